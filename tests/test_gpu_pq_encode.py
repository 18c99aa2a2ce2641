"""dc_pq_encode_bf16 against float64 distances."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,m,ds,nc", [
    (1, 32, 4, 256), (255, 32, 4, 256), (257, 16, 8, 256),      # below, at and past a block of 256 keys
    (3001, 32, 2, 256), (3001, 16, 16, 256),                    # the other subspace widths
    (700, 3, 4, 200), (513, 5, 8, 17), (300, 1, 4, 1),          # odd subspace counts, fewer centroids
])
def test_pq_encode_picks_a_nearest_centroid(n, m, ds, nc):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n * m + ds)
    x = torch.randn((n, m * ds + 16), generator=g, device=DEV).to(torch.bfloat16)[:, :m * ds]     # strided rows
    books = torch.randn((m, nc, ds), generator=g, device=DEV)
    if nc > 40:
        books[:, 33] = books[:, 7]          # equal centroids: the lower number
    codes = hip.pq_encode(x, books).long()
    assert codes.shape == (n, m) and int(codes.max()) < nc
    assert nc <= 40 or not bool((codes == 33).any())
    X, B = x.double().view(n, m, ds), books.double()
    for j in range(m):
        d = 0.5 * (B[j] ** 2).sum(-1)[None] - X[:, j] @ B[j].t()
        # ds + 3 fp32 roundings of terms no larger than their sum of magnitudes, on either side
        size = 0.5 * (B[j] ** 2).sum(-1)[None] + X[:, j].abs() @ B[j].abs().t()
        err = (ds + 3) * 2.0 ** -24 * size.amax(dim=1)
        got = d.gather(1, codes[:, j:j + 1])[:, 0]
        assert bool((got <= d.amin(dim=1) + 2 * err).all())
    if m == 32 and ds == 4 and n > 1:
        # a single nearest centroid wherever fp32 can tell: at most a handful of keys are undecided
        exact = torch.stack([torch.cdist(X[:, j], B[j]).argmin(1) for j in range(m)], 1)
        assert (exact != codes).float().mean() < 1e-3


@pytest.mark.parametrize("ds,nc", [(4, 17), (8, 33), (4, 255)])
def test_pq_encode_names_an_existing_centroid_for_any_key(ds, nc):
    """Keys whose products leave the range of fp32, and infinite and undefined ones, get the number of a
    centroid that exists, and leave the other keys' codes as they were."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(nc)
    x = torch.randn((600, 3 * ds), generator=g, device=DEV).to(torch.bfloat16)
    books = torch.randn((3, nc, ds), generator=g, device=DEV).abs() + 1.0
    plain = hip.pq_encode(x, books)
    odd = x.clone()
    for row, value in ((0, -3.3e38), (5, 3.3e38), (17, float("inf")), (33, float("-inf")), (64, float("nan"))):
        odd[row] = value
        odd[row + 300, 1] = value
    codes = hip.pq_encode(odd, books)
    assert int(codes.max()) < nc
    same = (odd == x).all(dim=1)
    assert torch.equal(codes[same], plain[same])


def test_encode_takes_what_it_took_before():
    """fp32 keys and subspace widths the kernel is not built for still go through torch's distances."""
    from diffcache_amd.pq import encode
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn((400, 24), generator=g, device=DEV)
    for m in (2, 6):
        books = torch.randn((m, 16, 24 // m), generator=g, device=DEV)
        for keys in (x, x.to(torch.bfloat16)):
            want = torch.stack([torch.cdist(keys.float().view(400, m, -1)[:, j].contiguous(), books[j]).argmin(1)
                                for j in range(m)], 1)
            assert (encode(keys, books).long() != want).float().mean() < 1e-2


@pytest.mark.parametrize("m,ds,n", [(32, 4, 33000), (3, 2, 90001), (16, 8, 33000), (5, 16, 30001), (300, 2, 700)])
def test_codes_do_not_depend_on_how_many_keys_there_are(m, ds, n):
    """Many keys: a block's waves take several batches each (from 2 ** 15 keys on at 8 columns of blocks), odd numbers of
    subspaces and columns of blocks that outnumber the CUs.  The same keys a few hundred at a time, a batch per wave, get the same codes."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn((n, m * ds), generator=g, device=DEV).to(torch.bfloat16)
    books = torch.randn((m, 256, ds), generator=g, device=DEV)
    codes = hip.pq_encode(x, books)
    for lo in (0, n // 2 - 100, n - 401):
        assert torch.equal(codes[lo:lo + 401], hip.pq_encode(x[lo:lo + 401].contiguous(), books))
    far = torch.randn((0, m * ds), device=DEV).to(torch.bfloat16)
    assert hip.pq_encode(far, books).shape == (0, m)


@pytest.mark.parametrize("m,ds,n", [(5, 8, 33000), (6, 16, 20001), (12, 8, 33000), (7, 2, 90001), (33, 4, 20001), (96, 2, 9001), (136, 2, 5003),
                                    (1, 8, 33000), (27, 16, 3001), (1040, 2, 700)])
def test_codes_of_columns_that_do_not_divide_the_grid(m, ds, n):
    """Columns of subspaces that do not divide an XCD's CUs, a last column of fewer subspaces, more columns than CUs."""
    test_codes_do_not_depend_on_how_many_keys_there_are(m, ds, n)


@pytest.mark.parametrize("m,ds,like,n", [(12, 8, 16, 200003), (24, 4, 32, 200003), (96, 2, 64, 100003), (272, 2, 128, 60001)])
def test_a_subspace_takes_no_longer_where_their_number_is_no_power_of_two(m, ds, like, n):
    """Blocks that the CUs or the XCDs hold unequal numbers of are twice as long; `like` subspaces fill both evenly."""
    from diffcache_amd import _hip as hip
    took = []
    for mm in (m, like):
        x = torch.randn((n, mm * ds), device=DEV).to(torch.bfloat16)
        books = torch.randn((mm, 256, ds), device=DEV)
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            hip.pq_encode(x, books)
            a.record()
            for _ in range(5):
                hip.pq_encode(x, books)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        took.append(min(times) / mm)
    assert took[0] < 1.3 * took[1]
