"""Codebook training and encoding for callers outside the encoding kernel's range (no GPU needed)."""
import pytest
import torch

from diffcache_amd.pq import train_codebooks


@pytest.mark.parametrize("n_centroids", [16, 256, 257, 600])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_training_is_lloyd_s_iteration_for_any_number_of_centroids(n_centroids, dtype):
    n, m, ds, iters = 3000, 2, 4, 3
    keys = torch.randn((n, m * ds), generator=torch.Generator().manual_seed(5)).to(dtype)
    got = train_codebooks(keys, m, iters=iters, seed=7, n_centroids=n_centroids)
    x, g = keys.float(), torch.Generator().manual_seed(7)
    for j in range(m):
        xs = x[:, j * ds:(j + 1) * ds].contiguous()
        c = xs[torch.randint(0, n, (n_centroids,), generator=g)].clone()
        for _ in range(iters):
            a = torch.cdist(xs, c).argmin(dim=1)
            for i in a.unique().tolist():
                c[i] = xs[a == i].mean(dim=0)
        # a cell's mean of at most 3000 values below 5 in fp32: 3000 * 2^-24 * 5 < 1e-3 on either side of
        # the sum's order; a key assigned to another cell moves means by 1e-2 and more
        assert torch.allclose(got[j], c, rtol=0.0, atol=1e-3), (got[j] - c).abs().max()


def test_no_keys_are_encoded_to_no_codes():
    """The C entry as well as the wrapper: an empty tensor's pointer is null, which is no error."""
    from diffcache_amd import _hip as hip
    assert hip.lib.dc_pq_encode_bf16(None, 128, 0, None, None, 32, 128, 32, 256, None) == 0
    assert hip.lib.dc_pq_encode_bf16(None, 128, 1, None, None, 32, 128, 32, 256, None) == -22
    assert hip.lib.dc_pq_encode_bf16(None, 128, 0, None, None, 32, 128, 33, 256, None) == -22


class Elsewhere:
    """What pq_encode_supported looks at of a tensor on some GPU."""

    def __init__(self, device, shape, dtype):
        self.device, self.shape, self.dtype, self.is_cuda = torch.device(device), shape, dtype, True

    def dim(self):
        return len(self.shape)

    def stride(self, i):
        return (self.shape[1], 1)[i]

    def data_ptr(self):
        return 4096


@pytest.mark.parametrize("keys_on,books_on,current,taken", [
    ("cuda:0", "cuda:0", 0, True), ("cuda:1", "cuda:1", 1, True),
    ("cuda:1", "cuda:1", 0, False),     # launched on GPU 0 it would work on GPU 1's memory, out of GPU 1's order
    ("cuda:0", "cuda:1", 0, False),     # torch's error, as for any two devices
])
def test_the_encoding_kernel_takes_operands_of_the_current_gpu_only(monkeypatch, keys_on, books_on, current, taken):
    from diffcache_amd import _hip as hip
    monkeypatch.setattr(torch.cuda, "current_device", lambda: current)
    keys, books = Elsewhere(keys_on, (100, 128), torch.bfloat16), Elsewhere(books_on, (32, 256, 4), torch.float32)
    assert hip.pq_encode_supported(keys, books) == taken


@pytest.mark.gpu
def test_no_keys_on_the_gpu():
    from diffcache_amd.pq import encode
    books = torch.zeros((32, 256, 4), device="cuda")
    for dtype in (torch.bfloat16, torch.float32):
        codes = encode(torch.zeros((0, 128), device="cuda", dtype=dtype), books)
        assert codes.shape == (0, 32) and codes.dtype == torch.uint8 and codes.is_cuda
