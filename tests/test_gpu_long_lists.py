"""More slices or chunks of one unit than the second dimension of a grid holds: an attended list of 4.2 Mi rows of 256 columns, a bf16
scan of 134 Mi rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_attention_over_more_slices_than_a_grid_dimension_holds():
    from diffcache_amd import _hip as hip
    hd, group, n = 256, 4, 65537 * 64 + 36
    g = torch.Generator(device=DEV).manual_seed(n)
    k, v = (torch.empty((1, 1, n, hd), device=DEV, dtype=torch.bfloat16).normal_(generator=g) for _ in range(2))
    q = torch.randn((1, group, hd), generator=g, device=DEV).to(torch.bfloat16)
    # rows that weigh about as much as all others together: either side of the places where a dimension ends, and the last
    far = [0, 32768 * 64 - 1, 32768 * 64, 65536 * 64 - 1, 65536 * 64, n - 1]
    for i, r in enumerate(far):
        k[0, 0, r] = q[0, i % group]
    out = hip.gather_attn(q, k, v, None, n_idx=0, region_lo=0, n_sink=0, recent_lo=0, n_recent=n)
    x = torch.cat([torch.matmul(q[0].double(), part.double().t()) for part in k[0, 0].split(1 << 19)], dim=1) * hd ** -0.5
    w = torch.softmax(x, dim=-1)
    want = sum(torch.matmul(a, part.double()) for a, part in zip(w.split(1 << 19, dim=1), v[0, 0].split(1 << 19)))
    # (a head's row scores |q|^2 / 16, the others' weights add up to n e^(1/2) = e^15.8: from |q|^2 = 200 on, 2.5 sigma below its mean, a share
    # of 0.036, which the tolerance below would not let go missing)
    assert float(w[:, far].sum(dim=1).min()) > 0.036
    # one rounding to bf16; fp32 sums of weights that add up to one, a slice's of 64 and one over the slices
    assert bool(((out[0].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


def test_scan_of_more_chunks_than_a_grid_dimension_holds():
    from diffcache_amd import _hip as hip
    hd, lead, chunk = 64, 16 * 256, 2048          # 16 blocks of one step, then blocks of eight
    n = lead + 65530 * chunk + 77
    g = torch.Generator(device=DEV).manual_seed(5)
    k = torch.empty((1, 1, n, hd), device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    q = torch.randn((1, hd), generator=g, device=DEV).to(torch.bfloat16)
    rows = [0, 255, 256, lead - 1, lead, n - 1, n - 78]
    for c in (1, 32750, 32751, 32752, 32753, 65518, 65519, 65520, 65529):
        rows += [lead + c * chunk - 1, lead + c * chunk]
    rows = sorted(set(rows))
    k[0, 0, rows] = 20 * q[0]                      # their score is some 8 times the largest of the others
    ids = hip.score_select(k, q, 0, n, len(rows), mode=hip.MODE_IP)
    assert sorted(ids[0].tolist()) == rows
