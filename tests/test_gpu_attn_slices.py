"""Slices of 64 rows instead of 128 in the gathered attention (few units): either side of the line, workspaces with and without
room for them, lists that end inside a slice; against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hd,group", [(64, 4), (128, 4), (128, 12)])
@pytest.mark.parametrize("units,n_idx", [(1, 1), (1, 63), (1, 64), (1, 65), (8, 2047), (8, 2048), (8, 2049), (16, 1000), (257, 40)])
def test_slices_of_64_rows_match_float64(units, n_idx, hd, group):
    from diffcache_amd import _hip as hip
    n = 2500
    g = torch.Generator(device=DEV).manual_seed(units * n_idx + hd)
    k, v = (torch.randn((1, units, n, hd), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((1, units * group, hd), generator=g, device=DEV).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(n, generator=g, device=DEV)[:n_idx] for _ in range(units)]).to(torch.int32)
    rows = idx.long()[:, :, None].expand(-1, -1, hd)
    kk, vv = k[0].gather(1, rows).double(), v[0].gather(1, rows).double()
    x = torch.matmul(q[0].double().view(units, group, hd), kk.transpose(1, 2).contiguous()) * hd ** -0.5
    want = torch.matmul(torch.softmax(x, dim=-1), vv).view(1, units * group, hd)
    kw = dict(n_idx=n_idx, region_lo=0, n_sink=0, recent_lo=n, n_recent=0)
    up = lambda x: (x + 255) // 256 * 256
    slices = units * ((n_idx + 127) // 128)
    least = up(slices * group * hd * 4) + up(slices * group * 8)      # room for the partials of slices of 128 rows
    assert least <= hip.lib.dc_attn_workspace_bytes(units, group, hd, n_idx)
    short = torch.empty((least + 255,), device=DEV, dtype=torch.uint8)
    short = short[-short.data_ptr() % 256:][:least]
    outs = [hip.gather_attn(q, k, v, idx, **kw), hip.gather_attn_static(q, k, v, idx, out=torch.empty_like(q), **kw),
            hip.gather_attn(q, k, v, idx, workspace=short, **kw)]
    for out in outs:
        # fp32 sums of at most 2049 weights that add up to one, then one rounding to bf16
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.parametrize("hd,group", [(64, 1), (128, 4), (128, 16)])
@pytest.mark.parametrize("units,n_idx,fine", [(1, 4096, True), (1, 4097, False), (4, 4096, True), (3, 5000, False), (1, 16000, False)])
def test_lists_of_more_slices_than_a_merge_takes_at_once(units, n_idx, fine, hd, group):
    """From 65 slices of 64 rows on a unit's list is split in slices of 128, with room for more or without: the same results bit for bit."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n_idx + hd)
    k, v = (torch.randn((1, units, 16384, hd), generator=g, device=DEV).to(torch.bfloat16) for _ in range(2))
    q = torch.randn((1, units * group, hd), generator=g, device=DEV).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(16384, generator=g, device=DEV)[:n_idx] for _ in range(units)]).to(torch.int32)
    rows = idx.long()[:, :, None].expand(-1, -1, hd)
    kk, vv = k[0].gather(1, rows).double(), v[0].gather(1, rows).double()
    x = torch.matmul(q[0].double().view(units, group, hd), kk.transpose(1, 2).contiguous()) * hd ** -0.5
    want = torch.matmul(torch.softmax(x, dim=-1), vv).view(1, units * group, hd)
    up = lambda x: (x + 255) // 256 * 256
    slices = units * ((n_idx + 127) // 128)
    outs, lses = [], []
    for nbytes in (up(slices * group * hd * 4) + up(slices * group * 8), 32 << 20):
        ws = torch.empty((nbytes + 255,), device=DEV, dtype=torch.uint8)
        ws = ws[-ws.data_ptr() % 256:][:nbytes]
        lses.append(torch.empty((1, units * group), device=DEV))
        outs.append(hip.gather_attn(q, k, v, idx, n_idx=n_idx, region_lo=0, n_sink=0, recent_lo=16384, n_recent=0, workspace=ws, lse=lses[-1]))
        # fp32 sums of weights that add up to one, then one rounding to bf16
        assert bool(((outs[-1].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        assert bool(((lses[-1].double() - torch.logsumexp(x, dim=-1).view(1, -1)).abs() < 1e-4).all())
    assert fine or (torch.equal(outs[0], outs[1]) and torch.equal(lses[0], lses[1]))
