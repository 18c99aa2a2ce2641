"""The dense bf16 scan (from 769 rows a unit to 1.75 Mi over all units: a 32-bit key for every row at the row's own place, classified in
tiles of 4096 rows): the edges of its blocks' shares and of those tiles, with ties, and live ends in front of the
capacity, for the sketch's dense scan as well.  Ids against oracle.topk_select of the GPU's dense scores (nsw.rs:592-630)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def keys_of(law, shape, g):
    k = torch.randn(shape, generator=g, device=DEV) * torch.exp(torch.randn((*shape[:2], 1, shape[3]), generator=g, device=DEV))
    if law == "integers":
        k = torch.randint(-1, 2, shape, generator=g, device=DEV).float()
    elif law == "equal":
        k[:, :, 1:] = k[:, :, :1]
    return k.to(torch.bfloat16).contiguous()


# 65549 rows a unit at 256 columns: more tiles than blocks; 458753 x 4 units: just beyond, where the scan lists its survivors
@pytest.mark.parametrize("hd,hkv", [(64, 3), (128, 2), (256, 1)])
@pytest.mark.parametrize("region", [1, 2, 255, 257, 4095, 4097, 65549, 262145])
@pytest.mark.parametrize("law", ["outliers", "integers", "equal"])
def test_dense_keys_are_exact_at_their_edges(law, hd, hkv, region):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(hd + region)
    k = keys_of(law, (1, hkv, region + 9, hd), g)
    q = torch.randn((hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
    for mode, budget in ((0, 1500), (1, 1), (1, 5000)):
        k_eff = min(budget, region)
        ws = hip.alloc_workspace(hip.score_select_workspace_bytes(hkv, region, budget), DEV)
        dense = hip.score(k, q, 4, region, mode).cpu().numpy()
        for order in (hip.ORDER_BEST, hip.ORDER_ANY):
            ids = hip.score_select(k, q, 4, region, budget, mode, order, workspace=ws).cpu().numpy()
            for u in range(hkv):
                want = orc.topk_select(dense[u], k_eff, mode)
                got = ids[u] if order == hip.ORDER_BEST else np.sort(ids[u])
                assert np.array_equal(got, want if order == hip.ORDER_BEST else np.sort(want)), (mode, budget, order, u)


@pytest.mark.parametrize("units_rows", [(4, 458752), (4, 458753), (600, 300)])
def test_both_sides_of_the_line_and_more_units_than_blocks(units_rows):
    from diffcache_amd import _hip as hip
    hkv, region = units_rows
    g = torch.Generator(device=DEV).manual_seed(region)
    k = keys_of("integers", (1, hkv, region, 64), g)
    q = torch.randn((hkv, 64), generator=g, device=DEV).to(torch.bfloat16)
    dense = hip.score(k, q, 0, region, 0).cpu().numpy()
    ids = hip.score_select(k, q, 0, region, 100, 0, hip.ORDER_BEST).cpu().numpy()
    for u in range(0, hkv, max(1, hkv // 8)):
        assert np.array_equal(ids[u], orc.topk_select(dense[u], 100, 0)), u


@pytest.mark.parametrize("sketch", [False, True])
def test_the_live_end_comes_from_the_device(sketch):
    """Launches laid out for 40 Ki rows, ends of less: the places behind the end hold no row."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(9)
    hkv, hd, cap, budget, sink = 3, 128, 40963, 700, 4
    k = keys_of("integers", (1, hkv, sink + cap, hd), g)
    q = torch.randn((1, hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, sink, cap) if sketch else None
    ws = hip.alloc_workspace(hip.layer_workspace_bytes(hkv, cap, budget, 1, hd, budget + sink), DEV)
    state = torch.zeros((4,), device=DEV, dtype=torch.int32)
    for i, region in enumerate((cap, 40961, 4096, 4097, 8195, 703, 700, cap - 1)):
        state[1:2].fill_(sink + region)
        idx = torch.full((hkv, budget), -1, device=DEV, dtype=torch.int32)
        hip.decode_layer(q, k, k, sink, sink + cap, 0, budget, None, idx, torch.empty_like(q), ws, mode=0, order=hip.ORDER_BEST,
                         one_kernel=hip.ONE_KERNEL_NEVER, select_state_ready=i > 0, sketch=sk,
                         n_recent_dev=state[0:1], region_hi_dev=state[1:2])
        dense = hip.score(k, q.view(hkv, hd), sink, region, 0).cpu().numpy()
        for u in range(hkv):
            assert np.array_equal(idx[u].cpu().numpy(), orc.topk_select(dense[u], budget, 0)), (region, u)


# up to 768 rows a unit the scan lists its survivors; up to 640 tiles of 256 rows in all every tile is a block's; other grids
# from 64 units on and above 1 Mi rows
@pytest.mark.parametrize("hkv,region,hd", [(3, 768, 64), (3, 769, 128), (2, 1023, 256), (24, 5424, 64), (24, 7000, 64), (64, 2561, 64),
                                           (33, 33000, 64), (16, 70001, 64), (9, 120001, 256)])
def test_every_grid_scans_every_row(hkv, region, hd):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(hkv + region)
    k = torch.randint(-1, 2, (1, hkv, region, hd), generator=g, device=DEV, dtype=torch.int8).to(torch.bfloat16)
    q = torch.randn((hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
    budget = min(region, 700)
    ws = hip.alloc_workspace(hip.score_select_workspace_bytes(hkv, region, budget), DEV)
    dense = hip.score(k, q, 0, region, 0)
    for order in (hip.ORDER_BEST, hip.ORDER_ANY):
        ids = hip.score_select(k, q, 0, region, budget, 0, order, workspace=ws).cpu().numpy()
        for u in range(0, hkv, 1 + hkv // 5):
            want, got = orc.topk_select(dense[u].cpu().numpy(), budget, 0), ids[u] if order == hip.ORDER_BEST else np.sort(ids[u])
            assert np.array_equal(got, want if order == hip.ORDER_BEST else np.sort(want)), (order, u)


@pytest.mark.parametrize("hkv,region,hd", [(64, 2561, 128), (700, 800, 128), (520, 1500, 256), (100, 5000, 256), (7, 20000, 128), (24, 7000, 128),
                                           (5, 300001, 128), (63, 9000, 128)])
def test_rotated_chunks_scan_every_row(hkv, region, hd):
    """More units than chunks, fewer, numbers that do not divide; blocks of one, two, three and more steps."""
    test_every_grid_scans_every_row(hkv, region, hd)
