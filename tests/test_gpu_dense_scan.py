"""The dense sketch scan (up to 4 Mi rows over all units: a bucket for every row at the row's own place, read back by the
exact pass in tiles of 2048 rows): the edges of its blocks' shares and of those tiles,
candidates that all sit in one tile.  Ids, best first, against oracle.topk_select of the GPU's dense scores
(nsw.rs:592-630)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("hd,hkv", [(64, 3), (128, 2), (256, 1)])
@pytest.mark.parametrize("region", [1, 255, 257, 2047, 2049, 40961, 262145])
def test_dense_scan_is_exact_at_its_edges(hd, hkv, region):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(hd + region)
    for law in ("outliers", "one_tile", "equal"):
        n = region + 9
        k = torch.randn((1, hkv, n, hd), generator=g, device=DEV) * torch.exp(torch.randn((1, hkv, 1, hd), generator=g, device=DEV))
        q = torch.randn((hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
        if law == "one_tile":       # every candidate between rows 100 and 1700: one block scores them in several rounds
            k[:, :, 100:1700] += 3.0 * torch.sign(q.float()).view(1, hkv, 1, hd)
        elif law == "equal":
            k[:, :, 1:] = k[:, :, :1]
        k = k.to(torch.bfloat16).contiguous()
        for mode, budget in ((0, 1500), (1, 1)):
            k_eff = min(budget, region)
            sk = hip.Sketch(k).build(k, 4, region)
            ws = hip.alloc_workspace(hip.sketch_select_workspace_bytes(hkv, region, budget), DEV)
            dense = hip.score(k, q, 4, region, mode).cpu().numpy()
            for ready in (False, True):
                ids = hip.score_select_sketch(k, sk, q, 4, region, budget, mode, hip.ORDER_BEST, workspace=ws, state_ready=ready)
                ids = ids.cpu().numpy()
                for u in range(hkv):
                    assert np.array_equal(ids[u], orc.topk_select(dense[u], k_eff, mode)), (law, mode, budget, ready, u)


# tiles of 512 rows up to 32 Ki rows a unit and 384 Ki in all, of 1024 up to 96 Ki and 1 Mi, of 2048 beyond
@pytest.mark.parametrize("hd,hkv,region", [(64, 3, 511), (128, 2, 513), (256, 2, 1025), (256, 1, 32768), (128, 1, 32769), (64, 2, 98304),
                                           (64, 1, 98305), (64, 24, 16384), (64, 24, 16385), (64, 16, 65536), (64, 16, 65537)])
def test_tiles_of_every_size_are_exact_at_their_edges(hd, hkv, region):
    test_dense_scan_is_exact_at_its_edges(hd, hkv, region)


@pytest.mark.parametrize("hkv,cap", [(3, 9001), (24, 20483)])
def test_the_live_end_cuts_a_tile_of_any_size(hkv, cap):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(cap)
    hd, budget, sink = 64, 300, 4
    k = torch.randn((1, hkv, sink + cap, hd), generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn((1, hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, sink, cap)
    ws = hip.alloc_workspace(hip.layer_workspace_bytes(hkv, cap, budget, 1, hd, budget + sink), DEV)
    state = torch.zeros((4,), device=DEV, dtype=torch.int32)
    for i, region in enumerate((cap, cap - 1, 8193, 8192, 4097, 1025, 513, 512, 303, 300, cap)):
        state[1:2].fill_(sink + region)
        idx = torch.full((hkv, budget), -1, device=DEV, dtype=torch.int32)
        hip.decode_layer(q, k, k, sink, sink + cap, 0, budget, None, idx, torch.empty_like(q), ws, mode=0, order=hip.ORDER_BEST,
                         one_kernel=hip.ONE_KERNEL_NEVER, select_state_ready=i > 0, sketch=sk,
                         n_recent_dev=state[0:1], region_hi_dev=state[1:2])
        dense = hip.score(k, q.view(hkv, hd), sink, region, 0).cpu().numpy()
        for u in range(0, hkv, 1 + hkv // 4):
            assert np.array_equal(idx[u].cpu().numpy(), orc.topk_select(dense[u], budget, 0)), (region, u)


# from 2.5 Mi rows in all on (128 columns) the scan lists its rows unless 1024 ids or more are selected
@pytest.mark.parametrize("region,budget", [(655360, 64), (655361, 64), (655361, 1023), (655361, 1024)])
def test_both_sides_of_the_line_for_few_ids(region, budget):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(region + budget)
    hkv, hd = 4, 128
    k = torch.randn((1, hkv, region, hd), generator=g, device=DEV, dtype=torch.bfloat16)
    q = torch.randn((hkv, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, 0, region)
    ws = hip.alloc_workspace(hip.sketch_select_workspace_bytes(hkv, region, budget), DEV)
    dense = hip.score(k, q, 0, region, 0).cpu().numpy()
    for ready in (False, True):
        ids = hip.score_select_sketch(k, sk, q, 0, region, budget, 0, hip.ORDER_BEST, workspace=ws, state_ready=ready).cpu().numpy()
        for u in range(hkv):
            assert np.array_equal(ids[u], orc.topk_select(dense[u], budget, 0)), (ready, u)
