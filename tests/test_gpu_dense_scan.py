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
