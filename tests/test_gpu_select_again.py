"""One scan, selected from several times: dc_sparse_select with reinit = 0 leaves histogram and survivors as the scan left
them, so any budget up to the scanned one may follow, in any order of ids; with reinit = 1 the next scan finds a cleared
state.  On both sides of the dense scan's line (1.75 Mi rows).  Against oracle.topk_select (nsw.rs:592-630)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("h,n", [(3, 20000), (4, 458753), (1, 700), (40, 4097)])
@pytest.mark.parametrize("mode", [0, 1])
def test_a_scan_can_be_selected_from_again(h, n, mode):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n + mode)
    k = torch.randn((1, h, n, 64), generator=g, device=DEV).to(torch.bfloat16)
    most = min(3000, n)
    ws = hip.alloc_workspace(hip.score_select_workspace_bytes(h, n, most), DEV)
    tail = (ws.data_ptr(), ws.numel(), hip._stream())
    idx = torch.zeros((h, most), device=DEV, dtype=torch.int32)
    hip._check(hip.lib.dc_select_state_init(h, n, most, *tail))
    for scan in range(2):
        q = torch.randn((h, 64), generator=g, device=DEV).to(torch.bfloat16)
        hip._check(hip.lib.dc_score_prune_bf16(k.data_ptr(), q.data_ptr(), 1, h, n, 64, h * n * 64, n * 64, 64, 1, most, mode, *tail))
        dense = hip.score(k, q, 0, n, mode).cpu().numpy()
        turns = [(most, hip.ORDER_ANY), (most // 3, hip.ORDER_ANY), (17, hip.ORDER_BEST), (most, hip.ORDER_BEST), (1, hip.ORDER_ANY),
                 (most // 2, hip.ORDER_BEST), (most // 2, hip.ORDER_ANY)]
        for i, (budget, order) in enumerate(turns):
            idx.fill_(-1)
            hip._check(hip.lib.dc_sparse_select(idx.data_ptr(), most, h, n, budget, mode, order, int(i == len(turns) - 1), *tail))
            got = idx[:, :budget].cpu().numpy()
            for u in range(0, h, 1 + h // 4):
                want = orc.topk_select(dense[u], budget, mode).astype(np.int64)
                ids = got[u].astype(np.int64)
                assert np.array_equal(ids if order == hip.ORDER_BEST else np.sort(ids), want if order == hip.ORDER_BEST else np.sort(want)), (scan, i, u)
