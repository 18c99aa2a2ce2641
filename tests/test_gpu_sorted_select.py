"""Best-first selection in one pass (select_sorted_kernel) against the dense route, which selects and sorts in
separate kernels: list lengths around the LDS capacity, selections up to the longest, keys that crowd."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _keys(law, n, g):
    k = torch.randn((1, 2, n, 64), generator=g, device=DEV)
    if law == "equal":              # one bin, ties by id throughout
        k[:] = k[:, :, :1]
    elif law == "steps":            # seven values, thousands of each
        k[:] = k[:, :, :1] * (1 + torch.arange(n, device=DEV) % 7).view(1, 1, n, 1)
    elif law == "outlier":          # one key far above the rest: the counting pass sees two bins
        k[:, :, n // 2] *= 1e4
    return k.to(torch.bfloat16)


@pytest.mark.parametrize("law,n,k", [
    ("normal", 1, 1), ("normal", 129, 128), ("normal", 5000, 1), ("normal", 5000, 1024), ("normal", 5000, 5000),
    ("normal", 60000, 4096), ("normal", 60000, 4097), ("equal", 3000, 700), ("equal", 12288, 4096),
    ("equal", 12289, 4096), ("steps", 9000, 2000), ("outlier", 20000, 2048),
])
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("sketch", [False, True])
def test_best_first_selection_matches_the_dense_route(law, n, k, mode, sketch):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n + k)
    store = _keys(law, n, g)
    q = torch.randn((2, 64), generator=g, device=DEV).to(torch.bfloat16)
    want = hip.topk_select(hip.score(store, q, 0, n, mode), k, mode, hip.ORDER_BEST)
    if sketch:
        sk = hip.Sketch(store).build(store, 0, n)
        ws = hip.alloc_workspace(hip.sketch_select_workspace_bytes(2, n, k), DEV)
        for ready in (False, True):         # the second call finds the state the first left
            got = hip.score_select_sketch(store, sk, q, 0, n, k, mode, hip.ORDER_BEST, workspace=ws, state_ready=ready)
            assert torch.equal(got, want)
    else:
        assert torch.equal(hip.score_select(store, q, 0, n, k, mode, hip.ORDER_BEST), want)
