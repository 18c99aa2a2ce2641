"""The sketch scan's integer weights (sketch_prune_kernel): every head dim's lane layout at row counts around a
wave's 64 rows and a block's 256, and weights whose largest is far from the rest, against the dense route."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _query(law, units, hd, g):
    q = torch.randn((units, hd), generator=g, device=DEV)
    if law == "outlier":        # one weight holds nearly all of the score: the others sit in the low digits
        q[:, hd // 3] *= 3e5
    elif law == "zero":
        q.zero_()
    elif law == "one_column":   # every other digit is zero, the last column of the last lane
        q[:, :-1] = 0
    elif law == "tiny":
        q *= 1e-30
    elif law == "huge":
        q *= 1e30
    return q.to(torch.bfloat16)


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("n,k", [(1, 1), (63, 5), (65, 64), (257, 100), (4096 + 17, 300), (20011, 1024)])
@pytest.mark.parametrize("law", ["normal", "outlier", "zero", "one_column", "tiny", "huge"])
def test_scan_keeps_the_top_rows(hd, n, k, law):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(hd + n)
    store = (torch.randn((1, 3, n + 2, hd), generator=g, device=DEV)
             * torch.exp(torch.randn((1, 3, 1, hd), generator=g, device=DEV))).to(torch.bfloat16)
    q = _query(law, 3, hd, g)
    sk = hip.Sketch(store).build(store, 1, n)
    for mode in (hip.MODE_IP, hip.MODE_REF_DIST):
        want = hip.topk_select(hip.score(store, q, 1, n, mode), k, mode, hip.ORDER_BEST)
        assert torch.equal(hip.score_select_sketch(store, sk, q, 1, n, k, mode, hip.ORDER_BEST), want)
