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


@pytest.mark.parametrize("hd,qg", [(64, 1), (128, 4), (256, 3)])
@pytest.mark.parametrize("rows", [237, 5003])
@pytest.mark.parametrize("mode", [0, 1])
def test_rows_without_a_number_are_selected_as_by_the_bf16_scan(mode, rows, hd, qg):
    """Infinite and undefined keys leave no bound: every row goes to the exact pass, also one whose approximation overflows, and a
    selection of all rows names all of them."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device="cuda").manual_seed(rows + hd)
    h = 6
    k = torch.randn((1, h, rows, hd), generator=g, device="cuda")
    for u, bad in enumerate((float("inf"), -float("inf"), float("nan"), 3e38, 1e-39)):
        k[0, u, torch.randint(0, rows, (20,), generator=g, device="cuda"), torch.randint(0, hd, (20,), generator=g, device="cuda")] = bad
    k = k.to(torch.bfloat16)
    q = (2 * torch.randn((h * qg, hd), generator=g, device="cuda")).to(torch.bfloat16)
    k[0, 5, rows // 2, 7] = float("inf")
    q[5 * qg:, 7] = 0.0                     # an infinite residual times zero
    sk = hip.Sketch(k).build(k, 0, rows)
    for budget in (rows, rows - 3, 200):
        want = hip.score_select(k, q, 0, rows, budget, mode=mode, order=hip.ORDER_BEST, q_group=qg)
        got = hip.score_select_sketch(k, sk, q, 0, rows, budget, mode=mode, order=hip.ORDER_BEST, q_group=qg)
        assert torch.equal(got, want), budget
