"""select_finish_kernel (ids in any order) at the edges of its lists: 8192 candidates stay in registers, 16384 in LDS, and
a threshold bin of more than 1024 is settled by radix passes.  Rows of few distinct scores make every row a candidate."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 1024, 1025, 8191, 8192, 8193, 16384, 16385])
@pytest.mark.parametrize("values", [1, 3, 40])      # distinct scores, all within the sketch's margin of each other
def test_the_best_of_a_list_of_any_length(n, values):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n + values)
    h, hd = 3, 64
    k = torch.randn((1, h, 1, hd), generator=g, device=DEV).expand(1, h, n, hd).contiguous()
    k *= 1.0 + torch.randint(0, values, (1, h, n, 1), generator=g, device=DEV) * 2.0 ** -7      # one step of bf16
    k = k.to(torch.bfloat16)
    q = torch.randn((h, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, 0, n)
    for mode in (0, 1):
        dense = hip.score(k, q, 0, n, mode).cpu().numpy()
        for budget in (1, n // 3 + 1, n):
            ids = hip.score_select_sketch(k, sk, q, 0, n, budget, mode, hip.ORDER_ANY).cpu().numpy()
            for u in range(h):
                want = orc.topk_select(dense[u], budget, mode).astype(np.int64)
                assert np.array_equal(np.sort(ids[u].astype(np.int64)), np.sort(want)), (mode, budget, u)


# lists that do not fit the LDS, of keys that tie: their ids settle the selection, counted in eight copies of a pass's bins
@pytest.mark.parametrize("n", [16385, 40001, 140001])
@pytest.mark.parametrize("values", [1, 2])
@pytest.mark.parametrize("order", ["ORDER_ANY", "ORDER_BEST", "ORDER_INDEX"])
def test_long_lists_of_ties(n, values, order):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(n + values)
    h, hd = 2, 64
    k = torch.randn((1, h, 1, hd), generator=g, device=DEV).expand(1, h, n, hd).contiguous()
    k *= 1.0 - 2.0 * torch.randint(0, values, (1, h, n, 1), generator=g, device=DEV)
    k = k.to(torch.bfloat16)
    q = torch.randn((h, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, 0, n)
    dense = hip.score(k, q, 0, n, 0).cpu().numpy()
    for budget in (1, 2000, n // 3):
        want = [orc.topk_select(dense[u], budget, 0).astype(np.int64) for u in range(h)]
        if order != "ORDER_BEST":
            want = [np.sort(w) for w in want]
        for got in (hip.score_select_sketch(k, sk, q, 0, n, budget, 0, getattr(hip, order)),
                    hip.score_select(k, q, 0, n, budget, 0, getattr(hip, order))):
            got = got.cpu().numpy().astype(np.int64)
            if order == "ORDER_ANY":
                got = np.sort(got, axis=1)
            assert np.array_equal(got, np.stack(want)), budget
