"""The PQ scan and its classify pass (buckets at the keys' own places) at the edges of their shares and tiles, with
ties, against the stepwise entry points (dense ADC scores, dc_topk_select), which add in the same order."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# around a wave (64 keys), a step of a block (1024), a tile of the classify pass (8192); more units than blocks
@pytest.mark.parametrize("b,h,n", [(1, 1, 1), (1, 2, 63), (1, 3, 1025), (2, 2, 8191), (1, 1, 8193), (1, 3, 40961), (20, 16, 1100)])
@pytest.mark.parametrize("m", [16, 32])
@pytest.mark.parametrize("law", ["codes", "few_codes", "one_code"])
def test_search_equals_the_stepwise_chain(b, h, n, m, law):
    from diffcache_amd.pq import PQIndex
    g = torch.Generator(device=DEV).manual_seed(n + m)
    hd = 64
    books = torch.randn((h, m, 256, hd // m), generator=g, device=DEV)
    most = {"codes": 256, "few_codes": 2, "one_code": 1}[law]     # ties by the dozen; every key a candidate
    codes = torch.randint(0, most, (b * h, n, m), generator=g, device=DEV, dtype=torch.uint8)
    if law == "few_codes":
        codes[:, :, 3:] = 7
    keys = torch.randn((b, h, n, hd), generator=g, device=DEV).to(torch.bfloat16)
    for n_cand, topk in ((300, 100), (1, 1), (2048, 300)):
        index = PQIndex(keys, books, codes, n_cand=n_cand, topk=topk)
        q = torch.randn((b * h, hd), generator=g, device=DEV).to(torch.bfloat16)
        want = index.search_stepwise(q)
        for _ in range(2):      # the second search finds the state as the first one left it
            assert torch.equal(index.search(q), want), (n_cand, topk)


# a block of the classify pass takes 2048 keys of short units, else 8192; above 512 or 1280 candidates it walks its keys in order
@pytest.mark.parametrize("b,h,n", [(1, 1, 512), (1, 2, 513), (1, 3, 2047), (1, 2, 2049), (1, 1, 262144), (1, 1, 262145), (16, 16, 8193)])
@pytest.mark.parametrize("m", [16, 32])
@pytest.mark.parametrize("most", [1, 2])
def test_many_candidates(b, h, n, m, most):
    from diffcache_amd.pq import PQIndex
    g = torch.Generator(device=DEV).manual_seed(n + m)
    hd = 64
    books = torch.randn((h, m, 256, hd // m), generator=g, device=DEV)
    codes = torch.full((b * h, n, m), 9, device=DEV, dtype=torch.uint8)
    codes[:, :, 0] += torch.randint(0, most, (b * h, n), generator=g, device=DEV, dtype=torch.uint8)
    keys = torch.randn((b, h, n, hd), generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn((b * h, hd), generator=g, device=DEV).to(torch.bfloat16)
    for n_cand in (1, min(n, 400), min(n, 3000)):
        index = PQIndex(keys, books, codes, n_cand=n_cand, topk=(n_cand + 1) // 2)
        assert torch.equal(index.search(q), index.search_stepwise(q)), n_cand
