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
