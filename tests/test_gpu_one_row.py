"""One row per unit and many units: the words that a dense scan leaves for a unit take 16 bytes, so the lists behind them
have to start after the last unit's.  Every unit's only row is its answer."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("units", [1, 33, 300])
def test_every_unit_finds_its_only_row(units):
    from diffcache_amd import _hip as hip
    from diffcache_amd.pq import PQIndex
    g = torch.Generator(device=DEV).manual_seed(units)
    hd, m = 64, 16
    k = torch.randn((1, units, 6, hd), generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn((units, hd), generator=g, device=DEV).to(torch.bfloat16)
    sk = hip.Sketch(k).build(k, 4, 1)
    for budget in (1, 7):
        for call in (lambda: hip.score_select(k, q, 4, 1, budget), lambda: hip.score_select_sketch(k, sk, q, 4, 1, budget)):
            for _ in range(3):
                assert torch.equal(call(), torch.zeros((units, 1), dtype=torch.int32, device=DEV)), budget
    index = PQIndex(k[:, :, :1].contiguous(), torch.randn((units, m, 256, hd // m), generator=g, device=DEV),
                    torch.randint(0, 256, (units, 1, m), generator=g, device=DEV, dtype=torch.uint8), n_cand=1, topk=1)
    for _ in range(3):
        assert torch.equal(index.search(q), torch.zeros((units, 1), dtype=torch.int32, device=DEV))
