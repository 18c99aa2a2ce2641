"""The group mean that the scans work out for themselves (dc_load_query) against dc_group_mean_bf16, for every way it goes: one
head, up to four, up to eight, more; powers of two, which are multiplied by the reciprocal, and other sizes, which are divided."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 7, 8, 9, 16, 17])
def test_scores_of_a_group_are_those_of_its_mean(group, hd):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(group * hd)
    k = torch.randn((2, 3, 300, hd), generator=g, device=DEV).to(torch.bfloat16)
    q = (torch.randn((2, 3 * group, hd), generator=g, device=DEV) * torch.exp(4 * torch.randn((2, 3 * group, hd), generator=g, device=DEV)))
    q = q.to(torch.bfloat16)
    q[0, :group] = 0.0                      # a mean of zeros of either sign
    q[0, 0] = -0.0
    mean = hip.group_mean(q, group, hd=hd)
    for mode in (hip.MODE_IP, hip.MODE_REF_DIST):
        assert torch.equal(hip.score(k, q, 0, 300, mode=mode, q_group=group), hip.score(k, mean, 0, 300, mode=mode))
