"""dc_gather_attn_bf16 at the edges of the merge kernel's batches of splits, against float64 attention."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


# a split is 128 rows (64 at head dim 256); a batch of the merge is 128, 64 and 32 splits
@pytest.mark.parametrize("hd,group,rows", [
    (64, 4, 1), (64, 1, 129), (64, 8, 16384), (64, 3, 16385), (128, 4, 128), (128, 7, 1025), (128, 4, 8192),
    (128, 4, 8193), (128, 2, 16500), (256, 4, 64), (256, 2, 257), (256, 4, 2048), (256, 4, 2049), (256, 1, 4200),
])
def test_merge_over_batches_of_splits(hd, group, rows):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(rows + hd)
    b, h = 2, 3
    k = torch.randn((b, h, rows, hd), generator=g, device=DEV).to(torch.bfloat16)
    v = (torch.randn((b, h, rows, hd), generator=g, device=DEV) + 1.0).to(torch.bfloat16)
    q = torch.randn((b, h * group, hd), generator=g, device=DEV).to(torch.bfloat16)
    # the last rows carry much of the weight: the largest logit is not in the first batch
    k[:, :, -1] = q.view(b, h, group, hd)[:, :, 0] / 2
    lse = torch.empty((b, h * group), device=DEV, dtype=torch.float32)
    out = hip.gather_attn(q, k, v, None, 0, 0, 0, 0, rows, lse=lse)
    K, V, Q = k.double().cpu(), v.double().cpu(), q.double().cpu().view(b, h, group, hd)
    logits = torch.matmul(Q, K.transpose(2, 3).contiguous()) / hd ** 0.5
    p = torch.softmax(logits, dim=-1)
    want = torch.matmul(p, V)
    # weights and output rounded to bf16 (2^-9 each, relative), twice that allowed
    bound = 2.0 ** -7 * torch.matmul(p, V.abs())
    got = out.double().cpu().view(b, h, group, hd)
    assert bool(((got - want).abs() <= bound).all())
    # fp32 logits of |x| < 2^6 and a sum of weights rounded to bf16 at most
    assert bool(((lse.double().cpu().view(b, h, group) - torch.logsumexp(logits, -1)).abs() <= 2.0 ** -8).all())
