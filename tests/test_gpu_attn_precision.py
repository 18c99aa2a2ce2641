"""Softmax weights are kept to 32 bits in P V, by the kernels with matrix instructions (csrc/dc_attn.h) as by the one
without (csrc/small.hip): values of either sign whose weights differ in the eleventh bit (base.py:134-142)."""
import pytest
import torch

DEV = "cuda:0"


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("route", ["short", "five_kernels", "one_kernel"])
def test_weights_are_kept_to_32_bits(route, hd):
    from diffcache_amd import _hip as hip
    n, group = 192, 4
    # a third of the rows each: weight 1 and value 0; weight exp(-s) and value 1; weight exp(-s - d) and value -1
    third = torch.arange(n) % 3
    k = torch.zeros((1, 1, n, hd))
    k[0, 0, :, 0] = -(third > 0).float()
    k[0, 0, :, 1] = -(third == 2).float()
    v = ((third == 1).float() - (third == 2).float()).reshape(1, 1, n, 1).expand(1, 1, n, hd)
    q = torch.zeros((1, group, hd))
    q[0, :, 0] = torch.tensor([0.3, 0.5, 0.6, 0.75])
    q[0, :, 1] = 2.0 ** -11
    k, v, q = (t.to(DEV, torch.bfloat16).contiguous() for t in (k, v, q))
    s, d = q[0, :, 0].double(), q[0, :, 1].double()
    pa, pb = torch.exp(-s), torch.exp(-s - d)
    want = (pa - pb) / (1.0 + pa + pb)
    out = torch.empty((1, group, hd), device=DEV, dtype=torch.bfloat16)
    idx = torch.empty((1, n), device=DEV, dtype=torch.int32)
    ws = hip.alloc_workspace(hip.layer_workspace_bytes(1, n, n, group, hd, n), DEV)
    args = (q, k, v, 0, n, 0, n, None, idx, out, ws)
    kw = dict(mode=hip.MODE_IP, scale=1.0, order=hip.ORDER_BEST if route == "five_kernels" else hip.ORDER_ANY,
              one_kernel=hip.ONE_KERNEL_EXCLUSIVE if route == "one_kernel" else hip.ONE_KERNEL_NEVER)
    assert (hip.decode_layer_route(*args, **kw) == hip.ROUTE_ONE_KERNEL) == (route == "one_kernel")
    assert hip.decode_layer_is_short(*args, **kw) == (route == "short")
    hip.decode_layer(*args, **kw)
    err = (out[0].double() / want[:, None] - 1.0).abs().max().item()
    # the output's rounding, 2^-9, and the two weights' own, a few 2^-24 of a weight over a difference of 2^-11 of it: 2^-10.
    # (weights of two bf16 values: 0.007 to 0.013)
    assert err < 2.0 ** -9 + 2.0 ** -10, err
