"""dc_decode_layer_step: the token's row and the step count carried along by a layer's own launches, against
dc_append_kv_bf16 + dc_decode_layer + dc_step_state_advance, on every route."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("route,hd,group,n,budget", [
    ("one_kernel", 128, 4, 3000, 256), ("one_kernel", 64, 1, 700, 64), ("one_kernel", 256, 8, 2048, 128),
    ("sketch", 128, 4, 9001, 512), ("sketch", 64, 7, 3000, 300), ("sketch", 256, 16, 2500, 100),
    ("stream", 128, 1, 5000, 512), ("stream", 256, 4, 2111, 64),
    ("attend_only", 128, 4, 3000, 0),
])
def test_a_step_carried_along_equals_the_three_calls(route, hd, group, n, budget):
    from diffcache_amd import _hip as hip
    b, h, sink, cap = 2, 3, 4, 32
    g = torch.Generator(device=DEV).manual_seed(n + hd)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    stores = [[rnd(b, h, n + sink + cap + 1, hd) for _ in range(2)]]
    stores.append([t.clone() for t in stores[0]])
    q = rnd(b, h * group, hd)
    hi = n + sink
    ws = [hip.alloc_workspace(hip.layer_workspace_bytes(b * h, n, budget, group, hd, budget + sink + cap + 1), DEV)
          for _ in range(2)]
    idx = [torch.zeros((b * h, max(budget, 1)), device=DEV, dtype=torch.int32) for _ in range(2)]
    out = [torch.empty_like(q) for _ in range(2)]
    # the window's first row, one inside, its last one, and a full window (nothing is stored, the step overflows)
    for count in (0, 5, cap - 1, cap):
        state = [torch.tensor([count, hi, hi + count, 0], device=DEV, dtype=torch.int32) for _ in range(2)]
        nk, nv = rnd(b, h, hd), rnd(b, h, hd)
        for i, (ks, vs) in enumerate(stores):
            sketch = None
            if route == "sketch":
                sketch = hip.Sketch(ks)
                sketch.build(ks, sink, n)
            kw = dict(sketch=sketch, n_recent_dev=state[i][0:1], order=hip.ORDER_INDEX if budget else hip.ORDER_ANY,
                      one_kernel=hip.ONE_KERNEL_NEVER)
            if route == "one_kernel":
                kw.update(order=hip.ORDER_ANY, one_kernel=hip.ONE_KERNEL_EXCLUSIVE)
            args = (q, ks, vs, sink, hi, cap, budget, None, idx[i], out[i], ws[i], nk, nv)
            if i == 0:
                hip.append_kv(ks, vs, nk, nv, hi, pos_dev=state[i][0:1], pos_end=hi + cap)
                hip.decode_layer(*args, **kw)
                hip.step_state_advance(state[i], 1, cap)
            else:
                hip.decode_layer(*args, append=(hi, state[i][0:1], hi + cap), advance=(state[i], cap), **kw)
                assert hip.last_route() == {"one_kernel": hip.ROUTE_ONE_KERNEL, "sketch": hip.ROUTE_SKETCH,
                                            "stream": hip.ROUTE_STREAM, "attend_only": hip.ROUTE_ATTEND_ONLY}[route]
        for a, c in zip(*stores):
            assert torch.equal(a, c)
            if count < cap:
                assert torch.equal(c[:, :, hi + count], nk if c is stores[1][0] else nv)
        if route == "one_kernel":
            # a block adds its rows in the order they were found, which differs between two launches: sums of at
            # most 300 terms of weight <= 1 in fp32 (300 * 2^-24 * |v| < 1e-4), then one bf16 rounding (2^-8)
            x, y = out[0].float(), out[1].float()
            assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-4).all())
        else:
            assert torch.equal(out[0], out[1])
        assert state[0].tolist() == state[1].tolist()
        assert state[1].tolist() == [min(count + 1, cap), hi, hi + min(count + 1, cap), int(count == cap)]


def test_a_step_s_arguments_are_checked():
    from diffcache_amd import _hip as hip
    ks = torch.zeros((1, 1, 64, 64), device=DEV, dtype=torch.bfloat16)
    q = torch.zeros((1, 1, 64), device=DEV, dtype=torch.bfloat16)
    ws = hip.alloc_workspace(hip.layer_workspace_bytes(1, 40, 8, 1, 64, 30), DEV)
    idx = torch.zeros((1, 8), device=DEV, dtype=torch.int32)
    args = (q, ks, ks, 4, 44, 16, 8, None, idx, torch.empty_like(q), ws)
    for nk, append in ((None, (44, None, 60)), (q, (-1, None, 60)), (q, (64, None, 64)), (q, (44, None, 44)),
                       (q[..., :32].contiguous(), (44, None, 60))):
        with pytest.raises(hip.DiffCacheError):
            hip.decode_layer(*args, nk, nk, append=append)
    with pytest.raises(hip.DiffCacheError):
        hip.decode_layer(*args, q, q, advance=(torch.zeros(4, dtype=torch.int32), 16))
