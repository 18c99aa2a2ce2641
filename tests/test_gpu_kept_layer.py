"""decode_layer with a LayerStep (arguments kept from step to step) against the same call without one: the struct is
filled anew whenever anything that it was filled from changes, and what is new in a call is checked in every call."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("with_sketch", [True, False])
def test_a_kept_layer_follows_its_tensors(with_sketch):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(31)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    b, h, group, hd, n, sink, cap, budget = 1, 2, 4, 64, 3000, 4, 8, 96
    hi = n - cap
    kept = hip.LayerStep()
    ks, vs, order = rnd(b, h, n, hd), rnd(b, h, n, hd), hip.ORDER_BEST

    def both(q, ks, vs, budget, state, ws, nk, nv, last):
        res, copies, count = [], (ks.clone(), vs.clone()), state.clone()
        for k in (kept, None):
            stores = (ks, vs) if k else copies      # the kept call works on the caller's own tensors
            sk = hip.Sketch(stores[0]).build(stores[0], sink, hi - sink) if with_sketch else None
            idx = torch.zeros((b * h, budget), device=DEV, dtype=torch.int32)
            out = torch.zeros((b, h * group, hd), device=DEV, dtype=torch.bfloat16)
            c = state if k else count
            hip.decode_layer(q, *stores, sink, hi, cap, budget, None, idx, out, ws, nk, nv, order=order, sketch=sk,
                             n_recent_dev=c[0:1], append=(hi, c[0:1], hi + cap), advance=(c, cap) if last else None, kept=k)
            torch.cuda.synchronize()
            res.append((idx, out, *stores, c.clone()))
        for x, y in zip(*res):
            assert torch.equal(x, y)

    ws = hip.alloc_workspace(hip.layer_workspace_bytes(b * h, hi - sink, 200, group, hd, 200 + sink + cap + 1), DEV)
    state = torch.tensor([2, hi, hi + 2, 0], device=DEV, dtype=torch.int32)
    q, nk, nv = rnd(b, h * group, hd), rnd(b, h, hd), rnd(b, h, hd)
    for last in (False, True, True):
        both(q, ks, vs, budget, state, ws, nk, nv, last)
    both(rnd(b, h * group, hd), ks, vs, budget, state, ws, rnd(b, h, hd), rnd(b, h, hd), True)  # a step's own tensors
    both(q, ks, vs, 150, state, ws, nk, nv, True)                                               # another size
    wide = rnd(b, h, n, 2 * hd)
    both(q, wide[..., :hd], wide[..., hd:], budget, state, ws, nk, nv, True)                    # other stores and strides
    both(q, ks, vs, budget, state.clone(), ws.clone(), nk, nv, True)                            # other counters, another workspace
    idx, out = torch.zeros((b * h, budget), device=DEV, dtype=torch.int32), torch.zeros((b, h * group, hd), device=DEV, dtype=torch.bfloat16)
    args = dict(order=order, n_recent_dev=state[0:1], append=(hi, state[0:1], hi + cap), kept=kept)
    good = (q, ks, vs, sink, hi, cap, budget, None, idx, out, ws, nk, nv)
    hip.decode_layer(*good, **args)
    for at, t in ((0, q.transpose(1, 2)), (0, q.cpu()), (9, out[:, :1]), (9, out.float()), (11, nk[:, :1]), (12, None), (12, nv.cpu())):
        with pytest.raises(hip.DiffCacheError):
            hip.decode_layer(*good[:at], t, *good[at + 1:], **args)
    with pytest.raises(hip.DiffCacheError):      # 32-bit ids only; a strided store's twin must share its strides
        hip.decode_layer(*good[:8], idx.long(), *good[9:], **args)
    with pytest.raises(hip.DiffCacheError):
        hip.decode_layer(q, ks, wide[..., :hd], *good[3:], **args)
    torch.cuda.synchronize()


def test_a_kept_layer_tells_the_append_positions_apart():
    """The token's row at pos + the window's counter, at pos + another counter, at pos alone: in any order, one LayerStep."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(32)
    rnd = lambda *s: torch.randn(s, generator=g, device=DEV).to(torch.bfloat16)
    b, h, group, hd, n, sink, cap, budget = 1, 2, 2, 64, 1000, 4, 8, 96
    hi = n - cap
    ws = hip.alloc_workspace(hip.layer_workspace_bytes(b * h, hi - sink, budget, group, hd, budget + sink + cap + 1), DEV)
    words = torch.tensor([2, 5], device=DEV, dtype=torch.int32)
    window, other = words[0:1], words[1:2]
    q, ks, vs = rnd(b, h * group, hd), rnd(b, h, n, hd), rnd(b, h, n, hd)
    idx, out = torch.zeros((b * h, budget), device=DEV, dtype=torch.int32), torch.zeros((b, h * group, hd), device=DEV, dtype=torch.bfloat16)
    kept = hip.LayerStep()
    for pos_dev, row in ((window, 2), (window, 2), (None, 0), (None, 0), (window, 2), (other, 5), (None, 0), (other, 5), (window, 2)):
        nk, nv, want_k, want_v = rnd(b, h, hd), rnd(b, h, hd), ks.clone(), vs.clone()
        want_k[:, :, hi + row], want_v[:, :, hi + row] = nk, nv
        hip.decode_layer(q, ks, vs, sink, hi, cap, budget, None, idx, out, ws, nk, nv, n_recent_dev=window,
                         append=(hi, pos_dev, hi + cap), kept=kept)
        torch.cuda.synchronize()
        assert torch.equal(ks, want_k) and torch.equal(vs, want_v), row
