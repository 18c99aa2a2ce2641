"""The chain of three kernels for short contexts (csrc/short.hip): every split of a unit finds the cutoff and its own
places of the list by itself, so what can go wrong is a split that counts differently from its neighbours or from the
oracle.  Ids against oracle.topk_select of the GPU's dense scores (nsw.rs:592-630, ties to the lower id), attention
against the float64 softmax over the oracle's rows (base.py:134-142)."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from oracle import oracle as orc

DEV = "cuda:0"


def bf16_rows(t):
    return t.cpu().view(torch.int16).numpy().view(np.uint16)


def keys_of(law, shape, g):
    b, h, n, hd = shape
    k = torch.randn(shape, generator=g, device=DEV)
    if law == "outliers":
        k *= torch.exp(torch.randn((1, h, 1, hd), generator=g, device=DEV))
    elif law == "integers":                     # ties by the dozen
        k = torch.randint(-2, 3, shape, generator=g, device=DEV).float()
    elif law == "two_values":                   # a threshold bucket of half the rows: not listed, ties settled by id
        k = torch.where(torch.rand((b, h, n, 1), generator=g, device=DEV) < 0.5, 1.0, -1.0) * k[:, :, :1]
    elif law == "constant":
        k = k[:, :, :1].expand(shape)
    elif law == "large":                        # scores beyond 32768, where d = 65536 - s has another grid than s
        k *= 3000.0
    elif law == "tiny":                         # every score in one bucket or in the negative half
        k *= 1e-7
    return k.to(torch.bfloat16).contiguous()


# region sizes at the edges of the key vectors per thread (2048 rows a vector; 2, 4, 8, 16 of them) and of a
# score block's parts; budgets at the edges of a split (128), beyond the region, and 1
@pytest.mark.gpu
@pytest.mark.parametrize("hd,group", [(64, 8), (128, 4), (256, 4), (128, 7)])
@pytest.mark.parametrize("law", ["outliers", "integers", "two_values", "constant", "large", "tiny"])
def test_short_chain_matches_the_oracle(law, hd, group):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(hd + group)
    for i, (region, budget) in enumerate([(64, 1), (65, 70), (511, 128), (2049, 129), (4096, 256), (4097, 1024), (8193, 127),
                                          (16385, 640), (32766, 1000)]):
        b, hkv, sink, recent, mode = 1, 2, i % 5, 13 * (i % 4), i % 2
        n, k_eff = sink + region + recent, min(budget, region)
        k, v = keys_of(law, (b, hkv, n, hd), g), torch.randn((b, hkv, n, hd), generator=g, device=DEV).to(torch.bfloat16)
        q = torch.randn((b, hkv * group, hd), generator=g, device=DEV).to(torch.bfloat16)
        ws = hip.alloc_workspace(hip.layer_workspace_bytes(b * hkv, region, budget, group, hd, k_eff + sink + recent), DEV)
        dense = hip.score(k, q, sink, region, mode, q_group=group).cpu().numpy()
        for ready in (False, True):             # the second call finds the state as the first one left it
            idx = torch.full((b * hkv, budget), -1, device=DEV, dtype=torch.int32)
            out = torch.empty((b, hkv * group, hd), device=DEV, dtype=torch.bfloat16)
            args = (q, k, v, sink, sink + region, recent, budget, None, idx, out, ws)
            kw = dict(mode=mode, order=hip.ORDER_ANY, one_kernel=hip.ONE_KERNEL_NEVER)
            assert hip.decode_layer_is_short(*args, **kw)
            hip.decode_layer(*args, select_state_ready=ready, **kw)
            torch.cuda.synchronize()
            for u in range(hkv):
                want = orc.topk_select(dense[u], k_eff, mode).astype(np.int64)
                got = idx[u, :k_eff].cpu().numpy().astype(np.int64)
                assert np.array_equal(np.sort(got), np.sort(want)), (region, budget, mode, ready, u)
                if law == "large":
                    # logits of 2e4: a sum of hd products in fp32 is good to hd * 2^-24 of sum |q k| * scale, 0.1 to 0.2
                    # here, so a softmax between near ties is not determined; the ids are what this law is for
                    continue
                rows = np.concatenate([want + sink, np.arange(sink), np.arange(sink + region, n)])
                o, _ = orc.sparse_attention(bf16_rows(q[0, u * group:(u + 1) * group]), bf16_rows(k[0, u])[rows],
                                            bf16_rows(v[0, u])[rows], None, None)
                x = out[0, u * group:(u + 1) * group].float().cpu().numpy()
                # outputs are convex sums of values, rounded to bf16 (2^-9); equal weights of equal values at most
                assert np.all(np.abs(x - o) <= np.maximum(2e-3, np.abs(o) * 2.0 ** -8)), (region, budget, mode, u)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [0, 1])
def test_rows_without_a_number_are_chosen_as_by_the_long_chain(mode):
    """Infinite and NaN elements: the ids of the streaming chain (best first; only the sets can be compared)."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(77)
    b, hkv, group, hd, region, budget = 1, 4, 2, 64, 5003, 300
    k = torch.randn((b, hkv, region, hd), generator=g, device=DEV)
    for u, bad in enumerate((float("inf"), -float("inf"), float("nan"), 3e38)):
        k[0, u, torch.randint(0, region, (40,), generator=g, device=DEV), 5] = bad
    k = k.to(torch.bfloat16)
    q = torch.randn((b, hkv * group, hd), generator=g, device=DEV).to(torch.bfloat16)
    ids = []
    for order in (hip.ORDER_ANY, hip.ORDER_BEST):
        ws = hip.alloc_workspace(hip.layer_workspace_bytes(b * hkv, region, budget, group, hd, budget), DEV)
        idx = torch.full((b * hkv, budget), -1, device=DEV, dtype=torch.int32)
        hip.decode_layer(q, k, k, 0, region, 0, budget, None, idx, torch.empty_like(q), ws, mode=mode, order=order,
                         one_kernel=hip.ONE_KERNEL_NEVER)
        torch.cuda.synchronize()
        ids.append(idx.sort(dim=1).values)
    assert torch.equal(*ids)


@pytest.mark.gpu
def test_the_live_end_of_the_region_comes_from_the_device():
    """Launches laid out for the largest region: shorter ends, the split's places and the padding of the last four keys
    move with the device word; every replay agrees with an eager call that passes the end as a size."""
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(5)
    b, hkv, group, hd, cap, budget, sink, window = 2, 2, 4, 128, 9001, 200, 4, 16
    n = sink + cap + window
    k, v = keys_of("integers", (b, hkv, n, hd), g), torch.randn((b, hkv, n, hd), generator=g, device=DEV).to(torch.bfloat16)
    q = torch.randn((b, hkv * group, hd), generator=g, device=DEV).to(torch.bfloat16)
    need = hip.layer_workspace_bytes(b * hkv, cap, budget, group, hd, budget + sink + window)
    ws = [hip.alloc_workspace(need, DEV) for _ in range(2)]
    state = torch.tensor([window, sink + cap, 0, 0], device=DEV, dtype=torch.int32)
    idx, out = [torch.zeros((b * hkv, budget), device=DEV, dtype=torch.int32) for _ in range(2)], [torch.empty_like(q) for _ in range(2)]

    def call(i, hi, ready, **kw):
        hip.decode_layer(q, k, v, sink, hi, window, budget, None, idx[i], out[i], ws[i], order=hip.ORDER_ANY,
                         select_state_ready=ready, one_kernel=hip.ONE_KERNEL_NEVER, **kw)
    on_device = dict(n_recent_dev=state[0:1], region_hi_dev=state[1:2])
    call(0, sink + cap, False, **on_device)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(0, sink + cap, True, **on_device)
    for region in (cap, 8192, 8191, 4094, 4095, 203, 200, cap - 1):
        state[1:2].fill_(sink + region)
        graph.replay()
        call(1, sink + region, False)
        torch.cuda.synchronize()
        # launches laid out for 4 Ki rows count in finer buckets, so the rows may come in another order: sums of at
        # most 221 terms of weight <= 1 in fp32 (221 * 2^-24 * |v| < 1e-4), then one bf16 rounding (2^-8) on either side
        assert torch.equal(idx[0].sort(dim=1).values, idx[1].sort(dim=1).values), region
        x, y = out[0].float(), out[1].float()
        assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-4).all()), region
        torch.randn(1000, device=DEV).sum().item()      # eager work between replays


def test_which_calls_take_the_short_chain():
    from diffcache_amd import _hip as hip

    def short(units=8, rows=4028, hd=128, group=4, order=hip.ORDER_ANY, budget=512, recent=64, sketch=0x1000, **kw):
        a = hip.LayerArgs()
        a.n_b, a.n_h, a.group, a.hd, a.budget, a.n_sink = 1, units, group, hd, budget, 4
        a.recent_lo, a.n_recent, a.order, a.kv_row_stride, a.sketch_codes = 4 + rows, recent, order, hd, sketch
        for name, value in kw.items():
            setattr(a, name, value)
        return hip.lib.dc_decode_layer_is_short(ctypes.byref(a))
    assert short() == short(sketch=None) == 1
    assert short(rows=64) == 1 and short(rows=63) == 0
    assert short(units=1, rows=32768) == 1 and short(units=1, rows=32769) == 0
    assert short(units=8, rows=32768, budget=4096) == 1 and short(units=9, rows=32768, budget=4096) == 0    # 64 MiB of keys
    assert short(units=7, rows=32768) == 1 and short(units=8, rows=32768) == 0      # 56 MiB, few rows selected
    assert short(units=8, rows=32768, sketch=None) == short(units=16, rows=16384) == 1
    assert short(hd=256, group=4) == 1 and short(hd=256, group=5) == 0 and short(group=8) == 1 and short(group=9) == 0
    assert short(order=hip.ORDER_BEST) == short(order=hip.ORDER_INDEX) == short(budget=0) == short(scores=0x1000) == 0
    assert short(kv_row_stride=1 << 20) == 0                                        # rows beyond 4 GiB of the unit's first


def test_the_valu_attention_is_kept_where_it_is_asked_for():
    """DIFFCACHE_ATTN_VALU=1 (read once per process): groups up to 8 leave this chain, whose attention is the matrix cores'."""
    code = """
import ctypes
import os
import subprocess
import sys
from diffcache_amd import _hip as hip
a = hip.LayerArgs()
a.n_b, a.n_h, a.hd, a.budget, a.n_sink, a.recent_lo, a.order, a.kv_row_stride, a.sketch_codes = 1, 8, 64, 512, 4, 4032, 0, 64, 0x1000
a.one_kernel = hip.ONE_KERNEL_NEVER
for g in (1, 8, 9, 16):
    a.group = g
    print(hip.lib.dc_decode_layer_is_short(ctypes.byref(a)), end=" ")
"""
    for value, want in (("1", "0 0 1 1"), ("0", "1 1 1 1")):
        res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env={**os.environ, "DIFFCACHE_ATTN_VALU": value},
                             cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
        assert res.stdout.split() == want.split(), (value, res.stdout, res.stderr[-300:])


@pytest.mark.gpu
def test_which_calls_run_as_one_kernel():
    from diffcache_amd import _hip as hip

    def route(units, rows, hd=128, group=4, sketch=0x1000, policy=hip.ONE_KERNEL_AUTO, region_hi_dev=None):
        a = hip.LayerArgs()
        a.n_b, a.n_h, a.group, a.hd, a.budget, a.n_sink = 1, units, group, hd, 512, 4
        a.recent_lo, a.n_recent, a.kv_row_stride, a.sketch_codes, a.one_kernel = 4 + rows, 64, hd, sketch, policy
        a.region_hi_dev = region_hi_dev
        return hip.lib.dc_decode_layer_route(ctypes.byref(a))
    one, chain, stream = hip.ROUTE_ONE_KERNEL, hip.ROUTE_SKETCH, hip.ROUTE_STREAM
    assert [route(8, n) for n in (4028, 16384, 32768, 40960)] == [chain] * 4
    assert [route(2, n) for n in (4028, 16384, 16385, 40960, 40961)] == [chain, chain, one, one, chain]
    assert [route(8, n, sketch=None) for n in (4028, 12288, 12289, 32768, 40960)] == [one, one, stream, stream, stream]
    assert [route(2, n, sketch=None) for n in (4028, 40960)] == [one, one]
    assert [route(8, n, policy=hip.ONE_KERNEL_EXCLUSIVE) for n in (4028, 32768)] == [one, one]
    assert route(8, 4028, policy=hip.ONE_KERNEL_NEVER) == chain and route(8, 4028, region_hi_dev=0x1000) == chain
    assert [route(8, n, hd=256, group=6) for n in (4028, 8192, 8193)] == [one, one, chain]


@pytest.mark.gpu
def test_small_groups_and_large_selections_run_as_one_kernel():
    """Both sides of the lines at which the one kernel takes less time than the chains."""
    from diffcache_amd import _hip as hip

    def one(units, rows, hd, group, budget, sketch=0x1000):
        a = hip.LayerArgs()
        a.n_b, a.n_h, a.group, a.hd, a.budget, a.n_sink = 1, units, group, hd, budget, 4
        a.recent_lo, a.n_recent, a.kv_row_stride, a.sketch_codes = 4 + rows, 64, hd, sketch
        return hip.lib.dc_decode_layer_route(ctypes.byref(a)) == hip.ROUTE_ONE_KERNEL
    for sketch in (0x1000, None):       # three kernels: many ids of narrow heads, a few units of wide ones
        rows = 12289                    # (without a sketch: beyond what stays with the one kernel anyway)
        assert one(12, rows, 64, 1, 4096, sketch) and not one(12, rows, 64, 1, 4095, sketch)
        assert one(16, rows, 64, 2, 4096, sketch) and not one(16, rows, 64, 2, 4095, sketch)
        assert one(24, rows, 64, 4, 4096, sketch) and not one(24, rows, 64, 4, 4095, sketch) and not one(24, rows, 64, 8, 4096, sketch)
        assert one(5, 13107, 256, 1, 1024, sketch) and not one(5, 13108, 256, 1, 1024, sketch)
        assert one(4, rows, 256, 2, 1024, sketch) and not one(3, rows, 256, 2, 1024, sketch) and not one(4, rows, 256, 4, 1024, sketch)
        assert one(4, rows, 256, 1, 3072, sketch) and not one(4, rows, 256, 1, 3073, sketch)
    assert one(24, 8124, 128, 1, 4096) and not one(24, 8124, 128, 1, 4095) and not one(24, 8124, 128, 2, 4096)
    assert one(3, 5120, 256, 1, 1024) and not one(3, 5119, 256, 1, 1024)
    # the sketch chain
    assert one(48, 13000, 64, 1, 1300) and not one(48, 13001, 64, 1, 1300) and one(32, 14000, 128, 1, 2000) and not one(32, 14001, 128, 1, 2000)
    assert one(16, 28000, 256, 1, 2000) and not one(16, 28001, 256, 1, 2000) and one(16, 14000, 256, 2, 2000) and not one(16, 14001, 256, 2, 2000)
    assert one(64, 8192, 256, 4, 4096) and not one(64, 8193, 256, 8, 4096)
    # the bf16 chain
    assert one(12, 49151, 128, 1, 512, None) and not one(12, 49152, 128, 1, 512, None) and not one(3, 49151, 128, 1, 512, None)
    assert one(12, 32767, 128, 2, 512, None) and not one(12, 32768, 128, 2, 512, None)
    assert one(12, 24000, 256, 4, 4000, None) and not one(12, 24001, 256, 4, 4000, None) and not one(12, 24000, 128, 4, 4000, None)


@pytest.mark.gpu
@pytest.mark.parametrize("policy", [-2, 2, 7])
def test_a_policy_that_does_not_exist_is_refused(policy):
    """Wherever the one kernel could run, whichever route is the faster one; before anything is launched."""
    from diffcache_amd import _hip as hip
    b, hkv, group, hd, budget = 1, 2, 4, 64, 64
    for rows, order in ((500, hip.ORDER_ANY), (9000, hip.ORDER_ANY)):
        k = torch.zeros((b, hkv, rows, hd), device=DEV, dtype=torch.bfloat16)
        q = torch.zeros((b, hkv * group, hd), device=DEV, dtype=torch.bfloat16)
        ws = hip.alloc_workspace(hip.layer_workspace_bytes(b * hkv, rows, budget, group, hd, budget), DEV)
        idx, out = torch.full((b * hkv, budget), -7, device=DEV, dtype=torch.int32), torch.full_like(q, 3.0)
        for sk in (None, hip.Sketch(k).build(k, 0, rows)):
            for ready in (False, True):
                with pytest.raises(hip.DiffCacheError, match="one_kernel policy"):
                    hip.decode_layer(q, k, k, 0, rows, 0, budget, None, idx, out, ws, order=order, sketch=sk, one_kernel=policy,
                                     select_state_ready=ready)
        torch.cuda.synchronize()
        assert bool((idx == -7).all()) and bool((out == 3.0).all())
