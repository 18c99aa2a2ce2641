"""When DiffCache tells a call that the workspace's select state is ready: only when the last call on the
workspace was of the same kind over the same region (dc_layer_args.select_state_ready).  The native calls are
replaced by recorders, so the rule runs without a GPU; the GPU tests below compare results.  Snapshots loaded
into such a cache are covered on the way."""
import pytest
import torch

LAYERS, WINDOW = 2, 16


class Layer:
    """Stands in for the data layer, which needs a GPU."""

    def __init__(self, **kw):
        self.ctx_len = 0

    def load(self, path, ctx_len):
        pass

    def update_r_sq(self, r_sq):
        pass


@pytest.fixture
def recorded(monkeypatch):
    """(make, calls, capture): a cache on the CPU; what its calls were told; a switch for "under capture"."""
    from diffcache_amd.kvcache import diffcache as mod
    calls, capture = [], []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capture))
    monkeypatch.setattr(mod, "DiffCacheHIP", Layer)
    for name in ("prefill_layer", "append_kv", "step_state_advance", "step_state_rollover", "group_mean"):
        monkeypatch.setattr(mod.hip, name, lambda *a, **k: None)
    monkeypatch.setattr(mod.hip.Sketch, "build", lambda self, *a, **k: self)
    monkeypatch.setattr(mod.hip, "decode_layer", lambda *a, **k: calls.append(k["select_state_ready"]))
    monkeypatch.setattr(mod.hip, "score_select_sketch", lambda *a, **k: calls.append(k["state_ready"]))
    monkeypatch.setattr(mod.hip, "score_select", lambda *a, **k: None)

    def make(r_sq=[[4.0, 4.0]] * LAYERS, **kw):
        return mod.DiffCache(num_layers=LAYERS, batch_size=1, max_length=4000, num_kv_heads=2, num_q_heads=4, head_dim=64,
                             retrieval_budget=64, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                             kvbuf_suffix_maxlen=WINDOW, attn_mass_threshold=0.9, k_check_seq=[100],
                             r_sq=r_sq, device="cpu", **kw)
    return make, calls, capture


def prefill(cache, n):
    k = torch.zeros((1, n, 2, 64), dtype=torch.bfloat16)
    for l in range(LAYERS):
        cache.prefill_update_kv_cache(k, k, l)


def step(cache, **kw):
    q, k = torch.zeros((1, 4, 64), dtype=torch.bfloat16), torch.zeros((1, 1, 2, 64), dtype=torch.bfloat16)
    for l in range(LAYERS):
        cache.decode_attention(l, q, k, k, **kw)


def hook_step(cache):
    for l in range(LAYERS):
        cache.decode_query_kvcache(l)


@pytest.mark.parametrize("one_step", [step, hook_step])
def test_a_prompt_of_another_length_finds_no_state_ready(recorded, one_step):
    make, calls, _ = recorded
    cache = make()
    for n in (3000, 700, 2000, 2000):
        prefill(cache, n)
        one_step(cache)
        one_step(cache)
    first, same = [False, True, True, True], [True] * 4
    assert calls == first + first + first + same


def snapshot(tmp_path):
    import json
    (tmp_path / "metadata.txt").write_text(json.dumps(dict(r_sq=[[1.0, 1.0]] * LAYERS, kvbuf_prefix_len=4,
                                                           kvbuf_suffix_len=8, retrieval_region_len=500)))
    for l in range(LAYERS):
        for kind, rows in (("p", 4), ("s", 8)):
            d = tmp_path / f"{kind}_l_{l:03d}"
            d.mkdir()
            for name in ("k.pt", "v.pt"):
                torch.save(torch.zeros((1, 2, rows, 64), dtype=torch.bfloat16), d / name)


def test_a_loaded_snapshot_of_another_length_finds_no_state_ready(recorded, tmp_path):
    make, calls, _ = recorded
    cache = make(key_sketch=False)
    prefill(cache, 3000)
    step(cache)
    snapshot(tmp_path)
    cache.load_prefill_cache(torch.zeros((1, 512)), str(tmp_path))
    step(cache)
    assert calls == [False, True, False, True]


def test_a_cache_that_is_only_loaded_needs_no_r_sq(recorded, tmp_path):
    make, _, _ = recorded
    cache = make(r_sq=None)
    assert cache.r_sq is None
    snapshot(tmp_path)
    cache.load_prefill_cache(torch.zeros((1, 512)), str(tmp_path))
    assert cache.r_sq == [[1.0, 1.0]] * LAYERS


def test_routes_and_orders_and_rollovers_do_not_share_a_state(recorded):
    from diffcache_amd import _hip as hip
    make, calls, _ = recorded
    cache = make()
    prefill(cache, 1000)
    step(cache)
    hook_step(cache)
    step(cache)
    step(cache, order=hip.ORDER_BEST)
    assert calls == [False, True] * 4
    del calls[:]
    while not cache.window_full():
        step(cache, order=hip.ORDER_BEST)
    assert all(calls)
    del calls[:]
    step(cache, order=hip.ORDER_BEST)       # rolls the window over first: the region grew
    assert cache.generation == 1 and calls == [False, True]


def test_a_call_that_raised_leaves_no_state_ready(recorded, monkeypatch):
    make, calls, _ = recorded
    from diffcache_amd import _hip as hip
    cache = make()
    prefill(cache, 1000)
    step(cache)
    good = hip.decode_layer

    def bad(*a, **k):
        raise hip.DiffCacheError("refused")
    monkeypatch.setattr(hip, "decode_layer", bad)
    with pytest.raises(hip.DiffCacheError):
        step(cache)
    monkeypatch.setattr(hip, "decode_layer", good)
    step(cache)
    assert calls == [False, True, False, True]


@pytest.mark.parametrize("one_step,kw", [
    (step, dict(key_sketch=True)),                       # the region's end on the device
    (step, dict(use_k_check=True)), (hook_step, {}),     # and where it is a launch parameter
])
def test_a_captured_step_and_eager_ones_do_not_share_a_state(recorded, monkeypatch, one_step, kw):
    from diffcache_amd import _hip as hip
    for name in ("score_gathered", "kcheck", "gather_attn"):
        monkeypatch.setattr(hip, name, lambda *a, **k: None)
    make, calls, capture = recorded
    cache = make(**kw)
    prefill(cache, 1000)
    for _ in range(2):              # before any eager call, and behind one
        for _ in range(2):          # captured again: the first capture has not run either
            del calls[:]
            capture.append(1)
            one_step(cache)
            capture.clear()
            assert calls == [False, True]   # a replay sets up what it finds, whatever ran before it
        del calls[:]
        one_step(cache)                     # nothing of the capture has run yet
        assert calls == [False, True]
    del calls[:]
    one_step(cache)
    assert calls == [True, True]
    cache.kvbuf_suffix_len = 8
    cache.advance_host_step(1)              # a replay in between, laid out its own way
    one_step(cache)
    cache.advance_host_step(-1)             # a token taken back: nothing ran
    one_step(cache)
    assert calls == [True, True, False, True, True, True]


def test_a_captured_search_does_not_ready_the_workspace_of_an_eager_one(monkeypatch):
    from diffcache_amd import pq
    calls, capture = [], [1]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capture))
    monkeypatch.setattr(pq.hip, "pq_build_lut", lambda *a: None)
    monkeypatch.setattr(pq.hip, "pq_search", lambda *a, **k: calls.append(k["state_ready"]))
    index = pq.PQIndex(torch.zeros((1, 1, 100, 64), dtype=torch.bfloat16), torch.zeros((1, 16, 256, 4)),
                       torch.zeros((1, 100, 16), dtype=torch.uint8))
    index.search(None)
    index.search(None)
    capture.clear()
    for _ in range(3):
        index.search(None)
    assert calls == [False, False, False, True, True]


@pytest.mark.gpu
@pytest.mark.parametrize("route", ["one_kernel", "sketch", "stream"])
def test_prompts_of_other_lengths_on_one_cache_equal_a_fresh_cache(route):
    from diffcache_amd import DiffCache, _hip as hip
    g = torch.Generator(device="cuda").manual_seed(17)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)

    def make():
        c = DiffCache(num_layers=LAYERS, batch_size=2, max_length=9000, num_kv_heads=4, num_q_heads=16, head_dim=128,
                      retrieval_budget=256, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                      kvbuf_suffix_maxlen=WINDOW, attn_mass_threshold=0.9, k_check_seq=[100],
                      r_sq=[[4.0] * 4] * LAYERS, key_sketch=route == "sketch")
        c.one_kernel = hip.ONE_KERNEL_EXCLUSIVE if route == "one_kernel" else hip.ONE_KERNEL_NEVER
        return c
    used = make()
    # the used cache's slots begin elsewhere for every one of these regions
    for n in (8500, 1501, 4003, 8999 - WINDOW, 700):
        fresh = make()
        kv = [(rnd(2, n, 4, 128), rnd(2, n, 4, 128)) for _ in range(LAYERS)]
        for cache in (used, fresh):
            for l, (k, v) in enumerate(kv):
                cache.prefill_update_kv_cache(k, v, l)
        for _ in range(2):
            for l in range(LAYERS):
                q, nk, nv = rnd(2, 16, 128), rnd(2, 1, 4, 128), rnd(2, 1, 4, 128)
                x, y = (c.decode_attention(l, q, nk, nv).float() for c in (used, fresh))
                if route == "one_kernel":
                    assert hip.last_route() == hip.ROUTE_ONE_KERNEL
                assert torch.equal(used.idx[l].sort(dim=1).values, fresh.idx[l].sort(dim=1).values), (n, l)
                # rows are added in the order they were found: at most 281 terms of weight <= 1 in fp32
                # (281 * 2^-24 * |v| < 1e-4), then one bf16 rounding (2^-8)
                assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-4).all()), (n, l)


@pytest.mark.gpu
@pytest.mark.parametrize("length", [6000, 100])     # with the region's end on the device, and as a launch parameter
def test_eager_steps_between_replays_and_tokens_taken_back(length):
    """One cache alternates eager steps, hook calls, replays of a captured step and tokens taken back; every step's
    ids, output and appended rows equal those of a cache that only steps eagerly."""
    from diffcache_amd import DiffCache, _hip as hip
    g = torch.Generator(device="cuda").manual_seed(23)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)
    used, plain = (DiffCache(num_layers=LAYERS, batch_size=2, max_length=9000, num_kv_heads=4, num_q_heads=16, head_dim=128,
                             retrieval_budget=256, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                             kvbuf_suffix_maxlen=40, attn_mass_threshold=0.9, k_check_seq=[100],
                             r_sq=[[4.0] * 4] * LAYERS) for _ in range(2))
    for l in range(LAYERS):
        k, v = rnd(2, length, 4, 128), rnd(2, length, 4, 128)
        for cache in (used, plain):
            cache.prefill_update_kv_cache(k, v, l)
    q, nk, nv, out = ([torch.zeros(s, device="cuda", dtype=torch.bfloat16) for _ in range(LAYERS)]
                      for s in ((2, 16, 128), (2, 1, 4, 128), (2, 1, 4, 128), (2, 16, 128)))
    for t in (*q, *nk, *nv):
        t.normal_(generator=g)

    def step(cache):
        for l in range(LAYERS):
            cache.decode_attention(l, q[l], nk[l], nv[l], out=out[l])

    def replay(cache):
        graph.replay()
        cache.advance_host_step()

    def take_back(cache):
        cache.advance_host_step(-1)
        hip.step_state_advance(cache._state, -1, cache.kvbuf_suffix_maxlen)

    used._ensure_workspace()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step(used)
    lo, hi = used._region()
    # the first eager step comes behind a capture that has not run
    for i, how in enumerate((step, replay, step, step, replay, "hooks", replay, step, "back", replay, "back", step, replay)):
        if how == "hooks":      # (only their use of the workspace matters here: the step they count is taken back)
            for l in range(LAYERS):
                used.decode_pre_query_operation(q[l])
                used.decode_query_kvcache(l)
            used.kvbuf_suffix_len -= 1
            hip.step_state_advance(used._state, -1, used.kvbuf_suffix_maxlen)
            continue
        if how == "back":
            for cache in (used, plain):
                take_back(cache)
                for store in (*cache.kstore, *cache.vstore):
                    store[:, :, hi + cache.kvbuf_suffix_len].fill_(7.0)     # a row that is not written again would show
            continue
        for t in (*q, *nk, *nv):
            t.normal_(generator=g)
        how(used)
        got, ids = [t.clone() for t in out], [t.clone() for t in used.idx]
        step(plain)
        n = hi + used.kvbuf_suffix_len
        assert used._state.tolist() == plain._state.tolist() == [n - hi, hi, n, 0], (i, how)
        for l in range(LAYERS):
            assert torch.equal(ids[l].sort(dim=1).values, plain.idx[l].sort(dim=1).values), (i, l)
            x, y = got[l].float(), out[l].float()
            # rows are added in another order on another route: at most 301 terms of weight <= 1 in fp32
            # (301 * 2^-24 * |v| < 1e-4), then one bf16 rounding (2^-8) on either side
            assert bool(((x - y).abs() <= 2.0 ** -7 * x.abs() + 1e-4).all()), (i, l)
            assert torch.equal(used.kstore[l][:, :, :n], plain.kstore[l][:, :, :n]), (i, l)
            assert torch.equal(used.vstore[l][:, :, :n], plain.vstore[l][:, :, :n]), (i, l)
