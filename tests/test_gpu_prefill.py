"""dc_prefill_layer_bf16: a prompt into one layer of a cache in one call, against torch's permutes and copies,
dc_sketch_build_bf16 of the same region, and a float64 reduction for the key norms."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("hd,b,h,seq,prefix,suffix", [
    (128, 1, 8, 1, 1, 0),            # one row, all of it prefix: no region, no sketch
    (128, 2, 3, 63, 4, 16),          # below one block, an odd number of heads
    (64, 1, 5, 64, 0, 0),            # exactly one block, no fixed rows
    (256, 2, 1, 65, 64, 1),          # one row past a block; the region is empty
    (128, 1, 8, 4133, 4, 64),        # ragged, several blocks per unit
    (64, 3, 4, 20011, 128, 128),     # blocks of more than 64 rows
    (256, 1, 2, 9001, 4, 64),
])
def test_prefill_layer_matches_copies_and_sketch_build(hd, b, h, seq, prefix, suffix):
    from diffcache_amd import _hip as hip
    g = torch.Generator(device=DEV).manual_seed(seq * hd)
    k = torch.randn((b, seq, h, hd), generator=g, device=DEV).mul_(
        torch.exp(torch.randn((1, 1, h, hd), generator=g, device=DEV))).to(torch.bfloat16)
    v = torch.randn((b, seq, h, hd), generator=g, device=DEV).to(torch.bfloat16)
    n_max, window = seq + 9, suffix + 7
    ks, vs = (torch.full((b, h, n_max, hd), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    kb, vb = (torch.full((b, h, 5 + prefix + window, hd), 9.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    sk, ref = hip.Sketch(ks), hip.Sketch(ks)
    for t in (sk.codes, ref.codes, sk.scale, sk.resid, ref.scale, ref.resid):
        t.fill_(3)                  # stale contents of an earlier prompt
    r_sq = torch.full((h,), 1e30, device=DEV)
    state = torch.tensor([5, 6, 7, 0], device=DEV, dtype=torch.int32)
    region = seq - prefix - suffix
    hip.prefill_layer(ks, vs, k, v, prefix, suffix, kb[:, :, 5:], vb[:, :, 5:], sketch=sk if region > 0 else None,
                      r_sq=r_sq, step_state=state)
    kt, vt = k.permute(0, 2, 1, 3), v.permute(0, 2, 1, 3)
    for store, src, buf in ((ks, kt, kb), (vs, vt, vb)):
        assert torch.equal(store[:, :, :seq], src) and bool((store[:, :, seq:] == 7.0).all())
        assert torch.equal(buf[:, :, 5:5 + prefix], src[:, :, :prefix])
        assert torch.equal(buf[:, :, 5 + prefix:5 + prefix + suffix], src[:, :, seq - suffix:])
        assert bool((buf[:, :, :5] == 9.0).all()) and bool((buf[:, :, 5 + prefix + suffix:] == 9.0).all())
    assert state.tolist() == [suffix, seq - suffix, seq, 0]
    if region > 0:
        ref.build(ks, prefix, region)
    assert torch.equal(sk.codes, ref.codes) and torch.equal(sk.scale, ref.scale) and torch.equal(sk.resid, ref.resid)
    # a sum of hd squares in fp32: relative error below hd * 2^-24
    want = k.double().pow(2).sum(-1).amax(dim=(0, 1))
    assert bool(((r_sq.double() - want).abs() <= hd * 2.0 ** -24 * want).all())


def test_prefill_carries_infinities_and_nans_to_the_norms():
    from diffcache_amd import _hip as hip
    k = torch.ones((1, 300, 3, 128), device=DEV, dtype=torch.bfloat16)
    k[0, 17, 1, 5] = float("inf")
    k[0, 299, 2, 0] = float("nan")
    store = torch.zeros((1, 3, 300, 128), device=DEV, dtype=torch.bfloat16)
    r_sq = torch.zeros((3,), device=DEV)
    hip.prefill_layer(store, torch.zeros_like(store), k, k, 0, 0, r_sq=r_sq)
    got = r_sq.tolist()
    assert got[0] == 128.0 and got[1] == float("inf") and got[2] != got[2]


def test_r_sq_of_a_prefill_reads_as_before():
    """DiffCache.r_sq and its data layers' r_sq: lists of floats, the bf16-rounded largest squared norm."""
    from diffcache_amd import DiffCache
    g = torch.Generator(device=DEV).manual_seed(3)
    mine = [[4.0, 4.0], [4.0, 4.0]]
    cache = DiffCache(num_layers=2, batch_size=2, max_length=700, num_kv_heads=2, num_q_heads=4, head_dim=64,
                      retrieval_budget=64, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                      kvbuf_suffix_maxlen=16, attn_mass_threshold=0.9, k_check_seq=[100], r_sq=mine)
    k = torch.randn((2, 600, 2, 64), generator=g, device=DEV).to(torch.bfloat16)
    cache.prefill_update_kv_cache(k, k, 1)
    want = k.float().pow(2).sum(-1).amax(dim=(0, 1)).to(torch.bfloat16).tolist()
    for got in (cache.data_layers[1].r_sq, cache.r_sq[1]):
        assert isinstance(got, list) and all(isinstance(x, float) for x in got)
        assert all(abs(a - b) <= 2.0 ** -7 * b for a, b in zip(got, want))     # one bf16 ulp
    assert cache.r_sq[0] == [4.0, 4.0] and mine == [[4.0, 4.0], [4.0, 4.0]]


def test_layers_prefilled_on_two_streams_share_nothing_and_r_sq_waits_for_its_own():
    """Layers ingested on different streams at the same time: each sketch is that of its own keys, and r_sq read
    from a third stream is the finished value."""
    from diffcache_amd import DiffCache, _hip as hip
    g = torch.Generator(device=DEV).manual_seed(11)
    cache = DiffCache(num_layers=2, batch_size=2, max_length=20100, num_kv_heads=4, num_q_heads=8, head_dim=128,
                      retrieval_budget=64, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                      kvbuf_suffix_maxlen=16, attn_mass_threshold=0.9, k_check_seq=[100], r_sq=[[4.0] * 4] * 2)
    ks = [torch.randn((2, 20011, 4, 128), generator=g, device=DEV).mul_(10.0 ** l).to(torch.bfloat16) for l in range(2)]
    want = [k.float().pow(2).sum(-1).amax(dim=(0, 1)).to(torch.bfloat16).tolist() for k in ks]
    torch.cuda.synchronize()
    for _ in range(3):
        for l, stream in enumerate((torch.cuda.Stream(), torch.cuda.Stream())):
            with torch.cuda.stream(stream):
                cache.prefill_update_kv_cache(ks[l], ks[l], l)
        for l in range(2):
            assert all(abs(a - b) <= 2.0 ** -7 * b for a, b in zip(cache.data_layers[l].r_sq, want[l]))   # one bf16 ulp
        torch.cuda.synchronize()
        for l in range(2):
            ref = hip.Sketch(cache.kstore[l])
            ref.build(cache.kstore[l], 4, 20011 - 12)
            assert torch.equal(cache.sketch[l].scale, ref.scale) and torch.equal(cache.sketch[l].resid, ref.resid)
            assert torch.equal(cache.sketch[l].codes[:, :, 4:20003], ref.codes[:, :, 4:20003])


def test_a_prefill_under_capture_is_refused():
    from diffcache_amd import DiffCache
    cache = DiffCache(num_layers=1, batch_size=1, max_length=300, num_kv_heads=1, num_q_heads=1, head_dim=64,
                      retrieval_budget=16, nsw_m=16, nsw_ef_cons=200, kvbuf_prefix_len=4, kvbuf_suffix_len=8,
                      kvbuf_suffix_maxlen=16, attn_mass_threshold=0.9, k_check_seq=[100], r_sq=[[4.0]])
    k = torch.ones((1, 200, 1, 64), device=DEV, dtype=torch.bfloat16)
    torch.cuda.synchronize()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        with pytest.raises(Exception, match="captured"):
            cache.prefill_update_kv_cache(k, k, 0)


@pytest.mark.parametrize("hd,b,h,seq,prefix,suffix", [
    (64, 41, 8, 300, 4, 64),         # one block to a unit's whole prompt
    (128, 11, 8, 7450, 4, 64),       # just beyond 80 Mi key elements of 88 units: shorter blocks, in pieces of 64 rows
    (256, 65, 1, 5043, 128, 128),    # the same of 256 columns, one unit beyond the line
])
def test_prefills_of_many_units_match_copies_and_sketch_build(hd, b, h, seq, prefix, suffix):
    test_prefill_layer_matches_copies_and_sketch_build(hd, b, h, seq, prefix, suffix)


@pytest.mark.parametrize("hd,b,h,seq", [(128, 3, 1, 262145), (64, 37, 8, 5333), (256, 2, 3, 65537)])
def test_long_prefills_without_a_sketch_match_copies(hd, b, h, seq):
    """Just beyond 96 Mi key elements: other blocks than with a sketch."""
    from diffcache_amd import _hip as hip
    assert 96 << 20 < b * h * seq * hd < 97 << 20
    g = torch.Generator(device=DEV).manual_seed(seq)
    k, v = (torch.empty((b, seq, h, hd), device=DEV, dtype=torch.bfloat16).normal_(generator=g) for _ in range(2))
    ks, vs = (torch.full((b, h, seq + 3, hd), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    kb, vb = (torch.full((b, h, 20, hd), 9.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
    r_sq = torch.full((h,), 1e30, device=DEV)
    hip.prefill_layer(ks, vs, k, v, 4, 9, kb, vb, r_sq=r_sq)
    for store, src, buf in ((ks, k, kb), (vs, v, vb)):
        src = src.permute(0, 2, 1, 3)
        assert torch.equal(store[:, :, :seq], src) and bool((store[:, :, seq:] == 7.0).all())
        assert torch.equal(buf[:, :, :13], torch.cat([src[:, :, :4], src[:, :, seq - 9:]], dim=2)) and bool((buf[:, :, 13:] == 9.0).all())
    want = k.double().pow(2).sum(-1).amax(dim=(0, 1))
    assert bool(((r_sq.double() - want).abs() <= hd * 2.0 ** -24 * want).all())
