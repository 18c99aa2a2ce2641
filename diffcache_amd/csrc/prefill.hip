// A prompt's keys and values into one layer of the cache, with everything the cache derives from
// them.  Replaces the permute + host copies of src/diffcache/kvcache/diffcache.py:142-147 with the
// memcpy of Index::prefill (diffcache_cpu/src/nsw.rs:503-508), the r_sq reduction
// (diffcache.py:151-156) and the prefix and suffix copies of diffcache.py:163-171.
//
// Two passes over the keys are the least there can be: the scales of the 8-bit sketch are known
// only when every key has been seen.  The first (prefill_copy_kernel) moves K and V from the
// model's layout into the store and, while the 16 bytes are in registers, takes the per-channel
// maxima for the scales, the largest |k|^2 of a head, and copies the rows that also belong to the
// assembled buffer; the second (sketch_quantise_kernel) reads K back.  Both are bound by HBM:
// 11 bytes per key element, 9 of which no implementation can do without.  At 16 units x 40003 rows
// of 128 channels a layer takes 152 us (902 MB moved: 5.9 TB/s, where a plain copy of 2 GiB reaches 5.0); with blocks that start one after
// the other and 17 instructions an element in the second pass 181, and the torch reduction for r_sq, the two ingest calls, the
// three-pass sketch build and the buffer copies they replace 7.8 ms, nearly all of it the reduction (one
// batched product per token and head) and the wait for its result.  (V stored past the caches and K through them, so that the
// second pass finds a part of it: both past them 30 us more, both through them 16.  V first and K second in every block: no gain.)
#include "dc_common.h"

namespace {

constexpr int kThreads = 256;
constexpr uint32_t kMaxFiniteMag = 0x7f7fu;  // largest finite bf16 magnitude, as in sketch.hip

struct PrefillCopy {
    const uint16_t *ks, *vs;  // (n_b, seq, n_h, hd)
    uint16_t *kd, *vd;        // the stores
    int64_t sb, sh, sr;
    uint16_t *kb, *vb;        // the assembled buffer at the row of its first prefix row, or null
    int64_t bb, bh, br;
    uint32_t *amax;           // (n_units, hd) float bits, or null
    uint32_t *r_sq;           // (n_h) float bits, or null
    int32_t *state;           // dc_step_state or null
    int n_units, n_h, seq, n_prefix, n_suffix, rows_per_block, k_blocks;
};

__global__ void prefill_zero_kernel(uint32_t *amax, uint32_t *resid, int64_t n, uint32_t *r_sq, int n_h) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        if (amax) amax[i] = 0u;
        if (resid) resid[i] = 0u;
    }
    if (r_sq && i < n_h) r_sq[i] = 0u;
}

// Blocks of K and V together: they all run at once (a CU holds eight) and end at about the same time.  Per layer, us, with 8192 blocks
// (fewer for short prompts), which start one after the other in the place of those that end / with 1280: 16 units x 40003 rows of
// 128 columns 183 / 159, 8 x 32768 108 / 76, 4 x 127284 184 / 133, 64 x 10000 188 / 162, 160 x 2048 123 / 88, 16 x 40003 of 64 123 /
// 94, 8 x 40003 of 256 179 / 159 (1024 blocks: as much, 2048: 2 to 4 more, 2560: 10 more, 512: 25 more).
constexpr int64_t kCopyBlocks = 1280;
// Beyond 64 units and 80 Mi key elements more and shorter blocks, which start one after the other: there a block of 1280 is a whole prompt of
// its unit or a large part of it.  Per layer, us, 8192 / 1280 / these: 256 units x 4000 rows of 128 columns 297 / 329 / 293, 160 x 8000 372 /
// 404 / 354, 320 x 4000 386 / 423 / 369, 400 x 4096 433 / 459 / 428, 400 x 4000 of 64 233 / 256 / 227, 328 x 2048 196 / 183 / 172; 320 x 4000
// of 64, just below, 205 / 185 / 193.  (Pieces of 64 rows: 200 x 4000 215 -> 209, 256 x 2000 of 256 columns 250 -> 242; 16 x 40003, below, 154 -> 157.)
constexpr int64_t kCopyBlocksMany = 6144, kManyUnits = 64, kManyElements = 80ll << 20;
// Without a sketch, whose pass over the keys is the other half of the time, and beyond 96 Mi key elements of any number of units, more and
// shorter ones still.  Per layer, us, 8192 / 1280 / 6144 / these: 32 units x 32000 rows of 128 columns 214 / 230 / 221 / 214, 1 x 2000000
// 402 / 422 / 412 / 395, 8 x 131072 223 / 225 / 223 / 212, 128 x 8000 216 / 229 / 223 / 216, 400 x 2000 of 256 315 / 347 / 322 / 316, 64 x
// 40000 of 64 281 / 289 / 283 / 280; below the line 64 x 10000 144 / 139 / 135 / 144, 16 x 40003 142 / 135 / 135 / 141.
constexpr int64_t kCopyBlocksLong = 12288, kLongElements = 96ll << 20;

// One block copies rows_per_block rows of one unit, of V (the first half of the grid) or of K.  A group of HD/8 lanes owns a row, 16 bytes per lane; a lane keeps its eight columns
// for the whole block, so the column maxima stay in registers.
template <int HD>
__global__ __launch_bounds__(kThreads) void prefill_copy_kernel(PrefillCopy a) {
    constexpr int LPR = HD / 8;
    constexpr int GROUPS = kThreads / LPR;
    constexpr int kInFlight = 4;
    __shared__ uint32_t smax[GROUPS][HD];
    __shared__ uint32_t s_sq[GROUPS];
    const bool is_k = (int)blockIdx.x >= a.k_blocks;
    const int id = (int)blockIdx.x - (is_k ? a.k_blocks : 0);
    const int unit = id % a.n_units, chunk = id / a.n_units;
    const int b = unit / a.n_h, h = unit % a.n_h;
    const int tid = threadIdx.x, grp = tid / LPR, col = tid % LPR;
    if (blockIdx.x == 0 && tid == 0 && a.state) {
        a.state[0] = a.n_suffix;
        a.state[1] = a.seq - a.n_suffix;
        a.state[2] = a.seq;
    }
    const int r0 = chunk * a.rows_per_block;
    const int r1 = r0 + a.rows_per_block < a.seq ? r0 + a.rows_per_block : a.seq;
    const int64_t tok = (int64_t)a.n_h * HD;
    const uint16_t *src = (is_k ? a.ks : a.vs) + (int64_t)b * a.seq * tok + (int64_t)h * HD + col * 8;
    uint16_t *dst = (is_k ? a.kd : a.vd) + b * a.sb + h * a.sh + col * 8;
    uint16_t *buf = is_k ? a.kb : a.vb;
    if (buf) buf += b * a.bb + h * a.bh + col * 8;
    const int s0 = a.seq - a.n_suffix;
    const bool stats = is_k && (a.amax || a.r_sq);
    uint32_t m[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) m[i] = 0u;
    uint32_t sq_max = 0u;
    for (int rb = r0 + grp; rb < r1; rb += GROUPS * kInFlight) {
        uint4 w[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            int r = rb + u * GROUPS;
            r = r < r1 ? r : r1 - 1;
            w[u] = dc_load_stream16(src + (int64_t)r * tok);
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const int r = rb + u * GROUPS;
            if (r >= r1) break;
            if (is_k) *reinterpret_cast<uint4 *>(dst + (int64_t)r * a.sr) = w[u];
            else dc_store_stream16(dst + (int64_t)r * a.sr, w[u]);
            const bool pre = r < a.n_prefix, suf = r >= s0;
            if (buf && (pre || suf))
                *reinterpret_cast<uint4 *>(buf + (int64_t)(pre ? r : a.n_prefix + (r - s0)) * a.br) = w[u];
            if (stats) {
                const uint32_t x[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
                if (!pre && !suf) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t lo = x[i] & 0x7fffu, hi = (x[i] >> 16) & 0x7fffu;
                        m[2 * i] = lo > m[2 * i] ? lo : m[2 * i];
                        m[2 * i + 1] = hi > m[2 * i + 1] ? hi : m[2 * i + 1];
                    }
                }
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    s = fmaf(dc_bf16_lo(x[i]), dc_bf16_lo(x[i]), s);
                    s = fmaf(dc_bf16_hi(x[i]), dc_bf16_hi(x[i]), s);
                }
                s = dc_group_sum<LPR>(s);
                // non-negative floats order like unsigned integers; a NaN is made the largest
                const uint32_t sb = (s == s) ? __float_as_uint(s) : 0x7fc00000u;
                sq_max = sb > sq_max ? sb : sq_max;
            }
        }
    }
    if (!stats) return;
#pragma unroll
    for (int i = 0; i < 8; ++i) smax[grp][col * 8 + i] = m[i];
    if (col == 0) s_sq[grp] = sq_max;
    __syncthreads();
    if (a.amax && tid < HD) {
        uint32_t v = 0;
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) v = smax[g][tid] > v ? smax[g][tid] : v;
        v = v > kMaxFiniteMag ? kMaxFiniteMag : v;
        if (v) atomicMax(&a.amax[(int64_t)unit * HD + tid], v << 16);
    }
    if (a.r_sq && tid == 0) {
        uint32_t v = 0;
        for (int g = 0; g < GROUPS; ++g) v = s_sq[g] > v ? s_sq[g] : v;
        if (v) atomicMax(&a.r_sq[h], v);
    }
}

}  // namespace

extern "C" size_t dc_prefill_workspace_bytes(int n_units, int hd) {
    return n_units > 0 && hd > 0 ? dc_align_up((size_t)n_units * (size_t)hd * 4, 256) : 256;
}

extern "C" int dc_prefill_layer_bf16(const dc_prefill_args *a, void *stream) {
    const char *who = "dc_prefill_layer_bf16";
    DC_REQUIRE(a, "%s: null args", who);
    DC_REQUIRE(a->k_src && a->v_src && a->k_store && a->v_store, "%s: null pointer", who);
    DC_REQUIRE(a->n_b >= 0 && a->n_h >= 1 && a->seq >= 0 && a->n_prefix >= 0 && a->n_suffix >= 0 &&
                   (int64_t)a->n_prefix + a->n_suffix <= a->seq,
               "%s: bad sizes", who);
    DC_REQUIRE(a->hd == 64 || a->hd == 128 || a->hd == 256, "%s: head_dim %d not in {64,128,256}", who, a->hd);
    DC_REQUIRE((a->k_buf == nullptr) == (a->v_buf == nullptr), "%s: k_buf and v_buf must both be set or both be null", who);
    DC_REQUIRE(dc_aligned16(a->k_src) && dc_aligned16(a->v_src) && dc_aligned16(a->k_store) && dc_aligned16(a->v_store) &&
                   dc_aligned16(a->k_buf) && dc_aligned16(a->v_buf),
               "%s: pointers must be 16-byte aligned", who);
    DC_REQUIRE(a->batch_stride % 8 == 0 && a->head_stride % 8 == 0 && a->row_stride % 8 == 0 && a->row_stride >= a->hd &&
                   a->buf_batch_stride % 8 == 0 && a->buf_head_stride % 8 == 0 && a->buf_row_stride % 8 == 0,
               "%s: strides must be multiples of 8 elements and row_stride >= hd", who);
    const int64_t n_units64 = (int64_t)a->n_b * a->n_h;
    DC_REQUIRE(n_units64 < (1 << 20), "%s: too many units", who);
    const int n_units = (int)n_units64;
    if (n_units == 0 || a->seq == 0) return DC_OK;
    const int region = a->seq - a->n_prefix - a->n_suffix;
    const bool sketch = a->codes && region > 0;
    if (sketch) {
        DC_REQUIRE(a->scale && a->resid && a->workspace, "%s: the sketch needs scale, resid and a workspace", who);
        DC_REQUIRE(dc_aligned16(a->codes) && dc_aligned16(a->workspace), "%s: codes and workspace must be 16-byte aligned", who);
        DC_REQUIRE(a->code_batch_stride % 16 == 0 && a->code_head_stride % 16 == 0 && a->code_row_stride % 16 == 0 &&
                       a->code_row_stride >= a->hd,
                   "%s: code strides must be multiples of 16 bytes and row_stride >= hd", who);
        if (a->workspace_bytes < dc_prefill_workspace_bytes(n_units, a->hd)) {
            dc_set_error("%s: workspace %zu bytes < %zu needed", who, a->workspace_bytes,
                         dc_prefill_workspace_bytes(n_units, a->hd));
            return DC_ENOMEM;
        }
    }
    hipStream_t st = (hipStream_t)stream;
    PrefillCopy p;
    p.ks = (const uint16_t *)a->k_src, p.vs = (const uint16_t *)a->v_src;
    p.kd = (uint16_t *)a->k_store, p.vd = (uint16_t *)a->v_store;
    p.sb = a->batch_stride, p.sh = a->head_stride, p.sr = a->row_stride;
    p.kb = (uint16_t *)a->k_buf, p.vb = (uint16_t *)a->v_buf;
    p.bb = a->buf_batch_stride, p.bh = a->buf_head_stride, p.br = a->buf_row_stride;
    p.amax = sketch ? (uint32_t *)a->workspace : nullptr;
    p.r_sq = (uint32_t *)a->r_sq;
    p.state = a->step_state;
    p.n_units = n_units, p.n_h = a->n_h, p.seq = a->seq, p.n_prefix = a->n_prefix, p.n_suffix = a->n_suffix;
    if (sketch || a->r_sq) {
        const int64_t n_sc = sketch ? n_units64 * a->hd : 0, n = n_sc > a->n_h ? n_sc : a->n_h;
        hipLaunchKernelGGL(prefill_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p.amax,
                           sketch ? (uint32_t *)a->resid : nullptr, n_sc, p.r_sq, a->n_h);
        DC_CHECK_LAUNCH(who);
    }
    // Equal shares for kCopyBlocks blocks, 64 rows at least; in long copies for more of them, whole pieces of 64 rows.
    const int64_t elements = n_units64 * a->seq * a->hd;
    int64_t most = kCopyBlocks;
    if (!sketch && elements > kLongElements) most = kCopyBlocksLong;
    else if (n_units64 > kManyUnits && elements > kManyElements) most = kCopyBlocksMany;
    int64_t chunks = most / (2 * n_units64);
    chunks = chunks < 1 ? 1 : chunks;
    int64_t rpb = ((int64_t)a->seq + chunks - 1) / chunks;
    if (most != kCopyBlocks) rpb = (rpb + 63) / 64 * 64;
    rpb = rpb < 64 ? 64 : rpb;
    const int64_t blocks = ((int64_t)a->seq + rpb - 1) / rpb * n_units64;
    DC_REQUIRE(2 * blocks < (1ll << 31), "%s: grid too large", who);
    p.rows_per_block = (int)rpb;
    p.k_blocks = (int)blocks;
    const dim3 grid((unsigned)(2 * blocks));
    if (a->hd == 64) hipLaunchKernelGGL(prefill_copy_kernel<64>, grid, dim3(kThreads), 0, st, p);
    else if (a->hd == 128) hipLaunchKernelGGL(prefill_copy_kernel<128>, grid, dim3(kThreads), 0, st, p);
    else hipLaunchKernelGGL(prefill_copy_kernel<256>, grid, dim3(kThreads), 0, st, p);
    DC_CHECK_LAUNCH(who);
    if (!sketch) return DC_OK;
    return dc_sketch_quantise_launch(who, (const uint16_t *)a->k_store + (int64_t)a->n_prefix * a->row_stride,
                                     a->codes + (int64_t)a->n_prefix * a->code_row_stride, (const float *)a->workspace,
                                     a->resid, n_units, a->n_h, region, a->hd, a->batch_stride, a->head_stride,
                                     a->row_stride, a->code_batch_stride, a->code_head_stride, a->code_row_stride, 1,
                                     a->scale, stream);
}
