// The 8-bit sketch of the key store that dc_score_select_sketch_bf16 scans.
//
// Per unit and channel d the sketch holds a scale a_d and a residual bound r_d;
// row i is stored as HD bytes u_id = c_id + 128 with c_id in [-127, 127] and
//   k_id = a_d * c_id + e_id,   |e_id| <= r_d   for every sketched row.
// r_d is measured while quantising (not assumed to be a_d / 2), so rows added
// later with values outside the range the scales were fitted to only raise r_d
// and the bound stays true.  No counterpart in the reference: the exact scan of
// diffcache_cpu/src/nsw.rs:592-630 reads every bf16 key; the sketch lets the GPU
// read half as many bytes and still return that scan's result.
#include "dc_common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kRowsPerBlock = 2048;

__global__ void sketch_zero_kernel(uint32_t *a, uint32_t *b, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        if (a) a[i] = 0;
        b[i] = 0;
    }
}

// largest finite bf16 magnitude (inf and NaN are clamped to it; their residual is inf)
constexpr uint32_t kMaxFiniteMag = 0x7f7fu;

// per (unit, channel) maximum |k| over the rows, as float bits (non-negative floats
// order like unsigned integers)
template <int HD>
__global__ __launch_bounds__(kThreads) void sketch_absmax_kernel(
    const uint16_t *__restrict__ K, uint32_t *__restrict__ amax_bits, int n_h, int n_rows, int64_t sb,
    int64_t sh, int64_t sr, int blocks_per_unit) {
    constexpr int LPR = HD / 8;
    constexpr int GROUPS = kThreads / LPR;
    __shared__ uint32_t smax[GROUPS][HD];
    const int unit = blockIdx.x / blocks_per_unit, blk = blockIdx.x % blocks_per_unit;
    const int b = unit / n_h, h = unit % n_h;
    const int grp = threadIdx.x / LPR, col = threadIdx.x % LPR;
    const uint16_t *Ku = K + b * sb + h * sh + col * 8;
    const int64_t r0 = (int64_t)blk * kRowsPerBlock;
    int64_t r1 = r0 + kRowsPerBlock;
    if (r1 > n_rows) r1 = n_rows;
    uint32_t m[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) m[i] = 0;
    for (int64_t r = r0 + grp; r < r1; r += GROUPS) {
        const uint4 w = dc_load_stream16(Ku + r * sr);
        const uint32_t x[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t lo = x[i] & 0x7fffu, hi = (x[i] >> 16) & 0x7fffu;
            m[2 * i] = lo > m[2 * i] ? lo : m[2 * i];
            m[2 * i + 1] = hi > m[2 * i + 1] ? hi : m[2 * i + 1];
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) smax[grp][col * 8 + i] = m[i];
    __syncthreads();
    if (threadIdx.x < HD) {
        uint32_t v = 0;
        for (int g = 0; g < GROUPS; ++g) v = smax[g][threadIdx.x] > v ? smax[g][threadIdx.x] : v;
        v = v > kMaxFiniteMag ? kMaxFiniteMag : v;
        if (v) atomicMax(&amax_bits[(int64_t)unit * HD + threadIdx.x], v << 16);
    }
}

// quantise rows with a_d = amax_d / 127 (scale_is_amax) or a_d = scale_d, write the
// codes, and raise resid_d to the largest |k - a c| seen; scale_out (or null) receives a_d
template <int HD>
__global__ __launch_bounds__(kThreads) void sketch_quantise_kernel(
    const uint16_t *__restrict__ K, uint8_t *__restrict__ C, const float *__restrict__ scale,
    uint32_t *__restrict__ resid_bits, int n_h, int n_rows, int64_t sb, int64_t sh, int64_t sr, int64_t cb,
    int64_t ch, int64_t cr, int n_units, int rows_per_block, int scale_is_amax, float *__restrict__ scale_out) {
    constexpr int LPR = HD / 8;
    constexpr int GROUPS = kThreads / LPR;
    constexpr int kInFlight = 4;  // rows of a lane group requested together
    __shared__ uint32_t smax[GROUPS][HD];
    const int unit = blockIdx.x % n_units, blk = blockIdx.x / n_units;
    const int b = unit / n_h, h = unit % n_h;
    const int grp = threadIdx.x / LPR, col = threadIdx.x % LPR;
    const uint16_t *Ku = K + b * sb + h * sh + col * 8;
    uint8_t *Cu = C + b * cb + h * ch + col * 8;
    float a[8], inv[8], res[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float s = scale[(int64_t)unit * HD + col * 8 + i];
        a[i] = scale_is_amax ? s / 127.0f : s;
        inv[i] = a[i] > 0.f ? 1.0f / a[i] : 0.f;
        res[i] = 0.f;
    }
    if (scale_out && blk == 0 && grp == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) scale_out[(int64_t)unit * HD + col * 8 + i] = a[i];
    }
    const int64_t r0 = (int64_t)blk * rows_per_block;
    int64_t r1 = r0 + rows_per_block;
    if (r1 > n_rows) r1 = n_rows;
    // Codes of numbers are rounded by adding a constant whose unit is one (halves go to the even neighbour there too), which leaves the
    // code in the low byte: 7.4 vector instructions an element instead of 17.  A key that is not finite leaves a residual that is infinite
    // or no number, whose maximum keeps it; the wave then works the batch out again with every comparison, and the rest of its block, as
    // it always does where a channel's scale is so small that a zero times its reciprocal is no number.
    constexpr float kRound = 12582912.0f + 128.0f;
    bool odd_scale = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) odd_scale |= inv[i] == __builtin_inff();
    odd_scale = __ballot(odd_scale) != 0ull;
    for (int64_t rb = r0 + grp; rb < r1; rb += GROUPS * kInFlight) {
        uint4 wv[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            int64_t r = rb + (int64_t)u * GROUPS;
            r = r < r1 ? r : r1 - 1;
            wv[u] = dc_load_stream16(Ku + r * sr);
        }
        uint2 packed[kInFlight];
        bool odd = odd_scale;
        if (!odd) {
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {  // (past the end the last row once more)
                const uint4 w = wv[u];
                const float kv[8] = {dc_bf16_lo(w.x), dc_bf16_hi(w.x), dc_bf16_lo(w.y), dc_bf16_hi(w.y),
                                     dc_bf16_lo(w.z), dc_bf16_hi(w.z), dc_bf16_lo(w.w), dc_bf16_hi(w.w)};
                uint32_t y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float f = __builtin_amdgcn_fmed3f(kv[i] * inv[i], -127.f, 127.f) + kRound;
                    y[i] = __float_as_uint(f);
                    res[i] = __builtin_elementwise_maximum(res[i], fabsf(fmaf(-a[i], f - kRound, kv[i])));
                }
                constexpr uint32_t kTwo = 0x0c0c0400u, kFour = 0x05040100u;  // the low bytes, the low halves of two words
                packed[u].x = __builtin_amdgcn_perm(__builtin_amdgcn_perm(y[3], y[2], kTwo), __builtin_amdgcn_perm(y[1], y[0], kTwo), kFour);
                packed[u].y = __builtin_amdgcn_perm(__builtin_amdgcn_perm(y[7], y[6], kTwo), __builtin_amdgcn_perm(y[5], y[4], kTwo), kFour);
            }
            bool wide = false;
#pragma unroll
            for (int i = 0; i < 8; ++i) wide |= !(res[i] < __builtin_inff());
            odd = __ballot(wide) != 0ull;
        }
        if (odd) {
            // a NaN residual must poison the bound, not vanish in the max
#pragma unroll
            for (int i = 0; i < 8; ++i) res[i] = res[i] == res[i] ? res[i] : __builtin_inff();
#pragma unroll
            for (int u = 0; u < kInFlight; ++u) {
                const uint4 w = wv[u];
                const float kv[8] = {dc_bf16_lo(w.x), dc_bf16_hi(w.x), dc_bf16_lo(w.y), dc_bf16_hi(w.y),
                                     dc_bf16_lo(w.z), dc_bf16_hi(w.z), dc_bf16_lo(w.w), dc_bf16_hi(w.w)};
                uint32_t code[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    float c = rintf(kv[i] * inv[i]);
                    c = c > 127.f ? 127.f : (c < -127.f ? -127.f : c);
                    if (!(c == c)) c = 0.f;  // NaN key or 0 * inf
                    const float e = fabsf(fmaf(-a[i], c, kv[i]));
                    if (!(e <= res[i])) res[i] = (e == e) ? e : __builtin_inff();
                    code[i] = (uint32_t)((int)c + 128);
                }
                packed[u].x = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
                packed[u].y = code[4] | (code[5] << 8) | (code[6] << 16) | (code[7] << 24);
            }
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const int64_t r = rb + (int64_t)u * GROUPS;
            if (r >= r1) break;
            dc_store_stream8(Cu + r * cr, packed[u]);
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) smax[grp][col * 8 + i] = __float_as_uint(res[i]);
    __syncthreads();
    if (threadIdx.x < HD) {
        uint32_t v = 0;
        for (int g = 0; g < GROUPS; ++g) v = smax[g][threadIdx.x] > v ? smax[g][threadIdx.x] : v;
        if (v) atomicMax(&resid_bits[(int64_t)unit * HD + threadIdx.x], v);
    }
}

__global__ void sketch_finalise_kernel(float *scale, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) scale[i] = scale[i] / 127.0f;  // the same expression the quantise kernel used
}

}  // namespace

// The quantising pass on its own: scale holds amax_d (scale_is_amax) or a_d, resid is raised from
// what it holds.  Arguments are the caller's to check.
int dc_sketch_quantise_launch(const char *who, const void *k, uint8_t *codes, const float *scale, float *resid,
                              int n_units, int n_h, int n_rows, int hd, int64_t sb, int64_t sh, int64_t sr, int64_t cb,
                              int64_t ch, int64_t cr, int scale_is_amax, float *scale_out, void *stream) {
    // Rows per block: 32 KB of keys, so that the blocks that run at a time walk the store together, as the copy that filled it did (longer
    // blocks are each somewhere else); 256 where there are few rows in all and a block's end, an LDS pass and HD atomics to its
    // unit's words, shows.  A prompt's layer, us, 32 KB / 64 KB / 128 KB: 16 units x 40003 rows of 128 columns 151 / 156 / 161, 8 x 131072
    // 244 / 249 / 258, 12 x 24683 of 256 144 / 145 / 148, 16 x 40003 of 64 87 / 88 / 89.  Below four units the atomics to a unit's words, one
    // behind the other, take longer than the keys: 64 KB for two units, 128 for one.  This pass alone, us: 2 x 131072 28.4 / 23.3 / 22.0, 2 x
    // 500000 88 / 68 / 73, 2 x 65536 17.0 / 13.9 / 15.8, 1 x 262144 45.9 / 32.3 / 26.5, 1 x 1000000 156 / 92 / 76, 1 x 500000 of 256 156 / 92 /
    // 76; 4 x 131072 40.7 / 42.7 / 40.0, 3 x 100000 24.4 / 23.6 / 26.1.
    const int64_t kb32 = 16384 / hd, each = n_units == 1 ? 4 : (n_units == 2 ? 2 : 1);
    const int64_t rpb = (int64_t)n_units * n_rows * hd >= (1ll << 24) ? kb32 * each : 256;
    const int64_t blocks = ((int64_t)n_rows + rpb - 1) / rpb * n_units;
    DC_REQUIRE(blocks < (1ll << 31), "%s: grid too large", who);
    const dim3 grid((unsigned)blocks);
    hipStream_t st = (hipStream_t)stream;
#define DC_LAUNCH_SKQ(HD)                                                                                   \
    hipLaunchKernelGGL(sketch_quantise_kernel<HD>, grid, dim3(kThreads), 0, st, (const uint16_t *)k, codes, scale, \
                       (uint32_t *)resid, n_h, n_rows, sb, sh, sr, cb, ch, cr, n_units, (int)rpb, scale_is_amax, scale_out)
    if (hd == 64) DC_LAUNCH_SKQ(64);
    else if (hd == 128) DC_LAUNCH_SKQ(128);
    else DC_LAUNCH_SKQ(256);
#undef DC_LAUNCH_SKQ
    DC_CHECK_LAUNCH(who);
    return DC_OK;
}

extern "C" int dc_sketch_build_bf16(const void *k, uint8_t *codes, float *scale, float *resid, int n_b,
                                    int n_h, int n_rows, int hd, int64_t sb, int64_t sh, int64_t sr,
                                    int64_t cb, int64_t ch, int64_t cr, int keep_scale, void *stream) {
    const char *who = "dc_sketch_build_bf16";
    DC_REQUIRE(k && codes && scale && resid, "%s: null pointer", who);
    DC_REQUIRE(n_b >= 0 && n_h >= 1 && n_rows >= 0, "%s: bad sizes", who);
    DC_REQUIRE(hd == 64 || hd == 128 || hd == 256, "%s: head_dim %d not in {64,128,256}", who, hd);
    DC_REQUIRE(dc_aligned16(k) && dc_aligned16(codes), "%s: k and codes must be 16-byte aligned", who);
    DC_REQUIRE(sb % 8 == 0 && sh % 8 == 0 && sr % 8 == 0 && sr >= hd,
               "%s: key strides must be multiples of 8 elements and row_stride >= hd", who);
    DC_REQUIRE(cb % 16 == 0 && ch % 16 == 0 && cr % 16 == 0 && cr >= hd,
               "%s: code strides must be multiples of 16 bytes and row_stride >= hd", who);
    const int64_t n_units = (int64_t)n_b * n_h;
    if (n_units == 0) return DC_OK;
    const int64_t bpu = n_rows > 0 ? ((int64_t)n_rows + kRowsPerBlock - 1) / kRowsPerBlock : 0;
    DC_REQUIRE(n_units * (bpu > 0 ? bpu : 1) < (1ll << 31), "%s: grid too large", who);
    hipStream_t st = (hipStream_t)stream;
    const int64_t n_sc = n_units * hd;
    const dim3 sgrid((unsigned)((n_sc + 255) / 256));
    if (!keep_scale) {
        hipLaunchKernelGGL(sketch_zero_kernel, sgrid, dim3(256), 0, st, (uint32_t *)scale, (uint32_t *)resid,
                           n_sc);
        DC_CHECK_LAUNCH(who);
    }
    if (bpu == 0) return DC_OK;
    const dim3 grid((unsigned)(n_units * bpu));
#define DC_LAUNCH_SKB(HD)                                                                            \
    hipLaunchKernelGGL(sketch_absmax_kernel<HD>, grid, dim3(kThreads), 0, st, (const uint16_t *)k,   \
                       (uint32_t *)scale, n_h, n_rows, sb, sh, sr, (int)bpu)
    if (!keep_scale) {
        if (hd == 64) DC_LAUNCH_SKB(64);
        else if (hd == 128) DC_LAUNCH_SKB(128);
        else DC_LAUNCH_SKB(256);
        DC_CHECK_LAUNCH(who);
    }
#undef DC_LAUNCH_SKB
    const int rc = dc_sketch_quantise_launch(who, k, codes, scale, resid, (int)n_units, n_h, n_rows, hd, sb, sh, sr, cb, ch,
                                             cr, keep_scale ? 0 : 1, nullptr, stream);
    if (rc) return rc;
    if (!keep_scale) {
        hipLaunchKernelGGL(sketch_finalise_kernel, sgrid, dim3(256), 0, st, scale, n_sc);
        DC_CHECK_LAUNCH(who);
    }
    return DC_OK;
}
