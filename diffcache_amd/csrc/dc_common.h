// Shared device helpers and host-side error plumbing for libdiffcache_hip.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/diffcache_hip.h"

#define DC_WAVE 64

// ---- host side -------------------------------------------------------------
void dc_set_error(const char *fmt, ...);

#define DC_REQUIRE(cond, ...)            \
    do {                                 \
        if (!(cond)) {                   \
            dc_set_error(__VA_ARGS__);   \
            return DC_EINVAL;            \
        }                                \
    } while (0)

#define DC_CHECK_LAUNCH(name)                                              \
    do {                                                                   \
        hipError_t e_ = hipGetLastError();                                 \
        if (e_ != hipSuccess) {                                            \
            dc_set_error("%s: launch failed: %s", name, hipGetErrorString(e_)); \
            return DC_ELAUNCH;                                             \
        }                                                                  \
    } while (0)

// select.hip: sort the selected ids of every unit (see the definition); n_rows = rows of
// the context the ids index into
int dc_sort_selected(const float *scores, int64_t scores_stride, const uint32_t *sel_keys,
                     uint32_t *idx_out, int64_t idx_stride, unsigned long long *scratch, int n_units,
                     int k_eff, int mode, int order, hipStream_t st, int n_rows);

// fused.hip: argument checks, state initialisation and the scan kernel of the sketch route
int dc_sketch_scan_launch(const char *who, const void *k, const uint8_t *codes, const float *scale,
                          const float *resid, const void *q, int n_b, int n_h, int n_rows, int hd, int64_t sb,
                          int64_t sh, int64_t sr, int64_t cb, int64_t ch, int64_t cr, int q_group, int budget,
                          int mode, int state_ready, void *workspace, size_t workspace_bytes,
                          void *ev_scan_begin, void *ev_scan_end, void *stream, const int32_t *hi_dev = nullptr,
                          int lo_row = 0);
// fused.hip: the bf16 scan of the streaming route (dc_score_prune_bf16 with an optional device-side region end)
int dc_score_prune_launch(const void *k, const void *q, int n_b, int n_h, int n_rows, int hd, int64_t sb, int64_t sh,
                          int64_t sr, int q_group, int budget, int mode, void *workspace, size_t workspace_bytes,
                          void *stream, const int32_t *hi_dev, int lo_row);
// fused.hip: dc_score_select_sketch_bf16 with an optional device-side region end
int dc_sketch_select_impl(const void *k, const uint8_t *codes, const float *scale, const float *resid, const void *q,
                          uint32_t *idx_out, int64_t idx_unit_stride, int n_b, int n_h, int n_rows, int hd,
                          int64_t sb, int64_t sh, int64_t sr, int64_t cb, int64_t ch, int64_t cr, int q_group,
                          int budget, int mode, int order, int state_ready, void *workspace, size_t workspace_bytes,
                          void *ev_scan_begin, void *ev_scan_end, void *stream, const int32_t *hi_dev, int lo_row);
// attn.hip: dc_gather_attn_bf16 with an optional device-side start of the suffix
int dc_gather_attn_common(const char *who, const void *q, const void *k, const void *v, const uint32_t *idx,
                          const void *new_k, const void *new_v, void *out, float *lse, int n_b, int n_h, int group,
                          int hd, int n_idx, int64_t idx_unit_stride, const uint32_t *n_idx_unit, int64_t region_lo,
                          int n_sink, int64_t recent_lo, int n_recent, const int32_t *n_recent_dev, int64_t ksb,
                          int64_t ksh, int64_t ksr, int64_t vsb, int64_t vsh, int64_t vsr, float scale,
                          void *workspace, size_t workspace_bytes, void *stream, const int32_t *recent_lo_dev,
                          const dc_step_args *step = nullptr);
bool dc_attn_valu(int group);  // the environment asks for the VALU version of the attention
int dc_merge_launch(const char *who, const float *acc, const float *ml, void *out, float *lse, int n_units, int group, int hd,
                    int n_splits, const dc_step_args *step, uint32_t *clear_hist, void *stream);
// short.hip: a decode layer in three kernels, for short contexts
bool dc_short_supported(const dc_layer_args *a, int region, int k_eff);
bool dc_one_kernel_first(const dc_layer_args *a, int region, int k_eff);
int dc_short_layer(const dc_layer_args *a, int region, int k_eff, void *sel_ws, void *attn_ws, size_t attn_ws_bytes,
                   void *stream, const dc_step_args *step);
// sketch.hip: the quantising pass of dc_sketch_build_bf16
int dc_sketch_quantise_launch(const char *who, const void *k, uint8_t *codes, const float *scale, float *resid,
                              int n_units, int n_h, int n_rows, int hd, int64_t sb, int64_t sh, int64_t sr, int64_t cb,
                              int64_t ch, int64_t cr, int scale_is_amax, float *scale_out, void *stream);
// small.hip: a whole decode layer in one kernel, for short contexts
bool dc_small_supported(int n_units, int region, int k_eff, int group, int hd, bool has_sketch);
size_t dc_small_workspace_bytes(int n_units, int region, int group, int hd);
size_t dc_small_cand_bytes(int n_units, int region);
int dc_small_state_init(int n_units, int region, void *cand, void *stream);
int dc_small_try(const dc_layer_args *a, int region, int k_eff, void *sel_ws, void *cand, void *attn_ws,
                 size_t attn_ws_bytes, void *stream, const dc_step_args *step);
bool dc_ws_state_trusted(const void *workspace);
void dc_ws_state_initialised(const void *workspace);

// kv.hip: the checks of dc_append_kv_bf16 on the append part of a step (DC_OK when there is none)
int dc_step_check(const char *who, const dc_layer_args *a, const dc_step_args *step);

static inline bool dc_aligned16(const void *p) { return (((uintptr_t)p) & 15u) == 0; }
static inline size_t dc_align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// ---- device side -----------------------------------------------------------
// dc_step_state_advance, by one thread
__device__ __forceinline__ void dc_state_advance(int32_t *s, int delta, int limit) {
    int64_t n = (int64_t)s[0] + delta;
    if (n > limit) {  // the window is full: this token has no row (the caller had to roll it over)
        s[3] = 1;
        n = limit;
    }
    if (n < 0) n = 0;
    s[0] = (int32_t)n;
    s[2] = s[1] + (int32_t)n;
}

// The token's row on its way into the store (dc_append_kv_bf16 inside another kernel): HD/4 threads of one
// block per unit carry 16 bytes each, the first half of K, the second of V.  load() goes in front of the
// block's last reduction, where registers are free, and store() behind it, so that nothing waits for it
// (in front of the gathered rows it costs the attention a fourth wave per SIMD).
struct DcAppend {
    uint16_t *k, *v;  // the stores (row 0 of unit (0, 0)); k null: nothing to append
    const int32_t *pos_dev;
    int64_t pos, pos_end;
};
inline DcAppend dc_append_of(const dc_step_args *step, const void *k, const void *v) {
    DcAppend a = {nullptr, nullptr, nullptr, 0, 0};
    if (step && step->append)
        a = {(uint16_t *)const_cast<void *>(k), (uint16_t *)const_cast<void *>(v), step->pos_dev, step->pos, step->pos_end};
    return a;
}
template <int HD>
struct DcNewRow {
    uint4 w;
    int64_t at;  // uniform
    bool live;
    __device__ __forceinline__ void load(const DcAppend &a, const uint16_t *new_k, const uint16_t *new_v, int unit, bool mine) {
        const int t = threadIdx.x;
        mine = mine && a.k;
        live = mine && t < HD / 4;
        at = a.pos;
        if (mine && a.pos_dev) at += (int64_t)*a.pos_dev;
        if (live) {
            const uint16_t *src = t < HD / 8 ? new_k : new_v;
            w = *reinterpret_cast<const uint4 *>(src + (int64_t)unit * HD + (t % (HD / 8)) * 8);
        }
    }
    // ku, vu: element offset of the unit's row 0 in the stores
    __device__ __forceinline__ void store(const DcAppend &a, int64_t ku, int64_t ksr, int64_t vu, int64_t vsr) const {
        const int t = threadIdx.x;
        if (live && at >= 0 && at < a.pos_end) {
            uint16_t *dst = t < HD / 8 ? a.k + ku + at * ksr : a.v + vu + at * vsr;
            *reinterpret_cast<uint4 *>(dst + (t % (HD / 8)) * 8) = w;
        }
    }
};

// 16-byte load of data that is read once (the scans stream gigabytes through the
// caches): the non-temporal hint keeps the lines from displacing what is reused, and the
// streaming kernels reach the plain read rate of the part with it (about 8 % faster).
__device__ __forceinline__ uint4 dc_load_stream16(const void *p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
    return make_uint4(t.x, t.y, t.z, t.w);
}

// the matching stores, for bulk data that the writing kernel does not read back
__device__ __forceinline__ void dc_store_stream16(void *p, uint4 v) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<u32x4 *>(p));
}
__device__ __forceinline__ void dc_store_stream8(void *p, uint2 v) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 t = {v.x, v.y};
    __builtin_nontemporal_store(t, reinterpret_cast<u32x2 *>(p));
}

__device__ __forceinline__ float dc_bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float dc_bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ float dc_bf16_to_f32(uint16_t v) { return __uint_as_float(((uint32_t)v) << 16); }

// round to nearest even; NaN -> canonical quiet NaN
__device__ __forceinline__ uint16_t dc_f32_to_bf16(float f) {
    uint32_t b = __float_as_uint(f);
    if ((b & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
    uint32_t lsb = (b >> 16) & 1u;
    return (uint16_t)((b + 0x7fffu + lsb) >> 16);
}

// order-preserving map f32 -> u32 (ascending)
__device__ __forceinline__ uint32_t dc_f2ord(float x) {
    uint32_t b = __float_as_uint(x);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Histogram bucket of a score (larger score = better = smaller bucket), a monotone
// map onto [0, DC_HIST_BINS).  Positive scores from 2^-20 up to 2^20 get 8 buckets
// per binade (the top-k of an attention scan lives there: a finer grid leaves
// fewer rows in the threshold bucket, a coarser one costs the scan fewer histogram
// atomics); smaller positives share the last fine bucket, larger ones the first;
// negative scores get two buckets per binade.
constexpr uint32_t kPosBinades = 40u, kSubBits = 3u;
constexpr uint32_t kPosBuckets = kPosBinades << kSubBits;
__device__ __forceinline__ uint32_t dc_score_bucket(float s) {
    const uint32_t b = __float_as_uint(s + 0.0f);  // -0 -> +0
    const uint32_t mag = b & 0x7fffffffu;
    if (b & 0x80000000u) return kPosBuckets + (mag >> 22);
    constexpr uint32_t lo = (127u - 20u) << 23, hi = ((127u - 20u + kPosBinades) << 23) - 1u;
    const uint32_t m = mag < lo ? lo : (mag > hi ? hi : mag);
    return (kPosBuckets - 1u) - ((m - lo) >> (23u - kSubBits));
}
static_assert(kPosBuckets + 512u <= DC_HIST_BINS, "bucket map exceeds the histogram");
// The same without a branch: for a lane that maps many scores in a row.
__device__ __forceinline__ uint32_t dc_score_bucket_flat(float s) {
    const uint32_t b = __float_as_uint(s + 0.0f), mag = b & 0x7fffffffu;
    constexpr uint32_t lo = (127u - 20u) << 23, hi = ((127u - 20u + kPosBinades) << 23) - 1u;
    const uint32_t m = mag < lo ? lo : (mag > hi ? hi : mag);
    const uint32_t pos = (kPosBuckets - 1u) - ((m - lo) >> (23u - kSubBits)), neg = kPosBuckets + (mag >> 22);
    return (b & 0x80000000u) ? neg : pos;
}

// 32-bit ordering key (smaller = better) and its histogram bucket.  The bucket is
// a monotone function of the key, so equal keys share a bucket.
// DC_MODE_IP:       key = ord(-(s + 0)),            bucket from s
// DC_MODE_REF_DIST: key = ord(d), d = f32(65536-s); bucket from s' = 65536 - d,
//                   which is exact and is s rounded onto d's grid.
__device__ __forceinline__ void dc_key_bucket(float s, int mode, uint32_t &key, uint32_t &bucket) {
    if (mode == DC_MODE_REF_DIST) {
        float d = 65536.0f - s;
        key = dc_f2ord(d);
        bucket = dc_score_bucket(65536.0f - d);
    } else {
        key = dc_f2ord(-(s + 0.0f));
        bucket = dc_score_bucket(s);
    }
}

// Margin of the sketch scan: a row can belong to the exact top-k only if
// approx + margin reaches the k-th largest approx.  e = sum_d |q_d| r_d bounds the
// quantisation error of one score, wabs = sum_d |q_d a_d| scales the fp32 rounding
// of both the approximate and the exact evaluation (128-term dots of values up to
// 127 a_d: below 1.5e-3 wabs together).  In DC_MODE_REF_DIST keys f32(65536 - s)
// of unequal scores can tie, within one ulp of the key: 2^-23 (65536 + |s|).
__device__ __forceinline__ float dc_sketch_margin(float e, float wabs, int mode) {
    const float ep = 1.02f * e + 4.0e-3f * wabs;
    float m = 2.0f * ep;
    if (mode == DC_MODE_REF_DIST) m += (65536.0f + 128.0f * wabs + e) * 4.8e-7f;
    return m;
}

// sum over the 16 lanes of a DPP row; every lane of the row receives the sum
__device__ __forceinline__ float dc_row16_sum(float v) {
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0x141, 0xF, 0xF, true);  // row_half_mirror
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0x140, 0xF, 0xF, true);  // row_mirror
    return v;
}

// sum over aligned groups of 8 lanes
__device__ __forceinline__ float dc_row8_sum(float v) {
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0xB1, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0x4E, 0xF, 0xF, true);
    v += __builtin_amdgcn_update_dpp(0.0f, v, 0x141, 0xF, 0xF, true);
    return v;
}

// sum over aligned groups of LPR lanes (8, 16 or 32)
template <int LPR>
__device__ __forceinline__ float dc_group_sum(float v) {
    if (LPR == 8) return dc_row8_sum(v);
    v = dc_row16_sum(v);
    if (LPR == 32) v += __shfl_xor(v, 16, 64);
    return v;
}

// Blocks of a grid whose first dimension is the units and whose others are the chunks of a unit, which need not fit the second (it and the
// third hold 65535): the kernel numbers them with dc_chunk() and leaves those beyond the last alone.
constexpr int kMostChunksY = 32768;
inline dim3 dc_unit_grid(int n_units, int64_t chunks) {
    return dim3((unsigned)n_units, (unsigned)(chunks < kMostChunksY ? chunks : kMostChunksY),
                (unsigned)((chunks + kMostChunksY - 1) / kMostChunksY));
}
__device__ __forceinline__ int dc_chunk() { return (int)(blockIdx.z * (unsigned)kMostChunksY + blockIdx.y); }

// A device word of the step (dc_step_state) that no block of the reading kernel changes: a scalar load, also where the compiler can no
// longer tell that nothing does.
__device__ __forceinline__ int32_t dc_step_word(const int32_t *p) {
    return *(const __attribute__((address_space(4))) int32_t *)p;
}

// Rows of a retrieval region that are live.  The kernels' grids and lists are laid out for
// n_cap rows; with hi_dev the region ends at the row that device word names (it moves up when the
// recent window is rolled over, between replays of a captured step), lo_row being its first row.
__device__ __forceinline__ int dc_live_rows(int n_cap, const int32_t *hi_dev, int lo_row) {
    if (!hi_dev) return n_cap;
    const int v = dc_step_word(hi_dev) - lo_row;
    return v < 0 ? 0 : (v < n_cap ? v : n_cap);
}

// 8 bf16 (one 16-byte load) dotted with 8 fp32 query values, added to acc
__device__ __forceinline__ float dc_dot8(const uint4 &w, const float (&q)[8], float acc) {
    acc = fmaf(dc_bf16_lo(w.x), q[0], acc);
    acc = fmaf(dc_bf16_hi(w.x), q[1], acc);
    acc = fmaf(dc_bf16_lo(w.y), q[2], acc);
    acc = fmaf(dc_bf16_hi(w.y), q[3], acc);
    acc = fmaf(dc_bf16_lo(w.z), q[4], acc);
    acc = fmaf(dc_bf16_hi(w.z), q[5], acc);
    acc = fmaf(dc_bf16_lo(w.w), q[6], acc);
    acc = fmaf(dc_bf16_hi(w.w), q[7], acc);
    return acc;
}

// This lane's 8 query values (columns col*8 .. col*8+7) of one unit.  A GQA
// group (q_group > 1) is averaged in fp32 in ascending head order, divided once
// and rounded to bf16, as torch's bf16 mean does (diffcache.py:193).  The loads
// of up to 8 heads are issued together, without a branch to a head (the last head again in the place of one that
// does not exist); a serial loop covers larger groups.  A group of a power of two is multiplied by the exact reciprocal.
__device__ __forceinline__ void dc_add_head(const uint4 &w, bool in, float (&acc)[8]) {
    const uint32_t x[4] = {in ? w.x : 0u, in ? w.y : 0u, in ? w.z : 0u, in ? w.w : 0u};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        acc[2 * i] += dc_bf16_lo(x[i]);
        acc[2 * i + 1] += dc_bf16_hi(x[i]);
    }
}
template <int HD>
__device__ __forceinline__ void dc_load_query(const uint16_t *__restrict__ Q, int64_t unit, int q_group, int col, float (&q)[8]) {
    const uint16_t *qp = Q + unit * q_group * HD + col * 8;
    auto head = [&](int g) __attribute__((always_inline)) {
        return *reinterpret_cast<const uint4 *>(qp + (g < q_group ? g : q_group - 1) * HD);
    };
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    if (q_group == 1) {
        dc_add_head(head(0), true, acc);
    } else if (q_group <= 4) {
        uint4 raw[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) raw[g] = head(g);
#pragma unroll
        for (int g = 0; g < 4; ++g) dc_add_head(raw[g], g < q_group, acc);
    } else {
        uint4 raw[8];
#pragma unroll
        for (int g = 0; g < 8; ++g) raw[g] = head(g);
#pragma unroll
        for (int g = 0; g < 8; ++g) dc_add_head(raw[g], g < q_group, acc);
        for (int g = 8; g < q_group; ++g) dc_add_head(*reinterpret_cast<const uint4 *>(qp + (int64_t)g * HD), true, acc);
    }
    if (q_group == 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = acc[i];
    } else if ((q_group & (q_group - 1)) == 0) {
        const float r = 1.0f / (float)q_group;
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = dc_bf16_to_f32(dc_f32_to_bf16(acc[i] * r));
    } else {
        const float n = (float)q_group;
#pragma unroll
        for (int i = 0; i < 8; ++i) q[i] = dc_bf16_to_f32(dc_f32_to_bf16(acc[i] / n));
    }
}
