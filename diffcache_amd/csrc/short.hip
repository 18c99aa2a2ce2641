// The chain of three kernels for contexts whose keys' scores fit a block's registers.
//
// A layer of a few thousand to a few ten thousand rows per unit is a chain of hand-overs, not of bytes, so
// the chain is as short as kernel boundaries make it:
//
//   1  short_score_kernel   scores every row (the arithmetic of dc_score_bf16), writes its 32-bit ordering key
//                           at the row's own place -- no list, no threshold to poll, no slot to reserve -- and adds
//                           the block's bucket counts to the unit's histogram
//   2  short_attend_kernel  every split of every unit finds the cutoff of its unit by itself, from the
//                           histogram and all keys of the unit in registers, picks the ids of its own 128 places of the
//                           attended list and attends to them (dc_attn_split_mfma): what other splits
//                           selected it never has to hear of, because all of them count the same keys in the same order
//   3  merge_kernel         the splits' softmax partials; leaves the histogram cleared
//
// Against the five kernels of the long-context routes (scan, exact pass, finish, attention, merge) that is two
// boundaries and three list hand-overs fewer; against the one kernel of small.hip it needs no resident grid, no wait
// between blocks and no exclusive GPU, so it also runs under capture and beside other streams.  A captured layer of
// 8 units x 16323 rows of 64 columns: 19.2 us, 24.8 us with the five kernels (8 query heads per unit; bytes: 2.2 us).
#include "dc_attn.h"
#include "dc_fused.h"

namespace {

constexpr int kSplitWaves = 8;                     // of a block of short_attend_kernel
constexpr int kSplitThreads = kSplitWaves * 64;
constexpr int kSplitRows = kSplitWaves * 16;       // list positions of a split: one tile of 16 per wave
constexpr int kShortMaxRows = 16 * 4 * kSplitThreads;  // 16 vectors of four keys per thread; places fit 16 bits
constexpr int kRankMost = 128;                     // rows of the threshold bucket that are ranked straight away
constexpr int kListMost = 2048;                    // rows of the threshold bucket that are listed
constexpr uint32_t kNoKey = 0xffffffffu;           // the key of no row

// The buckets of a histogram: those of dc_score_bucket, or, FINE, of half their width for positive scores (16 per binade
// from 2^-12 to 2^20).  Half as many candidates spare regions of up to 4 Ki rows a pass of the cutoff (8 units x 4028 rows:
// 17.1 -> 16.7 us, 2 x 4028 15.4 -> 14.8); in longer ones they cost as much in counts (8 x 16323 of 64 19.0 -> 19.5).
template <bool FINE>
struct ShortBuckets {
    static constexpr uint32_t kGrain = FINE ? 4u : kSubBits, kPos = FINE ? 512u : kPosBuckets;
    static constexpr uint32_t kLo = FINE ? (127u - 12u) << 23 : (127u - 20u) << 23;  // the least positive score told apart
    static_assert(kPos + 512u <= DC_HIST_BINS, "positive and negative buckets");
    static __device__ __forceinline__ uint32_t of(float s) {
        if (!FINE) return dc_score_bucket(s);
        const uint32_t b = __float_as_uint(s + 0.0f);  // -0 -> +0
        const uint32_t mag = b & 0x7fffffffu;
        if (b & 0x80000000u) return kPos + (mag >> 22);
        constexpr uint32_t hi = kLo + (kPos << (23u - kGrain)) - 1u;
        const uint32_t m = mag < kLo ? kLo : (mag > hi ? hi : mag);
        return (kPos - 1u) - ((m - kLo) >> (23u - kGrain));
    }
};

// Key (as dc_key_bucket) and bucket of a row; rows without a number go to either end of the order, as their bucket says.
template <bool FINE>
__device__ __forceinline__ void short_key(float s, int mode, uint32_t &key, uint32_t &bucket) {
    using B = ShortBuckets<FINE>;
    if (mode == DC_MODE_REF_DIST) {
        const float d = 65536.0f - s;
        key = dc_f2ord(d);
        bucket = B::of(65536.0f - d);
        if (!(s == s)) key = bucket < B::kPos ? 0u : kNoKey;
    } else {
        key = dc_f2ord(-(s + 0.0f));
        bucket = B::of(s);
    }
    key = key < kNoKey ? key : kNoKey - 1u;
}

// Bound by memory latency up to some 30 MB of keys (5 us at 8 units x 4028 rows of 128 columns, 7 at 8 x 16323 of 64,
// of which 2 are the launch), then by bandwidth (14.6 us at 8 x 32533 of 128: 4.6 TB/s).  A wave takes eight loads of 64 / LPR rows
// each at a time, two such parts in flight, the first of them on the way before the query is there.
template <int HD, bool FINE>
__global__ __launch_bounds__(kThreads) void short_score_kernel(
    const uint16_t *__restrict__ K, const uint16_t *__restrict__ Q, uint32_t *__restrict__ hist,
    uint32_t *__restrict__ keys, int64_t key_stride, int n_units, int n_h, int n_cap, int64_t sb, int64_t sh, int64_t sr,
    int q_group, int mode, int parts, const int32_t *__restrict__ hi_dev, int lo_row) {
    constexpr int LPR = HD / 8;
    constexpr int NL = 8;                     // loads of a lane per part
    constexpr int PART = 64 / LPR * NL;       // rows of a part
    constexpr int WAVES = kThreads / 64;
    __shared__ uint32_t lhist[DC_HIST_BINS];
    asm volatile("" ::"s"(K), "s"(Q), "s"(hist), "s"(keys), "s"(key_stride), "s"(n_units), "s"(n_h), "s"(n_cap), "s"(sb), "s"(sh), "s"(sr),
                 "s"(q_group), "s"(mode), "s"(parts), "s"(hi_dev), "s"(lo_row));  // all arguments at once
    const int n_rows = dc_live_rows(n_cap, hi_dev, lo_row);
    const int unit = blockIdx.x, blk = blockIdx.y;
    const int b = unit / n_h, h = unit % n_h;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int grp = lane / LPR, col = lane % LPR;
    const int64_t block_row0 = (int64_t)blk * parts * (WAVES * PART);
    if (block_row0 >= n_rows) return;  // the grid is laid out for n_cap rows
    const uint16_t *Ku = K + b * sb + h * sh + col * 8;
    const int64_t last = n_rows - 1;
    auto load_part = [&](int i, uint4 (&w)[NL]) __attribute__((always_inline)) {
        const int64_t row = block_row0 + (int64_t)(i * WAVES + wave) * PART + grp * NL;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const int64_t r = row + j > last ? last : row + j;
            w[j] = *reinterpret_cast<const uint4 *>(Ku + r * sr);
        }
    };
    uint4 wa[NL], wb[NL];
    load_part(0, wa);  // on the way with the query
    float q[8];
    dc_load_query<HD>(Q, unit, q_group, col, q);
    for (int i = tid; i < DC_HIST_BINS; i += kThreads) lhist[i] = 0;
    __syncthreads();
    uint32_t *ku = keys + (int64_t)unit * key_stride;
    auto work_part = [&](int i, const uint4 (&w)[NL]) __attribute__((always_inline)) {
        float mine = 0.f;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const float p = dc_group_sum<LPR>(dc_dot8(w[j], q, 0.f));
            mine = col == j ? p : mine;
        }
        const int64_t row = block_row0 + (int64_t)(i * WAVES + wave) * PART + grp * NL + col;
        if (col < NL && row < n_rows) {
            uint32_t key, bucket;
            short_key<FINE>(mine, mode, key, bucket);
            ku[row] = key;
            atomicAdd(&lhist[bucket], 1u);
        }
    };
    // the last vector of four is whole: what lies behind the last row reads as no row
    if (blk == 0 && tid < 3 && n_rows + tid < ((n_rows + 3) & ~3)) ku[n_rows + tid] = kNoKey;
    // (past the unit's last row the loads repeat it and nothing is kept)
    int i = 0;
    for (; i + 1 < parts; i += 2) {
        load_part(i + 1, wb);
        work_part(i, wa);
        load_part(i + 2, wa);
        work_part(i + 1, wb);
    }
    if (i < parts) work_part(i, wa);
    __syncthreads();
    uint32_t *hu = hist + (int64_t)unit * DC_HIST_BINS;
    for (int j = tid; j < DC_HIST_BINS; j += kThreads) {
        const uint32_t c = lhist[j];
        if (c) atomicAdd(&hu[j], c);
    }
}

// a value that is the same in all lanes, in a scalar register
__device__ __forceinline__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }

// Whether a key's bucket is `b` or worse (from the key alone).
template <bool FINE>
__device__ __forceinline__ bool key_reaches(uint32_t key, uint32_t b, int mode) {
    const float x = __uint_as_float((key & 0x80000000u) ? key & 0x7fffffffu : ~key);  // dc_f2ord, inverted
    return ShortBuckets<FINE>::of(mode == DC_MODE_REF_DIST ? 65536.0f - x : -x) >= b;
}

// The smallest key whose bucket is lane % 2 + bin or worse, in every lane of that parity: the ends of
// a bucket.  DC_MODE_IP: the map inverted.  DC_MODE_REF_DIST: the map inverted up to the rounding of d, the 32 keys
// around tried at once; scores beyond 32768, whose d has another grid than the score, may miss that window and
// are bisected.
template <bool FINE>
__device__ __forceinline__ uint32_t bucket_first_key(uint32_t bin, int mode) {
    constexpr uint32_t kLoMag = ShortBuckets<FINE>::kLo, kPos = ShortBuckets<FINE>::kPos, kGrain = ShortBuckets<FINE>::kGrain;
    constexpr uint32_t kFirst = 0x007fffffu, kLast = 0xff800000u;  // the keys of -inf and +inf
    const int lane = threadIdx.x & 63;
    const uint32_t b = bin + (uint32_t)(lane & 1);
    // the largest score in bucket b or a worse one
    const uint32_t mag = b < kPos ? kLoMag + ((kPos - b) << (23u - kGrain)) - 1u : (b - kPos) << 22;
    if (mode == DC_MODE_IP) {
        if (b == 0u) return 0u;
        if (b < kPos) return 0x7fffffffu - mag;
        return b - kPos < 512u ? 0x80000000u | mag : kNoKey;
    }
    const float s = __uint_as_float(b < kPos ? mag : 0x80000000u | mag);
    const uint32_t guess = dc_f2ord(65536.0f - (b < kPos + 511u ? s : -__builtin_inff()));
    uint32_t c = guess - 16u + (uint32_t)(lane >> 1);
    c = c < kFirst ? kFirst : (c > kLast ? kLast : c);
    unsigned long long hits = __ballot(key_reaches<FINE>(c, b, mode)) >> (lane & 1) & 0x5555555555555555ull;
    const int first = hits ? (int)__builtin_ctzll(hits) : 64;  // 2 * place in the window
    uint32_t out = guess - 16u + (uint32_t)(first >> 1);
    bool sure = first > 0 && first < 64;
    if (b == 0u) out = 0u, sure = true;
    if (b >= kPos + 511u) out = b == kPos + 511u ? kLast + 1u : kNoKey, sure = true;  // rows without a number
    if (__ballot(!sure)) {
        uint32_t lo = kFirst, hi = kLast;  // lo does not reach b > 0, hi does reach every b <= kPos + 510
        while (hi - lo > 1u) {
            const uint32_t mid = lo + (hi - lo) / 2u;
            if (key_reaches<FINE>(mid, b, mode)) hi = mid;
            else lo = mid;
        }
        if (!sure) out = hi;
    }
    return out;
}

struct ShortArgs {
    const uint32_t *hist, *keys;
    int64_t key_stride;
    uint32_t *idx_out;
    const int32_t *hi_dev;
    int n_cap, lo_row, k_eff, mode;
};

struct ShortShared {
    uint32_t lh[256];
    unsigned long long tie[kRankMost];
    uint32_t own[kSplitRows];  // the split's selected ids
    uint32_t wtot[kSplitWaves + 1];
    uint32_t n_tie;
    uint16_t list[kListMost];  // rows of the threshold bucket
};

// The bucket of the kk-th best key of a unit and how many of its keys are in; every wave for itself.  Without one
// (fewer rows than kk) the bucket is DC_HIST_BINS.
__device__ __forceinline__ void short_threshold(const uint32_t *__restrict__ hu, uint32_t kk, uint32_t &bin, uint32_t &rem) {
    constexpr int kPer = DC_HIST_BINS / 64;
    const int lane = threadIdx.x & 63;
    uint32_t h[kPer], sum = 0u;
#pragma unroll
    for (int i = 0; i < kPer / 4; ++i) {
        const uint4 t = reinterpret_cast<const uint4 *>(hu)[lane * (kPer / 4) + i];
        h[4 * i] = t.x, h[4 * i + 1] = t.y, h[4 * i + 2] = t.z, h[4 * i + 3] = t.w;
        sum += t.x + t.y + t.z + t.w;
    }
    const uint32_t incl = wave_incl_scan(sum, lane);
    const unsigned long long reach = __ballot(incl >= kk);
    uint32_t run = incl - sum, j = 0u;
#pragma unroll
    for (int i = 0; i < kPer - 1; ++i) {
        const bool go = run + h[i] < kk && j == (uint32_t)i;
        run += go ? h[i] : 0u;
        j += go ? 1u : 0u;
    }
    const int at = reach ? (int)__builtin_ctzll(reach) : 0;
    bin = reach ? (uint32_t)__builtin_amdgcn_readlane((int)(lane * kPer + j), at) : (uint32_t)DC_HIST_BINS;
    rem = kk - (uint32_t)__builtin_amdgcn_readlane((int)run, at);
}

// The rem-th smallest (key, id) of `n` candidates, rem < n: every candidate up to it is in.  each(f) calls f(key, id) for
// this thread's candidates.  Eight bits at a time, first of key - lo, then, among rows of one key, of the ids, until at
// most 64 are left, which are ranked.  Every wave reads the counts for itself, so a pass has two barriers.
template <typename Each>
__device__ __forceinline__ void short_cutoff(Each each, uint32_t n, uint32_t rem, uint32_t lo, uint32_t hi, int n_rows,
                                             ShortShared &sh, uint32_t &cut_key, uint32_t &cut_id) {
    const int tid = threadIdx.x, lane = tid & 63;
    uint32_t base = lo;  // of the values that are left: value - base <= span
    int top = hi == lo ? 0 : 32 - __clz((int)(hi - lo));
    bool by_id = false;
    uint32_t one = 0u;
    while (n > 64u) {
        if (top == 0) {  // one key; ids differ, so this happens once
            if (by_id) break;
            by_id = true;
            one = base;
            base = 0u;
            top = 32 - __clz(n_rows - 1);
        }
        const int width = top < 8 ? top : 8, shift = top - width;
        const uint32_t span = top >= 32 ? 0xffffffffu : (1u << top) - 1u;
        if (tid < 64) reinterpret_cast<uint4 *>(sh.lh)[tid] = make_uint4(0u, 0u, 0u, 0u);
        __syncthreads();
        each([&](bool live, uint32_t key, uint32_t id) __attribute__((always_inline)) {
            const uint32_t v = (by_id ? id : key) - base;
            const bool hit = live && v <= span && (!by_id || key == one);
            const unsigned long long hits = __ballot(hit);
            if (hits == 0ull) return;
            const int leader = (int)__builtin_ctzll(hits);
            const uint32_t place = v >> shift, lead = (uint32_t)__builtin_amdgcn_readlane((int)place, leader);
            if (__ballot(hit && place != lead) == 0ull) {  // long runs of one value: a wave adds its count once
                if (lane == leader) atomicAdd(&sh.lh[lead], (uint32_t)__popcll(hits));
            } else if (hit) {
                atomicAdd(&sh.lh[place], 1u);
            }
        });
        __syncthreads();
        const uint4 h4 = reinterpret_cast<const uint4 *>(sh.lh)[lane];
        const uint32_t sum = h4.x + h4.y + h4.z + h4.w, incl = wave_incl_scan(sum, lane);
        const unsigned long long reach = __ballot(incl >= rem);
        const int at = reach ? (int)__builtin_ctzll(reach) : 63;
        uint32_t run = incl - sum, j = 0u, c = h4.x;
        if (run + c < rem) run += c, j = 1u, c = h4.y;
        if (j == 1u && run + c < rem) run += c, j = 2u, c = h4.z;
        if (j == 2u && run + c < rem) run += c, j = 3u, c = h4.w;
        base += uniform((uint32_t)__builtin_amdgcn_readlane((int)(4u * lane + j), at)) << shift;
        rem -= (uint32_t)__builtin_amdgcn_readlane((int)run, at);
        n = (uint32_t)__builtin_amdgcn_readlane((int)c, at);
        top = shift;
        if (rem == n) break;  // the rest is in as a whole
        __syncthreads();      // the counts are cleared by the next pass
    }
    const uint32_t span = top >= 32 ? 0xffffffffu : (1u << top) - 1u;
    if (rem == n) {
        cut_key = by_id ? one : (hi - base < span ? hi : base + span);
        cut_id = by_id ? base + span : kNoKey;
        return;
    }
    if (tid == 0) sh.n_tie = 0u;
    if (tid < 64) sh.tie[tid] = ~0ull;
    __syncthreads();
    uint32_t zero = 0u;  // an address that the compiler cannot prove uniform: it would add once per wave, at length
    asm volatile("" : "+v"(zero));
    each([&](bool live, uint32_t key, uint32_t id) __attribute__((always_inline)) {
        const uint32_t v = (by_id ? id : key) - base;
        if (live && v <= span && (!by_id || key == one)) {
            const uint32_t e = atomicAdd(&sh.n_tie + zero, 1u);
            if (e < 64u) sh.tie[e] = ((unsigned long long)key << 32) | id;
        }
    });
    __syncthreads();
    const unsigned long long mine = sh.tie[lane];
    uint32_t rank = 0u;
    for (uint32_t e = 0; e < n; ++e) rank += sh.tie[e] < mine ? 1u : 0u;
    const unsigned long long is = __ballot((uint32_t)lane < n && rank == rem - 1u);
    const int at = is ? (int)__builtin_ctzll(is) : 0;
    cut_key = (uint32_t)__builtin_amdgcn_readlane((int)(mine >> 32), at);
    cut_id = (uint32_t)__builtin_amdgcn_readlane((int)mine, at);
}

// NV: vectors of four keys per thread.
//
// Bound by its chain and by instruction issue: at 8 units x 16323 rows (clock stamps) keys and counts arrive and the
// threshold is known after 1.7 us, its ends 0.3 later, the bits 0.7 (2.5 instructions a key; every split counts all keys of
// its unit, which no other block does for it), the places 0.6, the cutoff 1.8 in the splits that need one, the
// attention 2.1 (2.9 at 128 columns).  With the keys' comparisons kept in scalar registers and radix passes over all
// keys, 4 to 35 instructions a key and fifteen barriers, the kernel took 11.5 us instead of 9.0.
//
// Two bits per key decide most of it: whether its bucket is better than the threshold's (certain) and whether it
// is the threshold's (candidate).  The unit's list is [certain rows | candidates that are in], each in the order of
// threads and bits, so a place follows from one scan of the counts.  A split of certain rows alone writes out its bits
// and is done; one that reaches beyond them finds the cutoff among the candidates first.
template <int HD, int NV>
__global__ __launch_bounds__(kSplitThreads) void short_attend_kernel(AttnArgs a, int group, ShortArgs s) {
    constexpr int MW = (NV + 7) / 8;  // words of bits
    extern __shared__ float s_dyn[];
    __shared__ __align__(16) ShortShared sh;
    const int n_units = (int)(gridDim.x / (unsigned)a.n_splits);
    const int unit = blockIdx.x % n_units, split = blockIdx.x / n_units;
    const int tid = threadIdx.x;
    const uint32_t kk = (uint32_t)s.k_eff;
    const uint32_t slot0 = (uint32_t)split * kSplitRows;

    AttnFrame<HD> f;
    if (slot0 < kk) {  // splits of always-kept rows alone have nothing to select
        const int n_rows = dc_live_rows(s.n_cap, s.hi_dev, s.lo_row);
        const uint32_t *ku = s.keys + (int64_t)unit * s.key_stride;
        const uint4 *kp = reinterpret_cast<const uint4 *>(ku);
        uint4 kv[NV];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int v = i * kSplitThreads + tid;
            kv[i] = make_uint4(kNoKey, kNoKey, kNoKey, kNoKey);
            if (4 * v < n_rows) kv[i] = kp[v];
        }
        if (tid < kSplitRows) sh.own[tid] = 0u;
        uint32_t bin, rem;
        short_threshold(s.hist + (int64_t)unit * DC_HIST_BINS, kk, bin, rem);
        f.load(a, group, unit);
        uint32_t lo = kNoKey, hi = kNoKey - 1u;  // fewer rows than k: all are certain
        if (bin < (uint32_t)DC_HIST_BINS) {
            const uint32_t ends = bucket_first_key<NV <= 2>(bin, s.mode);
            lo = (uint32_t)__builtin_amdgcn_readlane((int)ends, 0);
            hi = (uint32_t)__builtin_amdgcn_readlane((int)ends, 1) - 1u;
        }
        uint32_t sure[MW], cand[MW];
#pragma unroll
        for (int w = 0; w < MW; ++w) sure[w] = cand[w] = 0u;
#pragma unroll
        for (int i = NV - 1; i >= 0; --i) {
            if (4 * i * kSplitThreads >= n_rows) continue;  // (the vectors go by the largest region)
            const uint32_t k4[4] = {kv[i].x, kv[i].y, kv[i].z, kv[i].w};
#pragma unroll
            for (int j = 3; j >= 0; --j) {
                sure[i / 8] += sure[i / 8] + (k4[j] < lo ? 1u : 0u);
                cand[i / 8] += cand[i / 8] + (k4[j] <= hi ? 1u : 0u);
            }
        }
        uint32_t cnt = 0u;
#pragma unroll
        for (int w = 0; w < MW; ++w) {
            cand[w] &= ~sure[w];
            cnt += (uint32_t)__popc(sure[w]) | (uint32_t)__popc(cand[w]) << 16;
        }
        uint32_t total;
        const uint32_t ex = block_excl_scan<kSplitThreads>(cnt, sh.wtot, &total);
        total = uniform(total);
        const uint32_t n_sure = total & 0xffffu, n_cand = total >> 16;
        // put(place, row) for every set bit
        auto each_bit = [&](const uint32_t(&bits)[MW], uint32_t place, auto put) __attribute__((always_inline)) {
#pragma unroll
            for (int w = 0; w < MW; ++w) {
                uint32_t m = bits[w];
                while (m) {
                    const uint32_t j = (uint32_t)__ffs(m) - 1u;
                    m &= m - 1u;
                    put(place++, (8u * w + (j >> 2)) * (4u * kSplitThreads) + 4u * tid + (j & 3u));
                }
            }
        };
        auto own = [&](uint32_t place, uint32_t row) __attribute__((always_inline)) {
            const uint32_t e = place - slot0;
            if (e < (uint32_t)kSplitRows) sh.own[e] = row;
        };
        const uint32_t p_sure = ex & 0xffffu, p_cand = ex >> 16;
        if (p_sure < slot0 + kSplitRows && p_sure + (cnt & 0xffffu) > slot0) each_bit(sure, p_sure, own);
        if (slot0 + kSplitRows > n_sure && n_sure < kk) {
            if (rem >= n_cand) {
                each_bit(cand, n_sure + p_cand, own);
            } else if (n_cand <= (uint32_t)kRankMost) {
                // few: the rank among them is the place
                if (NV <= 4) {
                    uint32_t e = p_cand;
#pragma unroll
                    for (int i = 0; i < NV; ++i) {
                        const uint32_t k4[4] = {kv[i].x, kv[i].y, kv[i].z, kv[i].w};
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (cand[0] >> (4 * i + j) & 1u)
                                sh.tie[e++] = ((unsigned long long)k4[j] << 32) | (uint32_t)(4 * (i * kSplitThreads + tid) + j);
                    }
                } else {
                    each_bit(cand, p_cand, [&](uint32_t place, uint32_t row) __attribute__((always_inline)) { sh.list[place] = (uint16_t)row; });
                    __syncthreads();
                    if (tid < (int)n_cand) {
                        const uint32_t row = sh.list[tid];
                        sh.tie[tid] = ((unsigned long long)ku[row] << 32) | row;
                    }
                }
                __syncthreads();
                constexpr int kLanes = kSplitThreads / kRankMost;  // lanes to an entry
                const uint32_t e = (uint32_t)(tid / kLanes);
                const unsigned long long mine = e < n_cand ? sh.tie[e] : ~0ull;
                uint32_t rank = 0u;
                for (uint32_t j = (uint32_t)(tid % kLanes); j < n_cand; j += kLanes) rank += sh.tie[j] < mine ? 1u : 0u;
#pragma unroll
                for (int d = 1; d < kLanes; d <<= 1) rank += (uint32_t)__shfl_xor((int)rank, d, 64);
                if (tid % kLanes == 0 && e < n_cand && rank < rem) own(n_sure + rank, (uint32_t)mine);
            } else if (n_cand <= (uint32_t)kListMost) {
                each_bit(cand, p_cand, [&](uint32_t place, uint32_t row) __attribute__((always_inline)) { sh.list[place] = (uint16_t)row; });
                __syncthreads();
                constexpr int kPer = kListMost / kSplitThreads;
                uint32_t ck[kPer], ci[kPer];
#pragma unroll
                for (int j = 0; j < kPer; ++j) {
                    const uint32_t e = j * kSplitThreads + tid;
                    ck[j] = kNoKey, ci[j] = 0u;
                    if (e < n_cand) {
                        ci[j] = sh.list[e];
                        ck[j] = ku[ci[j]];
                    }
                }
                auto each = [&](auto fn) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < kPer; ++j)
                        if (j * kSplitThreads < (int)n_cand) fn((uint32_t)(j * kSplitThreads + tid) < n_cand, ck[j], ci[j]);
                };
                uint32_t cut_key, cut_id, base = n_sure;
                short_cutoff(each, n_cand, rem, lo, hi, n_rows, sh, cut_key, cut_id);
                each([&](bool live, uint32_t key, uint32_t id) __attribute__((always_inline)) {
                    const bool in = live && (key < cut_key || (key == cut_key && id <= cut_id));
                    uint32_t n_in;
                    const uint32_t place = base + block_excl_scan<kSplitThreads>(in ? 1u : 0u, sh.wtot, &n_in);
                    if (in) own(place, id);
                    base += n_in;
                });
            } else {
                // a threshold bucket of thousands (rows that tie): the keys are read again for every pass
                auto each = [&](auto fn) __attribute__((always_inline)) {
                    for (int v0 = 0; 4 * v0 < n_rows; v0 += kSplitThreads) {
                        const int r = 4 * (v0 + tid);
                        uint4 k = make_uint4(kNoKey, kNoKey, kNoKey, kNoKey);
                        if (r < n_rows) k = kp[v0 + tid];
                        const uint32_t k4[4] = {k.x, k.y, k.z, k.w};
#pragma unroll
                        for (int j = 0; j < 4; ++j) fn(r + j < n_rows && k4[j] >= lo && k4[j] <= hi, k4[j], (uint32_t)(r + j));
                    }
                };
                uint32_t cut_key, cut_id, base = n_sure;
                short_cutoff(each, n_cand, rem, lo, hi, n_rows, sh, cut_key, cut_id);
                each([&](bool live, uint32_t key, uint32_t id) __attribute__((always_inline)) {
                    const bool in = live && (key < cut_key || (key == cut_key && id <= cut_id));
                    uint32_t n_in;
                    const uint32_t place = base + block_excl_scan<kSplitThreads>(in ? 1u : 0u, sh.wtot, &n_in);
                    if (in) own(place, id);
                    base += n_in;
                });
            }
        }
        __syncthreads();
        if (tid < kSplitRows && slot0 + tid < kk) s.idx_out[(int64_t)unit * a.idx_stride + slot0 + tid] = sh.own[tid];
    } else {
        f.load(a, group, unit);
    }
    const uint32_t *own = sh.own;
    dc_attn_split_mfma<HD, kSplitWaves, 1>(a, f, group, unit, split, s_dyn,
                                           [own, slot0](int, int p) { return own[((uint32_t)p - slot0) % kSplitRows]; });
}

// Blocks of the score kernel, where rows allow: two per CU.  Between 256 and 1024 a layer of up to 8 units x 8 Ki rows
// takes the same time; at 8 units x 32533 rows of 128 columns 1024 blocks cost 2.3 us more (every block
// adds its counts to the histogram), 256 cost 1.5 us more at 128 units x 4028.
constexpr int kScoreBlocks = 512;
// Bytes of the units' keys up to which the chain is taken: it reads all of them in bf16, the sketch chain half of
// that and another two kernels' worth of hand-overs.  Per layer, this chain / sketch chain, us: 8 units x 16316
// rows of 128 columns (33 MB) 21.9 / 27.3, x 24616 (50 MB) 26.4 / 28.8, x 32533 (67 MB) 30.1 / 29.9; 32 x 8124 (67 MB)
// 27.9 / 32.1, x 16316 (134 MB) 43.5 / 40.9; 64 x 4028 (66 MB) 28.4 / 33.5; 12 x 24615 of 256 (151 MB) 50.0 / 44.0;
// 8 x 16323 of 64 (17 MB) 19.2 / 24.8.  (With the dense scan of later the sketch chain takes 26.2, 27.7, 28.4; 29.7, 35.8; 32.5; 40.3;
// 22.7.)  It goes with k, 8 x 32533 x 128 with 4096 ids: 31.4 / 35.5, so long regions of which few rows are selected
// leave at kShortBytesFew.
constexpr int64_t kShortBytes = 64ll << 20, kShortBytesFew = 56ll << 20;

}  // namespace

// Whether a layer can take this chain: ids in any order, keys of a unit in a block's registers, row offsets of 32
// bits, the splits' partials in the LDS that a launch gets without asking, no wish for the VALU version of the attention; and
// whether it is short enough to.
bool dc_short_supported(const dc_layer_args *a, int region, int k_eff) {
    const int64_t n_units = (int64_t)a->n_b * a->n_h;
    return !dc_attn_valu(a->group) && a->order == DC_ORDER_ANY && !a->scores && k_eff > 0 && n_units > 0 && region >= 64 &&
           region <= kShortMaxRows &&
           n_units * region * a->hd * 2 <=
               (a->sketch_codes && region > 16 * 1024 && k_eff < region / 12 ? kShortBytesFew : kShortBytes) &&
           a->group >= 1 && a->group * a->hd <= 1024 && (a->hd == 64 || a->hd == 128 || a->hd == 256) && a->kv_row_stride > 0 &&
           (a->recent_lo + a->n_recent + 1) * a->kv_row_stride * 2 <= 0xffffffffll;
}

// Whether a layer that can run as one kernel (small.hip) does.  What decides is the time (us, one kernel / chain, G query heads to
// a unit, k ids).  The one kernel pays for every query head and every row of its serial phases; this chain pays for every split,
// all of which count all keys of their unit (units x k / 128 of them); the sketch chain for every candidate it
// scores again, and for two more kernels.
//   G >= 4       the chains: 8 x 4028 of 128 columns 19.5 / 16.5, x 16316 30.3 / 22.0, x 32533 34.4 / 27.7; 64 x 4028 37.3 / 28.8; 8 x
//                16316 of 64, G 8, 33.3 / 19.1; 12 x 24615 of 256 49.7 / 37.6; without a sketch 8 x 39932 36.9 / 33.7, 16 x 39932 of 64 34.9 / 32.7
//   G <= 2       this chain except, at 64 columns, from 48 Ki ids over all units on (64 Ki at G 2, 96 Ki at G 4: 12 x 20000, 4096 ids
//                22.7 / 25.2; 64 x 8124 33.7 / 43.3; 24 x 20000 at G 4 32.5 / 36.4), at 128 from 96 Ki (G 1: 32 x 8124, 4096 ids 34.4 /
//                37.2), and at 256 for a few units of 5 Ki rows and more (6 x 8124 20.0 / 22.0, 4 x 16316 22.4 / 24.0)
//   sketch chain except where much of the region is selected, 1/14 of it at 256 columns, 1/7 at 128 and 1/10 at 64, times G, half of it
//                at any G (24 x 12200 of 256, 4096 ids 56.5 / 66.2; G 4: 64 x 8124 115.8 / 151.4)
//   bf16 chain   except at G 1 up to 48 Ki rows, at G 2 up to 32 Ki, and at 256 columns from a sixth of the region on (12 x 24615 of 128
//                29.8 / 32.9; 16 x 16316 of 256 40.1 / 43.3; but 3 x 39932 of 128 29.0 / 27.1)
// Over 9000 shapes (1 to 64 units x 1000 to 65468 rows, 256 to 4096 ids, G 1 to 8) a layer takes 0.898 of what the one kernel alone
// took, 14 of them more than 1.05, none more than 1.10.  At most two units of more than 16 Ki rows, and callers without a
// sketch up to 12 Ki rows or two units, stay with the one kernel although this chain is mostly the faster one there too (2 x 16316
// of 128, G 4, 22.5 / 18.9).  Groups too large for this chain's attention: one kernel up to 32 MiB of keys (8 x 4028 of 256 at G 8, 256 ids
// 26.8 / 27.1, 1024 ids 32.2 / 30.7).
bool dc_one_kernel_first(const dc_layer_args *a, int region, int k_eff) {
    constexpr int64_t Ki = 1024;
    const int64_t n_units = (int64_t)a->n_b * a->n_h, k = k_eff;
    const int g = a->group, hd = a->hd;
    if (a->one_kernel == DC_ONE_KERNEL_EXCLUSIVE) return true;
    if (a->sketch_codes ? n_units <= 2 && region > 16 * Ki : n_units <= 2 || region <= 12 * Ki) return true;
    if (dc_short_supported(a, region, k_eff)) {
        if (hd == 64) return g <= 4 && n_units * k >= (g == 1 ? 48 : (g == 2 ? 64 : 96)) * Ki;
        if (hd == 128) return g == 1 && n_units * k >= 96 * Ki;
        return (g == 1 || (g == 2 && n_units >= 4)) && region >= 5 * Ki && n_units * region <= 64 * Ki && 4 * k <= region;
    }
    if (a->sketch_codes)
        return (region <= 16 * Ki && n_units * region * hd * 2 <= (32ll << 20)) || 2 * k >= region ||
               (hd == 64 ? 10 : (hd == 128 ? 7 : 14)) * k >= (int64_t)g * region;
    return (g == 1 && n_units > 3 && region < 48 * Ki) || (g == 2 && region < 32 * Ki) || (hd == 256 && g <= 4 && 6 * k >= region);
}

// The layer on `stream`.  sel_ws: the select part of the workspace, its histograms zero (and left so).
int dc_short_layer(const dc_layer_args *a, int region, int k_eff, void *sel_ws, void *attn_ws, size_t attn_ws_bytes,
                   void *stream, const dc_step_args *step) {
    const char *who = "dc_decode_layer(short context)";
    const int n_units = a->n_b * a->n_h, hd = a->hd;
    DC_REQUIRE((a->new_k == nullptr) == (a->new_v == nullptr), "%s: new_k and new_v must both be set or both be null", who);
    DC_REQUIRE(dc_aligned16(a->q) && dc_aligned16(a->k) && dc_aligned16(a->v) &&
                   (!a->new_k || (dc_aligned16(a->new_k) && dc_aligned16(a->new_v))),
               "%s: pointers must be 16-byte aligned", who);
    DC_REQUIRE(a->kv_batch_stride % 8 == 0 && a->kv_head_stride % 8 == 0 && a->kv_row_stride % 8 == 0 &&
                   a->kv_row_stride >= hd,
               "%s: strides must be multiples of 8 elements and row_stride >= hd", who);
    DC_REQUIRE(a->mode == DC_MODE_IP || a->mode == DC_MODE_REF_DIST, "%s: bad mode %d", who, a->mode);
    DC_REQUIRE(a->idx_unit_stride >= k_eff, "%s: idx_unit_stride < min(budget, region rows)", who);
    DC_REQUIRE(a->recent_lo + a->n_recent < 0xffffffffll, "%s: row numbers out of range", who);
    const FusedWs w = carve_fused(sel_ws, n_units, region, a->budget);
    const int n_total = k_eff + a->n_sink + a->n_recent + (a->new_k ? 1 : 0);
    const int n_splits = (n_total + kSplitRows - 1) / kSplitRows;
    const AttnWs aw = carve_attn(attn_ws, n_units, a->group, hd, n_splits);
    if (attn_ws_bytes < aw.bytes) {
        dc_set_error("%s: workspace %zu bytes < %zu needed", who, attn_ws_bytes, aw.bytes);
        return DC_ENOMEM;
    }
    DC_REQUIRE((int64_t)n_units * n_splits < (1ll << 31), "%s: grid too large", who);
    hipStream_t st = (hipStream_t)stream;
    // the survivor lists of the other routes hold the keys here (8 bytes a row there, 4 here)
    uint32_t *keys = reinterpret_cast<uint32_t *>(w.surv);
    const int64_t key_stride = ((int64_t)region + 3) & ~3ll;
    const uint16_t *k_region = (const uint16_t *)a->k + (int64_t)a->n_sink * a->kv_row_stride;

    const int part_rows = kThreads / 64 * (64 / (hd / 8)) * 8;
    const int64_t all_parts = (region + part_rows - 1) / part_rows;
    const int64_t parts = (n_units * all_parts + kScoreBlocks - 1) / kScoreBlocks;
    const int64_t bpu = (all_parts + parts - 1) / parts;
    const bool fine = region <= 2 * 4 * kSplitThreads;  // NV <= 2 of short_attend_kernel
    if (a->ev_scan_begin) (void)hipEventRecord((hipEvent_t)a->ev_scan_begin, st);
#define DC_LAUNCH_SSF(HD, FN)                                                                                         \
    hipLaunchKernelGGL((short_score_kernel<HD, FN>), dim3((unsigned)n_units, (unsigned)bpu), dim3(kThreads), 0, st, k_region,       \
                       (const uint16_t *)a->q, w.hist, keys, key_stride, n_units, a->n_h, region, a->kv_batch_stride,  \
                       a->kv_head_stride, a->kv_row_stride, a->group, a->mode, (int)parts, a->region_hi_dev, a->n_sink)
#define DC_LAUNCH_SS(HD)                    \
    do {                                    \
        if (fine) DC_LAUNCH_SSF(HD, true);  \
        else DC_LAUNCH_SSF(HD, false);      \
    } while (0)
    if (hd == 64) DC_LAUNCH_SS(64);
    else if (hd == 128) DC_LAUNCH_SS(128);
    else DC_LAUNCH_SS(256);
#undef DC_LAUNCH_SS
#undef DC_LAUNCH_SSF
    DC_CHECK_LAUNCH(who);
    if (a->ev_scan_end) (void)hipEventRecord((hipEvent_t)a->ev_scan_end, st);

    AttnArgs aa = {};
    aa.Q = (const uint16_t *)a->q;
    aa.K = (const uint16_t *)a->k;
    aa.V = (const uint16_t *)a->v;
    aa.new_k = (const uint16_t *)a->new_k;
    aa.new_v = (const uint16_t *)a->new_v;
    aa.ws_acc = aw.acc;
    aa.ws_ml = aw.ml;
    aa.n_recent_dev = a->n_recent_dev;
    aa.recent_lo_dev = a->region_hi_dev;
    aa.n_h = a->n_h;
    aa.n_idx = k_eff;
    aa.idx_stride = a->idx_unit_stride;
    aa.region_lo = a->n_sink;
    aa.n_sink = a->n_sink;
    aa.recent_lo = a->recent_lo;
    aa.n_recent = a->n_recent;
    aa.n_total = n_total;
    aa.n_splits = n_splits;
    aa.ksb = aa.vsb = a->kv_batch_stride, aa.ksh = aa.vsh = a->kv_head_stride, aa.ksr = aa.vsr = a->kv_row_stride;
    aa.scale = a->scale;
    aa.app = dc_append_of(step, a->k, a->v);
    ShortArgs sa;
    sa.hist = w.hist;
    sa.keys = keys;
    sa.key_stride = key_stride;
    sa.idx_out = a->idx_out;
    sa.hi_dev = a->region_hi_dev;
    sa.n_cap = region;
    sa.lo_row = a->n_sink;
    sa.k_eff = k_eff;
    sa.mode = a->mode;
    const dim3 grid((unsigned)(n_units * n_splits));
    const size_t lds = mfma_shared_bytes(hd, a->group, kSplitWaves);
#define DC_LAUNCH_SA(HD, NV) \
    hipLaunchKernelGGL((short_attend_kernel<HD, NV>), grid, dim3(kSplitThreads), lds, st, aa, a->group, sa)
#define DC_LAUNCH_SAV(HD)                                     \
    do {                                                      \
        if (region <= 2 * 4 * kSplitThreads) DC_LAUNCH_SA(HD, 2);      \
        else if (region <= 4 * 4 * kSplitThreads) DC_LAUNCH_SA(HD, 4); \
        else if (region <= 8 * 4 * kSplitThreads) DC_LAUNCH_SA(HD, 8); \
        else DC_LAUNCH_SA(HD, 16);                            \
    } while (0)
    if (hd == 64) DC_LAUNCH_SAV(64);
    else if (hd == 128) DC_LAUNCH_SAV(128);
    else DC_LAUNCH_SAV(256);
#undef DC_LAUNCH_SAV
#undef DC_LAUNCH_SA
    DC_CHECK_LAUNCH(who);
    return dc_merge_launch(who, aw.acc, aw.ml, a->out, a->lse, n_units, a->group, hd, n_splits, step, w.hist, stream);
}
