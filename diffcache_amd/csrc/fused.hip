// Streaming score + exact top-k in two kernels, without a dense score array.
// Same result as dc_score_bf16 followed by dc_topk_select (the set a size-k heap
// scan keeps, diffcache_cpu/src/nsw.rs:600-621), built for the case where the
// scores themselves are not wanted.
//
// Why: on MI355X every byte the scan writes costs several read bytes' worth of
// HBM time, so the 4 bytes/row of a dense score array are the main overhead of
// a kernel that otherwise streams 256 bytes/row at the read ceiling.
//
// score_prune_kernel streams the key rows like score_kernel, bins every key in
// the unit's bucket histogram, and keeps a row only if its bucket is not
// worse than the unit's running threshold bucket tb_run.  tb_run is the bucket
// of the k-th best key among the rows histogrammed so far; rows can only be
// added, so tb_run never undershoots the final threshold bucket and no member
// of the final top-k is ever dropped, however stale the value a block reads.
// Survivors are staged in LDS and appended to the unit's list as (id, score)
// with one atomic per block.  Blocks are ordered chunk-major so that all units
// advance together, and the first chunks of every unit are small so that a
// threshold exists early.
//
// classify_kernel (several blocks per unit) derives the exact threshold bucket
// from the complete histogram and splits the survivors into certain members and
// candidates; select_finish_kernel (one block per unit) finishes with the same
// radix select as finalize_kernel.
//
// The sketch route reads half the bytes for the same result: sketch_prune_kernel
// is the same scan over an 8-bit sketch of the keys (one byte per element, see
// sketch.hip) with a margin that makes its pruning safe, rescore_kernel computes
// the exact scores of the rows that survive it and lists them as candidates, and
// select_finish_kernel picks the k best of that list.
#include <stddef.h>
#include <type_traits>
#include "dc_common.h"
#include "dc_select.h"
#include "dc_fused.h"
#include "dc_pq.h"

namespace {

__global__ void init_state_kernel(uint32_t *hist, UnitState *state, int n_units) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t n_hist = (int64_t)n_units * DC_HIST_BINS;
    if (i < n_hist) hist[i] = 0;
    if (i < n_units) {
        state[i].tb_run = DC_HIST_BINS;  // nothing is pruned until a threshold exists
        state[i].surv_cnt = 0;
        state[i].win_cnt = 0;
        state[i].cand_cnt = 0;
        state[i].c_less = 0;
        state[i].margin = 0;
        state[i].sync_cnt = 0;
        state[i].sync_err = 0;
        state[i].cut_key = 0;
        state[i].cut_id = 0;
    }
}

// A block's copy of its unit's running threshold bucket, in LDS.  The poll of the unit's
// value crosses the chip (agent scope) and every younger load of the polling wave returns
// after it, so one wave of the block polls and the others read the copy.
__device__ __forceinline__ uint32_t lds_load_relaxed(const uint32_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_store_relaxed(uint32_t *p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// End of a scan block: append the block's survivors (staged per wave in LDS) to
// the unit's list with one returning atomic, flush the block's histogram, and in
// the blocks chosen by the caller refresh the unit's running threshold from
// whatever part of the histogram is visible.  Staleness only loosens the bound.
template <typename E = uint2>
__device__ __forceinline__ void prune_block_finish(uint32_t *lhist, const E *wstage, uint32_t wcnt,
                                                   uint32_t *s_wcnt, uint32_t *s_base, uint32_t *wtot,
                                                   UnitState *st, uint32_t *hu, E *surv_unit,
                                                   bool refresh, uint32_t kk) {
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) s_wcnt[wave] = wcnt;
    __syncthreads();

    // the atomic is in flight while the histogram is flushed
    uint32_t wbase = 0, cnt = 0;
#pragma unroll
    for (int w2 = 0; w2 < kThreads / 64; ++w2) {
        if (w2 < wave) wbase += s_wcnt[w2];
        cnt += s_wcnt[w2];
    }
    if (tid == 0) *s_base = cnt ? atomicAdd(&st->surv_cnt, cnt) : 0;
    for (int i = tid; i < DC_HIST_BINS; i += kThreads) {
        const uint32_t c = lhist[i];
        if (c) atomicAdd(&hu[i], c);
    }
    __syncthreads();
    {
        E *dst = surv_unit + *s_base + wbase;
        for (uint32_t i = lane; i < wcnt; i += 64) dst[i] = wstage[i];
    }
    if (!refresh) return;

    // Coalesced, L2-bypassing read of the unit's histogram into LDS (lhist is
    // free again), then kBinsPerThread adjacent bins per thread.
    {
        const unsigned long long *h64 = reinterpret_cast<const unsigned long long *>(hu);
        unsigned long long *l64 = reinterpret_cast<unsigned long long *>(lhist);
        for (int i = tid; i < DC_HIST_BINS / 2; i += kThreads)
            l64[i] = __hip_atomic_load(h64 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    constexpr int kBins = DC_HIST_BINS / kThreads;  // adjacent bins a thread owns
    static_assert(kBins * kThreads == DC_HIST_BINS, "bin split");
    uint32_t bins[kBins];
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < kBins; ++i) {
        bins[i] = lhist[tid * kBins + i];
        sum += bins[i];
    }
    uint32_t total;
    const uint32_t excl = block_excl_scan<kThreads>(sum, wtot, &total);
    if (excl < kk && kk <= excl + sum) {
        uint32_t run = excl;
        bool done = false;
#pragma unroll
        for (int i = 0; i < kBins; ++i) {
            if (!done && run + bins[i] >= kk) {
                atomicMin(&st->tb_run, (uint32_t)(tid * kBins + i));
                done = true;
            }
            run += bins[i];
        }
    }
}

constexpr uint32_t kNoRow = 0xffffffffu;  // in the place of a row's key: there is no such row
// words between the units of a dense scan's keys (16-byte rows of them)
__host__ __device__ __forceinline__ int64_t dense_key_stride(int n_cap) { return ((int64_t)n_cap + 3) & ~3ll; }

// DENSE: for scans of more than 768 rows a unit and up to 1.75 Mi in all (plan_dense_keys), as in the sketch scan below:
// every row's 32-bit key goes to the row's own place, nothing is polled, staged or listed, and blocks take equal shares; a CU
// runs four at a time, above 1 Mi rows some start late (plan_dense_keys).  Its loads come in halves of a step (quarters at 256 columns), two of them in flight, the first two ahead of the query; a
// step's sixteen at a time, behind the query and behind the step before them: per layer, us, 32 units x 49933 rows of 128 95.2 / 93.4, 4 x
// 127028 44.8 / 43.1, 16 x 65404 of 64 44.5 / 43.6, 64 x 16432 71.8 / 71.1, 8 x 131004 67.5 / 67.9.
template <int HD, bool DENSE>
__global__ __launch_bounds__(kThreads) void score_prune_kernel(
    const uint16_t *__restrict__ K, const uint16_t *__restrict__ Q, uint32_t *__restrict__ hist,
    UnitState *__restrict__ state, uint2 *__restrict__ surv, int n_units, int n_h, int n_cap,
    int64_t sb, int64_t sh, int64_t sr, int q_group, int mode, int k_eff, int small_chunks,
    int big_steps, int n_chunks, uint32_t apart, const int32_t *__restrict__ hi_dev, int lo_row) {
    if constexpr (DENSE)  // all arguments at once: read where they are first used, they are half a dozen round trips in a row
        asm volatile("" ::"s"(K), "s"(Q), "s"(hist), "s"(surv), "s"(n_units), "s"(n_h), "s"(n_cap), "s"(sb), "s"(sh), "s"(sr), "s"(q_group),
                     "s"(mode), "s"(big_steps), "s"(n_chunks), "s"(apart), "s"(hi_dev), "s"(lo_row));
    constexpr int LPR = HD / 8;
    constexpr int CH = LPR < 16 ? LPR : 16;
    __shared__ uint32_t lhist[DC_HIST_BINS];
    __shared__ uint2 stage[DENSE ? 1 : kStage];
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t s_wcnt[kThreads / 64];
    __shared__ uint32_t s_base;
    const int n_rows = dc_live_rows(n_cap, hi_dev, lo_row);

    const int unit = blockIdx.x, chunk = DENSE ? (int)blockIdx.y : dc_chunk();
    if (!DENSE && chunk >= n_chunks) return;
    const int b = unit / n_h, h = unit % n_h;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int grp = lane / LPR, col = lane % LPR;

    const bool small = !DENSE && chunk < small_chunks;
    // Units may sit a power of two apart in memory; rotating each unit's order of chunks keeps blocks that run together from walking
    // the same address offsets: large chunks of the listed scan by seven a unit; those of the dense scan, of which a grid holds few, so
    // that the units start evenly apart.  (Dense, per layer, us, without / by seven / evenly: 8 units of 131072 rows of 128 columns 74.1 / 65.2 /
    // 64.6, 4 of 262144 71.0 / 69.3 / 65.6, 8 of 65536 of 256 71.1 / 67.1 / 67.0, 4 of 131072 of 256 70.9 / 69.4 / 66.1; 8 of 140128 of 128 69.3 /
    // - / 70.1.  Not at 64 columns: 8 of 131072 40.7 / 41.9 / 42.0, 32 of 50129 57.9 / - / 60.1; in the dense sketch scan it changes nothing.)
    int big_id = chunk;
    if constexpr (!DENSE) {
        big_id = small ? 0 : (int)(((uint32_t)(chunk - small_chunks) + (uint32_t)unit * 7u) % (uint32_t)(n_chunks - small_chunks));
    } else if constexpr (HD > 64) {  // apart: n_chunks / n_units in 1/65536 (without a division here, in front of the first loads)
        big_id += (int)((uint32_t)unit * apart >> 16);
        big_id -= big_id < n_chunks ? 0 : n_chunks;
    }
    const int64_t block_row0 =
        small ? (int64_t)chunk * kRowsPerBlockStep
              : (int64_t)small_chunks * kRowsPerBlockStep + (int64_t)big_id * big_steps * kRowsPerBlockStep;
    const int steps = small ? 1 : big_steps;

    uint32_t *du = reinterpret_cast<uint32_t *>(surv) + (int64_t)unit * dense_key_stride(n_cap);
    if (DENSE) {  // places behind the live end, up to the capacity that the readers go by
        int64_t end = block_row0 + (int64_t)steps * kRowsPerBlockStep;
        end = end < dense_key_stride(n_cap) ? end : dense_key_stride(n_cap);
        for (int64_t r = (block_row0 > n_rows ? block_row0 : (int64_t)n_rows) + tid; r < end; r += kThreads) du[r] = kNoRow;
    }
    if (block_row0 >= n_rows) return;  // the grid is laid out for n_cap rows

    const uint16_t *Ku = K + b * sb + h * sh + col * 8;
    UnitState *st = state + unit;
    const int last = n_rows - 1;
    if constexpr (DENSE) {
        // A step's rows in parts of eight loads, two of them on the way at any time, the first two before the query is there; past the
        // end of the block its last row again, so that the number of loads in flight is known.
        constexpr int NL = 8, PARTS = LPR / NL;
        const int64_t blk_end = block_row0 + (int64_t)steps * kRowsPerBlockStep - 1;
        const int64_t blk_last = blk_end < (int64_t)last ? blk_end : (int64_t)last;
        auto load_part = [&](int i, uint4 (&w)[NL]) __attribute__((always_inline)) {
            const int64_t row = block_row0 + (int64_t)(i / PARTS) * kRowsPerBlockStep + wave * 64 + grp * LPR + i % PARTS * NL;
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                const int64_t at = row + j > blk_last ? blk_last : row + j;
                w[j] = dc_load_stream16(Ku + at * sr);
            }
        };
        uint4 wa[NL], wb[NL];
        load_part(0, wa);
        load_part(1, wb);
        for (int i = tid; i < DC_HIST_BINS; i += kThreads) lhist[i] = 0;
        float q[8];
        dc_load_query<HD>(Q, unit, q_group, col, q);
        __syncthreads();
        const int64_t first = block_row0 + wave * 64;
        int my_steps = 0;  // of this wave, those that hold rows
        if (first < n_rows) {
            const int64_t left = ((int64_t)n_rows - first + kRowsPerBlockStep - 1) / kRowsPerBlockStep;
            my_steps = left < steps ? (int)left : steps;
        }
        float mine = 0.f;
        auto work_part = [&](int i, const uint4 (&w)[NL]) __attribute__((always_inline)) {
            const int c0 = i % PARTS * NL;
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                const float p = dc_group_sum<LPR>(dc_dot8(w[j], q, 0.f));
                mine = col == c0 + j ? p : mine;
            }
            if (i % PARTS != PARTS - 1) return;
            const int64_t row = first + (int64_t)(i / PARTS) * kRowsPerBlockStep + lane;
            if (row < n_rows) {
                uint32_t key, bucket;
                dc_key_bucket(mine, mode, key, bucket);
                du[row] = key < kNoRow ? key : kNoRow - 1u;
                atomicAdd(&lhist[bucket], 1u);
            }
        };
        const int parts = my_steps * PARTS;
        int i = 0;
        // From 128 columns on the number of parts is even and the last two are worked on without further loads, which a short block would
        // wait for at its end (selections of 8 x 17940 rows of 128 19.2 -> 18.5 us; at 64 columns 32 x 49933 take 1 us longer with that).
        constexpr int kAhead = PARTS > 1 ? 3 : 1;
        for (; i + kAhead < parts; i += 2) {
            work_part(i, wa);
            load_part(i + 2, wa);
            work_part(i + 1, wb);
            load_part(i + 3, wb);
        }
        if (i < parts) {
            work_part(i, wa);
            if (PARTS > 1) work_part(i + 1, wb);
        }
        __syncthreads();
        uint32_t *hu = hist + (int64_t)unit * DC_HIST_BINS;
        for (int i = tid; i < DC_HIST_BINS; i += kThreads) {
            const uint32_t c = lhist[i];
            if (c) atomicAdd(&hu[i], c);
        }
        return;
    }
    for (int i = tid; i < DC_HIST_BINS; i += kThreads) lhist[i] = 0;
    uint32_t tb = load_relaxed(&st->tb_run);

    float q[8];
    dc_load_query<HD>(Q, unit, q_group, col, q);
    __syncthreads();

    // Each wave stages its survivors in its own slice of `stage` (at most 64 per
    // step), so the cursor is a wave-uniform register and no LDS atomic is needed.
    uint2 *wstage = stage + wave * (kBigSteps * 64);
    uint32_t wcnt = 0;
    const unsigned long long lt = (1ull << lane) - 1ull;

    for (int step = 0; step < steps; ++step) {
        const int64_t row0 = block_row0 + (int64_t)step * kRowsPerBlockStep + wave * 64;
        if (row0 >= n_rows) break;  // wave-uniform; no barrier inside the loop
        float mine = 0.f;
        uint32_t tb_next = tb;
#pragma unroll
        for (int c0 = 0; c0 < LPR; c0 += CH) {
            uint4 w[CH];
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                int64_t r = row0 + grp * LPR + c0 + j;
                r = r > last ? last : r;
                w[j] = dc_load_stream16(Ku + r * sr);
            }
            // the threshold for the next step queues up behind this step's rows
            if (c0 + CH >= LPR && step + 1 < steps) tb_next = load_relaxed(&st->tb_run);
#pragma unroll
            for (int j = 0; j < CH; ++j) {
                float p = dc_group_sum<LPR>(dc_dot8(w[j], q, 0.f));
                mine = (col == c0 + j) ? p : mine;
            }
        }
        const int64_t myrow = row0 + lane;
        const bool valid = myrow < n_rows;
        uint32_t key = 0, bucket = 0xffffffffu;
        if (valid) dc_key_bucket(mine, mode, key, bucket);
        // Only rows that can still matter are kept and counted: the final threshold
        // bucket is never worse than tb, so it is fixed by the counts of buckets <= tb.
        const bool keep = valid && bucket <= tb;
        if (keep) atomicAdd(&lhist[bucket], 1u);
        const unsigned long long mask = __ballot(keep);
        if (keep) wstage[wcnt + __popcll(mask & lt)] = make_uint2((uint32_t)myrow, __float_as_uint(mine));
        wcnt += (uint32_t)__popcll(mask);
        tb = tb_next;
    }
    // every 4th small block and every 8th large one refresh the running threshold
    const bool refresh = small ? (chunk & 3) == 3 : ((chunk - small_chunks) & 7) == 7;
    prune_block_finish(lhist, wstage, wcnt, s_wcnt, &s_base, wtot, st, hist + (int64_t)unit * DC_HIST_BINS,
                       surv + (int64_t)unit * n_cap, refresh, (uint32_t)k_eff);
}

// largest value of aligned groups of LPR lanes (8, 16 or 32), in every lane of the group
template <int LPR>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// Scan of the 8-bit sketch of the keys.  Row i of a unit is stored as codes
// u_id = c_id + 128 with k_id = a_d * c_id + e_id, |e_id| <= r_d (a: `scale`,
// r: `resid`, both per unit and channel).  The scan computes
//   approx_i = sum_d (q_d a_d) c_id,   |s_i - approx_i| <= E' for every row,
//   E' = sum_d |q_d| r_d + fp32 slack,
// where s_i is the fp32 score the exact kernels produce.  With A_k the k-th
// largest approx, every member of the exact top-k has approx_i >= A_k - 2E' - Q
// (Q: one quantisation step of the reference key in DC_MODE_REF_DIST, where equal
// keys of unequal scores tie).  So rows are histogrammed by bucket(approx_i), which
// yields the bucket of A_k exactly as in score_prune_kernel, and a row is kept when
// bucket(approx_i + margin) is not worse than the running threshold bucket,
// margin = 2E' + Q.  The kept rows are rescored exactly by rescore_kernel.
//
// The sums run on the matrix cores.  A weight q_d a_d is a whole multiple of 2^(e - 30), |q_d a_d| < 2^e, written
// as four signed digits of base 256; the codes less 128 are signed bytes; so v_mfma_i32_16x16x64_i8 sums every
// digit exactly and three fp32 additions put them together.  (Largest error against 64 bits, relative to
// sum |q_d a_d|: 5.5e-6 / 5.2e-6 / 3.4e-6 at head dims 64 / 128 / 256; 16 fp32 additions a lane and a tree over the
// lanes, biased codes, gave 1.6e-5 / 1.4e-5 / 7.4e-6.)  Sixteen query columns would fit where one is
// wanted: the sixteen rows of the left operand hold the digits instead, several times over with zeros elsewhere, so
// that a wave's 64 rows end up one to a lane.  From 128 columns on two lanes share a row (S = 2), because a load of
// 16 rows x 64 bytes takes half lines, which streaming loads fetch twice (205 us instead of 180 us at 64 units x
// 131004 rows of 128).  A step of 64 rows of 128 takes 284 vector instructions in all, 532 with fp32 arithmetic on the
// codes; the kernel is bound by memory latency at few units and by HBM at many.  The first rows, the
// query, scales and residuals are all requested at the block's start, one round trip instead of three, and little stands in
// front of them: the arguments are read at once, the unit and the chunk are the grid's dimensions, the heads of a group are asked for without
// a branch each.  (Clock stamps, 8 x 32533 rows of 128: the first rows are there after 2.8 to 4.5 us, 3.5 to 5.8 before that; the kernel
// ends after 8.1, 8.9 before.  Two steps of rows ahead instead of one, or the query in front of the rows: no earlier, the memory
// system is busy by then.)  Layers, us, before / after that and the like of it in the exact pass and the attention: 8 x 32533 29.6 / 28.7, 8 x
// 131004 46.8 / 46.2, 64 x 65420 126.3 / 123.5, 12 x 24615 of 256 38.9 / 38.0, 8 x 16316 (short chain) 24.5 / 23.6.
// Measured before / after (kernel trace): 8 x 131004 rows of 128 29.8 / 27.3 us, 4 x 127028 19.6 / 17.7, 64 x 131004
// 185.1 / 180.8, 8 x 1048508 183.1 / 179.1, 8 x 16323 of 64 11.1 / 9.5.
constexpr uint32_t kBulkKeep = 96;      // of the 128 rows of a wave's first two steps
// What the sketch scan keeps of a row: the row, and the bucket of (approximation + margin), which
// is all the exact pass asks of it (the exact pass keeps the row when that bucket is not worse
// than the final threshold bucket).  One word instead of (row, approximation): a byte the scan
// writes costs it several bytes read.  Rows of a unit beyond 2^22 do not fit: the callers send
// such regions down the bf16 route.
constexpr int kSketchRowBits = 22;
constexpr int kSketchMaxRows = 1 << kSketchRowBits;
static_assert(kSketchMaxRows / kRowsPerBlockStep <= 65535, "the chunks of a unit are the second dimension of the scan's grid");
static_assert(kSketchMaxRows == DC_SKETCH_MAX_ROWS && DC_HIST_BINS <= (1 << (32 - kSketchRowBits)), "row and bucket share a word");
__device__ __forceinline__ uint32_t sketch_entry(uint32_t bucket, uint32_t row) { return (bucket << kSketchRowBits) | row; }
// words of two bytes between the units of a dense scan's buckets (16-byte rows of them)
__host__ __device__ __forceinline__ int64_t dense_stride(int n_cap) { return ((int64_t)n_cap + 7) & ~7ll; }

// DENSE: for scans whose blocks all run at the same time.  There a threshold never comes early enough to drop a row
// worth its poll, so nothing is polled or listed: every row's bucket of (approximation + margin) goes to the row's
// own place, two bytes, and the exact pass reads them all.  That leaves out the block's closing round trip (the returning
// atomic that reserves its list slots) and the refresh of the threshold behind it, and the grid can be one of equal
// shares (sizes and times: plan_dense).  Nor is there a way out for rows that all tie, which a listed scan stops reading (bulk,
// below): selections among such rows take up to 14 % longer at 256 columns (1 x 131001 rows 140 -> 160 us, 32 x 65001 322 -> 355)
// and 6 % at 128 (32 x 65001 204 -> 215).
template <int HD, bool SHARED_POLL, bool DENSE>
__global__ __launch_bounds__(kThreads, HD <= 128 ? 4 : 1) void sketch_prune_kernel(
    const uint8_t *__restrict__ C, const uint16_t *__restrict__ Q, const float *__restrict__ scale,
    const float *__restrict__ resid, uint32_t *__restrict__ hist, UnitState *__restrict__ state,
    uint2 *__restrict__ surv, int n_units, int n_h, int n_cap, int64_t cb, int64_t ch, int64_t cr,
    int q_group, int mode, int k_eff, int small_chunks, int big_steps, const int32_t *__restrict__ hi_dev,
    int lo_row) {
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    constexpr int S = HD == 64 ? 1 : 2;   // lanes of 16 that share a row: a load takes whole 128-byte lines
    constexpr int KS = HD / (64 * S);     // matrix instructions per tile of 16 / S rows
    constexpr int TILES = 4 * S;          // tiles of a wave's 64 rows
    constexpr int kLoads = TILES * KS;    // 16-byte loads of a lane per step
    constexpr int LPQ = HD / 8;           // lanes that hold a copy of the weights, eight each
    // (all arguments at once: read where they are first used, they are half a dozen round trips in a row)
    asm volatile("" ::"s"(C), "s"(Q), "s"(scale), "s"(resid), "s"(hist), "s"(state), "s"(surv), "s"(n_units), "s"(n_h), "s"(n_cap), "s"(cb),
                 "s"(ch), "s"(cr), "s"(q_group), "s"(mode), "s"(k_eff), "s"(small_chunks), "s"(big_steps), "s"(hi_dev), "s"(lo_row));
    const int n_rows = dc_live_rows(n_cap, hi_dev, lo_row);
    __shared__ uint32_t lhist[DC_HIST_BINS];
    __shared__ __align__(16) uint8_t s_w[4][HD];  // the weights' digits, lowest first
    __shared__ uint32_t stage[DENSE ? 1 : kStage];  // kept rows as kSketchEntry words
    __shared__ uint32_t s_tb;  // the block's copy of the unit's running threshold bucket
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t s_wcnt[kThreads / 64];
    __shared__ uint32_t s_base;

    const int unit = blockIdx.x, chunk = blockIdx.y;
    const int b = unit / n_h, h = unit % n_h;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    // This lane loads 16 columns of row (lane & 15) / S of every tile; the row whose score it ends up with:
    const int grp = lane >> 4, side = S == 1 ? 0 : lane & 1, par = S == 1 ? 0 : (grp ^ lane) & 1;
    const int own_row = S == 1 ? lane : (4 * side + 2 * par + (grp >> 1)) * 8 + ((lane & 15) >> 1);

    const bool small = !DENSE && chunk < small_chunks;
    const int big_chunks = (int)gridDim.y - small_chunks;
    const int big_id = DENSE ? chunk : (small ? 0 : (int)(((uint32_t)(chunk - small_chunks) + (uint32_t)unit * 7u) % (uint32_t)big_chunks));
    const int64_t block_row0 =
        small ? (int64_t)chunk * kRowsPerBlockStep
              : (int64_t)small_chunks * kRowsPerBlockStep + (int64_t)big_id * big_steps * kRowsPerBlockStep;
    const int steps = small ? 1 : big_steps;

    if (block_row0 >= n_rows) return;  // the grid is laid out for n_cap rows

    const uint8_t *Cu = C + b * cb + h * ch + (grp * S + side) * 16;
    UnitState *st = state + unit;
    const int last = n_rows - 1;
    uint32_t tb = DENSE ? (uint32_t)DC_HIST_BINS : load_relaxed(&st->tb_run);
    uint16_t *du = reinterpret_cast<uint16_t *>(surv) + (int64_t)unit * dense_stride(n_cap);

    // Double buffering: the loads of the next step are issued before the current step is
    // worked on, so a wave always has a step's worth of bytes in flight.  The loads are
    // unconditional (past the block's end they repeat its last row), which lets the
    // compiler wait for exactly the older buffer instead of for every load in flight.
    const int64_t blk_end = block_row0 + (int64_t)steps * kRowsPerBlockStep - 1;
    const int64_t blk_last = blk_end < (int64_t)last ? blk_end : (int64_t)last;
    auto load_step = [&](int step, uint4 (&cv)[kLoads]) __attribute__((always_inline)) {
        const int64_t row0 = block_row0 + (int64_t)step * kRowsPerBlockStep + wave * 64;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            int64_t r = row0 + t * (16 / S) + (lane & 15) / S;
            r = r > blk_last ? blk_last : r;
            const uint8_t *p = Cu + r * cr;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) cv[t * KS + ks] = dc_load_stream16(p + ks * (64 * S));
        }
    };

    // the first rows are under way while the weights are worked out
    uint4 ca[kLoads], cb2[kLoads];
    load_step(0, ca);
    for (int i = tid; i < DC_HIST_BINS; i += kThreads) lhist[i] = 0;

    // The weights q_d * a_d as whole multiples of 2^w_exp, |multiple| < 2^30, in four signed digits
    // of base 256, and the margin.  Every wave works them out for itself and leaves one digit
    // in LDS for all.
    int w_exp;
    float margin, poison;
    {
        const int col = lane % LPQ;
        const float4 *ap = reinterpret_cast<const float4 *>(scale + (int64_t)unit * HD + col * 8);
        const float4 *rp = reinterpret_cast<const float4 *>(resid + (int64_t)unit * HD + col * 8);
        const float4 as[2] = {ap[0], ap[1]}, rs[2] = {rp[0], rp[1]};  // requested with the query, not behind it
        float qv[8];
        dc_load_query<HD>(Q, unit, q_group, col, qv);
        float w[8];
        float wabs = 0.f, wmax = 0.f, e = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float av[4] = {as[i].x, as[i].y, as[i].z, as[i].w}, rv[4] = {rs[i].x, rs[i].y, rs[i].z, rs[i].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float ww = qv[4 * i + j] * av[j];
                w[4 * i + j] = ww;
                wabs += fabsf(ww);
                wmax = fmaxf(wmax, fabsf(ww));
                e += fabsf(qv[4 * i + j]) * rv[j];
            }
        }
        wabs = dc_group_sum<LPQ>(wabs);
        e = dc_group_sum<LPQ>(e);
        wmax = group_max<LPQ>(wmax);
        margin = dc_sketch_margin(e, wabs, mode);
        // Weights or a margin that are not finite (an infinite residual; no number where the query is zero there) bound no row: all are kept,
        // their approximation being no number of positive sign, whose bucket is the best, whatever the margin's sign or an
        // approximation that overflows would make of their sum.
        const bool bound = wabs < __builtin_inff() && margin < __builtin_inff();
        poison = bound ? 0.f : __uint_as_float(0x7fc00000u);
        margin = bound ? margin : 0.f;
        w_exp = __builtin_amdgcn_frexp_expf(wmax) - 30;
        uint32_t dig[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)  // one digit per byte: carries out of the lower three are settled by the addition
            dig[i] = (((uint32_t)(int)rintf(__builtin_amdgcn_ldexpf(w[i], -w_exp)) + 0x00808080u) ^ 0x00808080u) >> (8 * wave);
        if (lane < LPQ) {
            uint2 pk;
            pk.x = (dig[0] & 0xffu) | ((dig[1] & 0xffu) << 8) | ((dig[2] & 0xffu) << 16) | (dig[3] << 24);
            pk.y = (dig[4] & 0xffu) | ((dig[5] & 0xffu) << 8) | ((dig[6] & 0xffu) << 16) | (dig[7] << 24);
            *reinterpret_cast<uint2 *>(&s_w[wave][col * 8]) = pk;
        }
    }
    if (chunk == 0 && tid == 0) st->margin = __float_as_uint(margin);
    if (tid == 0) s_tb = tb;
    __syncthreads();
    // The left operands: row m of 16 is digit m % 4 of the weights of one S-th of the columns, or zero.
    // S = 1: block t of four rows for tile t.  S = 2: rows 0-7 for even tiles and 8-15 for odd ones, a
    // block for the columns of even lanes and one for those of odd lanes, in this order or the other.
    constexpr int kOps = 4;
    i32x4 wd[kOps][KS];
    {
        const int m = lane & 15, blk = m >> 2;
#pragma unroll
        for (int o = 0; o < kOps; ++o) {
            const int part = S == 1 ? 0 : (blk & 1) ^ (o >> 1);
            const bool on = S == 1 ? blk == o : (blk >> 1) == (o & 1);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const i32x4 v = *reinterpret_cast<const i32x4 *>(&s_w[m & 3][ks * (64 * S) + (grp * S + part) * 16]);
                wd[o][ks] = on ? v : i32x4{0, 0, 0, 0};
            }
        }
    }

    uint32_t *wstage = stage + wave * (kBigSteps * 64);
    uint32_t wcnt = 0, marginal = 0;
    const unsigned long long lt = (1ull << lane) - 1ull;

    // COUNT: also count the rows kept although their own bucket is not better than the
    // threshold's (ties and near-ties); only the first two steps of a wave do.
    auto work_step = [&](int step, const uint4 (&cv)[kLoads], auto count) __attribute__((always_inline)) {
        const int64_t row0 = block_row0 + (int64_t)step * kRowsPerBlockStep + wave * 64;
        // Register i of a lane receives the sum of digit i for its column; tiles whose operands differ share an accumulator.
        constexpr int NACC = S == 1 ? 1 : 4;
        i32x4 ds[NACC];
#pragma unroll
        for (int d = 0; d < NACC; ++d) ds[d] = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            const int d = S == 1 ? 0 : t >> 1, o = S == 1 ? t : 2 * ((t >> 1) & 1) + (t & 1);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uint4 c = cv[t * KS + ks];
                const i32x4 cs = {(int)(c.x ^ 0x80808080u), (int)(c.y ^ 0x80808080u), (int)(c.z ^ 0x80808080u),
                                  (int)(c.w ^ 0x80808080u)};
                ds[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wd[o][ks], cs, ds[d], 0, 0, 0);
            }
        }
        auto value = [&](const i32x4 &v) __attribute__((always_inline)) {
            return fmaf(fmaf(fmaf((float)v[3], 256.f, (float)v[2]), 256.f, (float)v[1]), 256.f, (float)v[0]);
        };
        float mine;
        if constexpr (S == 1) {
            mine = value(ds[0]);
        } else {
            // two halves of two rows, whose other halves are in lane ^ 17: keep one row, hand over the other
            const float v0 = value(par ? ds[1] : ds[0]), v1 = value(par ? ds[3] : ds[2]);
            const int give = __float_as_int(side ? v0 : v1);
            mine = (side ? v1 : v0) + __int_as_float(__builtin_amdgcn_ds_swizzle(give, (17 << 10) | 0x1f));
        }
        mine = __builtin_amdgcn_ldexpf(mine, w_exp) + poison;
        const int64_t myrow = row0 + own_row;
        const bool valid = myrow < n_rows;
        const uint32_t lb = dc_score_bucket(mine), kb = dc_score_bucket(mine + margin);
        if constexpr (DENSE) {
            if (valid) {
                du[myrow] = (uint16_t)kb;
                atomicAdd(&lhist[lb], 1u);
            }
            return;
        }
        const bool keep = valid && kb <= tb;
        if (keep) atomicAdd(&lhist[lb], 1u);
        const unsigned long long mask = __ballot(keep);
        if (keep) wstage[wcnt + __popcll(mask & lt)] = sketch_entry(kb, (uint32_t)myrow);
        wcnt += (uint32_t)__popcll(mask);
        if (decltype(count)::value) marginal += (uint32_t)__popcll(__ballot(keep && lb >= tb));
    };
    // steps of this wave that hold rows (wave-uniform)
    int my_steps = 0;
    {
        const int64_t first = block_row0 + wave * 64;
        if (first < n_rows) {
            const int64_t left = (int64_t)n_rows - first;
            my_steps = (int)((left + kRowsPerBlockStep - 1) / kRowsPerBlockStep);
            my_steps = my_steps < steps ? my_steps : steps;
        }
    }
    bool bulk = false;
    const bool had_tb = tb < (uint32_t)DC_HIST_BINS;  // the first steps are judged against a real threshold
    // The threshold poll is issued before the prefetch: loads return in order, so waiting
    // for a poll that was issued last would also wait for the whole prefetch.
    int step = 0;
    // With few units the whole chip polls a handful of lines, and every poll holds back
    // the younger loads of its wave (the poll is an agent-scope load): then only wave 0
    // polls and passes the value on through LDS.  With many units every wave polls for
    // itself, which keeps its threshold one step fresher.
    // (SHARED_POLL is a template parameter: as a run-time choice it costs registers.)
    if constexpr (DENSE) {
        for (; step + 1 < my_steps; step += 2) {
            load_step(step + 1, cb2);
            work_step(step, ca, std::false_type{});
            load_step(step + 2, ca);
            work_step(step + 1, cb2, std::false_type{});
        }
        if (step < my_steps) work_step(step, ca, std::false_type{});
        __syncthreads();
        uint32_t *hu = hist + (int64_t)unit * DC_HIST_BINS;
        for (int i = tid; i < DC_HIST_BINS; i += kThreads) {
            const uint32_t c = lhist[i];
            if (c) atomicAdd(&hu[i], c);
        }
        return;
    }
    auto two_steps = [&](auto count) __attribute__((always_inline)) {
        uint32_t tb_next = tb;
        if (!SHARED_POLL || wave == 0) tb_next = load_relaxed(&st->tb_run);
        load_step(step + 1, cb2);
        work_step(step, ca, count);
        if (SHARED_POLL) {
            if (wave == 0 && lane == 0) lds_store_relaxed(&s_tb, tb_next);
            tb = lds_load_relaxed(&s_tb);
        } else {
            tb = tb_next;
        }
        if (!SHARED_POLL || wave == 0) tb_next = load_relaxed(&st->tb_run);
        load_step(step + 2, ca);
        work_step(step + 1, cb2, count);
        if (SHARED_POLL) {
            if (wave == 0 && lane == 0) lds_store_relaxed(&s_tb, tb_next);
            tb = lds_load_relaxed(&s_tb);
        } else {
            tb = tb_next;
        }
        step += 2;
    };
    if (my_steps >= 2) {
        two_steps(std::true_type{});
        // Degenerate data (rows that nearly all tie with the k-th best: the sketch prunes nothing):
        // a wave that kept three quarters of the rows of its first two steps without any of them
        // being better than the threshold stops reading codes and keeps the rest of its rows unseen.
        // An unseen row carries the best possible approximation, so the exact rescoring takes it
        // in any case, and it is left out of the histogram, which only loosens the threshold: the
        // selected ids are the same, the scan costs a quarter.
        bulk = had_tb && marginal >= kBulkKeep;
    }
    while (!bulk && step + 1 < my_steps) two_steps(std::false_type{});
    if (bulk) {
        for (; step < my_steps; ++step) {
            const int64_t myrow = block_row0 + (int64_t)step * kRowsPerBlockStep + wave * 64 + lane;
            const bool keep = myrow < n_rows;
            const unsigned long long mask = __ballot(keep);
            if (keep) wstage[wcnt + __popcll(mask & lt)] = sketch_entry(0u, (uint32_t)myrow);  // passes any threshold
            wcnt += (uint32_t)__popcll(mask);
        }
    } else if (step < my_steps) {
        work_step(step, ca, std::false_type{});  // an odd last step; its rows are already on the way
    }
    const bool refresh = small ? (chunk & 3) == 3 : ((chunk - small_chunks) & 7) == 7;
    prune_block_finish<uint32_t>(lhist, wstage, wcnt, s_wcnt, &s_base, wtot, st,
                                           hist + (int64_t)unit * DC_HIST_BINS,
                                           reinterpret_cast<uint32_t *>(surv) + (int64_t)unit * n_cap, refresh,
                                           (uint32_t)k_eff);
}

// The scan of the PQ baseline: a key's score is its ADC score (dc_pq.h), read from M code bytes per key, in DC_MODE_IP
// order.  One key per lane.  A block stages its unit's tables once and scans an equal share of the unit's keys; like the
// dense sketch scan it leaves every key's bucket at the key's own place, and the histogram.  Nothing is polled, listed
// or handed over before the block's end.
//
// Bound by instruction issue and HBM together (some 118 vector instructions per 64 keys, 32 of them the additions, 32 the
// addresses of the tables; 268 MB of codes in 46 us = 5.8 TB/s).  8 x 1048576 codes of 32 bytes: 46 us.  Listed, in blocks of
// 4096 keys, half of a block's life went into staging the tables and closing (76 us; 70 with the wide tables, sixteen
// waves per block).  One block of 1024 threads per CU: two 46.2, four 51; three steps of codes ahead 48.9, one 47.6;
// blocks of 512 threads 46.1, two of them 51.5.
constexpr int kPqBlocks = 256;

template <int M>
__global__ __launch_bounds__(kPqThreads, 4) void pq_scan_kernel(
    const uint8_t *__restrict__ codes, const float *__restrict__ lut, uint32_t *__restrict__ hist,
    uint2 *__restrict__ surv, int n_units, int n_rows, int steps) {
    constexpr int NW = M / 4;
    __shared__ float s_lut[kPqWideWords];
    __shared__ uint32_t lhist[DC_HIST_BINS];
    const int unit = blockIdx.x % n_units;
    const int chunk = blockIdx.x / n_units;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t block_row0 = (int64_t)chunk * steps * kPqThreads;
    const int64_t blk_end = block_row0 + (int64_t)steps * kPqThreads - 1;
    const int64_t blk_last = blk_end < (int64_t)n_rows - 1 ? blk_end : (int64_t)n_rows - 1;
    if (block_row0 >= n_rows) return;
    const uint8_t *cu = codes + (int64_t)unit * n_rows * M;
    uint16_t *du = reinterpret_cast<uint16_t *>(surv) + (int64_t)unit * dense_stride(n_rows);
    // rows are a multiple of 64 from the start of the unit: lane = key mod 64, as pq_adc_score expects
    auto load_row = [&](int64_t row0, uint32_t(&w)[NW]) __attribute__((always_inline)) {
        int64_t r = row0 + lane;
        r = r > blk_last ? blk_last : r;
        // plain loads: the two halves of a 32-byte row come from the same cache line
        const uint4 *cp = reinterpret_cast<const uint4 *>(cu + r * M);
#pragma unroll
        for (int i = 0; i < NW / 4; ++i) {
            const uint4 t = cp[i];
            w[4 * i + 0] = t.x;
            w[4 * i + 1] = t.y;
            w[4 * i + 2] = t.z;
            w[4 * i + 3] = t.w;
        }
    };
    // The codes of kAhead steps are in flight beyond the one that is scored; requests past the
    // block's end repeat its last row, so that their number is the same on every path.
    constexpr int kAhead = 2, kRing = kAhead + 1;
    uint32_t buf[kRing][NW];
    const int64_t wave_row0 = block_row0 + wave * 64;
    const int64_t rows_left = blk_last + 1 - wave_row0;
    const int my_steps = rows_left <= 0 ? 0 : (int)((rows_left + kPqThreads - 1) / kPqThreads);
#pragma unroll
    for (int j = 0; j < kAhead; ++j) load_row(wave_row0 + (int64_t)j * kPqThreads, buf[j]);
    for (int i = tid; i < DC_HIST_BINS; i += kPqThreads) lhist[i] = 0;
    pq_stage_lut_wide<M>(s_lut, lut + (int64_t)unit * M * 256, tid, kPqThreads);
    PqWideLane<M> ln;
    ln.init(lane);
    __syncthreads();
    for (int s0 = 0; s0 < my_steps; s0 += kRing) {
#pragma unroll
        for (int j = 0; j < kRing; ++j) {
            const int step = s0 + j;
            const int64_t row0 = wave_row0 + (int64_t)step * kPqThreads;
            load_row(row0 + (int64_t)kAhead * kPqThreads, buf[(j + kAhead) % kRing]);
            if (step < my_steps) {  // wave-uniform
                const float mine = pq_adc_score_wide<M>(buf[j], s_lut, ln);
                uint32_t key, bucket;
                dc_key_bucket(mine, DC_MODE_IP, key, bucket);
                if (row0 + lane <= blk_last) {
                    du[row0 + lane] = (uint16_t)bucket;
                    atomicAdd(&lhist[bucket], 1u);
                }
            }
        }
    }
    __syncthreads();
    uint32_t *hu = hist + (int64_t)unit * DC_HIST_BINS;
    for (int i = tid; i < DC_HIST_BINS; i += kPqThreads) {
        const uint32_t c = lhist[i];
        if (c) atomicAdd(&hu[i], c);
    }
}

// classify_kernel for the buckets that pq_scan_kernel left: keys in buckets better than the threshold bucket are certain
// members, keys in it become candidates, whose scores are worked out once more (the additions of pq_adc_score).  A block
// takes ROWS keys (pq_class_rows) and reserves its places in both lists with one returning atomic.  Few candidates are scored
// from the tables in memory, a chain of 3 us per 256 of them.  More are many of a block's keys (short units of which much is
// selected, keys that tie), and the block stages the tables and walks its keys in order as the scan does: 3 units x 5000 keys,
// 4096 of them selected, 6.6 us (12 from memory, in blocks of 8192); 5000 keys that tie 7.6 (65), 3 x 65000 11 (70).
static_assert(offsetof(UnitState, cand_cnt) == offsetof(UnitState, win_cnt) + 4 && offsetof(UnitState, win_cnt) % 8 == 0, "one word");

template <int M, int ROWS>
__global__ __launch_bounds__(kThreads) void pq_classify_kernel(
    const uint8_t *__restrict__ codes, const float *__restrict__ lut, const uint32_t *__restrict__ hist,
    UnitState *__restrict__ state, const uint2 *__restrict__ surv, uint32_t *__restrict__ cand_key,
    uint32_t *__restrict__ cand_idx, uint32_t *__restrict__ idx_out, int64_t idx_stride, int n_units, int n_rows, int k_eff) {
    constexpr int kVec = ROWS / kThreads / 8;  // vectors of eight buckets per thread
    constexpr int NW = M / 4;
    static_assert(kVec * 8 * kThreads == ROWS && ROWS % 64 == 0 && 4 * ROWS <= 4 * kPqLutWords, "whole vectors; both lists in the tables' place");
    __shared__ __align__(16) float s_lut[kPqLutWords];  // of blocks with many candidates; the lists before
    uint16_t *s_sure = reinterpret_cast<uint16_t *>(s_lut), *s_cand = s_sure + ROWS;
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t sres[2];
    __shared__ uint32_t sbase[2];
    const int unit = blockIdx.x % n_units, blk = blockIdx.x / n_units;
    const int tid = threadIdx.x;
    const int row0 = blk * ROWS;
    UnitState *st = state + unit;
    const uint16_t *du = reinterpret_cast<const uint16_t *>(surv) + (int64_t)unit * dense_stride(n_rows);
    uint4 v[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const int64_t r = (int64_t)row0 + (i * kThreads + tid) * 8;
        v[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
        if (r < n_rows) v[i] = *reinterpret_cast<const uint4 *>(du + r);
    }
    const uint32_t kk = (uint32_t)k_eff;
    uint32_t tb, c_less;
    unit_threshold(hist + (int64_t)unit * DC_HIST_BINS, kk, wtot, sres, tb, c_less);
    if (blk == 0 && tid == 0) st->c_less = c_less;
    uint32_t sure = 0, cand = 0;  // a bit per key
    static_assert(kVec * 8 <= 32, "bits of a thread's keys");
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const uint32_t w4[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t bucket = j & 1 ? w4[j / 2] >> 16 : w4[j / 2] & 0xffffu;
            const bool live = row0 + (i * kThreads + tid) * 8 + j < n_rows;
            sure |= live && bucket < tb ? 1u << (8 * i + j) : 0u;
            cand |= live && bucket == tb ? 1u << (8 * i + j) : 0u;
        }
    }
    uint32_t tot;
    const uint32_t ex = block_excl_scan<kThreads>(__popc(sure) | __popc(cand) << 16, wtot, &tot);
    const uint32_t n_sure = tot & 0xffffu, n_cand = tot >> 16;
    // (both lists with one addition: their cursors are the halves of one word, additions to which are served one after
    // the other, 128 of them per unit at a million keys)
    if (tid == 0) {
        unsigned long long at = 0ull;
        if (tot) at = atomicAdd(reinterpret_cast<unsigned long long *>(&st->win_cnt), (unsigned long long)n_cand << 32 | n_sure);
        sbase[0] = (uint32_t)at;
        sbase[1] = (uint32_t)(at >> 32);
    }
    auto list = [&](uint32_t bits, uint32_t at, uint16_t *dst) __attribute__((always_inline)) {
        while (bits) {
            const int b = __ffs(bits) - 1;
            bits &= bits - 1u;
            dst[at++] = (uint16_t)(((b >> 3) * kThreads + tid) * 8 + (b & 7));
        }
    };
    list(sure, ex & 0xffffu, s_sure);
    list(cand, ex >> 16, s_cand);
    __syncthreads();
    uint32_t *io = idx_out + (int64_t)unit * idx_stride;
    for (uint32_t i = tid; i < n_sure; i += kThreads) {
        const uint32_t at = sbase[0] + i;
        if (at < kk) io[at] = (uint32_t)row0 + s_sure[i];
    }
    const uint8_t *cu = codes + (int64_t)unit * n_rows * M;
    const float *lu = lut + (int64_t)unit * M * 256;
    uint32_t *ck = cand_key + (int64_t)unit * n_rows, *ci = cand_idx + (int64_t)unit * n_rows;
    auto load_codes = [&](uint32_t row, uint32_t (&w)[NW]) __attribute__((always_inline)) {
        const uint4 *cp = reinterpret_cast<const uint4 *>(cu + (int64_t)row * M);
#pragma unroll
        for (int x = 0; x < NW / 4; ++x) {
            const uint4 t = cp[x];
            w[4 * x] = t.x, w[4 * x + 1] = t.y, w[4 * x + 2] = t.z, w[4 * x + 3] = t.w;
        }
    };
    auto put = [&](uint32_t at, uint32_t row, float score) __attribute__((always_inline)) {
        uint32_t key, bucket;
        dc_key_bucket(score, DC_MODE_IP, key, bucket);
        if (at < (uint32_t)n_rows) {
            ck[at] = key;
            ci[at] = row;
        }
    };
    if (n_cand > (uint32_t)(ROWS / 8 + kThreads)) {
        __syncthreads();  // the lists are in the tables' place
        pq_stage_lut<M>(s_lut, lu, tid, kThreads);
        PqLane<M> ln;
        ln.init(tid & 63);
        __syncthreads();
        constexpr int kAtOnce = 4;
#pragma unroll 1
        for (int s0 = 0; s0 < ROWS && row0 + s0 < n_rows; s0 += kAtOnce * kThreads) {
            uint32_t w[kAtOnce][NW], bucket[kAtOnce];
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j) {
                const int row = row0 + s0 + j * kThreads + tid, r = row < n_rows ? row : n_rows - 1;
                bucket[j] = row < n_rows ? (uint32_t)du[r] : ~0u;
                load_codes((uint32_t)r, w[j]);
            }
#pragma unroll
            for (int j = 0; j < kAtOnce; ++j) {
                const bool in = bucket[j] == tb;
                if (__ballot(in) == 0ull) continue;
                const float score = pq_adc_score<M>(w[j], s_lut, ln);
                const uint32_t at = wave_reserve(in, &sbase[1]);
                if (in) put(at, (uint32_t)(row0 + s0 + j * kThreads + tid), score);
            }
        }
        return;
    }
    for (uint32_t i = tid; i < n_cand; i += kThreads) {
        const uint32_t row = (uint32_t)row0 + s_cand[i];
        uint32_t w[NW], rw[NW];
        load_codes(row, w);
        PqWideLane<M> ln;
        ln.init((int)(row & 63u));
        pq_rotate<M>(w, ln.rot, ln.sh, rw);
        float e[M], acc = 0.f;
#pragma unroll
        for (int j = 0; j < M; ++j) e[j] = lu[((row + j) % M) * 256 + ((rw[j / 4] >> (8 * (j % 4))) & 0xffu)];
#pragma unroll
        for (int j = 0; j < M; ++j) acc += e[j];
        put(sbase[1] + i, row, acc);
    }
}

// Several blocks per unit split the unit's survivor list: rows in buckets better
// than the threshold bucket are certain members and go straight to idx_out, rows
// in the threshold bucket become candidates.  Each block reserves its output
// ranges with one returning atomic per list.
constexpr int kClassifyBatch = 4;

__global__ __launch_bounds__(kThreads) void classify_kernel(
    const uint32_t *__restrict__ hist, UnitState *__restrict__ state, const uint2 *__restrict__ surv,
    uint32_t *__restrict__ cand_key, uint32_t *__restrict__ cand_idx, uint32_t *__restrict__ idx_out,
    int64_t idx_stride, uint32_t *__restrict__ sel_keys, int n_units, int n_rows, int k_eff, int mode,
    int nblk) {
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t sres[2];
    __shared__ uint32_t sbase[2];
    const int unit = blockIdx.x % n_units;
    const int blk = blockIdx.x / n_units;
    const int tid = threadIdx.x;
    UnitState *st = state + unit;
    const uint2 *su = surv + (int64_t)unit * n_rows;
    const uint32_t cap = (uint32_t)n_rows;
    uint32_t n_s = st->surv_cnt;
    if (n_s > cap) n_s = cap;
    // every block takes one contiguous slice of whole batches
    constexpr uint32_t kPer = kClassifyBatch * kThreads;
    const uint32_t per = ((n_s + (uint32_t)nblk - 1) / (uint32_t)nblk + kPer - 1) / kPer * kPer;
    const uint32_t lo = (uint32_t)blk * per;
    uint32_t hi = lo + per;
    if (hi > n_s) hi = n_s;
    if (lo >= n_s && blk != 0) return;

    const uint32_t kk = (uint32_t)k_eff;
    uint32_t tb, c_less;
    unit_threshold(hist + (int64_t)unit * DC_HIST_BINS, kk, wtot, sres, tb, c_less);
    if (blk == 0 && tid == 0) st->c_less = c_less;

    uint32_t *ck = cand_key + (int64_t)unit * n_rows;
    uint32_t *ci = cand_idx + (int64_t)unit * n_rows;
    uint32_t *io = idx_out + (int64_t)unit * idx_stride;
    uint32_t *ko = sel_keys ? sel_keys + (int64_t)unit * k_eff : nullptr;

    for (uint32_t i0 = lo; i0 < hi; i0 += kPer) {
        uint2 p[kClassifyBatch];
#pragma unroll
        for (int j = 0; j < kClassifyBatch; ++j) {
            const uint32_t i = i0 + j * kThreads + tid;
            p[j] = make_uint2(0u, 0u);
            if (i < hi) p[j] = su[i];
        }
        uint32_t keys[kClassifyBatch];
        uint32_t wmask = 0, cmask = 0;
#pragma unroll
        for (int j = 0; j < kClassifyBatch; ++j) {
            const uint32_t i = i0 + j * kThreads + tid;
            uint32_t key = 0, bucket = 0xffffffffu;
            if (i < hi) dc_key_bucket(__uint_as_float(p[j].y), mode, key, bucket);
            keys[j] = key;
            if (bucket < tb) wmask |= 1u << j;
            else if (bucket == tb) cmask |= 1u << j;
        }
        uint32_t tot;
        const uint32_t ex = block_excl_scan<kThreads>(__popc(wmask) | (__popc(cmask) << 16), wtot, &tot);
        if (tid == 0) {
            const uint32_t nw = tot & 0xffffu, nc = tot >> 16;
            sbase[0] = nw ? atomicAdd(&st->win_cnt, nw) : 0u;
            sbase[1] = nc ? atomicAdd(&st->cand_cnt, nc) : 0u;
        }
        __syncthreads();
        uint32_t wpos = sbase[0] + (ex & 0xffffu), cpos = sbase[1] + (ex >> 16);
#pragma unroll
        for (int j = 0; j < kClassifyBatch; ++j) {
            if (wmask & (1u << j)) {
                if (wpos < kk) {
                    io[wpos] = p[j].x;
                    if (ko) ko[wpos] = keys[j];
                }
                ++wpos;
            } else if (cmask & (1u << j)) {
                if (cpos < cap) {
                    ck[cpos] = keys[j];
                    ci[cpos] = p[j].x;
                }
                ++cpos;
            }
        }
        __syncthreads();  // sbase is rewritten by the next batch
    }
}

// classify_kernel for the keys that a dense score_prune_kernel left: a block takes kKeyClassRows rows and reserves its places
// in both lists with one returning atomic.  Bound by its chain: keys (6.4 MB at 32 units x 49933 rows) while the histogram is
// scanned, one atomic, the members' stores.
constexpr int kKeyClassRows = 4096;

__global__ __launch_bounds__(kThreads) void key_classify_kernel(
    const uint32_t *__restrict__ hist, UnitState *__restrict__ state, const uint2 *__restrict__ surv,
    uint32_t *__restrict__ cand_key, uint32_t *__restrict__ cand_idx, uint32_t *__restrict__ idx_out, int64_t idx_stride,
    uint32_t *__restrict__ sel_keys, int n_units, int n_rows, int k_eff, int mode) {
    constexpr int kVec = kKeyClassRows / kThreads / 4;
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t sres[2];
    __shared__ uint32_t sbase[2];
    const int unit = blockIdx.x % n_units, blk = blockIdx.x / n_units;
    const int tid = threadIdx.x;
    const int64_t row0 = (int64_t)blk * kKeyClassRows;
    UnitState *st = state + unit;
    const int64_t stride = dense_key_stride(n_rows);
    const uint32_t *du = reinterpret_cast<const uint32_t *>(surv) + (int64_t)unit * stride;
    uint32_t keys[4 * kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const int64_t r = row0 + (i * kThreads + tid) * 4;
        uint4 v = make_uint4(kNoRow, kNoRow, kNoRow, kNoRow);
        if (r < stride) v = *reinterpret_cast<const uint4 *>(du + r);
        keys[4 * i] = v.x, keys[4 * i + 1] = v.y, keys[4 * i + 2] = v.z, keys[4 * i + 3] = v.w;
    }
    const uint32_t kk = (uint32_t)k_eff;
    uint32_t tb, c_less;
    unit_threshold(hist + (int64_t)unit * DC_HIST_BINS, kk, wtot, sres, tb, c_less);
    if (blk == 0 && tid == 0) st->c_less = c_less;
    uint32_t sure = 0, cand = 0;  // a bit per row
#pragma unroll
    for (int j = 0; j < 4 * kVec; ++j) {
        const float x = __uint_as_float((keys[j] & 0x80000000u) ? keys[j] & 0x7fffffffu : ~keys[j]);  // dc_f2ord, inverted
        const uint32_t bucket = dc_score_bucket_flat(mode == DC_MODE_REF_DIST ? 65536.0f - x : -x);
        sure |= keys[j] != kNoRow && bucket < tb ? 1u << j : 0u;
        cand |= keys[j] != kNoRow && bucket == tb ? 1u << j : 0u;
    }
    uint32_t tot;
    const uint32_t ex = block_excl_scan<kThreads>(__popc(sure) | __popc(cand) << 16, wtot, &tot);
    if (tid == 0) {
        unsigned long long at = 0ull;
        if (tot) at = atomicAdd(reinterpret_cast<unsigned long long *>(&st->win_cnt), (unsigned long long)(tot >> 16) << 32 | (tot & 0xffffu));
        sbase[0] = (uint32_t)at;
        sbase[1] = (uint32_t)(at >> 32);
    }
    __syncthreads();
    uint32_t wpos = sbase[0] + (ex & 0xffffu), cpos = sbase[1] + (ex >> 16);
    uint32_t *ck = cand_key + (int64_t)unit * n_rows, *ci = cand_idx + (int64_t)unit * n_rows;
    uint32_t *io = idx_out + (int64_t)unit * idx_stride;
    uint32_t *ko = sel_keys ? sel_keys + (int64_t)unit * k_eff : nullptr;
#pragma unroll
    for (int j = 0; j < 4 * kVec; ++j) {
        const uint32_t row = (uint32_t)row0 + (uint32_t)(((j / 4) * kThreads + tid) * 4 + j % 4);
        if (sure >> j & 1u) {
            if (wpos < kk) {
                io[wpos] = row;
                if (ko) ko[wpos] = keys[j];
            }
            ++wpos;
        } else if (cand >> j & 1u) {
            if (cpos < (uint32_t)n_rows) {
                ck[cpos] = keys[j];
                ci[cpos] = row;
            }
            ++cpos;
        }
    }
}

// Second pass of the sketch path.  Several blocks per unit split the list the
// sketch scan left ((id, approx) pairs): a row stays a candidate when
// bucket(approx + margin) is not worse than the exact bucket of the k-th largest
// approx; candidates get their exact fp32 score from the bf16 row, computed lane for
// lane as score_kernel computes it, and their (key, id) go to the unit's candidate
// list, from which select_finish_kernel picks the k best (c_less = 0: the list
// holds every member of the top-k).
constexpr int kRescoreBatch = 4;

// PER > 0: the scan left a bucket for every row (sketch_prune_kernel); a block takes PER rows of a thread at a time, side
// by side, and the tiles of a unit are dealt to its blocks as they come (dense_per_thread).  PER == 0: the list.
template <int HD, int PER>
__global__ __launch_bounds__(kThreads) void rescore_kernel(
    const uint16_t *__restrict__ K, const uint16_t *__restrict__ Q, const uint32_t *__restrict__ hist,
    UnitState *__restrict__ state, const uint2 *__restrict__ surv, uint32_t *__restrict__ cand_key,
    uint32_t *__restrict__ cand_idx, int n_units, int n_h, int n_rows, int64_t sb, int64_t sh,
    int64_t sr, int q_group, int mode, int k_eff, int nblk, const int32_t *__restrict__ hi_dev, int lo_row) {
    constexpr int LPR = HD / 8;
    constexpr int GROUPS = kThreads / LPR;
    constexpr bool DENSE = PER > 0;
    if constexpr (DENSE)  // all arguments at once (in the scan, too); the pass over a list is 2 us slower with it
        asm volatile("" ::"s"(K), "s"(Q), "s"(hist), "s"(state), "s"(surv), "s"(cand_key), "s"(cand_idx), "s"(n_units), "s"(n_h), "s"(n_rows),
                     "s"(sb), "s"(sh), "s"(sr), "s"(q_group), "s"(mode), "s"(k_eff), "s"(nblk), "s"(hi_dev), "s"(lo_row));
    constexpr int kOwn = DENSE ? PER : kRescoreBatch;  // entries of a thread per batch
    constexpr uint32_t kPer = kOwn * kThreads;
    __shared__ uint32_t cid[kPer];
    __shared__ uint32_t ckey[kPer];
    __shared__ uint32_t wtot[kThreads / 64 + 1];
    __shared__ uint32_t sres[2];
    __shared__ uint32_t s_base;
    const int unit = blockIdx.x, blk = blockIdx.y;
    const int b = unit / n_h, h = unit % n_h;
    const int tid = threadIdx.x;
    const int grp = tid / LPR, col = tid % LPR;
    UnitState *st = state + unit;
    uint32_t opaque_zero = 0;
    asm volatile("" : "+v"(opaque_zero));
    // The list is dealt to the unit's blocks in tiles of kThreads entries, round robin:
    // the scan appends in the order its blocks finish, and the entries of late blocks
    // (tight threshold) pass the filter far more often than those of early ones, so
    // contiguous slices would leave a few blocks with most of the gathers.
    auto entry = [&](uint32_t t) { return ((uint32_t)blk + t * (uint32_t)nblk) * kThreads + (uint32_t)tid; };

    // The block's first batch of the list is requested before its length is known (what lies
    // beyond the length is stale and is masked below), together with the length, the histogram
    // and the query: one memory round trip for all of them.
    const uint32_t *su = reinterpret_cast<const uint32_t *>(surv) + (int64_t)unit * n_rows;
    const uint16_t *du = reinterpret_cast<const uint16_t *>(surv) + (int64_t)unit * dense_stride(n_rows);
    uint32_t p[4];
    auto load_dense = [&](uint32_t t) __attribute__((always_inline)) {
        const uint32_t i = (((uint32_t)blk + t * (uint32_t)nblk) * kThreads + (uint32_t)tid) * PER;
        p[0] = p[1] = p[2] = p[3] = ~0u;
        if (i >= (uint32_t)n_rows) return;
        if constexpr (PER == 8) {
            const uint4 v = *reinterpret_cast<const uint4 *>(du + i);
            p[0] = v.x, p[1] = v.y, p[2] = v.z, p[3] = v.w;
        } else if constexpr (PER == 4) {
            const uint2 v = *reinterpret_cast<const uint2 *>(du + i);
            p[0] = v.x, p[1] = v.y;
        } else {
            p[0] = *reinterpret_cast<const uint32_t *>(du + i);
        }
    };
    uint32_t n_s;
    UnitBins bins;
    if constexpr (DENSE) {
        load_dense(0u);
    } else {
#pragma unroll
        for (int j = 0; j < kRescoreBatch; ++j) {
            const uint32_t i = entry((uint32_t)j);
            p[j] = 0xffffffffu;
            if (i < (uint32_t)n_rows) p[j] = su[i];
        }
        n_s = st->surv_cnt;
    }
    bins.request(hist + (int64_t)unit * DC_HIST_BINS);
    __builtin_amdgcn_sched_barrier(0);  // (the query's sums are not worked out ahead of that)
    float q[8];
    dc_load_query<HD>(Q, unit, q_group, col, q);
    if constexpr (DENSE) n_s = (uint32_t)dc_live_rows(n_rows, hi_dev, lo_row);
    uint32_t tb, c_less;
    unit_threshold(bins, (uint32_t)k_eff, wtot, sres, tb, c_less);
    if (n_s > (uint32_t)n_rows) n_s = n_rows;
    constexpr uint32_t kTile = DENSE ? kPer : (uint32_t)kThreads;
    const uint32_t n_tiles = (n_s + kTile - 1) / kTile;
    if ((uint32_t)blk >= n_tiles) return;
    const uint32_t my_tiles = (n_tiles - (uint32_t)blk + (uint32_t)nblk - 1) / (uint32_t)nblk;
    if (blk == 0 && tid == 0) st->c_less = 0;
    const uint16_t *Ku = K + b * sb + h * sh + col * 8;
    uint32_t *ck = cand_key + (int64_t)unit * n_rows;
    uint32_t *ci = cand_idx + (int64_t)unit * n_rows;

    for (uint32_t t0 = 0; t0 < my_tiles; t0 += DENSE ? 1 : kRescoreBatch) {
        uint32_t pass = 0;
        const uint32_t row0 = (((uint32_t)blk + t0 * (uint32_t)nblk) * kThreads + (uint32_t)tid) * PER;  // DENSE
        if constexpr (DENSE) {
            if (t0 != 0) load_dense(t0);
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const uint32_t kb = j & 1 ? p[j / 2] >> 16 : p[j / 2] & 0xffffu;
                if (row0 + j < n_s && kb <= tb) pass |= 1u << j;
            }
        } else {
#pragma unroll
            for (int j = 0; j < kRescoreBatch; ++j) {
                const uint32_t t = t0 + (uint32_t)j;
                const uint32_t i = entry(t);
                const bool in = t < my_tiles && i < n_s;
                if (t0 != 0) {
                    p[j] = 0xffffffffu;
                    if (in) p[j] = su[i];
                }
                if (in && (p[j] >> kSketchRowBits) <= tb) pass |= 1u << j;
            }
        }
        uint32_t n_c;
        uint32_t pos = block_excl_scan<kThreads>(__popc(pass), wtot, &n_c);
#pragma unroll
        for (int j = 0; j < kOwn; ++j)
            if (pass & (1u << j)) cid[pos++] = DENSE ? row0 + j : p[j] & (uint32_t)(kSketchMaxRows - 1);
        // The list slot is reserved now and looked at after the rows are scored.  (Through an address
        // the compiler cannot prove uniform: it turns an atomic on a uniform address into one atomic
        // per wave plus a broadcast of the result and waits for that on the spot, a memory round
        // trip in front of the barrier below and of every row request behind it.)
        uint32_t base_reg = 0;
        if (tid == 0 && n_c) base_reg = atomicAdd(&st->cand_cnt + opaque_zero, n_c);
        __syncthreads();
        // exact scores: one LPR-lane group per row, kRowsInFlight rows of a group in flight
        constexpr int kRowsInFlight = 8;
        for (uint32_t j0 = 0; j0 < n_c; j0 += GROUPS * kRowsInFlight) {
            uint4 wv[kRowsInFlight];
#pragma unroll
            for (int u = 0; u < kRowsInFlight; ++u) {
                uint32_t j = j0 + u * GROUPS + grp;
                j = j < n_c ? j : n_c - 1;
                wv[u] = *reinterpret_cast<const uint4 *>(Ku + (int64_t)cid[j] * sr);
            }
#pragma unroll
            for (int u = 0; u < kRowsInFlight; ++u) {
                const uint32_t j = j0 + u * GROUPS + grp;
                const float sc = dc_group_sum<LPR>(dc_dot8(wv[u], q, 0.f));
                if (col == 0 && j < n_c) {
                    uint32_t key, bucket;
                    dc_key_bucket(sc, mode, key, bucket);
                    ckey[j] = key;
                }
            }
        }
        if (tid == 0) s_base = base_reg;
        __syncthreads();
        for (uint32_t i = tid; i < n_c; i += kThreads) {
            const uint32_t slot = s_base + i;
            if (slot < (uint32_t)n_rows) {
                ck[slot] = ckey[i];
                ci[slot] = cid[i];
            }
        }
        __syncthreads();  // cid, ckey and s_base are rewritten by the next batch
    }
}

// Exact scores of the rows the PQ scan selected: one LPR-lane group per row, the
// arithmetic of score_gathered_kernel.  Their (key, id) become the unit's candidate
// list, from which select_finish_kernel picks the best (c_less = 0).
template <int HD>
__global__ __launch_bounds__(kThreads) void pq_rescore_kernel(
    const uint16_t *__restrict__ K, const uint16_t *__restrict__ Q, const uint32_t *__restrict__ idx,
    UnitState *__restrict__ state, uint32_t *__restrict__ cand_key, uint32_t *__restrict__ cand_idx,
    int n_h, int n_idx, int64_t idx_stride, int n_rows, int64_t sb, int64_t sh, int64_t sr,
    int blocks_per_unit) {
    constexpr int LPR = HD / 8;
    constexpr int GROUPS = kThreads / LPR;
    const int unit = blockIdx.x / blocks_per_unit;
    const int chunk = blockIdx.x % blocks_per_unit;
    const int b = unit / n_h, h = unit % n_h;
    const int grp = threadIdx.x / LPR, col = threadIdx.x % LPR;
    if (chunk == 0 && threadIdx.x == 0) {
        state[unit].cand_cnt = (uint32_t)n_idx;
        state[unit].c_less = 0;
    }
    float q[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = dc_bf16_to_f32(Q[(int64_t)unit * HD + col * 8 + i]);
    const int j = chunk * GROUPS + grp;
    const int jj = j < n_idx ? j : n_idx - 1;
    const uint32_t id = idx[(int64_t)unit * idx_stride + jj];
    const uint4 w = *reinterpret_cast<const uint4 *>(K + b * sb + h * sh + (int64_t)id * sr + col * 8);
    const float p = dc_group_sum<LPR>(dc_dot8(w, q, 0.f));
    if (j < n_idx && col == 0) {
        uint32_t key, bucket;
        dc_key_bucket(p, DC_MODE_IP, key, bucket);
        cand_key[(int64_t)unit * n_rows + j] = key;
        cand_idx[(int64_t)unit * n_rows + j] = id;
    }
}

// One block per unit: a selection among the candidates of the threshold bucket
// fills idx_out[c_less, k).  Leaves the unit's list cursors at zero.  A chain of block barriers on few CUs.  Lists of up to
// kFinishRegs entries stay in registers, requested whole before their length is known: one counting pass over the
// highest 11 bits in which the keys differ hands out the slots (as dc_select_counted does), with six barriers: 5.3 us at 8
// units and 6.6 at 64 (2048 of about 3600 candidates), 5.9 and 7.3 with the list staged in LDS and eight barriers.
// (Counting a threshold bin of more than 96 once more instead of ranking it: no faster where it applies, 0.3 us slower else.)
// A radix pass whose members reserve slots wave by wave took 7.5 and 8.8 us.  Longer lists take dc_select_counted as long as they fit
// the LDS; lists that do not, and threshold bins of more than kFinalThreads (ties by the
// thousand), take the radix passes of dc_finalize_unit.  Keys that are all equal are not counted first (one bin: 8 units x
// 8000 rows that tie, a whole selection, 34 us with the count, 31 without).
constexpr int kFinishPer = 8, kFinishRegs = kFinishPer * kFinalThreads;

__global__ __launch_bounds__(kFinalThreads) void select_finish_kernel(
    uint32_t *__restrict__ hist, UnitState *__restrict__ state, uint32_t *__restrict__ cand_key,
    uint32_t *__restrict__ cand_idx, uint32_t *__restrict__ idx_out, int64_t idx_stride,
    uint32_t *__restrict__ sel_keys, int n_rows, int k_eff, int reinit) {
    asm volatile("" ::"s"(hist), "s"(state), "s"(cand_key), "s"(cand_idx), "s"(idx_out), "s"(idx_stride), "s"(sel_keys), "s"(n_rows), "s"(k_eff),
                 "s"(reinit));  // all arguments at once
    __shared__ uint32_t lh[kRadixBins];
    __shared__ uint32_t wtot[kFinalThreads / 64 + 1];
    __shared__ uint32_t sres[4];
    __shared__ uint32_t smisc[2];
    __shared__ uint32_t s_or[kFinalThreads / 64];
    __shared__ __align__(16) uint32_t s_list[2 * kCandLds];  // longer lists are staged in LDS when they fit
    uint32_t *const lck = s_list, *const lci = s_list + kCandLds;
    static_assert(kRadixCopies * kRadixBins <= 2 * kCandLds, "the counts of lists that do not fit take their place");
    __shared__ unsigned long long tie[kFinalThreads];
    const int unit = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    UnitState *st = state + unit;
    uint32_t *ck = cand_key + (int64_t)unit * n_rows;
    uint32_t *ci = cand_idx + (int64_t)unit * n_rows;
    // the list is fetched before its length is known: one memory round trip less
    uint32_t hk[kFinishPer], hi[kFinishPer];
#pragma unroll
    for (int j = 0; j < kFinishPer; ++j) {
        const int i = tid + j * kFinalThreads;
        hk[j] = hi[j] = 0;
        if (i < n_rows) {
            hk[j] = ck[i];
            hi[j] = ci[i];
        }
    }
    const uint32_t k0 = ck[0];
    uint32_t n_c = st->cand_cnt;
    const uint32_t c_less = st->c_less;
    reinterpret_cast<uint2 *>(lh)[tid] = make_uint2(0u, 0u);
    if (n_c > (uint32_t)n_rows) n_c = n_rows;
    const uint32_t kk = (uint32_t)k_eff;
    uint32_t *io = idx_out + (int64_t)unit * idx_stride;
    uint32_t *ko = sel_keys ? sel_keys + (int64_t)unit * k_eff : nullptr;
    const bool regs = n_c <= (uint32_t)kFinishRegs, staged = !regs && n_c <= (uint32_t)kCandLds;
    if (regs) {
        uint32_t diff = 0u;
#pragma unroll
        for (int j = 0; j < kFinishPer; ++j)
            if (j * kFinalThreads < (int)n_c) diff |= (uint32_t)(tid + j * kFinalThreads) < n_c ? hk[j] ^ k0 : 0u;
        diff = wave_or(diff);
        if (lane == 63) s_or[wave] = diff;
    } else if (staged) {
#pragma unroll
        for (int j = 0; j < kFinishPer; ++j) {
            lck[tid + j * kFinalThreads] = hk[j];
            lci[tid + j * kFinalThreads] = hi[j];
        }
        for (uint32_t i = tid + kFinishRegs; i < n_c; i += kFinalThreads) {
            lck[i] = ck[i];
            lci[i] = ci[i];
        }
    }
    __syncthreads();  // every thread has read the counters
    if (reinit) {
        // leave the unit's histogram and threshold ready for the next scan
        uint4 *hz = reinterpret_cast<uint4 *>(hist + (int64_t)unit * DC_HIST_BINS);
        if (tid < DC_HIST_BINS / 4) hz[tid] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (tid == 0) {
        if (reinit) {
            st->tb_run = DC_HIST_BINS;
            st->surv_cnt = 0;
        }
        st->win_cnt = 0;
        st->cand_cnt = 0;
    }
    if (c_less >= kk) return;
    uint32_t need = kk - c_less;
    if (need > n_c) need = n_c;
    auto put = [&](uint32_t slot, uint32_t key, uint32_t id) __attribute__((always_inline)) {
        io[c_less + slot] = id;
        if (ko) ko[c_less + slot] = key;
    };
    if (regs) {
        auto each = [&](auto fn) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < kFinishPer; ++j)
                if (j * kFinalThreads < (int)n_c && (uint32_t)(tid + j * kFinalThreads) < n_c)
                    fn((uint32_t)(tid + j * kFinalThreads), hk[j], hi[j]);
        };
        if (need == n_c) {  // all of them
            each(put);
            return;
        }
        uint32_t diff = 0u;
#pragma unroll
        for (int w = 0; w < kFinalThreads / 64; ++w) diff |= s_or[w];
        if (diff != 0u || n_c <= (uint32_t)kFinalThreads) {  // (equal keys are one bin)
            const int top = diff ? 32 - __clz((int)diff) : 0;
            const int shift = top > kRadixBits ? top - kRadixBits : 0;
            const uint32_t mask = diff ? (uint32_t)kRadixBins - 1u : 0u;  // the bits above are the same in every key
            each([&](uint32_t, uint32_t key, uint32_t) __attribute__((always_inline)) { atomicAdd(&lh[(key >> shift) & mask], 1u); });
            __syncthreads();
            const uint2 h2 = reinterpret_cast<const uint2 *>(lh)[tid];
            uint32_t total;
            const uint32_t excl = block_excl_scan<kFinalThreads>(h2.x + h2.y, wtot, &total);
            reinterpret_cast<uint2 *>(lh)[tid] = make_uint2(excl, excl + h2.x);
            if (excl < need && need <= excl + h2.x + h2.y) {
                const bool first = excl + h2.x >= need;
                sres[0] = 2 * tid + (first ? 0 : 1);
                sres[1] = first ? excl : excl + h2.x;
                sres[2] = first ? h2.x : h2.y;
            }
            __syncthreads();
            const uint32_t t_bin = sres[0], t_lo = sres[1], t_cnt = sres[2];
            if (t_cnt <= (uint32_t)kFinalThreads) {
                each([&](uint32_t, uint32_t key, uint32_t id) __attribute__((always_inline)) {
                    const uint32_t bin = (key >> shift) & mask;
                    if (bin > t_bin) return;
                    const uint32_t slot = atomicAdd(&lh[bin], 1u);
                    if (bin == t_bin) tie[slot - t_lo] = ((unsigned long long)key << 32) | id;
                    else put(slot, key, id);
                });
                __syncthreads();
                if ((uint32_t)tid < t_cnt) {
                    const unsigned long long mine = tie[tid];
                    uint32_t rank = t_lo;
                    for (uint32_t j = 0; j < t_cnt; ++j) rank += tie[j] < mine ? 1u : 0u;
                    if (rank < need) put(rank, (uint32_t)(mine >> 32), (uint32_t)mine);
                }
                return;
            }
        }
        // keys that crowd into one bin: from LDS like a longer list
        each([&](uint32_t i, uint32_t key, uint32_t id) __attribute__((always_inline)) { lck[i] = key, lci[i] = id; });
    }
    if (staged && dc_select_counted<false>(lck, lci, n_c, need, tie, lh, wtot, sres, smisc, put)) return;
    __syncthreads();
    // Two calls, so that the staged list is read with LDS instructions: through a pointer chosen
    // at run time every access would be a flat one, and waiting for a flat load also waits for
    // the stores issued above.
    if (regs || staged) dc_finalize_unit<true>(lck, lci, n_c, need, io + c_less, n_rows, lh, wtot, sres, smisc, ko ? ko + c_less : nullptr);
    else dc_finalize_unit(ck, ci, n_c, need, io + c_less, n_rows, lh, wtot, sres, smisc, ko ? ko + c_less : nullptr, s_list);
}

// The same for ids in best-first order (k <= kSortMost): the unit's certain members (which classify_kernel
// wrote to idx_out and sel_keys) and its candidates are ordered together by one counting pass
// (dc_select_counted), which is the selection as well.  4 units, 1024 of about 1400 candidates: 5.6 us,
// against 6.1 us for a selection and 8.6 us for a bitonic sort of its result in a kernel of its own.
// Lists that do not fit the LDS and keys that crowd into few bins take the selection above and the
// bitonic sort.
constexpr int kSortedLds = 12288;

__global__ __launch_bounds__(kFinalThreads) void select_sorted_kernel(
    uint32_t *__restrict__ hist, UnitState *__restrict__ state, const uint32_t *__restrict__ cand_key,
    const uint32_t *__restrict__ cand_idx, uint32_t *__restrict__ idx_out, int64_t idx_stride,
    uint32_t *__restrict__ sel_keys, int n_rows, int k_eff, int reinit) {
    __shared__ uint32_t lh[kRadixBins];
    __shared__ uint32_t wtot[kFinalThreads / 64 + 1];
    __shared__ uint32_t sres[4];
    __shared__ uint32_t smisc[2];
    __shared__ __align__(16) uint32_t s_list[2 * kSortedLds];
    uint32_t *const lck = s_list, *const lci = s_list + kSortedLds;
    static_assert(kRadixCopies * kRadixBins <= 2 * kSortedLds, "the counts of lists that do not fit take their place");
    __shared__ unsigned long long buf[kSortMost + kSortBinMost];
    const int unit = blockIdx.x;
    const int tid = threadIdx.x;
    UnitState *st = state + unit;
    const uint32_t *ck = cand_key + (int64_t)unit * n_rows;
    const uint32_t *ci = cand_idx + (int64_t)unit * n_rows;
    uint32_t *io = idx_out + (int64_t)unit * idx_stride;
    uint32_t *ko = sel_keys + (int64_t)unit * k_eff;
    // the head of the candidate list is fetched before its length is known
    constexpr int kHead = 4;
    uint32_t hk[kHead], hi[kHead];
#pragma unroll
    for (int j = 0; j < kHead; ++j) {
        const int i = tid + j * kFinalThreads;
        hk[j] = hi[j] = 0;
        if (i < n_rows) {
            hk[j] = ck[i];
            hi[j] = ci[i];
        }
    }
    uint32_t n_c = st->cand_cnt;
    const uint32_t kk = (uint32_t)k_eff;
    uint32_t c_less = st->c_less;
    if (n_c > (uint32_t)n_rows) n_c = n_rows;
    if (c_less > kk) c_less = kk;
    const uint32_t n = c_less + n_c, need = kk < n ? kk : n;
    const bool staged = n <= (uint32_t)kSortedLds;
    if (staged) {
        for (uint32_t i = tid; i < c_less; i += kFinalThreads) {
            lck[i] = ko[i];
            lci[i] = io[i];
        }
#pragma unroll
        for (int j = 0; j < kHead; ++j) {
            const uint32_t i = (uint32_t)(tid + j * kFinalThreads);
            if (i < n_c) {
                lck[c_less + i] = hk[j];
                lci[c_less + i] = hi[j];
            }
        }
        for (uint32_t i = tid + kHead * kFinalThreads; i < n_c; i += kFinalThreads) {
            lck[c_less + i] = ck[i];
            lci[c_less + i] = ci[i];
        }
    }
    __syncthreads();  // every thread has read the counters
    if (reinit) {
        uint4 *hz = reinterpret_cast<uint4 *>(hist + (int64_t)unit * DC_HIST_BINS);
        if (tid < DC_HIST_BINS / 4) hz[tid] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (tid == 0) {
        if (reinit) {
            st->tb_run = DC_HIST_BINS;
            st->surv_cnt = 0;
        }
        st->win_cnt = 0;
        st->cand_cnt = 0;
    }
    if (need == 0u) return;
    if (staged && dc_select_counted<true>(lck, lci, n, need, buf, lh, wtot, sres, smisc,
                                   [&](uint32_t rank, uint32_t, uint32_t id) { io[rank] = id; }))
        return;
    __syncthreads();
    if (c_less < need) {
        if (staged)
            dc_finalize_unit<true>(lck + c_less, lci + c_less, n_c, need - c_less, io + c_less, n_rows, lh, wtot, sres, smisc,
                                   ko + c_less);
        else
            dc_finalize_unit(ck, ci, n_c, need - c_less, io + c_less, n_rows, lh, wtot, sres, smisc, ko + c_less, s_list);
    }
    __syncthreads();
    int pow2 = 128;
    while (pow2 < (int)need) pow2 <<= 1;
    for (int i = tid; i < pow2; i += kFinalThreads)
        buf[i] = i < (int)need ? ((unsigned long long)ko[i] << 32) | io[i] : ~0ull;
    __syncthreads();
    dc_bitonic_lds(buf, pow2);
    for (int i = tid; i < (int)need; i += kFinalThreads) io[i] = (uint32_t)buf[i];
}

}  // namespace

extern "C" size_t dc_score_select_workspace_bytes(int n_units, int n_rows, int k) {
    return carve_fused(nullptr, n_units, n_rows, k).bytes;
}

extern "C" size_t dc_sketch_select_workspace_bytes(int n_units, int n_rows, int k) {
    return carve_fused(nullptr, n_units, n_rows, k).bytes;  // the same lists serve both paths
}

namespace {

constexpr int kFewFillBlocks = 512;  // see plan_fused

struct FusedPlan {
    int n_units, k_eff, small_chunks, big_steps;
    int64_t blocks;
};

int plan_fused(const char *who, int n_b, int n_h, int n_rows, int budget, FusedPlan *p,
               int big_steps = kBigSteps, int rows_per_step = kRowsPerBlockStep, int fill_div = 2048) {
    DC_REQUIRE(n_b >= 0 && n_h >= 1 && n_rows >= 0 && budget >= 0, "%s: bad sizes", who);
    const int64_t n_units64 = (int64_t)n_b * n_h;
    DC_REQUIRE(n_units64 < (1 << 20), "%s: too many units", who);
    p->n_units = (int)n_units64;
    p->k_eff = budget < n_rows ? budget : n_rows;
    // chunks per unit: up to kSmallChunks blocks of one step, then blocks of big_steps steps.
    // Short scans take fewer steps per block so that the grid still has fill_div blocks or
    // more: a block's steps run one after the other, and with few blocks the kernel
    // lasts as long as its longest block.  (2048 for the bf16 scan of many units.  With 512, for the sketch scan and the bf16
    // scan of few units, every scan that is listed at all -- more rows than plan_dense and plan_dense_keys take --
    // has blocks of big_steps: there a block's start and end cost more than its steps do.)
    const int64_t tiles = ((int64_t)n_rows + rows_per_step - 1) / rows_per_step;
    const int64_t fill = n_units64 * tiles / fill_div;
    if (fill < big_steps) big_steps = fill < 1 ? 1 : (int)fill;
    p->big_steps = big_steps;
    p->small_chunks = (int)(tiles < kSmallChunks ? tiles : kSmallChunks);
    const int64_t rest = (int64_t)n_rows - (int64_t)p->small_chunks * rows_per_step;
    const int64_t big_rows = (int64_t)p->big_steps * rows_per_step;
    const int64_t big_chunks = rest > 0 ? (rest + big_rows - 1) / big_rows : 0;
    p->blocks = n_units64 * (p->small_chunks + big_chunks);
    DC_REQUIRE(p->blocks < (1ll << 31), "%s: grid too large", who);
    return DC_OK;
}

// Whether the sketch scan of these sizes is a dense one, and its grid: blocks of equal shares, all running at once
// (four per CU at 64 columns, three at 128, two at 256; 256 per unit at most, because every block adds its counts to the unit's
// one histogram: 1 x 262107 of 64 columns 30.2 us with 1024 blocks, 20.1 with 256; listed 27.3).  Per layer, us, listed / dense: 8
// units x 131004 rows of 128 columns 48.9 / 45.1, x 65468 38.5 / 35.5, 16 x 131004 75.0 / 69.5, 32 x 131004 125.4 / 121.5, 4 x 1048508
// 135.5 / 121.8, 128 x 32700 138.6 / 135; 8 x 131004 of 64 38.4 / 32.0, 12 x 24615 of 256 44.7 / 41.4.  Beyond 4 Mi rows in all
// equal shares end at unequal times and the two bytes a row outweigh the list: 64 x 131004 225.8 / 237.7, 8 x 1048508 221.7 /
// 235.3.  From 128 columns on that shows from 2.5 Mi rows on where few rows are selected and the list is short: the selection
// alone, 64 x 65420 of 128, 64 ids 97.9 / 105.0, 1024 ids 107.2 / 107.4, 4096 ids 128.8 / 123.3; 32 x 130878 of 256, 64 ids 174.5 /
// 184.5, 2048 ids 197.3 / 195.8; but 24 x 109189 of 128, 64 ids 67.6 / 66.7, and 64 x 65420 of 64, 64 ids 61.7 / 62.8.
constexpr int64_t kDenseMostTiles = (4ll << 20) / kRowsPerBlockStep, kDenseFewTiles = (5ll << 19) / kRowsPerBlockStep;

// The grid of a dense scan of at least one unit and one tile: `most` blocks at the very most (one per unit where there are more
// units), which is as many as run at a time, so that none starts when the others end, but for the largest bf16 scans.  (Shares worked out from all tiles together gave a few blocks more where the
// tiles of a unit did not divide: 24 units x 65000 rows of 256 columns 106 against 94 us, 56 x 30011 of 128 68.1 against 65.5.)
void plan_shares(int64_t n_units, int64_t tiles, int64_t most, FusedPlan *p) {
    const int64_t each = most > n_units ? most / n_units : 1, steps = (tiles + each - 1) / each;
    p->small_chunks = 0;
    p->big_steps = (int)steps;
    p->blocks = n_units * ((tiles + steps - 1) / steps);
}

bool plan_dense(int64_t n_units, int n_rows, int hd, int k_eff, FusedPlan *p) {
    const int64_t tiles = ((int64_t)n_rows + kRowsPerBlockStep - 1) / kRowsPerBlockStep;
    if (n_units * tiles > (hd == 64 || k_eff >= 8 * hd ? kDenseMostTiles : kDenseFewTiles)) return false;
    const int64_t most = 256 * (hd == 64 ? 4 : (hd == 128 ? 3 : 2));
    if (p) plan_shares(n_units, tiles, most < 256 * n_units ? most : 256 * n_units, p);
    return true;
}

// Rows of a thread per tile of the exact pass of a dense scan: tiles of 512, 1024 or 2048 rows.  What a block scores one after
// the other is its tiles' candidates, so short regions, and those of which much is selected, take small tiles on many
// blocks; where every CU has work either way, a tile costs its barriers and its slot reservation.  Per selection, us, 512 / 1024 /
// 2048: 8 units x 8000 rows of 256 columns, 2048 ids 20.2 / 24.0 / 31.8, 1 x 16000 17.1 / 19.1 / 22.5, 32 x 8000 30.6 / 32.4 /
// 39.8, 8 x 60000 34.4 / 35.1 / 36.3, 8 x 131004 58.7 / 57.9 / 58.0, 8 x 262144 108.0 / 103.4 / 101.7; 64 x 16000 of 64, 64 ids 24.6 / 22.8 /
// 22.3.
// (The listed scan, which dealt its list out in pieces of 256 to one block per 1024 rows, took 26.1 in the first of these.)
int dense_per_thread(int64_t n_units, int n_rows) {
    const int64_t all = n_units * n_rows;
    if (n_rows <= 32 * 1024 && all <= 384 * 1024) return 2;
    return n_rows <= 96 * 1024 && all <= 1024 * 1024 ? 4 : 8;
}

// The same for the bf16 scan, whose rows take twice the bytes and leave four of them: two blocks per CU.  Per layer, us,
// listed / dense: 32 units x 49933 rows of 128 columns 101 / 95, 24 x 70000 100.3 / 95, 12 x 130001 95 / 89.6, 20 x 77771
// 98.5 / 91, 8 x 81852 53.0 / 49.3, 8 x 45000 39.0 / 35.9, 2 x 131004 40.0 / 35.3, 4 x 524000 125.6 / 111.4; 24 x 65000 of 64 59.2 /
// 55.4; 9 x 55555 of 256 71.3 / 68.8.  Beyond 1.75 Mi rows it is as often slower: 16 x 131004 112.2 / 115.5, 32 x 100000 163.6 /
// 166.2, 32 x 131004 204.1 / 208.3.  Up to 768 rows the listed scan's few blocks are the shorter chain (96 x 304 of 64 13.0 / 13.7).
//
// Its grid, selections alone, us: up to 640 tiles of 256 rows a block each (24 x 5424 of 128: 264 blocks of two tiles 19.7, 528
// of one 18.3); then 512 blocks, 1024 from 64 units on (64 x 16000 of 128 59.0 / 56.5, listed 55.1).  (768 instead of 512, per layer: 8 x 131004 of
// 128 67.1 -> 63.8, but 16 x 39932 48.5 -> 50.3, 4 x 199932 53.3 -> 55.2, 8 x 44932 35.6 -> 36.9, 8 x 99932 of 64 36.7 -> 38.3: no line between
// them is known.)  Above 1 Mi rows, where every share is long, 1280 blocks up to 32 units and 128 columns: a CU holds four, but the shorter
// shares outweigh the late start of some (per layer, 1024 / 1280: 32 x 49933 of 128 93.9 / 91.9, 16 x 99932 89.7 / 87.9; 16 x 100003 of 64
// 56.3 / 55.2, 32 x 49933 59.3 / 58.0, 8 x 199932 54.7 / 53.7); at 256 columns from 9 to 64 units one per CU (32 x 50000 144.5 / 139.5,
// listed 139.0).
constexpr int64_t kDenseKeyTiles = (7ll << 18) / kRowsPerBlockStep;  // 1.75 Mi rows
constexpr int kDenseKeyRows = 768;

bool plan_dense_keys(int64_t n_units, int n_rows, int hd, FusedPlan *p) {
    const int64_t tiles = ((int64_t)n_rows + kRowsPerBlockStep - 1) / kRowsPerBlockStep;
    if (n_rows <= kDenseKeyRows || n_units * tiles > kDenseKeyTiles) return false;
    if (!p) return true;
    const int64_t all = n_units * tiles;
    int64_t most = all <= 640 ? all : (n_units < 64 ? 512 : 1024);
    if (all > (1ll << 20) / kRowsPerBlockStep)
        most = hd == 256 ? (n_units > 8 && n_units <= 64 ? 256 : 512) : (n_units <= 32 ? 1280 : 512);
    plan_shares(n_units, tiles, most, p);
    return true;
}

int check_ws(const char *who, void *workspace, size_t workspace_bytes, int n_units, int n_rows,
             int budget, FusedWs *w) {
    DC_REQUIRE(workspace && (((uintptr_t)workspace) & 255u) == 0,
               "%s: workspace must be non-null and 256-byte aligned", who);
    *w = carve_fused(workspace, n_units, n_rows, budget);
    if (workspace_bytes < w->bytes) {
        dc_set_error("%s: workspace %zu bytes < %zu needed", who, workspace_bytes, w->bytes);
        return DC_ENOMEM;
    }
    return DC_OK;
}

}  // namespace

extern "C" int dc_select_state_init(int n_units, int n_rows, int budget, void *workspace,
                                    size_t workspace_bytes, void *stream) {
    DC_REQUIRE(n_units >= 0 && n_rows >= 0 && budget >= 0, "dc_select_state_init: bad sizes");
    if (n_units == 0) return DC_OK;
    FusedWs w;
    int rc = check_ws("dc_select_state_init", workspace, workspace_bytes, n_units, n_rows, budget, &w);
    if (rc) return rc;
    const int64_t n = (int64_t)n_units * DC_HIST_BINS;
    hipLaunchKernelGGL(init_state_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, w.hist, w.state, n_units);
    DC_CHECK_LAUNCH("dc_select_state_init");
    return DC_OK;
}

extern "C" int dc_score_prune_bf16(const void *k, const void *q, int n_b, int n_h, int n_rows, int hd,
                                   int64_t sb, int64_t sh, int64_t sr, int q_group, int budget,
                                   int mode, void *workspace, size_t workspace_bytes, void *stream) {
    return dc_score_prune_launch(k, q, n_b, n_h, n_rows, hd, sb, sh, sr, q_group, budget, mode, workspace,
                                 workspace_bytes, stream, nullptr, 0);
}

// hi_dev: null, or a device word holding the row at which the region ends at the time the kernel
// runs (lo_row: its first row); n_rows is then the capacity that the grid and the lists are laid
// out for.
int dc_score_prune_launch(const void *k, const void *q, int n_b, int n_h, int n_rows, int hd, int64_t sb, int64_t sh,
                          int64_t sr, int q_group, int budget, int mode, void *workspace, size_t workspace_bytes,
                          void *stream, const int32_t *hi_dev, int lo_row) {
    DC_REQUIRE(k && q, "dc_score_prune_bf16: null pointer");
    DC_REQUIRE(q_group >= 1, "dc_score_prune_bf16: bad q_group");
    DC_REQUIRE(hd == 64 || hd == 128 || hd == 256, "dc_score_prune_bf16: head_dim %d not in {64,128,256}", hd);
    DC_REQUIRE(mode == DC_MODE_IP || mode == DC_MODE_REF_DIST, "dc_score_prune_bf16: bad mode %d", mode);
    DC_REQUIRE(dc_aligned16(k), "dc_score_prune_bf16: k must be 16-byte aligned");
    DC_REQUIRE(sb % 8 == 0 && sh % 8 == 0 && sr % 8 == 0 && sr >= hd,
               "dc_score_prune_bf16: strides must be multiples of 8 elements and row_stride >= hd");
    FusedPlan p;
    // (short scans of up to 32 units: eight steps per block down to 512 blocks, like the sketch scan)
    int rc = plan_fused("dc_score_prune_bf16", n_b, n_h, n_rows, budget, &p, kBigSteps, kRowsPerBlockStep,
                        (int64_t)n_b * n_h <= 32 ? kFewFillBlocks : 2048);
    if (rc) return rc;
    if (p.n_units == 0 || p.k_eff == 0) return DC_OK;
    FusedWs w;
    rc = check_ws("dc_score_prune_bf16", workspace, workspace_bytes, p.n_units, n_rows, budget, &w);
    if (rc) return rc;
    const bool dense = plan_dense_keys(p.n_units, n_rows, hd, &p);
    const int n_chunks = (int)(p.blocks / p.n_units);
    // (dense: 1280 chunks at most, so that no unit's share of them leaves 32 bits)
    const uint32_t apart = dense ? ((uint32_t)n_chunks << 16) / (uint32_t)p.n_units : 0u;
    hipStream_t st = (hipStream_t)stream;
#define DC_LAUNCH_SPD(HD, DN)                                                                      \
    hipLaunchKernelGGL((score_prune_kernel<HD, DN>), dc_unit_grid(p.n_units, n_chunks), dim3(kThreads), 0, st, \
                       (const uint16_t *)k, (const uint16_t *)q, w.hist, w.state, w.surv,          \
                       p.n_units, n_h, n_rows, sb, sh, sr, q_group, mode, p.k_eff, p.small_chunks,  \
                       p.big_steps, n_chunks, apart, hi_dev, lo_row)
#define DC_LAUNCH_SP(HD)                    \
    do {                                    \
        if (dense) DC_LAUNCH_SPD(HD, true); \
        else DC_LAUNCH_SPD(HD, false);      \
    } while (0)
    if (hd == 64) DC_LAUNCH_SP(64);
    else if (hd == 128) DC_LAUNCH_SP(128);
    else DC_LAUNCH_SP(256);
#undef DC_LAUNCH_SP
#undef DC_LAUNCH_SPD
    DC_CHECK_LAUNCH("dc_score_prune_bf16");
    return DC_OK;
}

namespace {

// finish (+ sort): picks min(k, candidates) from the unit's candidate list
int launch_finish(const char *who, const FusedWs &w, uint32_t *idx_out, int64_t idx_unit_stride, int n_units,
                  int n_rows, int k_eff, int mode, int order, int reinit, hipStream_t st) {
    uint32_t *sel_keys = order == DC_ORDER_BEST ? w.sel_keys : nullptr;
    if (order == DC_ORDER_BEST && k_eff <= kSortMost) {
        hipLaunchKernelGGL(select_sorted_kernel, dim3(n_units), dim3(kFinalThreads), 0, st, w.hist, w.state,
                           w.cand_key, w.cand_idx, idx_out, idx_unit_stride, sel_keys, n_rows, k_eff, reinit);
        DC_CHECK_LAUNCH(who);
        return DC_OK;
    }
    hipLaunchKernelGGL(select_finish_kernel, dim3(n_units), dim3(kFinalThreads), 0, st, w.hist, w.state,
                       w.cand_key, w.cand_idx, idx_out, idx_unit_stride, sel_keys, n_rows, k_eff, reinit);
    DC_CHECK_LAUNCH(who);
    if (order != DC_ORDER_ANY)
        return dc_sort_selected(nullptr, 0, sel_keys, idx_out, idx_unit_stride, w.sort_scratch, n_units,
                                k_eff, mode, order, st, n_rows);
    return DC_OK;
}

// classify + finish (+ sort) on the survivor list of score_prune_kernel
int launch_select(const char *who, const FusedWs &w, uint32_t *idx_out, int64_t idx_unit_stride, int n_units,
                  int n_rows, int k_eff, int mode, int order, int reinit, hipStream_t st) {
    uint32_t *sel_keys = order == DC_ORDER_BEST ? w.sel_keys : nullptr;
    // blocks per unit for the classify pass: one per 4096 rows of context, as long as
    // the grid stays near 2048 blocks
    // one block per 4096 rows and at most 2048 blocks; below 3 Mi rows in all, one per 1024 rows
    // and at most 1024 blocks (8 x 131072 rows: 5.5 us against 7.1 us)
    if (plan_dense_keys(n_units, n_rows, 0, nullptr)) {
        const int64_t blocks = (int64_t)n_units * (((int64_t)n_rows + kKeyClassRows - 1) / kKeyClassRows);
        hipLaunchKernelGGL(key_classify_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, st, w.hist, w.state, w.surv, w.cand_key,
                           w.cand_idx, idx_out, idx_unit_stride, sel_keys, n_units, n_rows, k_eff, mode);
        DC_CHECK_LAUNCH(who);
        return launch_finish(who, w, idx_out, idx_unit_stride, n_units, n_rows, k_eff, mode, order, reinit, st);
    }
    const bool few = (int64_t)n_units * n_rows < (3ll << 20);
    int nblk = few ? (n_rows + 1023) / 1024 : (n_rows + 4095) / 4096;
    const int grid = few ? 1024 : 2048;
    const int cap = n_units >= grid ? 1 : grid / n_units;
    if (nblk > cap) nblk = cap;
    if (nblk < 1) nblk = 1;
    hipLaunchKernelGGL(classify_kernel, dim3((unsigned)n_units * (unsigned)nblk), dim3(kThreads), 0, st,
                       w.hist, w.state, w.surv, w.cand_key, w.cand_idx, idx_out, idx_unit_stride, sel_keys,
                       n_units, n_rows, k_eff, mode, nblk);
    DC_CHECK_LAUNCH(who);
    return launch_finish(who, w, idx_out, idx_unit_stride, n_units, n_rows, k_eff, mode, order, reinit, st);
}

}  // namespace

extern "C" int dc_sparse_select(uint32_t *idx_out, int64_t idx_unit_stride, int n_units, int n_rows,
                                int budget, int mode, int order, int reinit, void *workspace,
                                size_t workspace_bytes, void *stream) {
    DC_REQUIRE(idx_out, "dc_sparse_select: null pointer");
    DC_REQUIRE(n_units >= 0 && n_rows >= 0 && budget >= 0, "dc_sparse_select: bad sizes");
    DC_REQUIRE(mode == DC_MODE_IP || mode == DC_MODE_REF_DIST, "dc_sparse_select: bad mode %d", mode);
    DC_REQUIRE(order >= DC_ORDER_ANY && order <= DC_ORDER_INDEX, "dc_sparse_select: bad order %d", order);
    const int k_eff = budget < n_rows ? budget : n_rows;
    if (n_units == 0 || k_eff == 0) return DC_OK;
    DC_REQUIRE(idx_unit_stride >= k_eff, "dc_sparse_select: idx_unit_stride < min(budget, n_rows)");
    FusedWs w;
    int rc = check_ws("dc_sparse_select", workspace, workspace_bytes, n_units, n_rows, budget, &w);
    if (rc) return rc;
    return launch_select("dc_sparse_select", w, idx_out, idx_unit_stride, n_units, n_rows, k_eff, mode, order,
                         reinit, (hipStream_t)stream);
}

extern "C" int dc_score_select_bf16(const void *k, const void *q, uint32_t *idx_out,
                                    int64_t idx_unit_stride, int n_b, int n_h, int n_rows, int hd,
                                    int64_t sb, int64_t sh, int64_t sr, int q_group, int budget,
                                    int mode, int order, void *workspace, size_t workspace_bytes,
                                    void *stream) {
    DC_REQUIRE(n_b >= 0 && n_h >= 1, "dc_score_select_bf16: bad sizes");
    const int n_units = n_b * n_h;
    int rc = dc_select_state_init(n_units, n_rows, budget, workspace, workspace_bytes, stream);
    if (rc) return rc;
    rc = dc_score_prune_bf16(k, q, n_b, n_h, n_rows, hd, sb, sh, sr, q_group, budget, mode, workspace,
                             workspace_bytes, stream);
    if (rc) return rc;
    return dc_sparse_select(idx_out, idx_unit_stride, n_units, n_rows, budget, mode, order, 0, workspace,
                            workspace_bytes, stream);
}

extern "C" int dc_sketch_select_state_init(int n_units, int n_rows, int budget, void *workspace,
                                           size_t workspace_bytes, void *stream) {
    return dc_select_state_init(n_units, n_rows, budget, workspace, workspace_bytes, stream);
}

// Checks, state initialisation and the scan kernel of the sketch route; what follows the scan
// (exact pass, selection) is enqueued by the caller.
int dc_sketch_scan_launch(const char *who, const void *k, const uint8_t *codes, const float *scale,
                          const float *resid, const void *q, int n_b, int n_h, int n_rows, int hd, int64_t sb,
                          int64_t sh, int64_t sr, int64_t cb, int64_t ch, int64_t cr, int q_group, int budget,
                          int mode, int state_ready, void *workspace, size_t workspace_bytes,
                          void *ev_scan_begin, void *ev_scan_end, void *stream, const int32_t *hi_dev, int lo_row) {
    DC_REQUIRE(k && codes && scale && resid && q, "%s: null pointer", who);
    DC_REQUIRE(q_group >= 1, "%s: bad q_group", who);
    DC_REQUIRE(hd == 64 || hd == 128 || hd == 256, "%s: head_dim %d not in {64,128,256}", who, hd);
    DC_REQUIRE(mode == DC_MODE_IP || mode == DC_MODE_REF_DIST, "%s: bad mode %d", who, mode);
    DC_REQUIRE(dc_aligned16(k) && dc_aligned16(codes) && dc_aligned16(scale) && dc_aligned16(resid),
               "%s: k, codes, scale and resid must be 16-byte aligned", who);
    DC_REQUIRE(sb % 8 == 0 && sh % 8 == 0 && sr % 8 == 0 && sr >= hd,
               "%s: key strides must be multiples of 8 elements and row_stride >= hd", who);
    DC_REQUIRE(cb % 16 == 0 && ch % 16 == 0 && cr % 16 == 0 && cr >= hd,
               "%s: code strides must be multiples of 16 bytes and row_stride >= hd", who);
    DC_REQUIRE(n_rows <= kSketchMaxRows, "%s: %d rows per unit; the sketch scan takes at most %d (use the bf16 scan)", who,
               n_rows, kSketchMaxRows);
    FusedPlan p;
    int rc = plan_fused(who, n_b, n_h, n_rows, budget, &p, kBigSteps, kRowsPerBlockStep, kFewFillBlocks);
    if (rc) return rc;
    if (p.n_units == 0 || p.k_eff == 0) return DC_OK;
    const bool dense = plan_dense(p.n_units, n_rows, hd, p.k_eff, &p);
    DC_REQUIRE(workspace && (((uintptr_t)workspace) & 255u) == 0,
               "%s: workspace must be non-null and 256-byte aligned", who);
    const FusedWs w = carve_fused(workspace, p.n_units, n_rows, budget);
    if (workspace_bytes < w.bytes) {
        dc_set_error("%s: workspace %zu bytes < %zu needed", who, workspace_bytes, w.bytes);
        return DC_ENOMEM;
    }
    hipStream_t st = (hipStream_t)stream;
    if (!state_ready) {
        rc = dc_sketch_select_state_init(p.n_units, n_rows, budget, workspace, workspace_bytes, stream);
        if (rc) return rc;
    }
    if (ev_scan_begin) (void)hipEventRecord((hipEvent_t)ev_scan_begin, st);
#define DC_LAUNCH_SK(HD, SP, DN)                                                                    \
    hipLaunchKernelGGL((sketch_prune_kernel<HD, SP, DN>), dim3((unsigned)p.n_units, (unsigned)(p.blocks / p.n_units)), dim3(kThreads), 0, st,  \
                       codes, (const uint16_t *)q, scale, resid, w.hist, w.state, w.surv, p.n_units,    \
                       n_h, n_rows, cb, ch, cr, q_group, mode, p.k_eff, p.small_chunks, p.big_steps, hi_dev, lo_row)
    const bool shared_poll = p.n_units <= kSharedPollUnits;
#define DC_LAUNCH_SKH(HD)                                  \
    do {                                                   \
        if (dense) DC_LAUNCH_SK(HD, false, true);          \
        else if (shared_poll) DC_LAUNCH_SK(HD, true, false); \
        else DC_LAUNCH_SK(HD, false, false);               \
    } while (0)
    if (hd == 64) DC_LAUNCH_SKH(64);
    else if (hd == 128) DC_LAUNCH_SKH(128);
    else DC_LAUNCH_SKH(256);
#undef DC_LAUNCH_SKH
#undef DC_LAUNCH_SK
    DC_CHECK_LAUNCH(who);
    if (ev_scan_end) (void)hipEventRecord((hipEvent_t)ev_scan_end, st);
    return DC_OK;
}

extern "C" int dc_score_select_sketch_bf16(const void *k, const uint8_t *codes, const float *scale,
                                           const float *resid, const void *q, uint32_t *idx_out,
                                           int64_t idx_unit_stride, int n_b, int n_h, int n_rows, int hd,
                                           int64_t sb, int64_t sh, int64_t sr, int64_t cb, int64_t ch,
                                           int64_t cr, int q_group, int budget, int mode, int order,
                                           int state_ready, void *workspace, size_t workspace_bytes,
                                           void *ev_scan_begin, void *ev_scan_end, void *stream) {
    return dc_sketch_select_impl(k, codes, scale, resid, q, idx_out, idx_unit_stride, n_b, n_h, n_rows, hd, sb, sh, sr,
                                 cb, ch, cr, q_group, budget, mode, order, state_ready, workspace, workspace_bytes,
                                 ev_scan_begin, ev_scan_end, stream, nullptr, 0);
}

// hi_dev, lo_row: as in dc_score_prune_launch.  Only the scan needs the live length: the passes
// after it work on the lists the scan left, whose capacity is n_rows.
int dc_sketch_select_impl(const void *k, const uint8_t *codes, const float *scale, const float *resid, const void *q,
                          uint32_t *idx_out, int64_t idx_unit_stride, int n_b, int n_h, int n_rows, int hd,
                          int64_t sb, int64_t sh, int64_t sr, int64_t cb, int64_t ch, int64_t cr, int q_group,
                          int budget, int mode, int order, int state_ready, void *workspace, size_t workspace_bytes,
                          void *ev_scan_begin, void *ev_scan_end, void *stream, const int32_t *hi_dev, int lo_row) {
    const char *who = "dc_score_select_sketch_bf16";
    DC_REQUIRE(idx_out, "%s: null pointer", who);
    DC_REQUIRE(order >= DC_ORDER_ANY && order <= DC_ORDER_INDEX, "%s: bad order %d", who, order);
    int rc = dc_sketch_scan_launch(who, k, codes, scale, resid, q, n_b, n_h, n_rows, hd, sb, sh, sr, cb, ch, cr,
                                   q_group, budget, mode, state_ready, workspace, workspace_bytes,
                                   ev_scan_begin, ev_scan_end, stream, hi_dev, lo_row);
    if (rc) return rc;
    FusedPlan p;
    rc = plan_fused(who, n_b, n_h, n_rows, budget, &p);
    if (rc) return rc;
    if (p.n_units == 0 || p.k_eff == 0) return DC_OK;
    DC_REQUIRE(idx_unit_stride >= p.k_eff, "%s: idx_unit_stride < min(budget, n_rows)", who);
    const FusedWs w = carve_fused(workspace, p.n_units, n_rows, budget);
    hipStream_t st = (hipStream_t)stream;
    // Blocks per unit of the exact pass: one per 1024 rows of context, but a grid of at most 2048
    // blocks when the units hold 3 Mi rows or more between them and of 1024 below that (measured
    // at 8 to 128 units: 8 x 131072 rows 7.5 us against 9.1 us with half and 10.4 us with twice the
    // blocks; 64 x 131072 rows 18.9 us at 2048 blocks against 20.8 us at 1024 and 23.9 us at 4096).
    int nblk = (n_rows + 1023) / 1024;
    const int grid = (int64_t)p.n_units * n_rows >= (3ll << 20) ? 2048 : 1024;
    const int cap = p.n_units >= grid ? 1 : grid / p.n_units;
    if (nblk > cap) nblk = cap;
    if (nblk < 1) nblk = 1;
    const int per = plan_dense(p.n_units, n_rows, hd, p.k_eff, nullptr) ? dense_per_thread(p.n_units, n_rows) : 0;
    if (per) {
        const int tiles = (n_rows + kThreads * per - 1) / (kThreads * per);
        nblk = tiles < cap ? tiles : cap;
    }
#define DC_LAUNCH_RSP(HD, PER)                                                                        \
    hipLaunchKernelGGL((rescore_kernel<HD, PER>), dim3((unsigned)p.n_units, (unsigned)nblk), dim3(kThreads), 0, \
                       st, (const uint16_t *)k, (const uint16_t *)q, w.hist, w.state, w.surv, w.cand_key, \
                       w.cand_idx, p.n_units, n_h, n_rows, sb, sh, sr, q_group, mode, p.k_eff, nblk, hi_dev, lo_row)
#define DC_LAUNCH_RS(HD)                        \
    do {                                        \
        if (per == 2) DC_LAUNCH_RSP(HD, 2);     \
        else if (per == 4) DC_LAUNCH_RSP(HD, 4); \
        else if (per == 8) DC_LAUNCH_RSP(HD, 8); \
        else DC_LAUNCH_RSP(HD, 0);              \
    } while (0)
    if (hd == 64) DC_LAUNCH_RS(64);
    else if (hd == 128) DC_LAUNCH_RS(128);
    else DC_LAUNCH_RS(256);
#undef DC_LAUNCH_RS
#undef DC_LAUNCH_RSP
    DC_CHECK_LAUNCH(who);
    return launch_finish(who, w, idx_out, idx_unit_stride, p.n_units, n_rows, p.k_eff, mode, order, 1, st);
}

namespace {
// Keys of a block of pq_classify_kernel: 8192, or 2048 where those blocks would leave CUs idle and a unit has 128 of these at
// most, which all reserve their places with additions to one word.
int pq_class_rows(int64_t n_units, int n_rows) {
    return n_rows <= 128 * 2048 && n_units * ((n_rows + 8191) / 8192) < 512 ? 2048 : 8192;
}
}  // namespace

extern "C" size_t dc_pq_search_workspace_bytes(int n_units, int n_rows, int n_cand) {
    const FusedWs w = carve_fused(nullptr, n_units, n_rows, n_cand);
    const size_t nu = n_units > 0 ? n_units : 0;
    const size_t kc = (size_t)(n_cand < n_rows ? n_cand : n_rows);
    return w.bytes + dc_align_up(nu * (n_cand > 0 && n_rows > 0 ? kc : 0) * 4, 256);
}

extern "C" int dc_pq_search_bf16(const void *k, const uint8_t *codes, const float *lut, const void *q,
                                 uint32_t *idx_out, int64_t idx_unit_stride, int n_b, int n_h, int n_rows,
                                 int hd, int m, int64_t sb, int64_t sh, int64_t sr, int n_cand, int topk,
                                 int state_ready, void *workspace, size_t workspace_bytes,
                                 void *ev_scan_begin, void *ev_scan_end, void *stream) {
    const char *who = "dc_pq_search_bf16";
    DC_REQUIRE(k && codes && lut && q && idx_out, "%s: null pointer", who);
    DC_REQUIRE(hd == 64 || hd == 128 || hd == 256, "%s: head_dim %d not in {64,128,256}", who, hd);
    DC_REQUIRE(m == 16 || m == 32, "%s: m = %d subspaces unsupported (16 or 32)", who, m);
    DC_REQUIRE(n_cand >= 0 && topk >= 0 && topk <= n_cand, "%s: need 0 <= topk <= n_cand", who);
    DC_REQUIRE(dc_aligned16(k) && dc_aligned16(codes) && dc_aligned16(lut),
               "%s: k, codes and lut must be 16-byte aligned", who);
    DC_REQUIRE(sb % 8 == 0 && sh % 8 == 0 && sr % 8 == 0 && sr >= hd,
               "%s: key strides must be multiples of 8 elements and row_stride >= hd", who);
    FusedPlan p;
    int rc = plan_fused(who, n_b, n_h, n_rows, n_cand, &p);
    if (rc) return rc;
    const int k1 = p.k_eff;                   // candidates per unit
    const int k2 = topk < k1 ? topk : k1;     // results per unit
    if (p.n_units == 0 || k2 == 0) return DC_OK;
    DC_REQUIRE(idx_unit_stride >= k2, "%s: idx_unit_stride < min(topk, n_rows)", who);
    DC_REQUIRE(workspace && (((uintptr_t)workspace) & 255u) == 0,
               "%s: workspace must be non-null and 256-byte aligned", who);
    const FusedWs w = carve_fused(workspace, p.n_units, n_rows, n_cand);
    const size_t need = dc_pq_search_workspace_bytes(p.n_units, n_rows, n_cand);
    if (workspace_bytes < need) {
        dc_set_error("%s: workspace %zu bytes < %zu needed", who, workspace_bytes, need);
        return DC_ENOMEM;
    }
    uint32_t *cand = (uint32_t *)((char *)workspace + w.bytes);
    hipStream_t st = (hipStream_t)stream;
    if (!state_ready) {
        rc = dc_select_state_init(p.n_units, n_rows, n_cand, workspace, workspace_bytes, stream);
        if (rc) return rc;
    }
    // equal shares, a block per CU at most
    plan_shares(p.n_units, ((int64_t)n_rows + kPqThreads - 1) / kPqThreads, kPqBlocks, &p);
    const int64_t blocks = p.blocks, steps = p.big_steps;
    const int class_rows = pq_class_rows(p.n_units, n_rows);
    const int64_t class_blocks = p.n_units * (((int64_t)n_rows + class_rows - 1) / class_rows);
    DC_REQUIRE(blocks < (1ll << 31) && class_blocks < (1ll << 31), "%s: grid too large", who);
    if (ev_scan_begin) (void)hipEventRecord((hipEvent_t)ev_scan_begin, st);
    if (m == 16)
        hipLaunchKernelGGL(pq_scan_kernel<16>, dim3((unsigned)blocks), dim3(kPqThreads), 0, st, codes, lut, w.hist, w.surv,
                           p.n_units, n_rows, (int)steps);
    else
        hipLaunchKernelGGL(pq_scan_kernel<32>, dim3((unsigned)blocks), dim3(kPqThreads), 0, st, codes, lut, w.hist, w.surv,
                           p.n_units, n_rows, (int)steps);
    DC_CHECK_LAUNCH(who);
    if (ev_scan_end) (void)hipEventRecord((hipEvent_t)ev_scan_end, st);
    // the k1 best ADC scores of every unit, in no particular order
#define DC_LAUNCH_PC(M, ROWS)                                                                                             \
    hipLaunchKernelGGL((pq_classify_kernel<M, ROWS>), dim3((unsigned)class_blocks), dim3(kThreads), 0, st, codes, lut, w.hist, \
                       w.state, w.surv, w.cand_key, w.cand_idx, cand, (int64_t)k1, p.n_units, n_rows, k1)
    if (m == 16 && class_rows == 2048) DC_LAUNCH_PC(16, 2048);
    else if (m == 16) DC_LAUNCH_PC(16, 8192);
    else if (class_rows == 2048) DC_LAUNCH_PC(32, 2048);
    else DC_LAUNCH_PC(32, 8192);
#undef DC_LAUNCH_PC
    DC_CHECK_LAUNCH(who);
    rc = launch_finish(who, w, cand, k1, p.n_units, n_rows, k1, DC_MODE_IP, DC_ORDER_ANY, 1, st);
    if (rc) return rc;
    const int lpr = hd / 8, groups = kThreads / lpr;
    const int64_t bpu = ((int64_t)k1 + groups - 1) / groups;
    DC_REQUIRE((int64_t)p.n_units * bpu < (1ll << 31), "%s: grid too large", who);
#define DC_LAUNCH_PR(HD)                                                                              \
    hipLaunchKernelGGL(pq_rescore_kernel<HD>, dim3((unsigned)(p.n_units * bpu)), dim3(kThreads), 0, st, \
                       (const uint16_t *)k, (const uint16_t *)q, cand, w.state, w.cand_key, w.cand_idx, \
                       n_h, k1, (int64_t)k1, n_rows, sb, sh, sr, (int)bpu)
    if (hd == 64) DC_LAUNCH_PR(64);
    else if (hd == 128) DC_LAUNCH_PR(128);
    else DC_LAUNCH_PR(256);
#undef DC_LAUNCH_PR
    DC_CHECK_LAUNCH(who);
    return launch_finish(who, w, idx_out, idx_unit_stride, p.n_units, n_rows, k2, DC_MODE_IP, DC_ORDER_BEST, 1,
                         st);
}
