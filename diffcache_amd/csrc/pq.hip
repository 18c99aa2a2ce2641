// Product-quantisation baseline: per-query lookup tables and the asymmetric
// distance (ADC) scan.  The reference's PQ baseline directory
// (evaluation/impl/pqcache) is empty, so this follows the benchmark
// configuration only: M subspaces x 256 centroids, 8-bit codes, fp32 tables.
//
// The scan keeps the unit's tables in LDS (32 KB, laid out so that the reads of a
// wave never share a bank, see dc_pq.h) and gives each thread one key at a time:
// M code bytes, M table reads, M fp32 adds.  HBM traffic is M bytes per key.
#include "dc_common.h"
#include "dc_pq.h"

namespace {

constexpr int kThreads = 256;
constexpr int kKeysPerThread = 16;
constexpr int kKeysPerBlock = kThreads * kKeysPerThread;

__global__ __launch_bounds__(256) void pq_lut_kernel(const uint16_t *__restrict__ q,
                                                     const float *__restrict__ books,
                                                     float *__restrict__ lut, int n_h, int hd, int m) {
    const int um = blockIdx.x;  // unit * m + sub
    const int unit = um / m, sub = um % m;
    const int h = unit % n_h;
    const int ds = hd / m;
    const int c = threadIdx.x;
    const float *cb = books + (((int64_t)h * m + sub) * 256 + c) * ds;
    const uint16_t *qp = q + (int64_t)unit * hd + sub * ds;
    float acc = 0.f;
    for (int d = 0; d < ds; ++d) acc = fmaf(dc_bf16_to_f32(qp[d]), cb[d], acc);
    lut[(int64_t)um * 256 + c] = acc;
}

template <int M>
__global__ __launch_bounds__(kThreads) void pq_adc_kernel(
    const uint8_t *__restrict__ codes, const float *__restrict__ lut, float *__restrict__ scores,
    uint32_t *__restrict__ hist, int n_rows, int64_t scores_stride, int blocks_per_unit) {
    __shared__ float s_lut[kPqLutWords];
    __shared__ uint32_t lhist[DC_HIST_BINS];
    const int unit = blockIdx.x / blocks_per_unit;
    const int chunk = blockIdx.x % blocks_per_unit;
    const int tid = threadIdx.x;
    pq_stage_lut<M>(s_lut, lut + (int64_t)unit * M * 256, tid, kThreads);
    if (hist)
        for (int i = tid; i < DC_HIST_BINS; i += kThreads) lhist[i] = 0;
    PqLane<M> ln;
    ln.init(tid & 63);
    __syncthreads();
    const uint8_t *cu = codes + (int64_t)unit * n_rows * M;
    float *su = scores + (int64_t)unit * scores_stride;
    const int64_t base = (int64_t)chunk * kKeysPerBlock;  // a multiple of 64: lane = key mod 64
    for (int it = 0; it < kKeysPerThread; ++it) {
        const int64_t i = base + (int64_t)it * kThreads + tid;
        if (i >= n_rows) break;
        const uint4 *cp = reinterpret_cast<const uint4 *>(cu + i * M);
        uint32_t words[M / 4];
#pragma unroll
        for (int w = 0; w < M / 16; ++w) {
            const uint4 cw = cp[w];
            words[4 * w + 0] = cw.x;
            words[4 * w + 1] = cw.y;
            words[4 * w + 2] = cw.z;
            words[4 * w + 3] = cw.w;
        }
        const float acc = pq_adc_score<M>(words, s_lut, ln);
        su[i] = acc;
        if (hist) {
            uint32_t key, bucket;
            dc_key_bucket(acc, DC_MODE_IP, key, bucket);
            atomicAdd(&lhist[bucket], 1u);
        }
    }
    if (hist) {
        __syncthreads();
        uint32_t *hu = hist + (int64_t)unit * DC_HIST_BINS;
        for (int i = tid; i < DC_HIST_BINS; i += kThreads) {
            uint32_t c = lhist[i];
            if (c) atomicAdd(&hu[i], c);
        }
    }
}

// Codes of new keys: per subspace the nearest of (up to) 256 centroids.
//
// The distance that decides, |c|^2 / 2 - x.c, is a contraction over the few columns of a subspace,
// so it runs on the matrix cores: keys are bf16 already, a centroid's fp32 value is the exact
// sum of three bf16 values, and |c|^2 / 2 is three more with a factor of one, so the distances of 32
// keys to 32 centroids are one v_mfma_f32_32x32x16_bf16 (two at 8 columns, four at 16)
// of exact products with fp32 accumulation.  M = centroids and N = keys, so that a lane holds distances
// of ONE key: lane (h, c) = (lane / 32, lane % 32) supplies the first two parts of centroid c (h = 0), or the third and
// the bias (from 8 columns on one part per instruction), and the columns of key c, or ones against the bias.  Row
// 16 j + 8 u + 4 h + t of tile p is centroid 32 p + 16 j + 8 h + 4 u + t: a lane's sixteen results of a tile are two times
// eight neighbours, two "octets".
//
// What bounds the kernel is instruction issue on the vector ALUs, most of it the search for the minimum: 256 values per key
// and subspace.  Six instructions per eight values keep the least value and the octet it came from (four
// v_min3, a compare, a select).  At the end the two lanes of a key settle its octet, each lane
// for the key of one of the wave's two groups (v_permlane32_swap exchanges the halves), and that lane takes
// the least of the eight in fp32, from tables whose octets are padded apart so that lanes that look at the same place of
// different octets read different banks at fixed offsets.
//
// A CU holds one block, which stages the tables of its subspaces once and walks the keys; its waves take batches of 64 from a
// counter in LDS and meet at no barrier.  200003 keys of 128 columns, 32 subspaces: 68 us (275 instructions per wave and subspace,
// 192 of them the search, the vector ALUs issuing 95 % of the time that a CU is busy).  Blocks of 256 keys that stage for themselves took 75
// (347 instructions); walking with equal shares per wave 74, because the older waves of a SIMD run ahead and the youngest ends
// alone; two blocks of half the size per CU 69, one of which runs ahead; a tile's products asked for when the tile before has been searched
// 66 to 68, 87 % of the time issuing; the last batches dealt out by subspace 69; the octets' numbers as masks in scalar registers, 20
// instructions less, no faster.  Tiles of 16 x 16 x 16 (half the rate of the wider ones, four lanes to settle a key through LDS
// shuffles; 488 instructions) took 96 in the blocks of 256 keys, 32 x 32 x 8 90; torch's distance matrices, written to and read from
// HBM four times over, 11.8 ms.  16 subspaces of 8 columns 64 -> 55 us, 8 of 16 63 -> 51; 5000 keys 11.3 -> 10.6.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The upper halves of the three words sum up to x: 8 + 8 + 8 bits of its mantissa.
__device__ __forceinline__ void split3(float x, uint32_t &a, uint32_t &b, uint32_t &c) {
    a = __float_as_uint(x) & 0xffff0000u;
    const float r = x - __uint_as_float(a);
    b = __float_as_uint(r) & 0xffff0000u;
    c = __float_as_uint(r - __uint_as_float(b));
}

constexpr int kEncGroups = 2;                  // groups of 32 keys per wave: one per half of its lanes
constexpr int kEncBatch = 32 * kEncGroups;     // keys of a wave at a time
constexpr int kEncHalf = 12;                   // words of an octet's half norms, padded
// subspaces whose tables a block holds, and whose codes leave together (160 KB of LDS per CU)
__host__ __device__ constexpr int enc_subs(int ds) { return ds <= 8 ? 4 : 2; }
// threads of a block, of which a CU takes one
__host__ __device__ constexpr int enc_threads(int ds) { return ds <= 8 ? 1024 : 512; }

// Blocks of a column of subspaces, of the last one, which may have fewer of them, of all.
struct EncGrid {
    int per_column, last, blocks;
};

// A block per CU, in shares as equal as they come: the last column gets blocks by its number of subspaces.  Where the columns do not divide
// the CUs, or outnumber them, more and shorter blocks may fill them better in two or more turns, each of which costs a block about four
// batches to stage and start.  (256 / columns blocks of each, in a grid rounded up to eights, gave XCDs unequal numbers of them, some more than
// they have CUs.  200003 keys, us, blocks of 256 keys / that / this: 12 subspaces of 8 columns 50 / 67 / 43, 6 of 16 58 / 64 / 41, 24 of
// 4 58 / 94 / 53, 96 of 2 207 / 347 / 194, 5 of 8 29 / 25 / 20; 30001 keys, 272 of 2 95 / 276 / 93, 1040 of 2 384 / 2213 / 390.)
static bool plan_encode(int m, int subs, int64_t n, EncGrid *g) {
    const int64_t columns = (m + subs - 1) / subs, batches = (n + kEncBatch - 1) / kEncBatch;
    const int64_t whole = columns > 1 ? subs : m, last = m - (columns - 1) * subs;  // subspaces of a column, of the last
    auto last_of = [&](int64_t per) { return (per * last + whole - 1) / whole; };
    auto all_of = [&](int64_t per) { return (columns - 1) * per + last_of(per); };
    const int64_t most = (batches + 3) / 4;  // four batches each at least
    int64_t best = INT64_MAX, at = 1;
    for (int64_t turns = 1; turns <= 8; ++turns) {
        int64_t per = 256 * turns * whole / m + 1;
        while (per > 1 && all_of(per) > 256 * turns) --per;
        if (per > most) per = most;
        const int64_t cost = (all_of(per) + 255) / 256 * ((batches + per - 1) / per + 4);
        if (cost < best) best = cost, at = per;
        if (per == most || all_of(per) == 256 * turns) break;
    }
    if (all_of(at) >= (1ll << 31)) return false;
    g->per_column = (int)at;
    g->last = (int)last_of(at);
    g->blocks = (int)all_of(at);
    return true;
}

// (A CU's one block is four waves to a SIMD, of up to 128 registers, two of up to 256 at 16 columns: within 256 the compiler leaves the
// results of the matrix instructions in vector registers; with more it moves each through an accumulation register,
// one instruction per value, which is what the search costs.)
template <int DS>
__global__ __launch_bounds__(enc_threads(DS), enc_threads(DS) / 256) void pq_encode_kernel(
    const uint16_t *__restrict__ keys, int64_t key_stride, int64_t n, const float *__restrict__ books,
    uint8_t *__restrict__ codes, int64_t code_stride, int m, int nc, EncGrid grid) {
    constexpr int SUBS = enc_subs(DS), THREADS = enc_threads(DS);
    constexpr int KW = 4;                        // operand words per lane and instruction
    constexpr int NI = DS <= 4 ? 1 : 2;          // instructions per tile and eight columns (four, where there are no more)
    constexpr int KL = DS <= 4 ? 4 : 8;          // columns of a part of the centroid per lane and instruction
    constexpr int PARTS = DS <= 8 ? 1 : DS / 8;  // eights of columns
    constexpr int XW = (DS + 1) / 2;             // words of a key's columns
    constexpr int kOctet = 8 * DS + (DS < 4 ? DS : 4);  // words of an octet's centroids, padded
    // [tile][instruction][lane][word]: a wave's operand is one stretch
    __shared__ __align__(16) uint32_t s_a[SUBS][PARTS][8 * NI * 64 * KW];
    __shared__ __align__(16) float s_c[SUBS][32 * kOctet];
    __shared__ __align__(16) float s_half[SUBS][32 * kEncHalf];
    __shared__ uint32_t s_turn;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = lane >> 5, c = lane & 31;
    // The blocks that read the same keys (a few columns each, of lines they share) are next to each other in an order of which every XCD
    // takes an eighth in one piece: they run on one XCD at about the same time and find the lines in its L2.
    const int n_y = (m + SUBS - 1) / SUBS;
    const int xcd = blockIdx.x % 8, more = grid.blocks % 8;
    int at = xcd * (grid.blocks / 8) + (xcd < more ? xcd : more) + (int)blockIdx.x / 8;
    int place, col;  // among the blocks of the column; the column
    if (at < grid.last * n_y) {
        place = at / n_y;
        col = at % n_y;
    } else {  // the last column has no more
        at -= grid.last * n_y;
        place = grid.last + at / (n_y - 1);
        col = at % (n_y - 1);
    }
    const int per_column = col == n_y - 1 ? grid.last : grid.per_column;
    const int sub0 = col * SUBS;
    const int n_sub = m - sub0 < SUBS ? m - sub0 : SUBS;
    // stage the subspaces: the negated centroid in three bf16 parts, half its squared norm in three
    for (int s = tid / 256; s < n_sub; s += THREADS / 256) {
        const int at_c = tid & 255;  // this thread's centroid
        // and where it sits among the tiles' rows
        const int row = 16 * ((at_c >> 4) & 1) + 8 * ((at_c >> 2) & 1) + 4 * ((at_c >> 3) & 1) + (at_c & 3);
        const float *cp = books + ((int64_t)(sub0 + s) * nc + (at_c < nc ? at_c : nc - 1)) * DS;
        float cen[DS];
#pragma unroll
        for (int d = 0; d < DS; ++d) {
            const float v = cp[d];
            cen[d] = at_c < nc ? v : 0.f;
        }
        float half = 0.f;
#pragma unroll
        for (int d = 0; d < DS; ++d) half = fmaf(cen[d], cen[d], half);
        half = at_c < nc ? 0.5f * half : INFINITY;  // a centroid that does not exist is never the nearest, of no key
        s_half[s][(at_c >> 3) * kEncHalf + (at_c & 7)] = half;
#pragma unroll
        for (int d = 0; d < DS; ++d) s_c[s][(at_c >> 3) * kOctet + (at_c & 7) * DS + d] = cen[d];
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
            uint32_t e[4][KL];  // bf16 values in the upper halves: the three parts, the bias
#pragma unroll
            for (int j = 0; j < KL; ++j) {
                e[0][j] = e[1][j] = e[2][j] = e[3][j] = 0u;
                if (p * KL + j < DS) split3(-cen[p * KL + j < DS ? p * KL + j : 0], e[0][j], e[1][j], e[2][j]);
            }
            if (p == 0) split3(half, e[3][0], e[3][1], e[3][2]);
#pragma unroll
            for (int r = 0; r < 4; ++r)  // two instructions: r in lane 32 (r % 2) of number r / 2; one: parts 2 l and 2 l + 1 in half l
#pragma unroll
                for (int w = 0; w < KL / 2; ++w) {
                    const int at = NI == 2 ? ((at_c >> 5) * 128 + r * 32 + row) * KW + w : ((at_c >> 5) * 64 + (r / 2) * 32 + row) * KW + 2 * (r % 2) + w;
                    s_a[s][p][at] = __builtin_amdgcn_perm(e[r][2 * w + 1], e[r][2 * w], 0x07060302u);
                }
        }
    }
    const uint16_t *kp[kEncGroups];  // the batch that is loaded from
    auto point = [&](int64_t key0) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) {
            int64_t k = key0 + g * 32 + c;
            k = k < n ? k : n - 1;
            kp[g] = keys + k * key_stride + sub0 * DS;
        }
    };
    auto load_keys = [&](int s, uint32_t(&x)[kEncGroups][XW]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) {
            const uint16_t *p = kp[g] + s * DS;
            if constexpr (DS == 2) {
                x[g][0] = *reinterpret_cast<const uint32_t *>(p);
            } else if constexpr (DS == 4) {
                const uint2 t = *reinterpret_cast<const uint2 *>(p);
                x[g][0] = t.x, x[g][1] = t.y;
            } else {
#pragma unroll
                for (int w = 0; w < DS / 8; ++w) {
                    const uint4 t = reinterpret_cast<const uint4 *>(p)[w];
                    x[g][4 * w] = t.x, x[g][4 * w + 1] = t.y, x[g][4 * w + 2] = t.z, x[g][4 * w + 3] = t.w;
                }
            }
        }
    };
    // The block's waves take its batches as they come: the older waves of a SIMD run ahead of the younger ones, and with equal
    // shares the youngest would end alone.
    auto take = [&](int turn) __attribute__((always_inline)) { return ((int64_t)turn * per_column + place) * kEncBatch; };
    int64_t key0 = take(wave);
    uint32_t xw[kEncGroups][XW], xn[kEncGroups][XW];
    uint32_t word = 0u;  // the codes of key key0 + lane
    int s = 0;
    int64_t key_next = n;
    if (tid == 0) s_turn = THREADS / 64;
    point(key0);
    load_keys(0, xw);
    __syncthreads();
    while (key0 < n) {
        // the keys' operands: the columns, and ones against the bias
        uint32_t b[kEncGroups][PARTS][NI][KW];
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g)
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int w = 0; w < KW; ++w) {
                    const int xi = NI == 2 ? p * KW + w : w % 2, wb = NI == 2 ? w : w - 2;
                    const uint32_t x = xi < XW ? xw[g][xi < XW ? xi : 0] : 0u;
                    const uint32_t one = p != 0 ? 0u : (wb == 0 ? 0x3f803f80u : (wb == 1 ? 0x00003f80u : 0u));
                    b[g][p][0][w] = x;
                    if (NI == 2 || w >= 2) b[g][p][NI - 1][w] = h == 0 ? x : one;
                }
        // the next columns are on the way meanwhile (past the last key they repeat it)
        const bool last = s + 1 == n_sub;
        if (last) {
            uint32_t turn = 0u;
            if (lane == 0) turn = atomicAdd(&s_turn, 1u);
            key_next = take(__builtin_amdgcn_readfirstlane((int)turn));
            point(key_next);
        }
        load_keys(last ? 0 : s + 1, xn);
        float best[kEncGroups];
        uint32_t from[kEncGroups];  // 2 * tile + which of its octets
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) {
            best[g] = INFINITY;
            from[g] = 0u;
        }
        uint32_t aw[PARTS][NI][KW];
        auto load_tile = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(&s_a[s][p][((NI * t + i) * 64 + lane) * KW]);
                    aw[p][i][0] = v.x, aw[p][i][1] = v.y, aw[p][i][2] = v.z, aw[p][i][3] = v.w;
                }
        };
        // A tile's products are asked for before the tile ahead of it is searched, its operands another one earlier: a result is
        // dozens of cycles away from its instruction.
        f32x16 d[2][kEncGroups];
        auto products = [&](f32x16(&dst)[kEncGroups]) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int g = 0; g < kEncGroups; ++g) {
                        const uint4 av = make_uint4(aw[p][i][0], aw[p][i][1], aw[p][i][2], aw[p][i][3]);
                        const uint4 bv = make_uint4(b[g][p][i][0], b[g][p][i][1], b[g][p][i][2], b[g][p][i][3]);
                        const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                        dst[g] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), __builtin_bit_cast(bf16x8, bv),
                                                                         p == 0 && i == 0 ? zero : dst[g], 0, 0, 0);
                    }
        };
        load_tile(0);
        products(d[0]);
        load_tile(1);
#pragma unroll  // (whole: the octets' numbers are constants of their instructions then, and so are the tiles' addresses)
        for (int t = 0; t < 8; ++t) {
            __builtin_amdgcn_sched_barrier(0);
            if (t < 7) products(d[(t + 1) & 1]);
            if (t < 6) load_tile(t + 2);
            __builtin_amdgcn_sched_barrier(0);
            // each step of the search for all groups: a compare's mask is two cycles from its reader
            const f32x16(&dt)[kEncGroups] = d[t & 1];
#pragma unroll
            for (int o = 0; o < 2; ++o) {
                float v[kEncGroups];
                bool less[kEncGroups];
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(dt[g][8 * o], dt[g][8 * o + 1]), dt[g][8 * o + 2]);
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], dt[g][8 * o + 3]), dt[g][8 * o + 4]);
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], dt[g][8 * o + 5]), dt[g][8 * o + 6]);
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], dt[g][8 * o + 7]), best[g]);
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) less[g] = v[g] < best[g];
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) {
                    from[g] = less[g] ? (uint32_t)(2 * t + o) : from[g];
                    best[g] = v[g];
                }
            }
        }
        // The two lanes of a key hold its least value over their octets each.  The halves of the wave exchange a
        // group: half h ends with both lanes' values for group h.  (Equal values: the lower octet.)
        uint32_t oct[kEncGroups];
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) oct[g] = 2u * from[g] + (uint32_t)h;
        const auto bv = __builtin_amdgcn_permlane32_swap(__float_as_uint(best[0]), __float_as_uint(best[1]), false, false);
        const auto ov = __builtin_amdgcn_permlane32_swap(oct[0], oct[1], false, false);
        const float v0 = __uint_as_float(bv[0]), v1 = __uint_as_float(bv[1]);
        const bool second = v1 < v0 || (v1 == v0 && ov[1] < ov[0]);
        const uint32_t octet = second ? ov[1] : ov[0];
        // the least of the octet, in fp32, for key key0 + lane
        float xf[2 * XW];
#pragma unroll
        for (int w = 0; w < XW; ++w) {
            const uint32_t x = h ? xw[1][w] : xw[0][w];
            xf[2 * w] = dc_bf16_lo(x);
            xf[2 * w + 1] = dc_bf16_hi(x);
        }
        const float4 *hp = reinterpret_cast<const float4 *>(s_half[s] + octet * kEncHalf);
        const float4 h0 = hp[0], h1 = hp[1];
        const float hs[8] = {h0.x, h0.y, h0.z, h0.w, h1.x, h1.y, h1.z, h1.w};
        const float *cp = s_c[s] + octet * kOctet;
        float dist[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            dist[i] = hs[i];
#pragma unroll
            for (int k = 0; k < DS; ++k) dist[i] = fmaf(-xf[k], cp[i * DS + k], dist[i]);
        }
        float least = dist[0];
        uint32_t id = 0u;
#pragma unroll
        for (int i = 1; i < 8; ++i) {
            const bool take = dist[i] < least;
            least = take ? dist[i] : least;
            id = take ? (uint32_t)i : id;
        }
        word |= (octet * 8u + id) << (8 * s);
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g)
#pragma unroll
            for (int w = 0; w < XW; ++w) xw[g][w] = xn[g][w];
        ++s;
        if (!last) continue;
        const int64_t k = key0 + lane;
        if (k < n) {
            uint8_t *dst = codes + k * code_stride + sub0;
            if (SUBS == 4 && n_sub == SUBS && (code_stride & 3) == 0) {
                *reinterpret_cast<uint32_t *>(dst) = word;
            } else if (SUBS == 2 && n_sub == SUBS && (code_stride & 1) == 0) {
                *reinterpret_cast<uint16_t *>(dst) = (uint16_t)word;
            } else {
                for (int i = 0; i < n_sub; ++i) dst[i] = (uint8_t)(word >> (8 * i));
            }
        }
        key0 = key_next;
        s = 0;
        word = 0u;
    }
}

}  // namespace

extern "C" int dc_pq_encode_bf16(const void *keys, int64_t key_stride, int64_t n, const float *books, uint8_t *codes,
                                 int64_t code_stride, int hd, int m, int n_centroids, void *stream) {
    const char *who = "dc_pq_encode_bf16";
    DC_REQUIRE(n >= 0 && m >= 1 && hd >= m && hd % m == 0, "%s: bad sizes", who);
    if (n == 0) return DC_OK;  // an empty tensor has a null pointer
    DC_REQUIRE(keys && books && codes, "%s: null pointer", who);
    const int ds = hd / m;
    DC_REQUIRE(ds == 2 || ds == 4 || ds == 8 || ds == 16, "%s: %d columns per subspace unsupported (2, 4, 8 or 16)", who, ds);
    DC_REQUIRE(n_centroids >= 1 && n_centroids <= 256, "%s: %d centroids unsupported (1 to 256)", who, n_centroids);
    const int align = ds * 2 < 16 ? ds * 2 : 16;  // bytes of a key's columns read at a time
    DC_REQUIRE(((uintptr_t)keys) % align == 0 && key_stride >= hd && (key_stride * 2) % align == 0,
               "%s: keys must be %d-byte aligned, rows included", who, align);
    DC_REQUIRE((((uintptr_t)codes) & 3u) == 0 && code_stride >= m, "%s: codes must be 4-byte aligned, rows of at least m bytes", who);
    EncGrid g;
    DC_REQUIRE(plan_encode(m, enc_subs(ds), n, &g), "%s: grid too large", who);
    const dim3 grid((unsigned)g.blocks);
    hipStream_t st = (hipStream_t)stream;
#define DC_LAUNCH_ENC(DS)                                                                                            \
    hipLaunchKernelGGL(pq_encode_kernel<DS>, grid, dim3(enc_threads(DS)), 0, st, (const uint16_t *)keys, key_stride, n, books, \
                       codes, code_stride, m, n_centroids, g)
    if (ds == 2) DC_LAUNCH_ENC(2);
    else if (ds == 4) DC_LAUNCH_ENC(4);
    else if (ds == 8) DC_LAUNCH_ENC(8);
    else DC_LAUNCH_ENC(16);
#undef DC_LAUNCH_ENC
    DC_CHECK_LAUNCH(who);
    return DC_OK;
}

extern "C" int dc_pq_build_lut(const void *q, const float *books, float *lut, int n_b, int n_h,
                               int hd, int m, void *stream) {
    DC_REQUIRE(q && books && lut, "dc_pq_build_lut: null pointer");
    DC_REQUIRE(n_b >= 0 && n_h >= 1 && m >= 1 && hd >= m && hd % m == 0, "dc_pq_build_lut: bad sizes");
    const int64_t blocks = (int64_t)n_b * n_h * m;
    if (blocks == 0) return DC_OK;
    hipLaunchKernelGGL(pq_lut_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t *)q, books, lut, n_h, hd, m);
    DC_CHECK_LAUNCH("dc_pq_build_lut");
    return DC_OK;
}

extern "C" int dc_pq_adc_scan(const uint8_t *codes, const float *lut, float *scores, uint32_t *hist,
                              int n_units, int n_rows, int m, int64_t scores_unit_stride,
                              void *stream) {
    DC_REQUIRE(codes && lut && scores, "dc_pq_adc_scan: null pointer");
    DC_REQUIRE(n_units >= 0 && n_rows >= 0, "dc_pq_adc_scan: bad sizes");
    DC_REQUIRE(m == 16 || m == 32, "dc_pq_adc_scan: m = %d subspaces unsupported (16 or 32)", m);
    DC_REQUIRE(dc_aligned16(codes) && dc_aligned16(lut), "dc_pq_adc_scan: pointers must be 16-byte aligned");
    DC_REQUIRE(scores_unit_stride >= n_rows, "dc_pq_adc_scan: scores_unit_stride < n_rows");
    if (n_units == 0 || n_rows == 0) return DC_OK;
    const int64_t bpu = ((int64_t)n_rows + kKeysPerBlock - 1) / kKeysPerBlock;
    DC_REQUIRE(n_units * bpu < (1ll << 31), "dc_pq_adc_scan: grid too large");
    dim3 grid((unsigned)(n_units * bpu));
    hipStream_t st = (hipStream_t)stream;
    if (m == 16)
        hipLaunchKernelGGL(pq_adc_kernel<16>, grid, dim3(kThreads), 0, st, codes, lut, scores, hist,
                           n_rows, scores_unit_stride, (int)bpu);
    else
        hipLaunchKernelGGL(pq_adc_kernel<32>, grid, dim3(kThreads), 0, st, codes, lut, scores, hist,
                           n_rows, scores_unit_stride, (int)bpu);
    DC_CHECK_LAUNCH("dc_pq_adc_scan");
    return DC_OK;
}
