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
// sum of three bf16 values, and |c|^2 / 2 is three more with a factor of one, so the distances of 16
// keys to 16 centroids are one v_mfma_f32_16x16x16_bf16 (16x16x32 from 8 columns on, two of them for
// 16) of exact products with fp32 accumulation.  M = centroids and N = keys, so that a lane holds distances
// of ONE key: lane (q, c) = (lane / 16, lane % 16) supplies part q of a centroid (the three terms,
// then the bias) and the columns of key c (q < 3) or ones (q = 3).  Row 4 q + i of tile 2 p + h is
// centroid 32 p + 8 q + 4 h + i: a lane's eight results of two tiles are eight neighbours, an "octet".
//
// What bounds the kernel is the search for the minimum on the vector ALUs: 256 values per key and
// subspace.  Six instructions per eight values keep the least value and the octet it came from (four
// v_min3, a compare, a select).  At the end the four lanes of a key settle its octet, each lane
// for the key of one of the wave's four groups (an exchange that halves twice), and that lane takes
// the least of the eight in fp32.  200003 keys of 128 columns, 32
// subspaces: 94-98 us, the vector ALUs issuing 88 % of the kernel's time and the matrix cores busy 46 %
// (SQ counters); torch's distance matrices, written to and read from HBM four times over, took 11.8 ms.
// With the tables in plain order (bank conflicts where an octet is settled) it took 115 us, with a search
// of four values at a time 120 us.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The upper halves of the three words sum up to x: 8 + 8 + 8 bits of its mantissa.
__device__ __forceinline__ void split3(float x, uint32_t &a, uint32_t &b, uint32_t &c) {
    a = __float_as_uint(x) & 0xffff0000u;
    const float r = x - __uint_as_float(a);
    b = __float_as_uint(r) & 0xffff0000u;
    c = __float_as_uint(r - __uint_as_float(b));
}

constexpr int kEncGroups = 4;                              // groups of 16 keys per wave: one per quarter of its lanes
constexpr int kEncKeys = kThreads / 64 * 16 * kEncGroups;  // keys per block
constexpr int kEncSubs = 4;                                // subspaces per block: their codes leave as one word

// (At least two waves per SIMD asked for: with up to 256 registers the compiler leaves the results of the
// matrix instructions in vector registers; with more it moves each through an accumulation register,
// one instruction per value, which is what the search costs.)
template <int DS>
__global__ __launch_bounds__(kThreads, DS <= 4 ? 4 : 2) void pq_encode_kernel(
    const uint16_t *__restrict__ keys, int64_t key_stride, int64_t n, const float *__restrict__ books,
    uint8_t *__restrict__ codes, int64_t code_stride, int m, int nc) {
    constexpr int KL = DS <= 4 ? 4 : 8;         // operand elements per lane and instruction
    constexpr int KW = KL / 2;                   // the same in words
    constexpr int PARTS = DS <= 8 ? 1 : DS / 8;  // instructions per tile
    constexpr int XW = (DS + 1) / 2;             // words of a key's columns
    // [tile][q][row][word]: a wave's operand is one stretch
    __shared__ __align__(16) uint32_t s_a[PARTS][256 * 4 * KW];
    // Centroid i of an octet sits at place i ^ (octet & 7) of it, its half norm at i ^ 2 (octet / 8): lanes that
    // look at the same i of different octets read different banks.
    __shared__ __align__(16) float s_c[256 * DS];
    __shared__ __align__(16) float s_half[256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q = lane >> 4, c = lane & 15;
    // The blocks that read the same keys (a few columns each, of lines they share) are numbered 8 apart:
    // they run on one XCD at about the same time and find the lines in its L2.
    const int n_y = (m + kEncSubs - 1) / kEncSubs;
    const int xcd = blockIdx.x % 8, turn = blockIdx.x / 8;
    const int64_t kblk = (int64_t)(turn / n_y) * 8 + xcd;
    const int sub0 = (turn % n_y) * kEncSubs;
    const int n_sub = m - sub0 < kEncSubs ? m - sub0 : kEncSubs;
    const int64_t key0 = kblk * kEncKeys + wave * (16 * kEncGroups);
    if (kblk * kEncKeys >= n) return;  // the grid is a whole number of eights
    const uint16_t *kp[kEncGroups];
#pragma unroll
    for (int g = 0; g < kEncGroups; ++g) {
        int64_t k = key0 + g * 16 + c;
        k = k < n ? k : n - 1;
        kp[g] = keys + k * key_stride;
    }
    float cen[DS];  // this thread's centroid of a subspace
    auto load_centroid = [&](int sub) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < DS; ++d) cen[d] = 0.f;
        if (tid < nc) {
            const float *p = books + ((int64_t)sub * nc + tid) * DS;
#pragma unroll
            for (int d = 0; d < DS; ++d) cen[d] = p[d];
        }
    };
    uint32_t xw[kEncGroups][XW], xn[kEncGroups][XW];
    auto load_keys = [&](int sub, uint32_t(&x)[kEncGroups][XW]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) {
            const uint16_t *p = kp[g] + sub * DS;
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
    // where this thread's centroid sits among the tiles' rows
    const int tile = 2 * (tid >> 5) + ((tid >> 2) & 1), row = 4 * ((tid >> 3) & 3) + (tid & 3);
    const int c_slot = (tid & ~7) | ((tid ^ (tid >> 3)) & 7), half_slot = (tid & ~7) | ((tid ^ (2 * (tid >> 6))) & 7);
    uint32_t word = 0u;  // the codes of key key0 + lane
    load_centroid(sub0);
    load_keys(sub0, xw);
    for (int s = 0; s < n_sub; ++s) {
        // stage the subspace: the negated centroid in three bf16 parts, half its squared norm in three
        float half = 0.f;
#pragma unroll
        for (int d = 0; d < DS; ++d) half = fmaf(cen[d], cen[d], half);
        half = tid < nc ? 0.5f * half : INFINITY;  // a centroid that does not exist is never the nearest, of no key
        if (s > 0) __syncthreads();               // the last subspace's tables are no longer read
        s_half[half_slot] = half;
#pragma unroll
        for (int d = 0; d < DS; ++d) s_c[c_slot * DS + d] = cen[d];
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
            uint32_t e[4][KL];  // bf16 values in the upper halves
#pragma unroll
            for (int j = 0; j < KL; ++j) {
                e[0][j] = e[1][j] = e[2][j] = e[3][j] = 0u;
                if (p * KL + j < DS) split3(-cen[p * KL + j < DS ? p * KL + j : 0], e[0][j], e[1][j], e[2][j]);
            }
            if (p == 0) split3(half, e[3][0], e[3][1], e[3][2]);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int w = 0; w < KW; ++w)
                    s_a[p][((tile * 4 + r) * 16 + row) * KW + w] = __builtin_amdgcn_perm(e[r][2 * w + 1], e[r][2 * w], 0x07060302u);
        }
        __syncthreads();
        // the keys' operands: the columns for the lanes of the centroid's parts, ones for the bias
        uint32_t b[kEncGroups][PARTS][KW];
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g)
#pragma unroll
            for (int p = 0; p < PARTS; ++p)
#pragma unroll
                for (int w = 0; w < KW; ++w) {
                    const int xi = p * KW + w;
                    const uint32_t x = xi < XW ? xw[g][xi < XW ? xi : 0] : 0u;
                    const uint32_t one = p != 0 ? 0u : (w == 0 ? 0x3f803f80u : (w == 1 ? 0x00003f80u : 0u));
                    b[g][p][w] = q < 3 ? x : one;
                }
        if (s + 1 < n_sub) {  // the next subspace's centroids and columns are on the way meanwhile
            load_centroid(sub0 + s + 1);
            load_keys(sub0 + s + 1, xn);
        }
        float best[kEncGroups];
        uint32_t pair[kEncGroups];
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g) {
            best[g] = INFINITY;
            pair[g] = 0u;
        }
        uint32_t aw[2][PARTS][KW], an[2][PARTS][KW];
        auto load_pair = [&](int t2, uint32_t(&dst)[2][PARTS][KW]) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < PARTS; ++p) {
                    const uint32_t *src = &s_a[p][(((2 * t2 + h) * 4 + q) * 16 + c) * KW];
                    if constexpr (KW == 2) {
                        const uint2 v = *reinterpret_cast<const uint2 *>(src);
                        dst[h][p][0] = v.x, dst[h][p][1] = v.y;
                    } else {
                        const uint4 v = *reinterpret_cast<const uint4 *>(src);
                        dst[h][p][0] = v.x, dst[h][p][1] = v.y, dst[h][p][2] = v.z, dst[h][p][3] = v.w;
                    }
                }
        };
        load_pair(0, an);
#pragma unroll 2
        for (int t2 = 0; t2 < 8; ++t2) {
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int p = 0; p < PARTS; ++p)
#pragma unroll
                    for (int w = 0; w < KW; ++w) aw[h][p][w] = an[h][p][w];
            load_pair((t2 + 1) & 7, an);  // the next pair of tiles is on the way
            // all products first, then each step of the search for all groups: a result is a dozen
            // cycles away from its instruction, a compare's mask two from its reader
            f32x4 d[kEncGroups][2];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int g = 0; g < kEncGroups; ++g) {
                    d[g][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int p = 0; p < PARTS; ++p) {
                        if constexpr (KW == 2) {
                            const uint2 av = make_uint2(aw[h][p][0], aw[h][p][1]), bv = make_uint2(b[g][p][0], b[g][p][1]);
                            d[g][h] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, av),
                                                                                __builtin_bit_cast(s16x4, bv), d[g][h], 0, 0, 0);
                        } else {
                            const uint4 av = make_uint4(aw[h][p][0], aw[h][p][1], aw[h][p][2], aw[h][p][3]);
                            const uint4 bv = make_uint4(b[g][p][0], b[g][p][1], b[g][p][2], b[g][p][3]);
                            d[g][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av),
                                                                              __builtin_bit_cast(bf16x8, bv), d[g][h], 0, 0, 0);
                        }
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
            float v[kEncGroups];
            bool less[kEncGroups];
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(d[g][0][0], d[g][0][1]), d[g][0][2]);
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], d[g][0][3]), d[g][1][0]);
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], d[g][1][1]), d[g][1][2]);
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) v[g] = fminf(fminf(v[g], d[g][1][3]), best[g]);
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) less[g] = v[g] < best[g];
#pragma unroll
            for (int g = 0; g < kEncGroups; ++g) {
                pair[g] = less[g] ? (uint32_t)t2 : pair[g];
                best[g] = v[g];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // The four lanes of a key hold its least value over their octets each.  Lanes q and q ^ 2 exchange
        // two groups, then q and q ^ 1 one of the two that are left: lane q ends with group q.
        // (Equal values: the lower octet.)
        auto lesser = [](float &v, uint32_t &o, float v2, uint32_t o2) __attribute__((always_inline)) {
            const bool take = v2 < v || (v2 == v && o2 < o);
            v = take ? v2 : v;
            o = take ? o2 : o;
        };
        const bool up2 = (q & 2) != 0, up1 = (q & 1) != 0;
        float v2[2];
        uint32_t o2[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            v2[i] = up2 ? best[2 + i] : best[i];
            o2[i] = (up2 ? pair[2 + i] : pair[i]) * 4u + (uint32_t)q;
            const float vs = up2 ? best[i] : best[2 + i];
            const uint32_t os = (up2 ? pair[i] : pair[2 + i]) * 4u + (uint32_t)q;
            lesser(v2[i], o2[i], __shfl_xor(vs, 32, 64), (uint32_t)__shfl_xor((int)os, 32, 64));
        }
        float v1 = up1 ? v2[1] : v2[0];
        uint32_t octet = up1 ? o2[1] : o2[0];
        lesser(v1, octet, __shfl_xor(up1 ? v2[0] : v2[1], 16, 64), (uint32_t)__shfl_xor((int)(up1 ? o2[0] : o2[1]), 16, 64));
        // the least of the octet, in fp32, for key key0 + lane
        uint32_t x[XW];
#pragma unroll
        for (int w = 0; w < XW; ++w) {
            const uint32_t x0 = up1 ? xw[1][w] : xw[0][w], x1 = up1 ? xw[3][w] : xw[2][w];
            x[w] = up2 ? x1 : x0;
        }
        float least = 0.f;
        uint32_t id = 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float dist = s_half[octet * 8u + ((uint32_t)i ^ (2u * (octet >> 3)))];
            const float *cp = s_c + (octet * 8u + ((uint32_t)i ^ (octet & 7u))) * DS;
#pragma unroll
            for (int w = 0; w < XW; ++w) {
                dist = fmaf(-dc_bf16_lo(x[w]), cp[2 * w], dist);
                dist = fmaf(-dc_bf16_hi(x[w]), cp[2 * w + 1], dist);
            }
            const bool take = i == 0 || dist < least;
            least = take ? dist : least;
            id = take ? (uint32_t)i : id;
        }
        word |= (octet * 8u + id) << (8 * s);
#pragma unroll
        for (int g = 0; g < kEncGroups; ++g)
#pragma unroll
            for (int w = 0; w < XW; ++w) xw[g][w] = xn[g][w];
    }
    const int64_t k = key0 + lane;
    if (k >= n) return;
    uint8_t *dst = codes + k * code_stride + sub0;
    if (n_sub == kEncSubs && (code_stride & 3) == 0) {
        *reinterpret_cast<uint32_t *>(dst) = word;
    } else {
        for (int s = 0; s < n_sub; ++s) dst[s] = (uint8_t)(word >> (8 * s));
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
    const int64_t blocks = ((n + kEncKeys - 1) / kEncKeys + 7) / 8 * 8 * ((m + kEncSubs - 1) / kEncSubs);
    DC_REQUIRE(blocks < (1ll << 31), "%s: grid too large", who);
    const dim3 grid((unsigned)blocks);
    hipStream_t st = (hipStream_t)stream;
#define DC_LAUNCH_ENC(DS)                                                                                            \
    hipLaunchKernelGGL(pq_encode_kernel<DS>, grid, dim3(kThreads), 0, st, (const uint16_t *)keys, key_stride, n, books, \
                       codes, code_stride, m, n_centroids)
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
