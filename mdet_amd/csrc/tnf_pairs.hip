// All-pairs TNF graph on gfx950: the thresholded, per-row-capped edge list of
// gen_tnf_graph (cuda/Cuda2.cu:861-970) with the pair model of
// cal_tnf_pre_dist_d (cuda/Cuda2.cu:192-241).
//
// Pipeline (one mdet_tnf_edges call):
//   prep     per-contig: log-size -> Chebyshev coordinate, range check; the
//            row order and the rows' projection on 28 directions (tnf_order.hip);
//            for the Gram modes the TNF rows in BF16/FP16, K padded 136 -> 144,
//            in MFMA fragment order.  R = max over the length range of the edge
//            distance threshold.
//   scan     (k_box_scan) which 32 x 32 tiles of the upper triangle can hold a
//            pair within R: the gap of the tiles' boxes in the projection, then
//            MFMA products of the projected rows, a lower bound of every pair's
//            distance, with the threshold folded into K; small inputs skip it
//            and take every tile.
//            LEARNED (k_tile_scan): products of the TNF rows over the pairs of
//            cluster pairs chosen by the learned embeddings (tnf_ivf.hip).
//   select survivors of the listed tiles
//              EXACT_F32   FP32 sum of squared differences of every pair
//                          (k_tile_f32), d < R
//              *_REFINE    Gram d^2 = |a|^2 + |b|^2 - 2 a.b on MFMA
//                          (v_mfma_f32_32x32x16_{bf16,f16}), FP32 accumulate
//                          (k_tile_gram), d < R + the rounding of the rows
//   refine   (k_tile_refine) per survivor: FP32 sum of squared differences,
//            FP32 model via the Chebyshev form; a pair whose FP32 preProb lies
//            within EPS of the threshold (or whose model-1 value lies within EPS
//            of ln 9, where the model switches) is decided by the FP64
//            tie-breaker, which repeats the reference's device arithmetic
//            operation by operation.  Output: candidates (i, j, preProb).
//   select   candidates -> per-row lists (both endpoints) -> per row the
//            max_edges largest preProb (ties of FP32 values within 2*EPS of
//            the cut are re-ranked in FP64) -> edges i < j, sorted.
// Every pass before the refinement only has to keep a superset, so every mode
// returns the same edge set; the modes differ in the arithmetic of the pairs
// that the scan's bound does not rule out.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>
#include <vector>

#include "hip_common.h"
#include "ivf.h"
#include "model_tables.h"
#include "order.h"
#include "pass_lists.h"
#include "scan_spans.h"
#include "tnf_tables.h"

namespace {

using mdet::ITEM_TRI;
using mdet::PROJ_D;
using mdet::PROJ_KS;
constexpr int NT = 136;
constexpr int KS = 9;    // MFMA k-steps of 16 for TNF rows (K padded to 144)
constexpr int KS_E = 3;  // k-steps for 32-dimensional embeddings (K padded to 48)
constexpr float FLOOR32 = (float)MODEL_FLOOR_PREPROB;
// Bound on |preProb_fp32 - preProb_fp64| used for the tie band.  Measured
// errors of the FP32 evaluator are ~1e-5 (tests check < EPS/8).
constexpr float EPS_PRE = 2e-3f;
constexpr int SEL_CAP = 4096;  // candidates per row handled in LDS
constexpr int ZONE_CAP = 512;  // ties re-ranked in FP64 per row

__constant__ float c_cheb[4][MODEL_CX][MODEL_CY];

#define E17(a) a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15], a[16]
__constant__ double c_b1[18] = {E17(mdet::kB1), mdet::kB1[17]};
__constant__ double c_c1[18] = {E17(mdet::kC1), mdet::kC1[17]};
__constant__ double c_b2[17] = {E17(mdet::kB2)};
__constant__ double c_c2[19] = {E17(mdet::kC2), mdet::kC2[17], mdet::kC2[18]};
#undef E17

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

struct Cand {
    uint32_t i, j;
    float pre;
    uint32_t flags;  // bit 0: preProb from the FP64 tie-breaker
};
struct Adj {
    uint32_t partner;
    float pre;
};

// ------------------------------------------------------------ FP32 model --
__device__ inline float cheb_eval(int which, const float* Tx, const float* Ty) {
    float acc = 0.f;
#pragma unroll
    for (int p = 0; p < MODEL_CX; ++p) {
        float in = 0.f;
#pragma unroll
        for (int q = 0; q < MODEL_CY; ++q) in = fmaf(c_cheb[which][p][q], Ty[q], in);
        acc = fmaf(in, Tx[p], acc);
    }
    return acc;
}

struct Pre32 {
    float pre;   // full model
    float pre1;  // model 1 alone (decides which model applies)
};

// preProb of a pair from its distance d and the Chebyshev coordinates of the
// two log sizes.  t is increasing in the log size, so min/max commute.
__device__ inline Pre32 model32(float d, float ta, float tb) {
    const float tx = fminf(ta, tb), ty = fmaxf(ta, tb);
    float Tx[MODEL_CX], Ty[MODEL_CY];
    Tx[0] = 1.f;
    Tx[1] = tx;
#pragma unroll
    for (int p = 2; p < MODEL_CX; ++p) Tx[p] = fmaf(2.f * tx, Tx[p - 1], -Tx[p - 2]);
    Ty[0] = 1.f;
    Ty[1] = ty;
#pragma unroll
    for (int q = 2; q < MODEL_CY; ++q) Ty[q] = fmaf(2.f * ty, Ty[q - 1], -Ty[q - 2]);
    const float b1 = cheb_eval(0, Tx, Ty), c1 = cheb_eval(1, Tx, Ty);
    Pre32 r;
    r.pre1 = -fmaf(c1, d, b1);
    r.pre = r.pre1;
    if (r.pre1 <= FLOOR32) {
        const float b2 = cheb_eval(2, Tx, Ty), c2 = cheb_eval(3, Tx, Ty);
        r.pre = fminf(-fmaf(c2, d, b2), FLOOR32);
    }
    return r;
}

__device__ inline float dist2_f32(const float* __restrict__ a, const float* __restrict__ b) {
    const float4* a4 = reinterpret_cast<const float4*>(a);
    const float4* b4 = reinterpret_cast<const float4*>(b);
    float s0 = 0.f, s1 = 0.f;
#pragma unroll 2
    for (int q = 0; q < NT / 4; ++q) {
        float4 x = a4[q], y = b4[q];
        float d0 = x.x - y.x, d1 = x.y - y.y, d2 = x.z - y.z, d3 = x.w - y.w;
        s0 = fmaf(d0, d0, s0);
        s1 = fmaf(d1, d1, s1);
        s0 = fmaf(d2, d2, s0);
        s1 = fmaf(d3, d3, s1);
    }
    return s0 + s1;
}

// ------------------------------------------------------ FP64 tie-breaker --
// Operation-for-operation the device arithmetic of the reference,
// cuda/Cuda2.cu:192-241 compiled with fused multiply-add contraction:
// float differences and squares accumulated in double, every "acc + c*m" of
// the polynomials and "b + c*d" one fma, monomials as plain products.
__device__ inline double dist2_f64(const float* __restrict__ a, const float* __restrict__ b) {
#pragma clang fp contract(off)
    double d = 0;
#pragma unroll 4
    for (int q = 0; q < NT / 4; ++q) {
        const f32x4_t diff = reinterpret_cast<const f32x4_t*>(a)[q] - reinterpret_cast<const f32x4_t*>(b)[q];
        const f32x4_t sq = diff * diff;
        d += (double)sq.x;
        d += (double)sq.y;
        d += (double)sq.z;
        d += (double)sq.w;
    }
    return d;
}

// preProb from the squared distance.
__device__ double model64_d2(double d2, double r1, double r2) {
#pragma clang fp contract(off)
    const double d = sqrt(d2);
    double lw[19];
    lw[0] = r1 < r2 ? r1 : r2;
    lw[1] = r1 < r2 ? r2 : r1;
    lw[2] = lw[0] * lw[0];
    lw[4] = lw[2] * lw[0];
    lw[6] = lw[4] * lw[0];
    lw[8] = lw[6] * lw[0];
    lw[10] = lw[8] * lw[0];
    lw[11] = lw[10] * lw[0];
    lw[3] = lw[1] * lw[1];
    lw[5] = lw[3] * lw[1];
    lw[7] = lw[5] * lw[1];
    lw[9] = lw[7] * lw[1];
    lw[12] = lw[0] * lw[1];
    lw[14] = lw[4] * lw[5];
    lw[15] = lw[6] * lw[7];
    lw[16] = lw[8] * lw[9];
    lw[13] = lw[2] * lw[3];
    lw[18] = lw[9] * lw[1];
    double bb = c_b1[0], cc = c_c1[0];
#pragma unroll
    for (int t = 1; t < 18; ++t) {
        bb = __builtin_fma(c_b1[t], lw[t - 1], bb);
        cc = __builtin_fma(c_c1[t], lw[t - 1], cc);
    }
    double pre = -__builtin_fma(cc, d, bb);
    if (pre <= MODEL_FLOOR_PREPROB) {
        // b2 terms use lw[0..10], lw[18], lw[13..16]; c2 adds lw[11], lw[12]
        const int ib[16] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 18, 13, 14, 15, 16};
        const int ic[18] = {0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 18, 11, 12, 13, 14, 15, 16};
        bb = c_b2[0];
#pragma unroll
        for (int t = 1; t < 17; ++t) bb = __builtin_fma(c_b2[t], lw[ib[t - 1]], bb);
        cc = c_c2[0];
#pragma unroll
        for (int t = 1; t < 19; ++t) cc = __builtin_fma(c_c2[t], lw[ic[t - 1]], cc);
        pre = -__builtin_fma(cc, d, bb);
        if (pre > MODEL_FLOOR_PREPROB) pre = MODEL_FLOOR_PREPROB;
    }
    return pre;
}

__device__ double model64(const float* __restrict__ a, const float* __restrict__ b, double r1, double r2) {
    return model64_d2(dist2_f64(a, b), r1, r2);
}

// Order-preserving maps of floats and doubles to unsigned integers (for
// integer atomics and sorts; NaN is not expected).
__device__ inline uint32_t f2ord(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ inline float ord2f(uint32_t u) { return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u); }
__device__ inline unsigned long long d2ord(double f) {
    unsigned long long u = (unsigned long long)__double_as_longlong(f);
    return (u & 0x8000000000000000ull) ? ~u : (u | 0x8000000000000000ull);
}
__device__ inline double ord2d(unsigned long long u) {
    return __longlong_as_double((long long)((u & 0x8000000000000000ull) ? (u & 0x7fffffffffffffffull) : ~u));
}

// ------------------------------------------------------- wave utilities --
__device__ inline uint32_t lane_id() { return __lane_id(); }

// Inclusive prefix sum over the 64 lanes with DPP moves (no LDS round
// trips): row_shr 1, 2, 4, 8 within each 16-lane row, then row_bcast 15 and
// row_bcast 31 carry the row totals across rows.  All 64 lanes must be active.
__device__ inline uint32_t wave_incl_sum_dpp(uint32_t x) {
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);
    return x;
}

// Rows of the select stage are grouped in buckets of S_BUCKET consecutive
// positions of the scan's row order (a multiple of 64; measured while the rows
// were grouped in memory: at 200k contigs 64 rows selected 5-9% faster than 128,
// and 256 rows 28% slower, as more, shorter blocks balance better).  A bucket of
// 64 rows is also what k_bucket_select's LDS holds.
constexpr int S_BUCKET = 64;
static_assert(S_BUCKET >= 64 && S_BUCKET % 64 == 0, "the row scan gives each lane S_BUCKET / 64 rows");

// The active lanes by key: each lane's leader (the lowest lane with its key),
// rank among them and, in the leader, their number.  All 64 lanes call; the loop
// runs once per distinct key and touches no memory, so that a caller's atomics
// (one by each leader) go out together instead of one round trip per key.
struct KeyGroup {
    int leader;
    uint32_t rank, count;
};
__device__ inline KeyGroup wave_key_groups(uint32_t key, bool active) {
    KeyGroup g{-1, 0, 0};
    uint64_t pending = __ballot(active);
    const uint32_t lane = lane_id();
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const uint32_t k = (uint32_t)__builtin_amdgcn_readlane((int)key, leader);
        const uint64_t same = __ballot(active && key == k);
        if (active && key == k)
            g = KeyGroup{leader, (uint32_t)__popcll(same & ((1ull << lane) - 1ull)), (uint32_t)__popcll(same)};
        pending &= ~same;
    }
    return g;
}

// The same without the slots: counter[key] += lanes holding key (no return
// value is waited for).
__device__ inline void wave_aggregated_count(uint32_t* counter, uint32_t key, bool active) {
    uint64_t pending = __ballot(active);
    const uint32_t lane = lane_id();
    while (pending) {
        const int leader = __ffsll((long long)pending) - 1;
        const uint32_t k = __shfl(key, leader, 64);
        const uint64_t same = __ballot(active && key == k);
        if ((int)lane == leader) atomicAdd(&counter[k], (uint32_t)__popcll(same));
        pending &= ~same;
    }
}

// --------------------------------------------------------------- prep ----
// Chebyshev coordinate of each log size, domain check, min/max.  mm (zero
// before): [0] complement of the smallest log size's bits, [1] largest log
// size's bits, [2] count outside the domain.
__global__ void k_prep_rows(const double* __restrict__ ls, uint32_t n, float* __restrict__ tvec,
                            unsigned long long* __restrict__ mm) {
    __shared__ unsigned long long smin[4], smax[4];
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long lo = 0ull, hi = 0ull;
    bool bad = false;
    if (i < n) {
        const double v = ls[i];
        // domain: [log10 1500, log10 500000] up to rounding of the caller's log10
        bad = !(v >= MODEL_XLO - 1e-12 && v <= MODEL_XHI + 1e-12);
        tvec[i] = (float)((2.0 * v - (MODEL_XLO + MODEL_XHI)) / (MODEL_XHI - MODEL_XLO));
        if (v > 0) {
            hi = (unsigned long long)__double_as_longlong(v);
            lo = ~hi;
        }
    }
    const uint64_t nbad = __ballot(bad);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        lo = max(lo, (unsigned long long)__shfl_xor(lo, off, 64));
        hi = max(hi, (unsigned long long)__shfl_xor(hi, off, 64));
    }
    const uint32_t w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smin[w] = lo;
        smax[w] = hi;
        if (nbad) atomicAdd(&mm[2], (unsigned long long)__popcll(nbad));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t k = 1; k < blockDim.x / 64; ++k) {
            lo = max(lo, smin[k]);
            hi = max(hi, smax[k]);
        }
        atomicMax(&mm[0], lo);
        atomicMax(&mm[1], hi);
    }
}

__device__ inline uint16_t to_bf16_rne(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// FP32 rows in cluster order for the exact cover (position s holds contig
// perm[s]; zero rows past n).  One wave per row.
__global__ __launch_bounds__(256) void k_sort_rows(const float* __restrict__ tnf, const uint32_t* __restrict__ perm,
                                                   uint32_t n, uint32_t n_pad, float* __restrict__ tnfs) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t s = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (s >= n_pad) return;
    const bool real = s < n;
    const size_t src = real ? (size_t)perm[s] * NT : 0;
    float* dst = tnfs + (size_t)s * NT;
    for (uint32_t c = lane; c < (uint32_t)NT; c += 64) dst[c] = real ? tnf[src + c] : 0.f;
}

// Low-precision rows in MFMA fragment order.  For the 32-row tile t, k-step
// ks and lane l (row t*32 + l%32, k = 16*ks + 8*(l/32) .. +8), the 16 bytes
// sit at element offset ((t*9 + ks)*64 + l)*8: one coalesced 1 KiB load per
// wave serves an A or B operand of v_mfma_f32_32x32x16.
//
// K slots 136..143 carry the threshold so that the MFMA itself returns
//   acc = a.b - h_i - h_j,   h = |a~|^2/2 - R2/4,
// and "d~^2 < R2" is "acc > 0".  h is split into three pieces of the low
// format (hh + hm + hl = h to ~2^-24 relative), multiplied by exact ones:
//   column (B) role: slots 136..138 = 1, slots 139..141 = -hh, -hm, -hl
//   row (A) role:    slots 136..138 = -hh, -hm, -hl, slots 139..141 = 1
// The B-role rows are the main array; the A-role variant of the last k-step
// half (k = 136..143) is kept separately (one uint4 per row).
template <bool BF16>
__device__ inline uint16_t to_low(float v) {
    if (BF16) return to_bf16_rne(v);
    _Float16 x = (_Float16)v;
    return __builtin_bit_cast(uint16_t, x);
}
template <bool BF16>
__device__ inline float from_low(uint16_t h) {
    if (BF16) return from_bf16(h);
    return (float)__builtin_bit_cast(_Float16, h);
}
__device__ inline uint4 pack8(const uint16_t* h) {
    uint4 w;
    w.x = h[0] | ((uint32_t)h[1] << 16);
    w.y = h[2] | ((uint32_t)h[3] << 16);
    w.z = h[4] | ((uint32_t)h[5] << 16);
    w.w = h[6] | ((uint32_t)h[7] << 16);
    return w;
}

// Rows of D values (D = 136 TNF columns, or 32 embedding dimensions) padded
// to KSX k-steps of 16; the threshold slots are k = D .. D+5.  Every pair with
// |a - b| < R must pass, and |a~ - b~| <= |a - b| + e_a + e_b with e = |x - x~|,
// so each row carries its own share s = 2 (R/2 + e)^2 (+ a slack for the FP32
// accumulation, below 3e-5 for unit rows): s_a + s_b >= (R + e_a + e_b)^2,
// h = |x~|^2/2 - s/2, and acc > 0 iff |a~ - b~|^2 < s_a + s_b.
// TNF rows (EMB = false): e as the row's rounding gives it (~0.3 of the unit
// roundoff u times the norm: with u|x| for every row 0.7% more survivors, and
// twice the tiles the scan has to list for them).  Embeddings (EMB): e = u|x|.
// One block per 32-row tile: the rows (perm: position -> row; null: itself)
// pass through LDS once, so reads and the 16-byte fragment writes are both
// whole lines.
// With err: no share, acc = -|a~ - b~|^2 / 2 of the pair, err[row] = e; rows
// that hold a value that is not finite become padding with err = NaN, and a
// finite row of squared norm above PLAIN_NORM2 sets *outside.
constexpr float GRAM_SLACK = 5e-5f;
constexpr float PLAIN_NORM2 = 1.05f;

template <bool BF16, int D, int KSX, bool EMB = false>
__global__ __launch_bounds__(256) void k_prep_lowp(const float* __restrict__ x, const uint32_t* __restrict__ perm,
                                                   uint32_t n, float R, uint4* __restrict__ frag,
                                                   uint4* __restrict__ frag_a, float* __restrict__ err = nullptr,
                                                   uint32_t* __restrict__ outside = nullptr) {
    static_assert(D + 6 <= 16 * KSX && D % 8 == 0, "no room for the threshold slots");
    constexpr int STR = D + 4;
    __shared__ __align__(16) float X[32][STR];
    __shared__ uint32_t H[32][3];  // the pieces of each row's h
    const uint32_t tid = threadIdx.x, t = blockIdx.x;
    for (uint32_t e = tid; e < 32 * (D / 4); e += 256) {
        const uint32_t r = e / (D / 4), q = e % (D / 4), pos = t * 32 + r;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (pos < n) v = reinterpret_cast<const float4*>(x + (size_t)(perm ? perm[pos] : pos) * D)[q];
        *reinterpret_cast<float4*>(&X[r][4 * q]) = v;
    }
    __syncthreads();
    {  // eight lanes a row: squared norms of the rounded and the given values
        const uint32_t r = tid >> 3, s = tid & 7, pos = t * 32 + r;
        float part = 0.f, norm2 = 0.f, err2 = 0.f, nonfinite = 0.f;
        for (uint32_t k = s; k < (uint32_t)D; k += 8) {
            const float v = X[r][k], back = from_low<BF16>(to_low<BF16>(v));
            part = fmaf(back, back, part);
            norm2 = fmaf(v, v, norm2);
            err2 = fmaf(v - back, v - back, err2);
            nonfinite += v * 0.f;
        }
#pragma unroll
        for (int off = 4; off >= 1; off >>= 1) {
            part += __shfl_xor(part, off, 64);
            norm2 += __shfl_xor(norm2, off, 64);
            err2 += __shfl_xor(err2, off, 64);
            nonfinite += __shfl_xor(nonfinite, off, 64);
        }
        const bool pad = pos >= n || (err && nonfinite != 0.f);
        if (pad)
            for (uint32_t k = s; k < (uint32_t)D; k += 8) X[r][k] = 0.f;
        if (s == 0) {
            // padding rows get a large finite h (the split of +inf would be NaN)
            const float big = BF16 ? 1e30f : 6.0e4f;
            const float u = BF16 ? 1.0f / 256.0f : 1.0f / 2048.0f;
            const float e = EMB ? u * 1.0001f * sqrtf(norm2) : 1.001f * sqrtf(err2) + 1e-6f, half_r = 0.5f * R + e;
            const float share =
                err ? 0.f : 2.0f * half_r * half_r + (EMB ? 1e-5f : GRAM_SLACK) * (norm2 + 1.0f);
            float rem = pad ? big : fmaf(0.5f, part, -0.5f * share);
            if (err) {
                err[pos] = pad ? __builtin_nanf("") : e;
                if (!pad && norm2 > PLAIN_NORM2) *outside = 1u;
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const uint16_t p = to_low<BF16>(rem);
                H[r][q] = p;
                rem = rem - from_low<BF16>(p);
            }
        }
    }
    __syncthreads();
    const uint16_t one = to_low<BF16>(1.f);
    for (uint32_t e = tid; e < (uint32_t)KSX * 64; e += 256) {
        const uint32_t ks = e >> 6, l = e & 63, r = l & 31, k0 = 16 * ks + 8 * (l >> 5);
        uint16_t hb[8], ha[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            uint16_t v = 0, va = 0;
            if (k0 < (uint32_t)D) {  // whole octets of values (D is a multiple of 8)
                v = va = to_low<BF16>(X[r][k0 + i]);
            } else if (k0 == (uint32_t)D) {
                if (i < 3) {  // column role: 1, row role: -h pieces
                    v = one;
                    va = (uint16_t)H[r][i] ^ 0x8000u;
                } else if (i < 6) {  // column role: -h pieces, row role: 1
                    v = (uint16_t)H[r][i - 3] ^ 0x8000u;
                    va = one;
                }
            }
            hb[i] = v;
            ha[i] = va;
        }
        frag[((size_t)t * KSX + ks) * 64 + l] = pack8(hb);
        if (ks == KSX - 1) frag_a[(size_t)t * 64 + l] = pack8(ha);
    }
}

// ------------------------------------------------------------- tile scan --
// The first pass over the pairs: which 32 x 32 tiles hold a pair within the
// radius at all.  The exhaustive modes take k_box_scan (below), the learned
// filter k_tile_scan: block = 4 waves of RT row tiles each (held in registers for
// the whole column sweep of an item); columns stream through LDS CT tiles a
// step in fragment order, double buffered and filled by
// global_load_lds_dwordx4 (no register staging).  With the threshold folded
// into K the test of a pair is "acc > 0"; a tile with one goes to the list,
// which the second pass works off.  Nothing else leaves the kernel, so its cost
// is the MFMAs and the maximum tree.
//   KSX = 9, RT = 2, CT = 4: cluster pairs and full rows of the learned
//     filter, on the TNF rows themselves.
//   KSX = 3, RT = 2, CT = 4: the embedding radius of the learned filter.
// Both in BF16.  Measured and dropped in the full Gram form of this kernel (KSX =
// 9 over all pairs): B reads ahead by hand, ping-pong accumulators (one wave per
// SIMD), 8-wave blocks, s_setprio around the chains.
constexpr uint32_t SCAN_WAVES = 4;
constexpr uint32_t scan_rows(int rt) { return 32u * rt * SCAN_WAVES; }  // rows per item of row blocks
constexpr int PROJ_RT = 4;  // row tiles a wave of the projected scan
constexpr int GRAM_RT = 2, GRAM_CT = 4;
static_assert(scan_rows(GRAM_RT) == mdet::ITEM_ROWS, "cluster items hold one block's rows");
// Scan item: (r_lo, r_hi, c_lo, c_hi | ITEM_TRI) = pairs of row positions
// [r_lo, r_hi) and column positions [c_lo, c_hi), only i < j if ITEM_TRI;
// r_hi - (r_lo & ~31) <= the block's rows.  The fragment arrays must hold
// whole column steps from (c_lo & ~31) up to c_hi.

template <bool BF16>
__device__ inline f32x16_t mfma32(uint4 a, uint4 b, f32x16_t c) {
    if (BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                       c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                  0, 0);
}

// One step's column fragments (CT tiles x KSX k-steps x 64 lanes of 16 bytes)
// into LDS: each wave copies 1 KiB chunks, chunk m * 4 + wave.
template <int KSX, int CT>
__device__ inline void issue_btile(const uint4* __restrict__ frag, uint32_t c0, uint4* lds, int tid, int wave) {
    constexpr int STEP_U4 = CT * KSX * 64, THREADS = 64 * SCAN_WAVES;
    static_assert(STEP_U4 % 64 == 0, "whole 1 KiB chunks");
    const uint4* src = frag + (size_t)(c0 / 32) * KSX * 64;
#pragma unroll
    for (int m = 0; m < (STEP_U4 + THREADS - 1) / THREADS; ++m)
        if (STEP_U4 % THREADS == 0 || THREADS * m + 64 * wave < STEP_U4)
            __builtin_amdgcn_global_load_lds((const void*)(src + THREADS * m + tid),
                                             (__attribute__((address_space(3))) void*)(lds + THREADS * m + 64 * wave),
                                             16, 0, 0);
}

// Orders the LDS writes of a wave before its following LDS reads (the lanes
// of one wave execute each LDS instruction together and in program order; the
// fences keep the compiler from moving accesses across).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Squared distances of 64 pairs of rows in FP64, the sums in the order of
// dist2_f64: one pair a lane (all 64 lanes call; i, j < n also where the result
// is not used).  The rows pass through LDS 32 floats at a time, read eight lanes
// a row: whole 128-byte pieces instead of one 4-byte word of 64 rows per load.
// A row i that the pair before has too is loaded once.  4.1M edges of 47,111
// contigs (2.2 GB of rows j from the last-level cache, 7.8 TB/s): 287 us; one
// row a lane took 497 us, pieces of 16 floats (twice the waves, half lines)
// 341 us.  lds: DIST_LDS floats of the wave's own.
constexpr int DIST_STR = 36;  // floats between rows: 16 lanes' 16-byte reads cover all banks
constexpr int DIST_LDS = 128 * DIST_STR;
constexpr int DIST_WAVES = 2;

__device__ inline double wave_dist2_f64(const float* __restrict__ tnf, uint32_t i, uint32_t j, float* lds) {
#pragma clang fp contract(off)
    const uint32_t lane = lane_id(), sub = lane & 7, r0 = lane >> 3;
    const uint32_t before = (uint32_t)__shfl_up((int)i, 1, 64);  // by all lanes: an inactive one gives 0
    const uint64_t first = __ballot(lane == 0 || i != before);
    const uint32_t lead = 63 - __builtin_clzll(first & (~0ull >> (63 - lane)));
    uint32_t id[16];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        id[m] = (uint32_t)__shfl((int)i, (int)(r0 + 8 * m), 64);
        id[m + 8] = (uint32_t)__shfl((int)j, (int)(r0 + 8 * m), 64);
    }
    f32x4_t v[16];
    auto load = [&](uint32_t k) {
#pragma unroll
        for (int m = 0; m < 16; ++m)
            if (m >= 8 || (first >> (r0 + 8 * m) & 1))
                v[m] = *reinterpret_cast<const f32x4_t*>(tnf + (size_t)id[m] * NT + k + 4 * sub);
    };
    auto store = [&]() {
#pragma unroll
        for (int m = 0; m < 16; ++m)
            if (m >= 8 || (first >> (r0 + 8 * m) & 1))
                *reinterpret_cast<f32x4_t*>(lds + (r0 + 8 * m) * DIST_STR + 4 * sub) = v[m];
    };
    load(0);
    const f32x4_t* a = reinterpret_cast<const f32x4_t*>(lds + lead * DIST_STR);
    const f32x4_t* b = reinterpret_cast<const f32x4_t*>(lds + (64 + lane) * DIST_STR);
    double d = 0;
    auto add = [&](int q) {
        const f32x4_t diff = a[q] - b[q], sq = diff * diff;
        d += (double)sq.x;
        d += (double)sq.y;
        d += (double)sq.z;
        d += (double)sq.w;
    };
#pragma unroll 1
    for (uint32_t c = 0; c < 4; ++c) {
        store();
        wave_sync();
        if (c < 3 || sub < 2) load(32 * (c + 1));  // the last piece: 8 floats
#pragma unroll
        for (int q = 0; q < 8; ++q) add(q);
        wave_sync();
    }
    if (sub < 2) store();
    wave_sync();
    add(0);
    add(1);
    wave_sync();
    return d;
}

// Tile list: entries (row tile, column tile, item, 0); the counter keeps
// counting past the capacity so that the host learns the size needed.  A wave
// stages its tiles in LDS over all its items and appends 64 at a time: a
// returning atomic on one address costs ~15 ns of the whole chip's time, so a
// flush per item (240k items at 1M contigs) bound the scan: 24.6 ms.
struct TileList {
    uint4* buf;
    unsigned long long* cnt;
    unsigned long long cap;
};
constexpr uint32_t TILE_STAGE = 64;

__device__ inline unsigned long long lane0_u64(unsigned long long v) {
    return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), 0) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, 0);
}

__device__ inline void tiles_flush(const TileList& o, const uint4* stage, uint32_t& n, int lane) {
    if (n == 0) return;
    unsigned long long k = 0;
    if (lane == 0) k = atomicAdd(o.cnt, (unsigned long long)n);
    k = lane0_u64(k);
    wave_sync();
    if ((uint32_t)lane < n && k + lane < o.cap) o.buf[k + lane] = stage[lane];
    wave_sync();
    n = 0;
}

template <int KSX, int RT, int CT>
__device__ __forceinline__ void scan_item(const uint4* __restrict__ frag, const uint4* __restrict__ frag_a,
                                          const uint4 it, const uint32_t item, uint4* B0, uint4* B1,
                                          const int wave, uint4* stage, uint32_t& nstage,
                                          const TileList& out) {
    constexpr int CG = 4 / RT;  // column tiles a pass: 4 independent accumulator chains
    constexpr uint32_t STEP = 32 * CT;
    static_assert(CG >= 1 && CT % CG == 0, "whole passes");
    const uint32_t r_lo = it.x, r_hi = it.y, c_lo = it.z, c_hi = it.w & ~ITEM_TRI;
    const bool tri = (it.w & ITEM_TRI) != 0;
    const uint32_t c_begin = c_lo & ~31u;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t row0 = (r_lo & ~31u) + wave * (32 * RT);  // this wave's rows
    // a wave with no row of the item still takes its share of the column loads
    const bool active = row0 < r_hi;
    const uint32_t t0 = row0 >> 5;
    issue_btile<KSX, CT>(frag, c_begin, B0, tid, wave);
    uint4 a[RT][KSX];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        // row tiles past the item's rows are not in the arrays: the last one stands in (never listed)
        const uint32_t t = min(t0 + rt, (r_hi - 1) >> 5);
#pragma unroll
        for (int ks = 0; ks < KSX - 1; ++ks)
            a[rt][ks] = active ? frag[((size_t)t * KSX + ks) * 64 + lane] : make_uint4(0, 0, 0, 0);
        a[rt][KSX - 1] = active ? frag_a[(size_t)t * 64 + lane] : make_uint4(0, 0, 0, 0);
    }

    auto step = [&](const uint32_t c0, const uint4* B, uint4* next) __attribute__((always_inline)) {
        // The barrier keeps the fill of the other buffer after every wave's
        // reads of it in the step before, and the wait and barrier of the next
        // step keep the reads after every wave's fill.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (c0 + STEP < c_hi) issue_btile<KSX, CT>(frag, c0 + STEP, next, tid, wave);
        // steps wholly left of the wave's rows hold no pair i < j
        if (!active || (tri && c0 + STEP <= row0)) return;
#pragma unroll KSX == 9 ? CT / CG : 1
        for (int p = 0; p < CT / CG; ++p) {
            f32x16_t acc[RT][CG];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int c = 0; c < CG; ++c) acc[rt][c] = f32x16_t{};
            // let the scheduler interleave the B-fragment LDS reads with the
            // MFMA chains (measured 2% faster with KSX = 9)
            if (KSX == 9) __builtin_amdgcn_iglp_opt(0);
#pragma unroll
            for (int ks = 0; ks < KSX; ++ks) {
                uint4 b[CG];
#pragma unroll
                for (int c = 0; c < CG; ++c) b[c] = B[((CG * p + c) * KSX + ks) * 64 + lane];
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int c = 0; c < CG; ++c) acc[rt][c] = mfma32<true>(a[rt][ks], b[c], acc[rt][c]);
            }
            // per-lane maxima of each 32 x 32 tile.  acc > 0.0f exactly when
            // its bits, read as a signed int, are > 0, so the maxima are
            // integer max3 trees (a NaN may list its tile, never a pair).
            int tmax[RT][CG];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int c = 0; c < CG; ++c) {
                    const f32x16_t v = acc[rt][c];
                    int b[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) b[r] = __float_as_int(v[r]);
                    const int m0 = max(max(b[0], b[1]), b[2]), m1 = max(max(b[3], b[4]), b[5]);
                    const int m2 = max(max(b[6], b[7]), b[8]), m3 = max(max(b[9], b[10]), b[11]);
                    const int m4 = max(max(b[12], b[13]), b[14]);
                    tmax[rt][c] = max(max(max(m0, m1), m2), max(max(m3, m4), b[15]));
                }
            int hmax = 0;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int c = 0; c < CG; ++c) hmax = max(hmax, tmax[rt][c]);
            if (!__any(hmax > 0)) continue;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int c = 0; c < CG; ++c) {
                    if (!__any(tmax[rt][c] > 0)) continue;
                    const uint32_t tr = t0 + rt, tc = c0 / 32 + CG * p + c;
                    if ((tri && tc < tr) || 32 * tr >= r_hi || 32 * tc >= c_hi) continue;
                    if (lane == 0) stage[nstage] = make_uint4(tr, tc, item, 0u);
                    if (++nstage == TILE_STAGE) tiles_flush(out, stage, nstage, lane);
                }
        }
    };
    // two arrays by name: of one array's halves the compiler cannot tell the
    // fill's from the one read, and waits for the fill before the next reads
    // (1,000,000 contigs: 24.5 against 22.9 ms)
    for (uint32_t c0 = c_begin; c0 < c_hi; c0 += 2 * STEP) {
        step(c0, B0, B1);
        if (c0 + STEP < c_hi) step(c0 + STEP, B1, B0);
    }
}

// One block per item (item_ctr == nullptr: item = blockIdx.x), or persistent
// blocks that take items from a counter until the items are handed out.
template <int KSX, int RT, int CT, int WPE>
__global__ __launch_bounds__(64 * SCAN_WAVES, WPE) void k_tile_scan(const uint4* __restrict__ frag,
                                                                    const uint4* __restrict__ frag_a,
                                                                    const uint4* __restrict__ items, uint32_t nitems,
                                                                    uint32_t* __restrict__ item_ctr, TileList out) {
    __shared__ uint4 B0[CT * KSX * 64], B1[CT * KSX * 64];
    __shared__ uint4 stage_all[SCAN_WAVES][TILE_STAGE];
    __shared__ uint32_t s_item;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t item = blockIdx.x;
    if (item_ctr) {
        if (threadIdx.x == 0) s_item = atomicAdd(item_ctr, 1u);
        __syncthreads();
        item = s_item;
    }
    uint4* stage = stage_all[wave];
    uint32_t nstage = 0;
    while (item < nitems) {
        scan_item<KSX, RT, CT>(frag, frag_a, items[item], item, B0, B1, wave, stage, nstage, out);
        if (!item_ctr) break;
        __syncthreads();  // every wave is done with the buffers and s_item
        if (threadIdx.x == 0) s_item = atomicAdd(item_ctr, 1u);
        __syncthreads();
        item = s_item;
    }
    tiles_flush(out, stage, nstage, threadIdx.x & 63);
}

// Queues of k_box_scan with qbounds (item_order 1): the items come in 8 queues
// [qbounds[q], qbounds[q + 1]), one per XCD: block b serves queue b % 8 (the XCD
// workgroups are dispatched to round-robin) from counter item_ctr[16 q].
constexpr int PF_QUEUES = 8;
constexpr int PF_CTR_STRIDE = 16;  // counters 64 bytes apart

// The first pass of the exhaustive modes: the projected rows (order.h).  Before
// a pair of tiles is multiplied, the gap of their bounding boxes decides whether
// it can hold a close pair at all: a lane takes one column tile against the
// wave's PROJ_RT row tiles (their boxes from scalar loads), 64 column tiles at a
// time, and only the pairs left (10% at 50,000 contigs, 17% at 200,000, 30% at
// 1,000,000) go to MFMA: 2 products and a maximum tree.  Waves work on their own
// (no barrier in the loop): the columns left differ too much for a block to
// stage them together, so each wave reads its column fragments from L1/L2, the
// next ones ahead.  Bound by the box test (~480 instructions per 256 tile pairs:
// ~3 of 10.7 ms at 1,000,000 contigs) and by the products and trees of the pairs
// left, a wave's 2 products waiting on each other: six waves a SIMD (four: 11.6
// ms).  All pairs multiplied (row blocks of 512, columns staged in LDS): 23.5 ms
// and 929 us at 200,000 contigs, against 311 us.
struct BoxArgs {
    const uint4 *frag, *frag_a;
    uint32_t T;  // tiles per coordinate of box
    float R;
    const uint4* items;
    uint32_t nitems;
    uint32_t* item_ctr;
    const uint32_t* qbounds;
    TileList out;
};

__device__ __forceinline__ void box_item(const BoxArgs& A, const float2* __restrict__ box,
                                         const float* __restrict__ margin, const uint4 it, const uint32_t item, const int wave,
                                         const int lane, uint4* stage, uint32_t& nstage) {
    const uint32_t r_hi = it.y, c_hi = it.w & ~ITEM_TRI;
    const bool tri = (it.w & ITEM_TRI) != 0;
    // waves without rows of a short item take every 2nd or 4th step of columns
    const uint32_t groups = (r_hi - (it.x & ~31u) + 32 * PROJ_RT - 1) / (32 * PROJ_RT);
    const uint32_t split = groups == 1 ? 4 : groups == 2 ? 2 : 1, part = (uint32_t)wave / groups;
    if (part >= split) return;
    const uint32_t t0 = it.x / 32 + (uint32_t)wave % groups * PROJ_RT;
    uint4 a[PROJ_RT][PROJ_KS];
#pragma unroll
    for (int rt = 0; rt < PROJ_RT; ++rt) {
        const uint32_t t = min(t0 + rt, (r_hi - 1) >> 5);
        a[rt][0] = A.frag[(size_t)t * PROJ_KS * 64 + lane];
        a[rt][1] = A.frag_a[(size_t)t * 64 + lane];
    }
    float reach[PROJ_RT];
#pragma unroll
    for (int rt = 0; rt < PROJ_RT; ++rt) reach[rt] = A.R + margin[t0 + rt];
    uint32_t cb = it.z / 32;
    if (tri && cb < t0) cb += (t0 - cb) / 64 * 64;
    for (cb += 64 * part; 32 * cb < c_hi; cb += 64 * split) {
        const uint32_t tc = cb + lane;
        float s[PROJ_RT] = {};
        {
            const float2* bc = box + tc;
            const float2* br = box + t0;
#pragma unroll 4
            for (int d = 0; d < PROJ_D; ++d) {
                const float2 c = bc[(size_t)d * A.T];
#pragma unroll
                for (int rt = 0; rt < PROJ_RT; ++rt) {
                    const float2 r = br[(size_t)d * A.T + rt];
                    const float g = fmaxf(fmaxf(c.x - r.y, r.x - c.y), 0.f);
                    s[rt] = fmaf(g, g, s[rt]);
                }
            }
        }
        const float mc = margin[tc];
        uint64_t m[PROJ_RT], u = 0;
#pragma unroll
        for (int rt = 0; rt < PROJ_RT; ++rt) {
            const float th = (reach[rt] + mc) * (1.f + 1e-5f);
            m[rt] = __ballot(s[rt] < th * th && 32 * tc < c_hi && (!tri || tc >= t0 + rt) && 32 * (t0 + rt) < r_hi);
            u |= m[rt];
        }
        if (!u) continue;
        auto load = [&](uint64_t bits, uint4* b) {
            const uint32_t c = cb + (uint32_t)__builtin_ctzll(bits);
#pragma unroll
            for (int ks = 0; ks < PROJ_KS; ++ks) b[ks] = A.frag[((size_t)c * PROJ_KS + ks) * 64 + lane];
        };
        uint4 next[PROJ_KS];
        load(u, next);
        while (u) {
            const uint32_t c = (uint32_t)__builtin_ctzll(u);
            uint4 b[PROJ_KS];
#pragma unroll
            for (int ks = 0; ks < PROJ_KS; ++ks) b[ks] = next[ks];
            u &= u - 1;
            if (u) load(u, next);
#pragma unroll
            for (int rt = 0; rt < PROJ_RT; ++rt) {
                if (!(m[rt] >> c & 1)) continue;
                f32x16_t v = f32x16_t{};
#pragma unroll
                for (int ks = 0; ks < PROJ_KS; ++ks) v = mfma32<false>(a[rt][ks], b[ks], v);
                // acc > 0 exactly when its bits, read as a signed int, are > 0
                int x[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) x[r] = __float_as_int(v[r]);
                const int m0 = max(max(x[0], x[1]), x[2]), m1 = max(max(x[3], x[4]), x[5]);
                const int m2 = max(max(x[6], x[7]), x[8]), m3 = max(max(x[9], x[10]), x[11]);
                const int m4 = max(max(x[12], x[13]), x[14]);
                if (!__any(max(max(max(m0, m1), m2), max(max(m3, m4), x[15])) > 0)) continue;
                if (lane == 0) stage[nstage] = make_uint4(t0 + rt, cb + c, item, 0u);
                if (++nstage == TILE_STAGE) tiles_flush(A.out, stage, nstage, lane);
            }
        }
    }
}

__global__ __launch_bounds__(64 * SCAN_WAVES, 6) void k_box_scan(const BoxArgs A, const float2* __restrict__ box,
                                                                 const float* __restrict__ margin) {
    __shared__ uint4 stage_all[SCAN_WAVES][TILE_STAGE];
    __shared__ uint32_t s_item;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint32_t item = blockIdx.x, q_end = A.nitems, q_base = 0;
    uint32_t* ctr = A.item_ctr;
    if (ctr && A.qbounds) {
        const uint32_t q = blockIdx.x % PF_QUEUES;
        q_base = A.qbounds[q];
        q_end = A.qbounds[q + 1];
        ctr += q * PF_CTR_STRIDE;
    }
    uint4* stage = stage_all[wave];
    uint32_t nstage = 0;
    for (;;) {
        if (ctr) {
            __syncthreads();  // every wave has read s_item
            if (threadIdx.x == 0) s_item = q_base + atomicAdd(ctr, 1u);
            __syncthreads();
            item = (uint32_t)__builtin_amdgcn_readfirstlane((int)s_item);
        }
        if (item >= q_end) break;
        box_item(A, box, margin, A.items[item], item, wave, lane, stage, nstage);
        if (!ctr) break;
    }
    tiles_flush(A.out, stage, nstage, lane);
}

// Counters of one edge-list call (64-bit words of the zeroed block; the first
// CTR_HOST are copied to the host together).
enum : uint32_t {
    CTR_MM = 0,      // k_prep_rows: log-size range, out-of-domain count
    CTR_LIST = 3,    // listed tiles (everything from here on is cleared for a repeated pass)
    CTR_CAND,        // candidate records
    CTR_KEPT,        // kept candidates ...
    CTR_ADJ,         // ... and the ones decided in FP64 (k_adjudicate: the word after CTR_KEPT)
    CTR_AMB,         // tie-band list lengths, first pass and fallback
    CTR_AMB2,
    CTR_FULL,        // full rows of the fallback
    CTR_FB_LIST,     // its listed tiles
    CTR_SURV,        // tiles with survivors, first pass and fallback
    CTR_FB_SURV,
    CTR_ERR,         // select flags
    CTR_CAPPED,      // capped rows
    CTR_BIG,         // rows for the block-wide and the global-memory selection
    CTR_HUGE,
    CTR_EDGES,       // edges
    CTR_HOST,
    CTR_QUEUES = 24, // scan queues: PF_QUEUES counters PF_CTR_STRIDE 32-bit words apart
    CTR_FB_QUEUE = CTR_QUEUES + PF_QUEUES * PF_CTR_STRIDE / 2,
    CTR_WORDS = CTR_FB_QUEUE + 8,
};
static_assert(CTR_HOST <= CTR_QUEUES, "counter layout");

using mdet::PassCaps;
using mdet::PassCounts;

__host__ __device__ inline PassCounts pass_counts(const unsigned long long* ctr) {
    return PassCounts{ctr[CTR_LIST], ctr[CTR_SURV], ctr[CTR_FB_LIST], ctr[CTR_FB_SURV], ctr[CTR_CAND]};
}

// ------------------------------------------------------------ tile pairs --
// The second pass: the pairs of the listed tiles, decided in FP32.
//   k_tile_gram    the low-precision Gram (9 k-steps, or 3 on embeddings) of
//                  each listed tile: its survivor mask, and a second list of
//                  the tiles that have any.  One wave a tile, fragments
//                  straight from L2; bound by that traffic (18 KiB a tile).
//                  FULL: the learned filter's full rows (below): row positions
//                  past the appended rows' base map through full_pos, and only
//                  pairs that phase one did not decide are taken.
//   k_tile_f32     the same mask from FP32 differences of every pair of a
//                  listed tile (EXACT_F32).
//   k_tile_refine  the survivors' FP32 distances and model.
// Edge rule: RULE_PRE (gen_tnf_graph, cuda/Cuda2.cu:884: preProb > T) or
// RULE_PROB (the MetaBAT1 variant's TNF-only graph, cuda/Cuda.cu:1750-1753:
// 1 - prob >= required_min_p with prob as cal_tnf_dist_d forms it,
// cuda/Cuda.cu:152-162).  Both are pre ~ T with T = log(1/(1 - p) - 1) away
// from the tie band; inside it the FP64 value decides with the rule's own
// arithmetic: those candidates are listed (amb, count *amb_cnt) with their
// FP32 value and decided by k_adjudicate (inlined, the FP64 evaluator costs a
// third of the waves).
constexpr int RULE_PRE = 0, RULE_PROB = 1;
constexpr uint32_t TILE_CHUNK = 16;  // consecutive list entries that stay on one XCD

// Entry of step k of worker w (of W, a multiple of 8; worker w runs on XCD
// w % 8): the workers of an XCD take its chunks of TILE_CHUNK entries in
// order, so neighbouring tiles of one scan wave, which share rows, meet in one
// L2.  Increasing in k.
__device__ inline uint64_t chunk_entry(uint32_t w, uint32_t W, uint64_t k) {
    const uint64_t l = (w >> 3) + k * (W >> 3);
    return ((l / TILE_CHUNK) * 8 + (w & 7)) * TILE_CHUNK + l % TILE_CHUNK;
}

// Tiles with survivors: (row tile, column tile, first candidate record's low 32
// bits, survivors | its high bits << 11) and the 64 lanes' masks.  The tiles'
// slots and their candidate records are reserved TILE_BATCH tiles at a time
// (one returning atomic each costs ~15-25 ns of the whole chip's time: reserved
// tile by tile they bound the second pass, 1.9 ms at 200k contigs).
struct SurvTiles {
    uint4* buf;
    uint16_t* mask;
    unsigned long long* cnt;     // counts past the capacity
    unsigned long long cap;
    unsigned long long* n_cand;  // candidate records reserved
};
constexpr uint32_t TILE_BATCH = 32;

struct TileStage {
    uint16_t mask[TILE_BATCH][64];
    uint2 tile[TILE_BATCH];
    uint32_t count[TILE_BATCH];
};

// A wave's n staged tiles to the list from slot on, their records from base on.
__device__ inline void stage_write(const SurvTiles& o, const TileStage& st, uint32_t n, uint32_t lane,
                                   unsigned long long slot, unsigned long long base) {
    const uint32_t c = lane < n ? st.count[lane] : 0u;
    base += wave_incl_sum_dpp(c) - c;
    if (lane < n && slot + lane < o.cap)
        o.buf[slot + lane] = make_uint4(st.tile[lane].x, st.tile[lane].y, (uint32_t)base,
                                        c | (uint32_t)(base >> 32) << 11);
    for (uint32_t t = 0; t < n; ++t)
        if (slot + t < o.cap) o.mask[(slot + t) * 64 + lane] = st.mask[t][lane];
}

// Reserves and writes a wave's n staged tiles (n > 0).
__device__ inline void stage_flush(const SurvTiles& o, const TileStage& st, uint32_t n, uint32_t lane) {
    wave_sync();
    const uint32_t c = lane < n ? st.count[lane] : 0u;
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_sum_dpp(c), 63);
    unsigned long long slot = 0, base = 0;
    if (lane == 0) {
        slot = atomicAdd(o.cnt, (unsigned long long)n);
        base = atomicAdd(o.n_cand, (unsigned long long)total);
    }
    stage_write(o, st, n, lane, lane0_u64(slot), lane0_u64(base));
    wave_sync();
}

struct GramArgs {
    const uint4 *frag, *frag_a;
    const uint4* items;  // null: `whole`
    uint4 whole;
    const uint4* list;  // null: every tile (tr <= tc < ntiles) of the triangle
    const unsigned long long* n_list;
    unsigned long long list_cap;
    uint32_t ntiles;
    SurvTiles out;
    // FULL
    const uint32_t* full_pos;
    uint32_t full_base;
    const uint8_t* full;
    const uint32_t *cl, *bits;
    uint32_t k;
};

// Tile e of the triangle's tiles, column by column: column tc's tiles tr = 0 ..
// tc follow tc (tc + 1) / 2 others.
__device__ inline uint4 triangle_tile(uint64_t e) {
    uint32_t tc = (uint32_t)((sqrt(8.0 * (double)e + 1.0) - 1.0) * 0.5);
    while ((uint64_t)tc * (tc + 1) / 2 > e) --tc;
    while ((uint64_t)(tc + 1) * (tc + 2) / 2 <= e) ++tc;
    return make_uint4((uint32_t)(e - (uint64_t)tc * (tc + 1) / 2), tc, 0u, 0u);
}

template <bool BF16, int KSX, bool FULL>
__global__ __launch_bounds__(256) void k_tile_gram(const GramArgs A) {
    __shared__ TileStage stages[4];
    __shared__ uint32_t fin_n[4], fin_c[4];
    __shared__ unsigned long long s_slot, s_base;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    TileStage& st = stages[wave];
    uint32_t nst = 0;
    const unsigned long long n_ent =
        A.list ? min(*A.n_list, A.list_cap) : (unsigned long long)A.ntiles * (A.ntiles + 1) / 2;
    // the block's four waves take four neighbouring entries
    for (uint64_t step = 0;; ++step) {
        const uint64_t b = chunk_entry(blockIdx.x, gridDim.x, step);
        if (4 * b >= n_ent) break;
        const uint64_t e = 4 * b + wave;
        if (e >= n_ent) continue;
        const uint4 en = A.list ? A.list[e] : triangle_tile(e);
        const uint4 it = A.items ? A.items[en.z] : A.whole;
        const uint32_t r_lo = it.x, r_hi = it.y, c_lo = it.z, c_hi = it.w & ~ITEM_TRI;
        const bool tri = (it.w & ITEM_TRI) != 0;
        f32x16_t acc = f32x16_t{};
#pragma unroll
        for (int ks = 0; ks < KSX; ++ks) {
            const uint4 a = ks == KSX - 1 ? A.frag_a[(size_t)en.x * 64 + lane]
                                          : A.frag[((size_t)en.x * KSX + ks) * 64 + lane];
            acc = mfma32<BF16>(a, A.frag[((size_t)en.y * KSX + ks) * 64 + lane], acc);
        }
        // bit r: accumulator r of this lane is a survivor (row
        // 4 (l / 32) + r % 4 + 8 (r / 4), column l % 32)
        uint32_t bits = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) bits |= (acc[r] > 0.f ? 1u : 0u) << r;
        const uint32_t i0 = 32 * en.x + 4 * (lane >> 5), j = 32 * en.y + (lane & 31);
        if ((tri && en.x == en.y) || 32 * en.x < r_lo || 32 * en.x + 32 > r_hi || 32 * en.y < c_lo ||
            32 * en.y + 32 > c_hi) {  // the diagonal or an edge of the item
            uint32_t keep = 0;
            const bool j_in = j >= c_lo && j < c_hi;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t i = i0 + (r & 3) + 8 * (r >> 2);
                const bool ok = j_in & (i >= r_lo) & (i < r_hi) & (!tri | (i < j));
                keep |= (ok ? 1u : 0u) << r;
            }
            bits &= keep;
        }
        if (FULL && bits) {
            // not the row itself, not a probed cluster pair, and of two full
            // rows only from the smaller position
            const uint32_t cj = A.cl[j];
            const bool fj = A.full[j] != 0;
            for (uint32_t left = bits; left; left &= left - 1) {
                const int r = __builtin_ctz(left);
                const uint32_t pi = A.full_pos[i0 + (r & 3) + 8 * (r >> 2) - A.full_base];
                const uint64_t ab = (uint64_t)A.cl[pi] * A.k + cj;
                if (j == pi || ((A.bits[ab >> 5] >> (ab & 31)) & 1u) || (fj && j < pi)) bits &= ~(1u << r);
            }
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_sum_dpp((uint32_t)__popc(bits)), 63);
        if (total == 0) continue;
        st.mask[nst][lane] = (uint16_t)bits;
        if (lane == 0) {
            st.tile[nst] = make_uint2(en.x, en.y);
            st.count[nst] = total;
        }
        if (++nst == TILE_BATCH) {
            stage_flush(A.out, st, nst, lane);
            nst = 0;
        }
    }
    // what is left of the block's four waves in one reservation
    wave_sync();
    const uint32_t left = (uint32_t)__builtin_amdgcn_readlane(
        (int)wave_incl_sum_dpp(lane < nst ? st.count[lane] : 0u), 63);
    if (lane == 0) {
        fin_n[wave] = nst;
        fin_c[wave] = left;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t n = fin_n[0] + fin_n[1] + fin_n[2] + fin_n[3], c = fin_c[0] + fin_c[1] + fin_c[2] + fin_c[3];
        s_slot = n ? atomicAdd(A.out.cnt, (unsigned long long)n) : 0ull;
        s_base = n ? atomicAdd(A.out.n_cand, (unsigned long long)c) : 0ull;
    }
    __syncthreads();
    if (nst) {
        unsigned long long slot = s_slot, base = s_base;
        for (uint32_t w = 0; w < wave; ++w) {
            slot += fin_n[w];
            base += fin_c[w];
        }
        stage_write(A.out, st, nst, lane, slot, base);
    }
}

struct RowArgs {
    const float* tnf;
    const float* tvec;     // Chebyshev coordinates, by contig
    const uint32_t* perm;  // position -> contig (null: itself)
    uint32_t n;
    const uint32_t* full_pos;  // appended full rows: positions of rows full_base + t (null: none)
    uint32_t full_base;
};

// Contig of lane l of a tile: its row l for l < 32, its column l - 32 for the
// others; contig 0 past the rows, and for no tile (valid = false).
__device__ inline uint32_t tile_contig(const RowArgs& A, uint32_t tr, uint32_t tc, bool valid, uint32_t lane) {
    if (!valid) return 0u;
    uint32_t p = lane < 32 ? 32 * tr + lane : 32 * tc + (lane - 32);
    if (A.full_pos && lane < 32) p = p - A.full_base < A.n ? A.full_pos[p - A.full_base] : A.n;
    return p < A.n ? (A.perm ? A.perm[p] : p) : 0u;
}

// The 64 FP32 rows of a tile (32 of its rows, then 32 of its columns) pass
// through registers into LDS: 544-byte contiguous reads by contig, no sorted
// copy of the rows.  Four lanes a row, pieces lane % 4 + 4 m and piece 32 or 33
// (two lanes each).  The row stride of 35 float4 puts 16 different rows in
// different banks.
constexpr int TQ = NT / 4, TSTR = TQ + 1, TLOADS = 9;
static_assert(TQ == 34, "four lanes load a row in eight pieces each and two more");
struct TileRows {
    f32x4_t v[TLOADS];
    __device__ inline void load(const float* tnf, uint32_t contig, uint32_t tid) {
        const f32x4_t* src = reinterpret_cast<const f32x4_t*>(tnf + (size_t)contig * NT);
        const uint32_t q = tid & 3;
#pragma unroll
        for (int m = 0; m < TLOADS - 1; ++m) v[m] = src[q + 4 * m];
        v[TLOADS - 1] = src[32 + (q & 1)];
    }
    __device__ inline void store(f32x4_t (*rows)[TSTR], uint32_t tid) const {
        const uint32_t r = tid >> 2, q = tid & 3;
#pragma unroll
        for (int m = 0; m < TLOADS - 1; ++m) rows[r][q + 4 * m] = v[m];
        rows[r][32 + (q & 1)] = v[TLOADS - 1];
    }
};

// Squared FP32 distance of two LDS rows; every mode's similarity comes from
// this sum (eight accumulators, the same order everywhere).
__device__ inline float tile_dist2(const f32x4_t* x4, const f32x4_t* y4) {
    float s[8] = {};
#pragma unroll 1
    for (int q = 0; q < TQ; q += 2) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const f32x4_t x = x4[q + h], y = y4[q + h];
            const float d0 = x.x - y.x, d1 = x.y - y.y, d2 = x.z - y.z, d3 = x.w - y.w;
            s[4 * h] = fmaf(d0, d0, s[4 * h]);
            s[4 * h + 1] = fmaf(d1, d1, s[4 * h + 1]);
            s[4 * h + 2] = fmaf(d2, d2, s[4 * h + 2]);
            s[4 * h + 3] = fmaf(d3, d3, s[4 * h + 3]);
        }
    }
    return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}

struct F32Args {
    RowArgs rows;
    const uint4* list;  // null: every tile of the triangle
    const unsigned long long* n_list;
    unsigned long long list_cap;
    uint32_t ntiles;
    float R2;
    SurvTiles out;
};

// EXACT_F32's form of the survivor mask: FP32 differences of every pair of a
// listed tile, d^2 < R2.  One block a tile, 2 x 2 pairs a thread; the next
// tile's rows are in registers meanwhile.
__global__ __launch_bounds__(256, 3) void k_tile_f32(const F32Args A) {
    __shared__ __align__(16) f32x4_t rows[64][TSTR];
    __shared__ uint32_t id[2][64], smask[64];
    __shared__ TileStage st;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const unsigned long long n_ent =
        A.list ? min(*A.n_list, A.list_cap) : (unsigned long long)A.ntiles * (A.ntiles + 1) / 2;
    auto entry = [&](uint64_t e) {
        return e < n_ent ? (A.list ? A.list[e] : triangle_tile(e)) : make_uint4(0, 0, 0, 0);
    };
    uint64_t step = 0, e0 = chunk_entry(blockIdx.x, gridDim.x, 0);
    if (e0 >= n_ent) return;
    uint64_t e1 = chunk_entry(blockIdx.x, gridDim.x, 1);
    uint4 en = entry(e0), en1 = entry(e1);
    uint32_t next_id = 0, nst = 0;
    if (wave == 0) {
        id[0][lane] = tile_contig(A.rows, en.x, en.y, true, lane);
        next_id = tile_contig(A.rows, en1.x, en1.y, e1 < n_ent, lane);
    }
    __syncthreads();
    TileRows pre;
    pre.load(A.rows.tnf, id[0][tid >> 2], tid);
    for (int buf = 0;; buf ^= 1) {
        pre.store(rows, tid);
        if (wave == 0) {
            id[buf ^ 1][lane] = next_id;
            smask[lane] = 0;
        }
        __syncthreads();
        const bool more = e1 < n_ent;
        const uint64_t e2 = chunk_entry(blockIdx.x, gridDim.x, step + 2);
        const uint4 en2 = entry(e2);
        pre.load(A.rows.tnf, id[buf ^ 1][tid >> 2], tid);  // past the last tile: rows of no use
        if (wave == 0) next_id = tile_contig(A.rows, en2.x, en2.y, e2 < n_ent, lane);
        const uint32_t ty = tid >> 4, tx = tid & 15;
        float s[2][2][8] = {};
#pragma unroll 1
        for (int q = 0; q < TQ; q += 2)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                f32x4_t x[2], y[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    x[u] = rows[ty + 16 * u][q + h];
                    y[u] = rows[32 + tx + 16 * u][q + h];
                }
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const float d0 = x[u].x - y[v].x, d1 = x[u].y - y[v].y, d2 = x[u].z - y[v].z,
                                    d3 = x[u].w - y[v].w;
                        float* t = s[u][v] + 4 * h;
                        t[0] = fmaf(d0, d0, t[0]);
                        t[1] = fmaf(d1, d1, t[1]);
                        t[2] = fmaf(d2, d2, t[2]);
                        t[3] = fmaf(d3, d3, t[3]);
                    }
            }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const float* t = s[u][v];
                const float d2 = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
                const uint32_t r = ty + 16 * u, c = tx + 16 * v, i = 32 * en.x + r, j = 32 * en.y + c;
                // the mask's layout: lane 32 (r / 4 % 2) + c, bit r % 4 + 4 (r / 8)
                if (d2 < A.R2 && i < j && j < A.rows.n)
                    atomicOr(&smask[32 * ((r >> 2) & 1) + c], 1u << ((r & 3) + 4 * (r >> 3)));
            }
        __syncthreads();  // the mask is complete; rows and id[buf] are free again
        if (wave == 0) {
            const uint32_t bits = smask[lane];
            const uint32_t total =
                (uint32_t)__builtin_amdgcn_readlane((int)wave_incl_sum_dpp((uint32_t)__popc(bits)), 63);
            if (total) {
                st.mask[nst][lane] = (uint16_t)bits;
                if (lane == 0) {
                    st.tile[nst] = make_uint2(en.x, en.y);
                    st.count[nst] = total;
                }
                if (++nst == TILE_BATCH) {
                    stage_flush(A.out, st, nst, lane);
                    nst = 0;
                }
            }
        }
        if (!more) break;
        ++step;
        e1 = e2;
        en = en1;
        en1 = en2;
    }
    if (wave == 0 && nst) stage_flush(A.out, st, nst, lane);
}

struct RefineArgs {
    RowArgs rows;
    SurvTiles in;
    float T32;
    Cand* cand;
    unsigned long long cand_cap;
    unsigned long long* kept;
    uint32_t* bcnt;  // kept endpoints per select bucket
    uint64_t* amb;
    unsigned long long* amb_cnt;
};

// One block a tile: the rows in LDS, one survivor a thread: 68 16-byte LDS
// reads, 136 differences, the FP32 Chebyshev model.  The model's four
// polynomials of two sizes are folded per contig and tile into 7 coefficients
// each (the smaller size's variable summed up), so a pair takes two dot products
// of 7 (model_of_pair); evaluated in full it was 40% of the instructions, which
// bound this kernel (88% of the issue slots): 527 -> 485 us at 200,000
// contigs.  Now LDS does, busy in 79% of the cycles (39% of that bank conflicts
// of the survivors' rows) against 59% of the issue slots.  The next tile's rows
// are in registers while this tile is worked off (its contigs known one tile
// ahead), so the loads' latency is covered by this and the CU's other blocks.
// Survivors become candidate records {i, j, preProb, flags} in place: there is
// no survivor list to sort and pack, and a tile's kept pairs share one row and
// one column bucket of the selection, so two atomics a tile count them.
// Tie-band candidates are staged in LDS over the tiles.
// Before (four lanes a survivor streaming both rows from L2, 19.4M survivors at
// 200k contigs): 1.54 ms, and 0.3 ms to sort and pack the survivor list.
constexpr uint32_t AMB_STAGE = 192;

// Per contig of the tile: 4 x 8 folded coefficients (b1 c1 b2 c2), then the
// Chebyshev values T_0..T_6 of its size (an odd number of 16-byte units apart).
constexpr int FOLD_STR = 11;

// b + c d for the polynomials at F[0..1], F[2..3].
__device__ inline float folded(const f32x4_t* F, f32x4_t t0, f32x4_t t1, float d) {
    const f32x4_t b0 = F[0], b1 = F[1], c0 = F[2], c1 = F[3];
    float b = b0.x, c = c0.x;
    b = fmaf(b0.y, t0.y, b);
    c = fmaf(c0.y, t0.y, c);
    b = fmaf(b0.z, t0.z, b);
    c = fmaf(c0.z, t0.z, c);
    b = fmaf(b0.w, t0.w, b);
    c = fmaf(c0.w, t0.w, c);
    b = fmaf(b1.x, t1.x, b);
    c = fmaf(c1.x, t1.x, c);
    b = fmaf(b1.y, t1.y, b);
    c = fmaf(c1.y, t1.y, c);
    b = fmaf(b1.z, t1.z, b);
    c = fmaf(c1.z, t1.z, c);
    return fmaf(c, d, b);
}

// model32 from the folded coefficients of the pair's contigs (ta, tb: their sizes).
__device__ inline Pre32 model_of_pair(float d, const f32x4_t* a, const f32x4_t* b, float ta, float tb) {
    const f32x4_t* F = ta <= tb ? a : b;
    const f32x4_t* T = (ta <= tb ? b : a) + 8;
    const f32x4_t t0 = T[0], t1 = T[1];
    Pre32 r;
    r.pre1 = -folded(F, t0, t1, d);
    r.pre = r.pre1;
    if (r.pre1 <= FLOOR32) r.pre = fminf(-folded(F + 4, t0, t1, d), FLOOR32);
    return r;
}

__global__ __launch_bounds__(256, 3) void k_tile_refine(const RefineArgs A) {
    __shared__ __align__(16) f32x4_t rows[64][TSTR];
    __shared__ __align__(16) f32x4_t fold[64][FOLD_STR];
    __shared__ __align__(16) f32x4_t cheb[4][MODEL_CX][2];  // coefficients by degree in the smaller size
    __shared__ uint16_t pl[1024];  // survivors of the tile: row << 5 | column
    __shared__ uint32_t id[2][64];
    __shared__ float tv[2][64];
    __shared__ uint64_t amb_at[AMB_STAGE];  // staged tie-band records
    __shared__ uint32_t s_keep, s_amb;
    __shared__ unsigned long long s_dst;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const unsigned long long n_ent = min(*A.in.cnt, A.in.cap);
    const uint4 none = make_uint4(0, 0, 0, 0);
    uint64_t step = 0, e0 = chunk_entry(blockIdx.x, gridDim.x, 0);
    if (e0 >= n_ent) return;
    uint64_t e1 = chunk_entry(blockIdx.x, gridDim.x, 1);
    uint4 en = A.in.buf[e0], en1 = e1 < n_ent ? A.in.buf[e1] : none;
    uint32_t next_id = 0, bits = 0;
    if (wave == 0) {
        const uint32_t c = tile_contig(A.rows, en.x, en.y, true, lane);
        id[0][lane] = c;
        tv[0][lane] = A.rows.tvec[c];
        next_id = tile_contig(A.rows, en1.x, en1.y, e1 < n_ent, lane);
    }
    if (wave == 1) bits = A.in.mask[e0 * 64 + lane];
    if (tid == 0) s_amb = 0;
    if (tid < 4 * MODEL_CX * 8) {
        const int k = tid & 7;
        reinterpret_cast<float*>(cheb)[tid] = k < MODEL_CY ? c_cheb[tid >> 6][(tid >> 3) & 7][k < MODEL_CY ? k : 0] : 0.f;
    }
    __syncthreads();
    TileRows pre;
    pre.load(A.rows.tnf, id[0][tid >> 2], tid);
    unsigned int nkeep = 0;
    for (int buf = 0;; buf ^= 1) {
        // this tile's rows and survivor list to LDS, the next tile's contigs beside them
        pre.store(rows, tid);
        {  // four threads a contig, a polynomial each
            const uint32_t ct = tid >> 2, p = tid & 3;
            const float t = tv[buf][ct];
            float T[MODEL_CX];
            T[0] = 1.f;
            T[1] = t;
#pragma unroll
            for (int k = 2; k < MODEL_CX; ++k) T[k] = fmaf(2.f * t, T[k - 1], -T[k - 2]);
            f32x4_t f0 = {0.f, 0.f, 0.f, 0.f}, f1 = f0;
#pragma unroll
            for (int k = 0; k < MODEL_CX; ++k) {
                const f32x4_t c0 = cheb[p][k][0], c1 = cheb[p][k][1];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f0[e] = fmaf(c0[e], T[k], f0[e]);
                    f1[e] = fmaf(c1[e], T[k], f1[e]);
                }
            }
            fold[ct][2 * p] = f0;
            fold[ct][2 * p + 1] = f1;
            if (p < 2) fold[ct][8 + p] = f32x4_t{T[4 * p], T[4 * p + 1], T[4 * p + 2], T[4 * p + 3]};
        }
        if (wave == 0) id[buf ^ 1][lane] = next_id;
        if (wave == 1) {
            const uint32_t pc = (uint32_t)__popc(bits);
            uint32_t o = wave_incl_sum_dpp(pc) - pc;
            for (; bits; bits &= bits - 1) {
                const int r = __builtin_ctz(bits);
                pl[o++] = (uint16_t)((4 * (lane >> 5) + (r & 3) + 8 * (r >> 2)) << 5 | (lane & 31));
            }
        }
        if (tid == 0) s_keep = 0;
        __syncthreads();
        // the next tile's loads, and the one after's contigs
        const bool more = e1 < n_ent;
        const uint64_t e2 = chunk_entry(blockIdx.x, gridDim.x, step + 2);
        const uint4 en2 = e2 < n_ent ? A.in.buf[e2] : none;
        float next_tv = 0.f;
        pre.load(A.rows.tnf, id[buf ^ 1][tid >> 2], tid);  // past the last tile: rows of no use
        if (wave == 0) {
            next_tv = A.rows.tvec[next_id];
            next_id = tile_contig(A.rows, en2.x, en2.y, e2 < n_ent, lane);
        }
        if (wave == 1 && more) bits = A.in.mask[e1 * 64 + lane];
        // a tile past the capacity is left out (the host runs the pass again)
        const uint32_t c = en.w & 2047u;
        const unsigned long long base = (unsigned long long)(en.w >> 11) << 32 | en.z;
        const bool fits = base + c <= A.cand_cap;
        uint32_t kept_w = 0;
        for (uint32_t t0 = 0; t0 < c && fits; t0 += 256) {
            const uint32_t t = t0 + tid;
            bool keep = false;
            uint32_t r = 0;
            if (t < c) {
                r = pl[t] >> 5;
                const uint32_t col = 32 + (pl[t] & 31);
                const Pre32 m = model_of_pair(sqrtf(tile_dist2(rows[r], rows[col])), fold[r], fold[col], tv[buf][r],
                                              tv[buf][col]);
                const bool amb = fabsf(m.pre - A.T32) <= EPS_PRE || fabsf(m.pre1 - FLOOR32) <= EPS_PRE;
                keep = !amb && m.pre > A.T32;  // a tie-band pair is kept (or not) by k_adjudicate
                Cand cd;
                cd.i = id[buf][r];
                cd.j = id[buf][col];
                cd.pre = m.pre;
                cd.flags = (amb ? 1u : 0u) | (keep ? 2u : 0u);
                A.cand[base + t] = cd;
                if (amb) {
                    const uint32_t a = atomicAdd(&s_amb, 1u);
                    if (a < AMB_STAGE)
                        amb_at[a] = base + t;
                    else  // more ties than the stage holds: one by one
                        A.amb[atomicAdd(A.amb_cnt, 1ull)] = base + t;
                }
            }
            kept_w += (uint32_t)__popcll(__ballot(keep));
            if (A.rows.full_pos && keep)
                atomicAdd(&A.bcnt[A.rows.full_pos[32 * en.x + r - A.rows.full_base] / S_BUCKET], 1u);
        }
        if (lane == 0 && kept_w) atomicAdd(&s_keep, kept_w);
        if (more && wave == 0) tv[buf ^ 1][lane] = next_tv;
        __syncthreads();  // rows, pl, id[buf] and tv[buf] are free again; s_keep and s_amb are complete
        if (tid == 0 && s_keep) {
            if (!A.rows.full_pos) atomicAdd(&A.bcnt[32 * en.x / S_BUCKET], s_keep);
            atomicAdd(&A.bcnt[32 * en.y / S_BUCKET], s_keep);
            nkeep += s_keep;
        }
        const uint32_t na = min(s_amb, AMB_STAGE);  // block-uniform
        if (na && (!more || na >= AMB_STAGE / 2)) {
            if (tid == 0) s_dst = atomicAdd(A.amb_cnt, (unsigned long long)na);
            __syncthreads();
            for (uint32_t a = tid; a < na; a += 256) A.amb[s_dst + a] = amb_at[a];
            if (tid == 0) s_amb = 0;
        }
        if (!more) break;
        ++step;
        e1 = e2;
        en = en1;
        en1 = en2;
    }
    if (tid == 0 && nkeep) atomicAdd(A.kept, (unsigned long long)nkeep);
}

__device__ inline bool prob_rule_keeps(double pre64, double required_min_p) {
    // the FP64 tie-breaker returns exactly ln 9 where the variant's model 2
    // is above its floor (prob = 0.1 there)
    const double prob = pre64 == MODEL_FLOOR_PREPROB ? 0.1 : 1.0 / (1 + exp(pre64));
    return 1. - prob >= required_min_p;
}

__device__ inline uint32_t position_of(const uint32_t* __restrict__ iperm, uint32_t c) {
    return iperm ? iperm[c] : c;
}

// The FP64 decision of each listed tie-band candidate (cuda/Cuda2.cu:192-241
// arithmetic, model64): its preProb, kept flag, bucket counts and the kept /
// adjudicated totals.  The list length is read on the device.
__global__ __launch_bounds__(256) void k_adjudicate(const float* __restrict__ tnf, const double* __restrict__ ls,
                                                    const uint32_t* __restrict__ iperm, double T, int rule,
                                                    double min_p, const uint64_t* __restrict__ amb_list,
                                                    const unsigned long long* __restrict__ amb_ctr,
                                                    Cand* __restrict__ cand, unsigned long long* __restrict__ counters,
                                                    uint32_t* __restrict__ bcnt) {
    __shared__ unsigned int s_keep;
    if (threadIdx.x == 0) s_keep = 0;
    __syncthreads();
    const uint64_t n_amb = *amb_ctr;
    unsigned int nkeep = 0;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n_amb;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t idx = amb_list[t];
        const uint32_t i = cand[idx].i, j = cand[idx].j;
        const double p64 = model64(tnf + (size_t)i * NT, tnf + (size_t)j * NT, ls[i], ls[j]);
        const bool keep = rule == RULE_PROB ? prob_rule_keeps(p64, min_p) : p64 > T;
        cand[idx].pre = (float)p64;
        cand[idx].flags = 1u | (keep ? 2u : 0u);
        if (keep) {
            atomicAdd(&bcnt[position_of(iperm, i) / S_BUCKET], 1u);
            atomicAdd(&bcnt[position_of(iperm, j) / S_BUCKET], 1u);
            ++nkeep;
        }
    }
    if (nkeep) atomicAdd(&s_keep, nkeep);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s_keep) atomicAdd(&counters[0], (unsigned long long)s_keep);
        if (blockIdx.x == 0 && n_amb) atomicAdd(&counters[1], (unsigned long long)n_amb);
    }
}

// The candidate records as the passes left them, for the kernels that read them
// before the host has seen the counters: their number, or none if one of the
// lists was too small (the host then repeats the pass, and what these kernels
// leave out is not used).
struct Records {
    const Cand* cand;
    const unsigned long long* ctr;
    PassCaps caps;
};
__device__ inline uint64_t records_to_read(const Records& r) {
    const PassCounts n = pass_counts(r.ctr);
    return mdet::records_written(n, r.caps) ? n.cand : 0ull;
}

// ------------------------------------------- learned mode: exact fallback --
// The cluster index proposes pairs; a row whose proposals fill its max_edges
// slots (a "full row") may have missed a better partner, which would leave a
// wrong edge in its list.  Full rows are therefore evaluated again against
// every column with the BF16 Gram scan (their fragments appended to the
// fragment array as extra rows), and the survivors outside the probed cluster
// pairs (which phase one decided already) go through the same refinement and
// selection.  A full row's kept set is then the exhaustive one.

// Kept candidates per row (sorted positions).  Each endpoint recurs many
// times within a wave's 64 survivors (a 64-row group against a band of
// columns), and same-address atomics are serialised at the L2: the wave
// counts into a private LDS histogram over [min, max] of its keys (when that
// span is under KEPT_SPAN) and adds each nonzero slot to the global count
// once; wider spans take one atomic per distinct key.  The loop bound is
// wave-uniform.
constexpr uint32_t KEPT_SPAN = 256;

__device__ inline uint32_t wave_min_u32(uint32_t v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, off, 64));
    return v;
}
__device__ inline uint32_t wave_max_u32(uint32_t v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off, 64));
    return v;
}

__device__ inline void kept_count(uint32_t* __restrict__ h, uint32_t* __restrict__ cnt, uint32_t key, bool kept,
                                  uint32_t lane) {
    const uint32_t lo = wave_min_u32(kept ? key : 0xFFFFFFFFu);
    const uint32_t hi = wave_max_u32(kept ? key : 0u);
    if (hi - lo < KEPT_SPAN) {
        if (kept) atomicAdd(&h[key - lo], 1u);
        __builtin_amdgcn_s_waitcnt(0);  // the wave's LDS adds are done before its lanes read the slots
        for (uint32_t s = lane; s <= hi - lo; s += 64) {
            const uint32_t v = h[s];
            if (v) {
                atomicAdd(&cnt[lo + s], v);
                h[s] = 0u;
            }
        }
        __builtin_amdgcn_s_waitcnt(0);
    } else {
        wave_aggregated_count(cnt, key, kept);
    }
}

__global__ __launch_bounds__(256) void k_row_kept(const Records rec, const uint32_t* __restrict__ iperm,
                                                  uint32_t* __restrict__ cnt) {
    __shared__ uint32_t hist[4][2][KEPT_SPAN];
    const uint32_t w = threadIdx.x >> 6, lane = lane_id();
    for (uint32_t s = lane; s < KEPT_SPAN; s += 64) hist[w][0][s] = hist[w][1][s] = 0u;
    __builtin_amdgcn_s_waitcnt(0);
    const Cand* __restrict__ cand = rec.cand;
    const uint64_t nc = records_to_read(rec);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t base = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u); base < nc; base += stride) {
        const uint64_t k = base + lane;
        bool kept = false;
        uint2 p = make_uint2(0, 0);
        if (k < nc) {
            const Cand c = cand[k];
            if (c.flags & 2u) {
                p = make_uint2(iperm[c.i], iperm[c.j]);
                kept = true;
            }
        }
        if (!__any(kept)) continue;
        kept_count(hist[w][0], cnt, p.x, kept, lane);
        kept_count(hist[w][1], cnt, p.y, kept, lane);
    }
}

// full[p] = 1 for positions with at least `need` kept candidates.
__global__ __launch_bounds__(256) void k_full_flags(const uint32_t* __restrict__ cnt, uint32_t n, uint32_t need,
                                                    uint8_t* __restrict__ full) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n) full[p] = cnt[p] >= need ? 1 : 0;
}

// ids[t] = perm[pos[t]]: the contig of each full row (the fragment source).
__global__ __launch_bounds__(256) void k_gather_ids(const uint32_t* __restrict__ pos, const uint32_t* __restrict__ perm,
                                                    uint32_t m, uint32_t* __restrict__ ids) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) ids[t] = perm[pos[t]];
}

// Bit (a, b) of the k x k map: cluster pair (a, b) was probed (either way).
__global__ __launch_bounds__(256) void k_probed_bits(const uint32_t* __restrict__ probes, uint32_t k, uint32_t n_probe,
                                                     uint32_t* __restrict__ bits) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (uint64_t)k * n_probe) return;
    const uint32_t a = (uint32_t)(t / n_probe), b = probes[t];
    if (b >= k) return;
    const uint64_t ab = (uint64_t)a * k + b, ba = (uint64_t)b * k + a;
    atomicOr(&bits[ab >> 5], 1u << (ab & 31));
    atomicOr(&bits[ba >> 5], 1u << (ba & 31));
}

// ---------------------------------------------------------------- select --
// Kept candidates -> per row the max_edges largest preProb -> edges i < j,
// sorted by (i, j).  Rows are handled in buckets of S_BUCKET consecutive
// positions of the scan's row order.  A refined survivor run shares one
// row bucket and spans a few column buckets, so the bucket counts and slot
// reservations are aggregated per wave (one device atomic per distinct bucket
// among a wave's 64 candidates, instead of one per candidate endpoint) and a
// bucket's entries are written as a few contiguous runs.  One block per
// bucket then groups its entries by row with LDS atomics, and one wave per
// row selects and sorts in LDS; rows longer than W_CAP entries, and rows
// whose FP32 tie zone at the cut exceeds one wave, take the block-wide path.
constexpr int S_THREADS = 512;          // 8 waves per bucket block
constexpr int S_WAVES = S_THREADS / 64;
constexpr int W_CAP = 512;              // entries of a row sorted by one wave

struct Ent {
    uint32_t partner;
    float pre;
    uint32_t lrow;  // row within the bucket
};

__global__ __launch_bounds__(256) void k_iperm(const uint32_t* __restrict__ perm, uint32_t n,
                                               uint32_t* __restrict__ iperm) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n) iperm[perm[s]] = s;
}

// The candidate list runs tile by tile, so neighbouring candidates share row
// buckets: consecutive blocks take 256-candidate pieces FILL_SPREAD pieces
// apart (piece = (b % FILL_SPREAD) * per + b / FILL_SPREAD), which keeps the
// blocks in flight on different buckets' counters.  The list's length is read
// on the device.
constexpr uint32_t FILL_SPREAD = 2048;

__global__ __launch_bounds__(256) void k_bucket_fill(const Records rec, const uint32_t* __restrict__ iperm,
                                                     const uint64_t* __restrict__ boff, uint32_t* __restrict__ bcur,
                                                     Ent* __restrict__ ent) {
    const Cand* __restrict__ cand = rec.cand;
    const uint64_t nc = records_to_read(rec);
    const uint64_t pieces = (nc + 255) / 256, per = (pieces + FILL_SPREAD - 1) / FILL_SPREAD;
    for (uint64_t b = blockIdx.x; b < per * FILL_SPREAD; b += gridDim.x) {
        const uint64_t piece = (b % FILL_SPREAD) * per + b / FILL_SPREAD;
        if (piece >= pieces) continue;  // whole block: the wave collectives below see all lanes
        const uint64_t k = piece * 256 + threadIdx.x;
        bool act = false;
        Cand c{0, 0, 0.f, 0};
        uint32_t si = 0, sj = 0;
        if (k < nc) {
            c = cand[k];
            if (c.flags & 2u) {
                act = true;
                si = position_of(iperm, c.i);
                sj = position_of(iperm, c.j);
            }
        }
        const KeyGroup g1 = wave_key_groups(si / S_BUCKET, act), g2 = wave_key_groups(sj / S_BUCKET, act);
        const int lane = (int)lane_id();
        uint32_t b1 = 0, b2 = 0;
        uint64_t o1 = 0, o2 = 0;
        if (act) {
            if (g1.leader == lane) b1 = atomicAdd(&bcur[si / S_BUCKET], g1.count);
            if (g2.leader == lane) b2 = atomicAdd(&bcur[sj / S_BUCKET], g2.count);
            o1 = boff[si / S_BUCKET];
            o2 = boff[sj / S_BUCKET];
        }
        b1 = (uint32_t)__shfl((int)b1, g1.leader, 64);
        b2 = (uint32_t)__shfl((int)b2, g2.leader, 64);
        if (act) {
            ent[o1 + b1 + g1.rank] = Ent{c.j, c.pre, si % S_BUCKET};
            ent[o2 + b2 + g2.rank] = Ent{c.i, c.pre, sj % S_BUCKET};
        }
    }
}

// (pre desc, partner asc): true if x ranks before y
__device__ inline bool ranks_before(float px, uint32_t ix, float py, uint32_t iy) {
    return px > py || (px == py && ix < iy);
}

// Bitonic sort of sz (power of two) LDS entries by the whole block (BY_RANK:
// by ranks_before; else by id ascending), the key carried along.
template <bool BY_RANK>
__device__ void block_sort(float* key, uint32_t* id, int sz) {
    for (int k = 2; k <= sz; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int t = threadIdx.x; t < sz; t += blockDim.x) {
                const int u = t ^ j;
                if (u > t) {
                    const bool up = (t & k) == 0;
                    const bool before = BY_RANK ? ranks_before(key[u], id[u], key[t], id[t]) : (id[u] < id[t]);
                    if (before == up) {
                        const float tk = key[t];
                        key[t] = key[u];
                        key[u] = tk;
                        const uint32_t ti = id[t];
                        id[t] = id[u];
                        id[u] = ti;
                    }
                }
            }
            __syncthreads();
        }
}

__device__ inline int pow2_at_least(uint32_t v) {
    int sz = 1;
    while (sz < (int)v) sz <<= 1;
    return sz;
}

// x of lane (lane ^ J): DPP moves and lane swaps, no LDS round trip.
template <int J>
__device__ __forceinline__ uint32_t xor_lane(uint32_t x, int lane) {
    const int v = (int)x;
    if (J == 1) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);  // quad_perm 1 0 3 2
    if (J == 2) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);  // quad_perm 2 3 0 1
    if (J == 4) {  // mirror in 8 lanes, then in 4: 7 ^ 3
        const int m = __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);
        return (uint32_t)__builtin_amdgcn_mov_dpp(m, 0x1B, 0xF, 0xF, true);
    }
    if (J == 8) return (uint32_t)__builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);  // row_ror 8
    if (J == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
        return lane & 16 ? r[0] : r[1];
    }
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return lane & 32 ? r[0] : r[1];
}

template <int J, int E>
__device__ __forceinline__ void wave_exchange(float (&key)[E], uint32_t (&id)[E], int k, int lane) {
    const bool lower = (lane & J) == 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t pi = xor_lane<J>(id[e], lane);
        const float pk = __uint_as_float(xor_lane<J>(__float_as_uint(key[e]), lane));
        const bool up = ((e * 64 + lane) & k) == 0;
        if ((lower == up) != (id[e] < pi)) {
            key[e] = pk;
            id[e] = pi;
        }
    }
}

// Bitonic sort by id of 64 * E elements held in registers by one wave, element
// t = e * 64 + lane in slot e of lane t % 64 (the ids of a row are distinct;
// padding ids are equal).  Strides below 64 are exchanges between lanes, larger
// ones swap slots within a lane.
template <int E>
__device__ __forceinline__ void wave_sort_ids(float (&key)[E], uint32_t (&id)[E], int lane) {
#pragma unroll
    for (int k = 2; k <= 64 * E; k <<= 1)
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= 64) {
                const int sj = j / 64;
#pragma unroll
                for (int e = 0; e < E; ++e)
                    if ((e & sj) == 0) {
                        const int e2 = e | sj;
                        const bool up = ((e * 64 + lane) & k) == 0;
                        if ((id[e2] < id[e]) == up) {
                            const float tk = key[e];
                            key[e] = key[e2];
                            key[e2] = tk;
                            const uint32_t ti = id[e];
                            id[e] = id[e2];
                            id[e2] = ti;
                        }
                    }
            } else if (j == 32) {
                wave_exchange<32, E>(key, id, k, lane);
            } else if (j == 16) {
                wave_exchange<16, E>(key, id, k, lane);
            } else if (j == 8) {
                wave_exchange<8, E>(key, id, k, lane);
            } else if (j == 4) {
                wave_exchange<4, E>(key, id, k, lane);
            } else if (j == 2) {
                wave_exchange<2, E>(key, id, k, lane);
            } else {
                wave_exchange<1, E>(key, id, k, lane);
            }
        }
}

// cnt (<= 64 * E) compacted entries of LDS key/id: sort by id in registers and
// write them to adj[beg..].
template <int E>
__device__ void sort_ids_and_store(const float* key, const uint32_t* id, uint32_t cnt, Adj* __restrict__ adj,
                                   uint64_t beg, int lane) {
    float k[E];
    uint32_t v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t t = e * 64 + lane;
        const bool in = t < cnt;
        k[e] = in ? key[t] : 0.f;
        v[e] = in ? id[t] : 0xffffffffu;
    }
    wave_sort_ids<E>(k, v, lane);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t t = e * 64 + lane;
        if (t < cnt) adj[beg + t] = Adj{v[e], k[e]};
    }
}

// The K largest preProb of the row's deg (<= 64 * E, > K) entries in LDS
// key/id, FP32 ties within 2 * EPS of the K-th re-ranked in FP64: the partners
// above rid compacted to the front of key/id, their number returned; -1, with
// key/id as they were, if the tie zone is wider than a wave.  Only the K-th largest key is needed, not
// their order: it is found bit by bit, counting the keys not below a candidate
// (~25 rounds of E compares; a bitonic sort by rank took 45 exchange rounds).
template <int E>
__device__ int top_of_row(uint32_t deg, uint32_t rid, uint32_t K, const float* __restrict__ tnf,
                          const double* __restrict__ ls, float* key, uint32_t* id, int lane) {
    uint32_t k[E], v[E], hi = 0, lo = 0xffffffffu;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t t = e * 64 + lane;
        const bool in = t < deg;
        k[e] = in ? f2ord(key[t]) : 0u;
        v[e] = in ? id[t] : 0xffffffffu;
        hi = max(hi, k[e]);
        lo = min(lo, in ? k[e] : 0xffffffffu);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        hi = max(hi, (uint32_t)__shfl_xor((int)hi, off, 64));
        lo = min(lo, (uint32_t)__shfl_xor((int)lo, off, 64));
    }
    // all keys share the bits above the highest one in which hi and lo differ
    hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi);
    lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
    uint32_t kth = hi;
    if (hi != lo) {
        int bit = 31 - __builtin_clz(hi ^ lo);
        kth = bit == 31 ? 0u : hi & ~((2u << bit) - 1u);
        for (; bit >= 0; --bit) {
            const uint32_t c = kth | (1u << bit);
            uint32_t cnt = 0;
#pragma unroll
            for (int e = 0; e < E; ++e) cnt += (uint32_t)__popcll(__ballot(k[e] >= c));
            if (cnt >= K) kth = c;
            if (cnt == K) break;  // c lies above every key left out
        }
        // the smallest key not below it (the last round may have ended above that key)
        uint32_t least = 0xffffffffu;
#pragma unroll
        for (int e = 0; e < E; ++e) least = min(least, k[e] >= kth ? k[e] : 0xffffffffu);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) least = min(least, (uint32_t)__shfl_xor((int)least, off, 64));
        kth = (uint32_t)__builtin_amdgcn_readfirstlane((int)least);
    }
    const float vk = ord2f(kth);
    // entries above the zone are in; of the zone, the best by FP64
    uint32_t above = 0, zn = 0, zp[E];
    bool sel[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool in = e * 64 + lane < deg;
        const float x = ord2f(k[e]);
        const bool zone = in && fabsf(x - vk) <= 2.f * EPS_PRE;
        sel[e] = in && !zone && x > vk;
        const uint64_t zm = __ballot(zone);
        zp[e] = zone ? zn + (uint32_t)__popcll(zm & ((1ull << lane) - 1ull)) : 0xffffffffu;
        zn += (uint32_t)__popcll(zm);
        above += (uint32_t)__popcll(__ballot(sel[e]));
    }
    if (zn > 64) return -1;
    const uint32_t need = K - above;
    if (need < zn) {
        wave_sync();
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (zp[e] != 0xffffffffu) id[zp[e]] = v[e];
        wave_sync();
        double zk = 0.0;
        uint32_t zi = 0xffffffffu;
        if (lane < (int)zn) {
            zi = id[lane];
            zk = model64(tnf + (size_t)rid * NT, tnf + (size_t)zi * NT, ls[rid], ls[zi]);
        }
        uint32_t rk = 0;
        for (uint32_t u = 0; u < zn; ++u) {
            const double zu = __shfl(zk, (int)u, 64);
            const uint32_t iu = (uint32_t)__shfl((int)zi, (int)u, 64);
            rk += (zu > zk || (zu == zk && iu < zi)) ? 1u : 0u;
        }
        const uint64_t won = __ballot(lane < (int)zn && rk < need);
        wave_sync();
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (zp[e] != 0xffffffffu) sel[e] = won >> zp[e] & 1;
    } else {
#pragma unroll
        for (int e = 0; e < E; ++e) sel[e] = sel[e] || zp[e] != 0xffffffffu;
    }
    wave_sync();  // the row is in registers by here; its entries in LDS are overwritten
    uint32_t cnt = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool keep = sel[e] && v[e] > rid;
        const uint64_t m = __ballot(keep);
        if (keep) {
            const uint32_t o = cnt + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            key[o] = ord2f(k[e]);
            id[o] = v[e];
        }
        cnt += (uint32_t)__popcll(m);
    }
    return (int)cnt;
}

// Row `rid` (contig id), its deg entries in LDS key/id, which are overwritten:
// the kept ones, by id, to adj[beg..), by one wave.  Returns false, with key/id
// and adj as they were, if the row needs the block path (FP32 tie zone at the
// cut wider than a wave).  capped counts in LDS: one atomic per row on the
// call's counter serialised the 50,000 capped rows of a 50,000-contig input.
__device__ bool wave_row_select(Adj* __restrict__ adj, uint64_t beg, uint32_t deg, uint32_t rid, uint32_t K,
                                const float* __restrict__ tnf, const double* __restrict__ ls, float* key,
                                uint32_t* id, uint32_t* __restrict__ out_cnt, uint64_t* __restrict__ rbeg,
                                uint32_t* capped, int lane) {
    uint32_t cnt = 0;
    if (K && deg > K) {
        const int c = deg <= 64    ? top_of_row<1>(deg, rid, K, tnf, ls, key, id, lane)
                      : deg <= 128 ? top_of_row<2>(deg, rid, K, tnf, ls, key, id, lane)
                      : deg <= 256 ? top_of_row<4>(deg, rid, K, tnf, ls, key, id, lane)
                                   : top_of_row<8>(deg, rid, K, tnf, ls, key, id, lane);
        if (c < 0) return false;
        cnt = (uint32_t)c;
        if (lane == 0) atomicAdd(capped, 1u);
    } else {
        // every candidate is selected: gather the partners above the row.  An
        // entry moves to its own place or before it, so those not read yet stay.
        for (uint32_t t0 = 0; t0 < deg; t0 += 64) {
            const uint32_t t = t0 + lane;
            const uint32_t p = t < deg ? id[t] : 0u;
            const float x = t < deg ? key[t] : 0.f;
            const bool keep = t < deg && p > rid;
            const uint64_t m = __ballot(keep);
            wave_sync();
            if (keep) {
                const uint32_t o = cnt + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                key[o] = x;
                id[o] = p;
            }
            wave_sync();
            cnt += (uint32_t)__popcll(m);
        }
    }
    // sorted by id in registers
    wave_sync();
    if (cnt <= 64)
        sort_ids_and_store<1>(key, id, cnt, adj, beg, lane);
    else if (cnt <= 128)
        sort_ids_and_store<2>(key, id, cnt, adj, beg, lane);
    else if (cnt <= 256)
        sort_ids_and_store<4>(key, id, cnt, adj, beg, lane);
    else
        sort_ids_and_store<8>(key, id, cnt, adj, beg, lane);
    if (lane == 0) {
        out_cnt[rid] = cnt;
        rbeg[rid] = beg;
    }
    return true;
}

// Appends (rid, deg, beg) to a row list with its counter apart; err bit `ovf`
// if the list is full.
constexpr int BIG_REC = 4;  // uint32 words per row record: rid, deg, beg lo, beg hi
struct RowList {
    uint32_t* rec;
    uint32_t* cnt;
    uint32_t cap;
};
__device__ inline void push_row(const RowList& L, uint32_t rid, uint32_t deg, uint64_t beg,
                                unsigned int* __restrict__ err, unsigned int ovf) {
    const uint32_t q = atomicAdd(L.cnt, 1u);
    if (q < L.cap) {
        uint32_t* rec = L.rec + BIG_REC * q;
        rec[0] = rid;
        rec[1] = deg;
        rec[2] = (uint32_t)beg;
        rec[3] = (uint32_t)(beg >> 32);
    } else {
        atomicOr(err, ovf);
    }
}

// The same by the whole block, for rows of up to SEL_CAP entries and tie
// zones of up to ZONE_CAP entries.  Larger rows or zones are left untouched
// and listed in `huge` for k_hugerow_select (global-memory sort, no limit).
__device__ void block_row_select(Adj* __restrict__ adj, uint64_t beg, uint32_t deg, uint32_t rid, uint32_t K,
                                 const float* __restrict__ tnf, const double* __restrict__ ls, float* key,
                                 uint32_t* id, double* zkey, int* s_z, uint32_t* s_cnt,
                                 uint32_t* __restrict__ out_cnt, uint64_t* __restrict__ rbeg,
                                 const RowList& huge, unsigned int* __restrict__ err,
                                 unsigned long long* __restrict__ capped) {
    if (deg > SEL_CAP) {
        if (threadIdx.x == 0) push_row(huge, rid, deg, beg, err, 8u);
        return;
    }
    const int sz = pow2_at_least(deg);
    for (int t = threadIdx.x; t < sz; t += blockDim.x) {
        const bool in = t < (int)deg;
        const Adj e = in ? adj[beg + t] : Adj{0xffffffffu, 0.f};
        key[t] = in ? e.pre : -__builtin_inff();
        id[t] = in ? e.partner : 0xffffffffu;
    }
    __syncthreads();
    uint32_t nsel = deg;
    if (K && deg > K) {
        block_sort<true>(key, id, sz);
        const float vk = key[K - 1];
        if (threadIdx.x == 0) {
            s_z[0] = (int)deg;
            s_z[1] = 0;
        }
        __syncthreads();
        for (int t = threadIdx.x; t < (int)deg; t += blockDim.x)
            if (fabsf(key[t] - vk) <= 2.f * EPS_PRE) {
                atomicMin(&s_z[0], t);
                atomicMax(&s_z[1], t + 1);
            }
        __syncthreads();
        const int z0 = s_z[0], z1 = s_z[1], zn = z1 - z0;
        if (zn > ZONE_CAP) {  // block-uniform: adj is still untouched
            if (threadIdx.x == 0) push_row(huge, rid, deg, beg, err, 8u);
            __syncthreads();
            return;
        }
        if (threadIdx.x == 0) atomicAdd(capped, 1ull);
        if (zn > 1) {
            for (int t = threadIdx.x; t < zn; t += blockDim.x) {
                const uint32_t p = id[z0 + t];
                zkey[t] = model64(tnf + (size_t)rid * NT, tnf + (size_t)p * NT, ls[rid], ls[p]);
            }
            __syncthreads();
            // rank each zone entry by (FP64 key desc, partner asc)
            uint32_t myid[ZONE_CAP / S_THREADS + 1];
            float mykey[ZONE_CAP / S_THREADS + 1];
            int myrank[ZONE_CAP / S_THREADS + 1];
            int cntm = 0;
            for (int t = threadIdx.x; t < zn; t += blockDim.x, ++cntm) {
                int rk = 0;
                for (int u = 0; u < zn; ++u)
                    rk += (zkey[u] > zkey[t] || (zkey[u] == zkey[t] && id[z0 + u] < id[z0 + t])) ? 1 : 0;
                myid[cntm] = id[z0 + t];
                mykey[cntm] = key[z0 + t];
                myrank[cntm] = rk;
            }
            __syncthreads();
            for (int c = 0; c < cntm; ++c) {
                id[z0 + myrank[c]] = myid[c];
                key[z0 + myrank[c]] = mykey[c];
            }
            __syncthreads();
        }
        nsel = K;
    }
    for (int t = threadIdx.x; t < sz; t += blockDim.x)
        if (t >= (int)nsel || id[t] <= rid) id[t] = 0xffffffffu;
    if (threadIdx.x == 0) *s_cnt = 0;
    __syncthreads();
    block_sort<false>(key, id, sz);
    for (int t = threadIdx.x; t < sz; t += blockDim.x)
        if (id[t] != 0xffffffffu) atomicAdd(s_cnt, 1u);
    __syncthreads();
    const uint32_t cnt = *s_cnt;
    for (int t = threadIdx.x; t < (int)cnt; t += blockDim.x) adj[beg + t] = Adj{id[t], key[t]};
    if (threadIdx.x == 0) {
        out_cnt[rid] = cnt;
        rbeg[rid] = beg;
    }
    __syncthreads();
}

// One block per bucket: group the bucket's entries by row, then select every
// row by one wave.  Output per contig row: out_cnt (edges kept: partners above
// the row, sorted) and rbeg (where they are in adj, whose offsets are ent's).
// Rows the wave path declines go to a list for k_bigrow_select ((row id,
// degree, begin) records), their entries in adj.  Without records to read (and
// so without entries, whatever the bucket counts say) every row stays at no
// edges, as the call cleared out_cnt.
//
// The rows are grouped in LDS, where each is selected in place, as far as
// L_CAP entries go; only rows of more than W_CAP entries and those that end
// beyond L_CAP are grouped in adj, the latter staged through LDS once the
// rows in it are done.  Bound by vector instructions (the search of the K-th
// key, the FP64 zone, the sort) and by the latency of the entries' two passes.
// Grouped in adj, every row was written eight bytes here and there and read
// back: 385 us at 200k contigs, 1289 at 1M, 194 at 50k in FP32; grouped in LDS
// with two blocks a CU 350, 1111 and 201; with rows taken as waves become free
// 321, 1001 and 172; with three blocks a CU 298, 880 and 152 (80 registers, at
// the price of a few spills around the FP64 zone; four blocks: 307, 854 and
// 162); with eight loads in flight instead of four 290, 873 and 149.  L_CAP is
// what lets three blocks share a CU's 160 KB.  Taking the longest row first
// gave nothing.
constexpr uint32_t L_CAP = 6600;
static_assert(S_WAVES * W_CAP <= (int)L_CAP, "staging of the rows grouped in adj");

// Whether a row of deg entries from slot `at` of its bucket is grouped in LDS.
__device__ __forceinline__ bool in_lds(uint32_t at, uint32_t deg) {
    return deg <= (uint32_t)W_CAP && at <= L_CAP - deg;
}

__global__ __launch_bounds__(S_THREADS, 6) void k_bucket_select(
    const Records rec, const uint64_t* __restrict__ boff, const Ent* __restrict__ ent, Adj* __restrict__ adj,
    uint32_t n, uint32_t K, const uint32_t* __restrict__ perm, const float* __restrict__ tnf,
    const double* __restrict__ ls, uint32_t* __restrict__ out_cnt, uint64_t* __restrict__ rbeg, const RowList big,
    unsigned int* __restrict__ err, unsigned long long* __restrict__ capped) {
    constexpr int PER = S_BUCKET / 64;
    constexpr int BATCH = 8;
    __shared__ uint32_t hist[S_BUCKET], rstart[S_BUCKET], rcur[S_BUCKET], s_next[2], s_capped;
    __shared__ float lkey[L_CAP];
    __shared__ uint32_t lid[L_CAP];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint32_t b = blockIdx.x;
    const uint64_t e0 = boff[b], e1 = boff[b + 1];
    if (records_to_read(rec) == 0) return;  // the counters' loads go out with the bucket's
    const uint32_t row0 = b * S_BUCKET;
    const uint32_t rows = n - row0 < (uint32_t)S_BUCKET ? n - row0 : (uint32_t)S_BUCKET;
    for (int t = tid; t < S_BUCKET; t += S_THREADS) hist[t] = rcur[t] = 0;
    if (tid == 0) s_capped = s_next[0] = s_next[1] = 0;
    __syncthreads();
    // row histogram; BATCH independent loads in flight per thread
    for (uint64_t e = e0 + tid; e < e1; e += BATCH * S_THREADS) {
        uint32_t lr[BATCH];
#pragma unroll
        for (int q = 0; q < BATCH; ++q) lr[q] = e + q * S_THREADS < e1 ? ent[e + q * S_THREADS].lrow : 0xffffffffu;
#pragma unroll
        for (int q = 0; q < BATCH; ++q)
            if (lr[q] != 0xffffffffu) atomicAdd(&hist[lr[q]], 1u);
    }
    __syncthreads();
    if (wave == 0) {  // exclusive scan of the row counts, PER per lane
        uint32_t v[PER], sum = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            v[q] = hist[PER * lane + q];
            sum += v[q];
        }
        uint32_t x = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        uint32_t run = x - sum;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            rstart[PER * lane + q] = run;
            run += v[q];
        }
    }
    __syncthreads();
    for (uint64_t e = e0 + tid; e < e1; e += BATCH * S_THREADS) {
        Ent x[BATCH];
        bool ok[BATCH];
#pragma unroll
        for (int q = 0; q < BATCH; ++q) {
            ok[q] = e + q * S_THREADS < e1;
            if (ok[q]) x[q] = ent[e + q * S_THREADS];
        }
#pragma unroll
        for (int q = 0; q < BATCH; ++q)
            if (ok[q]) {
                const uint32_t lr = x[q].lrow, at = rstart[lr], deg = hist[lr];
                const uint32_t slot = at + atomicAdd(&rcur[lr], 1u);
                if (in_lds(at, deg)) {
                    lid[slot] = x[q].partner;
                    lkey[slot] = x[q].pre;
                } else {
                    adj[e0 + slot] = Adj{x[q].partner, x[q].pre};
                }
            }
    }
    __syncthreads();
    for (int pass = 0; pass < 2; ++pass) {  // the rows in LDS, then those staged through it
        if (pass == 1) {
            if (e1 - e0 <= L_CAP) break;
            __syncthreads();
        }
        // rows are taken as waves become free: their degrees differ widely
        for (;;) {
            uint32_t r = lane == 0 ? atomicAdd(&s_next[pass], 1u) : 0u;
            r = (uint32_t)__builtin_amdgcn_readfirstlane((int)r);
            if (r >= rows) break;
            const uint32_t deg = hist[r], at = rstart[r];
            const bool here = in_lds(at, deg), wide = deg > (uint32_t)W_CAP;
            if (pass == 1 && (here || wide)) continue;
            if (pass == 0 && !here && !wide) continue;
            const uint64_t beg = e0 + at;
            const uint32_t pos = row0 + r;
            const uint32_t rid = perm ? perm[pos] : pos;
            bool done = !wide;
            if (deg == 0) {
                if (lane == 0) {
                    out_cnt[rid] = 0;
                    rbeg[rid] = beg;
                }
            } else if (!wide) {
                float* key = here ? lkey + at : lkey + wave * W_CAP;
                uint32_t* id = here ? lid + at : lid + wave * W_CAP;
                if (!here) {
                    wave_sync();
                    for (uint32_t t = lane; t < deg; t += 64) {
                        const Adj a = adj[beg + t];
                        key[t] = a.pre;
                        id[t] = a.partner;
                    }
                    wave_sync();
                }
                done = wave_row_select(adj, beg, deg, rid, K, tnf, ls, key, id, out_cnt, rbeg, &s_capped, lane);
                if (!done && here)
                    for (uint32_t t = lane; t < deg; t += 64) adj[beg + t] = Adj{id[t], key[t]};
            }
            if (!done && lane == 0) push_row(big, rid, deg, beg, err, 4u);
        }
    }
    __syncthreads();
    if (tid == 0 && s_capped) atomicAdd(capped, (unsigned long long)s_capped);
}

// Rows the wave path declined (over W_CAP entries, or a tie zone wider than a
// wave): one block per row, blocks striding over the list.  err bit 4: the
// list overflowed its capacity.  Rows beyond the LDS capacities go on to the
// `huge` list (err bit 8 if that list overflowed).
__global__ __launch_bounds__(S_THREADS) void k_bigrow_select(
    const RowList big, Adj* __restrict__ adj, uint32_t K, const float* __restrict__ tnf,
    const double* __restrict__ ls, uint32_t* __restrict__ out_cnt, uint64_t* __restrict__ rbeg, const RowList huge,
    unsigned int* __restrict__ err, unsigned long long* __restrict__ capped) {
    __shared__ float bkey[SEL_CAP];
    __shared__ uint32_t bid[SEL_CAP];
    __shared__ double zkey[ZONE_CAP];
    __shared__ int s_z[2];
    __shared__ uint32_t s_cnt;
    const uint32_t nbig = *big.cnt;
    const uint32_t m = nbig < big.cap ? nbig : big.cap;
    for (uint32_t q = blockIdx.x; q < m; q += gridDim.x) {
        const uint32_t* rec = big.rec + BIG_REC * q;
        const uint64_t beg = (uint64_t)rec[2] | ((uint64_t)rec[3] << 32);
        block_row_select(adj, beg, rec[1], rec[0], K, tnf, ls, bkey, bid, zkey, s_z, &s_cnt, out_cnt, rbeg, huge,
                         err, capped);
    }
}

// Rows too large for LDS (more than SEL_CAP candidates, or more than ZONE_CAP
// near-ties at the cut): one block per listed row, sorting in global scratch
// (row q owns entries [soff[q], soff[q] + pow2(deg))).  Every candidate's
// preProb is recomputed by the FP64 tie-breaker and the row is ranked by
// (FP64 preProb desc, partner asc): the same selection as the FP32 rank with
// the FP64 re-rank of the tie zone, since the FP32 evaluator's error is far
// below the zone half-width.  Then the kept partners above the row are sorted
// by id into adj[beg..] as the other select paths leave them.
constexpr int HUGE_THREADS = 1024;

__device__ inline void global_step_sync() {
    __threadfence();  // the sort runs through global memory: device-scope visibility
    __syncthreads();
}

// Bitonic sort ascending of sz (power of two) entries by (k64, k32), v carried.
__device__ void global_bitonic(unsigned long long* k64, uint32_t* k32, uint32_t* v, uint32_t sz) {
    for (uint32_t k = 2; k <= sz; k <<= 1)
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t t = threadIdx.x; t < sz; t += blockDim.x) {
                const uint32_t u = t ^ j;
                if (u > t) {
                    const bool up = (t & k) == 0;
                    const unsigned long long a64 = k64[t], b64 = k64[u];
                    const uint32_t a32 = k32[t], b32 = k32[u];
                    const bool u_first = b64 < a64 || (b64 == a64 && b32 < a32);
                    if (u_first == up) {
                        k64[t] = b64;
                        k64[u] = a64;
                        k32[t] = b32;
                        k32[u] = a32;
                        const uint32_t tv = v[t];
                        v[t] = v[u];
                        v[u] = tv;
                    }
                }
            }
            global_step_sync();
        }
}

__global__ __launch_bounds__(HUGE_THREADS) void k_hugerow_select(
    const uint32_t* __restrict__ huge, const uint64_t* __restrict__ soff, Adj* __restrict__ adj, uint32_t K,
    const float* __restrict__ tnf, const double* __restrict__ ls, unsigned long long* __restrict__ sk64,
    uint32_t* __restrict__ sk32, uint32_t* __restrict__ sv, float* __restrict__ spre,
    uint32_t* __restrict__ out_cnt, uint64_t* __restrict__ rbeg, unsigned long long* __restrict__ capped) {
    __shared__ uint32_t s_cnt;
    const uint32_t* rec = huge + BIG_REC * blockIdx.x;
    const uint32_t rid = rec[0], deg = rec[1];
    const uint64_t beg = (uint64_t)rec[2] | ((uint64_t)rec[3] << 32);
    uint32_t sz = 1;
    while (sz < deg) sz <<= 1;
    const uint64_t o = soff[blockIdx.x];
    unsigned long long* k64 = sk64 + o;
    uint32_t *k32 = sk32 + o, *v = sv + o;
    float* pre = spre + o;
    for (uint32_t t = threadIdx.x; t < sz; t += blockDim.x) {
        if (t < deg) {
            const Adj e = adj[beg + t];
            const double p64 = model64(tnf + (size_t)rid * NT, tnf + (size_t)e.partner * NT, ls[rid], ls[e.partner]);
            k64[t] = ~d2ord(p64);  // ascending order = FP64 preProb descending
            k32[t] = e.partner;
            pre[t] = e.pre;
        } else {
            k64[t] = ~0ull;
            k32[t] = 0xffffffffu;
        }
        v[t] = t;
    }
    if (threadIdx.x == 0) s_cnt = 0;
    global_step_sync();
    const bool cap = K && deg > K;
    const uint32_t nsel = cap ? K : deg;
    if (cap) global_bitonic(k64, k32, v, sz);
    // keep ranks < nsel with partners above the row, then order them by id
    uint32_t mine = 0;
    for (uint32_t t = threadIdx.x; t < sz; t += blockDim.x) {
        const bool keep = t < nsel && k32[t] > rid && k32[t] != 0xffffffffu;
        if (!keep) k32[t] = 0xffffffffu;
        k64[t] = 0;
        mine += keep ? 1u : 0u;
    }
    if (mine) atomicAdd(&s_cnt, mine);
    global_step_sync();
    global_bitonic(k64, k32, v, sz);
    const uint32_t cnt = s_cnt;
    for (uint32_t t = threadIdx.x; t < cnt; t += blockDim.x) adj[beg + t] = Adj{k32[t], pre[v[t]]};
    if (threadIdx.x == 0) {
        out_cnt[rid] = cnt;
        rbeg[rid] = beg;
        if (cap) atomicAdd(capped, 1ull);
    }
}

// Edges of row r (contig order) to their place eoff[r]; a wave takes EMIT_ROWS
// rows, their offsets and first 128 entries in flight together.  *total = their
// number.  Moves 20 bytes an edge; with a row to a wave, its loads one after
// the other, 103 us at 200k contigs (15.2M edges) and 444 at 1M (50.8M), with
// four 74 and 287 (3.5 TB/s).
constexpr int EMIT_ROWS = 4;
__global__ void k_emit(const uint64_t* __restrict__ rbeg, const Adj* __restrict__ adj,
                       const uint32_t* __restrict__ out_cnt, const uint64_t* __restrict__ eoff, uint32_t n,
                       uint32_t* __restrict__ from, uint32_t* __restrict__ to, float* __restrict__ s,
                       unsigned long long* __restrict__ total) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *total = eoff[n];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t row0 = (blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6)) * EMIT_ROWS;
    uint32_t c[EMIT_ROWS];
    uint64_t src[EMIT_ROWS], dst[EMIT_ROWS];
    Adj e[EMIT_ROWS][2];
#pragma unroll
    for (int q = 0; q < EMIT_ROWS; ++q) {
        const bool in = row0 + q < n;
        c[q] = in ? out_cnt[row0 + q] : 0u;
        src[q] = in ? rbeg[row0 + q] : 0u;
        dst[q] = in ? eoff[row0 + q] : 0u;
    }
#pragma unroll
    for (int q = 0; q < EMIT_ROWS; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (h * 64 + lane < c[q]) e[q][h] = adj[src[q] + h * 64 + lane];
    auto put = [&](uint32_t row, uint64_t at, const Adj& a) {
        from[at] = row;
        to[at] = a.partner;
        s[at] = 1.f - 1.f / (1.f + expf(a.pre));
    };
#pragma unroll
    for (int q = 0; q < EMIT_ROWS; ++q) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (h * 64 + lane < c[q]) put(row0 + q, dst[q] + h * 64 + lane, e[q][h]);
        for (uint32_t t = 128 + lane; t < c[q]; t += 64) put(row0 + q, dst[q] + t, adj[src[q] + t]);
    }
}

// ------------------------------------------------------------- row max --
// Sampled row maxima of preProb (get_tnf_max_prob_sample, cuda/Cuda2.cu:
// 281-314): for each sampled position p < n_sample, the maximum over all
// positions q != p of preProb(idx[p], idx[q]).
//
// On MFMA: preProb falls with the distance for any two sizes, so bounds of a
// pair's distance give bounds of its preProb.  A first scan takes each sampled
// row's largest lower bound, a second lists the pairs whose upper bound reaches
// it, and only those are evaluated in FP64 (k_rm_exact).  Per 32 x 32 tile of
// pairs a scan forms three kinds of MFMA products of FP16 fragments:
//   -|a~ - b~|^2 / 2   the TNF Gram (9 k-steps); the distance itself differs by
//             the two rows' rounding errors (measured per row) and the FP32
//             accumulation (RM_D2)
//   b, c      the model's two polynomials of the sizes, preProb = -(b + c d):
//             with one size's variable folded into the coefficients each is a
//             dot product of 8 coefficients with the other's Chebyshev values,
//             as hi + lo FP16 pairs (2 k-steps; ~1e-6 of preProb, ~4e-4 where
//             subnormal parts are lost: EPS_PRE covers both)
// Positions are ordered by size, so which side of a tile is the smaller one
// (the model's x) is known for the whole tile; tiles around the diagonal run
// both ways under a per-pair condition, which leaves out q = p as well.
// RM_BEST1 bounds by model 1 alone (it applies above ln 9, where nearly every
// row's maximum lies); RM_BEST2 adds model 2 for blocks that hold a row without
// a pair above ln 9.  Block = 4 waves, a 32-row tile of sampled positions each
// (fragments in registers), over a segment of tiles of all positions, streamed
// through LDS in two buffers.  Bound by the VALU (a square root, three multiply-
// adds, an addition and half a minimum per pair: ~90 us at 20,011^2 pairs) and
// the 13 MFMAs a tile (65 us) beside each other.  All of 20,011 maxima: 0.55 ms
// (172 us RM_BEST1, 45 RM_BEST2, 199 RM_LIST); the direct form alone took 20.2 ms
// (FP32 differences and the whole model of every pair on the VALU, twice).
// One buffer array with halves by index: 207, 60 and 248 us.
// A finite row above PLAIN_NORM2 or more near-ties than the list holds leave
// everything to k_rowmax.
constexpr float RM_D2 = 4e-5f;  // |computed - exact| of |a~ - b~|^2 up to PLAIN_NORM2 (144 terms, 2^-24 each)
constexpr int RM_PKS = 2;       // k-steps of a polynomial's product
constexpr int RM_CHUNKS = KS + 2 * RM_PKS;  // 1 KiB chunks of a tile in LDS: Gram, b, c
constexpr uint32_t RM_STAGE = 64;
enum : int { RM_BEST1, RM_BEST2, RM_LIST };

// Sort key of each position: its size, and itself as the value.
__global__ __launch_bounds__(256) void k_rm_keys(const float* __restrict__ tvec, const uint64_t* __restrict__ idx,
                                                 uint32_t m, uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
    const uint32_t p = blockIdx.x * 256 + threadIdx.x;
    if (p >= m) return;
    key[p] = f2ord(tvec[(uint32_t)idx[p]]);
    val[p] = p;
}

// Per element s of the order: its contig, and rank[position] = s.
__global__ __launch_bounds__(256) void k_rm_contigs(const uint64_t* __restrict__ idx, const uint32_t* __restrict__ order,
                                                    uint32_t m, uint32_t* __restrict__ contig,
                                                    uint32_t* __restrict__ rank) {
    const uint32_t s = blockIdx.x * 256 + threadIdx.x;
    if (s >= m) return;
    const uint32_t p = order[s];
    contig[s] = (uint32_t)idx[p];
    if (rank) rank[p] = s;
}

__device__ inline uint4 rm_pack(const _Float16* x) {
    uint16_t h[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) h[k] = __builtin_bit_cast(uint16_t, x[k]);
    return pack8(h);
}

// All positions: the 8 folded coefficients of polynomial p (b1 c1 b2 c2) in
// role v (0: the position's is the smaller size), in the slots hi (k = 0..7),
// lo (8..15), hi (16..23), 0; and per tile the largest rounding error (NaN
// ones, of padding, aside).  Eight threads a position.
__global__ __launch_bounds__(256) void k_rm_poly(const float* __restrict__ tvec, const uint32_t* __restrict__ contig,
                                                 const float* __restrict__ err, uint32_t m,
                                                 uint4* __restrict__ pfrag, float* __restrict__ tile_err) {
    const uint32_t s = blockIdx.x * 32 + (threadIdx.x >> 3), v = (threadIdx.x >> 2) & 1, p = threadIdx.x & 3;
    const float x = s < m ? tvec[contig[s]] : 0.f;
    float T[MODEL_CX];
    T[0] = 1.f;
    T[1] = x;
#pragma unroll
    for (int k = 2; k < MODEL_CX; ++k) T[k] = fmaf(2.f * x, T[k - 1], -T[k - 2]);
    _Float16 hi[8], lo[8], zero[8] = {};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        float f = 0.f;
        if (v == 0) {
            if (k < MODEL_CY)
#pragma unroll
                for (int a = 0; a < MODEL_CX; ++a) f = fmaf(c_cheb[p][a][k], T[a], f);
        } else {
#pragma unroll
            for (int b = 0; b < MODEL_CY; ++b) f = fmaf(c_cheb[p][k][b], T[b], f);
        }
        hi[k] = (_Float16)f;
        lo[k] = (_Float16)(f - (float)hi[k]);
    }
    uint4* dst = pfrag + (((size_t)blockIdx.x * 2 + v) * 4 + p) * RM_PKS * 64 + (s & 31);
    dst[0] = dst[64] = rm_pack(hi);
    dst[32] = rm_pack(lo);
    dst[96] = rm_pack(zero);
    if (threadIdx.x < 64) {
        float e = threadIdx.x < 32 ? err[blockIdx.x * 32 + threadIdx.x] : 0.f;
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) e = fmaxf(e, __shfl_xor(e, off, 64));
        if (threadIdx.x == 0) tile_err[blockIdx.x] = e > 0.f ? e : 0.f;
    }
}

// Sampled positions: the Chebyshev values, slots hi, hi, lo, 0.
__global__ __launch_bounds__(256) void k_rm_cheb(const float* __restrict__ tvec, const uint32_t* __restrict__ contig,
                                                 uint32_t m, uint32_t tiles, uint4* __restrict__ tfrag) {
    const uint32_t s = blockIdx.x * 256 + threadIdx.x;
    if (s >= tiles * 32) return;
    const float x = s < m ? tvec[contig[s]] : 0.f;
    float T[8];
    T[0] = 1.f;
    T[1] = x;
    _Float16 hi[8], lo[8], zero[8] = {};
#pragma unroll
    for (int k = 2; k < 8; ++k) T[k] = fmaf(2.f * x, T[k - 1], -T[k - 2]);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        hi[k] = (_Float16)T[k];
        lo[k] = (_Float16)(T[k] - (float)hi[k]);
    }
    uint4* dst = tfrag + (size_t)(s >> 5) * RM_PKS * 64 + (s & 31);
    dst[0] = dst[32] = rm_pack(hi);
    dst[64] = rm_pack(lo);
    dst[96] = rm_pack(zero);
}

struct RmArgs {
    // all positions by size
    const uint4 *frag, *frag_a, *pfrag;
    const float* tile_err;
    const uint32_t* order;
    uint32_t n, tiles, seg;  // seg: tiles a block
    // sampled positions by size
    const uint4 *cfrag, *tfrag;
    const float* cerr;
    const uint32_t *corder, *rank;  // rank: of a position among all
    uint32_t ns, ctiles;
    uint32_t* best;  // per sampled element: largest lower bound (f2ord; 0: none)
    uint2* list;     // (sampled element, position)
    unsigned long long* n_list;
    uint32_t cap;
    const uint32_t* outside;
};

template <int PASS>
__global__ __launch_bounds__(256, 3) void k_rm_scan(const RmArgs A) {
    __shared__ uint4 R0[RM_CHUNKS * 64], R1[RM_CHUNKS * 64];
    __shared__ uint2 stage_all[PASS == RM_LIST ? 4 : 1][RM_STAGE];
    if (*A.outside) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t ct = 4 * blockIdx.x + wave, r0 = blockIdx.y * A.seg, r1 = min(A.tiles, r0 + A.seg);
    const bool active = ct < A.ctiles;
    const uint32_t col = 32 * ct + (lane & 31);
    const bool in = active && col < A.ns;
    const float ej = in ? A.cerr[col] : 0.f;
    const bool have = in && ej == ej;
    const float best = have && PASS != RM_BEST1 ? ord2f(A.best[col]) : 0.f;  // NaN: none
    const bool low = have && PASS != RM_BEST1 && !(best > FLOOR32);           // model 2 may decide
    bool need2 = false;
    if (PASS == RM_BEST2) {
        if (!__syncthreads_or(low)) return;
    } else if (PASS == RM_LIST) {
        need2 = __any(low);
    }
    uint4 B[KS], Tc[RM_PKS];
#pragma unroll
    for (int k = 0; k < KS; ++k) B[k] = active ? A.cfrag[((size_t)ct * KS + k) * 64 + lane] : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int k = 0; k < RM_PKS; ++k)
        Tc[k] = active ? A.tfrag[((size_t)ct * RM_PKS + k) * 64 + lane] : make_uint4(0, 0, 0, 0);
    const uint32_t rj = in ? A.rank[A.corder[col]] : 0u;
    // ranks are ascending along the sampled elements
    const uint32_t b_lo = A.rank[A.corder[128 * blockIdx.x]];
    const uint32_t b_hi = A.rank[A.corder[min(128 * blockIdx.x + 127, A.ns - 1)]];
    // role of tile rt's positions against the block's: 0 smaller, 1 larger, 2 both
    auto role = [&](uint32_t rt) { return 32 * rt + 31 < b_lo ? 0 : 32 * rt > b_hi ? 1 : 2; };
    constexpr int P0 = PASS == RM_BEST2 ? 2 : 0;  // polynomials in LDS: b1 c1, or b2 c2
    auto poly = [&](uint32_t rt, int v, int p) {
        return A.pfrag + (((size_t)rt * 2 + v) * 4 + p) * RM_PKS * 64;
    };
    auto fill = [&](uint32_t rt, uint4* buf) {
        const uint4* pf = poly(rt, role(rt) == 1, P0);
#pragma unroll
        for (int m = 0; m < (RM_CHUNKS + 3) / 4; ++m) {
            const int c = 4 * m + wave;
            if (c < RM_CHUNKS) {
                const uint4* src = c < KS - 1    ? A.frag + ((size_t)rt * KS + c) * 64
                                   : c == KS - 1 ? A.frag_a + (size_t)rt * 64
                                                 : pf + (c - KS) * 64;
                __builtin_amdgcn_global_load_lds((const void*)(src + lane),
                                                 (__attribute__((address_space(3))) void*)(buf + 64 * c), 16, 0, 0);
            }
        }
    };
    // in terms of w = -preProb: its smallest upper bound, and the listing limits
    // of model 1 and model 2 (where the maximum is known to be ln 9 at least, only
    // pairs that may lie above it)
    const float nfloor = -FLOOR32, inf = __builtin_inff();
    float wbest = inf, lim1 = 0.f, lim2 = 0.f;
    if (PASS == RM_LIST) {
        lim1 = have ? (best > FLOOR32 ? 2.f * EPS_PRE - best : nfloor + EPS_PRE) : -inf;
        lim2 = have && best < FLOOR32 ? 2.f * EPS_PRE - best : -inf;
    }
    uint2* stage = stage_all[PASS == RM_LIST ? wave : 0];
    uint32_t nst = 0;
    auto flush = [&]() {
        unsigned long long k = 0;
        if (lane == 0) k = atomicAdd(A.n_list, (unsigned long long)nst);
        k = lane0_u64(k);
        wave_sync();
        if ((uint32_t)lane < nst && k + lane < A.cap) A.list[k + lane] = stage[lane];
        wave_sync();
        nst = 0;
    };
    // the segment's largest rounding error: one a tile would have to be loaded
    // in the loop, and waited for behind the fill
    float E = 0.f;
    for (uint32_t rt = r0 + lane; rt < r1; rt += 64) E = fmaxf(E, A.tile_err[rt]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) E = fmaxf(E, __shfl_xor(E, off, 64));
    E += ej;
    auto step = [&](const uint32_t rt, const uint4* R, uint4* next) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (rt + 1 < r1) fill(rt + 1, next);
        if (!active) return;
        const int ro = role(rt);
        f32x16_t acc = f32x16_t{}, pb = f32x16_t{}, pc = f32x16_t{};
#pragma unroll
        for (int k = 0; k < KS; ++k) acc = mfma32<false>(R[k * 64 + lane], B[k], acc);
#pragma unroll
        for (int k = 0; k < RM_PKS; ++k) {
            pb = mfma32<false>(R[(KS + k) * 64 + lane], Tc[k], pb);
            pc = mfma32<false>(R[(KS + RM_PKS + k) * 64 + lane], Tc[k], pc);
        }
        const uint32_t i0 = 32 * rt + 4 * (lane >> 5);
        auto d_least = [&](float a) {
            return fmaxf(__builtin_amdgcn_sqrtf(fmaxf(fmaf(-2.f, a, -RM_D2), 0.f)) - E, 0.f);
        };
        if (PASS == RM_LIST && ro != 2 && !need2) {
            // most tiles hold no pair to list: all 16 at the shortest distance first
            float near = acc[0], least = inf;
#pragma unroll
            for (int r = 1; r < 16; ++r) near = fmaxf(near, acc[r]);
            const float dn = d_least(near);
#pragma unroll
            for (int r = 0; r < 16; ++r) least = fminf(least, fmaf(pc[r], dn, pb[r]));
            if (!__any(least <= lim1)) return;
        }
        float d[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            d[r] = PASS == RM_LIST ? d_least(acc[r]) : __builtin_amdgcn_sqrtf(fmaf(-2.f, acc[r], RM_D2)) + E;
        uint32_t bits = 0;  // RM_LIST: pairs to list among this lane's 16
        auto take = [&](const f32x16_t& b, const f32x16_t& c, uint32_t use, float lim) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float w = fmaf(c[r], d[r], b[r]);
                if (PASS == RM_LIST)
                    bits |= (w <= lim ? 1u : 0u) << r & use;
                else
                    wbest = fminf(wbest, use >> r & 1u ? w : inf);
            }
        };
        // positions of this lane's 16 on one side of its own (not itself)
        auto side = [&](bool larger) {
            uint32_t use = 0;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t i = i0 + (r & 3) + 8 * (r >> 2);
                use |= (i < A.n && (larger ? i > rj : i < rj) ? 1u : 0u) << r;
            }
            return use;
        };
        auto product = [&](int v, int p) {
            const uint4* f = poly(rt, v, p);
            f32x16_t x = f32x16_t{};
#pragma unroll
            for (int k = 0; k < RM_PKS; ++k) x = mfma32<false>(f[k * 64 + lane], Tc[k], x);
            return x;
        };
        if (ro != 2) {
            take(pb, pc, 0xffffu, lim1);
            if (PASS == RM_LIST && need2) take(product(ro, 2), product(ro, 3), 0xffffu, lim2);
        } else {
            take(pb, pc, side(false), lim1);
            take(product(1, P0), product(1, P0 + 1), side(true), lim1);
            if (PASS == RM_LIST && need2) {
                take(product(0, 2), product(0, 3), side(false), lim2);
                take(product(1, 2), product(1, 3), side(true), lim2);
            }
        }
        if (PASS == RM_LIST) {
            if (!__any(bits != 0)) return;
            const uint32_t cnt = (uint32_t)__popc(bits), incl = wave_incl_sum_dpp(cnt);
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            uint32_t o = incl - cnt, done = 0;
            while (done < total) {
                const uint32_t took = min(RM_STAGE - nst, total - done);
                while (bits && o < done + took) {
                    const int r = __builtin_ctz(bits);
                    bits &= bits - 1;
                    const uint32_t i = i0 + (r & 3) + 8 * (r >> 2);
                    stage[nst + (o - done)] = make_uint2(col, i < A.n ? A.order[i] : A.corder[col]);
                    ++o;
                }
                nst += took;
                done += took;
                if (nst == RM_STAGE) flush();
            }
        }
    };
    // two arrays by name: of one array's halves the compiler cannot tell the
    // fill's from the one read, and waits for the fill before the reads
    fill(r0, R0);
    for (uint32_t rt = r0; rt < r1; rt += 2) {
        step(rt, R0, R1);
        if (rt + 1 < r1) step(rt + 1, R1, R0);
    }
    if (PASS == RM_LIST) {
        if (nst) flush();
    } else {
        wbest = fminf(wbest, __shfl_xor(wbest, 32, 64));
        if (have && lane < 32 && wbest < inf) {
            // model 1's bound counts where it certainly applies; model 2's is clamped to ln 9
            if (PASS == RM_BEST1) {
                if (wbest < nfloor - EPS_PRE) atomicMax(&A.best[col], f2ord(-wbest));
            } else if (low) {
                atomicMax(&A.best[col], f2ord(-fmaxf(wbest + EPS_PRE, nfloor)));
            }
        }
    }
}

// FP64 preProb of the listed pairs, into each sampled position's maximum; a
// maximum known to be ln 9 at least starts there.
__global__ __launch_bounds__(64 * DIST_WAVES) void k_rm_exact(const RmArgs A, const float* __restrict__ tnf,
                                                              const double* __restrict__ ls,
                                                              const uint64_t* __restrict__ idx,
                                                              unsigned long long* __restrict__ m64) {
    __shared__ __align__(16) float X[DIST_WAVES][DIST_LDS];
    const unsigned long long m = *A.n_list;
    if (*A.outside || m > A.cap) return;
    const uint32_t g = blockIdx.x * (64 * DIST_WAVES) + threadIdx.x, step = gridDim.x * (64 * DIST_WAVES);
    for (uint32_t c = g; c < A.ns; c += step)
        if (A.best[c] && ord2f(A.best[c]) == FLOOR32) atomicMax(&m64[A.corder[c]], d2ord(MODEL_FLOOR_PREPROB));
    for (uint32_t k0 = g & ~63u; k0 < (uint32_t)m; k0 += step) {
        const uint32_t k = k0 + (threadIdx.x & 63);
        const bool in = k < (uint32_t)m;
        const uint2 e = in ? A.list[k] : make_uint2(0, 0);
        const uint32_t p = in ? A.corder[e.x] : 0u, i = in ? (uint32_t)idx[p] : 0u, j = in ? (uint32_t)idx[e.y] : 0u;
        const double d2 = wave_dist2_f64(tnf, i, j, X[threadIdx.x >> 6]);
        if (!in || p == e.y) continue;
        const double v = model64_d2(d2, ls[i], ls[j]);
        if (v == v) atomicMax(&m64[p], d2ord(v));
    }
}

// The direct form, for small inputs and the ones the bounds do not cover (with
// outside: only then).  Block = 64 sampled rows x a chunk of columns; both
// sides staged K-major in LDS, each thread owns a 4x4 block of pairs: FP32
// squared distance, FP32 model, running row maximum.  Pass 1 (EXACT=false)
// finds the FP32 maximum m32 of each row; pass 2 (EXACT=true) re-evaluates in
// FP64 every pair with FP32 preProb >= m32 - 2*EPS (the true maximum is among
// them) and keeps their FP64 maximum.
constexpr int RM_ROWS = 64, RM_COLS = 64, RM_CHUNK = 4096;


template <bool EXACT>
__global__ __launch_bounds__(256) void k_rowmax(const float* __restrict__ tnf, const double* __restrict__ ls,
                                                const float* __restrict__ tvec, const uint64_t* __restrict__ idx,
                                                uint32_t n, uint32_t n_sample, uint32_t* __restrict__ m32,
                                                unsigned long long* __restrict__ m64,
                                                const uint32_t* __restrict__ outside,
                                                const unsigned long long* __restrict__ n_list, uint32_t cap) {
    if (outside && !*outside && *n_list <= cap) return;
    __shared__ float As[NT][RM_ROWS + 1];
    __shared__ float Bs[NT][RM_COLS + 1];
    __shared__ uint32_t rid[RM_ROWS], cid[RM_COLS];
    const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
    const uint32_t p0 = blockIdx.x * RM_ROWS;
    const uint32_t q_begin = blockIdx.y * RM_CHUNK, q_end = min(q_begin + RM_CHUNK, n);
    if (tid < RM_ROWS) rid[tid] = (p0 + tid < n_sample) ? (uint32_t)idx[p0 + tid] : 0u;
    __syncthreads();
    for (int e = tid; e < RM_ROWS * NT; e += 256) {
        const int r = e / NT, k = e - r * NT;
        As[k][r] = tnf[(size_t)rid[r] * NT + k];
    }
    float best[4];
    float thr[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        best[a] = -__builtin_inff();
        const uint32_t p = p0 + ty + 16 * a;
        thr[a] = (EXACT && p < n_sample) ? ord2f(m32[p]) - 2.f * EPS_PRE : 0.f;
    }
    double best64[4] = {-1.0 / 0.0, -1.0 / 0.0, -1.0 / 0.0, -1.0 / 0.0};
    for (uint32_t q0 = q_begin; q0 < q_end; q0 += RM_COLS) {
        __syncthreads();
        if (tid < RM_COLS) cid[tid] = (q0 + tid < q_end) ? (uint32_t)idx[q0 + tid] : 0u;
        __syncthreads();
        for (int e = tid; e < RM_COLS * NT; e += 256) {
            const int c = e / NT, k = e - c * NT;
            Bs[k][c] = tnf[(size_t)cid[c] * NT + k];
        }
        __syncthreads();
        float acc[4][4] = {};
        for (int k = 0; k < NT; ++k) {
            float av[4], bv[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) av[a] = As[k][ty + 16 * a];
#pragma unroll
            for (int b = 0; b < 4; ++b) bv[b] = Bs[k][tx + 16 * b];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const float df = av[a] - bv[b];
                    acc[a][b] = fmaf(df, df, acc[a][b]);
                }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const uint32_t p = p0 + ty + 16 * a;
            if (p >= n_sample) continue;
            const uint32_t ri = rid[ty + 16 * a];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t q = q0 + tx + 16 * b;
                if (q >= q_end || q == p) continue;
                const uint32_t cj = cid[tx + 16 * b];
                const float pre = model32(sqrtf(acc[a][b]), tvec[ri], tvec[cj]).pre;
                if (!EXACT) {
                    best[a] = fmaxf(best[a], pre);
                } else if (pre >= thr[a]) {
                    const double v = model64(tnf + (size_t)ri * NT, tnf + (size_t)cj * NT, ls[ri], ls[cj]);
                    best64[a] = v > best64[a] ? v : best64[a];
                }
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const uint32_t p = p0 + ty + 16 * a;
        if (p >= n_sample) continue;
        if (!EXACT) {
            if (best[a] > -__builtin_inff()) atomicMax(&m32[p], f2ord(best[a]));
        } else if (best64[a] > -1.0 / 0.0) {
            atomicMax(&m64[p], d2ord(best64[a]));
        }
    }
}

// max_out[p] = 1 - 1/(1 + exp(max(DBL_MIN, m64[p]))): the running maximum of
// the reference starts at DBL_MIN (cuda/Cuda2.cu:287, 312).
__global__ void k_rowmax_final(const unsigned long long* __restrict__ m64, uint32_t n_sample,
                               double* __restrict__ out) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n_sample) return;
    double m = 2.2250738585072014e-308;
    if (m64[p]) {
        const double v = ord2d(m64[p]);
        if (v > m) m = v;
    }
    out[p] = 1. - (1. / (1. + exp(m)));
}

// Pairs with an index >= n are counted in *bad_idx and get NaN (no row read).
__global__ void k_preprob_pairs(const float* __restrict__ tnf, const double* __restrict__ ls,
                                const float* __restrict__ tvec, uint32_t n, const uint32_t* __restrict__ pi,
                                const uint32_t* __restrict__ pj, uint64_t np, float* __restrict__ p32,
                                double* __restrict__ p64, unsigned int* __restrict__ bad_idx) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= np) return;
    const uint32_t i = pi[k], j = pj[k];
    if (i >= n || j >= n) {
        atomicAdd(bad_idx, 1u);
        if (p32) p32[k] = __builtin_nanf("");
        if (p64) p64[k] = __builtin_nan("");
        return;
    }
    const float* a = tnf + (size_t)i * NT;
    const float* b = tnf + (size_t)j * NT;
    if (p32) p32[k] = model32(sqrtf(dist2_f32(a, b)), tvec[i], tvec[j]).pre;
    if (p64) p64[k] = model64(a, b, ls[i], ls[j]);
}

// FP64 similarity of listed pairs, 1 - 1/(1 + exp(preProb)) with preProb from
// the FP64 tie-breaker: the value get_tnf_graph2 stores (cuda/Cuda2.cu:257-258).
// Pairs with an index >= n are counted in *bad_idx and get NaN.
__global__ __launch_bounds__(64 * DIST_WAVES) void k_similarity64(
    const float* __restrict__ tnf, const double* __restrict__ ls, uint32_t n, const uint32_t* __restrict__ pi,
    const uint32_t* __restrict__ pj, uint64_t np, double* __restrict__ s64, unsigned int* __restrict__ bad_idx) {
    __shared__ __align__(16) float X[DIST_WAVES][DIST_LDS];
    const uint64_t k = (uint64_t)blockIdx.x * (64 * DIST_WAVES) + threadIdx.x;
    const bool in = k < np;
    const uint32_t i = in ? pi[k] : 0u, j = in ? pj[k] : 0u;
    const bool ok = in && i < n && j < n;
    if (in && !ok) {
        atomicAdd(bad_idx, 1u);
        s64[k] = __builtin_nan("");
    }
    if (!__any(ok)) return;  // n may be 0
    const double d2 = wave_dist2_f64(tnf, ok ? i : 0u, ok ? j : 0u, X[threadIdx.x >> 6]);
    if (ok) s64[k] = 1. - 1. / (1. + exp(model64_d2(d2, ls[i], ls[j])));
}

}  // namespace

namespace mdet {

int ensure_model(mdet_ctx* ctx) {
    if (ctx->model_ready) return MDET_OK;
    ModelCheb m;
    model_cheb_tables(&m);
    MDET_HIP(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_cheb), m.c, sizeof m.c, 0, hipMemcpyHostToDevice, ctx->stream));
    MDET_HIP(hipStreamSynchronize(ctx->stream));
    ctx->model_ready = true;
    return MDET_OK;
}

}  // namespace mdet

using namespace mdet;

namespace {

struct Timer {
    mdet_ctx* ctx;
    int base;
    int record(int k) {
        hipEvent_t e;
        MDET_TRY(ctx_event(ctx, base + k, &e));
        MDET_HIP(hipEventRecord(e, ctx->stream));
        return MDET_OK;
    }
    double ms(int a, int b) {
        float v = 0;
        if (hipEventElapsedTime(&v, ctx->events[base + a], ctx->events[base + b]) != hipSuccess) return 0;
        return v;
    }
};

template <class T>
int read_scalar(mdet_ctx* ctx, const T* dev, T* out) {
    void* st;
    MDET_TRY(ctx_host_stage(ctx, 64, &st));
    MDET_HIP(hipMemcpyAsync(st, dev, sizeof(T), hipMemcpyDeviceToHost, ctx->stream));
    MDET_HIP(hipStreamSynchronize(ctx->stream));
    memcpy(out, st, sizeof(T));
    return MDET_OK;
}

int exclusive_scan_u32_to_u64(mdet_ctx* ctx, const uint32_t* in, uint64_t* out, uint32_t n) {
    // out[0..n] = exclusive prefix sums of in[0..n-1], out[n] = total
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, in, out, (int)n + 1, ctx->stream));
    void* t;
    MDET_TRY(ctx_buf(ctx, "cub.tmp", tmp, &t));
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(t, tmp, in, out, (int)n + 1, ctx->stream));
    return MDET_OK;
}

// Scan items over the whole triangle: (row block of `rows`, column begin,
// column end), each row block's columns from its diagonal in segments of seg
// columns.  With one queue (row-block major) the survivor-heavy diagonal item
// of every row block is one of ~n/seg items in flight; with per-XCD queues
// (column start major within a queue of every 8th row block) the diagonal
// items still come spread over time and XCDs, while an XCD's blocks share
// column ranges in its L2: memory-side traffic 19.4 -> 3.5 GB and 10% faster
// at 200k contigs in the full Gram over 256-row blocks.
// order 0: one list, row-block major.  order 1: PF_QUEUES lists (row blocks
// rb with rb % PF_QUEUES == q), each ordered by column start then row block,
// so the blocks of one XCD work on neighbouring column ranges together;
// qbounds[0..PF_QUEUES] delimit the lists.
int build_items(mdet_ctx* ctx, uint32_t n, uint32_t rows, uint32_t seg, uint32_t order, uint4** items_dev,
                uint32_t* nitems, uint32_t** qbounds_dev) {
    if (ctx->items_n == n && ctx->items_rows == rows && ctx->items_seg == seg && ctx->items_order == order &&
        ctx->nitems) {
        auto it = ctx->bufs.find("pairs.items");
        auto iq = ctx->bufs.find("pairs.item_qb");
        if (it != ctx->bufs.end() && iq != ctx->bufs.end()) {
            *items_dev = static_cast<uint4*>(it->second.p);
            *qbounds_dev = static_cast<uint32_t*>(iq->second.p);
            *nitems = ctx->nitems;
            return MDET_OK;
        }
    }
    std::vector<uint4> items;
    std::vector<uint32_t> qb(PF_QUEUES + 1, 0);
    const uint32_t nrb = (n + rows - 1) / rows;
    auto row_items = [&](uint32_t rb, std::vector<uint4>& v) {
        for (uint32_t c = rb * rows; c < n; c += seg)
            v.push_back(make_uint4(rb * rows, std::min(rb * rows + rows, n), c, std::min<uint32_t>(c + seg, n) | ITEM_TRI));
    };
    if (order == 0) {
        for (uint32_t rb = 0; rb < nrb; ++rb) row_items(rb, items);
        for (int q = 1; q <= PF_QUEUES; ++q) qb[q] = (uint32_t)items.size();
    } else {
        for (int q = 0; q < PF_QUEUES; ++q) {
            std::vector<uint4> qi;
            for (uint32_t rb = q; rb < nrb; rb += PF_QUEUES) row_items(rb, qi);
            std::stable_sort(qi.begin(), qi.end(), [](const uint4& x, const uint4& y) { return x.z < y.z; });
            qb[q] = (uint32_t)items.size();
            items.insert(items.end(), qi.begin(), qi.end());
        }
        qb[PF_QUEUES] = (uint32_t)items.size();
    }
    *nitems = (uint32_t)items.size();
    ctx->nitems = 0;  // not cached until the upload is queued
    MDET_TRY(ctx_buf(ctx, "pairs.items", items.size(), items_dev));
    MDET_TRY(ctx_buf(ctx, "pairs.item_qb", PF_QUEUES + 1, qbounds_dev));
    MDET_HIP(hipMemcpyAsync(*items_dev, items.data(), items.size() * sizeof(uint4), hipMemcpyHostToDevice,
                            ctx->stream));
    MDET_HIP(hipMemcpyAsync(*qbounds_dev, qb.data(), qb.size() * sizeof(uint32_t), hipMemcpyHostToDevice,
                            ctx->stream));
    MDET_HIP(hipStreamSynchronize(ctx->stream));
    ctx->items_n = n;
    ctx->items_rows = rows;
    ctx->items_seg = seg;
    ctx->items_order = order;
    ctx->nitems = *nitems;
    return MDET_OK;
}

constexpr int PREP_EVENT = 6;  // context event index marking the log-size range's copy
// Exhaustive modes up to this many contigs skip the row order and the first
// pass: every tile goes to the second one.  What that costs goes with the square
// of the contigs, the order's ~190 us do not; BF16, us direct / ordered at 100,
// 200 and 300 contigs a genome: 6,300 contigs 392 / 359, 487 / 438, 587 / 526;
// 8,000 491 / 369, 607 / 445, 694 / 535.  Only inputs with next to no pair in
// range would take a later line (8,000 contigs of 4,000 genomes 210 / 312).
constexpr uint32_t DIRECT_MAX = 6144;
// Contigs above which the selection's buffers go by the counted candidates: 52
// bytes each of 128 a contig are 7.5 KB a contig, more than half of a call's
// memory (12.2 KB a contig; counted 7.8 with 86 survivors a contig and 4.8 with
// hardly any), and the wait of ~20 us is nothing beside the 20 ms of such an
// input.
constexpr uint32_t COUNTED_SELECT = 1u << 20;
// Pairs of full rows and contigs, and of the probed clusters, from which on the
// learned filter scans projected rows as the exhaustive modes do: the projection
// takes ~190 us at 200,000 contigs (110 of them at any size) and serves both;
// multiplying all tile pairs takes 135 us per 1e9 pairs of full rows and 250 of
// the ragged cluster pairs, the box scan 25 and 200.
constexpr uint64_t PROBE_PROJ_PAIRS = 750000000;
constexpr uint64_t PROJ_PAIRS = 1500000000;
// Resident refinement blocks per CU at most (52 KiB of LDS each).
constexpr uint32_t REFINE_PER_CU = 3;

int edges_impl(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n, double cutoff,
               uint32_t max_edges, int precision, mdet_mlp* mlp, float radius2, uint32_t n_clusters,
               uint32_t n_probe, mdet_edges* out, mdet_pair_stats* stats, int rule = RULE_PRE) {
    MDET_TRY(check_ctx(ctx));
    if (!out) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges: null output");
    ctx->last_pairs = 0;
    *out = mdet_edges{0, nullptr, nullptr, nullptr};
    mdet_pair_stats st{};
    st.pairs_total = (uint64_t)n * (n ? n - 1 : 0) / 2;
    if (!(cutoff > 0.0 && cutoff < 1.0)) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges: cutoff %g not in (0, 1)", cutoff);
    if (precision < MDET_EXACT_F32 || precision > MDET_LEARNED)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges: unknown precision %d", precision);
    if (precision == MDET_LEARNED && !(radius2 > 0 || (radius2 == 0.f && n_probe > 0)))
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges_learned: needs a positive radius (radius2 = 0 only with probes)");
    // the exact cover clusters a fixed projection of the TNF rows: no network needed
    if (precision == MDET_LEARNED && !mlp && !(ctx->learned_exact_cover && radius2 == 0.f))
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges_learned: needs a network (none only with the exact cover)");
    if (n > (1u << 30)) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_edges: n = %u too large", n);
    if (n < 2) {
        if (stats) *stats = st;
        return MDET_OK;
    }
    if (!tnf_dev || !logsize_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges: null tnf or logsize");
    MDET_TRY(ensure_model(ctx));
    // threshold on preProb exactly as cuda/Cuda2.cu:884
    const double T = log((1.0 / (1. - cutoff)) - 1.0);
    Timer tm{ctx, 0};
    MDET_TRY(tm.record(0));

    // -- counters and per-call arrays that start at zero, in one allocation:
    // CTR_WORDS counters (64-bit), then kept endpoints per select bucket, the
    // buckets' fill cursors, and the edges per row
    const uint32_t nb = (n + S_BUCKET - 1) / S_BUCKET;
    unsigned long long* ctr;
    const size_t zero_words = 2 * (size_t)CTR_WORDS + (nb + 1) + nb + ((size_t)n + 1);
    MDET_TRY(ctx_buf(ctx, "pairs.zero", (zero_words + 1) / 2, &ctr));
    uint32_t* bcnt = reinterpret_cast<uint32_t*>(ctr + CTR_WORDS);
    uint32_t* bcur = bcnt + nb + 1;
    uint32_t* out_cnt = bcur + nb;
    MDET_HIP(hipMemsetAsync(ctr, 0, zero_words * 4, ctx->stream));

    // -- prep rows: the log sizes' range goes to the host, which finds the
    // radius while the device orders the rows
    float* tvec;
    MDET_TRY(ctx_buf(ctx, "pairs.tvec", n, &tvec));
    hipLaunchKernelGGL(k_prep_rows, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, logsize_dev, n, tvec, ctr + CTR_MM);
    MDET_HIP(hipGetLastError());
    void* stage_host;
    MDET_TRY(ctx_host_stage(ctx, 8 * CTR_HOST, &stage_host));
    unsigned long long* host = static_cast<unsigned long long*>(stage_host);
    hipEvent_t prep_done;
    MDET_TRY(ctx_event(ctx, PREP_EVENT, &prep_done));
    MDET_HIP(hipMemcpyAsync(host, ctr + CTR_MM, 3 * 8, hipMemcpyDeviceToHost, ctx->stream));
    MDET_HIP(hipEventRecord(prep_done, ctx->stream));
    // small inputs: every 32 x 32 tile of the triangle goes straight to the
    // second pass, in contig order
    const bool gram_all = precision != MDET_LEARNED;  // the exhaustive modes
    const bool direct = gram_all && n <= DIRECT_MAX;
    const bool cluster = precision == MDET_LEARNED && n_probe > 0;
    ProjOrder order;
    if (!direct && !cluster)
        MDET_TRY(proj_order(ctx, tnf_dev, n,
                            precision == MDET_BF16_REFINE ? PROJ_BF16 : precision == MDET_F16_REFINE ? PROJ_F16 : PROJ_F32,
                            &order));
    MDET_HIP(hipEventSynchronize(prep_done));
    if (host[2] != 0)
        MDET_FAIL(MDET_E_RANGE,
                  "mdet_tnf_edges: %u log sizes outside [log10 1500, log10 500000] (contigs shorter than 1500 "
                  "are not allowed in the graph)",
                  (unsigned int)host[2]);
    double xlo, xhi;
    {
        const unsigned long long a = ~host[0], b = host[1];
        memcpy(&xlo, &a, 8);
        memcpy(&xhi, &b, 8);
    }
    // the radius cache key: the threshold, offset for the probability rule
    // (|T| < 40 for any cutoff in (0, 1) representable here)
    const double rkey = rule == RULE_PROB ? T + 1e6 : T;
    if (!(ctx->radius_valid && ctx->radius_key[0] == xlo && ctx->radius_key[1] == xhi && ctx->radius_key[2] == rkey)) {
        if (rule == RULE_PROB) {
            // s = 1 - prob >= p: model 1 passes where preProb >= T (all of it
            // above ln 9 if T < ln 9); model 2 where preProb2 >= T, and also,
            // if p <= 0.9, wherever it is above its floor (prob = 0.1 there)
            const double fl = MODEL_FLOOR_PREPROB;
            const bool m2 = T < fl || 0.9 >= cutoff;
            ctx->radius = model_dthr_max(xlo, xhi, T > fl ? T : fl, m2, T < fl ? T : fl);
        } else {
            ctx->radius = model_dthr_max(xlo, xhi, T);
        }
        ctx->radius_key[0] = xlo;
        ctx->radius_key[1] = xhi;
        ctx->radius_key[2] = rkey;
        ctx->radius_valid = true;
    }
    const double R = ctx->radius;
    mdet_edges result{0, nullptr, nullptr, nullptr};

    if (R > 0) {
        const mdet_ctx::Tune tune = ctx->tune[precision];
        const bool bf = precision != MDET_F16_REFINE;      // format of the Gram
        const bool f32 = precision == MDET_EXACT_F32;
        const bool tnf_gram = !(radius2 > 0.f);            // Gram of the TNF rows (else of embeddings)
        // exact cover: the cluster pairs that can hold a pair within
        // the radius R (TNF-space triangle bound) instead of probes;
        // then no row can miss a partner and no row is completed
        const bool exact_cover = cluster && tnf_gram && ctx->learned_exact_cover;
        // rows per scan item, and the rows padded to whole blocks
        const uint32_t item_rows = gram_all ? scan_rows(PROJ_RT) : ITEM_ROWS;
        const uint32_t n_pad = (n + item_rows - 1) / item_rows * item_rows;
        // distance below which the Gram must keep every pair, and the distance
        // beyond which the second pass keeps none: the FP32 mode's own bound,
        // or what the Gram adds to its radius: its slack (2 GRAM_SLACK (|x|^2 +
        // 1) on the square for unit rows) here, and twice each row's rounding
        // in the row's own margin
        const float gram_r = (float)(R * (1.0 + 1e-6)) + 1e-5f;
        const float f32_r2 = (float)(R * R * (1.0 + 1e-4)) + 1e-6f;
        const float reach = std::sqrt(f32 ? f32_r2 : gram_r * gram_r + 4.4f * GRAM_SLACK) * (1.f + 1e-5f) + 1e-6f;

        // -- fragments of the Gram in the scan's row order
        uint32_t* perm = order.perm;  // position -> contig (null: itself)
        uint4 *frag = nullptr, *frag_a = nullptr, *pfrag = nullptr, *pfrag_a = nullptr;
        float2* pbox = nullptr;
        float* pbox_margin = nullptr;
        const uint32_t box_tiles = (n_pad / 32 + 127) / 64 * 64;  // a whole step past the last tile
        uint4* items = nullptr;
        uint32_t nitems = 0;
        uint32_t* qbounds = nullptr;
        IvfIndex ivf;
        const int ks = tnf_gram ? KS : KS_E;
        // cluster items start column steps anywhere: room for one more block;
        // with the TNF Gram also for the fallback's full rows, appended after
        // the first n_frag
        const uint32_t n_frag = cluster ? n_pad + ITEM_ROWS : n_pad;
        const uint32_t n_alloc = cluster && tnf_gram ? n_frag + n_pad : n_frag;
        if (!f32) {
            MDET_TRY(ctx_buf(ctx, gram_all ? "pairs.frag" : "learn.frag", (size_t)n_alloc / 32 * ks * 64, &frag));
            MDET_TRY(ctx_buf(ctx, gram_all ? "pairs.frag_a" : "learn.frag_a", (size_t)n_alloc / 32 * 64, &frag_a));
        }
        const uint32_t seg = tune.seg_cols ? tune.seg_cols : seg_cols_for(n);
        const dim3 fgrid(n_frag / 32);
        if (gram_all) {
            if (!f32 && bf)
                hipLaunchKernelGGL((k_prep_lowp<true, NT, KS>), fgrid, dim3(256), 0, ctx->stream, tnf_dev, perm, n,
                                   gram_r, frag, frag_a);
            else if (!f32)
                hipLaunchKernelGGL((k_prep_lowp<false, NT, KS>), fgrid, dim3(256), 0, ctx->stream, tnf_dev, perm, n,
                                   gram_r, frag, frag_a);
            if (!direct) {
                MDET_TRY(ctx_buf(ctx, "pairs.pfrag", (size_t)n_pad / 32 * PROJ_KS * 64, &pfrag));
                MDET_TRY(ctx_buf(ctx, "pairs.pfrag_a", (size_t)n_pad / 32 * 64, &pfrag_a));
                MDET_TRY(proj_frags(ctx, order, n, n_pad, reach, pfrag, pfrag_a));
                MDET_TRY(ctx_buf(ctx, "pairs.pbox", (size_t)PROJ_D * box_tiles, &pbox));
                MDET_TRY(ctx_buf(ctx, "pairs.pbox_m", (size_t)box_tiles, &pbox_margin));
                MDET_TRY(proj_boxes(ctx, order, n, box_tiles, box_tiles, pbox, pbox_margin));
                const uint32_t ord = tune.persistent ? tune.item_order : 0u;
                MDET_TRY(build_items(ctx, n, item_rows, seg, ord, &items, &nitems, &qbounds));
                if (!ord) qbounds = nullptr;
            }
        } else {
            // embedding rows (n x 32) in BF16, threshold = calibrated radius^2;
            // with probes, only the pairs of probed cluster pairs (items of
            // the cluster index), else every pair.  radius2 == 0 with probes:
            // the BF16 TNF Gram (as BF16_REFINE) decides within the probed
            // cluster pairs instead of the embedding radius.
            float* emb;
            MDET_TRY(ctx_buf(ctx, "learn.emb", (size_t)n * 32, &emb));
            if (exact_cover)
                MDET_TRY(ivf_cover_space(ctx, tnf_dev, n, emb));
            else
                MDET_TRY(mdet_mlp_embed(mlp, tnf_dev, n, emb));
            if (cluster) {
                MDET_TRY(ivf_launch(ctx, emb, n, n_clusters, n_probe, exact_cover, &ivf));
                perm = ivf.perm;
            }
            if (tnf_gram)
                hipLaunchKernelGGL((k_prep_lowp<true, NT, KS>), fgrid, dim3(256), 0, ctx->stream, tnf_dev, perm, n,
                                   gram_r, frag, frag_a);
            else
                hipLaunchKernelGGL((k_prep_lowp<true, 32, KS_E, true>), fgrid, dim3(256), 0, ctx->stream, emb, perm, n,
                                   std::sqrt(radius2), frag, frag_a);
            if (exact_cover) {
                // FP32 rows in cluster order for the cover's passes
                float* tnfs;
                MDET_TRY(ctx_buf(ctx, "pairs.tnfs", (size_t)n_pad * NT, &tnfs));
                hipLaunchKernelGGL(k_sort_rows, dim3(n_pad / 4), dim3(256), 0, ctx->stream, tnf_dev, perm, n, n_pad,
                                   tnfs);
                // the cover's radius: every pair the BF16 Gram can keep (unit
                // rows: the rounding of one row is at most u = 1/256)
                MDET_TRY(ivf_cover(ctx, frag, tnfs, n, (double)reach + 4.0 / 256.0 * 1.0001, &ivf));
            }
            if (cluster) {
                MDET_TRY(ivf_finish(ctx, &ivf));
                items = ivf.items_dev;
                nitems = ivf.nitems;
            } else {
                MDET_TRY(build_items(ctx, n, item_rows, seg, 0, &items, &nitems, &qbounds));
            }
            qbounds = nullptr;  // one queue
        }
        // projected rows in cluster order for the learned filter's scans (with
        // room for the fallback's full rows behind them)
        float* proj_y = nullptr;
        const uint32_t proj_T = (n_alloc / 32 + 127) / 64 * 64;
        auto project_clusters = [&]() -> int {
            MDET_TRY(proj_rows(ctx, tnf_dev, n, PROJ_BF16, &proj_y));
            MDET_TRY(ctx_buf(ctx, "pairs.pfrag", (size_t)n_alloc / 32 * PROJ_KS * 64, &pfrag));
            MDET_TRY(ctx_buf(ctx, "pairs.pfrag_a", (size_t)n_alloc / 32 * 64, &pfrag_a));
            MDET_TRY(ctx_buf(ctx, "pairs.pbox", (size_t)PROJ_D * proj_T, &pbox));
            MDET_TRY(ctx_buf(ctx, "pairs.pbox_m", (size_t)proj_T, &pbox_margin));
            const ProjOrder all{perm, proj_y};
            MDET_TRY(proj_frags(ctx, all, n, n_frag, reach, pfrag, pfrag_a));
            return proj_boxes(ctx, all, n, proj_T, proj_T, pbox, pbox_margin);
        };
        if (cluster && tnf_gram && !ivf.exact && ivf.pairs >= PROBE_PROJ_PAIRS) MDET_TRY(project_clusters());
        uint32_t* iperm = nullptr;
        if (perm) {
            MDET_TRY(ctx_buf(ctx, "sel.iperm", (size_t)n, &iperm));
            hipLaunchKernelGGL(k_iperm, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, perm, n, iperm);
        }
        MDET_HIP(hipGetLastError());
        st.pairs_evaluated = cluster ? ivf.pairs : st.pairs_total;

        // -- both passes over the pairs and the selection, again with larger
        // buffers if a list did not fit (its counter says how much it needs)
        const uint64_t ntiles = (n + 31) / 32;
        PassCaps caps{};
        caps.list = std::min<uint64_t>(ntiles * (ntiles + 1) / 2, std::max<uint64_t>(1u << 16, 8ull * n));
        caps.surv = direct ? ntiles * (ntiles + 1) / 2 : std::max<uint64_t>(1u << 16, 2ull * n);
        caps.cand = 128ull * n + 65536;
        if (auto it = ctx->bufs.find("pairs.tiles"); it != ctx->bufs.end())
            caps.list = std::max<uint64_t>(caps.list, it->second.bytes / sizeof(uint4));
        if (auto it = ctx->bufs.find("pairs.stiles"); it != ctx->bufs.end())
            caps.surv = std::max<uint64_t>(caps.surv, it->second.bytes / sizeof(uint4));
        if (auto it = ctx->bufs.find("pairs.cand"); it != ctx->bufs.end())
            caps.cand = std::max<uint64_t>(caps.cand, it->second.bytes / sizeof(Cand));
        for (int attempt = 0;; ++attempt) {
            if (attempt == mdet::PASS_MAX) MDET_FAIL(MDET_E_STATE, "mdet_tnf_edges: survivor count grew between passes");
            if (attempt) MDET_HIP(hipMemsetAsync(ctr + CTR_LIST, 0, (zero_words - 2 * CTR_LIST) * 4, ctx->stream));
            uint4* list = nullptr;
            Cand* cand;
            uint64_t* amb;
            MDET_TRY(ctx_buf(ctx, "pairs.cand", caps.cand, &cand));
            MDET_TRY(ctx_buf(ctx, "pairs.amb", caps.cand, &amb));
            if (!direct) MDET_TRY(ctx_buf(ctx, "pairs.tiles", caps.list, &list));
            // -- first pass: the tiles
            MDET_TRY(tm.record(1));
            if (!direct && nitems) {
                // persistent blocks: the resident ones pull items from a
                // counter, or with per-XCD queues (qbounds) each from its
                // queue's counter (the grid then covers every queue)
                uint32_t* pf_ctr = tune.persistent ? reinterpret_cast<uint32_t*>(ctr + CTR_QUEUES) : nullptr;
                const TileList tl{list, ctr + CTR_LIST, (unsigned long long)caps.list};
                auto grid = [&](uint32_t per_cu) {
                    const uint32_t resident = (uint32_t)ctx->num_cus * per_cu;
                    if (!pf_ctr) return dim3(nitems);
                    if (qbounds)
                        return dim3((std::max<uint32_t>(resident, PF_QUEUES) + PF_QUEUES - 1) / PF_QUEUES * PF_QUEUES);
                    return dim3(std::min<uint32_t>(nitems, resident));
                };
                const dim3 block(64 * SCAN_WAVES);
                if (proj_y)
                    // tens of thousands of small items: a block each (a returning
                    // atomic an item on the one queue bound it, 300 us at 200,000)
                    hipLaunchKernelGGL(k_box_scan, dim3(nitems), block, 0, ctx->stream,
                                       BoxArgs{pfrag, pfrag_a, proj_T, reach, items, nitems, nullptr, nullptr, tl},
                                       pbox, pbox_margin);
                else if (gram_all)
                    hipLaunchKernelGGL(k_box_scan, grid(6), block, 0, ctx->stream,
                                       BoxArgs{pfrag, pfrag_a, box_tiles, reach, items, nitems, pf_ctr, qbounds, tl},
                                       pbox, pbox_margin);
                else if (tnf_gram)
                    hipLaunchKernelGGL((k_tile_scan<KS, GRAM_RT, GRAM_CT, 2>), grid(2), block, 0, ctx->stream, frag,
                                       frag_a, items, nitems, pf_ctr, tl);
                else
                    hipLaunchKernelGGL((k_tile_scan<KS_E, GRAM_RT, GRAM_CT, 4>), grid(4), block, 0, ctx->stream, frag,
                                       frag_a, items, nitems, pf_ctr, tl);
                MDET_HIP(hipGetLastError());
            }
            MDET_TRY(tm.record(2));
            // -- second pass: the tiles' pairs
            SurvTiles sv{nullptr, nullptr, ctr + CTR_SURV, (unsigned long long)caps.surv, ctr + CTR_CAND};
            MDET_TRY(ctx_buf(ctx, "pairs.stiles", caps.surv, &sv.buf));
            MDET_TRY(ctx_buf(ctx, "pairs.smask", caps.surv * 64, &sv.mask));
            const RowArgs rows{tnf_dev, tvec, perm, n, nullptr, 0};
            // persistent blocks over the device's counts (a multiple of 8: one
            // XCD each in turn), no more than a small input has tiles for
            auto work_grid = [&](uint64_t per_cu, uint64_t most) {
                return dim3((unsigned)((std::min<uint64_t>(ctx->num_cus * per_cu, most) + 7) / 8 * 8));
            };
            const uint64_t most = direct ? ntiles * (ntiles + 1) / 2 : ~0ull;
            const dim3 ggrid = work_grid(8, most / 8 + 1);
            const dim3 rgrid = work_grid(std::min<uint32_t>(tune.refine_blocks, REFINE_PER_CU), most);
            GramArgs ga{};
            ga.frag = frag;
            ga.frag_a = frag_a;
            ga.items = direct ? nullptr : items;
            ga.whole = make_uint4(0, n, 0, n | ITEM_TRI);
            ga.list = list;
            ga.n_list = ctr + CTR_LIST;
            ga.list_cap = caps.list;
            ga.ntiles = (uint32_t)ntiles;
            ga.out = sv;
            if (f32) {
                const F32Args fa{rows, list, ctr + CTR_LIST, (unsigned long long)caps.list, (uint32_t)ntiles, f32_r2,
                                 sv};
                hipLaunchKernelGGL(k_tile_f32, rgrid, dim3(256), 0, ctx->stream, fa);
            } else if (!tnf_gram) {
                hipLaunchKernelGGL((k_tile_gram<true, KS_E, false>), ggrid, dim3(256), 0, ctx->stream, ga);
            } else if (bf) {
                hipLaunchKernelGGL((k_tile_gram<true, KS, false>), ggrid, dim3(256), 0, ctx->stream, ga);
            } else {
                hipLaunchKernelGGL((k_tile_gram<false, KS, false>), ggrid, dim3(256), 0, ctx->stream, ga);
            }
            RefineArgs ra{rows, sv, (float)T, cand, (unsigned long long)caps.cand, ctr + CTR_KEPT, bcnt, amb,
                          ctr + CTR_AMB};
            hipLaunchKernelGGL(k_tile_refine, rgrid, dim3(256), 0, ctx->stream, ra);
            const dim3 agrid(2 * ctx->num_cus);
            hipLaunchKernelGGL(k_adjudicate, agrid, dim3(256), 0, ctx->stream, tnf_dev, logsize_dev, iperm, T, rule,
                               cutoff, amb, ctr + CTR_AMB, cand, ctr + CTR_KEPT, bcnt);
            MDET_HIP(hipGetLastError());
            // what kernels may read of the candidates without the host, and
            // whether the counters at host[] ask for another pass
            const Records records{cand, ctr, caps};
            auto too_small = [&]() { return mdet::grow_lists(pass_counts(host), caps); };
            // -- learned mode with the cluster index and the TNF Gram: the exact
            // fallback for full rows
            uint64_t ns1 = 0;
            const bool fallback = cluster && tnf_gram && max_edges > 0 && ctx->learned_fallback && !ivf.exact;
            if (fallback) {
                // rows whose proposals fill all but max_edges / margin_div of the
                // slots (a row that missed more partners than that and still
                // exceeds max_edges in truth can keep a wrong edge)
                const uint32_t need = max_edges - max_edges / ctx->learned_margin_div;
                uint32_t *kept, *full_pos, *full_ids;
                uint8_t* full;
                MDET_TRY(ctx_buf(ctx, "fb.kept", (size_t)n, &kept));
                MDET_TRY(ctx_buf(ctx, "fb.full", (size_t)n, &full));
                MDET_TRY(ctx_buf(ctx, "fb.pos", (size_t)n, &full_pos));
                MDET_TRY(ctx_buf(ctx, "fb.ids", (size_t)n, &full_ids));
                uint32_t* n_full_dev = reinterpret_cast<uint32_t*>(ctr + CTR_FULL);
                MDET_HIP(hipMemsetAsync(kept, 0, (size_t)n * 4, ctx->stream));
                hipLaunchKernelGGL(k_row_kept, dim3(8u * ctx->num_cus), dim3(256), 0, ctx->stream, records, iperm,
                                   kept);
                hipLaunchKernelGGL(k_full_flags, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, kept, n, need, full);
                hipcub::CountingInputIterator<uint32_t> pos_it(0);
                size_t tmp = 0;
                MDET_HIP(hipcub::DeviceSelect::Flagged(nullptr, tmp, pos_it, full, full_pos, n_full_dev, (int)n,
                                                       ctx->stream));
                void* t;
                MDET_TRY(ctx_buf(ctx, "cub.selecttmp", tmp, &t));
                MDET_HIP(hipcub::DeviceSelect::Flagged(t, tmp, pos_it, full, full_pos, n_full_dev, (int)n, ctx->stream));
                MDET_HIP(hipMemcpyAsync(host, ctr, 8 * CTR_HOST, hipMemcpyDeviceToHost, ctx->stream));
                MDET_HIP(hipStreamSynchronize(ctx->stream));
                if (too_small()) continue;
                ns1 = host[CTR_CAND];
                const uint32_t n_full = ns1 ? (uint32_t)host[CTR_FULL] : 0;
                st.fallback_rows = n_full;
                if (n_full) {
                    const bool projected = proj_y || (uint64_t)n_full * n >= PROJ_PAIRS;
                    // the full rows' fragments after the first n_frag rows
                    hipLaunchKernelGGL(k_gather_ids, dim3((n_full + 255) / 256), dim3(256), 0, ctx->stream, full_pos,
                                       perm, n_full, full_ids);
                    const uint32_t n_fpad = (n_full + ITEM_ROWS - 1) / ITEM_ROWS * ITEM_ROWS;
                    hipLaunchKernelGGL((k_prep_lowp<true, NT, KS>), dim3(n_fpad / 32), dim3(256), 0, ctx->stream,
                                       tnf_dev, full_ids, n_full, gram_r, frag + (size_t)n_frag / 32 * KS * 64,
                                       frag_a + (size_t)n_frag / 32 * 64);
                    // items: a block's full rows x 4096 columns, taken by resident blocks
                    // in column-segment-major order, so that the blocks in flight
                    // share a segment's column fragments in L2 (the full rows'
                    // fragments are the small, reused side)
                    constexpr uint32_t FB_SEG = 4096;
                    uint32_t w = 0;
                    const uint32_t nseg = (n + FB_SEG - 1) / FB_SEG;
                    void* hi;
                    MDET_TRY(ctx_host_buf(ctx, "fb.h_items", (size_t)(n_fpad / ITEM_ROWS) * nseg * sizeof(uint4), &hi));
                    const uint32_t fb_rows = projected ? scan_rows(PROJ_RT) : ITEM_ROWS;
                    uint4* hitems = static_cast<uint4*>(hi);
                    for (uint32_t c0 = 0; c0 < n; c0 += FB_SEG)
                        for (uint32_t r0 = 0; r0 < n_full; r0 += fb_rows)
                            hitems[w++] = make_uint4(n_frag + r0, n_frag + std::min(r0 + fb_rows, n_full), c0,
                                                     std::min(c0 + FB_SEG, n));
                    uint4* fitems;
                    MDET_TRY(ctx_buf(ctx, "fb.items", (size_t)w, &fitems));
                    MDET_HIP(hipMemcpyAsync(fitems, hitems, (size_t)w * sizeof(uint4), hipMemcpyHostToDevice,
                                            ctx->stream));
                    uint32_t* pbits;
                    const uint64_t nbits = (uint64_t)ivf.k * ivf.k;
                    MDET_TRY(ctx_buf(ctx, "fb.pbits", (size_t)(nbits + 31) / 32, &pbits));
                    MDET_HIP(hipMemsetAsync(pbits, 0, (size_t)(nbits + 31) / 32 * 4, ctx->stream));
                    hipLaunchKernelGGL(k_probed_bits, dim3((unsigned)(((uint64_t)ivf.k * ivf.n_probe + 255) / 256)),
                                       dim3(256), 0, ctx->stream, ivf.probes_dev, ivf.k, ivf.n_probe, pbits);
                    caps.fb_list = std::max<uint64_t>(caps.fb_list, std::max<uint64_t>(1u << 16, 64ull * n_full));
                    if (auto it = ctx->bufs.find("fb.tiles"); it != ctx->bufs.end())
                        caps.fb_list = std::max<uint64_t>(caps.fb_list, it->second.bytes / sizeof(uint4));
                    uint4* flist;
                    uint64_t* amb2;
                    MDET_TRY(ctx_buf(ctx, "fb.tiles", caps.fb_list, &flist));
                    MDET_TRY(ctx_buf(ctx, "fb.amb", caps.cand, &amb2));
                    const TileList tl{flist, ctr + CTR_FB_LIST, (unsigned long long)caps.fb_list};
                    uint32_t* const fb_ctr = reinterpret_cast<uint32_t*>(ctr + CTR_FB_QUEUE);
                    auto fb_grid = [&](uint32_t per_cu) {
                        return dim3(std::min<uint32_t>(w, (uint32_t)ctx->num_cus * per_cu));
                    };
                    if (projected) {
                        if (!proj_y) MDET_TRY(project_clusters());
                        ProjOrder some{full_ids, proj_y};
                        const uint32_t ct = n_frag / 32;
                        MDET_TRY(proj_frags(ctx, some, n_full, n_fpad, reach, pfrag + (size_t)ct * PROJ_KS * 64,
                                            pfrag_a + (size_t)ct * 64));
                        MDET_TRY(proj_boxes(ctx, some, n_full, proj_T - ct, proj_T, pbox + ct, pbox_margin + ct));
                        hipLaunchKernelGGL(k_box_scan, fb_grid(6), dim3(64 * SCAN_WAVES), 0, ctx->stream,
                                           BoxArgs{pfrag, pfrag_a, proj_T, reach, fitems, w, fb_ctr, nullptr, tl}, pbox,
                                           pbox_margin);
                    } else {
                        hipLaunchKernelGGL((k_tile_scan<KS, GRAM_RT, GRAM_CT, 2>), fb_grid(2), dim3(64 * SCAN_WAVES), 0,
                                           ctx->stream, frag, frag_a, fitems, w, fb_ctr, tl);
                    }
                    // its survivor tiles after the first phase's are worked off
                    sv.cnt = ctr + CTR_FB_SURV;
                    ga.items = fitems;
                    ga.list = flist;
                    ga.n_list = ctr + CTR_FB_LIST;
                    ga.list_cap = caps.fb_list;
                    ga.out = sv;
                    ga.full_pos = full_pos;
                    ga.full_base = n_frag;
                    ga.full = full;
                    ga.cl = ivf.cluster_dev;
                    ga.bits = pbits;
                    ga.k = ivf.k;
                    ra.in = sv;
                    ra.amb = amb2;
                    ra.amb_cnt = ctr + CTR_AMB2;
                    ra.rows.full_pos = full_pos;
                    ra.rows.full_base = n_frag;
                    hipLaunchKernelGGL((k_tile_gram<true, KS, true>), ggrid, dim3(256), 0, ctx->stream, ga);
                    hipLaunchKernelGGL(k_tile_refine, rgrid, dim3(256), 0, ctx->stream, ra);
                    hipLaunchKernelGGL(k_adjudicate, agrid, dim3(256), 0, ctx->stream, tnf_dev, logsize_dev, iperm, T,
                                       rule, cutoff, amb2, ctr + CTR_AMB2, cand, ctr + CTR_KEPT, bcnt);
                    MDET_HIP(hipGetLastError());
                }
            }
            MDET_TRY(tm.record(3));

            // -- select: no host round trip up to the edges, with every buffer
            // sized by the candidates' capacity; large inputs wait for the
            // counters and take what the kept candidates need
            uint64_t sel_cap = caps.cand;
            if (n > COUNTED_SELECT) {
                MDET_HIP(hipMemcpyAsync(host, ctr, 8 * CTR_HOST, hipMemcpyDeviceToHost, ctx->stream));
                MDET_HIP(hipStreamSynchronize(ctx->stream));
                if (too_small()) continue;
                sel_cap = std::max<uint64_t>(host[CTR_KEPT], 1);
            }
            uint64_t *boff, *eoff, *rbeg;
            Ent* ent;
            Adj* adj;
            MDET_TRY(ctx_buf(ctx, "sel.boff", (size_t)nb + 1, &boff));
            MDET_TRY(ctx_buf(ctx, "sel.rbeg", (size_t)n, &rbeg));
            MDET_TRY(ctx_buf(ctx, "sel.eoff", (size_t)n + 1, &eoff));
            MDET_TRY(ctx_buf(ctx, "sel.ent", 2 * sel_cap, &ent));
            MDET_TRY(ctx_buf(ctx, "sel.adj", 2 * sel_cap, &adj));
            unsigned int* err = reinterpret_cast<unsigned int*>(ctr + CTR_ERR);
            unsigned long long* capped = ctr + CTR_CAPPED;
            // rows for the block-wide path (big) and for the global-memory path (huge)
            const uint32_t big_cap = std::min<uint32_t>(n, 1u << 20);
            uint32_t *big_rec, *huge_rec;
            MDET_TRY(ctx_buf(ctx, "sel.big", (size_t)BIG_REC * big_cap, &big_rec));
            MDET_TRY(ctx_buf(ctx, "sel.huge", (size_t)BIG_REC * big_cap, &huge_rec));
            const RowList big{big_rec, reinterpret_cast<uint32_t*>(ctr + CTR_BIG), big_cap};
            const RowList huge{huge_rec, reinterpret_cast<uint32_t*>(ctr + CTR_HUGE), big_cap};
            uint32_t *from, *to;
            float* s;
            MDET_TRY(ctx_buf(ctx, "out.from", sel_cap, &from));
            MDET_TRY(ctx_buf(ctx, "out.to", sel_cap, &to));
            MDET_TRY(ctx_buf(ctx, "out.s", sel_cap, &s));
            MDET_TRY(exclusive_scan_u32_to_u64(ctx, bcnt, boff, nb));
            const uint64_t pieces = (caps.cand + 255) / 256;
            hipLaunchKernelGGL(k_bucket_fill, dim3((unsigned)std::min<uint64_t>(pieces, 16u * ctx->num_cus)), dim3(256),
                               0, ctx->stream, records, iperm, boff, bcur, ent);
            hipLaunchKernelGGL(k_bucket_select, dim3(nb), dim3(S_THREADS), 0, ctx->stream, records, boff, ent, adj, n,
                               max_edges, perm, tnf_dev, logsize_dev, out_cnt, rbeg, big, err, capped);
            hipLaunchKernelGGL(k_bigrow_select, dim3(ctx->num_cus), dim3(S_THREADS), 0, ctx->stream, big, adj,
                               max_edges, tnf_dev, logsize_dev, out_cnt, rbeg, huge, err, capped);
            MDET_HIP(hipGetLastError());
            auto emit = [&]() -> int {
                MDET_TRY(exclusive_scan_u32_to_u64(ctx, out_cnt, eoff, n));
                hipLaunchKernelGGL(k_emit, dim3((n + 4 * EMIT_ROWS - 1) / (4 * EMIT_ROWS)), dim3(256), 0,
                                   ctx->stream, rbeg, adj, out_cnt, eoff, n, from, to, s, ctr + CTR_EDGES);
                MDET_HIP(hipGetLastError());
                MDET_HIP(hipMemcpyAsync(host, ctr, 8 * CTR_HOST, hipMemcpyDeviceToHost, ctx->stream));
                MDET_TRY(tm.record(4));
                MDET_HIP(hipStreamSynchronize(ctx->stream));
                return MDET_OK;
            };
            MDET_TRY(emit());
            if (too_small()) continue;
            if ((unsigned int)host[CTR_ERR] & 4u)
                MDET_FAIL(MDET_E_CAPACITY, "mdet_tnf_edges: more than %u rows need the block-wide selection", big_cap);
            if ((unsigned int)host[CTR_ERR] & 8u)
                MDET_FAIL(MDET_E_CAPACITY, "mdet_tnf_edges: more than %u rows need the global-memory selection",
                          big_cap);
            const uint32_t nhuge = (uint32_t)host[CTR_HUGE];
            if (nhuge) {
                // rows beyond the LDS capacities: sort them in global scratch
                uint32_t* rec_h;
                MDET_TRY(ctx_host_buf(ctx, "sel.huge_h", (size_t)BIG_REC * 4 * nhuge, (void**)&rec_h));
                uint64_t* soff_h;
                MDET_TRY(ctx_host_buf(ctx, "sel.huge_off_h", (size_t)8 * nhuge, (void**)&soff_h));
                MDET_HIP(hipMemcpyAsync(rec_h, huge_rec, (size_t)BIG_REC * 4 * nhuge, hipMemcpyDeviceToHost,
                                        ctx->stream));
                MDET_HIP(hipStreamSynchronize(ctx->stream));
                uint64_t total = 0;
                for (uint32_t q = 0; q < nhuge; ++q) {
                    uint64_t sz = 1;
                    while (sz < rec_h[BIG_REC * q + 1]) sz <<= 1;
                    soff_h[q] = total;
                    total += sz;
                }
                unsigned long long* sk64;
                uint32_t *sk32, *sv;
                float* spre;
                uint64_t* soff;
                MDET_TRY(ctx_buf(ctx, "sel.huge_k64", total, &sk64));
                MDET_TRY(ctx_buf(ctx, "sel.huge_k32", total, &sk32));
                MDET_TRY(ctx_buf(ctx, "sel.huge_v", total, &sv));
                MDET_TRY(ctx_buf(ctx, "sel.huge_pre", total, &spre));
                MDET_TRY(ctx_buf(ctx, "sel.huge_off", nhuge, &soff));
                MDET_HIP(hipMemcpyAsync(soff, soff_h, (size_t)8 * nhuge, hipMemcpyHostToDevice, ctx->stream));
                hipLaunchKernelGGL(k_hugerow_select, dim3(nhuge), dim3(HUGE_THREADS), 0, ctx->stream, huge_rec, soff,
                                   adj, max_edges, tnf_dev, logsize_dev, sk64, sk32, sv, spre, out_cnt, rbeg, capped);
                MDET_HIP(hipGetLastError());
                MDET_TRY(emit());
            }
            st.survivors = ns1 ? ns1 : host[CTR_CAND];
            st.fallback_pairs = ns1 ? host[CTR_CAND] - ns1 : 0;
            st.fallback_chunks = host[CTR_FB_LIST];
            st.pairs_evaluated += st.fallback_rows * (uint64_t)(n - 1);  // some counted in phase one too
            st.candidates = host[CTR_KEPT];
            st.adjudicated = host[CTR_ADJ];
            st.rows_block = std::min<uint64_t>((uint32_t)host[CTR_BIG], big_cap);
            st.rows_global = nhuge;
            st.rows_capped = host[CTR_CAPPED];
            ctx->last_pairs = st.survivors;
            result = mdet_edges{host[CTR_EDGES], from, to, s};
            break;
        }
    } else {
        MDET_TRY(tm.record(1));
        MDET_TRY(tm.record(2));
        MDET_TRY(tm.record(3));
        MDET_TRY(tm.record(4));
        MDET_HIP(hipEventSynchronize(ctx->events[4]));
    }
    st.ms_prefilter = tm.ms(1, 2);
    st.ms_refine = tm.ms(2, 3);
    st.ms_select = tm.ms(3, 4);
    st.ms_total = tm.ms(0, 4);
    *out = result;
    if (stats) *stats = st;
    return MDET_OK;
}

}  // namespace

extern "C" {

int mdet_tnf_edges(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n, double cutoff,
                   uint32_t max_edges, int precision, mdet_edges* out, mdet_pair_stats* stats) {
    if (precision == MDET_LEARNED)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_edges: the learned mode needs mdet_tnf_edges_learned");
    return edges_impl(ctx, tnf_dev, logsize_dev, n, cutoff, max_edges, precision, nullptr, 0.f, 0, 0, out, stats);
}

int mdet_tnf_prob_edges(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n,
                        double required_min_p, int precision, mdet_edges* out, mdet_pair_stats* stats) {
    if (precision == MDET_LEARNED)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_prob_edges: precision must be EXACT_F32, BF16_REFINE or F16_REFINE");
    return edges_impl(ctx, tnf_dev, logsize_dev, n, required_min_p, 0, precision, nullptr, 0.f, 0, 0, out, stats,
                      RULE_PROB);
}

int mdet_tnf_edges_learned(mdet_ctx* ctx, mdet_mlp* mlp, const float* tnf_dev, const double* logsize_dev, uint32_t n,
                           double cutoff, uint32_t max_edges, float radius2, uint32_t n_clusters, uint32_t n_probe,
                           mdet_edges* out, mdet_pair_stats* stats) {
    return edges_impl(ctx, tnf_dev, logsize_dev, n, cutoff, max_edges, MDET_LEARNED, mlp, radius2, n_clusters, n_probe,
                      out, stats);
}

int mdet_tune_get(mdet_ctx* ctx, int precision, mdet_tune* out) {
    MDET_TRY(check_ctx(ctx));
    if (precision < MDET_EXACT_F32 || precision > MDET_LEARNED || !out)
        MDET_FAIL(MDET_E_INVALID, "mdet_tune_get: bad precision %d or null output", precision);
    const mdet_ctx::Tune& t = ctx->tune[precision];
    *out = mdet_tune{t.seg_cols, t.persistent, t.refine_blocks, t.item_order, t.ms_prefilter, t.ms_refine};
    return MDET_OK;
}

int mdet_learned_set_fallback(mdet_ctx* ctx, int enabled) {
    MDET_TRY(check_ctx(ctx));
    ctx->learned_fallback = enabled != 0;
    return MDET_OK;
}

int mdet_learned_set_exact_cover(mdet_ctx* ctx, int enabled) {
    MDET_TRY(check_ctx(ctx));
    ctx->learned_exact_cover = enabled != 0;
    return MDET_OK;
}

int mdet_learned_set_fallback_margin(mdet_ctx* ctx, uint32_t margin_div) {
    MDET_TRY(check_ctx(ctx));
    if (margin_div == 0) MDET_FAIL(MDET_E_INVALID, "mdet_learned_set_fallback_margin: divisor 0");
    ctx->learned_margin_div = margin_div;
    return MDET_OK;
}

int mdet_tune_set(mdet_ctx* ctx, int precision, const mdet_tune* in) {
    MDET_TRY(check_ctx(ctx));
    if (precision < MDET_EXACT_F32 || precision > MDET_LEARNED || !in)
        MDET_FAIL(MDET_E_INVALID, "mdet_tune_set: bad precision %d or null input", precision);
    if (in->seg_cols != 0 && (in->seg_cols < ITEM_ROWS || in->seg_cols > 65536 || in->seg_cols % ITEM_ROWS))
        MDET_FAIL(MDET_E_RANGE, "mdet_tune_set: seg_cols %u is neither 0 nor a multiple of %d in [%d, 65536]",
                  in->seg_cols, (int)ITEM_ROWS, (int)ITEM_ROWS);
    if (in->persistent > 1) MDET_FAIL(MDET_E_RANGE, "mdet_tune_set: persistent must be 0 or 1");
    if (in->refine_blocks < 1 || in->refine_blocks > 64)
        MDET_FAIL(MDET_E_RANGE, "mdet_tune_set: refine_blocks %u outside [1, 64]", in->refine_blocks);
    if (in->item_order > 1) MDET_FAIL(MDET_E_RANGE, "mdet_tune_set: item_order must be 0 or 1");
    mdet_ctx::Tune& t = ctx->tune[precision];
    t.seg_cols = in->seg_cols;
    t.persistent = in->persistent;
    t.refine_blocks = in->refine_blocks;
    t.item_order = in->item_order;
    t.ms_prefilter = in->ms_prefilter;
    t.ms_refine = in->ms_refine;
    return MDET_OK;
}

}  // extern "C"

namespace {

// Times the launch shapes of the first pass on this input and keeps the
// fastest in ctx->tune[precision]: item column span for the Gram modes x {one
// block per item, persistent blocks with one queue, persistent blocks with
// per-XCD queues}, by the median stage time over reps calls, the shape of an
// untuned context first and kept unless another beats it (tuned_shape_wins).
// Inputs that skip the pass leave the shape as it is: there is nothing to time,
// and a larger input on the same context uses it.  The refinement launches the
// blocks that fit (REFINE_PER_CU), one launch for all settings from there on:
// it stays at the default and is timed at it.  Every shape gives the same edge
// list; the last call's list stays in ctx.
int autotune_impl(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n, double cutoff,
                  uint32_t max_edges, int precision, mdet_mlp* mlp, float radius2, uint32_t n_clusters,
                  uint32_t n_probe, uint32_t reps, mdet_tune* out) {
    MDET_TRY(check_ctx(ctx));
    if (precision < MDET_EXACT_F32 || precision > MDET_LEARNED)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_autotune: bad precision %d", precision);
    reps = std::max<uint32_t>(1, std::min<uint32_t>(reps, 15));
    mdet_ctx::Tune& t = ctx->tune[precision];
    const mdet_ctx::Tune saved = t;
    mdet_edges e;
    mdet_pair_stats st;
    auto call = [&]() {
        return edges_impl(ctx, tnf_dev, logsize_dev, n, cutoff, max_edges, precision, mlp, radius2, n_clusters,
                          n_probe, &e, &st);
    };
    auto median_of = [&](double mdet_pair_stats::*field, double* ms) -> int {
        std::vector<double> v;
        for (uint32_t r = 0; r < reps; ++r) {
            MDET_TRY(call());
            v.push_back(st.*field);
        }
        std::sort(v.begin(), v.end());
        *ms = v[v.size() / 2];
        return MDET_OK;
    };
    auto fail = [&](int rc) {
        t = saved;
        return rc;
    };
    if (int rc = call(); rc != MDET_OK) return fail(rc);  // first-call allocations at the current shape
    // 1. the first pass's shape
    struct Shape {
        uint32_t seg, pers, order;
    };
    std::vector<Shape> shapes;
    if (precision == MDET_BF16_REFINE || precision == MDET_F16_REFINE) {
        for (uint32_t seg : n > DIRECT_MAX ? tune_spans(n) : std::vector<uint32_t>())
            for (const Shape sh : {Shape{seg, 1u, 1u}, Shape{seg, 1u, 0u}, Shape{seg, 0u, 0u}}) shapes.push_back(sh);
    } else if (precision == MDET_LEARNED) {
        for (uint32_t pers : {1u, 0u}) shapes.push_back({t.seg_cols, pers, t.item_order});
    }
    double best_pre = 0;
    if (!shapes.empty()) {
        best_pre = 1e300;
        Shape best = shapes[0];
        for (const auto& sh : shapes) {
            t.seg_cols = sh.seg;
            t.persistent = sh.pers;
            t.item_order = sh.order;
            double ms;
            if (int rc = median_of(&mdet_pair_stats::ms_prefilter, &ms); rc != MDET_OK) return fail(rc);
            if (tuned_shape_wins(ms, best_pre)) {
                best_pre = ms;
                best = sh;
            }
        }
        t.seg_cols = best.seg;
        t.persistent = best.pers;
        t.item_order = best.order;
    }
    // 2. the refinement at that shape
    t.refine_blocks = mdet_ctx::Tune().refine_blocks;
    double best_ref;
    if (int rc = median_of(&mdet_pair_stats::ms_refine, &best_ref); rc != MDET_OK) return fail(rc);
    t.ms_prefilter = best_pre;
    t.ms_refine = best_ref;
    if (out) *out = mdet_tune{t.seg_cols, t.persistent, t.refine_blocks, t.item_order, t.ms_prefilter, t.ms_refine};
    return MDET_OK;
}

// Up to here k_rowmax alone (one step of columns a block); from n = 300 on it
// took 4x and more of the scans' time.
constexpr uint32_t RM_DIRECT_MAX = 64;
constexpr uint32_t RM_LIST_PER_ROW = 32;  // list capacity (2-5 a row measured)

// The MFMA row maxima (see k_rm_scan): m64 of every sampled position unless
// *outside is set or the list (its length: *n_list) overflows.
int rowmax_mfma(mdet_ctx* ctx, const float* tnf_dev, const double* ls, const float* tvec, const uint64_t* idx,
                uint32_t n, uint32_t ns, uint32_t* best, unsigned long long* m64, unsigned long long* n_list,
                RmArgs* out) {
    const hipStream_t s = ctx->stream;
    const uint32_t tiles = (n + 31) / 32, ctiles = (ns + 31) / 32, m2 = ns == n ? 0 : ns;  // a second order
    uint32_t *key, *val, *order, *contig, *rank;
    uint4 *frag, *frag_a, *pfrag, *tfrag;
    float *err, *tile_err;
    const size_t all = (size_t)tiles * 32 + (m2 ? (size_t)ctiles * 32 : 0);
    MDET_TRY(ctx_buf(ctx, "rm.key", 2 * (size_t)n, &key));
    MDET_TRY(ctx_buf(ctx, "rm.val", n, &val));
    MDET_TRY(ctx_buf(ctx, "rm.order", all, &order));
    MDET_TRY(ctx_buf(ctx, "rm.contig", all, &contig));
    MDET_TRY(ctx_buf(ctx, "rm.rank", n, &rank));
    MDET_TRY(ctx_buf(ctx, "rm.frag", all * 2 * KS, &frag));
    MDET_TRY(ctx_buf(ctx, "rm.frag_a", all * 2, &frag_a));
    MDET_TRY(ctx_buf(ctx, "rm.err", all, &err));
    MDET_TRY(ctx_buf(ctx, "rm.pfrag", (size_t)tiles * 2 * 4 * RM_PKS * 64, &pfrag));
    MDET_TRY(ctx_buf(ctx, "rm.tile_err", tiles, &tile_err));
    MDET_TRY(ctx_buf(ctx, "rm.tfrag", (size_t)ctiles * RM_PKS * 64, &tfrag));
    RmArgs A{};
    A.cap = RM_LIST_PER_ROW * ns;
    MDET_TRY(ctx_buf(ctx, "rm.list", (size_t)A.cap, &A.list));
    A.n_list = n_list;
    uint32_t* outside = reinterpret_cast<uint32_t*>(n_list + 1);
    A.outside = outside;
    A.best = best;
    auto sorted = [&](uint32_t m, uint32_t off, uint32_t* rk) -> int {
        const dim3 g((m + 255) / 256), b(256);
        hipLaunchKernelGGL(k_rm_keys, g, b, 0, s, tvec, idx, m, key, val);
        size_t tmp = 0;
        MDET_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key, key + n, val, order + off, (int)m, 0, 32, s));
        void* t;
        MDET_TRY(ctx_buf(ctx, "cub.tmp", tmp, &t));
        MDET_HIP(hipcub::DeviceRadixSort::SortPairs(t, tmp, key, key + n, val, order + off, (int)m, 0, 32, s));
        hipLaunchKernelGGL(k_rm_contigs, g, b, 0, s, idx, order + off, m, contig + off, rk);
        hipLaunchKernelGGL((k_prep_lowp<false, NT, KS>), dim3((m + 31) / 32), b, 0, s, tnf_dev, contig + off, m, 0.f,
                           frag + (size_t)off * 2 * KS, frag_a + (size_t)off * 2, err + off, outside);
        return MDET_OK;
    };
    MDET_TRY(sorted(n, 0, rank));
    const uint32_t off = m2 ? tiles * 32 : 0;
    if (m2) MDET_TRY(sorted(ns, off, nullptr));
    hipLaunchKernelGGL(k_rm_poly, dim3(tiles), dim3(256), 0, s, tvec, contig, err, n, pfrag, tile_err);
    hipLaunchKernelGGL(k_rm_cheb, dim3((ctiles * 32 + 255) / 256), dim3(256), 0, s, tvec, contig + off, ns, ctiles,
                       tfrag);
    A.frag = frag;
    A.frag_a = frag_a;
    A.pfrag = pfrag;
    A.tile_err = tile_err;
    A.order = order;
    A.n = n;
    A.tiles = tiles;
    A.cfrag = frag + (size_t)off * 2 * KS;
    A.tfrag = tfrag;
    A.cerr = err + off;
    A.corder = order + off;
    A.rank = rank;
    A.ns = ns;
    A.ctiles = ctiles;
    // about 8 blocks a CU
    const uint32_t gx = (ctiles + 3) / 4, gy = std::min(tiles, std::max(1u, (8 * (uint32_t)ctx->num_cus + gx - 1) / gx));
    A.seg = (tiles + gy - 1) / gy;
    const dim3 grid(gx, (tiles + A.seg - 1) / A.seg), block(256);
    hipLaunchKernelGGL(k_rm_scan<RM_BEST1>, grid, block, 0, s, A);
    hipLaunchKernelGGL(k_rm_scan<RM_BEST2>, grid, block, 0, s, A);
    hipLaunchKernelGGL(k_rm_scan<RM_LIST>, grid, block, 0, s, A);
    hipLaunchKernelGGL(k_rm_exact, dim3(4 * (uint32_t)ctx->num_cus), dim3(64 * DIST_WAVES), 0, s, A, tnf_dev, ls, idx, m64);
    MDET_HIP(hipGetLastError());
    *out = A;
    return MDET_OK;
}

}  // namespace

extern "C" {

int mdet_tnf_autotune(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n, double cutoff,
                      uint32_t max_edges, int precision, uint32_t reps, mdet_tune* out) {
    if (precision == MDET_LEARNED)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_autotune: the learned mode needs mdet_tnf_autotune_learned");
    return autotune_impl(ctx, tnf_dev, logsize_dev, n, cutoff, max_edges, precision, nullptr, 0.f, 0, 0, reps, out);
}

int mdet_tnf_autotune_learned(mdet_ctx* ctx, mdet_mlp* mlp, const float* tnf_dev, const double* logsize_dev,
                              uint32_t n, double cutoff, uint32_t max_edges, float radius2, uint32_t n_clusters,
                              uint32_t n_probe, uint32_t reps, mdet_tune* out) {
    return autotune_impl(ctx, tnf_dev, logsize_dev, n, cutoff, max_edges, MDET_LEARNED, mlp, radius2, n_clusters,
                         n_probe, reps, out);
}

int mdet_last_pairs(mdet_ctx* ctx, const void** records_dev, uint64_t* count) {
    MDET_TRY(check_ctx(ctx));
    if (!records_dev || !count) MDET_FAIL(MDET_E_INVALID, "mdet_last_pairs: null output");
    auto it = ctx->bufs.find("pairs.cand");
    *records_dev = it == ctx->bufs.end() ? nullptr : it->second.p;
    *count = it == ctx->bufs.end() ? 0 : ctx->last_pairs;
    return MDET_OK;
}

int mdet_tnf_rowmax(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n, const uint64_t* idx_dev,
                    uint32_t n_sample, double* max_out_dev) {
    MDET_TRY(check_ctx(ctx));
    if (n_sample == 0) return MDET_OK;
    if (!tnf_dev || !logsize_dev || !idx_dev || !max_out_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_rowmax: null argument");
    if (n_sample > n) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_rowmax: n_sample %u > n %u", n_sample, n);
    MDET_TRY(ensure_model(ctx));
    float* tvec;
    unsigned long long* mm;
    unsigned long long* m64;
    MDET_TRY(ctx_buf(ctx, "rm.tvec", n, &tvec));
    MDET_TRY(ctx_buf(ctx, "rm.mm", 8, &mm));
    // m64, then m32 and the bounds (32 bits each)
    MDET_TRY(ctx_buf(ctx, "rm.max", (size_t)2 * n_sample, &m64));
    uint32_t* m32 = reinterpret_cast<uint32_t*>(m64 + n_sample);
    // mm: [0..2] log-size range and out-of-domain count, [3] listed pairs, [4] rows outside the bounds
    MDET_HIP(hipMemsetAsync(mm, 0, 64, ctx->stream));
    hipLaunchKernelGGL(k_prep_rows, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, logsize_dev, n, tvec, mm);
    unsigned long long bad = 0;
    MDET_TRY(read_scalar(ctx, mm + 2, &bad));
    if ((unsigned int)bad != 0)
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_rowmax: %u log sizes outside [log10 1500, log10 500000]", (unsigned int)bad);
    MDET_HIP(hipMemsetAsync(m64, 0, (size_t)n_sample * 16, ctx->stream));
    const uint32_t* outside = nullptr;
    uint32_t cap = 0;
    if (n > RM_DIRECT_MAX) {
        RmArgs A;
        MDET_TRY(rowmax_mfma(ctx, tnf_dev, logsize_dev, tvec, idx_dev, n, n_sample, m32 + n_sample, m64, mm + 3, &A));
        outside = A.outside;
        cap = A.cap;
    }
    const dim3 grid((n_sample + RM_ROWS - 1) / RM_ROWS, (n + RM_CHUNK - 1) / RM_CHUNK);
    hipLaunchKernelGGL(k_rowmax<false>, grid, dim3(256), 0, ctx->stream, tnf_dev, logsize_dev, tvec, idx_dev, n,
                       n_sample, m32, m64, outside, mm + 3, cap);
    hipLaunchKernelGGL(k_rowmax<true>, grid, dim3(256), 0, ctx->stream, tnf_dev, logsize_dev, tvec, idx_dev, n,
                       n_sample, m32, m64, outside, mm + 3, cap);
    hipLaunchKernelGGL(k_rowmax_final, dim3((n_sample + 255) / 256), dim3(256), 0, ctx->stream, m64, n_sample,
                       max_out_dev);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

int mdet_tnf_similarity64(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n,
                          const uint32_t* pi_dev, const uint32_t* pj_dev, uint64_t np, double* s64_dev) {
    MDET_TRY(check_ctx(ctx));
    if (np == 0) return MDET_OK;
    if (!tnf_dev || !logsize_dev || !pi_dev || !pj_dev || !s64_dev)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_similarity64: null argument");
    unsigned int* bad;
    MDET_TRY(ctx_buf(ctx, "s64.bad", 16, &bad));
    MDET_HIP(hipMemsetAsync(bad, 0, 16, ctx->stream));
    hipLaunchKernelGGL(k_similarity64, dim3((unsigned)((np + 64 * DIST_WAVES - 1) / (64 * DIST_WAVES))),
                       dim3(64 * DIST_WAVES), 0, ctx->stream, tnf_dev,
                       logsize_dev, n, pi_dev, pj_dev, np, s64_dev, bad);
    MDET_HIP(hipGetLastError());
    unsigned int nbad = 0;
    MDET_TRY(read_scalar(ctx, bad, &nbad));
    if (nbad)
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_similarity64: %u pairs index a contig >= n = %u (their outputs are NaN)",
                  nbad, n);
    return MDET_OK;
}

int mdet_tnf_preprob(mdet_ctx* ctx, const float* tnf_dev, const double* logsize_dev, uint32_t n,
                     const uint32_t* pi_dev, const uint32_t* pj_dev, uint64_t np, float* pre32_dev,
                     double* pre64_dev) {
    MDET_TRY(check_ctx(ctx));
    if (np == 0) return MDET_OK;
    if (!tnf_dev || !logsize_dev || !pi_dev || !pj_dev)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_preprob: null argument");
    if (n == 0) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_preprob: n = 0 with pairs to evaluate");
    MDET_TRY(ensure_model(ctx));
    float* tvec;
    unsigned long long* mm;
    MDET_TRY(ctx_buf(ctx, "pp.tvec", n, &tvec));
    MDET_TRY(ctx_buf(ctx, "pp.mm", 8, &mm));
    // [0..1] log-size range, [2] out-of-domain count, [3] bad indices
    MDET_HIP(hipMemsetAsync(mm, 0, 32, ctx->stream));
    hipLaunchKernelGGL(k_prep_rows, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, logsize_dev, n, tvec, mm);
    hipLaunchKernelGGL(k_preprob_pairs, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, ctx->stream, tnf_dev,
                       logsize_dev, tvec, n, pi_dev, pj_dev, np, pre32_dev, pre64_dev,
                       reinterpret_cast<unsigned int*>(mm + 3));
    MDET_HIP(hipGetLastError());
    unsigned long long chk[2];
    {
        void* st_host;
        MDET_TRY(ctx_host_stage(ctx, 64, &st_host));
        MDET_HIP(hipMemcpyAsync(st_host, mm + 2, 16, hipMemcpyDeviceToHost, ctx->stream));
        MDET_HIP(hipStreamSynchronize(ctx->stream));
        memcpy(chk, st_host, 16);
    }
    if ((unsigned int)chk[0] != 0)
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_preprob: %u log sizes outside [log10 1500, log10 500000]",
                  (unsigned int)chk[0]);
    if ((unsigned int)chk[1] != 0)
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_preprob: %u pairs index a contig >= n = %u (their outputs are NaN)",
                  (unsigned int)chk[1], n);
    return MDET_OK;
}

}  // extern "C"
