// Row order and projection of the exhaustive pair stage on gfx950 (no
// reference counterpart: the reference evaluates every pair in full).
//
// Almost every pair of contigs is far apart in a few leading directions of the
// TNF rows already.  A projection P with |P v| <= |v| gives a lower bound of
// every distance, so a 32 x 32 tile of pairs none of which is within the
// radius after 28 dimensions (2 MFMA k-steps instead of 9) needs no further
// work.  The directions come from the rows: with C their covariance over a
// sample, the span of C^2 W for a fixed random W holds most of the spread
// (measured on 200,000 contigs of 1,000 genomes: 0.8% of the tiles keep a pair
// within the radius in 28 such dimensions, 0.65% in the 28 leading principal
// components, 32% in 28 random ones).  The quality of the directions only
// decides how many tiles are dropped, never a result: the bound holds for any
// P with norm <= 1, which k_basis enforces on what it computed.
//
// The rows are visited in the order of their nearest of up to 4,096 centres
// ("row order" below): 0.14% of the 32 x 32 tiles then hold a pair within the
// radius at 200,000 contigs, against 0.44% in the order of a Morton key of the
// rows' leading coordinates and 13% in that of GC content.
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "order.h"

namespace {

using mdet::PROJ_D;
using mdet::PROJ_KS;
using mdet::PROJ_W;

constexpr int NT = 136;
constexpr uint32_t COV_SAMPLE = 2048, COV_SPLITS = 64;

// Words PROJ_D.. of a projected row.
constexpr int PW_PART = 28;  // sum of squares of the FP16-rounded coordinates
constexpr int PW_NY = 29;    // |y|
constexpr int PW_MARGIN = 30;  // what the row adds to half the radius
constexpr int PW_KIND = 31;  // 0 bounded; 1 holds a NaN or infinity (never within any radius); 2 too long for FP16

// v rounded to BF16, to nearest even (finite v)
__device__ inline float bf16_rne(float v) {
    uint32_t u = __float_as_uint(v);
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}
__device__ inline bool finite_bits(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// Sums of products, sums and count of COV_SPLITS slices of the sampled rows
// (row s * n / S); rows with a non-finite value are left out.  Thread t < 289
// owns an 8 x 8 block of the 136 x 136 products.
__global__ __launch_bounds__(320) void k_cov_part(const float* __restrict__ tnf, uint32_t n, uint32_t S,
                                                  float* __restrict__ part, float* __restrict__ msum) {
    constexpr int R = 32;
    __shared__ __align__(16) float X[R][NT + 4];
    __shared__ uint32_t bad[R];
    const uint32_t tid = threadIdx.x, per = (S + COV_SPLITS - 1) / COV_SPLITS;
    const uint32_t s0 = blockIdx.x * per, s1 = min(S, s0 + per);
    const int ti = tid / 17, tj = tid % 17;
    float acc[8][8] = {};
    float csum = 0.f, cnt = 0.f;
    for (uint32_t r0 = s0; r0 < s1; r0 += R) {
        __syncthreads();
        if (tid < R) bad[tid] = r0 + tid >= s1;
        __syncthreads();
        for (uint32_t e = tid; e < R * (NT / 4); e += 320) {
            const uint32_t r = e / (NT / 4), q = e % (NT / 4);
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r0 + r < s1) {
                const uint64_t row = (uint64_t)(r0 + r) * n / S;
                v = reinterpret_cast<const float4*>(tnf + row * NT)[q];
                if (!(finite_bits(v.x) && finite_bits(v.y) && finite_bits(v.z) && finite_bits(v.w))) bad[r] = 1;
            }
            *reinterpret_cast<float4*>(&X[r][4 * q]) = v;
        }
        __syncthreads();
        for (int r = 0; r < R; ++r) {
            if (bad[r]) continue;  // block-uniform
            if (tid < 289) {
                float a[8], b[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) a[i] = X[r][8 * ti + i];
#pragma unroll
                for (int j = 0; j < 8; ++j) b[j] = X[r][8 * tj + j];
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
            }
            if (tid < NT) csum += X[r][tid];
            cnt += 1.f;
        }
    }
    if (tid < 289)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                part[((size_t)blockIdx.x * NT + 8 * ti + i) * NT + 8 * tj + j] = acc[i][j];
    if (tid < NT) msum[blockIdx.x * (NT + 1) + tid] = csum;
    if (tid == 0) msum[blockIdx.x * (NT + 1) + NT] = cnt;
}

// Covariance C[136 x 136] and mean from the slices, added in slice order.
__global__ __launch_bounds__(256) void k_cov_sum(const float* __restrict__ part, const float* __restrict__ msum,
                                                 float* __restrict__ C, float* __restrict__ mean) {
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e >= NT * NT) return;
    const uint32_t i = e / NT, j = e % NT;
    float c = 0.f, mi = 0.f, mj = 0.f, cnt = 0.f;
#pragma unroll 8
    for (uint32_t s = 0; s < COV_SPLITS; ++s) {
        c += part[(size_t)s * NT * NT + e];
        mi += msum[s * (NT + 1) + i];
        mj += msum[s * (NT + 1) + j];
        cnt += msum[s * (NT + 1) + NT];
    }
    const float inv = cnt > 0.f ? 1.f / cnt : 0.f;
    C[e] = c * inv - (mi * inv) * (mj * inv);
    if (j == 0) mean[i] = mi * inv;
}

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// The directions, one block: V = W (random signs), twice V = orthonormal basis
// of C V (Cholesky QR of the 28 columns, the second time repeated for
// accuracy), columns ordered by their variance, then scaled so that the
// largest row sum of |P^T P|, a bound of |P|^2, is below 1.  Everything stays
// in one CU's LDS; the products are FP32 MFMAs (v_mfma_f32_32x32x2, a wave per
// 32 rows), the 28 x 28 factorisation and its inverse one wave's registers.
// Bound by these serial chains: 54 us (116 us with scalar products and a
// barrier per factorisation step).
// basis: P as [4][136][8] (coordinate 7 g + j of group g at [g][k][j]); off:
// P mean [28]; sig: standard deviation of each coordinate.
constexpr int B_THREADS = 512, B_WAVES = B_THREADS / 64, B_TILES = (NT + 31) / 32;
constexpr int B_STR = PROJ_W + 1;  // rows apart by an odd number of banks: columns are read too

// Y[136 x 32] = A B: A(m, k) row m of 136, K even, B(k, n).
template <int K, class FA, class FB>
__device__ inline void basis_product(FA A, FB B, float (*Y)[B_STR]) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int c = lane & 31, h = lane >> 5;
    if (wave < B_TILES) {
        const int m = min(32 * wave + c, NT - 1);
        f32x16_t acc = {};
#pragma unroll 4
        for (int k = 0; k < K; k += 2) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(A(m, k + h), B(k + h, c), acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 32 * wave + (r & 3) + 8 * (r >> 2) + 4 * h;
            if (row < NT) Y[row][c] = acc[r];
        }
    }
    __syncthreads();
}

// G = A^T B of two 136 x 32 matrices, the rows split over the waves.
__device__ inline void basis_gram(const float (*A)[B_STR], const float (*B)[B_STR], float (*part)[PROJ_W][B_STR],
                                  float (*G)[B_STR]) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int c = lane & 31, h = lane >> 5;
    f32x16_t acc = {};
    constexpr int PER = (NT / 2 + B_WAVES - 1) / B_WAVES;  // row pairs a wave
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int k = 2 * (wave * PER + q) + h;
        const float x = k < NT ? A[k][c] : 0.f, y = k < NT ? B[k][c] : 0.f;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][(r & 3) + 8 * (r >> 2) + 4 * h][c] = acc[r];
    __syncthreads();
    for (int e = threadIdx.x; e < PROJ_W * PROJ_W; e += B_THREADS) {
        float g = 0.f;
#pragma unroll
        for (int w = 0; w < B_WAVES; ++w) g += part[w][e / PROJ_W][e % PROJ_W];
        G[e / PROJ_W][e % PROJ_W] = g;
    }
    __syncthreads();
}

__device__ inline float lane_value(float v, int lane) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}

// V = orthonormal columns spanning Y's (Y may be V); columns whose remainder
// vanishes become zero.  G = Y^T Y = L L^T, V = Y L^-T.
__device__ inline void basis_orth(const float (*Y)[B_STR], float (*V)[B_STR], float (*part)[PROJ_W][B_STR],
                                  float (*G)[B_STR], float (*T)[B_STR]) {
    basis_gram(Y, Y, part, G);
    if (threadIdx.x < 64) {
        const int i = threadIdx.x & 31;
        float g[PROJ_D], diag[PROJ_D];  // row i of G, of L as it comes; 1 / L[k][k] (0: dropped)
        float gmax = 0.f;
#pragma unroll
        for (int k = 0; k < PROJ_D; ++k) {
            g[k] = G[i][k];
            gmax = fmaxf(gmax, G[k][k]);
        }
#pragma unroll
        for (int k = 0; k < PROJ_D; ++k) {
            const float p = lane_value(g[k], k);
            diag[k] = p > 1e-7f * gmax ? __builtin_amdgcn_rsqf(p) : 0.f;
            g[k] *= diag[k];
#pragma unroll
            for (int j = k + 1; j < PROJ_D; ++j) g[j] = fmaf(-g[k], lane_value(g[k], j), g[j]);
        }
        float x[PROJ_D];  // column i of L^-1
#pragma unroll
        for (int r = 0; r < PROJ_D; ++r) {
            float s = r == i ? 1.f : 0.f;
#pragma unroll
            for (int k = 0; k < r; ++k) s = fmaf(-lane_value(g[k], r), x[k], s);
            x[r] = s * diag[r];
        }
        if (threadIdx.x < 32)
#pragma unroll
            for (int r = 0; r < PROJ_W; ++r) T[i][r] = r < PROJ_D && i < PROJ_D ? x[r < PROJ_D ? r : 0] : 0.f;
    }
    __syncthreads();
    // (a wave reads its own 32 rows before it writes them)
    basis_product<PROJ_W>([&](int m, int k) { return Y[m][k]; }, [&](int k, int n) { return T[k][n]; }, V);
}

__global__ __launch_bounds__(B_THREADS, 2) void k_basis(const float* __restrict__ Cg, const float* __restrict__ mean,
                                                     float* __restrict__ basis, float* __restrict__ off,
                                                     float* __restrict__ sig) {
    __shared__ __align__(16) float C[NT][NT];
    __shared__ float V[NT][B_STR], Y[NT][B_STR], part[B_WAVES][PROJ_W][B_STR];
    __shared__ float G[PROJ_W][B_STR], T[PROJ_W][B_STR];
    __shared__ float var[PROJ_W], rowsum[PROJ_W], pm[16][PROJ_W], scale;
    __shared__ int place[PROJ_W];
    const int tid = threadIdx.x;
    {  // all 16-byte loads of C at once
        constexpr int LOADS = (NT * NT / 4 + B_THREADS - 1) / B_THREADS;
        f32x4_t v[LOADS];
#pragma unroll
        for (int q = 0; q < LOADS; ++q)
            v[q] = reinterpret_cast<const f32x4_t*>(Cg)[min(tid + q * B_THREADS, NT * NT / 4 - 1)];
#pragma unroll
        for (int q = 0; q < LOADS; ++q)
            if (tid + q * B_THREADS < NT * NT / 4) reinterpret_cast<f32x4_t*>(&C[0][0])[tid + q * B_THREADS] = v[q];
    }
    for (int e = tid; e < NT * PROJ_W; e += B_THREADS) {
        uint32_t h = (uint32_t)e * 0x9E3779B9u + 0x7F4A7C15u;
        h = (h ^ (h >> 16)) * 0x85EBCA6Bu;
        h = (h ^ (h >> 13)) * 0xC2B2AE35u;
        V[e / PROJ_W][e % PROJ_W] = e % PROJ_W < PROJ_D ? ((h >> 31) ? 1.f : -1.f) : 0.f;
    }
    __syncthreads();
    // C is symmetric: row k, consecutive lanes
    auto mul = [&]() {
        basis_product<NT>([&](int m, int k) { return C[k][m]; }, [&](int k, int n) { return V[k][n]; }, Y);
    };
    // one loop: straight-line copies of the factorisation are instruction misses
#pragma unroll 1
    for (int pass = 0; pass < 4; ++pass) {
        if (pass != 2) mul();
        if (pass < 3) basis_orth(pass == 2 ? V : Y, V, part, G, T);
    }
    basis_gram(V, Y, part, T);  // variances on its diagonal
    basis_gram(V, V, part, G);
    if (tid < PROJ_W) {
        var[tid] = tid < PROJ_D ? fmaxf(T[tid][tid], 0.f) : -1.f;
        float s = 0.f;
#pragma unroll
        for (int b = 0; b < PROJ_D; ++b) s += fabsf(G[tid][b]);
        rowsum[tid] = s;
    }
    {  // P mean, unscaled: 16 slices of the rows
        const int c = tid & 31, q = tid >> 5;
        float s = 0.f;
        for (int k = q; k < NT; k += 16) s = fmaf(V[k][c], mean[k], s);
        pm[q][c] = s;
    }
    __syncthreads();
    if (tid < 64) {
        const int c = tid & 31;
        float m = c < PROJ_D ? rowsum[c] : 0.f;
        const bool fine = c >= PROJ_D || (finite_bits(m) && finite_bits(var[c]));
        const bool ok = __all(fine);
#pragma unroll
        for (int o = 16; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        // |P|^2 <= the largest row sum; a basis that did not come out finite is dropped (P = 0: no tile is)
        if (tid == 0) scale = ok && m > 0.f ? 1.f / sqrtf(m * (1.f + 1e-5f)) : 0.f;
        if (tid < PROJ_D) {  // rank by variance, ties by index
            int p = 0;
#pragma unroll
            for (int d = 0; d < PROJ_D; ++d)
                p += (var[d] > var[tid] || (var[d] == var[tid] && d < tid)) ? 1 : 0;
            place[tid] = ok ? p : tid;  // not a permutation otherwise
        }
    }
    __syncthreads();
    for (int e = tid; e < NT * PROJ_D; e += B_THREADS) {
        const int k = e / PROJ_D, c = e % PROJ_D, p = place[c];
        basis[((p / 7) * NT + k) * 8 + p % 7] = scale > 0.f ? V[k][c] * scale : 0.f;
    }
    for (int e = tid; e < 4 * NT; e += B_THREADS) basis[e * 8 + 7] = 0.f;
    if (tid < PROJ_D) {
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < 16; ++q) s += pm[q][tid];
        off[place[tid]] = scale > 0.f ? s * scale : 0.f;
        sig[place[tid]] = scale > 0.f ? sqrtf(var[tid]) * scale : 0.f;
    }
}

// Projected rows, 64 rows a block: the rows pass through LDS
// once (lane = row, odd stride), wave g forms coordinates 7 g .. 7 g + 6 with
// the directions from scalar loads.  100 us for 200,000 contigs, 1.3 TB/s of 544
// bytes in and 128 out a row: bound by latency, not by that traffic.  45 KB of
// LDS leave three blocks a CU, whose waves spend two thirds of their time
// waiting for the rows and then for the directions; the vector units issue in
// 40% of the cycles, LDS is busy in 15%.
constexpr int PJ_ROWS = 64;

__global__ __launch_bounds__(256) void k_project(const float* __restrict__ tnf, uint32_t n,
                                                 const float* __restrict__ basis, const float* __restrict__ off,
                                                 float* __restrict__ y, int fmt) {
    __shared__ float X[PJ_ROWS][NT + 1];
    __shared__ float Ys[PJ_ROWS][PROJ_W + 1];
    __shared__ float nx2[4][PJ_ROWS], ne2[4][PJ_ROWS];
    __shared__ uint32_t bad[PJ_ROWS];
    const uint32_t tid = threadIdx.x, r0 = blockIdx.x * PJ_ROWS;
    const uint32_t rows = min((uint32_t)PJ_ROWS, n - r0);
    if (tid < PJ_ROWS) bad[tid] = 0;
    __syncthreads();
    const float4* src = reinterpret_cast<const float4*>(tnf + (size_t)r0 * NT);
    for (uint32_t e = tid; e < PJ_ROWS * (NT / 4); e += 256) {
        const uint32_t r = e / (NT / 4), q = e % (NT / 4);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (r < rows) v = src[e];
        if (!(finite_bits(v.x) && finite_bits(v.y) && finite_bits(v.z) && finite_bits(v.w))) bad[r] = 1;
        X[r][4 * q] = v.x;
        X[r][4 * q + 1] = v.y;
        X[r][4 * q + 2] = v.z;
        X[r][4 * q + 3] = v.w;
    }
    __syncthreads();
    const uint32_t lane = tid & 63, g = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* P = basis + (size_t)g * NT * 8;
    float acc[7] = {}, n2 = 0.f, e2 = 0.f;
#pragma unroll 4
    for (int k = 0; k < NT; ++k) {
        const float x = X[lane][k];
#pragma unroll
        for (int j = 0; j < 7; ++j) acc[j] = fmaf(x, P[k * 8 + j], acc[j]);
    }
    for (int k = 34 * (int)g; k < 34 * (int)g + 34; ++k) {
        const float x = X[lane][k];
        const float d = fmt == mdet::PROJ_BF16 ? x - bf16_rne(x) : fmt == mdet::PROJ_F16 ? x - (float)(_Float16)x : 0.f;
        n2 = fmaf(x, x, n2);
        e2 = fmaf(d, d, e2);
    }
    nx2[g][lane] = n2;
    ne2[g][lane] = e2;
#pragma unroll
    for (int j = 0; j < 7; ++j) Ys[lane][7 * g + j] = acc[j] - off[7 * g + j];
    __syncthreads();
    if (tid < rows) {
        float part = 0.f, ny2 = 0.f;
#pragma unroll
        for (int c = 0; c < PROJ_D; ++c) {
            const float v = Ys[tid][c], h = (float)(_Float16)v;
            part = fmaf(h, h, part);
            ny2 = fmaf(v, v, ny2);
        }
        const float ny = sqrtf(ny2);
        Ys[tid][PW_PART] = part;
        Ys[tid][PW_NY] = ny;
        const float nx = sqrtf(nx2[0][tid] + nx2[1][tid] + nx2[2][tid] + nx2[3][tid]);
        const float ne = sqrtf(ne2[0][tid] + ne2[1][tid] + ne2[2][tid] + ne2[3][tid]);
        Ys[tid][PW_MARGIN] = 2.002f * ne + 2e-6f + ny * (1.0001f / 2048.0f) + 5e-5f * (nx + 1.f);
        Ys[tid][PW_KIND] = bad[tid] ? 1.f : (ny < 100.f && nx < 1e4f && ne < 1e4f ? 0.f : 2.f);
    }
    __syncthreads();
    for (uint32_t e = tid; e < rows * PROJ_W; e += 256) y[(size_t)r0 * PROJ_W + e] = Ys[e / PROJ_W][e % PROJ_W];
}

// ------------------------------------------------------- row order --
// Rows of one population belong in the same 32-row tiles: the scan lists a tile
// pair, and the passes behind it work on it, if any of its 1,024 pairs is close.
// The order is by nearest of k centres (one Lloyd step on a sample of the rows;
// k = n / 96 or so, a few tiles each), the centres by a Morton key of their
// leading coordinates, and within a centre by the signs of the row's offset
// from it.  Against a Morton key of the rows alone the tiles with a close pair
// fell from 0.44% to 0.14% of all at 200,000 contigs and from 0.24% to 0.04% at
// 1,000,000, the listed ones from 0.52% to 0.16% and 0.53% to 0.10%.
constexpr uint32_t CL_SAMPLE = 16384, CL_ROWS = 96, CL_MIN = 64, CL_MAX = 4096;
constexpr int CL_SIGNS = 12;
constexpr float CL_FIX = 16384.f;  // fixed point of the centres' sums (sums that do not depend on the order)

// Centres c [k][PROJ_W]: from the sample's rows (sums == null), or the means of
// the rows assigned to them (a centre without rows stays); their MFMA fragments
// (row role: coordinates, then 4 - |c|^2 / 2 in two FP16 pieces against ones)
// and Morton keys.  A wave each half: lane = centre, half the k-steps.
__global__ __launch_bounds__(64) void k_cl_centres(const float* __restrict__ y, uint32_t n, uint32_t S, uint32_t k,
                                                   int* __restrict__ sums, const float* __restrict__ sig,
                                                   float* __restrict__ c, uint4* __restrict__ frag,
                                                   uint32_t* __restrict__ key, bool first) {
    const uint32_t i = blockIdx.x * 64 + threadIdx.x;  // k is a multiple of 64
    float v[PROJ_W];
    if (first) {
        const uint32_t s = (uint32_t)((uint64_t)i * S / k);
        const float* src = y + (size_t)((uint64_t)s * n / S) * PROJ_W;
        const bool ok = src[PW_KIND] == 0.f;
#pragma unroll
        for (int d = 0; d < PROJ_D; ++d) v[d] = ok ? fminf(fmaxf(src[d], -2.f), 2.f) : 0.f;
    } else {
        const int cnt = sums[(size_t)i * PROJ_W + PROJ_D];
        const float inv = 1.f / (CL_FIX * (float)cnt);
#pragma unroll
        for (int d = 0; d < PROJ_D; ++d)
            v[d] = cnt ? (float)sums[(size_t)i * PROJ_W + d] * inv : c[(size_t)i * PROJ_W + d];
    }
    float h = 0.f;
    uint32_t hi = 0, lo = 0;
#pragma unroll
    for (int d = 0; d < PROJ_D; ++d) {
        v[d] = (float)(_Float16)v[d];
        h = fmaf(v[d], v[d], h);
        c[(size_t)i * PROJ_W + d] = v[d];
        if (d < CL_SIGNS) {  // quartile of a normal coordinate: 2 bits
            const float t = 0.6745f * sig[d];
            hi = 2 * hi + (v[d] > 0.f ? 1u : 0u);
            lo = 2 * lo + ((v[d] > 0.f ? v[d] > t : v[d] > -t) ? 1u : 0u);
        }
    }
    key[i] = (hi << CL_SIGNS) | lo;
    h = 4.f - 0.5f * h;
    v[PROJ_D] = (float)(_Float16)h;
    v[PROJ_D + 1] = h - v[PROJ_D];
    v[PROJ_D + 2] = v[PROJ_D + 3] = 0.f;
#pragma unroll
    for (int o = 0; o < 4; ++o) {  // octet o: k-step o / 2, half o % 2
        f16x8_t w;
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = (_Float16)v[8 * o + e];
        frag[((size_t)(i >> 5) * PROJ_KS + (o >> 1)) * 64 + 32 * (o & 1) + (i & 31)] = __builtin_bit_cast(uint4, w);
    }
    // the sums of the coming step
    if (first)
        for (int d = 0; d <= PROJ_D; ++d) sums[(size_t)i * PROJ_W + d] = 0;
}

// rank[i]: place of centre i by key.
__global__ __launch_bounds__(256) void k_cl_rank(const uint32_t* __restrict__ key, uint32_t k,
                                                 uint32_t* __restrict__ rank) {
    __shared__ uint32_t ks[CL_MAX];
    for (uint32_t e = threadIdx.x; e < k; e += 256) ks[e] = key[e];
    __syncthreads();
    const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63), quarter = threadIdx.x >> 6;  // a wave each quarter
    __shared__ uint32_t part[4][64];
    uint32_t p = 0;
    const uint32_t mine = ks[i], q0 = quarter * (k / 4), q1 = q0 + k / 4;
    for (uint32_t e = q0; e < q1; ++e) p += (ks[e] < mine || (ks[e] == mine && e < i)) ? 1u : 0u;
    part[quarter][threadIdx.x & 63] = p;
    __syncthreads();
    if (quarter == 0) rank[i] = part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x];
}

// Nearest centre (largest y.c - |c|^2/2, on MFMA; FP16 coordinates) of every
// row, or of the sampled ones.  Sample: adds the row to its centre's sums;
// otherwise key[row] = (rank of the centre, signs of the offset from it), rows
// holding a NaN or an infinity last.  A wave takes CL_TILES x 32 rows (a row a
// lane, both halves) past all centres, whose fragments come from L1/L2; the
// 4-bit place among a lane's 16 centres rides in the product's low bits.
constexpr int CL_TILES = 2;

template <bool SAMPLE>
__global__ __launch_bounds__(256) void k_cl_assign(const float* __restrict__ y, uint32_t n, uint32_t S, uint32_t k,
                                                   const float* __restrict__ c, const uint4* __restrict__ frag,
                                                   const uint32_t* __restrict__ rank, int* __restrict__ sums,
                                                   uint32_t* __restrict__ key, uint32_t* __restrict__ idx) {
    constexpr int T = SAMPLE ? 1 : CL_TILES;
    const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, m = SAMPLE ? S : n;
    f16x8_t b[T][PROJ_KS];
    int best[T], at[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t s = (wave * T + t) * 32 + (lane & 31);
        const uint64_t row = SAMPLE ? (uint64_t)s * n / S : s;
#pragma unroll
        for (int q = 0; q < PROJ_KS; ++q) {
            const int d0 = 16 * q + 8 * (int)(lane >> 5);
            float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
            if (s < m) {
                v0 = *reinterpret_cast<const float4*>(y + row * PROJ_W + d0);
                v1 = *reinterpret_cast<const float4*>(y + row * PROJ_W + d0 + 4);
            }
            if (d0 == PROJ_D - 4) v1 = make_float4(1.f, 1.f, 0.f, 0.f);
            b[t][q] = f16x8_t{(_Float16)v0.x, (_Float16)v0.y, (_Float16)v0.z, (_Float16)v0.w,
                              (_Float16)v1.x, (_Float16)v1.y, (_Float16)v1.z, (_Float16)v1.w};
        }
        best[t] = INT32_MIN;
        at[t] = 0;
    }
    auto load = [&](uint32_t ct, f16x8_t* a) {
#pragma unroll
        for (int q = 0; q < PROJ_KS; ++q)
            a[q] = __builtin_bit_cast(f16x8_t, frag[((size_t)ct * PROJ_KS + q) * 64 + lane]);
    };
    f16x8_t a[PROJ_KS], next[PROJ_KS];
    load(0, next);
    for (uint32_t ct = 0; ct < k / 32; ++ct) {
#pragma unroll
        for (int q = 0; q < PROJ_KS; ++q) a[q] = next[q];
        load(min(ct + 1, k / 32 - 1), next);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            f32x16_t acc = f32x16_t{};
#pragma unroll
            for (int q = 0; q < PROJ_KS; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[q], b[t][q], acc, 0, 0, 0);
            int g = INT32_MIN;
#pragma unroll
            for (int r = 0; r < 16; ++r) g = max(g, (__float_as_int(acc[r]) & ~15) | r);
            if (g > best[t]) {
                best[t] = g;
                at[t] = (int)ct;
            }
        }
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int r = best[t] & 15;
        uint32_t at_c = 32u * at[t] + (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5);
        const int other = __shfl_xor(best[t], 32, 64);
        const uint32_t other_c = (uint32_t)__shfl_xor((int)at_c, 32, 64);
        if (other > best[t] || (other == best[t] && lane >= 32)) at_c = other_c;
        const uint32_t s = (wave * T + t) * 32 + (lane & 31);
        if (s >= m) continue;
        const float* row = y + (SAMPLE ? (uint64_t)s * n / S : (uint64_t)s) * PROJ_W;
        if (SAMPLE) {
            if (row[PW_KIND] != 0.f) continue;
            const int d0 = (lane >> 5) * (PROJ_D / 2);
            for (int d = d0; d < d0 + PROJ_D / 2; ++d)
                atomicAdd(&sums[(size_t)at_c * PROJ_W + d],
                          (int)rintf(CL_FIX * fminf(fmaxf(row[d], -2.f), 2.f)));
            if (lane < 32) atomicAdd(&sums[(size_t)at_c * PROJ_W + PROJ_D], 1);
        } else if (lane < 32) {
            uint32_t signs = 0;
#pragma unroll
            for (int d = 0; d < CL_SIGNS; ++d) signs = 2 * signs + (row[d] > c[(size_t)at_c * PROJ_W + d] ? 1u : 0u);
            key[s] = row[PW_KIND] == 1.f ? (CL_MAX << CL_SIGNS) : (rank[at_c] << CL_SIGNS) | signs;
            idx[s] = s;
        }
    }
}

// One thread per fragment entry (tile t, k-step ks, lane l: row t*32 + l%32,
// dimensions 16*ks + 8*(l/32) .. +8).  Slots 28..31 of the last octet carry
// the threshold (column role: 1, 1, -hh, -hl; row role: -hh, -hl, 1, 1) with
// h = |y~|^2/2 - s/2 in two FP16 pieces.  s is the row's share of the squared
// radius: for any pair |y~_a - y~_b| <= |a - b| + sum over both of u |y| (the
// FP16 rounding) + 5e-5 (|x| + 1) (the FP32 projection).  With the margin m of
// these and of twice the caller's rounding error, s = 2 (R/2 + m)^2 and a slack
// for the FP32 accumulation, |y~_a - y~_b|^2 < s_a + s_b for every pair within
// R + 2 (both errors), and the product a.b - h_a - h_b is positive.
__global__ __launch_bounds__(256) void k_proj_frags(const float* __restrict__ y, const uint32_t* __restrict__ perm,
                                                    uint32_t n, uint32_t n_pad, float R, uint4* __restrict__ frag,
                                                    uint4* __restrict__ frag_a) {
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n_pad / 32 * PROJ_KS * 64) return;
    const uint32_t t = e / (PROJ_KS * 64), ks = (e / 64) % PROJ_KS, l = e & 63, half = l >> 5;
    const uint32_t r = t * 32 + (l & 31);
    float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    float h = 6.0e4f;  // padding, and rows holding a NaN or an infinity: never within the radius
    if (r < n) {
        const float4* row = reinterpret_cast<const float4*>(y + (size_t)perm[r] * PROJ_W);
        const float4 w = row[PROJ_D / 4];  // part, |y|, margin, kind
        if (w.w == 0.f) {
            const float4 a = row[4 * ks + 2 * half], b = row[4 * ks + 2 * half + 1];
            v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
            v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
            const float half_r = 0.5f * R + w.z;
            const float share = 2.f * half_r * half_r + 1e-5f * (w.y * w.y + 1.f);
            h = 0.5f * w.x - 0.5f * share;
        } else if (w.w == 2.f) {
            h = -3.0e4f;  // longer than FP16 holds: passes against every bounded row
        }
    }
    _Float16 c[8], a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) c[k] = a[k] = (_Float16)v[k];
    const bool last = ks == PROJ_KS - 1;
    if (last && half) {
        const _Float16 hh = (_Float16)h, hl = (_Float16)(h - (float)hh), one = (_Float16)1.f;
        c[4] = c[5] = a[6] = a[7] = one;
        a[4] = c[6] = -hh;
        a[5] = c[7] = -hl;
    }
    auto pack = [](const _Float16* x) {
        uint4 w;
        w.x = __builtin_bit_cast(uint16_t, x[0]) | ((uint32_t)__builtin_bit_cast(uint16_t, x[1]) << 16);
        w.y = __builtin_bit_cast(uint16_t, x[2]) | ((uint32_t)__builtin_bit_cast(uint16_t, x[3]) << 16);
        w.z = __builtin_bit_cast(uint16_t, x[4]) | ((uint32_t)__builtin_bit_cast(uint16_t, x[5]) << 16);
        w.w = __builtin_bit_cast(uint16_t, x[6]) | ((uint32_t)__builtin_bit_cast(uint16_t, x[7]) << 16);
        return w;
    };
    frag[e] = pack(c);
    if (last) frag_a[(size_t)t * 64 + l] = pack(a);
}

// Bounding boxes of the 32-row tiles in the projection, box[d * T + t] =
// (lowest, highest) and the largest margin, for `tiles` tiles; ones without a bounded
// row get empty boxes, ones with a row too long for FP16 boundless boxes.  A
// thread per tile and coordinate: a row is one 128-byte read of 32 lanes.
__global__ __launch_bounds__(256) void k_tile_boxes(const float* __restrict__ y, const uint32_t* __restrict__ perm,
                                                    uint32_t n, uint32_t tiles, uint32_t T,
                                                    float2* __restrict__ box, float* __restrict__ margin) {
    const uint32_t t = blockIdx.x * 8 + (threadIdx.x >> 5), d = threadIdx.x & 31;
    if (t >= tiles) return;  // the 32 lanes of a tile together
    float lo = 3e38f, hi = -3e38f, mg = 0.f;
    // all loads of 16 rows go out at once: past the end the last row, left out
    for (uint32_t r0 = 0; r0 < 32; r0 += 16) {
        float v[16];
#pragma unroll
        for (uint32_t r = 0; r < 16; ++r) v[r] = y[(size_t)perm[min(t * 32 + r0 + r, n - 1)] * PROJ_W + d];
#pragma unroll
        for (uint32_t r = 0; r < 16; ++r) {
            const float word = __shfl(v[r], PW_KIND, 32);
            const float kind = t * 32 + r0 + r < n ? word : 1.f;
            if (kind != 1.f) {
                lo = fminf(lo, kind == 2.f ? -3e38f : v[r]);
                hi = fmaxf(hi, kind == 2.f ? 3e38f : v[r]);
                mg = fmaxf(mg, kind == 2.f ? 0.f : v[r]);
            }
        }
    }
    if (d < PROJ_D) box[(size_t)d * T + t] = make_float2(lo, hi);
    if (d == PW_MARGIN) margin[t] = mg;
}

}  // namespace

namespace mdet {

static_assert(PROJ_D == 28 && PROJ_KS == 2 && PROJ_W == 32, "k_project's groups and k_proj_frags' slots");

namespace {
// proj_rows, with the deviations of the coordinates (device, context buffer).
int project(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, float** y, float** sig) {
    hipStream_t s = ctx->stream;
    float *part, *msum, *cov, *mean, *basis;
    MDET_TRY(ctx_buf(ctx, "proj.part", (size_t)COV_SPLITS * NT * NT, &part));
    MDET_TRY(ctx_buf(ctx, "proj.msum", (size_t)COV_SPLITS * (NT + 1), &msum));
    MDET_TRY(ctx_buf(ctx, "proj.cov", (size_t)NT * NT, &cov));
    MDET_TRY(ctx_buf(ctx, "proj.vec", (size_t)NT + 2 * PROJ_W, &mean));  // mean, offsets, deviations
    float* off = mean + NT;
    *sig = off + PROJ_W;
    MDET_TRY(ctx_buf(ctx, "proj.basis", (size_t)4 * NT * 8, &basis));
    MDET_TRY(ctx_buf(ctx, "proj.y", (size_t)n * PROJ_W, y));
    hipLaunchKernelGGL(k_cov_part, dim3(COV_SPLITS), dim3(320), 0, s, tnf_dev, n, std::min(n, COV_SAMPLE), part, msum);
    hipLaunchKernelGGL(k_cov_sum, dim3((NT * NT + 255) / 256), dim3(256), 0, s, part, msum, cov, mean);
    hipLaunchKernelGGL(k_basis, dim3(1), dim3(B_THREADS), 0, s, cov, mean, basis, off, *sig);
    hipLaunchKernelGGL(k_project, dim3((n + PJ_ROWS - 1) / PJ_ROWS), dim3(256), 0, s, tnf_dev, n, basis, off, *y,
                       (int)fmt);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}
}  // namespace

int proj_rows(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, float** y) {
    float* sig;
    return project(ctx, tnf_dev, n, fmt, y, &sig);
}

int proj_order(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, ProjOrder* out) {
    hipStream_t s = ctx->stream;
    float* sig;
    uint32_t *key, *key2, *idx;
    MDET_TRY(project(ctx, tnf_dev, n, fmt, &out->y, &sig));
    MDET_TRY(ctx_buf(ctx, "proj.key", (size_t)n, &key));
    MDET_TRY(ctx_buf(ctx, "proj.key2", (size_t)n, &key2));
    MDET_TRY(ctx_buf(ctx, "proj.idx", (size_t)n, &idx));
    MDET_TRY(ctx_buf(ctx, "proj.perm", (size_t)n, &out->perm));
    uint32_t k = CL_MIN;
    while (k < CL_MAX && k * CL_ROWS * 3 / 2 < n) k *= 2;
    const uint32_t S = std::min({n, CL_SAMPLE, 4 * k});
    uint32_t *ckey, *rank;
    float* cen;
    int* sums;
    uint4* cfrag;
    MDET_TRY(ctx_buf(ctx, "proj.cen", (size_t)k * PROJ_W, &cen));
    MDET_TRY(ctx_buf(ctx, "proj.csum", (size_t)k * PROJ_W, &sums));
    MDET_TRY(ctx_buf(ctx, "proj.cfrag", (size_t)k / 32 * PROJ_KS * 64, &cfrag));
    MDET_TRY(ctx_buf(ctx, "proj.ckey", (size_t)2 * k, &ckey));
    rank = ckey + k;
    hipLaunchKernelGGL(k_cl_centres, dim3(k / 64), dim3(64), 0, s, out->y, n, S, k, sums, sig, cen, cfrag, ckey, true);
    hipLaunchKernelGGL(k_cl_assign<true>, dim3((S + 127) / 128), dim3(256), 0, s, out->y, n, S, k, cen, cfrag, rank,
                       sums, key, idx);
    hipLaunchKernelGGL(k_cl_centres, dim3(k / 64), dim3(64), 0, s, out->y, n, S, k, sums, sig, cen, cfrag, ckey, false);
    hipLaunchKernelGGL(k_cl_rank, dim3(k / 64), dim3(256), 0, s, ckey, k, rank);
    hipLaunchKernelGGL(k_cl_assign<false>, dim3((n + 128 * CL_TILES - 1) / (128 * CL_TILES)), dim3(256), 0, s, out->y,
                       n, S, k, cen, cfrag, rank, sums, key, idx);
    MDET_HIP(hipGetLastError());
    constexpr int KEY_BITS = CL_SIGNS + 13;
    static_assert((CL_MAX << CL_SIGNS) < 1u << KEY_BITS, "sort key");
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key, key2, idx, out->perm, (int)n, 0, KEY_BITS, s));
    void* t;
    MDET_TRY(ctx_buf(ctx, "cub.sorttmp", tmp, &t));
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(t, tmp, key, key2, idx, out->perm, (int)n, 0, KEY_BITS, s));
    return MDET_OK;
}

int proj_boxes(mdet_ctx* ctx, const ProjOrder& o, uint32_t n, uint32_t tiles, uint32_t T, float2* box,
               float* margin) {
    hipLaunchKernelGGL(k_tile_boxes, dim3((tiles + 7) / 8), dim3(256), 0, ctx->stream, o.y, o.perm, n, tiles, T, box,
                       margin);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

int proj_frags(mdet_ctx* ctx, const ProjOrder& o, uint32_t n, uint32_t n_pad, float R, uint4* frag, uint4* frag_a) {
    const uint32_t total = n_pad / 32 * PROJ_KS * 64;
    hipLaunchKernelGGL(k_proj_frags, dim3((total + 255) / 256), dim3(256), 0, ctx->stream, o.y, o.perm, n, n_pad, R,
                       frag, frag_a);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

}  // namespace mdet
