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
// The rows are visited in the order of a Morton key of the 12 leading
// coordinates (2 bits each): 0.4% of the 32 x 32 tiles then hold a pair within
// the radius, against 13% in the order of GC content.
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "order.h"

namespace {

using mdet::PROJ_D;
using mdet::PROJ_KS;
using mdet::PROJ_W;

constexpr int NT = 136;
constexpr uint32_t COV_SAMPLE = 2048, COV_SPLITS = 32;
constexpr int KEY_DIMS = 12;

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

// The directions, one block: V = W (random signs), twice V = orthonormal basis
// of C V (Cholesky QR of the 28 columns, the second time repeated for
// accuracy), columns ordered by their variance, then scaled so that the
// largest row sum of |P^T P|, a bound of |P|^2, is below 1.  Bound by the
// latency of one CU (three 136 x 136 x 32 products and 28-step
// factorisations); everything stays in its LDS.
// basis: P as [4][136][8] (coordinate 7 g + j of group g at [g][k][j]); off:
// P mean [28]; sig: standard deviation of each coordinate.
constexpr int B_THREADS = 1024;

__device__ inline void basis_mul(const float (*C)[NT], const float (*V)[PROJ_W], float (*Y)[PROJ_W]) {
    for (int t = threadIdx.x; t < NT * 8; t += B_THREADS) {
        const int r = t >> 3, c = (t & 7) * 4;
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int k = 0; k < NT; ++k) {
            const float x = C[r][k];
            const float4 v = *reinterpret_cast<const float4*>(&V[k][c]);
            a.x = fmaf(x, v.x, a.x);
            a.y = fmaf(x, v.y, a.y);
            a.z = fmaf(x, v.z, a.z);
            a.w = fmaf(x, v.w, a.w);
        }
        *reinterpret_cast<float4*>(&Y[r][c]) = a;
    }
    __syncthreads();
}

// V = orthonormal columns spanning Y's (Y may be V); columns whose remainder
// vanishes become zero.
__device__ inline void basis_orth(const float (*Y)[PROJ_W], float (*V)[PROJ_W], float (*G)[PROJ_W + 1]) {
    const int i = threadIdx.x >> 5, j = threadIdx.x & 31;
    float g = 0.f;
    for (int k = 0; k < NT; ++k) g = fmaf(Y[k][i], Y[k][j], g);
    G[i][j] = g;
    __syncthreads();
    float gmax = 0.f;
    for (int k = 0; k < PROJ_D; ++k) gmax = fmaxf(gmax, G[k][k]);
    __syncthreads();
    for (int k = 0; k < PROJ_D; ++k) {  // right-looking Cholesky, L in the lower triangle
        const float p = G[k][k];
        const float r = p > 1e-7f * gmax ? 1.f / sqrtf(p) : 0.f;
        const float lik = i > k ? G[i][k] * r : 0.f, ljk = j > k ? G[j][k] * r : 0.f;
        __syncthreads();
        if (j == k && i > k) G[i][k] = lik;
        if (i == k && j == k) G[k][k] = r;  // the reciprocal of the diagonal
        if (i > k && j > k && j <= i) G[i][j] -= lik * ljk;
        __syncthreads();
    }
    for (int r = threadIdx.x; r < NT; r += B_THREADS) {  // v L^T = y, row by row
        float v[PROJ_D];
#pragma unroll
        for (int c = 0; c < PROJ_D; ++c) {
            float s = Y[r][c];
#pragma unroll
            for (int k = 0; k < c; ++k) s = fmaf(-v[k], G[c][k], s);
            v[c] = s * G[c][c];
        }
#pragma unroll
        for (int c = 0; c < PROJ_D; ++c) V[r][c] = v[c];
#pragma unroll
        for (int c = PROJ_D; c < PROJ_W; ++c) V[r][c] = 0.f;
    }
    __syncthreads();
}

__global__ __launch_bounds__(B_THREADS) void k_basis(const float* __restrict__ Cg, const float* __restrict__ mean,
                                                     float* __restrict__ basis, float* __restrict__ off,
                                                     float* __restrict__ sig) {
    __shared__ __align__(16) float C[NT][NT];
    __shared__ __align__(16) float V[NT][PROJ_W], Y[NT][PROJ_W];
    __shared__ float G[PROJ_W][PROJ_W + 1];
    __shared__ float var[PROJ_W], scale;
    __shared__ int place[PROJ_W];
    const int tid = threadIdx.x;
    for (int e = tid; e < NT * NT; e += B_THREADS) C[e / NT][e % NT] = Cg[e];
    for (int e = tid; e < NT * PROJ_W; e += B_THREADS) {
        uint32_t h = (uint32_t)e * 0x9E3779B9u + 0x7F4A7C15u;
        h = (h ^ (h >> 16)) * 0x85EBCA6Bu;
        h = (h ^ (h >> 13)) * 0xC2B2AE35u;
        V[e / PROJ_W][e % PROJ_W] = e % PROJ_W < PROJ_D ? ((h >> 31) ? 1.f : -1.f) : 0.f;
    }
    __syncthreads();
    basis_mul(C, V, Y);
    basis_orth(Y, V, G);
    basis_mul(C, V, Y);
    basis_orth(Y, V, G);
    basis_orth(V, V, G);
    basis_mul(C, V, Y);
    if (tid < PROJ_W) {
        float s = 0.f;
        for (int k = 0; k < NT; ++k) s = fmaf(V[k][tid], Y[k][tid], s);
        var[tid] = tid < PROJ_D ? fmaxf(s, 0.f) : -1.f;
    }
    const int i = tid >> 5, j = tid & 31;
    float g = 0.f;
    for (int k = 0; k < NT; ++k) g = fmaf(V[k][i], V[k][j], g);
    G[i][j] = fabsf(g);
    __syncthreads();
    if (tid < PROJ_D) {  // rank by variance, ties by index
        int p = 0;
        for (int c = 0; c < PROJ_D; ++c) p += (var[c] > var[tid] || (var[c] == var[tid] && c < tid)) ? 1 : 0;
        place[tid] = p;
    }
    if (tid == 0) {
        float m = 0.f;
        bool ok = true;
        for (int a = 0; a < PROJ_D; ++a) {
            float s = 0.f;
            for (int b = 0; b < PROJ_D; ++b) s += G[a][b];
            ok = ok && finite_bits(s);
            m = fmaxf(m, s);
        }
        for (int a = 0; a < PROJ_D; ++a) ok = ok && finite_bits(var[a]);
        // |P|^2 <= the largest row sum; a basis that did not come out finite is dropped (P = 0: no tile is)
        scale = ok && m > 0.f ? 1.f / sqrtf(m * (1.f + 1e-5f)) : 0.f;
    }
    __syncthreads();
    if (!(scale > 0.f))  // place may not be a permutation
        for (int e = tid; e < PROJ_D; e += B_THREADS) place[e] = e;
    __syncthreads();
    for (int e = tid; e < NT * PROJ_D; e += B_THREADS) {
        const int k = e / PROJ_D, c = e % PROJ_D, p = place[c];
        basis[((p / 7) * NT + k) * 8 + p % 7] = scale > 0.f ? V[k][c] * scale : 0.f;
    }
    for (int e = tid; e < 4 * NT; e += B_THREADS) basis[e * 8 + 7] = 0.f;
    if (tid < PROJ_D) {
        float s = 0.f;
        if (scale > 0.f)
            for (int k = 0; k < NT; ++k) s = fmaf(V[k][tid] * scale, mean[k], s);
        off[place[tid]] = s;
        sig[place[tid]] = scale > 0.f ? sqrtf(var[tid]) * scale : 0.f;
    }
}

// Projected rows and Morton keys, 64 rows a block: the rows pass through LDS
// once (lane = row, odd stride), wave g forms coordinates 7 g .. 7 g + 6 with
// the directions from scalar loads.  Bound by reading the rows (544 bytes in,
// 132 out per row).
constexpr int PJ_ROWS = 64;

__global__ __launch_bounds__(256) void k_project(const float* __restrict__ tnf, uint32_t n,
                                                 const float* __restrict__ basis, const float* __restrict__ off,
                                                 const float* __restrict__ sig, float* __restrict__ y,
                                                 uint32_t* __restrict__ key, uint32_t* __restrict__ idx, int fmt) {
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
        uint32_t hi = 0, lo = 0;
#pragma unroll
        for (int c = 0; c < PROJ_D; ++c) {
            const float v = Ys[tid][c], h = (float)(_Float16)v;
            part = fmaf(h, h, part);
            ny2 = fmaf(v, v, ny2);
            if (c < KEY_DIMS) {  // quartile of a normal coordinate: 2 bits
                const float t = 0.6745f * sig[c];
                hi = 2 * hi + (v > 0.f ? 1u : 0u);
                lo = 2 * lo + ((v > 0.f ? v > t : v > -t) ? 1u : 0u);
            }
        }
        const float ny = sqrtf(ny2);
        Ys[tid][PW_PART] = part;
        Ys[tid][PW_NY] = ny;
        const float nx = sqrtf(nx2[0][tid] + nx2[1][tid] + nx2[2][tid] + nx2[3][tid]);
        const float ne = sqrtf(ne2[0][tid] + ne2[1][tid] + ne2[2][tid] + ne2[3][tid]);
        Ys[tid][PW_MARGIN] = 2.002f * ne + 2e-6f + ny * (1.0001f / 2048.0f) + 5e-5f * (nx + 1.f);
        Ys[tid][PW_KIND] = bad[tid] ? 1.f : (ny < 100.f && nx < 1e4f && ne < 1e4f ? 0.f : 2.f);
        key[r0 + tid] = bad[tid] ? 0xffffffu : (hi << KEY_DIMS) | lo;
        idx[r0 + tid] = r0 + tid;
    }
    __syncthreads();
    for (uint32_t e = tid; e < rows * PROJ_W; e += 256) y[(size_t)r0 * PROJ_W + e] = Ys[e / PROJ_W][e % PROJ_W];
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

}  // namespace

namespace mdet {

static_assert(PROJ_D == 28 && PROJ_KS == 2 && PROJ_W == 32, "k_project's groups and k_proj_frags' slots");

int proj_order(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, ProjFormat fmt, ProjOrder* out) {
    hipStream_t s = ctx->stream;
    float *part, *msum, *cov, *mean, *basis, *off, *sig;
    uint32_t *key, *key2, *idx;
    MDET_TRY(ctx_buf(ctx, "proj.part", (size_t)COV_SPLITS * NT * NT, &part));
    MDET_TRY(ctx_buf(ctx, "proj.msum", (size_t)COV_SPLITS * (NT + 1), &msum));
    MDET_TRY(ctx_buf(ctx, "proj.cov", (size_t)NT * NT, &cov));
    MDET_TRY(ctx_buf(ctx, "proj.vec", (size_t)NT + 2 * PROJ_W, &mean));  // mean, offsets, deviations
    off = mean + NT;
    sig = off + PROJ_W;
    MDET_TRY(ctx_buf(ctx, "proj.basis", (size_t)4 * NT * 8, &basis));
    MDET_TRY(ctx_buf(ctx, "proj.y", (size_t)n * PROJ_W, &out->y));
    MDET_TRY(ctx_buf(ctx, "proj.key", (size_t)n, &key));
    MDET_TRY(ctx_buf(ctx, "proj.key2", (size_t)n, &key2));
    MDET_TRY(ctx_buf(ctx, "proj.idx", (size_t)n, &idx));
    MDET_TRY(ctx_buf(ctx, "proj.perm", (size_t)n, &out->perm));
    hipLaunchKernelGGL(k_cov_part, dim3(COV_SPLITS), dim3(320), 0, s, tnf_dev, n, std::min(n, COV_SAMPLE), part, msum);
    hipLaunchKernelGGL(k_cov_sum, dim3((NT * NT + 255) / 256), dim3(256), 0, s, part, msum, cov, mean);
    hipLaunchKernelGGL(k_basis, dim3(1), dim3(B_THREADS), 0, s, cov, mean, basis, off, sig);
    hipLaunchKernelGGL(k_project, dim3((n + PJ_ROWS - 1) / PJ_ROWS), dim3(256), 0, s, tnf_dev, n, basis, off, sig,
                       out->y, key, idx, (int)fmt);
    MDET_HIP(hipGetLastError());
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, key, key2, idx, out->perm, (int)n, 0, 2 * KEY_DIMS, s));
    void* t;
    MDET_TRY(ctx_buf(ctx, "cub.sorttmp", tmp, &t));
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(t, tmp, key, key2, idx, out->perm, (int)n, 0, 2 * KEY_DIMS, s));
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
