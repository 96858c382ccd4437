// Learned candidate filter for the TNF graph: an MLP 136 -> 256 -> 256 -> 32
// (GELU, BF16 weights, FP32 accumulation) whose embedding distance predicts
// whether a contig pair can clear the edge threshold.  No reference
// counterpart: the reference evaluates every pair.
//
// Training (all on the device, kernels below): a batch of labelled pairs
// (i, j, y) gathers 2B input rows (standardised TNF), runs the forward pass
// keeping pre-activations, evaluates the contrastive margin loss
//     L = mean over pairs of  y * D + (1 - y) * relu(m - D),
//     D = |e_i - e_j|^2,
// back-propagates through the three layers and applies Adam to the FP32
// master weights, refreshing their BF16 copies that the forward pass reads.
//
// Three launches a batch: forward and backward of 16 rows a block with
// everything between in LDS and registers (k_train_rows), the weight gradients
// split by rows (k_weight_grad), and the sums over blocks and splits
// (k_grad_sum).  All products are FP32 (v_mfma_f32_16x16x4, 32x32x2): the
// network is 109,088 weights and a batch of 512 pairs 0.67 GFLOP, so launches
// and latency are the cost: 30 + 10 + 4 us at 512 pairs, against 288 us in 21
// launches of one product, activation or sum each (64 x 64 tiles on the VALU, 16
// to 64 blocks a launch).  The all-pairs embedding Gram that uses the network
// at inference is in tnf_pairs.hip.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "hip_common.h"

namespace {

constexpr int D_IN = 136, D_H = 256, D_E = 32;
constexpr int N_W1 = D_H * D_IN, N_W2 = D_H * D_H, N_W3 = D_E * D_H;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + N_W1, OFF_W2 = OFF_B1 + D_H, OFF_B2 = OFF_W2 + N_W2, OFF_W3 = OFF_B2 + D_H,
              OFF_B3 = OFF_W3 + N_W3, N_PARAMS = OFF_B3 + D_E;  // 109,088

__device__ inline float bf16_round(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return f;
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
}

// erf by Abramowitz & Stegun, Handbook of Mathematical Functions, formula
// 7.1.26: for u >= 0, erf(u) = 1 - (a1 t + a2 t^2 + a3 t^3 + a4 t^4 + a5 t^5)
// exp(-u^2) with t = 1 / (1 + p u), |error| <= 1.5e-7; odd in u.  Branch-free
// (one reciprocal, one exponential), far inside the BF16 rounding of the
// activations it feeds.
__device__ inline float erf_as(float u) {
    const float a = fabsf(u);
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, a, 1.f));
    float poly = fmaf(1.061405429f, t, -1.453152027f);
    poly = fmaf(poly, t, 1.421413741f);
    poly = fmaf(poly, t, -0.284496736f);
    poly = fmaf(poly, t, 0.254829592f);
    const float r = 1.f - poly * t * __expf(-a * a);
    return copysignf(r, u);
}
__device__ inline float gelu(float x) { return 0.5f * x * (1.f + erf_as(x * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float x) {
    const float cdf = 0.5f * (1.f + erf_as(x * 0.70710678118654752f));
    const float pdf = 0.39894228040143268f * expf(-0.5f * x * x);
    return cdf + x * pdf;
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// ------------------------------------------------------------ training --
// Rows 2b and 2b + 1 of a batch are pair b's two contigs; block = 16 rows, 16
// waves of one 16-column tile each.  A product's k index runs as 16 s + 4 g + j
// (s the step, g = lane / 16, j the element of the lane's 4): A comes as 16-byte
// LDS reads (row strides of an odd number of 16-byte units), B either as 16
// bytes of a weight's row (products with the transposed weights) or as one
// float of each of 4 rows.  Bound by the MFMAs of one CU a block (~22,000 cycles
// a SIMD, 9 us) and the latency of the weights from L2 before them.
constexpr int TR_ROWS = 16, TR_WAVES = 16;
constexpr int X_STR = D_IN + 4, H_STR = D_H + 4, E_STR = D_E + 4;
constexpr int N_BIAS = 2 * D_H + D_E;  // b1, b2, b3

// acc += A[16 x K] * W^T for the columns n0 .. n0 + 15 (W row-major, ldw).
template <int K>
__device__ inline f32x4_t mul_wt(const float* a, int stride, const float* __restrict__ W, int ldw, int lane) {
    const int c = lane & 15, g = lane >> 4;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
    constexpr int FULL = K / 16;
    static_assert(K % 8 == 0, "half steps");
#pragma unroll
    for (int s = 0; s < FULL; ++s) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + c * stride + 16 * s + 4 * g);
        const f32x4_t w = *reinterpret_cast<const f32x4_t*>(W + (size_t)c * ldw + 16 * s + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], w[j], acc, 0, 0, 0);
    }
    if (K % 16) {
        f32x4_t x = {0.f, 0.f, 0.f, 0.f}, w = x;
        if (g < 2) {
            x = *reinterpret_cast<const f32x4_t*>(a + c * stride + 16 * FULL + 4 * g);
            w = *reinterpret_cast<const f32x4_t*>(W + (size_t)c * ldw + 16 * FULL + 4 * g);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], w[j], acc, 0, 0, 0);
    }
    return acc;
}

// A[16 x K] * W for 16 columns (W: first of them, row-major, ldw).
template <int K>
__device__ inline f32x4_t mul_w(const float* a, int stride, const float* __restrict__ W, int ldw, int lane) {
    const int c = lane & 15, g = lane >> 4;
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < K / 16; ++s) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + c * stride + 16 * s + 4 * g);
        float w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = W[(size_t)(16 * s + 4 * g + j) * ldw + c];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], w[j], acc, 0, 0, 0);
    }
    return acc;
}

// Sum over the block's 16 rows of a tile's column (lane % 16).
__device__ inline float column_sum(const f32x4_t v) {
    float s = (v[0] + v[1]) + (v[2] + v[3]);
    s += __shfl_xor(s, 16, 64);
    return s + __shfl_xor(s, 32, 64);
}

struct TrainArgs {
    const float* tnf;
    const uint32_t *pi, *pj;
    const float* label;
    uint32_t B;
    float margin;
    const float *mean, *istd;
    const float* w;  // BF16-rounded weights and FP32 biases
    float *X, *A1, *A2, *dE, *dZ2, *dZ1;  // rows for the weight gradients
    float* bias;  // per block: N_BIAS sums over its rows, then its loss
};

__global__ __launch_bounds__(64 * TR_WAVES) void k_train_rows(const TrainArgs A) {
    __shared__ __align__(16) float xs[TR_ROWS * X_STR], h1[TR_ROWS * H_STR], h2[TR_ROWS * H_STR], de[TR_ROWS * E_STR];
    __shared__ float ep[8][TR_ROWS][D_E + 1], ls[TR_ROWS / 2];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 15, r4 = 4 * (lane >> 4);  // this lane's column and first row of a result tile
    const uint32_t row0 = blockIdx.x * TR_ROWS, M = 2 * A.B;
    for (int e = tid; e < TR_ROWS * D_IN; e += 64 * TR_WAVES) {
        const uint32_t r = e / D_IN, k = e % D_IN, row = row0 + r;
        float v = 0.f;
        if (row < M) {
            const uint32_t contig = (row & 1) ? A.pj[row >> 1] : A.pi[row >> 1];
            v = A.tnf[(size_t)contig * D_IN + k];
            if (v != v) v = 0.f;  // rows with no valid window
            v = (v - A.mean[k]) * A.istd[k];
            A.X[(size_t)row * D_IN + k] = v;
        }
        xs[r * X_STR + k] = v;
    }
    __syncthreads();
    const int n0 = 16 * wave, n = n0 + c;
    // a tile to its rows in LDS and in memory
    auto put = [&](const f32x4_t v, float* lds, float* out) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (lds) lds[(r4 + r) * H_STR + n] = v[r];
            if (row0 + r4 + r < M) out[(size_t)(row0 + r4 + r) * D_H + n] = v[r];
        }
    };
    f32x4_t z1 = mul_wt<D_IN>(xs, X_STR, A.w + OFF_W1 + n0 * D_IN, D_IN, lane), z2, t;
    const float b1 = A.w[OFF_B1 + n], b2 = A.w[OFF_B2 + n];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        z1[r] += b1;
        t[r] = gelu(z1[r]);
    }
    put(t, h1, A.A1);
    __syncthreads();
    z2 = mul_wt<D_H>(h1, H_STR, A.w + OFF_W2 + n0 * D_H, D_H, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        z2[r] += b2;
        t[r] = gelu(z2[r]);
    }
    put(t, h2, A.A2);
    __syncthreads();
    {  // the 32 embedding columns, K in 8 slices of 32
        const int e0 = 16 * (wave & 1), s = wave >> 1;
        t = mul_wt<32>(h2 + 32 * s, H_STR, A.w + OFF_W3 + e0 * D_H + 32 * s, D_H, lane);
#pragma unroll
        for (int r = 0; r < 4; ++r) ep[s][r4 + r][e0 + c] = t[r];
    }
    __syncthreads();
    if (tid < TR_ROWS / 2 * D_E) {  // a pair's dimension a thread
        const int p = tid >> 5, d = tid & 31;
        const uint32_t pair = row0 / 2 + p;
        float e[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            e[i] = A.w[OFF_B3 + d];
#pragma unroll
            for (int s = 0; s < 8; ++s) e[i] += ep[s][2 * p + i][d];
        }
        const float diff = pair < A.B ? e[0] - e[1] : 0.f;
        float D = diff * diff;
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) D += __shfl_xor(D, off, 32);
        const float lab = pair < A.B ? A.label[pair] : 0.f;
        const float l = lab * D + (1.f - lab) * fmaxf(A.margin - D, 0.f);
        const float dldD = (lab + (1.f - lab) * (D < A.margin ? -1.f : 0.f)) / (float)A.B;
        const float g = pair < A.B ? dldD * 2.f * diff : 0.f;
        de[2 * p * E_STR + d] = g;
        de[(2 * p + 1) * E_STR + d] = -g;
        if (pair < A.B) {
            A.dE[(size_t)2 * pair * D_E + d] = g;
            A.dE[(size_t)(2 * pair + 1) * D_E + d] = -g;
        }
        if (d == 0) ls[p] = pair < A.B ? l / (float)A.B : 0.f;
    }
    __syncthreads();
    float* bias = A.bias + (size_t)blockIdx.x * (N_BIAS + 1);
    t = mul_w<D_E>(de, E_STR, A.w + OFF_W3 + n0, D_H, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] *= gelu_grad(z2[r]);
    put(t, h1, A.dZ2);  // h1: every wave is past the second layer
    float s = column_sum(t);
    if (lane < 16) bias[D_H + n] = s;
    if (tid < D_E) {
        float v = 0.f;
        for (int r = 0; r < TR_ROWS; ++r) v += de[r * E_STR + tid];
        bias[2 * D_H + tid] = v;
    }
    if (tid == 64) {
        float v = 0.f;
        for (int p = 0; p < TR_ROWS / 2; ++p) v += ls[p];
        bias[N_BIAS] = v;
    }
    __syncthreads();
    t = mul_w<D_H>(h1, H_STR, A.w + OFF_W2 + n0, D_H, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) t[r] *= gelu_grad(z1[r]);
    put(t, nullptr, A.dZ1);
    s = column_sum(t);
    if (lane < 16) bias[n] = s;
}

// dW = dZ^T A over the rows of a split, one 32 x 32 tile of one weight a wave
// (two rows a product, both operands straight from memory: 128-byte reads).
// part: [split][N_PARAMS], the weights' places.
constexpr int WG_T1 = D_H / 32 * ((D_IN + 31) / 32), WG_T2 = D_H / 32 * (D_H / 32), WG_T3 = D_E / 32 * (D_H / 32);
constexpr int WG_TILES = WG_T1 + WG_T2 + WG_T3;

__global__ __launch_bounds__(64) void k_weight_grad(const float* __restrict__ X, const float* __restrict__ A1,
                                                    const float* __restrict__ A2, const float* __restrict__ dE,
                                                    const float* __restrict__ dZ2, const float* __restrict__ dZ1,
                                                    uint32_t M, uint32_t per, float* __restrict__ part) {
    const int lane = threadIdx.x, c = lane & 31, h = lane >> 5;
    int t = blockIdx.x;
    const float *dz, *a;
    int rows, cols, off;
    if (t < WG_T1) {
        dz = dZ1, a = X, rows = D_H, cols = D_IN, off = OFF_W1;
    } else if (t < WG_T1 + WG_T2) {
        dz = dZ2, a = A1, rows = D_H, cols = D_H, off = OFF_W2, t -= WG_T1;
    } else {
        dz = dE, a = A2, rows = D_E, cols = D_H, off = OFF_W3, t -= WG_T1 + WG_T2;
    }
    const int n0 = 32 * (t % (rows / 32)), k0 = 32 * (t / (rows / 32)), k = k0 + c;
    const uint32_t m0 = blockIdx.y * per, m1 = min(M, m0 + per);  // per is even, M is even
    const bool in = k < cols;
    const float* pz = dz + (size_t)m0 * rows + (size_t)h * rows + n0 + c;
    const float* pa = a + (size_t)m0 * cols + (size_t)h * cols + (in ? k : 0);
    f32x16_t acc = {};
    constexpr int U = 8;
    for (uint32_t m = m0; m < m1; m += 2 * U) {
        float x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool ok = m + 2 * u < m1;
            x[u] = ok ? pz[(size_t)2 * u * rows] : 0.f;
            y[u] = ok && in ? pa[(size_t)2 * u * cols] : 0.f;
        }
        pz += (size_t)2 * U * rows;
        pa += (size_t)2 * U * cols;
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[u], y[u], acc, 0, 0, 0);
    }
    float* out = part + (size_t)blockIdx.y * N_PARAMS + off + k;
    if (in)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[(size_t)(n0 + (r & 3) + 8 * (r >> 2) + 4 * h) * cols] = acc[r];
}

// g: the weights' partial sums over the splits, the biases' and the loss over
// the row blocks, in order; a thread a weight, a wave a bias.
__device__ inline bool is_bias(uint32_t k) {
    return (k >= (uint32_t)OFF_B1 && k < (uint32_t)OFF_W2) || (k >= (uint32_t)OFF_B2 && k < (uint32_t)OFF_W3) ||
           k >= (uint32_t)OFF_B3;
}
constexpr uint32_t GS_WEIGHTS = (N_PARAMS + 255) / 256, GS_BLOCKS = GS_WEIGHTS + (N_BIAS + 1 + 3) / 4;

__global__ __launch_bounds__(256) void k_grad_sum(const float* __restrict__ part, uint32_t splits,
                                                  const float* __restrict__ bias, uint32_t blocks,
                                                  float* __restrict__ g, float* __restrict__ loss) {
    if (blockIdx.x < GS_WEIGHTS) {
        const uint32_t k = blockIdx.x * 256 + threadIdx.x;
        if (k >= (uint32_t)N_PARAMS || is_bias(k)) return;
        float t = 0.f;
#pragma unroll 8
        for (uint32_t z = 0; z < splits; ++z) t += part[(size_t)z * N_PARAMS + k];
        g[k] = t;
        return;
    }
    const uint32_t b = (blockIdx.x - GS_WEIGHTS) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (b > (uint32_t)N_BIAS) return;
    float t = 0.f;
    for (uint32_t z = lane; z < blocks; z += 64) t += bias[(size_t)z * (N_BIAS + 1) + b];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) t += __shfl_xor(t, off, 64);
    if (lane) return;
    if (b == (uint32_t)N_BIAS)
        *loss = t;
    else
        g[b < (uint32_t)D_H ? OFF_B1 + b : b < (uint32_t)(2 * D_H) ? OFF_B2 + b - D_H : OFF_B3 + b - 2 * D_H] = t;
}

// Adam on the FP32 master copy; writes the BF16-rounded weights the forward
// pass reads (biases stay FP32).
__global__ void k_adam(float* __restrict__ p, float* __restrict__ wq, const float* __restrict__ g,
                       float* __restrict__ m1, float* __restrict__ m2, uint32_t count, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const float gk = g[k];
    const float a = b1 * m1[k] + (1.f - b1) * gk;
    const float v = b2 * m2[k] + (1.f - b2) * gk * gk;
    m1[k] = a;
    m2[k] = v;
    const float w = p[k] - lr * (a / c1) / (sqrtf(v / c2) + eps);
    p[k] = w;
    wq[k] = is_bias(k) ? w : bf16_round(w);
}

// One parameter block [off, off + count): weights are rounded to BF16, biases
// copied.  The block kind is a launch argument, uniform over the grid: a
// per-lane bias test here (branching between a copy and the rounding) was
// compiled by this hipcc into a store whose address register the range compare
// had overwritten, so all-bias waves wrote one element each.
__global__ void k_quantize(const float* __restrict__ p, float* __restrict__ wq, uint32_t off, uint32_t count,
                           int round) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= count) return;
    const float v = p[off + k];
    wq[off + k] = round ? bf16_round(v) : v;
}


// ------------------------------------------------------------ inference --
// Embeddings on MFMA (v_mfma_f32_32x32x16_bf16): BF16 weights, inputs and
// hidden activations, FP32 accumulation.  One wave per 32 rows, 128 rows per
// block.  Layer 1's A fragments come straight from the FP32 TNF rows
// (standardised, NaN -> 0, rounded to BF16, K padded 136 -> 144).  A row of a
// row-major BF16 weight matrix is an MFMA B fragment (lane l: output column
// l % 32, inputs 8 * (l / 32) .. +8 of the k-step).  Between layers, bias +
// GELU + BF16 rounding go through a per-wave LDS buffer of 32 rows x 256
// (rows padded by 16 bytes against bank conflicts).  Fragment conventions as
// in the pair prefilter: accumulator r of a lane holds row
// 4 * (l / 32) + r % 4 + 8 * (r / 4), column l % 32.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int K1_PAD = 144;             // layer-1 inputs padded to 9 k-steps
constexpr int H_STRIDE = D_H + 8;       // BF16 elements per LDS row
constexpr int EMB_ROWS = 128;

__device__ inline uint16_t bf16_bits(float f) { return (uint16_t)(__float_as_uint(bf16_round(f)) >> 16); }

__device__ inline uint4 pack_bf16x8(const float* v) {
    uint4 w;
    w.x = bf16_bits(v[0]) | ((uint32_t)bf16_bits(v[1]) << 16);
    w.y = bf16_bits(v[2]) | ((uint32_t)bf16_bits(v[3]) << 16);
    w.z = bf16_bits(v[4]) | ((uint32_t)bf16_bits(v[5]) << 16);
    w.w = bf16_bits(v[6]) | ((uint32_t)bf16_bits(v[7]) << 16);
    return w;
}

__device__ inline f32x16_t mfma_bf16(uint4 a, uint4 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                    c, 0, 0, 0);
}

// Weights (already BF16-valued in wq) as BF16 bits, row-major [out][in]:
// W1 [256][144] (inputs 136..143 zero), W2 [256][256], W3 [32][256].
__global__ void k_pack_weights(const float* __restrict__ wq, uint16_t* __restrict__ w1, uint16_t* __restrict__ w2,
                               uint16_t* __restrict__ w3) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    constexpr uint32_t N1 = D_H * K1_PAD, N2 = D_H * D_H, N3 = D_E * D_H;
    if (e < N1) {
        const uint32_t o = e / K1_PAD, i = e % K1_PAD;
        w1[e] = i < (uint32_t)D_IN ? bf16_bits(wq[OFF_W1 + o * D_IN + i]) : (uint16_t)0;
    } else if (e < N1 + N2) {
        w2[e - N1] = bf16_bits(wq[OFF_W2 + (e - N1)]);
    } else if (e < N1 + N2 + N3) {
        w3[e - N1 - N2] = bf16_bits(wq[OFF_W3 + (e - N1 - N2)]);
    }
}

// One hidden layer's output tile set (4 column tiles of 32) to LDS:
// H[row][col] = bf16(gelu(acc + bias[col])).
__device__ inline void store_hidden(uint16_t* H, const f32x16_t* acc, int tile0, const float* __restrict__ bias,
                                    int lane) {
    const int lr = lane & 31, rb = 4 * (lane >> 5);
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
        const int col = 32 * (tile0 + ct) + lr;
        const float bv = bias[col];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = rb + (r & 3) + 8 * (r >> 2);
            H[row * H_STRIDE + col] = bf16_bits(gelu(acc[ct][r] + bv));
        }
    }
}

__device__ inline void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(256) void k_embed_mfma(const float* __restrict__ tnf, uint32_t n,
                                                    const float* __restrict__ norm, const uint16_t* __restrict__ w1,
                                                    const uint16_t* __restrict__ w2, const uint16_t* __restrict__ w3,
                                                    const float* __restrict__ wq, float* __restrict__ emb) {
    __shared__ uint16_t hbuf[4][32 * H_STRIDE];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t row0 = blockIdx.x * EMB_ROWS + wave * 32;
    if (row0 >= n) return;  // no block-wide synchronisation below
    const int lr = lane & 31, kh = 8 * (lane >> 5);
    const uint32_t r = row0 + lr;
    uint16_t* H = hbuf[wave];

    // layer 1: A fragments from the TNF row
    uint4 a[16];
#pragma unroll
    for (int ks = 0; ks < 9; ++ks) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = 16 * ks + kh + e;
            float x = 0.f;
            if (r < n && k < D_IN) {
                float t = tnf[(size_t)r * D_IN + k];
                if (t != t) t = 0.f;  // rows with no valid window
                x = (t - norm[k]) * norm[D_IN + k];
            }
            v[e] = x;
        }
        a[ks] = pack_bf16x8(v);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        f32x16_t acc[4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) acc[ct] = f32x16_t{};
#pragma unroll
        for (int ks = 0; ks < 9; ++ks)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                const int c = 32 * (4 * half + ct) + lr;
                const uint4 b = *reinterpret_cast<const uint4*>(w1 + (size_t)c * K1_PAD + 16 * ks + kh);
                acc[ct] = mfma_bf16(a[ks], b, acc[ct]);
            }
        store_hidden(H, acc, 4 * half, wq + OFF_B1, lane);
    }
    wave_lds_sync();

    // layer 2: A fragments from LDS (all read before the buffer is rewritten)
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) a[ks] = *reinterpret_cast<const uint4*>(H + lr * H_STRIDE + 16 * ks + kh);
    wave_lds_sync();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        f32x16_t acc[4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) acc[ct] = f32x16_t{};
#pragma unroll
        for (int ks = 0; ks < 16; ++ks)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                const int c = 32 * (4 * half + ct) + lr;
                const uint4 b = *reinterpret_cast<const uint4*>(w2 + (size_t)c * D_H + 16 * ks + kh);
                acc[ct] = mfma_bf16(a[ks], b, acc[ct]);
            }
        store_hidden(H, acc, 4 * half, wq + OFF_B2, lane);
    }
    wave_lds_sync();

    // layer 3: 32 outputs, FP32
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) a[ks] = *reinterpret_cast<const uint4*>(H + lr * H_STRIDE + 16 * ks + kh);
    f32x16_t acc = f32x16_t{};
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
        const uint4 b = *reinterpret_cast<const uint4*>(w3 + (size_t)lr * D_H + 16 * ks + kh);
        acc = mfma_bf16(a[ks], b, acc);
    }
    const float bv = wq[OFF_B3 + lr];
    const int rb = 4 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const uint32_t row = row0 + rb + (q & 3) + 8 * (q >> 2);
        if (row < n) emb[(size_t)row * D_E + lr] = acc[q] + bv;
    }
}
}  // namespace

struct mdet_mlp {
    mdet_ctx* ctx = nullptr;
    float* p = nullptr;   // FP32 master parameters
    float* wq = nullptr;  // parameters as the forward pass uses them (BF16-rounded weights)
    float* g = nullptr;   // gradient
    float* m1 = nullptr;
    float* m2 = nullptr;
    float* norm = nullptr;  // mean[136], inv std[136]
    uint64_t step = 0;
    // activations of the last batch (rows = 2 * batch)
    std::vector<void*> owned;
};

namespace {

using namespace mdet;

// Host<->device transfers go through the context's stream and complete before
// returning: that stream is non-blocking, so a null-stream hipMemcpy would not
// be ordered before the kernels launched on it afterwards.
int mlp_copy(mdet_mlp* m, void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
    MDET_HIP(hipMemcpyAsync(dst, src, bytes, kind, m->ctx->stream));
    MDET_HIP(hipStreamSynchronize(m->ctx->stream));
    return MDET_OK;
}

// wq = p with the weights rounded to BF16, block by block
int mlp_quantize(mdet_mlp* m) {
    static const uint32_t blocks[6][3] = {{OFF_W1, N_W1, 1}, {OFF_B1, D_H, 0}, {OFF_W2, N_W2, 1},
                                          {OFF_B2, D_H, 0}, {OFF_W3, N_W3, 1}, {OFF_B3, D_E, 0}};
    for (const auto& b : blocks)
        hipLaunchKernelGGL(k_quantize, dim3((b[1] + 255) / 256), dim3(256), 0, m->ctx->stream, m->p, m->wq, b[0], b[1],
                           (int)b[2]);
    MDET_HIP(hipGetLastError());
    MDET_HIP(hipStreamSynchronize(m->ctx->stream));
    return MDET_OK;
}

int mlp_alloc(mdet_mlp* m, size_t bytes, void** out) {
    hipError_t e = hipMalloc(out, bytes ? bytes : 4);
    if (e != hipSuccess) MDET_FAIL(MDET_E_NOMEM, "mlp: hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
    m->owned.push_back(*out);
    return MDET_OK;
}

struct Scratch {
    float* loss;
};

// The weight gradients' sums over the batch's rows: at most WG_SPLITS splits of
// at least WG_MIN_ROWS rows (one partial product each, summed in order, so the
// result depends on the batch size only); 128 rows a split put ~900 waves to
// work at 512 pairs.
constexpr uint32_t WG_SPLITS = 32, WG_MIN_ROWS = 128;

// loss + gradient (into m->g) of one batch of pairs
int mlp_grad(mdet_mlp* m, const float* tnf, const uint32_t* pi, const uint32_t* pj, const float* y, uint32_t B,
             float margin, Scratch* S) {
    hipStream_t s = m->ctx->stream;
    mdet_ctx* c = m->ctx;
    const uint32_t M = 2 * B, blocks = (M + TR_ROWS - 1) / TR_ROWS;
    const uint32_t want = std::max(1u, std::min(WG_SPLITS, M / WG_MIN_ROWS));
    const uint32_t per = ((M + want - 1) / want + 1) / 2 * 2, splits = (M + per - 1) / per;
    TrainArgs A{tnf, pi, pj, y, B, margin, m->norm, m->norm + D_IN, m->wq};
    float* part;
    MDET_TRY(ctx_buf(c, "mlp.X", (size_t)M * D_IN, &A.X));
    MDET_TRY(ctx_buf(c, "mlp.A1", (size_t)M * D_H, &A.A1));
    MDET_TRY(ctx_buf(c, "mlp.A2", (size_t)M * D_H, &A.A2));
    MDET_TRY(ctx_buf(c, "mlp.dE", (size_t)M * D_E, &A.dE));
    MDET_TRY(ctx_buf(c, "mlp.dZ2", (size_t)M * D_H, &A.dZ2));
    MDET_TRY(ctx_buf(c, "mlp.dZ1", (size_t)M * D_H, &A.dZ1));
    MDET_TRY(ctx_buf(c, "mlp.bias", (size_t)blocks * (N_BIAS + 1), &A.bias));
    MDET_TRY(ctx_buf(c, "mlp.part", (size_t)splits * N_PARAMS, &part));
    MDET_TRY(ctx_buf(c, "mlp.loss", 4, &S->loss));
    hipLaunchKernelGGL(k_train_rows, dim3(blocks), dim3(64 * TR_WAVES), 0, s, A);
    hipLaunchKernelGGL(k_weight_grad, dim3(WG_TILES, splits), dim3(64), 0, s, A.X, A.A1, A.A2, A.dE, A.dZ2, A.dZ1, M,
                       per, part);
    hipLaunchKernelGGL(k_grad_sum, dim3(GS_BLOCKS), dim3(256), 0, s, part, splits, A.bias, blocks, m->g, S->loss);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

// Xavier-uniform weights from a splitmix64 stream, zero biases.
void init_params(std::vector<float>& p, uint64_t seed) {
    uint64_t x = seed ^ 0x5DEECE66Dull;
    auto next = [&]() {
        uint64_t z = (x += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return ((z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    p.assign(N_PARAMS, 0.f);
    auto fill = [&](int off, int fan_out, int fan_in) {
        const double a = std::sqrt(6.0 / (fan_in + fan_out));
        for (int k = 0; k < fan_out * fan_in; ++k) p[off + k] = (float)((2 * next() - 1) * a);
    };
    fill(OFF_W1, D_H, D_IN);
    fill(OFF_W2, D_H, D_H);
    fill(OFF_W3, D_E, D_H);
}

}  // namespace

namespace mdet {
mdet_ctx* mlp_context(mdet_mlp* m) { return m ? m->ctx : nullptr; }
}  // namespace mdet

extern "C" {

int mdet_mlp_create(mdet_ctx* ctx, uint64_t seed, mdet_mlp** out) {
    MDET_TRY(check_ctx(ctx));
    if (!out) MDET_FAIL(MDET_E_INVALID, "mdet_mlp_create: null output");
    mdet_mlp* m = new mdet_mlp();
    m->ctx = ctx;
    int rc = MDET_OK;
    void* v;
    if ((rc = mlp_alloc(m, N_PARAMS * 4, &v)) == MDET_OK) m->p = (float*)v;
    if (!rc && (rc = mlp_alloc(m, N_PARAMS * 4, &v)) == MDET_OK) m->wq = (float*)v;
    if (!rc && (rc = mlp_alloc(m, N_PARAMS * 4, &v)) == MDET_OK) m->g = (float*)v;
    if (!rc && (rc = mlp_alloc(m, N_PARAMS * 4, &v)) == MDET_OK) m->m1 = (float*)v;
    if (!rc && (rc = mlp_alloc(m, N_PARAMS * 4, &v)) == MDET_OK) m->m2 = (float*)v;
    if (!rc && (rc = mlp_alloc(m, 2 * D_IN * 4, &v)) == MDET_OK) m->norm = (float*)v;
    if (rc) {
        mdet_mlp_destroy(m);
        return rc;
    }
    std::vector<float> p;
    init_params(p, seed);
    std::vector<float> norm(2 * D_IN, 0.f);
    for (int k = 0; k < D_IN; ++k) norm[D_IN + k] = 1.f;
    if ((rc = mlp_copy(m, m->p, p.data(), N_PARAMS * 4, hipMemcpyHostToDevice)) ||
        (rc = mlp_copy(m, m->norm, norm.data(), 2 * D_IN * 4, hipMemcpyHostToDevice))) {
        mdet_mlp_destroy(m);
        return rc;
    }
    MDET_HIP(hipMemsetAsync(m->m1, 0, N_PARAMS * 4, ctx->stream));
    MDET_HIP(hipMemsetAsync(m->m2, 0, N_PARAMS * 4, ctx->stream));
    if ((rc = mlp_quantize(m))) {
        mdet_mlp_destroy(m);
        return rc;
    }
    *out = m;
    return MDET_OK;
}

int mdet_mlp_destroy(mdet_mlp* m) {
    if (!m) return MDET_OK;
    if (m->ctx) (void)hipStreamSynchronize(m->ctx->stream);
    for (void* p : m->owned) (void)hipFree(p);
    delete m;
    return MDET_OK;
}

uint64_t mdet_mlp_param_count(void) { return N_PARAMS; }

int mdet_mlp_set_input_norm(mdet_mlp* m, const float* mean136, const float* istd136) {
    if (!m || !mean136 || !istd136) MDET_FAIL(MDET_E_INVALID, "mdet_mlp_set_input_norm: null argument");
    MDET_TRY(check_ctx(m->ctx));
    MDET_TRY(mlp_copy(m, m->norm, mean136, D_IN * 4, hipMemcpyHostToDevice));
    MDET_TRY(mlp_copy(m, m->norm + D_IN, istd136, D_IN * 4, hipMemcpyHostToDevice));
    return MDET_OK;
}

int mdet_mlp_get_params(mdet_mlp* m, float* out, uint64_t count) {
    if (!m || !out || count < N_PARAMS) MDET_FAIL(MDET_E_INVALID, "mdet_mlp_get_params: need %d floats", N_PARAMS);
    MDET_TRY(mlp_copy(m, out, m->p, N_PARAMS * 4, hipMemcpyDeviceToHost));
    // with room for twice the parameters, also the copy the forward pass reads
    if (count >= 2 * (uint64_t)N_PARAMS) MDET_TRY(mlp_copy(m, out + N_PARAMS, m->wq, N_PARAMS * 4, hipMemcpyDeviceToHost));
    return MDET_OK;
}

int mdet_mlp_set_params(mdet_mlp* m, const float* in, uint64_t count) {
    if (!m || !in || count != N_PARAMS) MDET_FAIL(MDET_E_INVALID, "mdet_mlp_set_params: need %d floats", N_PARAMS);
    MDET_TRY(mlp_copy(m, m->p, in, N_PARAMS * 4, hipMemcpyHostToDevice));
    return mlp_quantize(m);
}

int mdet_mlp_grad(mdet_mlp* m, const float* tnf_dev, const uint32_t* pi_dev, const uint32_t* pj_dev,
                  const float* label_dev, uint32_t batch, float margin, float* grad_out, float* loss_out) {
    if (!m) MDET_FAIL(MDET_E_INVALID, "null mdet_mlp");
    MDET_TRY(check_ctx(m->ctx));
    if (batch == 0 || !tnf_dev || !pi_dev || !pj_dev || !label_dev)
        MDET_FAIL(MDET_E_INVALID, "mdet_mlp_grad: empty batch or null argument");
    Scratch S;
    MDET_TRY(mlp_grad(m, tnf_dev, pi_dev, pj_dev, label_dev, batch, margin, &S));
    if (grad_out) MDET_TRY(mlp_copy(m, grad_out, m->g, N_PARAMS * 4, hipMemcpyDeviceToHost));
    if (loss_out) MDET_TRY(mlp_copy(m, loss_out, S.loss, 4, hipMemcpyDeviceToHost));
    MDET_HIP(hipStreamSynchronize(m->ctx->stream));
    return MDET_OK;
}

int mdet_mlp_train_step(mdet_mlp* m, const float* tnf_dev, const uint32_t* pi_dev, const uint32_t* pj_dev,
                        const float* label_dev, uint32_t batch, float lr, float margin, float* loss_out) {
    if (!m) MDET_FAIL(MDET_E_INVALID, "null mdet_mlp");
    MDET_TRY(check_ctx(m->ctx));
    if (batch == 0 || !tnf_dev || !pi_dev || !pj_dev || !label_dev)
        MDET_FAIL(MDET_E_INVALID, "mdet_mlp_train_step: empty batch or null argument");
    Scratch S;
    MDET_TRY(mlp_grad(m, tnf_dev, pi_dev, pj_dev, label_dev, batch, margin, &S));
    m->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - (float)std::pow((double)b1, (double)m->step);
    const float c2 = 1.f - (float)std::pow((double)b2, (double)m->step);
    hipLaunchKernelGGL(k_adam, dim3((N_PARAMS + 255) / 256), dim3(256), 0, m->ctx->stream, m->p, m->wq, m->g, m->m1,
                       m->m2, (uint32_t)N_PARAMS, lr, b1, b2, 1e-8f, c1, c2);
    MDET_HIP(hipGetLastError());
    if (loss_out) {
        MDET_HIP(hipMemcpyAsync(loss_out, S.loss, 4, hipMemcpyDeviceToHost, m->ctx->stream));
        MDET_HIP(hipStreamSynchronize(m->ctx->stream));
    }
    return MDET_OK;
}

int mdet_mlp_embed(mdet_mlp* m, const float* tnf_dev, uint32_t n, float* emb_dev) {
    if (!m) MDET_FAIL(MDET_E_INVALID, "null mdet_mlp");
    MDET_TRY(check_ctx(m->ctx));
    if (n == 0) return MDET_OK;
    if (!tnf_dev || !emb_dev) MDET_FAIL(MDET_E_INVALID, "mdet_mlp_embed: null argument");
    uint16_t *w1, *w2, *w3;
    mdet_ctx* c = m->ctx;
    MDET_TRY(ctx_buf(c, "mlp.w1bf", (size_t)D_H * K1_PAD, &w1));
    MDET_TRY(ctx_buf(c, "mlp.w2bf", (size_t)D_H * D_H, &w2));
    MDET_TRY(ctx_buf(c, "mlp.w3bf", (size_t)D_E * D_H, &w3));
    const uint32_t nw = D_H * K1_PAD + D_H * D_H + D_E * D_H;
    hipLaunchKernelGGL(k_pack_weights, dim3((nw + 255) / 256), dim3(256), 0, c->stream, m->wq, w1, w2, w3);
    hipLaunchKernelGGL(k_embed_mfma, dim3((n + EMB_ROWS - 1) / EMB_ROWS), dim3(256), 0, c->stream, tnf_dev, n,
                       m->norm, w1, w2, w3, m->wq, emb_dev);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

}  // extern "C"
