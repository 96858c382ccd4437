// Cluster index of the learned proposal filter (no reference counterpart: the
// reference evaluates every pair).
//
// The filter's embedding puts a contig's partners close to it, but the
// embeddings do not form tiles compact enough to skip 32x32 blocks of pairs
// by bounds.  They do cluster: k-means with one centroid per ~192 contigs puts
// most partner pairs in the same cluster, and almost all of the rest in one of
// the few clusters whose centroids are nearest.  So the learned path runs its
// prefilter (the BF16 TNF Gram, or the embedding Gram with a radius) only on
// the pairs of probed cluster pairs:
//   1. k-means (Lloyd) on a sample of the rows, 4-8 iterations, distances on
//      FP16 MFMA (hi/lo split); centroid sums in 2^-20 fixed point (integer
//      atomics: the result does not depend on the order of the additions),
//      then one assignment of every row;
//   2. rows sorted by cluster (radix sort, stable), cluster offsets;
//   3. per cluster the n_probe nearest non-empty centroids (itself first);
//   4. on the host: the distinct unordered cluster pairs (a, b) with b in a's
//      probes or a in b's, each turned into prefilter items over a's rows x
//      b's rows (pairs i < j within one cluster).
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "ivf.h"

namespace {

constexpr int E_D = 32;                 // embedding dimensions
constexpr uint32_t KM_MAX_K = 16384;
constexpr double KM_FIX = 1048576.0;    // fixed-point scale of the centroid sums
// Lloyd iterations x sampled rows per centroid, by the number of centroids.
// Measured: at 1M contigs (5208 centroids, 32 probes) the edge recall is
// 0.9983 with 4 x 16, 0.9992 with 8 x 32, 0.9993 with 8 x 64; at 200k
// contigs (1042 centroids) 4 x 16 keeps as many partner pairs as 8 x 32, and
// the sampled passes (bound by the centroid-sum atomics) cost 1.3 ms more.
constexpr uint32_t KM_FEW_CLUSTERS = 2048;
inline int km_iters(uint32_t k) { return k <= KM_FEW_CLUSTERS ? 4 : 8; }
inline uint32_t km_sample_per_cluster(uint32_t k) { return k <= KM_FEW_CLUSTERS ? 16 : 32; }

// centroid c <- row c * n / k (rows are in input order)
__global__ void k_km_init(const float* __restrict__ emb, uint32_t n, uint32_t k, float* __restrict__ cent) {
    const uint32_t c = blockIdx.x, d = threadIdx.x;
    if (c >= k || d >= (uint32_t)E_D) return;
    const uint64_t src = (uint64_t)c * n / k;
    cent[(size_t)c * E_D + d] = emb[src * E_D + d];
}

// ---- assignment on MFMA (v_mfma_f32_32x32x16_f16, FP32 accumulate)
// Coordinates are split into FP16 pairs hi + lo (hi = fp16(v), lo =
// fp16(v - hi)), and the MFMA accumulates, for a point x and a centroid c,
//   -xh.ch - xh.cl - xl.ch                       (the dropped xl.cl and the
//                                                 FP32 sums: ~2^-21 relative)
//   + 1 * (hi, lo halves of s^2 |c - o|^2 / 2)
//   + (s^2 |x - o|^2 / 2 * (1 + 2^-6) + 2^-8) * 1
// over x, c in the frame (origin o = mean of the initial centroids, scale
// s = 2^e with s |x - o| <= KM_SPAN for every point, so all operands are in
// the FP16 range; centroids stay in the points' hull).  That is
// s^2 |x - c|^2 / 2 + delta_x, with delta_x > 0 far above the rounding error
// wherever |x - c| is small, so every value is positive and its float bits
// order like the values.  A point's nearest centroid is the smallest key
// (value bits with the low 8 bits replaced by the 32-centroid tile index),
// then the smallest index among equal keys: values within 2^-15 relative of
// each other count as equal.
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// fragments per 32 points or centroids: hi dims 0-15, 16-31, lo dims 0-15,
// 16-31, the norm slots
constexpr int KM_KF = 5;
constexpr float KM_SPAN = 128.f;  // bound on s |x - o|
constexpr uint32_t KM_TILES_MAX = KM_MAX_K / 32;
static_assert(KM_TILES_MAX <= 512, "tile index must fit the key's low 9 bits");
// bits of the key that hold the tile index: 8 up to 256 tiles (values within
// 2^-15 relative count as equal), 9 above (2^-14)
inline uint32_t km_tile_bits(uint32_t k) { return (k + 31) / 32 <= 256 ? 8u : 9u; }

struct KmFrame {
    float o[E_D];
    unsigned int maxd2;  // float bits of max |x - o|^2 over the points
};

__device__ inline float km_scale(const KmFrame* fr) {
    const float m = __uint_as_float(fr->maxd2);
    if (!(m > 0.f) || !(m < __builtin_inff())) return 1.f;
    const int e2 = ilogbf(KM_SPAN * KM_SPAN / m);  // 2^e2 <= SPAN^2 / m
    const int e = e2 >= 0 ? e2 / 2 : -((1 - e2) / 2);  // floor(e2 / 2)
    return ldexpf(1.f, e);
}

__device__ inline f32x16_t km_mfma(uint4 a, uint4 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                  0, 0, 0);
}

__device__ inline uint4 km_pack(const float* v) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const _Float16 lo = (_Float16)v[2 * e], hi = (_Float16)v[2 * e + 1];
        w[e] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// o = mean of the k centroids (fixed summation order); clears maxd2.  One block of 1024.
__global__ __launch_bounds__(1024) void k_km_center(const float* __restrict__ cent, uint32_t k, KmFrame* __restrict__ fr) {
    __shared__ float part[32][E_D];
    const int d = threadIdx.x % E_D, ch = threadIdx.x / E_D;
    float sum = 0.f;
#pragma unroll 8
    for (uint32_t c = ch; c < k; c += 32) sum += cent[(size_t)c * E_D + d];
    part[ch][d] = sum;
    __syncthreads();
    if (threadIdx.x < E_D) {
        float t = 0.f;
        for (int q = 0; q < 32; ++q) t += part[q][threadIdx.x];
        fr->o[threadIdx.x] = t / (float)k;
        if (threadIdx.x == 0) fr->maxd2 = 0u;
    }
}

// maxd2 = max over the n points of |x - o|^2 (order-free maximum of
// non-negative float bits; grid-stride, one atomic per block)
__global__ __launch_bounds__(256) void k_km_extent(const float* __restrict__ emb, uint32_t n, KmFrame* __restrict__ fr) {
    __shared__ uint32_t wmax[4];
    uint32_t u = 0;
    for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        const float4* x4 = reinterpret_cast<const float4*>(emb + (size_t)q * E_D);
        float d2 = 0.f;
#pragma unroll
        for (int v = 0; v < E_D / 4; ++v) {
            const float4 x = x4[v];
            const float a = x.x - fr->o[4 * v], b = x.y - fr->o[4 * v + 1], c = x.z - fr->o[4 * v + 2],
                        e = x.w - fr->o[4 * v + 3];
            d2 = fmaf(a, a, fmaf(b, b, fmaf(c, c, fmaf(e, e, d2))));
        }
        u = max(u, __float_as_uint(d2));  // NaN rows: bits above +inf, scale falls back to 1
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) u = max(u, (uint32_t)__shfl_xor((int)u, off, 64));
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = u;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t b = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
        if (b) atomicMax(&fr->maxd2, b);
    }
}

__device__ inline void km_split(float v, float& hi, float& lo) {
    hi = (float)(_Float16)v;
    lo = v - hi;
}

// Centroid fragments: tile t (centroids 32t..32t+31) x KM_KF x 64 lanes;
// lane l holds column l % 32, k = 8 (l / 32) + 0..7 of the fragment's 16.
// Coordinates enter negated.  Centroids past k get an unbeatable norm slot.
__global__ __launch_bounds__(256) void k_km_cfrag(const float* __restrict__ cent, uint32_t k,
                                                  const KmFrame* __restrict__ fr, uint4* __restrict__ cfrag) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t ntiles = (k + 31) / 32;
    if (g >= ntiles * 64) return;
    const uint32_t t = g / 64, lane = g % 64;
    const uint32_t c = t * 32 + (lane & 31), half = lane >> 5;
    const float s = km_scale(fr);
    float vh[8], vl[8], v[8];
    uint4 f[KM_KF];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
    if (c < k) {
        const float* cr = cent + (size_t)c * E_D;
        float n2 = 0.f;
        for (int d = 0; d < E_D; ++d) {
            const float y = s * (cr[d] - fr->o[d]);
            n2 = fmaf(y, y, n2);
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
#pragma unroll
            for (int e = 0; e < 8; ++e) km_split(-s * (cr[16 * st + 8 * half + e] - fr->o[16 * st + 8 * half + e]),
                                                 vh[e], vl[e]);
            f[st] = km_pack(vh);
            f[2 + st] = km_pack(vl);
        }
        if (half == 0) {
            km_split(0.5f * n2, v[0], v[1]);
            v[2] = 1.f;
        }
    } else {
        f[0] = f[1] = f[2] = f[3] = make_uint4(0, 0, 0, 0);
        if (half == 0) {
            v[0] = 65504.f;
            v[1] = 65504.f;
            v[2] = 1.f;
        }
    }
    f[4] = km_pack(v);
#pragma unroll
    for (int q = 0; q < KM_KF; ++q) cfrag[((size_t)t * KM_KF + q) * 64 + lane] = f[q];
}

// Nearest centroid of the points q * stride, q < m.  Block = 32 R points x W
// waves: every wave holds the points' A fragments and scans the centroid
// tiles t = w, w + W, ... (7 MFMAs per 32 x 32 tile: hi.hi, hi.lo, lo.hi
// over two k-steps each, and the norm slots); per element one AND-OR (key)
// and a running minimum; the 32 lanes of a column half then reduce each
// row, and the W
// waves' results are merged in LDS.  mode 1: counts[best] += 1; mode 2: also
// the point's coordinates into the fixed-point sums of its centroid.  err
// bit 0: a point outside the frame (only non-finite or overflowing rows).
template <int R, int W>
__global__ __launch_bounds__(64 * W) void k_km_assign(const float* __restrict__ emb, uint32_t m, uint32_t stride,
                                                      const KmFrame* __restrict__ fr, const uint4* __restrict__ cfrag,
                                                      uint32_t k, uint32_t* __restrict__ assign,
                                                      uint32_t* __restrict__ counts,
                                                      unsigned long long* __restrict__ sums, int mode,
                                                      unsigned int* __restrict__ err, uint32_t tbits) {
    __shared__ uint32_t sv[W][32 * R], si[W][32 * R];
    const uint32_t vmask = 0xffffffffu << tbits, tmask = ~vmask;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t half = lane >> 5, p0 = blockIdx.x * 32 * R;
    const float s = km_scale(fr);
    // a[r]: hi dims 0-15, hi 16-31, lo 0-15, lo 16-31, norm slots
    uint4 a[R][KM_KF];
    bool bad = false;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t q = p0 + 32 * r + (lane & 31);
        const bool valid = q < m;
        const float* x = emb + (size_t)(valid ? q : 0) * stride * E_D;
        float vh[8], vl[8], n2 = 0.f;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int d = 16 * st + 8 * half + e;
                const float v = valid ? s * (x[d] - fr->o[d]) : 0.f;
                n2 = fmaf(v, v, n2);
                km_split(v, vh[e], vl[e]);
            }
            a[r][st] = km_pack(vh);
            a[r][2 + st] = km_pack(vl);
        }
        n2 += __shfl_xor(n2, 32, 64);
        bad |= valid && !(n2 <= KM_SPAN * KM_SPAN * 1.0001f);
#pragma unroll
        for (int e = 0; e < 8; ++e) vh[e] = 0.f;
        if (half == 0) {
            vh[0] = 1.f;
            vh[1] = 1.f;
            vh[2] = fmaf(0.5f * n2, 1.f + 0x1p-6f, 0x1p-8f);
        }
        a[r][4] = km_pack(vh);
    }
    if (bad) atomicOr(err, 1u);
    uint32_t best[R][16];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 16; ++e) best[r][e] = 0xffffffffu;
    const uint32_t ntiles = (k + 31) / 32;
    for (uint32_t t = wave; t < ntiles; t += W) {
        const uint4* bt = cfrag + (size_t)t * KM_KF * 64 + lane;
        uint4 b[KM_KF];
#pragma unroll
        for (int f = 0; f < KM_KF; ++f) b[f] = bt[64 * f];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            f32x16_t acc = {};
            acc = km_mfma(a[r][0], b[0], acc);  // xh.ch
            acc = km_mfma(a[r][1], b[1], acc);
            acc = km_mfma(a[r][0], b[2], acc);  // xh.cl
            acc = km_mfma(a[r][1], b[3], acc);
            acc = km_mfma(a[r][2], b[0], acc);  // xl.ch
            acc = km_mfma(a[r][3], b[1], acc);
            acc = km_mfma(a[r][4], b[4], acc);  // norm slots
#pragma unroll
            for (int e = 0; e < 16; ++e) best[r][e] = min(best[r][e], (__float_as_uint(acc[e]) & vmask) | t);
        }
    }
    // per row: (value bits, centroid) minimum over the 32 lanes of the half.
    // Each step halves a lane's elements: it keeps the half its lane bit names
    // and gives the other away (15 exchanges and a last one instead of 80, which
    // were most of this kernel: 175 -> 125 us for 200,000 points and 1,042 centroids).
#pragma unroll
    for (int r = 0; r < R; ++r) {
        uint32_t v[16], c[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const uint32_t key = best[r][e];
            v[e] = key & vmask;
            c[e] = key == 0xffffffffu ? 0xffffffffu : (key & tmask) * 32 + (lane & 31);
        }
        auto merge = [&](int e, uint32_t v2, uint32_t c2) {
            if (v2 < v[e] || (v2 == v[e] && c2 < c[e])) {
                v[e] = v2;
                c[e] = c2;
            }
        };
#pragma unroll
        for (int h = 8; h >= 1; h >>= 1) {
            const bool up = (lane & (2 * h)) != 0;
#pragma unroll
            for (int e = 0; e < h; ++e) {
                const uint32_t gv = up ? v[e] : v[e + h], gc = up ? c[e] : c[e + h];
                v[e] = up ? v[e + h] : v[e];
                c[e] = up ? c[e + h] : c[e];
                merge(e, (uint32_t)__shfl_xor((int)gv, 2 * h, 64), (uint32_t)__shfl_xor((int)gc, 2 * h, 64));
            }
        }
        merge(0, (uint32_t)__shfl_xor((int)v[0], 1, 64), (uint32_t)__shfl_xor((int)c[0], 1, 64));
        const uint32_t e = (lane >> 1) & 15;  // the element this lane ended up with
        if ((lane & 1) == 0) {
            const uint32_t row = 32 * r + 8 * (e / 4) + 4 * half + (e % 4);
            sv[wave][row] = v[0];
            si[wave][row] = c[0];
        }
    }
    __syncthreads();
    const uint32_t t = threadIdx.x;
    if (t < 32 * R) {
        uint32_t bv = sv[0][t], bi = si[0][t];
#pragma unroll
        for (int w = 1; w < W; ++w) {
            const uint32_t v2 = sv[w][t], c2 = si[w][t];
            if (v2 < bv || (v2 == bv && c2 < bi)) {
                bv = v2;
                bi = c2;
            }
        }
        if (bi >= k) bi = 0;  // only reachable with non-finite coordinates
        const uint32_t q = p0 + t;
        if (q < m) {
            if (assign) assign[q] = bi;
            if (mode >= 1) atomicAdd(&counts[bi], 1u);
        }
        si[0][t] = bi;
    }
    if (mode < 2) return;
    __syncthreads();
    // fixed-point sums: lanes of an instruction cover 2 points x 32
    // consecutive dimensions (contiguous centroid rows)
    for (uint32_t g = threadIdx.x; g < 32 * R * E_D; g += 64 * W) {
        const uint32_t pt = g / E_D, d = g % E_D, q = p0 + pt;
        if (q < m)
            atomicAdd(&sums[(size_t)si[0][pt] * E_D + d],
                      (unsigned long long)llrint((double)emb[(size_t)q * stride * E_D + d] * KM_FIX));
    }
}

// centroid <- mean of its points (unchanged if it has none); clears the sums
// and counts for the next iteration.  32 threads (one per dimension) per
// centroid.
__global__ __launch_bounds__(256) void k_km_update(unsigned long long* __restrict__ sums, uint32_t* __restrict__ counts,
                                                   uint32_t k, float* __restrict__ cent) {
    const uint32_t c = blockIdx.x * (blockDim.x / E_D) + threadIdx.x / E_D;
    const uint32_t d = threadIdx.x % E_D;
    const bool ok = c < k;
    const uint32_t cnt = ok ? counts[c] : 0u;
    if (ok) {
        const size_t e = (size_t)c * E_D + d;
        const long long v = (long long)sums[e];
        sums[e] = 0ull;
        if (cnt) cent[e] = (float)((double)v / KM_FIX / (double)cnt);
    }
    __syncthreads();  // every lane has read counts[c] before it is cleared
    if (ok && d == 0) counts[c] = 0;
}

// Per cluster a (one wave; 4 clusters per block): its n_probe (<= KM_MAX_PROBE)
// nearest non-empty centroids, itself first, by (distance, index).  Each lane
// keeps the KM_MAX_PROBE best of the centroids b = lane, lane + 64, ... in
// registers (insertion into a sorted list; b increases, so ties keep the
// lower index), the lists go to LDS, and n_probe rounds take the wave-wide
// minimum of the lanes' list heads, the owning lane advancing its head.
constexpr uint32_t KM_MAX_PROBE = 32;

__device__ inline void probe_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ __launch_bounds__(256) void k_km_probe(const float* __restrict__ cent, const uint32_t* __restrict__ counts,
                                                  uint32_t k, uint32_t n_probe, uint32_t* __restrict__ probes) {
    __shared__ float dk[4][KM_MAX_PROBE * 64];
    __shared__ uint32_t di[4][KM_MAX_PROBE * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t a = blockIdx.x * 4 + wave;
    if (a >= k) return;  // no block-wide synchronisation below
    float ca[E_D];
#pragma unroll
    for (int d = 0; d < E_D; ++d) ca[d] = cent[(size_t)a * E_D + d];
    float bd[KM_MAX_PROBE];
    uint32_t bx[KM_MAX_PROBE];
#pragma unroll
    for (uint32_t t = 0; t < KM_MAX_PROBE; ++t) {
        bd[t] = __builtin_inff();
        bx[t] = 0xffffffffu;
    }
    // KM_SCAN candidates b = b0 + 64 u per lane and round, loaded together
    // (clamped index, masked after) so their latencies overlap; inserted in
    // increasing b as before
    constexpr uint32_t KM_SCAN = 4;
    for (uint32_t b0 = lane; b0 < k; b0 += 64 * KM_SCAN) {
        float dists[KM_SCAN];
#pragma unroll
        for (uint32_t u = 0; u < KM_SCAN; ++u) {
            const uint32_t b = b0 + 64 * u;
            const uint32_t bc = b < k ? b : k - 1;
            const bool nonempty = counts[bc] != 0;
            const float4* cb = reinterpret_cast<const float4*>(cent + (size_t)bc * E_D);
            float s = 0.f;
#pragma unroll
            for (int v = 0; v < E_D / 4; ++v) {
                const float4 y = cb[v];
                const float t0 = ca[4 * v] - y.x, t1 = ca[4 * v + 1] - y.y, t2 = ca[4 * v + 2] - y.z,
                            t3 = ca[4 * v + 3] - y.w;
                s = fmaf(t0, t0, s);
                s = fmaf(t1, t1, s);
                s = fmaf(t2, t2, s);
                s = fmaf(t3, t3, s);
            }
            dists[u] = (b < k && nonempty) ? (b == a ? -1.f : s) : __builtin_inff();
        }
#pragma unroll
        for (uint32_t u = 0; u < KM_SCAN; ++u) {
            if (!(dists[u] < bd[KM_MAX_PROBE - 1])) continue;
            float cd = dists[u];
            uint32_t cx = b0 + 64 * u;
#pragma unroll
            for (uint32_t t = 0; t < KM_MAX_PROBE; ++t) {
                if (cd < bd[t]) {
                    const float td = bd[t];
                    const uint32_t tx = bx[t];
                    bd[t] = cd;
                    bx[t] = cx;
                    cd = td;
                    cx = tx;
                }
            }
        }
    }
    float* sd = dk[wave];
    uint32_t* sx = di[wave];
#pragma unroll
    for (uint32_t t = 0; t < KM_MAX_PROBE; ++t) {
        sd[t * 64 + lane] = bd[t];
        sx[t * 64 + lane] = bx[t];
    }
    probe_wave_sync();
    // every centroid index sits in exactly one lane's list, so one lane holds the minimum
    uint32_t head = 0;
    for (uint32_t r = 0; r < n_probe; ++r) {
        const float v = head < KM_MAX_PROBE ? sd[head * 64 + lane] : __builtin_inff();
        const uint32_t x = head < KM_MAX_PROBE ? sx[head * 64 + lane] : 0xffffffffu;
        float mv = v;
        uint32_t mx = x;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            const float v2 = __shfl_xor(mv, off, 64);
            const uint32_t x2 = (uint32_t)__shfl_xor((int)mx, off, 64);
            if (v2 < mv || (v2 == mv && x2 < mx)) {
                mv = v2;
                mx = x2;
            }
        }
        if (v == mv && x == mx) ++head;
        if (lane == 0) probes[(size_t)a * n_probe + r] = mv < __builtin_inff() ? mx : 0xffffffffu;
    }
}

__global__ void k_iota(uint32_t* __restrict__ v, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = i;
}

// ---- exact cover: which cluster pairs can hold a pair within the radius R
// of the pre > T test (d(i, j) < R for every pair that can pass; R covers
// every size pair of the input).  With a TNF-space centre c_b and radius
// r_b >= max_{j in b} |x_j - c_b| of each cluster, the triangle inequality
// gives, for i in a and j in b,
//   d(i, j) >= |x_i - c_b| - r_b >= M[a][b] - r_b,
//   M[a][b] = min_{i in a} |x_i - c_b|,
// so no pair of (a, b) passes unless M[a][b] - r_b < R and M[b][a] - r_a < R.
// M comes from the BF16 MFMA: x~, c~ the BF16 roundings (|x - x~| <= 2^-9
// |x|, the same for c), |x~ - c~|^2 = |x~|^2 + |c~|^2 - 2 x~.c~ with the
// products exact and the FP32 sums within 1e-5 (|x| + |c|)^2 (136 terms),
// hence |x - c| >= sqrt(max(0, D - 1e-5 s^2)) - 2^-8 s with s = |x| + |c| and
// D the computed value.  Rows with no valid window (NaN) pass no test and
// take no part in the bounds.
constexpr int CV_NT = 136;   // TNF columns
constexpr int CV_KS = 9;     // k-steps of 16 over the TNF columns (K padded to 144)
constexpr int CV_CAP = (int)mdet::IVF_COVER_CAP;  // listed partners per cluster; more: "every cluster"

__device__ inline uint16_t cv_bf16(float f) {  // round to nearest even (finite inputs)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ inline float cv_from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline f32x16_t cv_mfma(uint4 a, uint4 b, f32x16_t c) {
    typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// The clustering space of the exact cover: y = S x with a fixed 32 x 136
// matrix of signs (a Johnson-Lindenstrauss projection, so that k-means
// clusters are compact in TNF space; the bound is exact whatever the
// clusters).  Rows with no valid window map to 0.  One wave per row.
__device__ inline float cv_sign(uint32_t col, uint32_t dim) {
    uint32_t h = col * 32u + dim + 0x9e3779b9u;
    h ^= h >> 16;
    h *= 0x7feb352du;
    h ^= h >> 15;
    h *= 0x846ca68bu;
    h ^= h >> 16;
    return (h & 1u) ? 1.f : -1.f;
}

__global__ __launch_bounds__(256) void k_cover_project(const float* __restrict__ tnf, uint32_t n,
                                                       float* __restrict__ y) {
    constexpr uint32_t RW = 4;  // rows a wave projects per pass
    constexpr uint32_t HALF = CV_NT / 2;
    constexpr uint32_t SST = 33;  // sign table row stride: the two lane halves on different banks
    static_assert(HALF % 4 == 0, "each half of the columns in float4 pieces");
    __shared__ float sgn[CV_NT * SST];
    __shared__ __align__(16) float row[4][RW][CV_NT];
    for (uint32_t e = threadIdx.x; e < (uint32_t)CV_NT * 32; e += blockDim.x)
        sgn[(e / 32) * SST + (e % 32)] = cv_sign(e / 32, e % 32);
    __syncthreads();
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // lane: output dimension lane % 32 over the columns of half lane / 32
    const uint32_t d = lane & 31, c0 = (lane >> 5) * HALF;
    for (uint32_t i0 = (blockIdx.x * 4 + wave) * RW; i0 < n; i0 += gridDim.x * 4 * RW) {
        for (uint32_t e = lane; e < RW * CV_NT; e += 64) {
            const uint32_t q = e / CV_NT, c = e - q * CV_NT;
            row[wave][q][c] = i0 + q < n ? tnf[(size_t)(i0 + q) * CV_NT + c] : 0.f;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float acc[RW];
#pragma unroll
        for (uint32_t q = 0; q < RW; ++q) acc[q] = 0.f;
#pragma unroll 2
        for (uint32_t j = 0; j < HALF; j += 4) {
            const float s0 = sgn[(c0 + j) * SST + d], s1 = sgn[(c0 + j + 1) * SST + d];
            const float s2 = sgn[(c0 + j + 2) * SST + d], s3 = sgn[(c0 + j + 3) * SST + d];
#pragma unroll
            for (uint32_t q = 0; q < RW; ++q) {
                const float4 v = *reinterpret_cast<const float4*>(&row[wave][q][c0 + j]);
                acc[q] = fmaf(s0, v.x, acc[q]);
                acc[q] = fmaf(s1, v.y, acc[q]);
                acc[q] = fmaf(s2, v.z, acc[q]);
                acc[q] = fmaf(s3, v.w, acc[q]);
            }
        }
#pragma unroll
        for (uint32_t q = 0; q < RW; ++q) {
            const float t = acc[q] + __shfl_xor(acc[q], 32, 64);
            if (lane < 32 && i0 + q < n) y[(size_t)(i0 + q) * 32 + lane] = t == t ? t : 0.f;  // no valid window: 0
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();  // the rows are read before the next pass overwrites them
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// |x~|^2 of every sorted position (+inf for a row with no valid window).
// One wave per row of the sorted FP32 rows.
__global__ __launch_bounds__(256) void k_cover_xn2(const float* __restrict__ rows, uint32_t n,
                                                   float* __restrict__ xn2) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t s = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (s >= n) return;
    const float* x = rows + (size_t)s * CV_NT;
    float q = 0.f, raw = 0.f;
    for (uint32_t c = lane; c < (uint32_t)CV_NT; c += 64) {
        const float v = x[c];
        raw += v;
        const float b = v == v ? cv_from_bf16(cv_bf16(v)) : 0.f;
        q = fmaf(b, b, q);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        q += __shfl_xor(q, off, 64);
        raw += __shfl_xor(raw, off, 64);
    }
    if (lane == 0) xn2[s] = raw == raw ? q : __builtin_inff();
}

// The centres and radii, in passes over (cluster, part) blocks: a cluster's
// rows are split over CV_SPLIT blocks (32-row steps), so a large cluster does
// not hold the launch.  Sums are in 2^-40 fixed point (TNF values are in
// [0, 1]): integer atomics, a result independent of their order.
constexpr uint32_t CV_SPLIT = 8;
constexpr double CV_FIX = 1099511627776.0;  // 2^40

// Column sums and counts of the valid member rows.  sums (k x 144), cnt (k)
// zero before.  Wave w of part s takes the rows p0 + 4 (s + CV_SPLIT j) + w.
__global__ __launch_bounds__(256) void k_cover_sums(const float* __restrict__ rows, const uint32_t* __restrict__ off,
                                                    unsigned long long* __restrict__ sums, uint32_t* __restrict__ cnt) {
    __shared__ unsigned long long ws[4][144];
    __shared__ uint32_t wc[4];
    const uint32_t a = blockIdx.x, part = blockIdx.y;
    const uint32_t p0 = off[a], p1 = off[a + 1];
    if (p0 + 4 * part >= p1) return;  // block-uniform: no row for this part
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63;
    unsigned long long ps[3] = {0, 0, 0};
    uint32_t pc = 0;
    for (uint32_t p = p0 + 4 * part + w; p < p1; p += 4 * CV_SPLIT) {
        const float* x = rows + (size_t)p * CV_NT;
        const float v0 = x[l], v1 = x[l + 64], v2 = l + 128 < (uint32_t)CV_NT ? x[l + 128] : 0.f;
        if (v0 == v0) {  // a row is all NaN or all finite
            ps[0] += (unsigned long long)llrint((double)v0 * CV_FIX);
            ps[1] += (unsigned long long)llrint((double)v1 * CV_FIX);
            ps[2] += (unsigned long long)llrint((double)v2 * CV_FIX);
            ++pc;
        }
    }
    ws[w][l] = ps[0];
    ws[w][l + 64] = ps[1];
    if (l + 128 < 144) ws[w][l + 128] = ps[2];
    if (l == 0) wc[w] = pc;
    __syncthreads();
    const uint32_t t = threadIdx.x;
    if (t < (uint32_t)CV_NT) {
        const unsigned long long v = ws[0][t] + ws[1][t] + ws[2][t] + ws[3][t];
        if (v) atomicAdd(&sums[(size_t)a * 144 + t], v);
    }
    if (t == 0) {
        const uint32_t c = wc[0] + wc[1] + wc[2] + wc[3];
        if (c) atomicAdd(&cnt[a], c);
    }
}

// One block per cluster: the centre c (FP32, k x 136), its BF16 fragment
// (lane layout of the row fragments, zeros beyond column 136: a product with
// a row fragment is the plain dot product whatever the rows carry in their
// threshold slots) and info = (|c~|^2, |c|): +inf / 0 without a valid row.
__global__ __launch_bounds__(256) void k_cover_centre(const unsigned long long* __restrict__ sums,
                                                      const uint32_t* __restrict__ cnt, uint32_t k,
                                                      float* __restrict__ cen, uint4* __restrict__ cfrag,
                                                      float4* __restrict__ info) {
    __shared__ float c[144];
    __shared__ uint16_t cb[144];
    const uint32_t a = blockIdx.x, tid = threadIdx.x;
    const uint32_t m = cnt[a];
    if (tid < 144) {
        const float cv = (tid < (uint32_t)CV_NT && m) ? (float)((double)sums[(size_t)a * 144 + tid] / CV_FIX / m) : 0.f;
        c[tid] = cv;
        cb[tid] = cv_bf16(cv);
        if (tid < (uint32_t)CV_NT) cen[(size_t)a * CV_NT + tid] = cv;
    }
    __syncthreads();
    if (tid < 2 * CV_KS) {  // fragment k-step tid / 2, lane half tid % 2
        const uint32_t ks = tid >> 1, half = tid & 1, e0 = 16 * ks + 8 * half;
        uint4 w;
        w.x = cb[e0] | ((uint32_t)cb[e0 + 1] << 16);
        w.y = cb[e0 + 2] | ((uint32_t)cb[e0 + 3] << 16);
        w.z = cb[e0 + 4] | ((uint32_t)cb[e0 + 5] << 16);
        w.w = cb[e0 + 6] | ((uint32_t)cb[e0 + 7] << 16);
        cfrag[((size_t)(a / 32) * CV_KS + ks) * 64 + (a % 32) + 32 * half] = w;
    }
    if (tid == 0) {
        float cn2 = 0.f, c2 = 0.f;
        for (int q = 0; q < CV_NT; ++q) {
            const float bq = cv_from_bf16(cb[q]);
            cn2 = fmaf(bq, bq, cn2);
            c2 = fmaf(c[q], c[q], c2);
        }
        info[a] = m ? make_float4(cn2, sqrtf(c2) * (1.f + 1.0f / 4096.f), 0.f, 0.f)
                    : make_float4(__builtin_inff(), 0.f, 0.f, 0.f);
    }
}

// The members' largest squared distance from the centre and largest squared
// norm, as float bits (squares are >= 0: the bits order like the values;
// r2b, x2b zero before).  Rows as in k_cover_sums.
__global__ __launch_bounds__(256) void k_cover_radius(const float* __restrict__ rows, const uint32_t* __restrict__ off,
                                                      const float* __restrict__ cen, uint32_t* __restrict__ r2b,
                                                      uint32_t* __restrict__ x2b) {
    const uint32_t a = blockIdx.x, part = blockIdx.y;
    const uint32_t p0 = off[a], p1 = off[a + 1];
    if (p0 + 4 * part >= p1) return;
    const uint32_t w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const float* ca = cen + (size_t)a * CV_NT;
    const float c0 = ca[l], c1 = ca[l + 64], c2 = l + 128 < (uint32_t)CV_NT ? ca[l + 128] : 0.f;
    uint32_t rb = 0, xb = 0;
    for (uint32_t p = p0 + 4 * part + w; p < p1; p += 4 * CV_SPLIT) {
        const float* x = rows + (size_t)p * CV_NT;
        const float v0 = x[l], v1 = x[l + 64], v2 = l + 128 < (uint32_t)CV_NT ? x[l + 128] : 0.f;
        const float t0 = v0 - c0, t1 = v1 - c1, t2 = v2 - c2;
        float d2 = fmaf(t0, t0, fmaf(t1, t1, t2 * t2));
        float x2 = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            d2 += __shfl_xor(d2, o, 64);
            x2 += __shfl_xor(x2, o, 64);
        }
        if (d2 == d2) {
            rb = max(rb, __float_as_uint(d2));
            xb = max(xb, __float_as_uint(x2));
        }
    }
    if (l == 0 && rb) {
        atomicMax(&r2b[a], rb);
        atomicMax(&x2b[a], xb);
    }
}

// M2[a][b] = min over the valid rows i of cluster a of the computed
// |x~_i - c~_b|^2 (clamped at 0; float bits, +inf before).  Block (a, s):
// the chunks s, s + CV_SPLIT, ... of CV_MAXT of a's 32-row tiles; wave w
// holds tile w of the chunk in registers, and the centre fragments stream
// through LDS CV_CT tiles a step (two buffers filled with global_load_lds,
// shared by the block's waves).  The MFMA's rows are the contigs (A), its
// columns the centres (B): each lane keeps the minimum over its 16 rows, one
// exchange between the lane halves finishes a wave's column, and an LDS
// minimum over the waves the block's; a cluster of one chunk stores it, a
// larger one takes the minimum with atomics.
constexpr uint32_t CV_MAXT = 4;  // row tiles a chunk: one a wave
constexpr uint32_t CV_CT = 4;    // centre tiles a step (36 KiB of fragments)
constexpr uint32_t CV_STEP_U4 = CV_CT * CV_KS * 64;

__global__ __launch_bounds__(256) void k_cover_min(const uint4* __restrict__ frag, const float* __restrict__ xn2,
                                                   const uint4* __restrict__ cfrag, const float4* __restrict__ info,
                                                   const uint32_t* __restrict__ off, uint32_t k,
                                                   uint32_t* __restrict__ m2b) {
    __shared__ uint4 Bl[2][CV_STEP_U4];
    __shared__ uint32_t smin[CV_CT * 32];
    const uint32_t a = blockIdx.x, part = blockIdx.y;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint32_t p0 = off[a], p1 = off[a + 1];
    if (p1 == p0) return;  // block-uniform
    const uint32_t ntc = (k + 31) / 32;
    const uint32_t rbase = 4 * (lane >> 5);
    const uint32_t t0 = p0 / 32, nt = (p1 - 1) / 32 - t0 + 1;
    const bool single = nt <= CV_MAXT;  // one chunk: each entry has one writer
    // the fragments of centre tiles [c0, c0 + CV_CT) into buf; entries past
    // the last tile are not loaded (tile boundaries are multiples of 64
    // entries, so the guard is uniform in a wave)
    auto fill = [&](uint32_t c0, uint4* buf) {
        const uint32_t valid = (min(ntc, c0 + CV_CT) - c0) * CV_KS * 64;
        const uint4* src = cfrag + (size_t)c0 * CV_KS * 64;
#pragma unroll
        for (uint32_t m = 0; m < CV_STEP_U4 / 256; ++m)
            if (256 * m + 64 * wave < valid)
                __builtin_amdgcn_global_load_lds((const void*)(src + 256 * m + tid),
                                                 (__attribute__((address_space(3))) void*)(buf + 256 * m + 64 * wave),
                                                 16, 0, 0);
    };
    static_assert(CV_STEP_U4 % 256 == 0, "a step's fragments in whole 256-entry pieces");
    for (uint32_t ch = part * CV_MAXT; ch < nt; ch += CV_SPLIT * CV_MAXT) {
        const uint32_t nc = min(CV_MAXT, nt - ch);
        const bool active = wave < nc;
        const uint32_t t = t0 + ch + wave;
        uint4 A[CV_KS];
        float xr[16];
#pragma unroll
        for (int ks = 0; ks < CV_KS; ++ks) A[ks] = active ? frag[((size_t)t * CV_KS + ks) * 64 + lane] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t pos = 32 * t + rbase + (r & 3) + 8 * (r >> 2);
            xr[r] = (active && pos >= p0 && pos < p1) ? xn2[pos] : __builtin_inff();  // other clusters: never minimal
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // the previous chunk's last step is done with Bl and smin
        for (uint32_t e = tid; e < CV_CT * 32; e += blockDim.x) smin[e] = 0x7f800000u;
        fill(0, Bl[0]);
        // |c~|^2 of this lane's column in each tile of a step, one step ahead
        auto norms = [&](uint32_t c0, float* out) {
#pragma unroll
            for (uint32_t c = 0; c < CV_CT; ++c) {
                const uint32_t col = (c0 + c) * 32 + (lane & 31);
                out[c] = col < k ? info[col].x : __builtin_inff();
            }
        };
        float cn[CV_CT], cnn[CV_CT];
        norms(0, cn);
        int buf = 0;
        for (uint32_t c0 = 0; c0 < ntc; c0 += CV_CT, buf ^= 1) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();  // this step's fragments and the smin reset are visible
            if (c0 + CV_CT < ntc) {
                fill(c0 + CV_CT, Bl[buf ^ 1]);
                norms(c0 + CV_CT, cnn);
            }
            if (active) {
#pragma unroll
                for (uint32_t c = 0; c < CV_CT; ++c) {
                    if (c0 + c >= ntc) break;
                    const float cn2 = cn[c];
                    f32x16_t acc = {};
#pragma unroll
                    for (int ks = 0; ks < CV_KS; ++ks) acc = cv_mfma(A[ks], Bl[buf][(c * CV_KS + ks) * 64 + lane], acc);
                    float m = __builtin_inff();
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float d = xr[r] + cn2 - 2.f * acc[r];
                        m = d < m ? d : m;  // NaN (no valid window) never lowers it
                    }
                    const float o = __shfl_xor(m, 32, 64);
                    m = o < m ? o : m;
                    if (lane < 32) atomicMin(&smin[c * 32 + lane], __float_as_uint(fmaxf(m, 0.f)));
                }
            }
#pragma unroll
            for (uint32_t c = 0; c < CV_CT; ++c) cn[c] = cnn[c];
            __syncthreads();  // every wave's minima are in smin
            for (uint32_t e = tid; e < CV_CT * 32; e += blockDim.x) {
                const uint32_t col = c0 * 32 + e;
                const uint32_t v = smin[e];
                if (col < k) {
                    if (single)
                        m2b[(size_t)a * k + col] = v;
                    else if (v != 0x7f800000u)
                        atomicMin(&m2b[(size_t)a * k + col], v);
                }
                smin[e] = 0x7f800000u;
            }
        }
    }
}

// Directed lists: list[a] = every b with the bound M[a][b] - r_b below R
// (ascending b; the first CV_CAP of them), cnt[a] = their number.  r bounds
// the members' distances from above (FP32 sums of 136 squares are within
// 1e-5 relative), xm their norms.  One wave per cluster.
__global__ __launch_bounds__(256) void k_cover_lists(const uint32_t* __restrict__ m2b, const float4* __restrict__ info,
                                                     const uint32_t* __restrict__ members,
                                                     const uint32_t* __restrict__ r2b, const uint32_t* __restrict__ x2b,
                                                     uint32_t k, float Rk, uint32_t* __restrict__ cnt,
                                                     uint32_t* __restrict__ list) {
    const uint32_t a = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (a >= k) return;
    const bool valid = members[a] != 0;
    const float xm = sqrtf(__uint_as_float(x2b[a])) * (1.f + 1.0f / 4096.f);
    uint32_t total = 0;
    for (uint32_t b0 = 0; b0 < k && valid; b0 += 64) {
        const uint32_t b = b0 + lane;
        bool keep = false;
        if (b < k && members[b]) {
            const float d2 = __uint_as_float(m2b[(size_t)a * k + b]);
            const float rb = sqrtf(__uint_as_float(r2b[b])) * (1.f + 1.0f / 4096.f) + 1e-6f;
            if (d2 < __builtin_inff()) {
                const float sm = xm + info[b].y;
                const float lb = sqrtf(fmaxf(d2 - 1e-5f * sm * sm, 0.f)) - sm * (1.0f / 256.0f);
                keep = lb - rb <= Rk;
            }
        }
        const uint64_t mk = __ballot(keep);
        const uint32_t o = total + (uint32_t)__popcll(mk & ((1ull << lane) - 1ull));
        if (keep && o < (uint32_t)CV_CAP) list[(size_t)a * CV_CAP + o] = b;
        total += (uint32_t)__popcll(mk);
    }
    if (lane == 0) cnt[a] = total;
}

// Mutual partners: mlist[a] = every b > a with b in a's list and a in b's
// (a list longer than the cap holds every cluster), ascending, the first
// CV_MCAP of them; mcnt[a] = their number (above CV_MCAP: the host takes
// every b > a).  One wave per cluster; membership by binary search in the
// ascending directed list.
constexpr uint32_t CV_MCAP = mdet::IVF_COVER_MCAP;

__device__ inline bool cv_listed(const uint32_t* __restrict__ cnt, const uint32_t* __restrict__ list, uint32_t a,
                                 uint32_t b) {
    const uint32_t c = cnt[a];
    if (c > (uint32_t)CV_CAP) return true;
    const uint32_t* L = list + (size_t)a * CV_CAP;
    uint32_t lo = 0, hi = c;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (L[mid] < b) lo = mid + 1; else hi = mid;
    }
    return lo < c && L[lo] == b;
}

__global__ __launch_bounds__(256) void k_cover_mutual(const uint32_t* __restrict__ cnt,
                                                      const uint32_t* __restrict__ list, uint32_t k,
                                                      uint32_t* __restrict__ mcnt, uint32_t* __restrict__ mlist,
                                                      uint32_t* __restrict__ ovf, uint32_t ovf_cap,
                                                      uint32_t* __restrict__ mstart) {
    const uint32_t a = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (a >= k) return;
    const bool full = cnt[a] > (uint32_t)CV_CAP;
    const uint32_t span = full ? k : cnt[a];  // candidates: every cluster, or a's list
    uint32_t total = 0;
    for (uint32_t q0 = 0; q0 < span; q0 += 64) {
        const uint32_t q = q0 + lane;
        bool keep = false;
        uint32_t b = 0;
        if (q < span) {
            b = full ? q : list[(size_t)a * CV_CAP + q];
            keep = b > a && cv_listed(cnt, list, b, a);
        }
        const uint64_t mk = __ballot(keep);
        const uint32_t o = total + (uint32_t)__popcll(mk & ((1ull << lane) - 1ull));
        if (keep && o < CV_MCAP) mlist[(size_t)a * CV_MCAP + o] = b;
        total += (uint32_t)__popcll(mk);
    }
    if (lane == 0) mcnt[a] = total;
    if (total <= CV_MCAP) return;
    // past the cap: the whole list once more into the overflow region
    // (ovf[0] counts the entries taken; mstart[a] = ~0 if it is full)
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(&ovf[0], total);
    base = (uint32_t)__shfl((int)base, 0, 64);
    if ((uint64_t)base + total > ovf_cap) {
        if (lane == 0) mstart[a] = 0xffffffffu;
        return;
    }
    if (lane == 0) mstart[a] = base;
    uint32_t w = 0;
    for (uint32_t q0 = 0; q0 < span; q0 += 64) {
        const uint32_t q = q0 + lane;
        bool keep = false;
        uint32_t b = 0;
        if (q < span) {
            b = full ? q : list[(size_t)a * CV_CAP + q];
            keep = b > a && cv_listed(cnt, list, b, a);
        }
        const uint64_t mk = __ballot(keep);
        if (keep) ovf[1 + base + w + (uint32_t)__popcll(mk & ((1ull << lane) - 1ull))] = b;
        w += (uint32_t)__popcll(mk);
    }
}

}  // namespace

namespace mdet {

constexpr int IVF_EVENT = 8;  // context event index marking the host copies

int ivf_launch(mdet_ctx* ctx, const float* emb, uint32_t n, uint32_t k, uint32_t n_probe, bool exact,
               IvfIndex* out) {
    if (!out || !emb || n == 0 || (n_probe == 0 && !exact)) MDET_FAIL(MDET_E_INVALID, "ivf_build: bad arguments");
    if (exact) n_probe = 1;  // the probe lists are not built
    // the cover's bound is tight only when a cluster holds one population:
    // more clusters than the probes use.  Measured at 200,000 contigs of
    // 1,000 genomes (bound with the model radius alone): n/128 clusters
    // 4.6 ms a call (0.64% of the pairs evaluated), n/96 5.4 ms, n/64 6.6 ms
    // (0.12%: above 2,048 clusters the k-means passes grow), n/160 4.7 ms
    // (3.2%); at 1,000,000 contigs of 5,000 genomes (shorter, noisier
    // contigs) n/128 66 ms (8.7%), n/84 46 ms (0.79%).  So n/128 while that
    // keeps the cheaper k-means schedule, n/84 above.
    if (k == 0 && exact) {
        const uint32_t k128 = std::max<uint32_t>(1, (n + 64) / 128);
        k = k128 <= 2048 ? k128 : (n + 42) / 84;
    }
    if (k == 0) k = std::max<uint32_t>(1, (n + 96) / 192);
    k = std::min<uint32_t>(std::min<uint32_t>(k, KM_MAX_K), n);
    if (n_probe > KM_MAX_PROBE)
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_edges_learned: n_probe %u above %u", n_probe, KM_MAX_PROBE);
    n_probe = std::min(n_probe, k);
    hipStream_t s = ctx->stream;
    float* cent;
    uint32_t *counts, *assign, *keys_sorted, *idx, *perm, *off, *probes, *err;
    unsigned long long* sums;
    KmFrame* frame;
    uint4* cfrag;
    const uint32_t ntiles = (k + 31) / 32;
    MDET_TRY(ctx_buf(ctx, "ivf.cent", (size_t)k * E_D, &cent));
    MDET_TRY(ctx_buf(ctx, "ivf.frame", 1, &frame));
    MDET_TRY(ctx_buf(ctx, "ivf.cfrag", (size_t)ntiles * KM_KF * 64, &cfrag));
    MDET_TRY(ctx_buf(ctx, "ivf.err", 1, &err));
    MDET_TRY(ctx_buf(ctx, "ivf.counts", (size_t)k + 1, &counts));
    MDET_TRY(ctx_buf(ctx, "ivf.sums", (size_t)k * E_D, &sums));
    MDET_TRY(ctx_buf(ctx, "ivf.assign", (size_t)n, &assign));
    MDET_TRY(ctx_buf(ctx, "ivf.keys", (size_t)n, &keys_sorted));
    MDET_TRY(ctx_buf(ctx, "ivf.idx", (size_t)n, &idx));
    MDET_TRY(ctx_buf(ctx, "ivf.perm", (size_t)n, &perm));
    MDET_TRY(ctx_buf(ctx, "ivf.off", (size_t)k + 1, &off));
    MDET_TRY(ctx_buf(ctx, "ivf.probes", (size_t)k * n_probe, &probes));

    // 1. k-means on a sample (every stride-th row), then every row
    hipLaunchKernelGGL(k_km_init, dim3(k), dim3(E_D), 0, s, emb, n, k, cent);
    hipLaunchKernelGGL(k_km_center, dim3(1), dim3(1024), 0, s, cent, k, frame);
    hipLaunchKernelGGL(k_km_extent, dim3(std::min<uint32_t>((n + 255) / 256, 4u * (uint32_t)ctx->num_cus)), dim3(256),
                       0, s, emb, n, frame);
    MDET_HIP(hipMemsetAsync(sums, 0, (size_t)k * E_D * 8, s));
    MDET_HIP(hipMemsetAsync(counts, 0, ((size_t)k + 1) * 4, s));
    MDET_HIP(hipMemsetAsync(err, 0, 4, s));
    const uint32_t stride =
        std::max<uint32_t>(1, n / std::max<uint32_t>(1, k * km_sample_per_cluster(exact ? 1 : k)));
    const uint32_t m = (n - 1) / stride + 1;
    // 2 row tiles x 4 waves per block where that still gives >= 8 blocks per
    // CU (measured 0.7 ms faster at 1M contigs than 4 row tiles, which hold
    // 2 waves per SIMD instead of 4), else 1 row tile x 8 waves (the
    // centroids split over more waves)
    const uint32_t tbits = km_tile_bits(k);
    auto assign_pass = [&](uint32_t pts, uint32_t str, uint32_t* out, unsigned long long* sm, int mode) {
        if ((pts + 63) / 64 >= 8u * (uint32_t)ctx->num_cus)
            hipLaunchKernelGGL((k_km_assign<2, 4>), dim3((pts + 63) / 64), dim3(256), 0, s, emb, pts, str, frame,
                               cfrag, k, out, counts, sm, mode, err, tbits);
        else
            hipLaunchKernelGGL((k_km_assign<1, 8>), dim3((pts + 31) / 32), dim3(512), 0, s, emb, pts, str, frame,
                               cfrag, k, out, counts, sm, mode, err, tbits);
    };
    const dim3 cf_grid((ntiles * 64 + 255) / 256);
    // the exact cover is exact whatever the clusters: the cheaper schedule
    // (measured at 1M contigs and 11,905 clusters: the 8 x 32 one took
    // 13 of the call's 47 ms)
    const int iters = exact ? km_iters(1) : km_iters(k);
    for (int it = 0; it < iters; ++it) {
        hipLaunchKernelGGL(k_km_cfrag, cf_grid, dim3(256), 0, s, cent, k, frame, cfrag);
        assign_pass(m, stride, (uint32_t*)nullptr, sums, 2);
        hipLaunchKernelGGL(k_km_update, dim3((k + 7) / 8), dim3(256), 0, s, sums, counts, k, cent);
    }
    hipLaunchKernelGGL(k_km_cfrag, cf_grid, dim3(256), 0, s, cent, k, frame, cfrag);
    assign_pass(n, 1u, assign, (unsigned long long*)nullptr, 1);
    MDET_HIP(hipGetLastError());

    // 2. rows sorted by cluster (stable), cluster offsets
    hipLaunchKernelGGL(k_iota, dim3((n + 255) / 256), dim3(256), 0, s, idx, n);
    int end_bit = 1;
    while ((1u << end_bit) < k) ++end_bit;
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, assign, keys_sorted, idx, perm, (int)n, 0, end_bit, s));
    void* t;
    MDET_TRY(ctx_buf(ctx, "ivf.sorttmp", tmp, &t));
    MDET_HIP(hipcub::DeviceRadixSort::SortPairs(t, tmp, assign, keys_sorted, idx, perm, (int)n, 0, end_bit, s));
    size_t tmp2 = 0;
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp2, counts, off, (int)k + 1, s));
    void* t2;
    MDET_TRY(ctx_buf(ctx, "ivf.scantmp", tmp2, &t2));
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(t2, tmp2, counts, off, (int)k + 1, s));

    // 3. probe lists
    if (!exact) hipLaunchKernelGGL(k_km_probe, dim3((k + 3) / 4), dim3(256), 0, s, cent, counts, k, n_probe, probes);
    MDET_HIP(hipGetLastError());

    // 4. copies for the host part
    void* hb;
    MDET_TRY(ctx_host_buf(ctx, "ivf.h_index", ((size_t)k + 2 + (size_t)k * n_probe) * 4, &hb));
    uint32_t* h_off = static_cast<uint32_t*>(hb);
    uint32_t* h_err = h_off + k + 1;  // read by ivf_finish as the word after the offsets
    uint32_t* h_probes = h_err + 1;
    MDET_HIP(hipMemcpyAsync(h_off, off, ((size_t)k + 1) * 4, hipMemcpyDeviceToHost, s));
    if (!exact) MDET_HIP(hipMemcpyAsync(h_probes, probes, (size_t)k * n_probe * 4, hipMemcpyDeviceToHost, s));
    MDET_HIP(hipMemcpyAsync(h_err, err, 4, hipMemcpyDeviceToHost, s));
    hipEvent_t ev;
    MDET_TRY(ctx_event(ctx, IVF_EVENT, &ev));
    MDET_HIP(hipEventRecord(ev, s));
    out->h_off = h_off;
    out->h_probes = h_probes;
    out->n_probe = n_probe;
    out->perm = perm;
    out->probes_dev = probes;
    out->cluster_dev = keys_sorted;
    out->off_dev = off;
    out->k = k;
    out->exact = exact;
    return MDET_OK;
}

int ivf_cover_space(mdet_ctx* ctx, const float* tnf_dev, uint32_t n, float* y_dev) {
    if (!tnf_dev || !y_dev || n == 0) MDET_FAIL(MDET_E_INVALID, "ivf_cover_space: bad arguments");
    const uint32_t grid = std::min<uint32_t>((n + 15) / 16, 8u * (uint32_t)ctx->num_cus);
    hipLaunchKernelGGL(k_cover_project, dim3(grid), dim3(256), 0, ctx->stream, tnf_dev, n, y_dev);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

int ivf_cover(mdet_ctx* ctx, const uint4* frag, const float* rows, uint32_t n, double R, IvfIndex* out) {
    if (!out || !out->exact || !frag || !rows) MDET_FAIL(MDET_E_INVALID, "ivf_cover: bad arguments");
    hipStream_t s = ctx->stream;
    const uint32_t k = out->k, ntc = (k + 31) / 32;
    float* xn2;
    float4* info;
    uint4* cfrag;
    uint32_t *cnt, *list;
    unsigned long long* sums;
    uint32_t *members, *r2b, *x2b, *m2b;
    float* cen;
    MDET_TRY(ctx_buf(ctx, "cover.xn2", (size_t)n, &xn2));
    MDET_TRY(ctx_buf(ctx, "cover.info", (size_t)k, &info));
    MDET_TRY(ctx_buf(ctx, "cover.cfrag", (size_t)ntc * CV_KS * 64, &cfrag));
    MDET_TRY(ctx_buf(ctx, "cover.sums", (size_t)k * 144, &sums));
    MDET_TRY(ctx_buf(ctx, "cover.members", (size_t)k * 3, &members));  // members, r2 bits, x2 bits
    MDET_TRY(ctx_buf(ctx, "cover.cen", (size_t)k * CV_NT, &cen));
    MDET_TRY(ctx_buf(ctx, "cover.m2", (size_t)k * k, &m2b));
    MDET_TRY(ctx_buf(ctx, "cover.cnt", (size_t)k, &cnt));
    MDET_TRY(ctx_buf(ctx, "cover.list", (size_t)k * CV_CAP, &list));
    r2b = members + k;
    x2b = members + 2 * (size_t)k;
    MDET_HIP(hipMemsetAsync(sums, 0, (size_t)k * 144 * 8, s));
    MDET_HIP(hipMemsetAsync(members, 0, (size_t)k * 3 * 4, s));
    MDET_HIP(hipMemsetD32Async((hipDeviceptr_t)m2b, 0x7f800000u, (size_t)k * k, s));  // +inf
    hipLaunchKernelGGL(k_cover_xn2, dim3((n + 3) / 4), dim3(256), 0, s, rows, n, xn2);
    hipLaunchKernelGGL(k_cover_sums, dim3(k, CV_SPLIT), dim3(256), 0, s, rows, out->off_dev, sums, members);
    hipLaunchKernelGGL(k_cover_centre, dim3(k), dim3(256), 0, s, sums, members, k, cen, cfrag, info);
    hipLaunchKernelGGL(k_cover_radius, dim3(k, CV_SPLIT), dim3(256), 0, s, rows, out->off_dev, cen, r2b, x2b);
    hipLaunchKernelGGL(k_cover_min, dim3(k, CV_SPLIT), dim3(256), 0, s, frag, xn2, cfrag, info, out->off_dev, k, m2b);
    const float Rk = (float)(R * (1.0 + 1e-6)) + 1e-6f;
    hipLaunchKernelGGL(k_cover_lists, dim3((k + 3) / 4), dim3(256), 0, s, m2b, info, members, r2b, x2b, k, Rk, cnt,
                       list);
    uint32_t *mcnt, *mlist, *ovf;
    MDET_TRY(ctx_buf(ctx, "cover.mcnt", (size_t)k * 2, &mcnt));  // counts, then overflow starts
    MDET_TRY(ctx_buf(ctx, "cover.mlist", (size_t)k * CV_MCAP, &mlist));
    MDET_TRY(ctx_buf(ctx, "cover.ovf", (size_t)IVF_COVER_OVF + 1, &ovf));
    MDET_HIP(hipMemsetAsync(ovf, 0, 4, s));
    hipLaunchKernelGGL(k_cover_mutual, dim3((k + 3) / 4), dim3(256), 0, s, cnt, list, k, mcnt, mlist, ovf,
                       (uint32_t)IVF_COVER_OVF, mcnt + k);
    MDET_HIP(hipGetLastError());
    void* hb;
    MDET_TRY(ctx_host_buf(ctx, "ivf.h_cover", ((size_t)2 * k + (size_t)k * CV_MCAP + IVF_COVER_OVF + 1) * 4, &hb));
    uint32_t* h_cnt = static_cast<uint32_t*>(hb);     // k counts, k overflow starts
    uint32_t* h_list = h_cnt + 2 * (size_t)k;
    uint32_t* h_ovf = h_list + (size_t)k * CV_MCAP;  // taken count, entries
    MDET_HIP(hipMemcpyAsync(h_cnt, mcnt, (size_t)2 * k * 4, hipMemcpyDeviceToHost, s));
    MDET_HIP(hipMemcpyAsync(h_list, mlist, (size_t)k * CV_MCAP * 4, hipMemcpyDeviceToHost, s));
    MDET_HIP(hipMemcpyAsync(h_ovf, ovf, ((size_t)IVF_COVER_OVF + 1) * 4, hipMemcpyDeviceToHost, s));
    hipEvent_t ev;
    MDET_TRY(ctx_event(ctx, IVF_EVENT, &ev));
    MDET_HIP(hipEventRecord(ev, s));
    out->h_cnt = h_cnt;
    out->h_list = h_list;
    out->h_ovf = h_ovf;
    return MDET_OK;
}

int ivf_finish(mdet_ctx* ctx, IvfIndex* out) {
    hipEvent_t ev;
    MDET_TRY(ctx_event(ctx, IVF_EVENT, &ev));
    MDET_HIP(hipEventSynchronize(ev));
    const uint32_t k = out->k, n_probe = out->n_probe;
    // the pinned copies are slow to read from the host: what the loops below
    // touch is copied into ordinary memory first (sequential reads)
    thread_local std::vector<uint32_t> off_local;
    off_local.assign(out->h_off, out->h_off + k + 2);
    const uint32_t* offh = off_local.data();
    const uint32_t* probeh = out->h_probes;
    if (offh[k + 1] & 1u)  // the error word follows the offsets
        MDET_FAIL(MDET_E_RANGE, "mdet_tnf_edges_learned: an embedding row is non-finite or too large to cluster");
    auto usable = [&](uint32_t b) { return b < k && offh[b + 1] > offh[b]; };
    std::vector<uint64_t> cp;  // (rows cluster << 32) | column cluster, rows <= columns
    uint64_t nitems = 0;
    auto count_items = [&](uint32_t lo, uint32_t hi) {
        // items: the rows of cluster lo in pieces ending at 32-aligned
        // ITEM_ROWS boundaries (a single-row diagonal piece has no pair)
        for (uint32_t rs = offh[lo], r1 = offh[lo + 1]; rs < r1;) {
            const uint32_t re = std::min<uint32_t>((rs & ~31u) + ITEM_ROWS, r1);
            nitems += (lo != hi || rs + 1 < r1) ? 1 : 0;
            rs = re;
        }
    };
    if (out->exact) {
        // the mutual partners b > a of each cluster (k_cover_mutual), with
        // the diagonal pairs; a list over its cap: every b > a (more pairs,
        // none missed).  Host reads of the pinned copies are slow: the
        // lengths are read once, of the lists only the entries in use.
        thread_local std::vector<uint32_t> mc;
        mc.assign(out->h_cnt, out->h_cnt + 2 * (size_t)k);  // counts, overflow starts
        const uint32_t* ml = out->h_list;  // only the listed entries are read
        const uint32_t* ov = out->h_ovf + 1;
        out->cover_full = 0;
        for (uint32_t a = 0; a < k; ++a) {
            const bool over = mc[a] > IVF_COVER_MCAP, lost = over && mc[k + a] == 0xffffffffu;
            if (lost) ++out->cover_full;
            if (!usable(a)) continue;
            cp.push_back(((uint64_t)a << 32) | a);
            count_items(a, a);
            auto take = [&](uint32_t b) {
                if (!usable(b)) return;
                cp.push_back(((uint64_t)a << 32) | b);
                count_items(a, b);
            };
            if (lost)  // no room left in the overflow region: every b > a
                for (uint32_t b = a + 1; b < k; ++b) take(b);
            else if (over)
                for (uint32_t q = 0; q < mc[a]; ++q) take(ov[mc[k + a] + q]);
            else
                for (uint32_t q = 0; q < mc[a]; ++q) take(ml[(size_t)a * IVF_COVER_MCAP + q]);
        }
    } else {
        // distinct unordered cluster pairs {a, b} with b in a's probes or a in
        // b's, each once: emitted by a for b >= a, and for b < a only when a is
        // not among b's probes (then b emits it).  Bitmap of (b, a) listings.
        thread_local std::vector<uint64_t> listed;  // all zero between calls
        if (listed.size() < ((size_t)k * k + 63) / 64) listed.assign(((size_t)k * k + 63) / 64, 0ull);
        for (uint32_t b = 0; b < k; ++b)
            for (uint32_t p = 0; p < n_probe; ++p) {
                const uint32_t a = probeh[(size_t)b * n_probe + p];
                if (a < k) listed[((size_t)b * k + a) >> 6] |= 1ull << (((size_t)b * k + a) & 63);
            }
        auto is_listed = [&](uint32_t b, uint32_t a) {
            return (listed[((size_t)b * k + a) >> 6] >> (((size_t)b * k + a) & 63)) & 1ull;
        };
        cp.reserve((size_t)k * n_probe);
        for (uint32_t a = 0; a < k; ++a) {
            if (!usable(a)) continue;
            for (uint32_t p = 0; p < n_probe; ++p) {
                const uint32_t b = probeh[(size_t)a * n_probe + p];
                if (!usable(b) || (b < a && is_listed(b, a))) continue;
                const uint32_t lo = std::min(a, b), hi = std::max(a, b);
                cp.push_back(((uint64_t)lo << 32) | hi);
                count_items(lo, hi);
            }
        }
        for (uint32_t b = 0; b < k; ++b)
            for (uint32_t p = 0; p < n_probe; ++p) {
                const uint32_t a = probeh[(size_t)b * n_probe + p];
                if (a < k) listed[((size_t)b * k + a) >> 6] = 0ull;
            }
    }
    if (nitems > 0x7fffffffull) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_edges_learned: too many cluster items");
    uint4* items = nullptr;
    if (nitems) {
        // the previous call's upload from this buffer finished before that call returned
        void* hb;
        MDET_TRY(ctx_host_buf(ctx, "ivf.h_items", nitems * sizeof(uint4), &hb));
        items = static_cast<uint4*>(hb);
    }
    uint64_t pairs = 0, w = 0;
    for (uint64_t key : cp) {
        const uint32_t a = (uint32_t)(key >> 32), b = (uint32_t)key;
        const uint32_t a0 = offh[a], a1 = offh[a + 1], b0 = offh[b], b1 = offh[b + 1];
        for (uint32_t rs = a0; rs < a1;) {
            const uint32_t re = std::min<uint32_t>((rs & ~31u) + ITEM_ROWS, a1);
            if (a == b) {
                if (rs + 1 < a1) items[w++] = make_uint4(rs, re, rs, a1 | ITEM_TRI);
                // pairs i < j, i in [rs, re), j in [rs, a1): sum of (a1 - 1 - i)
                const uint64_t cnt = re - rs;
                pairs += cnt * (a1 - 1) - (cnt * (2 * (uint64_t)rs + cnt - 1)) / 2;
            } else {
                items[w++] = make_uint4(rs, re, b0, b1);
                pairs += (uint64_t)(re - rs) * (b1 - b0);
            }
            rs = re;
        }
    }
    out->pairs = pairs;
    out->probe_pairs = (uint32_t)cp.size();
    out->nitems = (uint32_t)nitems;
    MDET_TRY(ctx_buf(ctx, "ivf.items", std::max<size_t>(nitems, 1), &out->items_dev));
    if (nitems)
        MDET_HIP(hipMemcpyAsync(out->items_dev, items, nitems * sizeof(uint4), hipMemcpyHostToDevice, ctx->stream));
    return MDET_OK;
}

}  // namespace mdet
