// TNF counting on gfx950: 2-bit packed stream -> per-contig canonical
// tetranucleotide counts -> L2-normalised FP32 rows.
//
// Reference semantics: openmp/TNF.cpp:160-219 (oracle), cuda/Cuda2.cu:1823-1864
// and cuda/Cuda.cu:222-269 (GPU variant: one thread walks a whole contig).
//
// Layout and work split (MI355X-first):
//   * The packed stream (16 bases per uint32) is cut into fixed chunks of
//     CNT_CHUNK bases of window END positions, one 256-thread block each, so
//     every block streams the same number of bytes whatever the contig
//     lengths (1.5 kb .. 2 Mb).  The 3-base halo of a window is read from the
//     previous word, which the neighbouring lane loads anyway (L1/L2 hit).
//   * Thread t reads words 4t .. 4t+3 of the chunk with one 16-byte load
//     (a wave's load covers 1 KB) and the word before them for the halo:
//     64 window ends per lane, so the per-lane tests (contig boundaries, N)
//     are paid once per 64 windows, as bit masks.  Windows go two at a time
//     where both count towards one contig, the rest one by one, and lanes
//     spanning three contigs (contigs under 64 bases) window by window.
//   * Windows are binned by their raw codes (10 bits a pair, 8 a window) into
//     block-shared LDS histograms per contig segment of the chunk; the fold to
//     the 136 canonical columns (code and reverse complement) happens once per
//     segment at flush, so the per-pair work is extract + mask test + one LDS
//     add.
//   * N bases come as a sorted run list; a block whose chunk meets runs turns
//     them into an LDS bitmap of the chunk once, and a lane's N mask is then
//     three dwords of it.  Contig boundaries of the pass sit in registers.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <mutex>

#include "hip_common.h"
#include "tnf_tables.h"

namespace {

constexpr int CNT_THREADS = 256;
constexpr int CNT_WORDS = 4;  // consecutive words per thread (64 window ends)
constexpr uint64_t CNT_CHUNK = (uint64_t)CNT_THREADS * CNT_WORDS * 16;
constexpr int CNT_MAXSEG = 4;  // contig segments histogrammed per pass
// LDS adds bound the counting, so two neighbouring windows (5 bases) are one add
// into a histogram of 1,024 codes wherever both count towards one contig;
// the others, at contig ends and N runs, go one by one
// into a histogram of 256 codes.  The fold adds a 4-base code's windows up from
// the 5-base codes that begin or end with it.  With the larger code space adds
// of one wave instruction to one bin are rare, so one copy of it does; 4
// segments keep the block at 23 KB of LDS.  2.65e9 windows: 622 us (LDS and VALU
// about half busy each, the rest latency of the short blocks); one add
// a window (four copies of 256 codes): 752 us.
constexpr int CNT_PAIRS = 1024, CNT_SEGSZ = CNT_PAIRS + 256;  // words of a segment's histograms
// dwords of the per-chunk N bitmap: positions -32 .. CNT_CHUNK + 31
constexpr int CNT_NBM = (int)(CNT_CHUNK / 32) + 2;

__constant__ int16_t c_colmap[256] = {
#define M(i) mdet::kColumnMap.col[i]
#define R8(i) M(i), M(i + 1), M(i + 2), M(i + 3), M(i + 4), M(i + 5), M(i + 6), M(i + 7)
#define R64(i) R8(i), R8(i + 8), R8(i + 16), R8(i + 24), R8(i + 32), R8(i + 40), R8(i + 48), R8(i + 56)
    R64(0), R64(64), R64(128), R64(192)
#undef R64
#undef R8
#undef M
};

// upper_bound(a[0..len), v) - 1: last index with a[i] <= v, -1 if none.
__device__ inline int64_t last_le(const uint64_t* a, int64_t len, uint64_t v) {
    int64_t lo = 0, hi = len;  // answer in [lo-1, hi-1]
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (a[mid] <= v) lo = mid + 1;
        else hi = mid;
    }
    return lo - 1;
}

// First run index k in [0, nr) whose end runs[2k+1] > v (ends are sorted).
__device__ inline int64_t first_end_gt(const uint64_t* runs, int64_t nr, uint64_t v) {
    int64_t lo = 0, hi = nr;
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (runs[2 * mid + 1] > v) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}
// First run index k whose start runs[2k] >= v.
__device__ inline int64_t first_start_ge(const uint64_t* runs, int64_t nr, uint64_t v) {
    int64_t lo = 0, hi = nr;
    while (lo < hi) {
        int64_t mid = (lo + hi) >> 1;
        if (runs[2 * mid] >= v) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// Per chunk: the contigs holding its first and last base and the N runs that
// can touch its windows (binary searches, one thread per chunk, so the
// counting blocks do not start with a chain of dependent loads).
// meta = (first contig, last contig, first run, end run); contig -1 -> 0.
//
// The same launch clears the counts (a kernel, not hipMemsetAsync, so that
// callers may capture the no-allocation entry point in a graph), and with `edges` (host memory) hands the
// caller base_off[0] and base_off[n]; offsets that do not fit n_bases set
// *refused, and then this and the kernels behind it leave counts and rows as
// they are.  One launch ahead of the counting instead of two copies, a wait, a
// clear and a launch: 2,000 contigs 59 -> 26 us.
__global__ __launch_bounds__(256) void k_count_begin(uint64_t n_bases, const uint64_t* __restrict__ runs,
                                                     uint64_t n_runs, const uint64_t* __restrict__ base_off,
                                                     uint32_t n, uint64_t nchunks, longlong4* __restrict__ meta,
                                                     uint32_t* __restrict__ counts, uint64_t* edges,
                                                     uint32_t* __restrict__ refused) {
    if (edges) {
        const uint64_t e0 = base_off[0], e1 = base_off[n];
        const bool bad = e1 < e0 || e1 > n_bases;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            edges[0] = e0;
            edges[1] = e1;
            *refused = bad ? 1u : 0u;
        }
        if (bad) return;
    }
    const uint64_t meta_blocks = (nchunks + 255) / 256;
    if (blockIdx.x >= meta_blocks) {
        const uint64_t zero_blocks = gridDim.x - meta_blocks, words = (uint64_t)n * 136;
        for (uint64_t i = (blockIdx.x - meta_blocks) * 256 + threadIdx.x; i < words; i += zero_blocks * 256) counts[i] = 0;
        return;
    }
    const uint64_t c = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= nchunks) return;
    const uint64_t chunk_lo = c * CNT_CHUNK;
    const uint64_t chunk_hi = min(chunk_lo + CNT_CHUNK, n_bases);
    int64_t c0 = last_le(base_off, (int64_t)n + 1, chunk_lo);
    int64_t c1 = last_le(base_off, (int64_t)n + 1, chunk_hi - 1);
    c0 = c0 < 0 ? 0 : c0;
    c1 = c1 > (int64_t)n - 1 ? (int64_t)n - 1 : c1;
    const uint64_t lo = chunk_lo >= 3 ? chunk_lo - 3 : 0;
    const int64_t r0 = n_runs ? first_end_gt(runs, (int64_t)n_runs, lo) : 0;
    const int64_t r1 = n_runs ? first_start_ge(runs, (int64_t)n_runs, chunk_hi) : 0;
    meta[c] = make_longlong4(c0, c1, r0, r1);
}

// Bits [a, b) of a 64-bit mask, a and b clamped to [0, 64].
__device__ inline uint64_t bit_range(int32_t a, int32_t b) {
    a = a < 0 ? 0 : a;
    b = b > 64 ? 64 : b;
    if (a >= b) return 0ull;
    const uint64_t below_b = b == 64 ? ~0ull : ((1ull << b) - 1ull);
    return below_b & (~0ull << a);
}

__global__ __launch_bounds__(CNT_THREADS) void k_count_packed(const uint32_t* __restrict__ packed, uint64_t n_bases,
                                                              const uint64_t* __restrict__ runs,
                                                              const uint64_t* __restrict__ base_off,
                                                              const longlong4* __restrict__ meta,
                                                              uint32_t* __restrict__ counts,
                                                              const uint32_t* __restrict__ refused) {
    constexpr int SEGSZ = CNT_SEGSZ;
    __shared__ __align__(16) uint32_t hist[CNT_MAXSEG][SEGSZ];
    __shared__ uint32_t fold[CNT_MAXSEG][136];
    // positions relative to the chunk start, as int32, clamped to [-4,
    // length + 17]: every comparison with a window of the chunk keeps its
    // outcome, and the per-lane tests stay 32-bit
    __shared__ int32_t seg[CNT_MAXSEG + 1];
    // N bitmap of the chunk: bit b is position b - 32 (the halo before the
    // chunk included); built once per chunk with N runs
    __shared__ uint32_t nbm[CNT_NBM];

    const int tid = threadIdx.x;
    const uint64_t chunk_lo = (uint64_t)blockIdx.x * CNT_CHUNK;
    const uint64_t chunk_hi = min(chunk_lo + CNT_CHUNK, n_bases);
    const int32_t clen = (int32_t)(chunk_hi - chunk_lo);
    const longlong4 mt = meta[blockIdx.x];
    if (refused && *refused) return;

    // This lane's 64 window ends q0 .. q0 + 63: words 4 tid .. 4 tid + 3 of the
    // chunk (one 16-byte load where aligned and whole) and the word before
    // them (the 3-base halo of the first windows).  A block lives for a few
    // microseconds, most of them waiting: these loads, then the runs' and the
    // boundaries' go out before the histograms are cleared.
    const int32_t q0 = tid * 64;
    const uint64_t w0 = chunk_lo / 16;
    const uint64_t n_words = (n_bases + 15) / 16;
    const uint32_t last_lw = (uint32_t)min<uint64_t>(n_words - 1 - w0, CNT_CHUNK / 16 - 1);
    uint32_t W[4] = {0u, 0u, 0u, 0u}, H = 0u;
    if (q0 < clen) {
        const uint32_t i0 = 4u * tid;
        if (i0 + 3 <= last_lw && ((uintptr_t)packed & 15u) == 0) {
            const uint4 v = *reinterpret_cast<const uint4*>(packed + w0 + i0);
            W[0] = v.x;
            W[1] = v.y;
            W[2] = v.z;
            W[3] = v.w;
        } else {
#pragma unroll
            for (int m = 0; m < 4; ++m) W[m] = packed[w0 + min(i0 + m, last_lw)];
        }
        if (w0 + i0 > 0) H = packed[w0 + i0 - 1];
    }
    const int64_t c_first = mt.x, c_last = mt.y;
    const int64_t r_first = mt.z, r_last = mt.w;
    auto rel = [&](uint64_t p) {
        const int64_t d = (int64_t)p - (int64_t)chunk_lo;
        return (int32_t)(d < -4 ? -4 : (d > clen + 17 ? clen + 17 : d));
    };
    const int nr = (int)(r_last - r_first);
    const bool any_n = nr > 0;
    uint64_t rs0 = 0, re0 = 0, off0 = 0;
    if (tid < nr) {
        rs0 = runs[2 * (r_first + tid)];
        re0 = runs[2 * (r_first + tid) + 1];
    }
    const int nseg0 = (int)min<int64_t>(CNT_MAXSEG, c_last - c_first + 1);
    if (tid <= CNT_MAXSEG && tid <= nseg0) off0 = base_off[c_first + tid];
    auto clear = [&](int nseg) {
        for (int i = tid; i < nseg * SEGSZ / 4; i += CNT_THREADS)
            reinterpret_cast<uint4*>(&hist[0][0])[i] = make_uint4(0u, 0u, 0u, 0u);
        for (int i = tid; i < CNT_MAXSEG * 136; i += CNT_THREADS) (&fold[0][0])[i] = 0;
    };
    clear(nseg0);
    // the N bitmap: each run ORs its bits into the dwords it covers (runs are
    // disjoint; most cover one or two dwords)
    if (any_n) {
        for (int d = tid; d < CNT_NBM; d += CNT_THREADS) nbm[d] = 0u;
        __syncthreads();
        for (int r = tid; r < nr; r += CNT_THREADS) {
            if (r != tid) {
                rs0 = runs[2 * (r_first + r)];
                re0 = runs[2 * (r_first + r) + 1];
            }
            const int32_t rs = rel(rs0) + 32, re = rel(re0) + 32;
            // bits [rs, re) of the bitmap; rel() keeps both in [28, clen + 49]
            for (int32_t d = rs >> 5; d <= (re - 1) >> 5 && rs < re; ++d) {
                const int32_t x0 = max(rs - 32 * d, 0), x1 = min(re - 32 * d, 32);
                atomicOr(&nbm[d], (uint32_t)(((1ull << x1) - 1ull) & ~((1ull << x0) - 1ull)));
            }
        }
    }
    // boundaries past the pass's last segment read as "never reached"
    if (tid <= CNT_MAXSEG) seg[tid] = tid <= nseg0 ? rel(off0) : INT32_MAX;
    __syncthreads();
    // window k's N test: bit k of nvalid (bases q0 + k - 3 .. q0 + k N-free)
    uint64_t nvalid = ~0ull;
    if (any_n) {
        const uint32_t d0 = (uint32_t)q0 >> 5;  // bitmap bits q0 + 29 .. q0 + 95
        const uint32_t m0 = nbm[d0], m1 = nbm[d0 + 1], m2 = nbm[d0 + 2];
        const uint64_t A = (uint64_t)(m0 >> 29) | ((uint64_t)m1 << 3) | ((uint64_t)m2 << 35);
        const uint64_t B = m2 >> 29;  // positions q0 + 61 .. q0 + 63
        nvalid = ~(A | (A >> 1) | (A >> 2) | (A >> 3) | (B << 61) | (B << 62) | (B << 63));
    }

    for (int64_t cs = c_first; cs <= c_last; cs += CNT_MAXSEG) {
        const int nseg = (int)min<int64_t>(CNT_MAXSEG, c_last - cs + 1);
        if (cs != c_first) {  // a chunk of more contigs: again for the next ones
            __syncthreads();
            if (tid <= CNT_MAXSEG) seg[tid] = tid <= nseg ? rel(base_off[cs + tid]) : INT32_MAX;
            clear(nseg);
            __syncthreads();
        }
        int32_t sg[CNT_MAXSEG + 1];
#pragma unroll
        for (int k = 0; k <= CNT_MAXSEG; ++k) sg[k] = seg[k];
        // the window codes are formed inside the pass: hoisted out of the
        // (mostly single-pass) loop they would hold 64+ registers
        asm volatile("" : "+v"(W[0]), "+v"(W[1]), "+v"(W[2]), "+v"(W[3]), "+v"(H));
        // segment t of position q0 and the next two boundaries
        int t = 0;
        int32_t s_lo = sg[0], s_hi = sg[1], s_hi2 = sg[2];
#pragma unroll
        for (int k = 1; k < CNT_MAXSEG; ++k)
            if (sg[k] <= q0) {
                t = k;
                s_lo = sg[k];
                s_hi = sg[k + 1];
                s_hi2 = k + 2 <= CNT_MAXSEG ? sg[k + 2 <= CNT_MAXSEG ? k + 2 : CNT_MAXSEG] : INT32_MAX;
            }
        const int32_t end = min(clen, q0 + 64);  // window ends of the lane in the chunk: [q0, end)
        const bool mine = q0 < clen && q0 + 64 > sg[0] && t < nseg;
        // more than one boundary among the lane's windows (contigs under 64
        // bases): counted window by window below
        const bool general = mine && s_hi2 < end;
        // windows of segment t, then of t + 1 from s_hi on (each window's
        // first base in its own contig): V = counted (N-free), S = in t + 1
        uint64_t V = 0ull, S = 0ull;
        if (mine && !general) {
            V = bit_range(s_lo + 3 - q0, min(s_hi, end) - q0);
            if (t + 1 < nseg) {
                S = bit_range(s_hi + 3 - q0, end - q0);
                V |= S;
            }
            V &= nvalid;
            S &= V;
        }
        uint32_t* const h0 = &hist[t][0];
        // windows in pairs (bit 2k of P: both of a pair count, into one
        // segment), 8 pairs of a word at a time, the increment 0 or 1 and, where
        // a lane's word meets a contig's end, the segment (t or t + 1) from the
        // masks; what is left, U, window by window
        const uint64_t P = V & (V >> 1) & ~(S ^ (S >> 1)) & 0x5555555555555555ull;
        uint64_t U = V & ~(P | (P << 1));
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint64_t x = ((uint64_t)W[m] << 32) | (m ? W[m > 0 ? m - 1 : 0] : H);
            const uint32_t p16 = (uint32_t)(P >> (16 * m)) & 0xFFFFu, s16 = (uint32_t)(S >> (16 * m)) & 0xFFFFu;
            // (N bases are scattered: in nearly every word some lane has one)
            if (__all(s16 == 0u || s16 == 0xFFFFu)) {
                uint32_t* const h = s16 ? h0 + SEGSZ : h0;
#pragma unroll
                for (int k = 0; k < 16; k += 2)
                    atomicAdd(&h[(uint32_t)(x >> (26 + 2 * k)) & 0x3FFu], (p16 >> k) & 1u);
            } else {
#pragma unroll
                for (int k = 0; k < 16; k += 2)
                    atomicAdd(&h0[((s16 >> k) & 1u) * SEGSZ + ((uint32_t)(x >> (26 + 2 * k)) & 0x3FFu)],
                              (p16 >> k) & 1u);
            }
        }
        for (; __any(U != 0); U &= U - 1) {
            if (!U) continue;
            const int k = __builtin_ctzll(U), m = k >> 4;
            const uint32_t hi = m == 0 ? W[0] : m == 1 ? W[1] : m == 2 ? W[2] : W[3];
            const uint32_t lo = m == 0 ? H : m == 1 ? W[0] : m == 2 ? W[1] : W[2];
            const uint64_t x = ((uint64_t)hi << 32) | lo;
            atomicAdd(&h0[(uint32_t)((S >> k) & 1u) * SEGSZ + CNT_PAIRS + ((uint32_t)(x >> (26 + 2 * (k & 15))) & 0xFFu)],
                      1u);
        }
        if (general) {
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const uint64_t x = ((uint64_t)W[m] << 32) | (m ? W[m > 0 ? m - 1 : 0] : H);
#pragma unroll 1
                for (int k = 0; k < 16; ++k) {
                    const int32_t p = q0 + 16 * m + k;
                    int u = 0;
#pragma unroll
                    for (int j = 1; j <= CNT_MAXSEG; ++j) u += sg[j] <= p ? 1 : 0;
                    const int32_t u_lo = seg[u < CNT_MAXSEG ? u : CNT_MAXSEG];
                    const bool ok = p < clen && u < nseg && p >= u_lo + 3 && ((nvalid >> (16 * m + k)) & 1ull);
                    if (ok) atomicAdd(&hist[u][CNT_PAIRS + ((uint32_t)(x >> (26 + 2 * k)) & 0xFFu)], 1u);
                }
            }
        }
        __syncthreads();
        // fold raw codes into canonical columns, then one global add per
        // nonzero column (a contig may span several chunks)
        for (int s = 0; s < nseg; ++s) {
            const uint4 last = *reinterpret_cast<const uint4*>(&hist[s][4 * tid]);  // pairs whose second window it is
            uint32_t v = hist[s][CNT_PAIRS + tid] + ((last.x + last.y) + (last.z + last.w));
#pragma unroll
            for (int c = 0; c < 4; ++c) v += hist[s][256 * c + tid];  // ... whose first
            if (v) atomicAdd(&fold[s][c_colmap[tid]], v);
        }
        __syncthreads();
        for (int i = tid; i < nseg * 136; i += CNT_THREADS) {
            int s = i / 136, col = i - s * 136;
            uint32_t v = fold[s][col];
            if (v) atomicAdd(&counts[(uint64_t)(cs + s) * 136 + col], v);
        }
    }
}

// One wavefront per contig: exact integer sum of squares, FP64 sqrt and
// division (both correctly rounded), one rounding to FP32.  Equals
// (float)(c / sqrt(sum c^2)) of openmp/TNF.cpp:208-217 bit for bit.
__global__ __launch_bounds__(256) void k_normalize(const uint32_t* __restrict__ counts, uint32_t n,
                                                   float* __restrict__ tnf, const uint32_t* __restrict__ refused) {
    if (refused && *refused) return;
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= n) return;
    const uint32_t* c = counts + r * 136;
    uint32_t v0 = c[lane], v1 = c[lane + 64], v2 = lane < 8 ? c[lane + 128] : 0u;
    uint64_t ss = (uint64_t)v0 * v0 + (uint64_t)v1 * v1 + (uint64_t)v2 * v2;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_xor(ss, off, 64);
    const double rsum = sqrt((double)ss);
    float* t = tnf + r * 136;
    t[lane] = (float)((double)v0 / rsum);
    t[lane + 64] = (float)((double)v1 / rsum);
    if (lane < 8) t[lane + 128] = (float)((double)v2 / rsum);
}

// ---- raw-byte input (get_TNF's [begin | end] index, cuda/Cuda.cu:222-226) --
// Contig c is bytes [index[c], index[n+c]).  Its windows (start positions
// 0 .. len-4) are cut into chunks of ASC_CHUNK starts; one 256-thread block
// per chunk stages the chunk's bytes (+3) in LDS, each thread forms 16 window
// codes, and the block's 256-bin histogram is folded into the contig's 136
// columns with one global add per nonzero column.
constexpr int ASC_THREADS = 256;
constexpr int ASC_CHUNK = ASC_THREADS * 16;

__global__ void k_ascii_chunks(const uint64_t* __restrict__ index, uint32_t n, uint32_t* __restrict__ nch) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c > n) return;
    if (c == n) {
        nch[n] = 0;
        return;
    }
    const uint64_t b = index[c], e = index[n + c];
    const uint64_t nw = e > b + 3 ? e - b - 3 : 0;  // window starts
    nch[c] = (uint32_t)((nw + ASC_CHUNK - 1) / ASC_CHUNK);
}

__device__ inline uint32_t ascii_code(uint8_t ch) {
    // A/a=0 C/c=1 G/g=2 T/t=3, anything else 4
    switch (ch | 0x20) {
        case 'a': return 0;
        case 'c': return 1;
        case 'g': return 2;
        case 't': return 3;
        default: return 4;
    }
}

__global__ __launch_bounds__(ASC_THREADS) void k_count_ascii(const char* __restrict__ seqs,
                                                             const uint64_t* __restrict__ index, uint32_t n,
                                                             const uint64_t* __restrict__ choff,
                                                             uint32_t* __restrict__ counts) {
    __shared__ uint8_t code[ASC_CHUNK + 3];
    __shared__ uint32_t hist[256];
    __shared__ uint32_t fold[136];
    __shared__ int64_t s_c;
    const int tid = threadIdx.x;
    const uint64_t blk = blockIdx.x;
    if (tid == 0) s_c = last_le(choff, (int64_t)n + 1, blk);
    hist[tid] = 0;
    if (tid < 136) fold[tid] = 0;
    __syncthreads();
    const int64_t c = s_c;  // choff[c] <= blk < choff[c+1] (empty contigs skipped)
    const uint64_t b = index[c], e = index[n + c];
    const uint64_t w0 = (blk - choff[c]) * (uint64_t)ASC_CHUNK;  // first window start of the chunk
    const uint64_t nw = e - b - 3;
    const uint32_t wn = (uint32_t)min<uint64_t>(ASC_CHUNK, nw - w0);
    for (uint32_t k = tid; k < wn + 3; k += ASC_THREADS) code[k] = (uint8_t)ascii_code((uint8_t)seqs[b + w0 + k]);
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < 16; ++k) {
        const uint32_t w = tid * 16 + k;
        if (w < wn) {
            const uint32_t c0 = code[w], c1 = code[w + 1], c2 = code[w + 2], c3 = code[w + 3];
            if ((c0 | c1 | c2 | c3) < 4) atomicAdd(&hist[c0 | (c1 << 2) | (c2 << 4) | (c3 << 6)], 1u);
        }
    }
    __syncthreads();
    if (hist[tid]) atomicAdd(&fold[c_colmap[tid]], hist[tid]);
    __syncthreads();
    if (tid < 136 && fold[tid]) atomicAdd(&counts[(uint64_t)c * 136 + tid], fold[tid]);
}

// Scratch of the no-allocation entry point (mdet_tnf_count_noalloc): the
// per-chunk metadata of k_count_begin, for up to NOALLOC_CHUNKS chunks of
// CNT_CHUNK bases (2^21 x 16,384 = 34.4e9 bases), 64 MiB held on every device
// the library runs on until the process ends.  Host code never passes
// `scratch` itself: its device address comes from hipGetSymbolAddress, once
// per device (count_scratch_setup), kept in g_scratch_ptr.
constexpr uint64_t NOALLOC_CHUNKS = 1ull << 21;
static __device__ __align__(256) longlong4 scratch[NOALLOC_CHUNKS];

constexpr int COUNT_EVENT = 7;  // context event index marking k_count_begin

void count_begin(mdet_ctx* ctx, uint64_t n_bases, const uint64_t* runs, uint64_t n_runs, const uint64_t* base_off,
                 uint32_t n, uint64_t nchunks, longlong4* meta, uint32_t* counts, uint64_t* edges, uint32_t* refused) {
    const uint64_t zero = std::min<uint64_t>(((uint64_t)n * 136 + 1023) / 1024, 2048), most = (nchunks + 255) / 256 + zero;
    hipLaunchKernelGGL(k_count_begin, dim3((unsigned)most), dim3(256), 0, ctx->stream, n_bases, runs, n_runs, base_off,
                       n, nchunks, meta, counts, edges, refused);
}

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
longlong4* g_scratch_ptr[MAX_DEVICES] = {};

}  // namespace

using namespace mdet;

namespace mdet {

int count_scratch_setup(int device) {
    if (device < 0 || device >= MAX_DEVICES)
        MDET_FAIL(MDET_E_RANGE, "device %d beyond the %d devices the library supports", device, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[device]) return MDET_OK;
    void* p = nullptr;
    MDET_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));  // the caller made `device` current
    if (!p) MDET_FAIL(MDET_E_HIP, "hipGetSymbolAddress returned a null address for the counting scratch");
    g_scratch_ptr[device] = static_cast<longlong4*>(p);
    return MDET_OK;
}

}  // namespace mdet

extern "C" {

int mdet_tnf_count(mdet_ctx* ctx, const uint32_t* packed_dev, uint64_t n_bases, const uint64_t* runs_dev,
                   uint64_t n_runs, const uint64_t* base_off_dev, uint32_t n, uint32_t* counts_dev,
                   float* tnf_dev) {
    MDET_TRY(check_ctx(ctx));
    if (n == 0) return MDET_OK;
    if (!base_off_dev || !tnf_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count: null base_off or tnf");
    if (n_bases && !packed_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count: null packed stream");
    if (n_runs && !runs_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count: n_runs > 0 with null runs");
    if (n > (1u << 31)) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_count: n = %u contigs exceeds 2^31", n);
    // The kernel reads only base_off[0..n], words below ceil(n_bases/16) and
    // runs[0..2*n_runs); base_off beyond n_bases only drops windows.
    const uint64_t nchunks = (n_bases + CNT_CHUNK - 1) / CNT_CHUNK;
    if (nchunks > 0x7fffffffu) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_count: %llu bases is too many", (unsigned long long)n_bases);
    uint32_t *counts = counts_dev, *refused;
    longlong4* meta = nullptr;
    void* host;
    hipEvent_t begun;
    if (!counts) MDET_TRY(ctx_buf(ctx, "count.counts", (size_t)n * 136, &counts));
    if (nchunks) MDET_TRY(ctx_buf(ctx, "count.meta", (size_t)nchunks, &meta));
    MDET_TRY(ctx_buf(ctx, "count.refused", 4, &refused));
    MDET_TRY(ctx_host_stage(ctx, 64, &host));
    MDET_TRY(ctx_event(ctx, COUNT_EVENT, &begun));
    uint64_t* edge = static_cast<uint64_t*>(host);
    count_begin(ctx, n_bases, runs_dev, n_runs, base_off_dev, n, nchunks, meta, counts, edge, refused);
    MDET_HIP(hipEventRecord(begun, ctx->stream));
    if (nchunks)
        hipLaunchKernelGGL(k_count_packed, dim3((unsigned)nchunks), dim3(CNT_THREADS), 0, ctx->stream, packed_dev,
                           n_bases, runs_dev, base_off_dev, meta, counts, refused);
    hipLaunchKernelGGL(k_normalize, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, counts, n, tnf_dev, refused);
    MDET_HIP(hipGetLastError());
    MDET_HIP(hipEventSynchronize(begun));
    if (edge[1] < edge[0]) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count: base_off is not non-decreasing");
    if (edge[1] > n_bases)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count: base_off[n] = %llu exceeds n_bases = %llu",
                  (unsigned long long)edge[1], (unsigned long long)n_bases);
    return MDET_OK;
}

int mdet_tnf_count_noalloc(mdet_ctx* ctx, const uint32_t* packed_dev, uint64_t n_bases, const uint64_t* runs_dev,
                           uint64_t n_runs, const uint64_t* base_off_dev, uint32_t n, uint32_t* counts_dev,
                           float* tnf_dev) {
    MDET_TRY(check_ctx(ctx));
    if (n == 0) return MDET_OK;
    if (!base_off_dev || !tnf_dev || !counts_dev)
        MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count_noalloc: null base_off, counts or tnf");
    if (n_bases && !packed_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count_noalloc: null packed stream");
    if (n_runs && !runs_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count_noalloc: n_runs > 0 with null runs");
    if (n > (1u << 31)) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_count_noalloc: n = %u contigs exceeds 2^31", n);
    const uint64_t nchunks = (n_bases + CNT_CHUNK - 1) / CNT_CHUNK;
    if (nchunks > NOALLOC_CHUNKS)
        MDET_FAIL(MDET_E_RANGE,
                  "mdet_tnf_count_noalloc: %llu bases need %llu chunks of %llu; the static scratch holds %llu "
                  "(%llu bases)",
                  (unsigned long long)n_bases, (unsigned long long)nchunks, (unsigned long long)CNT_CHUNK,
                  (unsigned long long)NOALLOC_CHUNKS, (unsigned long long)(NOALLOC_CHUNKS * CNT_CHUNK));
    longlong4* meta = g_scratch_ptr[ctx->device];
    if (!meta) MDET_FAIL(MDET_E_STATE, "mdet_tnf_count_noalloc: scratch of device %d not set up", ctx->device);
    count_begin(ctx, n_bases, runs_dev, n_runs, base_off_dev, n, nchunks, meta, counts_dev, nullptr, nullptr);
    if (nchunks)
        hipLaunchKernelGGL(k_count_packed, dim3((unsigned)nchunks), dim3(CNT_THREADS), 0, ctx->stream, packed_dev,
                           n_bases, runs_dev, base_off_dev, meta, counts_dev, (const uint32_t*)nullptr);
    hipLaunchKernelGGL(k_normalize, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, counts_dev, n, tnf_dev,
                       (const uint32_t*)nullptr);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

int mdet_tnf_count_ascii(mdet_ctx* ctx, const char* seqs_dev, const uint64_t* index_dev, uint32_t n,
                         uint32_t* counts_dev, float* tnf_dev) {
    MDET_TRY(check_ctx(ctx));
    if (n == 0) return MDET_OK;
    if (!seqs_dev || !index_dev || !tnf_dev) MDET_FAIL(MDET_E_INVALID, "mdet_tnf_count_ascii: null argument");
    if (n > (1u << 31)) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_count_ascii: n = %u contigs exceeds 2^31", n);
    uint32_t* counts = counts_dev;
    if (!counts) MDET_TRY(ctx_buf(ctx, "count.counts", (size_t)n * 136, &counts));
    uint32_t* nch;
    uint64_t* choff;
    MDET_TRY(ctx_buf(ctx, "ascii.nch", (size_t)n + 1, &nch));
    MDET_TRY(ctx_buf(ctx, "ascii.choff", (size_t)n + 1, &choff));
    MDET_HIP(hipMemsetAsync(counts, 0, (size_t)n * 136 * sizeof(uint32_t), ctx->stream));
    hipLaunchKernelGGL(k_ascii_chunks, dim3((n + 256) / 256), dim3(256), 0, ctx->stream, index_dev, n, nch);
    MDET_HIP(hipGetLastError());
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, nch, choff, (int)n + 1, ctx->stream));
    void* t;
    MDET_TRY(ctx_buf(ctx, "cub.tmp", tmp, &t));
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(t, tmp, nch, choff, (int)n + 1, ctx->stream));
    uint64_t total = 0;
    MDET_HIP(hipMemcpyAsync(&total, choff + n, sizeof total, hipMemcpyDeviceToHost, ctx->stream));
    MDET_HIP(hipStreamSynchronize(ctx->stream));
    if (total > 0x7fffffffull) MDET_FAIL(MDET_E_RANGE, "mdet_tnf_count_ascii: input too large");
    if (total)
        hipLaunchKernelGGL(k_count_ascii, dim3((unsigned)total), dim3(ASC_THREADS), 0, ctx->stream, seqs_dev,
                           index_dev, n, choff, counts);
    MDET_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_normalize, dim3((n + 3) / 4), dim3(256), 0, ctx->stream, counts, n, tnf_dev,
                       (const uint32_t*)nullptr);
    MDET_HIP(hipGetLastError());
    return MDET_OK;
}

}  // extern "C"
