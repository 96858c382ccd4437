// Sequence ingest on gfx950: ASCII bases of the joined contigs -> the 2-bit
// packed stream and the N-run list the counting kernel reads.
//
// The reference keeps the FASTA text in pinned host memory and walks it per
// contig (cuda/Cuda2.cu:1436-1572 reader, 1823-1864 TNF loop; the MetaBAT1
// variant copies the raw bytes to the device, cuda/Cuda.cu:1706-1736).  Here
// the joined sequence bytes (kseq semantics: line breaks removed, as
// extra/kseq.h:190-229 reads them) are packed on the device, so the stream the
// TNF kernels read never passes through the host at 2 bits per base.
//
// Format (identical to the host packer mdet_pack_ascii): base p at bits
// 2*(p%16) of word p/16, A/a=0 C/c=1 G/g=2 T/t=3; any other byte is an N,
// stored as 0 and listed in maximal runs [start, end) of global positions.
//
// Work split: a thread packs 16 bases into one word, a wave a chunk of 64 words
// (1 KiB of text) at a time; per chunk one word says how many N runs start in
// it, whether it holds an N at all and whether its last base is one, and only
// chunks with an N store their per-word N masks.  A scan over blocks of 64
// chunks gives each block its first run index; the second pass reads the chunk
// words and visits only chunks in which a run starts or ends.  (The k-th end
// closes the k-th run: before a position as many runs have ended as have
// started, less the one that is open.)  Bound by reading the text and writing
// the stream: 656 MB + 164 MB in 161 us, 213 us in all; a thread a word with four 4-byte
// loads and ~140 instructions of decoding, and the runs counted and written from
// all masks in strides of 16 words a thread, took 552 us.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstring>

#include "hip_common.h"

namespace {

constexpr int ING_THREADS = 256;
constexpr int ING_CHUNKS = 64;   // chunks of a block ...
constexpr int ING_WAVE = 16;     // ... and of each of its waves
constexpr uint64_t ING_BLOCK_WORDS = 64 * ING_CHUNKS;
constexpr uint32_t CHUNK_ANY = 1u << 30;   // chunk word: holds an N
constexpr uint32_t CHUNK_LAST = 1u << 31;  // its last base is an N
constexpr uint32_t CHUNK_STARTS = 0xffffu;

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Four characters: their 2-bit codes a byte each (a/c/g/t in either case: 0..3
// from bits 1 and 2, ((x>>1)^(x>>2)) & 3), and what they differ by from the
// letters of those codes (zero bytes: A/C/G/T).
__device__ inline void decode4(uint32_t x, uint32_t& code, uint32_t& diff) {
    const uint32_t lo = x | 0x20202020u;
    code = ((lo ^ (lo >> 1)) >> 1) & 0x03030303u;
    diff = lo ^ __builtin_amdgcn_perm(0u, 0x74676361u, code);  // "acgt"
}
// Four 2-bit codes, one per byte, side by side.
__device__ inline uint32_t pack4(uint32_t code) { return __builtin_amdgcn_udot4(code, 0x40100401u, 0u, false); }
// 1 in each byte that is not zero.
__device__ inline uint32_t nonzero_bytes(uint32_t d) {
    return ((((d & 0x7f7f7f7fu) + 0x7f7f7f7fu) | d) >> 7) & 0x01010101u;
}

__device__ inline u32x4_t load16(const char* __restrict__ seq, uint64_t p, uint64_t total, bool aligned) {
    if (aligned && p + 16 <= total) return *reinterpret_cast<const u32x4_t*>(seq + p);
    u32x4_t v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t x = 0;
        for (int k = 0; k < 4; ++k) {
            const uint64_t at = p + 4 * q + k;
            x |= (uint32_t)(at < total ? (uint8_t)seq[at] : (uint8_t)'A') << (8 * k);
        }
        v[q] = x;
    }
    return v;
}

__device__ inline bool is_n(char c) {
    uint32_t code, diff;
    decode4((uint8_t)c, code, diff);
    return (diff & 0xffu) != 0;
}

// m shifted by one base: bit k = base p0 + k - 1 of the lane's word is an N.
__device__ inline uint32_t shifted_mask(uint32_t m, bool before, int lane) {
    const uint32_t prev = (uint32_t)__shfl_up((int)(m >> 15), 1, 64);
    return (m << 1) | (lane ? prev & 1u : before ? 1u : 0u);
}

// Bases past the end are packed as A (0) and not N.
__global__ __launch_bounds__(ING_THREADS) void k_pack_words(const char* __restrict__ seq, uint64_t total,
                                                           uint64_t nw, bool aligned, uint32_t* __restrict__ packed,
                                                           uint16_t* __restrict__ nmask,
                                                           uint32_t* __restrict__ chunk,
                                                           uint64_t* __restrict__ nstart) {
    constexpr int U = 4;  // chunks in flight
    __shared__ uint32_t s_starts;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (threadIdx.x == 0) s_starts = 0;
    __syncthreads();
    const uint64_t c0 = (uint64_t)blockIdx.x * ING_CHUNKS + wave * ING_WAVE;
    uint32_t starts = 0;
    for (int k = 0; k < ING_WAVE && (c0 + k) * 64 < nw; k += U) {
        u32x4_t x[U];
        char before[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t p = ((c0 + k + u) * 64 + lane) * 16;
            x[u] = load16(seq, p, total, aligned);
            const uint64_t first = (c0 + k + u) * 1024;
            before[u] = first && first <= total ? seq[first - 1] : 'A';
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t c = c0 + k + u, w = c * 64 + lane;
            if (c * 64 >= nw) break;
            uint32_t code[4], diff[4], word = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                decode4(x[u][q], code[q], diff[q]);
                word |= pack4(code[q]) << (8 * q);
            }
            uint32_t info = 0;
            if (__any((diff[0] | diff[1] | diff[2] | diff[3]) != 0)) {
                uint32_t m = 0;
                word = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t nz = nonzero_bytes(diff[q]);
                    m |= __builtin_amdgcn_udot4(nz, 0x08040201u, 0u, false) << (4 * q);
                    word |= pack4(code[q] & ~(nz * 3u)) << (8 * q);
                }
                if (w < nw) nmask[w] = (uint16_t)m;
                const uint32_t s = m & ~shifted_mask(m, is_n(before[u]), lane);
                uint32_t cnt = (uint32_t)__popc(s & 0xffffu);
#pragma unroll
                for (int off = 32; off >= 1; off >>= 1) cnt += (uint32_t)__shfl_xor((int)cnt, off, 64);
                const uint32_t last = (uint32_t)__builtin_amdgcn_readlane((int)m, 63) >> 15 & 1u;
                info = CHUNK_ANY | (last ? CHUNK_LAST : 0u) | cnt;
                starts += cnt;
            }
            if (w < nw) packed[w] = word;
            if (lane == 0) chunk[c] = info;
        }
    }
    if (lane == 0 && starts) atomicAdd(&s_starts, starts);
    __syncthreads();
    if (threadIdx.x == 0) nstart[blockIdx.x] = s_starts;
}

__global__ __launch_bounds__(ING_THREADS) void k_run_write(const uint16_t* __restrict__ nmask,
                                                          const uint32_t* __restrict__ chunk, uint64_t nw,
                                                          uint64_t total, const uint64_t* __restrict__ ostart,
                                                          uint64_t* __restrict__ runs, uint64_t cap) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    // a chunk a lane: what it holds, whether a run is open before it, the runs started before it
    const uint64_t b0 = (uint64_t)blockIdx.x * ING_CHUNKS, mine = b0 + lane;
    const bool in = mine * 64 < nw;
    const uint32_t info = in ? chunk[mine] : 0u;
    const uint32_t open = in && mine ? chunk[mine - 1] >> 31 : 0u;
    uint32_t incl = info & CHUNK_STARTS;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)incl, off, 64);
        if (lane >= off) incl += y;
    }
    const uint32_t excl = incl - (info & CHUNK_STARTS);
    uint64_t work = __ballot((info & CHUNK_ANY) || open) >> (wave * ING_WAVE) & ((1u << ING_WAVE) - 1u);
    if (!work) return;
    const uint64_t base = ostart[blockIdx.x];
    for (; work; work &= work - 1) {
        const int c = wave * ING_WAVE + __builtin_ctzll(work);
        const uint32_t ci = (uint32_t)__builtin_amdgcn_readlane((int)info, c);
        const bool co = __builtin_amdgcn_readlane((int)open, c) != 0;
        const uint64_t w = (b0 + c) * 64 + lane, p0 = w * 16;
        const uint32_t m = (ci & CHUNK_ANY) && w < nw ? nmask[w] : 0u;
        const uint32_t shifted = shifted_mask(m, co, lane);
        uint32_t s = m & ~shifted & 0xffffu, e = 0;
        if (w < nw) {
            const uint32_t len = total - p0 < 16 ? (uint32_t)(total - p0) : 16u;
            e = ~m & shifted & ((1u << len) - 1u);                          // non-N after N
            if (p0 + len == total && ((m >> (len - 1)) & 1u)) e |= 1u << len;  // the sequence ends in N
        }
        uint32_t sx = (uint32_t)__popc(s), ex = (uint32_t)__popc(e);
        const uint32_t sn = sx, en = ex;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t a = (uint32_t)__shfl_up((int)sx, off, 64), b = (uint32_t)__shfl_up((int)ex, off, 64);
            if (lane >= off) {
                sx += a;
                ex += b;
            }
        }
        const uint64_t first = base + (uint32_t)__builtin_amdgcn_readlane((int)excl, c);
        uint64_t ks = first + (sx - sn), ke = first - (co ? 1u : 0u) + (ex - en);
        for (; s; s &= s - 1, ++ks)
            if (ks < cap) runs[2 * ks] = p0 + __builtin_ctz(s);
        for (; e; e &= e - 1, ++ke)
            if (ke < cap) runs[2 * ke + 1] = p0 + __builtin_ctz(e);
    }
}

}  // namespace

using namespace mdet;

extern "C" {

int mdet_pack_ascii_dev(mdet_ctx* ctx, const char* seq_dev, uint64_t n_bases, uint32_t* packed_dev,
                        uint64_t packed_words, uint64_t* runs_dev, uint64_t runs_cap, uint64_t* n_runs) {
    MDET_TRY(check_ctx(ctx));
    if (!n_runs) MDET_FAIL(MDET_E_INVALID, "mdet_pack_ascii_dev: null n_runs");
    *n_runs = 0;
    if (n_bases == 0) return MDET_OK;
    if (!seq_dev || !packed_dev) MDET_FAIL(MDET_E_INVALID, "mdet_pack_ascii_dev: null sequence or packed buffer");
    if (runs_cap && !runs_dev) MDET_FAIL(MDET_E_INVALID, "mdet_pack_ascii_dev: runs_cap > 0 with null runs");
    const uint64_t nw = (n_bases + 15) / 16;
    if (nw > packed_words)
        MDET_FAIL(MDET_E_CAPACITY, "mdet_pack_ascii_dev: packed buffer holds %llu words, need %llu",
                  (unsigned long long)packed_words, (unsigned long long)nw);
    const uint64_t nblk = (nw + ING_BLOCK_WORDS - 1) / ING_BLOCK_WORDS;
    if ((nw + ING_THREADS - 1) / ING_THREADS > 0x7fffffffull)
        MDET_FAIL(MDET_E_RANGE, "mdet_pack_ascii_dev: %llu bases is too many", (unsigned long long)n_bases);
    uint16_t* nmask;
    uint32_t* chunk;
    uint64_t *bst, *ost;
    MDET_TRY(ctx_buf(ctx, "ingest.nmask", nw, &nmask));
    MDET_TRY(ctx_buf(ctx, "ingest.chunk", (size_t)nblk * ING_CHUNKS, &chunk));
    MDET_TRY(ctx_buf(ctx, "ingest.bst", nblk + 1, &bst));
    MDET_TRY(ctx_buf(ctx, "ingest.ost", nblk + 1, &ost));
    const bool aligned = ((uintptr_t)seq_dev & 3u) == 0;
    hipLaunchKernelGGL(k_pack_words, dim3((unsigned)nblk), dim3(ING_THREADS), 0, ctx->stream, seq_dev, n_bases, nw,
                       aligned, packed_dev, nmask, chunk, bst);
    MDET_HIP(hipGetLastError());
    // exclusive scan over the blocks (the last entry receives the total and is not read)
    size_t tmp = 0;
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, bst, ost, (int)nblk + 1, ctx->stream));
    void* t;
    MDET_TRY(ctx_buf(ctx, "cub.tmp", tmp, &t));
    MDET_HIP(hipcub::DeviceScan::ExclusiveSum(t, tmp, bst, ost, (int)nblk + 1, ctx->stream));
    hipLaunchKernelGGL(k_run_write, dim3((unsigned)nblk), dim3(ING_THREADS), 0, ctx->stream, nmask, chunk, nw, n_bases,
                       ost, runs_dev, runs_cap);
    MDET_HIP(hipGetLastError());
    uint64_t tot[1];
    {
        void* st_host;
        MDET_TRY(ctx_host_stage(ctx, 64, &st_host));
        MDET_HIP(hipMemcpyAsync(st_host, ost + nblk, 8, hipMemcpyDeviceToHost, ctx->stream));
        MDET_HIP(hipStreamSynchronize(ctx->stream));
        memcpy(tot, st_host, 8);
    }
    *n_runs = tot[0];
    if (tot[0] > runs_cap)
        MDET_FAIL(MDET_E_CAPACITY, "mdet_pack_ascii_dev: %llu N runs, capacity %llu", (unsigned long long)tot[0],
                  (unsigned long long)runs_cap);
    return MDET_OK;
}

}  // extern "C"
