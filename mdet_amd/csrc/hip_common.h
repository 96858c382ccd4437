// Device-side plumbing shared by the HIP translation units: error checks,
// the context object, grow-only scratch buffers and stage timers.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <unordered_map>
#include <vector>

#include "host_common.h"

#define MDET_HIP(call)                                                                        \
    do {                                                                                      \
        hipError_t _e = (call);                                                               \
        if (_e != hipSuccess) {                                                               \
            ::mdet::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(_e), __FILE__, \
                              __LINE__);                                                      \
            return MDET_E_HIP;                                                                \
        }                                                                                     \
    } while (0)

#define MDET_TRY(expr)               \
    do {                             \
        int _r = (expr);             \
        if (_r != MDET_OK) return _r; \
    } while (0)

struct mdet_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    struct Buf {
        void* p = nullptr;
        size_t bytes = 0;
    };
    std::unordered_map<std::string, Buf> bufs;   // scratch, grown on demand
    std::unordered_map<std::string, Buf> hbufs;  // pinned host buffers, grown on demand
    std::vector<hipEvent_t> events;
    // pinned host staging for small device->host reads (counters)
    void* host_stage = nullptr;
    size_t host_stage_bytes = 0;
    bool model_ready = false;  // FP32 model constants uploaded
    int num_cus = 0;
    // cached prefilter radius for (min log size, max log size, threshold)
    double radius_key[3] = {0, 0, 0};
    double radius = 0;
    bool radius_valid = false;
    // cached scan items for a row count, rows per block and column span
    uint32_t items_n = 0;
    uint32_t items_rows = 0;
    uint32_t items_seg = 0;
    uint32_t items_order = 0;
    uint32_t nitems = 0;
    // pair-stage launch shapes per precision mode (set by hand or by the
    // autotuner): prefilter item column span, persistent prefilter blocks,
    // refine blocks per CU, item order of the persistent blocks; the
    // autotuner's stage times at that shape
    struct Tune {
        uint32_t seg_cols = 0;  // 0: by size (seg_cols_for)
        uint32_t persistent = 1;
        uint32_t refine_blocks = 64;
        uint32_t item_order = 1;  // 1: per-XCD queues, column-segment major
        double ms_prefilter = 0, ms_refine = 0;
    } tune[4];
    uint64_t last_pairs = 0;  // refine records of the last edge-list call
    bool learned_fallback = true;  // learned mode: evaluate full rows again against every column
    uint32_t learned_margin_div = 32;  // full row: at least max_edges - max_edges / div kept proposals
    bool learned_exact_cover = false;  // learned mode: cluster pairs from the TNF-space bound, not probes
};

namespace mdet {

// Device scratch buffer `key` of at least `bytes` bytes, owned by the
// context (contents are not preserved across growth).
int ctx_buf(mdet_ctx* ctx, const char* key, size_t bytes, void** out);
template <class T>
int ctx_buf(mdet_ctx* ctx, const char* key, size_t count, T** out) {
    void* p = nullptr;
    int r = ctx_buf(ctx, key, count * sizeof(T), &p);
    *out = static_cast<T*>(p);
    return r;
}
int ctx_host_stage(mdet_ctx* ctx, size_t bytes, void** out);
// Pinned host buffer `key` of at least `bytes` bytes, owned by the context.
int ctx_host_buf(mdet_ctx* ctx, const char* key, size_t bytes, void** out);
int ctx_event(mdet_ctx* ctx, int idx, hipEvent_t* out);
int check_ctx(mdet_ctx* ctx);

// Upload of the FP32 model constants (Chebyshev coefficients) to the device.
int ensure_model(mdet_ctx* ctx);

// Device address of the counting path's static scratch array on the current
// device, looked up once per device (called by mdet_ctx_create).
int count_scratch_setup(int device);

}  // namespace mdet
