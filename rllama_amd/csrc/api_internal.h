// api_internal.h -- what the translation units behind the C ABI (api.hip, api_ops.hip) share: the context and tensor
// objects, the error helpers and the context lock.
#pragma once

#include "../../include/rllama_hip.h"
#include "kernels.h"
#include "tensor_pool.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <initializer_list>
#include <mutex>

namespace rlh {
// records the calling thread's error text (rlh_last_error) and returns `code`
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
int set_error(int code, const char *msg);
} // namespace rlh

#define HIP_TRY(expr)                                                                                          \
    do {                                                                                                       \
        hipError_t _e = (expr);                                                                                \
        if (_e != hipSuccess) {                                                                                \
            return rlh::fail(_e == hipErrorOutOfMemory ? RLH_ERR_OOM : RLH_ERR_HIP, "%s failed: %s (%s:%d)",   \
                             #expr, hipGetErrorString(_e), __FILE__, __LINE__);                                \
        }                                                                                                      \
    } while (0)

// Work memory of the op-level entry points that need more than their operands (rlh_attn_decode, rlh_argmax_greedy):
// allocated on first use, kept until rlh_shutdown.
struct OpScratch {
    rlh::DecodeState *state = nullptr;
    float *attn_ws = nullptr;      // partial triples of a split sequence
    size_t attn_ws_floats = 0;
    unsigned *tickets = nullptr;   // [kOpMaxHeads]
    int32_t *token = nullptr;      // one id
    void *gemm_ws = nullptr;       // partial sums of products cut along K and the parts of an fp32 operand (gemm_work_reserve)
    size_t gemm_ws_bytes = 0;
};
constexpr int kOpMaxHeads = 1024;

// The library's switches.  Read from the environment (RLLAMA_HIP_<NAME>) once, when the context is made, and changed
// afterwards only through rlh_set_option under the context lock: no launch path reads the environment.
struct Tunables {
    rlh::GemmTune gemm{};
    int gemv_burst_fixed = 0;      // GEMV_BURST=0: single-row products always issue bursts of 8 loads per lane
    int attn_chunk = -1;           // ATTN_CHUNK: positions per workgroup of a split sequence: N >= 16, 0 = 128, -1 = about one workgroup per compute unit
    int attn_single_max = 384;     // ATTN_SINGLE_MAX=N: longest sequence one workgroup per head handles alone
    int attn_merge_mode = 2;       // ATTN_MERGE=0: the pieces of a split sequence are combined by a second launch; 2: inside the kernel
    int attn_lds = 0;              // ATTN_LDS=1: cache rows staged through LDS (comparison form)
    int prefill_attn_gemm = 0;     // PREFILL_ATTN=gemm: multi-token attention as two batched GEMMs around a softmax kernel
    int prefill_attn_order = 2;    // PREFILL_ATTN_ORDER=0/1/2: launch order of the query blocks of the one-kernel attention
    int decode_graph = 0;          // DECODE_GRAPH=1: greedy decode loops replay one captured HIP graph per token
    int decode_fold = 1;           // DECODE_FOLD=0: embedding row and greedy pick as launches of their own instead of inside the first and last product of a token step
};

namespace rlh {
// applies NAME=value (value nullptr: back to the default); false if the name or the value is not known
bool tunables_set(Tunables &t, const char *name, const char *value);
void tunables_from_env(Tunables &t);
} // namespace rlh

constexpr size_t kStageBytes = (size_t)1 << 20;

struct rlh_ctx {
    int device = 0;
    int verbose = 0;
    hipStream_t stream = nullptr;
    hipDeviceProp_t prop;
    std::recursive_mutex mu;
    OpScratch ops;
    // Buffers of freed tensors, guarded by mu.  Everything that touches a tensor's buffer is ordered on the context's one stream (tensors
    // that another context's operation used are not kept: rlh_tensor::lent), so a buffer may be handed out while work of its former owner
    // is still queued.  Given back when memory runs out (device_alloc) and by rlh_shutdown.
    rlh::TensorPool pool;
    Tunables tun;
    unsigned tun_version = 0;        // bumped by rlh_set_option: captured decode steps of an older version are dropped
    // Page-locked staging of small host transfers, [0, kStageBytes) for uploads and as much again for downloads: a call holds mu from its first
    // transfer until the stream is idle, so one call uses it at a time.  Null until the first use, or where it could not be allocated.
    char *stage = nullptr;
    bool stage_busy = false; // an upload from it may still be queued; every call that uploads ends with stage_download, unless it fails
    void *noalloc_scratch = nullptr; // this device's address of the library's static work memory (api_ops.hip)
};

struct rlh_tensor {
    rlh_ctx *ctx = nullptr;
    void *p = nullptr;
    int rows = 0, cols = 0, dtype = RLH_F16;
    size_t capacity = 0; // bytes allocated at p
    // an operation of another context has read or written the buffer: work on that context's stream may still be queued when the tensor
    // is freed, so the buffer is not handed out again but freed, which waits for the device
    mutable std::atomic<bool> lent{false};
    size_t esize() const { return dtype == RLH_F16 ? 2 : 4; }
    size_t count() const { return (size_t)rows * cols; }
};

struct rlh_event {
    rlh_ctx *ctx = nullptr;
    hipEvent_t ev = nullptr;
};

struct CtxLock {
    std::lock_guard<std::recursive_mutex> g;
    explicit CtxLock(rlh_ctx *c) : g(c->mu) { (void)hipSetDevice(c->device); }
};

namespace rlh {
// Transfers between the caller's pageable memory and the device with the context locked, through page-locked staging where they fit.
// stage_upload: `host` is the caller's again at once.  stage_download: waits for the stream.
hipError_t stage_upload(rlh_ctx *ctx, void *dev, const void *host, size_t bytes);
hipError_t stage_download(rlh_ctx *ctx, void *host, const void *dev, size_t bytes);
void pool_release(rlh_ctx *ctx); // waits for the stream and frees the kept buffers
// hipMalloc for everything the library holds on the device: when memory runs out, the context's kept buffers are freed first
hipError_t device_alloc(rlh_ctx *ctx, void **p, size_t bytes);
// Work memory of products: kGemmPartialBytes, and where `need` (split3_work_bytes) is more, as much of that as kGemmWorkMax allows -- or
// what there is already, if memory runs out on the way: products then go in more passes.  Growing waits for the context's stream.
hipError_t gemm_work_reserve(rlh_ctx *ctx, void **p, size_t *bytes, size_t need);
} // namespace rlh

// Notes that an operation of `user` is about to use the tensors.
inline void lend(const rlh_ctx *user, std::initializer_list<const rlh_tensor *> tensors) {
    for (const rlh_tensor *t : tensors)
        if (t->ctx != user) t->lent.store(true, std::memory_order_relaxed);
}

namespace rlh {
void ops_release(rlh_ctx *ctx); // frees the op-level work memory (rlh_shutdown)
// looks up the context's device address of the static work memory of rlh_attn_decode_noalloc; rlh_init calls it with the
// device current
int noalloc_setup(rlh_ctx *ctx);
// how many blocks per head the decode attention uses at sequence length T
int attn_splits_rule(int T, int n_heads, int compute_units, int single_max, int chunk, int max_splits);
} // namespace rlh
