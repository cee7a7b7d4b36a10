// Shared host-side plumbing of libnncase_hip.so: context object, error
// recording, argument checks, small device helpers.  gfx950 only.
#pragma once

#include <hip/hip_runtime.h>

#include <cerrno>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/nncase_hip.h"
#include "once_per_kernel.hpp"
#include "weight_fetch.hpp"

struct nncase_hip_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    bool owns_stream = false;
    int compute_units = 0;
    int clock_khz = 0;
    size_t hbm_bytes = 0;
    // paged-attention partials and completion counters, owned by the context (calls on one context
    // are ordered on its stream, so they can share them).  Sized when an attention operator is
    // recorded into a function or first called eagerly; never moved while a captured graph holds
    // their addresses (attn_pins = captured functions with an attention operator).
    void *attn_ws = nullptr;
    size_t attn_ws_bytes = 0;
    void *attn_done = nullptr; // counters live apart from the partials: they must stay zero between calls
    size_t attn_done_bytes = 0;
    int attn_pins = 0;
    // this GPU's copy of the static scratch of nncase_hip_paged_attention_decode_noalloc (its device address, taken
    // when the context is created so that the entry point itself makes no runtime call but launches)
    void *attn_static = nullptr;
    // hostcall.hip: pinned host memory through which small operands travel (in flight until a host call has drained the
    // stream), and device scratch of calls on host tensors; both made on first use, bounded, kept with the context
    uint8_t *stage = nullptr;
    size_t stage_used = 0;
    void *arena = nullptr;
    size_t arena_bytes = 0;
    hipStream_t copy_stream = nullptr; // results on their way to the host beside the context's stream
    static constexpr int kCopySlots = 8;
    hipEvent_t copy_events[kCopySlots] = {nullptr};
    // function.hip: lanes 1.. of captured functions run on streams of their own, forked from the context's stream and joined back
    // into it; made when the first function with lanes is captured, kept with the context (calls on one context are ordered on its
    // stream, so its functions can share them)
    hipStream_t lane_streams[NNCASE_HIP_MAX_LANES] = {nullptr};
    hipEvent_t lane_events[NNCASE_HIP_MAX_LANES] = {nullptr}; // 0: the fork, l: the end of lane l
    std::mutex lane_lock;                                     // two threads' forks and joins do not mix
    char last_error[512] = {0};
};

namespace nnhip {

// Device address of the static scratch array of the attention entry point that allocates nothing, on `device`
// (which must be current).  attn.hip, where the array lives.
hipError_t attn_static_scratch_address(void **ptr);

// Asks for a dynamic LDS limit of `limit` bytes, always the same for one kernel (a call slow next to a launch: once per kernel and device).
template <auto Kernel> hipError_t raise_dynamic_lds(int device, int limit) {
    return once_per_kernel<Kernel>(device, [&] { return hipFuncSetAttribute(reinterpret_cast<const void *>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, limit); });
}

// hostcall.hip: device scratch of at least `bytes`, valid until the next call (`*temporary`: larger than what a context
// keeps, the caller gives it back with hipFree when the stream has drained); what a context holds for host calls.
int scratch_reserve(nncase_hip_ctx *ctx, size_t bytes, void **ptr, bool *temporary);
// Copies on the context's stream.  The one to the device may still be under way when it returns, but src may then be changed
// only once the stream has drained (small ones: at once); the other returns when dst holds the data.
int copy_to_device(nncase_hip_ctx *ctx, void *dst_dev, const void *src_host, size_t bytes);
int copy_to_host(nncase_hip_ctx *ctx, void *dst_host, const void *src_dev, size_t bytes);
int mark_result(nncase_hip_ctx *ctx, int slot);
int fetch_result(nncase_hip_ctx *ctx, int slot, void *dst_pinned, const void *src_dev, size_t bytes); // under way when it returns, on ctx->copy_stream
int drain_host_calls(nncase_hip_ctx *ctx); // waits for the context's stream
bool host_is_pinned(const void *ptr);      // a block of nncase_hip_host_malloc
void hostcall_attach();
void hostcall_release(nncase_hip_ctx *ctx);

// function.hip: the context's lane streams and events, up to `lanes`; given back with the context.
int lane_streams_reserve(nncase_hip_ctx *ctx, int lanes);
void lane_streams_release(nncase_hip_ctx *ctx);

// function.hip: a loaded model's list prepared for, and run with, results that go to host memory (complete on return).
void function_hoist_outputs(nncase_hip_function_t *fn, void *const *outputs_dev, int n);
int function_run_to_host(nncase_hip_function_t *fn, int n, void *const *outputs_dev, void *const *outputs_host, const size_t *bytes);

inline int fail(nncase_hip_ctx *ctx, int code, const char *fmt, ...) {
    if (ctx) {
        va_list ap;
        va_start(ap, fmt);
        vsnprintf(ctx->last_error, sizeof(ctx->last_error), fmt, ap);
        va_end(ap);
    }
    return code;
}

inline int hip_fail(nncase_hip_ctx *ctx, hipError_t e, const char *what) {
    return fail(ctx, -(NNCASE_HIP_ERR_HIP_BASE + (int)e), "%s: %s", what, hipGetErrorString(e));
}

#define NNHIP_CHECK_CTX(ctx)                                                                                           \
    do {                                                                                                               \
        if (!(ctx)) return -EINVAL;                                                                                    \
    } while (0)

#define NNHIP_REQUIRE(ctx, cond, code, ...)                                                                            \
    do {                                                                                                               \
        if (!(cond)) return ::nnhip::fail((ctx), (code), __VA_ARGS__);                                                 \
    } while (0)

#define NNHIP_HIP(ctx, expr)                                                                                           \
    do {                                                                                                               \
        hipError_t e__ = (expr);                                                                                       \
        if (e__ != hipSuccess) return ::nnhip::hip_fail((ctx), e__, #expr);                                            \
    } while (0)

// Checks the launch itself (bad configuration etc.); execution errors surface
// at the next synchronising call.
#define NNHIP_LAUNCH_CHECK(ctx, name)                                                                                  \
    do {                                                                                                               \
        hipError_t e__ = hipGetLastError();                                                                            \
        if (e__ != hipSuccess) return ::nnhip::hip_fail((ctx), e__, name);                                             \
    } while (0)

inline int dtype_size(int dt) {
    switch (dt) {
    case NNCASE_HIP_DT_I8:
    case NNCASE_HIP_DT_U8: return 1;
    case NNCASE_HIP_DT_I16:
    case NNCASE_HIP_DT_F16: return 2;
    case NNCASE_HIP_DT_I32:
    case NNCASE_HIP_DT_F32: return 4;
    default: return 0;
    }
}

// src/Native/include/nncase/kernels/kernel_utils.h:86-93
inline int32_t windowed_output_size(int32_t size, int32_t filter, int32_t stride, int32_t dilation, int32_t before,
                                    int32_t after) {
    const int32_t eff = (filter - 1) * dilation + 1;
    return (size + before + after - eff + stride) / stride;
}

// Division of a 31-bit numerator by a runtime constant as multiply-high +
// shift (round-up method): q = (n * mul) >> (32 + shift).
struct FastDiv {
    uint32_t mul;
    uint32_t shift;
    uint32_t div;
};

inline FastDiv make_fastdiv(uint32_t d) {
    FastDiv f;
    f.div = d;
    if (d == 1) {
        f.mul = 0;
        f.shift = 0;
        return f;
    }
    uint32_t l = 0;
    while ((1u << l) < d) l++;
    // mul = ceil(2^(32+l) / d) - 2^32, used as q = (umulhi(n, mul) + n) >> l
    const uint64_t m = ((uint64_t(1) << 32) * ((uint64_t(1) << l) - d)) / d + 1;
    f.mul = (uint32_t)m;
    f.shift = l;
    return f;
}

__device__ __forceinline__ uint32_t fastdiv(uint32_t n, const FastDiv &f) {
    // exact for n < 2^31 (Granlund-Montgomery / Hacker's Delight 10-9 form)
    // (a select, not a branch, for the divisor 1: callers count on straight-line code around their loads)
    const uint32_t t = __umulhi(n, f.mul);
    const uint32_t q = (t + ((n - t) >> 1)) >> ((f.shift - 1) & 31u);
    return f.div == 1 ? n : q;
}

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

template <typename TQ> struct QLimits;
template <> struct QLimits<uint8_t> { static constexpr float lo = 0.f, hi = 255.f; };
template <> struct QLimits<int8_t> { static constexpr float lo = -128.f, hi = 127.f; };
template <> struct QLimits<int16_t> { static constexpr float lo = -32768.f, hi = 32767.f; };

// rne(v) then saturate.  The clamp is done on the float before rounding: the
// limits are integers, so clamp and round-half-even commute, and values
// beyond the int32 range saturate instead of wrapping.
template <typename TQ> __device__ __forceinline__ TQ quantize_one(float x, float scale, float bias) {
    float v = x / scale + bias;
    v = fminf(fmaxf(v, QLimits<TQ>::lo), QLimits<TQ>::hi); // NaN -> lo
    return (TQ)(int32_t)rintf(v);
}


// attn.hip: checks the geometry and sizes the context's paged-attention workspace for it
// (-EBUSY if that needs a reallocation while a captured graph refers to it or the stream is capturing).
int attn_reserve(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *geometry);
// Bytes of split partials and of counters paged attention needs for a geometry, and the launch on areas the caller
// brings (the counters zero before the first launch; every launch leaves them zero again).
int attn_scratch_sizes(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *geometry, size_t *partial_bytes, size_t *counter_bytes);
int attn_decode_on(nncase_hip_ctx *ctx, const void *q_dev, const void *k_cache_dev, const void *v_cache_dev, const int32_t *block_table_dev,
                   const int32_t *ctx_lens_dev, void *out_dev, const nncase_hip_paged_attn_args_t *geometry, void *partials,
                   size_t partial_bytes, void *counters, size_t counter_bytes, const WeightFetches *fetch);
// The launch on the context's own areas.  `fetch` (may be null): weights that the operators behind it will read.
int attn_decode_on_context(nncase_hip_ctx *ctx, const void *q_dev, const void *k_cache_dev, const void *v_cache_dev,
                           const int32_t *block_table_dev, const int32_t *ctx_lens_dev, void *out_dev,
                           const nncase_hip_paged_attn_args_t *geometry, const WeightFetches *fetch);
// llm.hip: which weights each block of a product of m rows reads; false where its launch is of another kind.  rope: the q / k / v
// projection that rotates and appends.
bool w8a16_weight_fetch(const nncase_hip_ctx *ctx, const nncase_hip_w8a16_t *w, int m, int mode, bool normalises,
                        const nncase_hip_paged_attn_args_t *rope, WeightFetch *f);

// glue.hip: a max pool of stride 1 over its own result, `levels` times, and the channel concat of the tensor and all levels.
struct MaxPoolChain {
    const uint8_t *in;
    uint8_t *level[NNCASE_HIP_MAX_CONCAT - 1], *cat;
    int levels, batch, h, w, channels, kernel;
    nncase_hip_quant_param_t qp[NNCASE_HIP_MAX_CONCAT], cat_qp; // of the tensor and of every level
};
bool maxpool_chain_supported(const MaxPoolChain &c);
int launch_maxpool_chain(nncase_hip_ctx *ctx, const MaxPoolChain &c);

} // namespace nnhip
