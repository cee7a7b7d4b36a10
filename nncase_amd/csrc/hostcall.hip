// Calls on host tensors: how operands cross the host bus, and the convolution and matmul that take host arrays as the
// reference's kernels do (one call: operands up, weights packed, product, result down).
#include "qconv.hpp"

#include <algorithm>
#include <mutex>
#include <vector>

namespace nnhip {

constexpr size_t kStageBytes = 1 << 20;        // pinned memory of a context
// Largest upload or download of a host call that goes through it (convolution 96 -> 128 3x3 of 28 x 28, 190 KB up, 100 KB down:
// 98 us with the runtime's copies, 55 so; at a megabyte the host's own copy costs what the engines' start did).
constexpr size_t kStageMost = 512 << 10;
constexpr size_t kArenaMost = (size_t)256 << 20; // device scratch a context keeps

// A small copy is a kernel that reads or writes the pinned memory itself: the copy engines take about as long to be
// started and waited for as a chain of small kernels runs.
__global__ __launch_bounds__(256) void bus_copy_kernel(uint8_t *dst, const uint8_t *src, uint32_t bytes) {
    const uint32_t v = (blockIdx.x * 256 + threadIdx.x) * 16;
    if (v + 16 <= bytes) {
        *reinterpret_cast<uint4 *>(dst + v) = *reinterpret_cast<const uint4 *>(src + v);
    } else {
        for (uint32_t i = v; i < bytes; i++) dst[i] = src[i];
    }
}

static int launch_bus_copy(nncase_hip_ctx *ctx, void *dst, const void *src, size_t bytes) {
    hipLaunchKernelGGL(bus_copy_kernel, dim3((unsigned)((bytes + 4095) / 4096)), dim3(256), 0, ctx->stream, (uint8_t *)dst, (const uint8_t *)src,
                       (uint32_t)bytes);
    NNHIP_LAUNCH_CHECK(ctx, "bus_copy_kernel");
    return 0;
}

static bool capturing(nncase_hip_ctx *ctx) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

int drain_host_calls(nncase_hip_ctx *ctx) {
    NNHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    ctx->stage_used = 0;
    return 0;
}

// `bytes` of the pinned memory, 256-byte aligned; waits for the stream when it is used up.  Null: too large, no pinned
// memory to be had, or the stream is being recorded (the copy has to fail or run as an ordinary one).
static uint8_t *stage_take(nncase_hip_ctx *ctx, size_t bytes) {
    const size_t need = (bytes + 255) & ~(size_t)255;
    if (need > kStageBytes || capturing(ctx)) return nullptr;
    if (!ctx->stage && hipHostMalloc((void **)&ctx->stage, kStageBytes, hipHostMallocDefault) != hipSuccess) {
        ctx->stage = nullptr;
        (void)hipGetLastError();
        return nullptr;
    }
    if (ctx->stage_used + need > kStageBytes && drain_host_calls(ctx)) return nullptr;
    uint8_t *p = ctx->stage + ctx->stage_used;
    ctx->stage_used += need;
    return p;
}

int copy_to_device(nncase_hip_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (bytes <= kStageMost) {
        if (uint8_t *s = stage_take(ctx, bytes)) {
            memcpy(s, src, bytes);
            return launch_bus_copy(ctx, dst, s, bytes);
        }
    }
    NNHIP_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
    return 0;
}

int copy_to_host(nncase_hip_ctx *ctx, void *dst, const void *src, size_t bytes) {
    if (bytes <= kStageMost) {
        if (uint8_t *s = stage_take(ctx, bytes)) {
            int rc = launch_bus_copy(ctx, s, src, bytes);
            if (!rc) rc = drain_host_calls(ctx);
            if (!rc) memcpy(dst, s, bytes);
            return rc;
        }
    }
    NNHIP_HIP(ctx, hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    return drain_host_calls(ctx);
}

int scratch_reserve(nncase_hip_ctx *ctx, size_t bytes, void **ptr, bool *temporary) {
    *temporary = bytes > kArenaMost;
    if (*temporary) {
        const hipError_t e = hipMalloc(ptr, bytes);
        if (e == hipErrorOutOfMemory) return fail(ctx, -ENOMEM, "out of device memory (%zu bytes of scratch)", bytes);
        NNHIP_HIP(ctx, e);
        return 0;
    }
    if (bytes > ctx->arena_bytes) {
        if (ctx->arena) {
            const int rc = drain_host_calls(ctx);
            if (rc) return rc;
            NNHIP_HIP(ctx, hipFree(ctx->arena));
        }
        ctx->arena = nullptr, ctx->arena_bytes = 0;
        const size_t want = std::min(kArenaMost, std::max<size_t>(bytes + bytes / 2, 4 << 20));
        const hipError_t e = hipMalloc(&ctx->arena, want);
        if (e == hipErrorOutOfMemory) return fail(ctx, -ENOMEM, "out of device memory (%zu bytes of scratch)", want);
        NNHIP_HIP(ctx, e);
        ctx->arena_bytes = want;
    }
    *ptr = ctx->arena;
    return 0;
}

// Pinned memory for results.  The runtime brings 8 MB to pageable memory at 17 GB/s and to pinned memory at 56, but pinning
// costs more than that saves, so blocks are kept for the next result.  Shared by all contexts of the process; at most
// kHostPoolMost bytes in all, given back with the last context.
namespace {
constexpr size_t kHostPoolMost = (size_t)256 << 20;
struct HostBlock {
    void *ptr;
    size_t bytes;
    bool used;
};
struct HostPool {
    std::mutex mu;
    std::vector<HostBlock> blocks;
    size_t total = 0;
    int contexts = 0;

    void trim(size_t until) { // frees idle blocks, largest first, until the total is at most `until`
        while (total > until) {
            auto worst = blocks.end();
            for (auto it = blocks.begin(); it != blocks.end(); ++it)
                if (!it->used && (worst == blocks.end() || it->bytes > worst->bytes)) worst = it;
            if (worst == blocks.end()) return;
            (void)hipHostFree(worst->ptr);
            total -= worst->bytes;
            blocks.erase(worst);
        }
    }
};
HostPool &host_pool() {
    static HostPool *p = new HostPool; // (results may be dropped while the process ends)
    return *p;
}
} // namespace

// A result complete on the context's stream, marked where it is enqueued and fetched while later work runs.  The wait is the
// host's: it has nothing else to do by then, and making one stream wait for another on the device costs 25 us a time.
int mark_result(nncase_hip_ctx *ctx, int slot) {
    if (!ctx->copy_stream) NNHIP_HIP(ctx, hipStreamCreateWithFlags(&ctx->copy_stream, hipStreamNonBlocking));
    if (!ctx->copy_events[slot]) NNHIP_HIP(ctx, hipEventCreateWithFlags(&ctx->copy_events[slot], hipEventDisableTiming));
    NNHIP_HIP(ctx, hipEventRecord(ctx->copy_events[slot], ctx->stream));
    return 0;
}

int fetch_result(nncase_hip_ctx *ctx, int slot, void *dst_pinned, const void *src, size_t bytes) {
    NNHIP_HIP(ctx, hipEventSynchronize(ctx->copy_events[slot]));
    NNHIP_HIP(ctx, hipMemcpyAsync(dst_pinned, src, bytes, hipMemcpyDeviceToHost, ctx->copy_stream));
    return 0;
}

bool host_is_pinned(const void *ptr) {
    std::lock_guard<std::mutex> guard(host_pool().mu);
    for (const HostBlock &b : host_pool().blocks)
        if (b.ptr == ptr && b.used) return true;
    return false;
}

void hostcall_attach() {
    std::lock_guard<std::mutex> guard(host_pool().mu);
    host_pool().contexts++;
}

void hostcall_release(nncase_hip_ctx *ctx) {
    {
        std::lock_guard<std::mutex> guard(host_pool().mu);
        if (--host_pool().contexts == 0) host_pool().trim(0);
    }
    for (hipEvent_t &e : ctx->copy_events) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (ctx->copy_stream) (void)hipStreamDestroy(ctx->copy_stream);
    ctx->copy_stream = nullptr;
    if (ctx->stage) (void)hipHostFree(ctx->stage);
    if (ctx->arena) (void)hipFree(ctx->arena);
    ctx->stage = nullptr, ctx->arena = nullptr;
    ctx->stage_used = ctx->arena_bytes = 0;
}

namespace {

struct Carve { // consecutive 256-byte aligned pieces of the scratch
    size_t total = 0;
    size_t take(size_t bytes) {
        const size_t at = total;
        total += (bytes + 255) & ~(size_t)255;
        return at;
    }
};

// One dense layer on host operands.  x: NCHW (relayout) or rows as they are; the result in the same order.
int dense_host_call(nncase_hip_ctx *ctx, nncase_hip_weights *w, const uint8_t *x_host, const RawWeights &raw_host, const int32_t *bias_host,
                    void *y_host, const nncase_hip_conv2d_args_t *a, int out_h, int out_w, bool nchw) {
    int rc = igemm_plan(ctx, w, bias_host);
    if (rc) return rc;
    const int es = a->out_dtype == NNCASE_HIP_DT_U8 ? 1 : 4;
    const size_t x_bytes = (size_t)a->batch * a->in_h * a->in_w * w->in_channels;
    const size_t w_bytes = (size_t)w->out_channels * w->g_ic * w->kernel_h * w->kernel_w;
    const size_t y_bytes = (size_t)a->batch * out_h * out_w * w->out_channels * es;
    const bool move_x = nchw && a->in_h * a->in_w > 1 && w->in_channels > 1, move_y = nchw && out_h * out_w > 1 && w->out_channels > 1;
    Carve c;
    // what goes up lies first and together, so that small operands are one copy: weights, bias, activations
    const size_t o_w = c.take(w_bytes);
    const size_t o_b = c.take(sizeof(int32_t) * w->out_channels), o_x = c.take(x_bytes), up = c.total;
    const size_t o_c = c.take(igemm_const_bytes(w)), o_xn = move_x ? c.take(x_bytes) : o_x, o_y = c.take(y_bytes), o_yn = move_y ? c.take(y_bytes) : o_y;
    void *base = nullptr;
    bool temporary = false;
    rc = scratch_reserve(ctx, c.total, &base, &temporary);
    if (rc) return rc;
    uint8_t *const d = reinterpret_cast<uint8_t *>(base);
    igemm_place(w, d + o_c);
    w->d_bias = reinterpret_cast<int32_t *>(d + o_b);
    auto run = [&]() -> int {
        if (uint8_t *s = up <= kStageMost ? stage_take(ctx, up) : nullptr) {
            memcpy(s + o_w, raw_host.ptr, w_bytes);
            if (bias_host) memcpy(s + o_b, bias_host, sizeof(int32_t) * w->out_channels);
            else memset(s + o_b, 0, sizeof(int32_t) * w->out_channels);
            memcpy(s + o_x, x_host, x_bytes);
            if (int r = launch_bus_copy(ctx, d, s, up)) return r;
        } else {
            if (int r = copy_to_device(ctx, d + o_w, raw_host.ptr, w_bytes)) return r;
            if (bias_host) {
                if (int r = copy_to_device(ctx, d + o_b, bias_host, sizeof(int32_t) * w->out_channels)) return r;
            } else {
                NNHIP_HIP(ctx, hipMemsetAsync(d + o_b, 0, sizeof(int32_t) * w->out_channels, ctx->stream));
            }
            if (int r = copy_to_device(ctx, d + o_x, x_host, x_bytes)) return r;
        }
        RawWeights raw = raw_host;
        raw.ptr = d + o_w;
        if (int r = igemm_pack(ctx, w, raw)) return r;
        if (move_x)
            if (int r = nncase_hip_nchw_to_nhwc(ctx, d + o_x, d + o_xn, 1, a->batch, w->in_channels, a->in_h, a->in_w)) return r;
        if (int r = nncase_hip_qconv2d(ctx, d + o_xn, w, d + o_yn, a)) return r;
        if (move_y) {
            // (a small result is brought into the caller's order on its way over the bus)
            uint8_t *const s = y_bytes <= kStageMost ? stage_take(ctx, y_bytes) : nullptr;
            if (int r = nncase_hip_nhwc_to_nchw(ctx, d + o_yn, s ? s : d + o_y, es, a->batch, w->out_channels, out_h, out_w)) return r;
            if (s) {
                if (int r = drain_host_calls(ctx)) return r;
                memcpy(y_host, s, y_bytes);
                return 0;
            }
        }
        return copy_to_host(ctx, y_host, d + o_y, y_bytes);
    };
    rc = run();
    if (rc || temporary) (void)hipStreamSynchronize(ctx->stream);
    if (temporary) (void)hipFree(base);
    return rc;
}

} // namespace
} // namespace nnhip

using namespace nnhip;

extern "C" int nncase_hip_host_malloc(nncase_hip_ctx_t *ctx, size_t bytes, void **ptr) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, ptr, -EINVAL, "host_malloc: null out pointer");
    *ptr = nullptr;
    const size_t need = (std::max<size_t>(bytes, 1) + 65535) & ~(size_t)65535;
    HostPool &p = host_pool();
    std::lock_guard<std::mutex> guard(p.mu);
    HostBlock *best = nullptr;
    for (HostBlock &b : p.blocks)
        if (!b.used && b.bytes >= need && b.bytes <= 2 * need && (!best || b.bytes < best->bytes)) best = &b;
    if (!best) {
        if (need > kHostPoolMost) return -ENOMEM; // (not an error to report: the caller takes ordinary memory)
        p.trim(kHostPoolMost - need);
        if (p.total + need > kHostPoolMost) return -ENOMEM;
        HostBlock b{nullptr, need, false};
        NNHIP_HIP(ctx, hipSetDevice(ctx->device));
        NNHIP_HIP(ctx, hipHostMalloc(&b.ptr, need, hipHostMallocDefault));
        p.total += need;
        p.blocks.push_back(b);
        best = &p.blocks.back();
    }
    best->used = true;
    *ptr = best->ptr;
    return 0;
}

extern "C" int nncase_hip_host_free(void *ptr) {
    if (!ptr) return 0;
    HostPool &p = host_pool();
    std::lock_guard<std::mutex> guard(p.mu);
    for (HostBlock &b : p.blocks)
        if (b.ptr == ptr && b.used) {
            b.used = false;
            if (p.contexts == 0) p.trim(0);
            return 0;
        }
    return -EINVAL;
}

extern "C" int nncase_hip_qconv2d_host(nncase_hip_ctx_t *ctx, const nncase_hip_conv2d_desc_t *desc, const uint8_t *x_nchw_host,
                                       const uint8_t *weights_oihw_host, const int32_t *bias_host, void *y_nchw_host,
                                       const nncase_hip_conv2d_args_t *a) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, desc && x_nchw_host && weights_oihw_host && y_nchw_host && a, -EINVAL, "qconv2d_host: null argument");
    NNHIP_REQUIRE(ctx, a->batch > 0 && a->in_h > 0 && a->in_w > 0 && a->stride_h > 0 && a->stride_w > 0 && a->dilation_h > 0 && a->dilation_w > 0,
                  -EINVAL, "qconv2d_host: non-positive shape, stride or dilation");
    NNHIP_REQUIRE(ctx, !a->residual_dev && !a->out_channel_stride && !a->out_channel_offset && !a->dequantize_output, -EINVAL,
                  "qconv2d_host: no residual, output slice or dequantised output");
    nncase_hip_weights w;
    int rc = describe_weights(ctx, &w, desc, "qconv2d_host");
    if (rc) return rc;
    NNHIP_REQUIRE(ctx, w.kind == nncase_hip_weights::kIgemm, -EINVAL, "qconv2d_host: dense and grouped convolutions only");
    const int out_h = windowed_output_size(a->in_h, w.kernel_h, a->stride_h, a->dilation_h, a->pad_h_before, a->pad_h_after);
    const int out_w = windowed_output_size(a->in_w, w.kernel_w, a->stride_w, a->dilation_w, a->pad_w_before, a->pad_w_after);
    NNHIP_REQUIRE(ctx, out_h > 0 && out_w > 0, -NNCASE_HIP_ERR_SHAPE_MISMATCH, "qconv2d_host: window larger than padded input");
    w.pixels_hint = (int64_t)a->batch * out_h * out_w;
    const int64_t taps = (int64_t)w.kernel_h * w.kernel_w;
    return dense_host_call(ctx, &w, x_nchw_host, RawWeights{weights_oihw_host, w.g_ic * taps, taps, (size_t)(w.g_oc * w.g_ic * taps)}, bias_host,
                           y_nchw_host, a, out_h, out_w, true);
}

extern "C" int nncase_hip_qmatmul_host(nncase_hip_ctx_t *ctx, const uint8_t *a_host, const uint8_t *b_host, int32_t k, int32_t n,
                                       nncase_hip_quant_param_t b_qp, const int32_t *bias_host, void *y_host, const nncase_hip_matmul_args_t *m) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, a_host && b_host && y_host && m, -EINVAL, "qmatmul_host: null argument");
    NNHIP_REQUIRE(ctx, m->m > 0 && k > 0 && n > 0, -EINVAL, "qmatmul_host: non-positive dimension");
    nncase_hip_conv2d_desc_t desc{};
    desc.in_channels = k, desc.out_channels = n, desc.kernel_h = desc.kernel_w = desc.groups = 1;
    desc.w_qp = b_qp, desc.expected_pixels = m->m;
    nncase_hip_weights w;
    int rc = describe_weights(ctx, &w, &desc, "qmatmul_host");
    if (rc) return rc;
    nncase_hip_conv2d_args_t a;
    memset(&a, 0, sizeof(a));
    a.batch = 1, a.in_h = m->m, a.in_w = 1;
    a.stride_h = a.stride_w = a.dilation_h = a.dilation_w = 1;
    a.x_qp = m->a_qp, a.y_qp = m->y_qp, a.clamp_min = m->clamp_min, a.clamp_max = m->clamp_max, a.out_dtype = m->out_dtype;
    return dense_host_call(ctx, &w, a_host, RawWeights{b_host, 1, n, 0}, bias_host, y_host, &a, m->m, 1, false);
}
