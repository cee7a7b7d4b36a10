// Quantize / Dequantize streaming kernels and the u8 elementwise glue
// (residual add, global average pool).  All HBM-bound: every thread moves
// pieces of up to 16 bytes, all requested before the first is used, and a
// block owns neighbouring ones.
//
// Arithmetic contracts (each fp32 step is a single IEEE operation; the file
// is compiled with -ffp-contract=off):
//   quantize    q = sat_T((int32) rne(x / scale + bias))          reference/quantize.cpp:36-43
//   dequantize  y = ((float) q - bias) * scale                    reference/dequantize.cpp:36-39
#include "qconv.hpp"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace nnhip {

constexpr int kEwThreads = 256;
constexpr int kEwUnroll = 4;

// V neighbouring elements at any address a T may have; PAST: through the caches without a stay there
template <int BYTES> struct PieceWord;
template <> struct PieceWord<1> { typedef uint8_t type; };
template <> struct PieceWord<2> { typedef uint16_t type __attribute__((aligned(1))); };
template <> struct PieceWord<4> { typedef uint32_t type __attribute__((aligned(1))); };
template <> struct PieceWord<8> { typedef uint32_t type __attribute__((ext_vector_type(2), aligned(1))); };
template <> struct PieceWord<16> { typedef uint32_t type __attribute__((ext_vector_type(4), aligned(1))); };
template <bool PAST, int V, typename T> __device__ __forceinline__ void load_piece(const T *p, T (&v)[V]) {
    typedef typename PieceWord<sizeof(T) * V>::type W;
    const W raw = PAST ? __builtin_nontemporal_load(reinterpret_cast<const W *>(p)) : *reinterpret_cast<const W *>(p);
    __builtin_memcpy(v, &raw, sizeof(v));
}
template <bool PAST, int V, typename T> __device__ __forceinline__ void store_piece(T *p, const T (&v)[V]) {
    typedef typename PieceWord<sizeof(T) * V>::type W;
    W raw;
    __builtin_memcpy(&raw, v, sizeof(v));
    if (PAST) __builtin_nontemporal_store(raw, reinterpret_cast<W *>(p));
    else *reinterpret_cast<W *>(p) = raw;
}
// Elements per load and store: up to 16 bytes of either, but no more than 4 codes of a byte read at once (u8 -> f16 by 8: 1.5 % slower).
template <typename A, typename B> constexpr int piece_elements() { return sizeof(A) == 2 && sizeof(B) <= 2 ? 8 : 4; }

template <typename T> __device__ __forceinline__ float to_f32(T v) { return (float)v; }
template <> __device__ __forceinline__ float to_f32<__half>(__half v) { return __half2float(v); }

// A block owns U * kEwThreads neighbouring pieces, each read and written where it lies; the last block's last elements, fewer than a
// piece, take a thread each.
template <int U, bool PAST, typename A, typename B, class F> __device__ __forceinline__ void for_pieces(const A *in, B *out, size_t count, F &&f) {
    constexpr int V = piece_elements<A, B>();
    const size_t first = (size_t)blockIdx.x * (U * kEwThreads * V), i = first + threadIdx.x * V;
    if (first + U * kEwThreads * V <= count) {
        A v[U][V];
#pragma unroll
        for (int u = 0; u < U; u++) load_piece<PAST, V>(in + i + u * kEwThreads * V, v[u]);
        __builtin_amdgcn_sched_barrier(0); // (every request before the first piece is waited for)
#pragma unroll
        for (int u = 0; u < U; u++) {
            B w[V];
            f(v[u], w);
            store_piece<PAST, V>(out + i + u * kEwThreads * V, w);
        }
        return;
    }
    for (size_t k = i; k + V <= count; k += kEwThreads * V) {
        A v[V];
        B w[V];
        load_piece<PAST, V>(in + k, v);
        f(v, w);
        store_piece<PAST, V>(out + k, w);
    }
    const size_t k = count / V * V + threadIdx.x;
    if (k < count) {
        const A v[1] = {in[k]};
        B w[1];
        f(v, w);
        out[k] = w[0];
    }
}

// What quantize divides by.  QUICK: x / scale by the reciprocal, 3 instructions instead of some 11, which bound the kernel (25 M
// elements f16 -> u8: 14.9 -> 12.0 us, 6.3 TB/s; 3.3 M f32 -> u8 4.5 -> 3.3).  q0 = x * r is within 1.5 ulp of the quotient and
// q0 + (x - scale * q0) * r, rounded once, is the quotient's nearest float: Markstein's theorem of the quotient corrected by a correctly
// rounded reciprocal, which asks for a q0 within one ulp; the rest was held by enumeration of every pair of mantissas whose quotient
// lies near enough to the middle of two floats.  A q0 far past every code is cut to +-2^40, so that an infinity leaves no difference of two infinities behind; a NaN stays
// one up to the conversion, which makes the lowest code of it like the general form.
struct Divisor {
    float scale, reciprocal, bias;
};
constexpr float kReach = 0x1p40f;
// scales from 2^-60 to 2^60: no quotient that a code depends on, nor its residual, leaves the range of normal floats
inline bool quick_divisor(float scale) { return std::fabs(scale) >= 0x1p-60f && std::fabs(scale) <= 0x1p60f; }

template <typename TQ, int V, typename TIn> __device__ __forceinline__ void quantize_quick(const TIn (&x)[V], TQ (&q)[V], const Divisor &d) {
    float v[V];
#pragma unroll
    for (int e = 0; e < V; e++) {
        const float f = to_f32(x[e]), q0 = __builtin_amdgcn_fmed3f(f * d.reciprocal, -kReach, kReach);
        v[e] = __builtin_fmaf(__builtin_fmaf(-d.scale, q0, f), d.reciprocal, q0) + d.bias;
    }
    if constexpr (std::is_same_v<TQ, uint8_t> && V % 4 == 0) {
        uint32_t w[V / 4];
#pragma unroll
        for (int e = 0; e < V; e++) w[e / 4] = __builtin_amdgcn_cvt_pk_u8_f32(v[e], e % 4, e % 4 ? w[e / 4] : 0u);
        __builtin_memcpy(q, w, sizeof(q));
    } else {
#pragma unroll
        for (int e = 0; e < V; e++) q[e] = (TQ)(int32_t)rintf(__builtin_amdgcn_fmed3f(v[e], QLimits<TQ>::lo, QLimits<TQ>::hi));
    }
}

template <typename TIn, typename TQ, int U, bool PAST, bool QUICK>
__global__ __launch_bounds__(kEwThreads) void quantize_kernel(const TIn *__restrict__ in, TQ *__restrict__ out, size_t count, const Divisor d) {
    for_pieces<U, PAST>(in, out, count, [&](const auto &x, auto &q) {
        constexpr int V = sizeof(x) / sizeof(TIn);
        if constexpr (QUICK) {
            quantize_quick<TQ, V>(x, q, d);
        } else {
#pragma unroll
            for (int e = 0; e < V; e++) q[e] = quantize_one<TQ>(to_f32(x[e]), d.scale, d.bias);
        }
    });
}

template <typename TOut> __device__ __forceinline__ TOut from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
// (the fp32 value is hidden from the optimiser first: where it sees the multiply that produced it, it may merge
// multiply and conversion into one mixed-precision instruction that rounds once, and does so in some copies of a
// loop body and not in others; the result is defined as the fp16 nearest to the rounded fp32 product)
template <> __device__ __forceinline__ __half from_f32<__half>(float v) {
    asm volatile("" : "+v"(v));
    return __float2half_rn(v);
}

template <typename TQ, typename TOut, int U, bool PAST>
__global__ __launch_bounds__(kEwThreads) void dequantize_kernel(const TQ *__restrict__ in, TOut *__restrict__ out, size_t count, float scale, float bias) {
    for_pieces<U, PAST>(in, out, count, [&](const auto &q, auto &y) {
#pragma unroll
        for (int e = 0; e < (int)(sizeof(q) / sizeof(TQ)); e++) y[e] = from_f32<TOut>(((float)q[e] - bias) * scale);
    });
}

// Strided forms: element `index` of a tensor of `rank` dimensions is read at sum(index[d] * in_strides[d]) and
// written at sum(index[d] * out_strides[d]) (strides in elements), as the reference's kernels address their
// operands (apply(in_shape, ...) with offset(strides, index), reference/quantize.cpp:36-47, dequantize.cpp:36-44).
// One element per thread and trip, innermost dimension fastest, so dense inner rows still coalesce.
constexpr int kMaxStridedRank = 6;
struct StridedArgs {
    int rank;
    uint32_t count;
    FastDiv dim[kMaxStridedRank];          // innermost first
    uint32_t in_stride[kMaxStridedRank];   // innermost first
    uint32_t out_stride[kMaxStridedRank];
};

__device__ __forceinline__ void strided_offsets(const StridedArgs &a, uint32_t i, uint32_t *in_off, uint32_t *out_off) {
    uint32_t io = 0, oo = 0;
#pragma unroll
    for (int d = 0; d < kMaxStridedRank; d++) {
        if (d < a.rank) {
            const uint32_t q = fastdiv(i, a.dim[d]);
            const uint32_t r = i - q * a.dim[d].div;
            io += r * a.in_stride[d];
            oo += r * a.out_stride[d];
            i = q;
        }
    }
    *in_off = io, *out_off = oo;
}

template <typename TIn, typename TQ>
__global__ __launch_bounds__(kEwThreads) void quantize_strided_kernel(const TIn *__restrict__ in, TQ *__restrict__ out, const StridedArgs a,
                                                                      float scale, float bias) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.count; i += gridDim.x * blockDim.x) {
        uint32_t io, oo;
        strided_offsets(a, i, &io, &oo);
        out[oo] = quantize_one<TQ>(to_f32(in[io]), scale, bias);
    }
}

template <typename TQ, typename TOut>
__global__ __launch_bounds__(kEwThreads) void dequantize_strided_kernel(const TQ *__restrict__ in, TOut *__restrict__ out, const StridedArgs a,
                                                                        float scale, float bias) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < a.count; i += gridDim.x * blockDim.x) {
        uint32_t io, oo;
        strided_offsets(a, i, &io, &oo);
        out[oo] = from_f32<TOut>(((float)in[io] - bias) * scale);
    }
}

// out = Q(clamp(DQ(a) + DQ(b))) on bytes; the clamp and the u8 saturation are folded into
// one clamp on the requantised value, the division is the exact FMA form (see qconv.hpp).
__global__ __launch_bounds__(kEwThreads) void qadd_kernel(const uint8_t *__restrict__ a, const uint8_t *__restrict__ b,
                                                          uint8_t *__restrict__ out, size_t count, float za, float sa,
                                                          float zb, float sb, const Epilogue ep, int vec_ok) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nthreads = (size_t)gridDim.x * blockDim.x;
    // the requantised sum before rounding to a byte
    auto value = [&](uint32_t qa, uint32_t qb) -> float {
        const float fa = ((float)qa - za) * sa;
        const float fb = ((float)qb - zb) * sb;
        return __builtin_amdgcn_fmed3f(div_rn(fa + fb, ep.sy, ep.rsy) + ep.zy, ep.qlo, ep.qhi);
    };
    auto one = [&](uint32_t qa, uint32_t qb) -> uint32_t { return __builtin_amdgcn_cvt_pk_u8_f32(value(qa, qb), 0, 0u); };
    // 16 bytes per thread per step
    const size_t nvec = vec_ok ? count / 16 : 0;
    for (size_t i = tid; i < nvec; i += nthreads) {
        const uint4 va = *reinterpret_cast<const uint4 *>(a + i * 16);
        const uint4 vb = *reinterpret_cast<const uint4 *>(b + i * 16);
        const uint32_t wa[4] = {va.x, va.y, va.z, va.w}, wb[4] = {vb.x, vb.y, vb.z, vb.w};
        uint32_t wo[4];
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) w = __builtin_amdgcn_cvt_pk_u8_f32(value((wa[d] >> (8 * e)) & 0xffu, (wb[d] >> (8 * e)) & 0xffu), e, w);
            wo[d] = w;
        }
        *reinterpret_cast<uint4 *>(out + i * 16) = uint4{wo[0], wo[1], wo[2], wo[3]};
    }
    for (size_t j = nvec * 16 + tid; j < count; j += nthreads) out[j] = (uint8_t)one(a[j], b[j]);
}

// Global average pool over NHWC u8.  One thread per (image, channel): the sum
// runs over the pixels in (y, x) order with a float accumulator, exactly the
// order of the reference's window loop, so the result is bit-identical.
// Adjacent threads read adjacent channels, so every load is coalesced.
__global__ __launch_bounds__(kEwThreads) void qglobal_avgpool_kernel(const uint8_t *__restrict__ x,
                                                                     uint8_t *__restrict__ out, int batch, int hw,
                                                                     int channels, float zx, float sx, float zy,
                                                                     float sy) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= batch * channels) return;
    const int n = idx / channels, c = idx - n * channels;
    const uint8_t *p = x + (size_t)n * hw * channels + c;
    float value = 0.f;
    for (int i = 0; i < hw; i++) value = value + ((float)p[(size_t)i * channels] - zx) * sx;
    const float mean = value / (float)hw;
    float t = mean / sy + zy;
    t = fminf(fmaxf(t, 0.f), 255.f);
    out[idx] = (uint8_t)(int32_t)rintf(t);
}

// The same for 4 adjacent channels per thread (dword loads), the loads of 64 pixels (a whole 7x7 map) issued before
// their values are added: with one or two waves per SIMD the kernel is a chain of memory round trips, and this
// leaves one per 64 pixels.  Each channel's additions keep their order.
__global__ __launch_bounds__(kEwThreads) void qglobal_avgpool4_kernel(const uint8_t *__restrict__ x, uint8_t *__restrict__ out,
                                                                      int batch, int hw, int channels, float zx, float sx,
                                                                      float zy, float sy) {
    const int cq = channels >> 2;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= batch * cq) return;
    const int n = idx / cq, c = (idx - n * cq) * 4;
    const uint32_t q = global_avgpool4(x + (size_t)n * hw * channels + c, hw, channels, zx, sx, zy, sy);
    *reinterpret_cast<uint32_t *>(out + (size_t)n * channels + c) = q;
}

inline int ew_grid(const nncase_hip_ctx *ctx, size_t work_items) {
    size_t blocks = (work_items + kEwThreads - 1) / kEwThreads;
    const size_t cap = (size_t)ctx->compute_units * 16; // 16 blocks of 4 waves per CU
    if (blocks > cap) blocks = cap;
    if (blocks == 0) blocks = 1;
    return (int)blocks;
}

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Quantize / dequantize: a block per U * kEwThreads neighbouring pieces, however many that makes.  Blocks that
// run at the same time then read and write neighbouring addresses (measured on 100 M elements against a capped grid that
// strides over the tensor: quantize f32 -> u8 114 -> 96 us, dequantize i32 -> f32 202 -> 136 us).  Four pieces a thread where that leaves
// two blocks per compute unit (one of bytes), else one (0.5 M f32 -> u8 3.3 -> 2.5 us; 1.04 M u8 -> f16 2.6 with four, 2.8 with one).
template <typename A, typename B> inline unsigned piece_blocks(size_t count, int unroll) {
    const size_t per_block = (size_t)unroll * kEwThreads * piece_elements<A, B>();
    return (unsigned)((count + per_block - 1) / per_block);
}
// Both sides' bytes from which on next to nothing of them is in a cache when the next operator comes (the memory side's holds 256 MiB;
// us through the caches / past them: f32 -> u8 of 275 MB 42.8 / 46.0, of 300 MB 48.7 / 48.3, of 375 MB 70.6 / 62.4, i32 -> f32 of 428 MB
// 76.7 / 68.6)
constexpr size_t kPastCaches = 300000000;
// go(pieces per thread, past the caches)
template <typename A, typename B, class F> void with_piece_form(const nncase_hip_ctx *ctx, size_t count, F &&go) {
    const bool several = count >= (size_t)(sizeof(A) == 1 ? 1 : 2) * ctx->compute_units * (kEwUnroll * kEwThreads * piece_elements<A, B>());
    if (!several) go(std::integral_constant<int, 1>(), std::false_type());
    else if (count * (sizeof(A) + sizeof(B)) < kPastCaches) go(std::integral_constant<int, kEwUnroll>(), std::false_type());
    else go(std::integral_constant<int, kEwUnroll>(), std::true_type());
}

template <typename TIn, typename TQ>
int launch_quantize(nncase_hip_ctx *ctx, const void *in, void *out, size_t count, float scale, float bias) {
    const Divisor d{scale, 1.f / scale, bias};
    with_piece_form<TIn, TQ>(ctx, count, [&](auto u, auto past) {
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(piece_blocks<TIn, TQ>(count, u)), dim3(kEwThreads), 0, ctx->stream, (const TIn *)in, (TQ *)out, count, d);
        };
        if (quick_divisor(scale)) go(quantize_kernel<TIn, TQ, u, past, true>);
        else go(quantize_kernel<TIn, TQ, u, past, false>);
    });
    NNHIP_LAUNCH_CHECK(ctx, "quantize_kernel");
    return 0;
}

template <typename TQ, typename TOut>
int launch_dequantize(nncase_hip_ctx *ctx, const void *in, void *out, size_t count, float scale, float bias) {
    with_piece_form<TQ, TOut>(ctx, count, [&](auto u, auto past) {
        hipLaunchKernelGGL((dequantize_kernel<TQ, TOut, u, past>), dim3(piece_blocks<TQ, TOut>(count, u)), dim3(kEwThreads), 0, ctx->stream,
                           (const TQ *)in, (TOut *)out, count, scale, bias);
    });
    NNHIP_LAUNCH_CHECK(ctx, "dequantize_kernel");
    return 0;
}

// Validates a strided operand pair and fills the kernel's arguments.  *dense is set when both sides are the
// plain row-major layout of the shape (the caller then takes the vector kernels).
int make_strided(nncase_hip_ctx *ctx, const char *what, int32_t rank, const int64_t *shape, const int64_t *in_strides,
                 const int64_t *out_strides, StridedArgs *a, bool *dense) {
    NNHIP_REQUIRE(ctx, rank >= 1 && rank <= kMaxStridedRank, -EINVAL, "%s: rank %d (1..%d are supported)", what, rank, kMaxStridedRank);
    NNHIP_REQUIRE(ctx, shape && in_strides && out_strides, -EINVAL, "%s: null shape or strides", what);
    memset(a, 0, sizeof(*a));
    a->rank = rank;
    int64_t count = 1, in_extent = 0, out_extent = 0, row_major = 1;
    *dense = true;
    for (int d = rank - 1; d >= 0; d--) { // innermost first
        NNHIP_REQUIRE(ctx, shape[d] >= 0 && in_strides[d] >= 0 && out_strides[d] >= 0, -EINVAL, "%s: negative extent or stride", what);
        NNHIP_REQUIRE(ctx, shape[d] < ((int64_t)1 << 31) && in_strides[d] < ((int64_t)1 << 31) && out_strides[d] < ((int64_t)1 << 31),
                      -EINVAL, "%s: extent or stride of 2^31 or more", what);
        count *= shape[d];
        NNHIP_REQUIRE(ctx, count < ((int64_t)1 << 31), -EINVAL, "%s: 2^31 elements or more", what);
        if (shape[d] > 0) {
            in_extent += (shape[d] - 1) * in_strides[d];
            out_extent += (shape[d] - 1) * out_strides[d];
        }
        NNHIP_REQUIRE(ctx, in_extent < ((int64_t)1 << 31) && out_extent < ((int64_t)1 << 31), -EINVAL, "%s: operand spans 2^31 elements or more", what);
        const int k = rank - 1 - d;
        a->dim[k] = make_fastdiv((uint32_t)std::max<int64_t>(shape[d], 1));
        a->in_stride[k] = (uint32_t)in_strides[d];
        a->out_stride[k] = (uint32_t)out_strides[d];
        if (shape[d] != 1 && (in_strides[d] != row_major || out_strides[d] != row_major)) *dense = false;
        row_major *= shape[d];
    }
    a->count = (uint32_t)count;
    return 0;
}

} // namespace nnhip

using namespace nnhip;

extern "C" int nncase_hip_quantize(nncase_hip_ctx_t *ctx, const void *in_dev, int in_dtype, void *out_dev,
                                   int out_dtype, size_t count, nncase_hip_quant_param_t qp) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, (in_dev && out_dev) || count == 0, -EINVAL, "quantize: null buffer");
    NNHIP_REQUIRE(ctx, qp.scale != 0.f, -EINVAL, "quantize: scale is zero");
    if (count == 0) return 0;
    const float bias = (float)qp.zero_point;
#define NNHIP_Q_CASE(IN_DT, TIn, OUT_DT, TQ)                                                                           \
    if (in_dtype == IN_DT && out_dtype == OUT_DT)                                                                      \
    return launch_quantize<TIn, TQ>(ctx, in_dev, out_dev, count, qp.scale, bias)
    NNHIP_Q_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_U8, uint8_t);
    NNHIP_Q_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_I8, int8_t);
    NNHIP_Q_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_I16, int16_t);
    NNHIP_Q_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_U8, uint8_t);
    NNHIP_Q_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_I8, int8_t);
    NNHIP_Q_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_I16, int16_t);
#undef NNHIP_Q_CASE
    return fail(ctx, -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "quantize: unsupported types in=0x%x out=0x%x", in_dtype,
                out_dtype);
}

extern "C" int nncase_hip_dequantize(nncase_hip_ctx_t *ctx, const void *in_dev, int in_dtype, void *out_dev,
                                     int out_dtype, size_t count, nncase_hip_quant_param_t qp) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, (in_dev && out_dev) || count == 0, -EINVAL, "dequantize: null buffer");
    if (count == 0) return 0;
    const float bias = (float)qp.zero_point;
#define NNHIP_DQ_CASE(IN_DT, TQ, OUT_DT, TOut)                                                                         \
    if (in_dtype == IN_DT && out_dtype == OUT_DT)                                                                      \
    return launch_dequantize<TQ, TOut>(ctx, in_dev, out_dev, count, qp.scale, bias)
    NNHIP_DQ_CASE(NNCASE_HIP_DT_U8, uint8_t, NNCASE_HIP_DT_F32, float);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I8, int8_t, NNCASE_HIP_DT_F32, float);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I16, int16_t, NNCASE_HIP_DT_F32, float);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I32, int32_t, NNCASE_HIP_DT_F32, float);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_U8, uint8_t, NNCASE_HIP_DT_F16, __half);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I8, int8_t, NNCASE_HIP_DT_F16, __half);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I16, int16_t, NNCASE_HIP_DT_F16, __half);
    NNHIP_DQ_CASE(NNCASE_HIP_DT_I32, int32_t, NNCASE_HIP_DT_F16, __half);
#undef NNHIP_DQ_CASE
    return fail(ctx, -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "dequantize: unsupported types in=0x%x out=0x%x", in_dtype,
                out_dtype);
}

extern "C" int nncase_hip_quantize_strided(nncase_hip_ctx_t *ctx, const void *in_dev, int in_dtype, void *out_dev, int out_dtype,
                                           int32_t rank, const int64_t *shape, const int64_t *in_strides, const int64_t *out_strides,
                                           nncase_hip_quant_param_t qp) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, qp.scale != 0.f, -EINVAL, "quantize: scale is zero");
    StridedArgs a;
    bool dense;
    const int rc = make_strided(ctx, "quantize", rank, shape, in_strides, out_strides, &a, &dense);
    if (rc) return rc;
    if (a.count == 0) return 0;
    NNHIP_REQUIRE(ctx, in_dev && out_dev, -EINVAL, "quantize: null buffer");
    if (dense) return nncase_hip_quantize(ctx, in_dev, in_dtype, out_dev, out_dtype, a.count, qp);
    const float bias = (float)qp.zero_point;
    const int grid = ew_grid(ctx, a.count);
#define NNHIP_QS_CASE(IN_DT, TIn, OUT_DT, TQ)                                                                          \
    if (in_dtype == IN_DT && out_dtype == OUT_DT) {                                                                    \
        hipLaunchKernelGGL((quantize_strided_kernel<TIn, TQ>), dim3(grid), dim3(kEwThreads), 0, ctx->stream,           \
                           (const TIn *)in_dev, (TQ *)out_dev, a, qp.scale, bias);                                     \
        NNHIP_LAUNCH_CHECK(ctx, "quantize_strided_kernel");                                                            \
        return 0;                                                                                                      \
    }
    NNHIP_QS_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_U8, uint8_t)
    NNHIP_QS_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_I8, int8_t)
    NNHIP_QS_CASE(NNCASE_HIP_DT_F32, float, NNCASE_HIP_DT_I16, int16_t)
    NNHIP_QS_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_U8, uint8_t)
    NNHIP_QS_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_I8, int8_t)
    NNHIP_QS_CASE(NNCASE_HIP_DT_F16, __half, NNCASE_HIP_DT_I16, int16_t)
#undef NNHIP_QS_CASE
    return fail(ctx, -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "quantize: unsupported types in=0x%x out=0x%x", in_dtype, out_dtype);
}

extern "C" int nncase_hip_dequantize_strided(nncase_hip_ctx_t *ctx, const void *in_dev, int in_dtype, void *out_dev, int out_dtype,
                                             int32_t rank, const int64_t *shape, const int64_t *in_strides, const int64_t *out_strides,
                                             nncase_hip_quant_param_t qp) {
    NNHIP_CHECK_CTX(ctx);
    StridedArgs a;
    bool dense;
    const int rc = make_strided(ctx, "dequantize", rank, shape, in_strides, out_strides, &a, &dense);
    if (rc) return rc;
    if (a.count == 0) return 0;
    NNHIP_REQUIRE(ctx, in_dev && out_dev, -EINVAL, "dequantize: null buffer");
    if (dense) return nncase_hip_dequantize(ctx, in_dev, in_dtype, out_dev, out_dtype, a.count, qp);
    const float bias = (float)qp.zero_point;
    const int grid = ew_grid(ctx, a.count);
#define NNHIP_DQS_CASE(IN_DT, TQ, OUT_DT, TOut)                                                                        \
    if (in_dtype == IN_DT && out_dtype == OUT_DT) {                                                                    \
        hipLaunchKernelGGL((dequantize_strided_kernel<TQ, TOut>), dim3(grid), dim3(kEwThreads), 0, ctx->stream,        \
                           (const TQ *)in_dev, (TOut *)out_dev, a, qp.scale, bias);                                    \
        NNHIP_LAUNCH_CHECK(ctx, "dequantize_strided_kernel");                                                          \
        return 0;                                                                                                      \
    }
    NNHIP_DQS_CASE(NNCASE_HIP_DT_U8, uint8_t, NNCASE_HIP_DT_F32, float)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I8, int8_t, NNCASE_HIP_DT_F32, float)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I16, int16_t, NNCASE_HIP_DT_F32, float)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I32, int32_t, NNCASE_HIP_DT_F32, float)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_U8, uint8_t, NNCASE_HIP_DT_F16, __half)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I8, int8_t, NNCASE_HIP_DT_F16, __half)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I16, int16_t, NNCASE_HIP_DT_F16, __half)
    NNHIP_DQS_CASE(NNCASE_HIP_DT_I32, int32_t, NNCASE_HIP_DT_F16, __half)
#undef NNHIP_DQS_CASE
    return fail(ctx, -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "dequantize: unsupported types in=0x%x out=0x%x", in_dtype, out_dtype);
}

extern "C" int nncase_hip_qadd(nncase_hip_ctx_t *ctx, const uint8_t *a_dev, nncase_hip_quant_param_t a_qp,
                               const uint8_t *b_dev, nncase_hip_quant_param_t b_qp, uint8_t *out_dev,
                               nncase_hip_quant_param_t y_qp, float clamp_min, float clamp_max, size_t count) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, (a_dev && b_dev && out_dev) || count == 0, -EINVAL, "qadd: null buffer");
    if (count == 0) return 0;
    NNHIP_REQUIRE(ctx, std::isfinite(a_qp.scale) && std::isfinite(b_qp.scale) && std::fabs(a_qp.scale) <= 0x1p20f &&
                           std::fabs(b_qp.scale) <= 0x1p20f,
                  -ERANGE, "qadd: input scale outside the supported range");
    Epilogue ep;
    // the sum's magnitude is bounded by 255 * (|sa| + |sb|); mult is unused here
    const int rc = make_epilogue(ctx, &ep, 1.f, 1.f, y_qp, clamp_min, clamp_max, NNCASE_HIP_DT_U8, "qadd");
    if (rc) return rc;
    const int vec_ok = aligned16(a_dev) && aligned16(b_dev) && aligned16(out_dev);
    const int grid = ew_grid(ctx, (count + 15) / 16);
    hipLaunchKernelGGL(qadd_kernel, dim3(grid), dim3(kEwThreads), 0, ctx->stream, a_dev, b_dev, out_dev, count,
                       (float)a_qp.zero_point, a_qp.scale, (float)b_qp.zero_point, b_qp.scale, ep, vec_ok);
    NNHIP_LAUNCH_CHECK(ctx, "qadd_kernel");
    return 0;
}

extern "C" int nncase_hip_qglobal_avgpool(nncase_hip_ctx_t *ctx, const uint8_t *x_dev, uint8_t *out_dev, int32_t batch,
                                          int32_t h, int32_t w, int32_t channels, nncase_hip_quant_param_t x_qp,
                                          nncase_hip_quant_param_t y_qp) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, x_dev && out_dev, -EINVAL, "qglobal_avgpool: null buffer");
    NNHIP_REQUIRE(ctx, batch > 0 && h > 0 && w > 0 && channels > 0, -EINVAL, "qglobal_avgpool: bad shape");
    NNHIP_REQUIRE(ctx, (int64_t)batch * channels < (int64_t)1 << 31, -EINVAL, "qglobal_avgpool: too large");
    NNHIP_REQUIRE(ctx, y_qp.scale != 0.f, -EINVAL, "qglobal_avgpool: output scale is zero");
    if (channels % 4 == 0 && (reinterpret_cast<uintptr_t>(x_dev) & 3u) == 0 && (reinterpret_cast<uintptr_t>(out_dev) & 3u) == 0) {
        const int total4 = batch * (channels / 4);
        hipLaunchKernelGGL(qglobal_avgpool4_kernel, dim3((total4 + kEwThreads - 1) / kEwThreads), dim3(kEwThreads), 0, ctx->stream,
                           x_dev, out_dev, batch, h * w, channels, (float)x_qp.zero_point, x_qp.scale, (float)y_qp.zero_point,
                           y_qp.scale);
        NNHIP_LAUNCH_CHECK(ctx, "qglobal_avgpool4_kernel");
        return 0;
    }
    const int total = batch * channels;
    hipLaunchKernelGGL(qglobal_avgpool_kernel, dim3((total + kEwThreads - 1) / kEwThreads), dim3(kEwThreads), 0,
                       ctx->stream, x_dev, out_dev, batch, h * w, channels, (float)x_qp.zero_point, x_qp.scale,
                       (float)y_qp.zero_point, y_qp.scale);
    NNHIP_LAUNCH_CHECK(ctx, "qglobal_avgpool_kernel");
    return 0;
}
