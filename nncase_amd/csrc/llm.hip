// The rest of an LLM decode step around paged attention (fp16 activations, W8A16 weights):
// RMSNorm, the small-M weight-streaming GEMM, rotary embedding + KV append into the block-paged
// cache, arg-max, embedding gather and the per-step advance of the context lengths.
//
// A decode step multiplies a handful of token rows (M = batch, <= 64) with every weight matrix, so
// each int8 weight byte is read from HBM exactly once and the step is bound by that stream
// (~0.5 GB for a Qwen2-0.5B-shaped model).  The GEMM is organised around it: weights are
// pre-packed so that a wave's load of one k-step is a contiguous 1 KiB fragment (16 bytes per
// lane), converted int8 -> fp16 in registers (exactly: (w + 128) | 0x6400 is the fp16 1024 + w + 128)
// and fed to v_mfma_f32_16x16x32_f16 as the A operand (16 output channels), the token rows being
// the B operand; a lane ends up with 4 consecutive output channels of one token.  The four waves
// of a block split the reduction and combine through LDS.  Per-output-channel scales, bias, the
// residual add and the SwiGLU gate are applied in the epilogue.
#include "common.hpp"
#include "w8a16_rules.hpp"

#include <hip/hip_fp16.h>

#include <cmath>
#include <type_traits>
#include <new>
#include <vector>

namespace nnhip {

typedef _Float16 h16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef uint32_t lu32x4 __attribute__((ext_vector_type(4)));

constexpr int kLlmThreads = 256;
constexpr int kMaxRows = 64; // token rows per GEMM call (4 MFMA column tiles)

} // namespace nnhip

// Pre-packed W8A16 matrix: out[m, n] = scale[n] * sum_k a[m, k] * w[n, k] (+ bias[n]).
struct nncase_hip_w8a16 {
    int k = 0, n = 0;      // reduction length (multiple of 64), output channels (multiple of 16)
    int ntiles = 0, ksteps = 0;
    void *d_packed = nullptr; // [ntiles][ksteps][64 lanes][16 B]: lane (i = l % 16, kg = l / 16) holds
                              // w[tile * 16 + i][ks * 64 + kg * 16 .. + 15], each as the unsigned byte w + 128
    float *d_scale = nullptr; // [n]
    float *d_bias = nullptr;  // [n] or null
};

namespace nnhip {

struct RopeArgs {
    const __half *qkv; // [batch][(hq + 2 * hkv) * d]: q heads, then k heads, then v heads
    __half *q_out;     // [batch][hq][d]
    __half *k_cache;   // [blocks][hkv][block][d]
    __half *v_cache;   // [blocks][hkv][d][block]
    const int32_t *block_table, *ctx_lens; // the new token of sequence b goes to position ctx_lens[b]
    int batch, hq, hkv, d, block_size, max_blocks, num_blocks;
    float theta;
};

struct GemmArgs {
    const uint16_t *a; // [m][k] fp16
    const lu32x4 *w;
    const float *scale, *bias;
    const uint16_t *residual; // [m][n_out] fp16 or null
    void *out;                // [m][n_out] fp16 or fp32
    int m, k, n_out, ksteps, out_f32;
    int up_tile_offset; // SwiGLU: tile t of the gate pairs with tile t + up_tile_offset of the up projection
    // RMS normalisation of the token rows in front of the product (null: none): the block computes every row's
    // 1 / sqrt(mean(x^2) + eps) the way rmsnorm_f16_kernel does, and a token slice becomes
    // fp16(x * r * weight) as it is loaded, so the result is what the two kernels give one after the other
    const uint16_t *ln_w; // [k] fp16
    float ln_eps;
    // ROPE kernels: the product is a q / k / v projection whose rows do not go to `out` but, rotated, to the query buffer
    // and the paged cache (rope.qkv unused)
    RopeArgs rope;
};

// 1 / sqrt(mean(x^2) + eps) of a row, the way every kernel here forms it.  A lane owns the 8 consecutive elements
// 8 * lane .. 8 * lane + 7 of every 512-element piece of the row (one 16-byte load per piece); it adds their squares
// in index order, piece after piece, and a butterfly adds the 64 lanes.  The order is part of the definition: the
// product kernel that normalises its own rows must arrive at the same bits as rmsnorm_f16_kernel.
//
// Squares and scalings are one instruction per element: v_fma_mix_f32 takes halves where they lie in a dword (a conversion and a
// multiplication or addition otherwise, each rounding where this one does: the square of a half is exact in fp32, and a sum with -0
// is the other summand).
__device__ __forceinline__ void add_squares8(const lu32x4 &v, float &ss) {
    const h16x8 h = __builtin_bit_cast(h16x8, v);
#pragma unroll
    for (int e = 0; e < 8; e++) ss = __builtin_fmaf((float)h[e], (float)h[e], ss);
}
// fp16(x * r * w) of eight elements, both products and the conversion rounding by themselves (see rmsnorm_f16_kernel): the second product
// passes an assembly statement, or the compiler would make one rounding of it and the conversion.
__device__ __forceinline__ lu32x4 normalise8(const lu32x4 &x, float r, const lu32x4 &w) {
    typedef float f32x2v __attribute__((ext_vector_type(2)));
    const h16x8 xh = __builtin_bit_cast(h16x8, x), wh = __builtin_bit_cast(h16x8, w);
    float zero = -0.0f;
    asm("" : "+s"(zero)); // (or the compiler would make a multiplication of it, behind a conversion)
    lu32x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        f32x2v p;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            float v = __builtin_fmaf(__builtin_fmaf((float)xh[2 * e + q], r, zero), (float)wh[2 * e + q], zero);
            asm("" : "+v"(v));
            p[q] = v;
        }
        y[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(p, h16x2));
    }
    return y;
}
// The sum over the wave's lanes, in every lane, bit for bit the butterfly `for (o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o)`
// (a sum of two does not mind their order) on row swaps and DPP moves: a shuffle goes through the LDS crossbar and back, six of
// them in a row a quarter of a microsecond in front of every product that normalises its rows.
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float v) {
    // (the builtin of the swaps takes two equal operands for two equal results; the wait states are those it would insert)
    float other = v;
    asm("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(v), "+v"(other)); // lanes 0..31 twice, lanes 32..63 twice
    v += other;
    other = v;
    asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(v), "+v"(other)); // the even rows of 16 twice, the odd ones twice
    v += other;
    v += dpp_move<0x128>(v); // row_ror:8
    v += dpp_move<0x124>(v); // row_ror:4 (the lanes of a row repeat with period 8 by now)
    v += dpp_move<0x4e>(v);  // quad_perm 2 3 0 1
    return v + dpp_move<0xb1>(v); // quad_perm 1 0 3 2
}
__device__ __forceinline__ float rstd_from_sum(float ss, int hidden, float eps) {
    return 1.0f / sqrtf(wave_sum(ss) / (float)hidden + eps);
}
// R rows at once (row r0 + i * stride for i < R, those below `rows`): the loads of one piece of all of them are in
// flight together.  hidden is a multiple of 8 and the rows are 16-byte aligned.
template <int R>
__device__ __forceinline__ void rms_rstd_rows(const __half *x, int hidden, int rows, int r0, int stride, int lane, float eps,
                                              float (&out)[R]) {
    float ss[R];
#pragma unroll
    for (int i = 0; i < R; i++) ss[i] = 0.f;
    for (int e0 = lane * 8; e0 < ((hidden + 511) & ~511); e0 += 512) {
        lu32x4 v[R];
#pragma unroll
        for (int i = 0; i < R; i++) {
            const int r = r0 + i * stride;
            v[i] = lu32x4{0, 0, 0, 0}; // (+0 squares leave a sum as it is)
            if (r < rows && e0 < hidden) v[i] = *reinterpret_cast<const lu32x4 *>(x + (size_t)r * hidden + e0);
        }
#pragma unroll
        for (int i = 0; i < R; i++) add_squares8(v[i], ss[i]);
    }
#pragma unroll
    for (int i = 0; i < R; i++) out[i] = rstd_from_sum(ss[i], hidden, eps);
}
// any row length and alignment: the same order with one element per load
__device__ __forceinline__ float rms_rstd_scalar(const __half *xr, int hidden, float eps, int lane) {
    float ss = 0.f;
    for (int e0 = lane * 8; e0 < ((hidden + 511) & ~511); e0 += 512)
        for (int e = 0; e < 8; e++)
            if (e0 + e < hidden) {
                const float f = __half2float(xr[e0 + e]);
                ss += f * f;
            }
    return rstd_from_sum(ss, hidden, eps);
}

// One rotate-half pair of the new token of sequence b: elements i and i + d/2 of head h (q heads, then k heads, then
// v heads), given as the fp16 values the projection stores.  q goes rotated to the query buffer, k rotated and v as it
// is to position ctx_lens[b] of the paged cache.  The one definition of that arithmetic: the rope kernel and the
// projection that rotates in its own epilogue both use it.
//
// In two halves: where the pair goes and its angle (two dependent loads, a power, a sine and a cosine) do not depend on
// the values, so a projection has them ready before its products are.
struct RopePair {
    int h, i, pos, in_block;
    int pb; // the physical block, not used before the pair is stored: its load may still be under way
    bool fits;
    float c, s;
};
__device__ __forceinline__ RopePair rope_pair(const RopeArgs &a, int b, int h, int i, int pos /* ctx_lens[b] */) {
    RopePair r;
    r.h = h, r.i = i, r.pos = pos;
    const int lb = pos / a.block_size;
    r.in_block = pos - lb * a.block_size;
    r.fits = pos >= 0 && lb < a.max_blocks; // a negative length appends nothing (it would index before the block)
    r.pb = a.block_table[(size_t)b * a.max_blocks + (r.fits ? lb : 0)];
    const float inv = powf(a.theta, -2.0f * (float)i / (float)a.d);
    const float ang = (float)pos * inv;
    r.c = cosf(ang), r.s = sinf(ang);
    return r;
}
__device__ __forceinline__ void rope_store(const RopeArgs &a, int b, const RopePair &r, float x0, float x1) {
    const int half = a.d / 2;
    const int pb = min(max(r.pb, 0), a.num_blocks - 1);
    if (r.h < a.hq + a.hkv) {
        const __half y0 = __float2half_rn(x0 * r.c - x1 * r.s), y1 = __float2half_rn(x1 * r.c + x0 * r.s);
        if (r.h < a.hq) {
            __half *dst = a.q_out + ((size_t)b * a.hq + r.h) * a.d;
            dst[r.i] = y0, dst[r.i + half] = y1;
        } else if (r.fits) {
            __half *dst = a.k_cache + ((((size_t)pb * a.hkv + (r.h - a.hq)) * a.block_size) + r.in_block) * a.d;
            dst[r.i] = y0, dst[r.i + half] = y1;
        }
    } else if (r.fits) {
        __half *dst = a.v_cache + ((size_t)pb * a.hkv + (r.h - a.hq - a.hkv)) * a.d * a.block_size + r.in_block;
        dst[(size_t)r.i * a.block_size] = __float2half_rn(x0);
        dst[(size_t)(r.i + half) * a.block_size] = __float2half_rn(x1);
    }
}

// 8 packed weights -> 8 fp16, exact: the byte w + 128 under 0x64 is the half 1024 + w + 128.
__device__ __forceinline__ h16x8 w8_to_f16(uint32_t lo, uint32_t hi) {
    uint32_t h[4];
    h[0] = __builtin_amdgcn_perm(0x64646464u, lo, 0x07010700u); // [b0, 0x64, b1, 0x64]
    h[1] = __builtin_amdgcn_perm(0x64646464u, lo, 0x07030702u);
    h[2] = __builtin_amdgcn_perm(0x64646464u, hi, 0x07010700u);
    h[3] = __builtin_amdgcn_perm(0x64646464u, hi, 0x07030702u);
    h16x8 v;
    __builtin_memcpy(&v, h, 16);
    return v - (_Float16)1152.0f; // 1024 + (w + 128) - 1152 = w, exact in fp16
}

// Epilogue of 4 consecutive output channels of one token, at element o of `out`: SwiGLU gate, residual (its four halves in `res`),
// conversion, store.
template <int G> __device__ __forceinline__ void store_gemm_row(const float (&v)[G][4], size_t o, bool has_residual, uint2 res, void *out, int out_f32) {
    float y[4];
    __half rh[4];
    __builtin_memcpy(rh, &res, 8);
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (G == 2) y[r] = v[0][r] / (1.f + __expf(-v[0][r])) * v[G - 1][r]; // silu(gate) * up
        else y[r] = v[0][r];
        if (has_residual) y[r] += __half2float(rh[r]);
    }
    if (out_f32) {
        *reinterpret_cast<float4 *>(reinterpret_cast<float *>(out) + o) = float4{y[0], y[1], y[2], y[3]};
    } else {
        __half h[4];
#pragma unroll
        for (int r = 0; r < 4; r++) h[r] = __float2half_rn(y[r]);
        uint2 pk;
        __builtin_memcpy(&pk, h, 8);
        *reinterpret_cast<uint2 *>(reinterpret_cast<__half *>(out) + o) = pk;
    }
}

// The same for one channel.
template <int G> __device__ __forceinline__ void store_gemm_one(const float (&v)[G], size_t o, bool has_residual, uint16_t res, void *out, int out_f32) {
    float y = G == 2 ? v[0] / (1.f + __expf(-v[0])) * v[G - 1] : v[0];
    if (has_residual) y += __half2float(__builtin_bit_cast(__half, res));
    if (out_f32) reinterpret_cast<float *>(out)[o] = y;
    else reinterpret_cast<__half *>(out)[o] = __float2half_rn(y);
}

// MT = 16-token column tiles (m <= 16 * MT); G = matrices multiplied at once (2: SwiGLU gate and up).
// grid.x = output tiles of 16 channels.  The eight waves of a block split the reduction; a wave
// requests the weights and token slices of four k-steps before it multiplies any of them, so a
// whole share of a short reduction (896 / 8 waves = 2 k-steps) is a single memory round trip.
constexpr int kGemmWaves = 8;
constexpr int kGemmThreads = kGemmWaves * 64;
constexpr int kGemmBatch = 4; // k-steps a wave requests before it multiplies any
constexpr int kRedPitch = 64 + 16; // floats

// SPLIT: the block's waves share one output tile and split its reduction (few tiles, long reductions);
// otherwise every wave owns a tile of its own and the whole reduction (many tiles: the vocabulary head).
// PAIRED: a wave's even and odd k-steps are summed apart, as w8a16_small_tile_kernel does.
template <int MT, int G, bool SPLIT, bool PAIRED = false> __global__ __launch_bounds__(kGemmThreads) void w8a16_gemm_kernel(const GemmArgs a) {
    constexpr int B = kGemmBatch, P = PAIRED ? 2 : 1;
    static_assert(B % 2 == 0, "a batch starts with an even k-step of the wave's share");
    __shared__ float red[SPLIT ? kGemmWaves : 1][P][G][MT][64][4];
    __shared__ float rstd[MT * 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    if (a.ln_w) { // (uniform; before any wave leaves the block)
        constexpr int R = MT * 16 / kGemmWaves; // rows per wave
        float rs[R];
        rms_rstd_rows<R>(reinterpret_cast<const __half *>(a.a), a.k, a.m, wave, kGemmWaves, lane, a.ln_eps, rs);
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < R; i++)
                if (wave + i * kGemmWaves < a.m) rstd[wave + i * kGemmWaves] = rs[i];
        }
        __syncthreads();
    }
    const int per = SPLIT ? (a.ksteps + kGemmWaves - 1) / kGemmWaves : a.ksteps;
    const int ks0 = SPLIT ? wave * per : 0, ks1 = min(a.ksteps, ks0 + per);
    const int out_tile = SPLIT ? (int)blockIdx.x : (int)blockIdx.x * kGemmWaves + wave;
    if (out_tile >= a.up_tile_offset) return; // SPLIT: never; otherwise the last block's spare waves (uniform per wave)
    f32x4v acc[P][G][MT];
#pragma unroll
    for (int q = 0; q < P; q++)
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int t = 0; t < MT; t++) acc[q][g][t] = f32x4v{0.f, 0.f, 0.f, 0.f};

    const int tile[2] = {out_tile, out_tile + a.up_tile_offset};
    // token rows of this lane (clamped: rows past m read row m - 1 and are never stored)
    const uint16_t *arow[MT];
    float rrow[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) {
        arow[t] = a.a + (size_t)min(t * 16 + i16, a.m - 1) * a.k + kg * 16;
        rrow[t] = a.ln_w ? rstd[min(t * 16 + i16, a.m - 1)] : 1.f;
    }

    // The epilogue's operands (SPLIT: of the token tile this wave finishes) are asked for before the products: the
    // launch is a chain of memory round trips, and this takes the last one out of it (5 rows of 2880 to 208, normalised, 7.5 -> 7.2 us).
    // (not with four token tiles: their slices leave no registers for it)
    constexpr bool kPre = SPLIT && MT <= 2;
    float4 sc[G], bs[G];
    uint2 res_pre = uint2{0u, 0u};
    if (kPre) {
#pragma unroll
        for (int g = 0; g < G; g++) {
            sc[g] = *reinterpret_cast<const float4 *>(a.scale + tile[g] * 16 + kg * 4);
            bs[g] = float4{0.f, 0.f, 0.f, 0.f};
            if (a.bias) bs[g] = *reinterpret_cast<const float4 *>(a.bias + tile[g] * 16 + kg * 4);
        }
        const int m_pre = min(min(wave, MT - 1) * 16 + i16, a.m - 1);
        if (a.residual) res_pre = *reinterpret_cast<const uint2 *>(a.residual + (size_t)m_pre * a.n_out + out_tile * 16 + kg * 4);
    }
    for (int kb = ks0; kb < ks1; kb += B) {
        lu32x4 wv[B][G];
        lu32x4 av[B][MT][2];
        lu32x4 lw[B][2]; // the normalisation weights of the lane's 16 reduction indices
#pragma unroll
        for (int u = 0; u < B; u++) {
            const int ks = min(kb + u, ks1 - 1); // steps past the share re-read the last one and are not multiplied
#pragma unroll
            for (int g = 0; g < G; g++) wv[u][g] = a.w[((size_t)tile[g] * a.ksteps + ks) * 64 + lane];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                av[u][t][0] = *reinterpret_cast<const lu32x4 *>(arow[t] + ks * 64);
                av[u][t][1] = *reinterpret_cast<const lu32x4 *>(arow[t] + ks * 64 + 8);
            }
            if (a.ln_w) {
                lw[u][0] = *reinterpret_cast<const lu32x4 *>(a.ln_w + ks * 64 + kg * 16);
                lw[u][1] = *reinterpret_cast<const lu32x4 *>(a.ln_w + ks * 64 + kg * 16 + 8);
            }
        }
        if (a.ln_w) {
#pragma unroll
            for (int u = 0; u < B; u++)
                if (MT > 2 || kb + u < ks1) // (uniform for the wave: the slices past its share are not multiplied; four token tiles have no registers to spare for the branch)
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int hlf = 0; hlf < 2; hlf++) av[u][t][hlf] = normalise8(av[u][t][hlf], rrow[t], lw[u][hlf]);
        }
#pragma unroll
        for (int u = 0; u < B; u++) {
            if (kb + u < ks1) { // uniform for the wave
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const h16x8 w0 = w8_to_f16(wv[u][g][0], wv[u][g][1]), w1 = w8_to_f16(wv[u][g][2], wv[u][g][3]);
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        h16x8 x0, x1;
                        __builtin_memcpy(&x0, &av[u][t][0], 16);
                        __builtin_memcpy(&x1, &av[u][t][1], 16);
                        f32x4v &to = acc[u % P][g][t];
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, x0, to, 0, 0, 0);
                        to = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, x1, to, 0, 0, 0);
                    }
                }
            }
        }
    }
    // ---- combine the waves' partial sums ------------------------------------------------------------
    if (SPLIT) {
#pragma unroll
        for (int q = 0; q < P; q++)
#pragma unroll
            for (int g = 0; g < G; g++)
#pragma unroll
                for (int t = 0; t < MT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) red[wave][q][g][t][lane][r] = acc[q][g][t][r];
        __syncthreads();
        if (wave >= MT) return; // wave w finishes token tile w
    }
    // lane (i16 = token within the tile, kg): channels tile * 16 + kg * 4 + r
#pragma unroll
    for (int tt = 0; tt < (SPLIT ? 1 : MT); tt++) {
        const int t = SPLIT ? wave : tt;
        const int m = t * 16 + i16;
        float v[G][4];
#pragma unroll
        for (int g = 0; g < G; g++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float s = 0.f;
                if (SPLIT) {
#pragma unroll
                    for (int w = 0; w < kGemmWaves; w++) // fixed order: deterministic
#pragma unroll
                        for (int q = 0; q < P; q++) s += red[w][q][g][t][lane][r];
                } else {
                    s = acc[0][g][tt][r];
                }
                if (kPre) {
                    const float scv[4] = {sc[g].x, sc[g].y, sc[g].z, sc[g].w}, bsv[4] = {bs[g].x, bs[g].y, bs[g].z, bs[g].w};
                    s *= scv[r];
                    if (a.bias) s += bsv[r];
                } else {
                    const int ch = tile[g] * 16 + kg * 4 + r;
                    s *= a.scale[ch];
                    if (a.bias) s += a.bias[ch];
                }
                v[g][r] = s;
            }
        }
        if (m >= a.m) continue;
        const size_t o = (size_t)m * a.n_out + out_tile * 16 + kg * 4;
        const uint2 res = kPre ? res_pre : a.residual ? *reinterpret_cast<const uint2 *>(a.residual + o) : uint2{0u, 0u};
        store_gemm_row<G>(v, o, a.residual != nullptr, res, a.out, a.out_f32);
    }
}

// Kernel arguments that are used at different times, asked for together: a scalar load behind a branch or a wait is a wait of its own.
template <typename A, typename B, typename C, typename D, typename E, typename F>
__device__ __forceinline__ void request_together(const A &a, const B &b, const C &c, const D &d, const E &e, const F &f) {
    asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d), "s"(e), "s"(f));
}

// One tile of 16 output channels (G = 2: a gate tile and its up tile; ROPE: the two tiles that hold the halves of eight
// rotate-half pairs, up_tile_offset = head_dim / 32 apart) times 16 token rows per block, the reduction split over the block's
// eight waves and combined through LDS in a fixed order: the products of a decode step, a few dozen to a few hundred tiles.
//
// What bounds such a launch is not its bytes (a block's share of the weights is 14 to 78 KiB) but its chain of waits, so the
// chain is as short as it can be: every argument is requested at once, then, without a branch between them, the rows, the weights
// and the epilogue's operands, in the order in which they are needed and with addresses clamped where there is nothing to read.
// (Loads behind branches cannot be waited for one by one: the normalisation waited for the weights' trip to memory, and the
// products for the scales'.)  More than 16 rows are more blocks, not longer ones: those of one tile run on one die where the
// number of tiles is a multiple of 8, and the weights come out of its L2.
// Between the waits it is instructions: a wave issues one every 4 to 9 cycles, so the hundred that one wave runs while the others
// wait for it are a quarter of a microsecond.  Hence rows scaled with v_fma_mix_f32, weights converted ahead of the barrier, an output
// per lane on four waves behind the last one, the rotation on waves that have fewer rows to bring in (one operator over 24 layers, us,
// before / after: 1 row gate / up 4.86 / 4.34, q / k / v 4.16 / 3.60, output 2.55 / 2.29; 16 rows 6.34 / 5.53, 5.06 / 4.72, 2.89 /
// 2.61; 64 rows gate / up 11.6 / 9.3).
//
// KS: k-steps of 64 a wave may have, all requested at once (k <= 512 * KS).
// R: the products read the rows from LDS, and wave w brings in rows w and, with R = 2, w + 8, PIECES pieces of 512 elements each: whole
// lines, where an operand read of the rows where they lie (R = 0: too long for LDS, or few) takes 32 bytes of each of 64 lines (14 rows of
// 640 to 4768 columns 4.3 -> 3.5 us, 50 of 704 to 7760 10.8 -> 7.3).
// NORM: the rows are RMS-normalised on the way (see rms_rstd_rows for the order).
template <int G, int KS, bool NORM, int R, int PIECES, bool ROPE>
__global__ __launch_bounds__(kGemmThreads) void w8a16_tile_kernel(const GemmArgs a) {
    static_assert(!ROPE || G == 2, "the rotating epilogue pairs two tiles of one block");
    constexpr bool LDS = R > 0;
    static_assert(LDS || !NORM, "rows are normalised on their way to LDS");
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[]; // LDS: [16][k halves + padding]
    // a wave's sums: [four channels][16 rows][channel of the four], the rows of the next four 16 banks on
    __shared__ float red[kGemmWaves][G][4][kRedPitch];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int k = a.k, ksteps = a.ksteps, off = a.up_tile_offset, n_out = a.n_out, out_f32 = a.out_f32;
    const float eps = a.ln_eps;
    const uint16_t *const x = a.a, *const ln_w = a.ln_w, *const residual = a.residual;
    const lu32x4 *const w = a.w;
    const float *const scale = a.scale, *const bias = a.bias ? a.bias : a.scale;
    void *const out = a.out;
    const bool has_bias = a.bias != nullptr;
    request_together(eps, out, out_f32, residual, n_out, a.m);
    const int row0 = (int)blockIdx.y * 16, rows = min(16, a.m - row0), last = row0 + rows - 1;
    const int tile0 = ROPE ? (int)blockIdx.x / off * (2 * off) + (int)blockIdx.x % off : (int)blockIdx.x;
    const int tile[2] = {tile0, tile0 + off};

    // ---- requests ---------------------------------------------------------------------------------------
    int rope_pos = 0;
    if constexpr (ROPE) rope_pos = a.rope.ctx_lens[min(row0 + (wave & 3) * 4 + kg, last)]; // (loads return in order: asked for first, it is there first)
    const int per = (ksteps + kGemmWaves - 1) / kGemmWaves, ks0 = wave * per, ks1 = min(ksteps, ks0 + per);
    const uint16_t *xrow = x + (size_t)min(row0 + i16, last) * k + kg * 16;
    lu32x4 v[LDS ? R : 1][LDS ? PIECES : 1], lwp[NORM ? PIECES : 1], wv[KS][G], av[LDS ? 1 : KS][2];
    if constexpr (LDS) {
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            const int e0 = min(lane * 8 + p * 512, k - 8); // (past the row: masked below)
#pragma unroll
            for (int i = 0; i < R; i++) v[i][p] = *reinterpret_cast<const lu32x4 *>(x + (size_t)min(row0 + wave + i * kGemmWaves, last) * k + e0);
            if constexpr (NORM) lwp[p] = *reinterpret_cast<const lu32x4 *>(ln_w + e0);
        }
    }
    // The lane's output, of the four waves that finish the tile: row fw * 4 + lane / 16, channel lane % 16.
    const int fw = ROPE ? wave - 4 : wave, frow = (fw & 3) * 4 + kg, fch = tile0 * 16 + i16;
    float sc[G], bs[G]; // (ahead of the products' operands: behind their thirty loads a cold line of scales would arrive last)
#pragma unroll
    for (int g = 0; g < G; g++) sc[g] = scale[fch + g * off * 16], bs[g] = bias[fch + g * off * 16];
    const size_t o = (size_t)min(row0 + frow, last) * n_out + fch;
    const uint16_t res = *(residual ? residual + o : x);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < KS; u++) {
        const int ks = max(min(ks0 + u, ks1 - 1), 0);
#pragma unroll
        for (int g = 0; g < G; g++) wv[u][g] = w[((size_t)tile[g] * ksteps + ks) * 64 + lane];
        if constexpr (!LDS) {
            av[u][0] = *reinterpret_cast<const lu32x4 *>(xrow + ks * 64), av[u][1] = *reinterpret_cast<const lu32x4 *>(xrow + ks * 64 + 8);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- rows --------------------------------------------------------------------------------------------
    RopePair rope;
    if constexpr (ROPE) {
        // The angle is computed while the rows and weights travel, by the waves that finish the tile: the upper four, which have fewer
        // rows to bring in or none.
        if (fw >= 0 && fw * 4 < rows) rope = rope_pair(a.rope, min(row0 + frow, last), fch / a.rope.d, fch % a.rope.d, rope_pos);
        __builtin_amdgcn_sched_barrier(0);
    }
    const int pitch = rows_in_lds_pitch(k);
    if constexpr (LDS) {
        if (wave < rows) { // (uniform; what LDS holds in the place of rows past m meets no row that is stored)
            if constexpr (NORM) {
                float ss[R];
#pragma unroll
                for (int i = 0; i < R; i++) ss[i] = 0.f;
#pragma unroll
                for (int p = 0; p < PIECES; p++)
#pragma unroll
                    for (int i = 0; i < R; i++) {
                        if (lane * 8 + p * 512 >= k) v[i][p] = lu32x4{0, 0, 0, 0}; // (+0 squares leave a sum as it is)
                        add_squares8(v[i][p], ss[i]);
                    }
#pragma unroll
                for (int i = 0; i < R; i++) ss[i] = 1.0f / sqrtf(wave_sum(ss[i]) / (float)k + eps); // rstd_from_sum's formula
#pragma unroll
                for (int p = 0; p < PIECES; p++)
#pragma unroll
                    for (int i = 0; i < R; i++) v[i][p] = normalise8(v[i][p], ss[i], lwp[p]);
            }
#pragma unroll
            for (int p = 0; p < PIECES; p++)
                if (lane * 8 + p * 512 < k) {
#pragma unroll
                    for (int i = 0; i < R; i++) *reinterpret_cast<lu32x4 *>(xs + (size_t)(wave + i * kGemmWaves) * pitch + (lane * 8 + p * 512) * 2) = v[i][p];
                }
        }
    }
    // (converted ahead of the barrier: by the waves without a row while the others normalise theirs)
    h16x8 wf[KS][G][2];
#pragma unroll
    for (int u = 0; u < KS; u++)
#pragma unroll
        for (int g = 0; g < G; g++) wf[u][g][0] = w8_to_f16(wv[u][g][0], wv[u][g][1]), wf[u][g][1] = w8_to_f16(wv[u][g][2], wv[u][g][3]);
    if constexpr (LDS) __syncthreads();

    // ---- products ------------------------------------------------------------------------------------------
    f32x4v acc[G];
#pragma unroll
    for (int g = 0; g < G; g++) acc[g] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const uint8_t *xl = xs + (size_t)i16 * pitch + kg * 32; // the lane's 16 reduction indices of a k-step
#pragma unroll
    for (int u = 0; u < KS; u++) {
        if (ks0 + u < ks1) { // uniform
            h16x8 x0, x1;
            if constexpr (LDS) {
                x0 = *reinterpret_cast<const h16x8 *>(xl + (ks0 + u) * 128), x1 = *reinterpret_cast<const h16x8 *>(xl + (ks0 + u) * 128 + 16);
            } else {
                __builtin_memcpy(&x0, &av[u][0], 16), __builtin_memcpy(&x1, &av[u][1], 16);
            }
#pragma unroll
            for (int g = 0; g < G; g++) {
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[u][g][0], x0, acc[g], 0, 0, 0);
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[u][g][1], x1, acc[g], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++) *reinterpret_cast<f32x4v *>(&red[wave][g][kg][i16 * 4]) = acc[g];
    __syncthreads();
    // An output per lane, by as many waves as the rows need: what follows is a chain of some hundred instructions, and with four
    // channels a lane on one wave it was twice as long.
    if (fw < 0 || fw * 4 >= rows) return; // (uniform)
    float y[G];
#pragma unroll
    for (int g = 0; g < G; g++) {
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < kGemmWaves; q++) s += red[q][g][i16 >> 2][frow * 4 + (i16 & 3)]; // fixed order: deterministic
        y[g] = s * sc[g];
        if (has_bias) y[g] += bs[g];
    }
    if (frow >= rows) return;
    // (rounded to fp16 as the projection's output would be stored; the partner is d / 2 channels further)
    if constexpr (ROPE) rope_store(a.rope, row0 + frow, rope, __half2float(__float2half_rn(y[0])), __half2float(__float2half_rn(y[1])));
    else store_gemm_one<G>(y, o, residual != nullptr, res, out, out_f32);
}

// The same product for long reductions over few tiles (the down projection), where a block of the kernel above has its compute
// unit to itself and is bound by what passes through that unit's L1: tiles of 8 channels by 8 rows.  The matrix instruction's 16
// rows are 8 channels of two consecutive k-steps, its 16 columns the 8 token rows of the same two; the two blocks of the result
// on the diagonal are wanted, the other two are not.  A block then reads half the weights and half the rows for a quarter of the
// outputs, and a wave half as many fragments.  The order of the sum: a wave's even steps and its odd steps, then the waves' two
// sums after one another (w8a16_gemm_kernel with PAIRED adds in it too).
// Two blocks share a 16-channel tile of the packed weights; both on one die, so that its L2 keeps the halves together.
template <int KP> __global__ __launch_bounds__(kGemmThreads) void w8a16_small_tile_kernel(const GemmArgs a) {
    __shared__ float red[kGemmWaves][64][4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i8 = lane & 7, odd = lane >> 3 & 1, kg = lane >> 4;
    const int k = a.k, ksteps = a.ksteps, n_out = a.n_out, out_f32 = a.out_f32;
    const uint16_t *const x = a.a, *const residual = a.residual;
    const lu32x4 *const w = a.w;
    const float *const scale = a.scale, *const bias = a.bias ? a.bias : a.scale;
    void *const out = a.out;
    const bool has_bias = a.bias != nullptr;
    request_together(k, out, out_f32, residual, n_out, a.m);
    const int group = (int)blockIdx.x / 16 * 8, in_group = min(8, a.up_tile_offset - group), r16 = (int)blockIdx.x % 16;
    const int half = r16 >= in_group, tile = group + r16 - half * in_group;
    const int row0 = (int)blockIdx.y * 8, rows = min(8, a.m - row0), last = row0 + rows - 1;
    const int per = (ksteps + kGemmWaves - 1) / kGemmWaves, ks0 = wave * per, ks1 = min(ksteps, ks0 + per);
    // the output of wave 0's lane: row lane / 8, channel lane % 8 of the eight
    const int frow = lane >> 3, ch = tile * 16 + half * 8 + i8;
    const size_t o = (size_t)min(row0 + frow, last) * n_out + ch;
    const float sc = scale[ch], bs = bias[ch];
    const uint16_t res = *(residual ? residual + o : x);
    const lu32x4 *wl = w + (size_t)tile * ksteps * 64 + kg * 16 + half * 8 + i8;
    const uint16_t *xl = x + (size_t)min(row0 + i8, last) * k + kg * 16;
    lu32x4 wv[KP], av[KP][2];
#pragma unroll
    for (int u = 0; u < KP; u++) {
        const int ks = max(min(ks0 + 2 * u + odd, ks1 - 1), 0); // steps past the share: cleared below
        wv[u] = wl[ks * 64];
        av[u][0] = *reinterpret_cast<const lu32x4 *>(xl + ks * 64), av[u][1] = *reinterpret_cast<const lu32x4 *>(xl + ks * 64 + 8);
        __builtin_amdgcn_sched_barrier(0);
    }
    f32x4v acc = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < KP; u++) {
        if (ks0 + 2 * u < ks1) { // uniform
            if (ks0 + 2 * u + 1 >= ks1 && odd) wv[u] = av[u][0] = av[u][1] = lu32x4{0, 0, 0, 0};
            h16x8 x0, x1;
            __builtin_memcpy(&x0, &av[u][0], 16), __builtin_memcpy(&x1, &av[u][1], 16);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w8_to_f16(wv[u][0], wv[u][1]), x0, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w8_to_f16(wv[u][2], wv[u][3]), x1, acc, 0, 0, 0);
        }
    }
    *reinterpret_cast<f32x4v *>(red[wave][lane]) = acc;
    __syncthreads();
    if (wave != 0) return;
    float y[1] = {0.f};
#pragma unroll
    for (int q = 0; q < kGemmWaves; q++) { // fixed order: deterministic
        y[0] += red[q][(i8 >> 2) * 16 + frow][i8 & 3];
        y[0] += red[q][((i8 >> 2) + 2) * 16 + 8 + frow][i8 & 3];
    }
    y[0] *= sc;
    if (has_bias) y[0] += bs;
    if (frow >= rows) return;
    store_gemm_one<1>(y, o, residual != nullptr, res, out, out_f32);
}

constexpr int kRowsBatch = 8;
// Many output tiles and a reduction short enough for the token rows to fit in LDS (the vocabulary head): a wave owns a
// tile (G = 2: the gate tile and its up tile) and the whole reduction, as in the kernel above without SPLIT, but the
// block's waves share the token rows through LDS.  A wave brings in whole rows (row wave, wave + 8, ...): it adds their
// squares in rms_rstd_rows' order as they arrive and, knowing 1 / sqrt(mean + eps) of its own rows without asking another
// wave, normalises them on the way to LDS -- one trip to memory and one barrier in front of the products, and every element
// normalised once per block instead of once per wave.  A wave has the weights of KB k-steps in flight, the first KB from the
// start of the kernel.  The arithmetic per element and the order of the multiply-adds are those of the kernel above.
template <int MT, int G, int KB, int PIECES> __global__ __launch_bounds__(kGemmThreads) void w8a16_gemm_rows_in_lds_kernel(const GemmArgs a) {
    constexpr int WAVES = kGemmWaves;
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[]; // [MT * 16][k halves + padding]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int pitch = rows_in_lds_pitch(a.k);
    // The weights do not depend on the rows: the first KB k-steps of this wave's share are requested before anything
    // else, so that their trip to memory runs beside the one that brings the rows in (a spare wave of the last block
    // reads the last tile's and multiplies nothing).
    // A block walks the groups of WAVES tiles blockIdx.x, blockIdx.x + gridDim.x, ...: a launch with fewer
    // blocks than groups (the vocabulary head) brings the rows in and normalises them once per block, not once per group.
    int group = (int)blockIdx.x;
    int out_tile = group * WAVES + wave;
    const int ks1 = a.ksteps;
    int first = min(out_tile, a.up_tile_offset - 1);
    int tile[2] = {first, first + a.up_tile_offset};
    lu32x4 wv[KB][G];
    auto request_first = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < KB; u++) {
            const int ks = min(u, ks1 - 1); // steps past the end re-read the last one and are not multiplied
#pragma unroll
            for (int g = 0; g < G; g++) wv[u][g] = a.w[((size_t)tile[g] * a.ksteps + ks) * 64 + lane];
        }
    };
    request_first();
    {
        constexpr int R = MT * 16 / WAVES; // rows per wave
        // The wave's rows stay in registers from the load to the one LDS write: their sums of squares, the butterflies
        // and the normalisation run for all R rows side by side (independent chains), element by element in the order
        // rms_rstd_rows and rmsnorm_f16_kernel use.
        lu32x4 v[R][PIECES], lwp[PIECES];
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            const int e0 = lane * 8 + p * 512;
            lwp[p] = lu32x4{0, 0, 0, 0};
            if (a.ln_w && e0 < a.k) lwp[p] = *reinterpret_cast<const lu32x4 *>(a.ln_w + e0);
#pragma unroll
            for (int i = 0; i < R; i++) {
                const int r = wave + i * WAVES;
                v[i][p] = lu32x4{0, 0, 0, 0}; // rows past m: zeros (their products are never stored)
                if (r < a.m && e0 < a.k) v[i][p] = *reinterpret_cast<const lu32x4 *>(a.a + (size_t)r * a.k + e0);
            }
        }
        if (a.ln_w) {
            float ss[R];
#pragma unroll
            for (int i = 0; i < R; i++) ss[i] = 0.f;
#pragma unroll
            for (int p = 0; p < PIECES; p++)
#pragma unroll
                for (int i = 0; i < R; i++) add_squares8(v[i][p], ss[i]); // (pieces past the row are zeros: +0 leaves a sum as it is)
#pragma unroll
            for (int i = 0; i < R; i++) ss[i] = wave_sum(ss[i]);
            float rr[R];
#pragma unroll
            for (int i = 0; i < R; i++) rr[i] = 1.0f / sqrtf(ss[i] / (float)a.k + a.ln_eps); // rstd_from_sum's formula
#pragma unroll
            for (int p = 0; p < PIECES; p++)
#pragma unroll
                for (int i = 0; i < R; i++) v[i][p] = normalise8(v[i][p], rr[i], lwp[p]);
        }
#pragma unroll
        for (int p = 0; p < PIECES; p++) {
            const int e0 = lane * 8 + p * 512;
            if (e0 < a.k) {
#pragma unroll
                for (int i = 0; i < R; i++) *reinterpret_cast<lu32x4 *>(xs + (size_t)(wave + i * WAVES) * pitch + e0 * 2) = v[i][p];
            }
        }
    }
    __syncthreads();
    const int groups = (a.up_tile_offset + WAVES - 1) / WAVES;
    for (;;) {
    if (out_tile >= a.up_tile_offset) return; // the last group's spare waves (uniform per wave; no group follows it)
    f32x4v acc[G][MT];
#pragma unroll
    for (int g = 0; g < G; g++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[g][t] = f32x4v{0.f, 0.f, 0.f, 0.f};
    const uint8_t *xl = xs + (size_t)i16 * pitch + kg * 32; // the lane's 16 reduction indices of a k-step
    float4 sc[G], bs[G]; // the epilogue's operands, asked for before the products
#pragma unroll
    for (int g = 0; g < G; g++) {
        sc[g] = *reinterpret_cast<const float4 *>(a.scale + tile[g] * 16 + kg * 4);
        bs[g] = float4{0.f, 0.f, 0.f, 0.f};
        if (a.bias) bs[g] = *reinterpret_cast<const float4 *>(a.bias + tile[g] * 16 + kg * 4);
    }
    for (int kb = 0; kb < ks1; kb += KB) {
        if (kb != 0) { // (the first batch is on its way since the start)
#pragma unroll
            for (int u = 0; u < KB; u++) {
                const int ks = min(kb + u, ks1 - 1); // steps past the end re-read the last one and are not multiplied
#pragma unroll
                for (int g = 0; g < G; g++) wv[u][g] = a.w[((size_t)tile[g] * a.ksteps + ks) * 64 + lane];
            }
        }
#pragma unroll
        for (int u = 0; u < KB; u++) {
            if (kb + u < ks1) { // uniform
                h16x8 x0[MT], x1[MT];
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const uint8_t *xp = xl + (size_t)t * 16 * pitch + (size_t)(kb + u) * 128;
                    x0[t] = *reinterpret_cast<const h16x8 *>(xp), x1[t] = *reinterpret_cast<const h16x8 *>(xp + 16);
                }
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const h16x8 w0 = w8_to_f16(wv[u][g][0], wv[u][g][1]), w1 = w8_to_f16(wv[u][g][2], wv[u][g][3]);
#pragma unroll
                    for (int t = 0; t < MT; t++) {
                        acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, x0[t], acc[g][t], 0, 0, 0);
                        acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, x1[t], acc[g][t], 0, 0, 0);
                    }
                }
            }
        }
    }
    // the next group's first weights are requested as soon as this one's are multiplied: they travel under the epilogue
    group += (int)gridDim.x;
    const bool more = group < groups;
    const int next_tile = group * WAVES + wave;
    if (more) {
        first = min(next_tile, a.up_tile_offset - 1);
        tile[0] = first, tile[1] = first + a.up_tile_offset;
        request_first();
    }
    // lane (i16 = token within the tile, kg): channels tile * 16 + kg * 4 + r
#pragma unroll
    for (int t = 0; t < MT; t++) {
        const int m = t * 16 + i16;
        float v[G][4];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const float scv[4] = {sc[g].x, sc[g].y, sc[g].z, sc[g].w}, bsv[4] = {bs[g].x, bs[g].y, bs[g].z, bs[g].w};
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float s = acc[g][t][r] * scv[r];
                if (a.bias) s += bsv[r];
                v[g][r] = s;
            }
        }
        if (m >= a.m) continue;
        const size_t o = (size_t)m * a.n_out + out_tile * 16 + kg * 4;
        const uint2 res = a.residual ? *reinterpret_cast<const uint2 *>(a.residual + o) : uint2{0u, 0u};
        store_gemm_row<G>(v, o, a.residual != nullptr, res, a.out, a.out_f32);
    }
    if (!more) return;
    out_tile = next_tile;
    }
}

// out[r, :] = x[r, :] * rsqrt(mean(x[r, :]^2) + eps) * weight, fp32 arithmetic; one wave per row.
__global__ __launch_bounds__(kLlmThreads) void rmsnorm_f16_kernel(const __half *__restrict__ x, const __half *__restrict__ w,
                                                                 __half *__restrict__ out, int rows, int hidden, float eps) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= rows) return;
    const __half *xr = x + (size_t)row * hidden;
    float r;
    if ((hidden & 7) == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
        float rs[1];
        rms_rstd_rows<1>(x, hidden, rows, row, 1, lane, eps, rs);
        r = rs[0];
    } else {
        r = rms_rstd_scalar(xr, hidden, eps, lane);
    }
    for (int i = lane; i < hidden; i += 64) {
        // The fp32 product is rounded before it is converted to fp16.  Left to itself the compiler turns multiply and
        // conversion into one mixed-precision instruction (a single rounding) in some copies of this loop's body
        // and not in others, so the same input could round either way depending on where it sits in the row.
        float pr = __half2float(xr[i]) * r * __half2float(w[i]);
        asm volatile("" : "+v"(pr));
        out[(size_t)row * hidden + i] = __float2half_rn(pr);
    }
}

// Rotary embedding (rotate-half pairing: element i with i + d/2, angle pos * theta^(-2i/d)) of the q
// and k heads of the new token, and the append of the rotated k and of v at position ctx_lens[b]
// of the paged cache.  One thread per (sequence, head, pair).
__global__ __launch_bounds__(kLlmThreads) void rope_append_kernel(const RopeArgs a) {
    const int half = a.d / 2;
    const int heads = a.hq + 2 * a.hkv;
    const int gid = blockIdx.x * kLlmThreads + threadIdx.x;
    if (gid >= a.batch * heads * half) return;
    const int i = gid % half, h = (gid / half) % heads, b = gid / (half * heads);
    const __half *src = a.qkv + ((size_t)b * heads + h) * a.d;
    rope_store(a, b, rope_pair(a, b, h, i, a.ctx_lens[b]), __half2float(src[i]), __half2float(src[i + half]));
}

// Index of the largest element of every row (the lowest index among equals); one block of 1024
// threads per row, 16-byte loads, so that a 152 K-entry vocabulary row is a few dozen independent
// loads per thread.
constexpr int kArgmaxThreads = 1024;
__device__ __forceinline__ void argmax_take(float v, int i, float &best, int &bi) {
    if (v > best || (v == best && i < bi)) best = v, bi = i;
}
__global__ __launch_bounds__(kArgmaxThreads) void argmax_f32_kernel(const float *__restrict__ x, int32_t *__restrict__ out, int cols) {
    __shared__ float sv[kArgmaxThreads / 64];
    __shared__ int si[kArgmaxThreads / 64];
    const float *row = x + (size_t)blockIdx.x * cols;
    float best = -INFINITY;
    int bi = 0x7fffffff;
    // rows start 16-byte aligned when cols is a multiple of 4 (x itself is aligned by the allocator)
    const int nvec = ((cols & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) ? cols / 4 : 0;
    // eight 16-byte loads per thread are requested before any of them is compared: a row of the vocabulary is five
    // memory round trips, not one per load
    constexpr int U = 8;
    for (int i0 = threadIdx.x; i0 < nvec; i0 += U * kArgmaxThreads) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = reinterpret_cast<const float4 *>(row)[min(i0 + u * kArgmaxThreads, nvec - 1)];
        // the batch's maximum first (one instruction per element); only a batch that beats the running maximum -- a
        // handful per thread -- is searched for where (its first such element: indices grow with u and i0)
        float m = -INFINITY;
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u * kArgmaxThreads < nvec) m = fmaxf(m, fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w)));
        if (m > best) {
            best = m;
            bi = 0x7fffffff;
#pragma unroll
            for (int u = U - 1; u >= 0; u--) {
                const int i = i0 + u * kArgmaxThreads;
                if (i < nvec) {
                    bi = v[u].w == m ? 4 * i + 3 : bi;
                    bi = v[u].z == m ? 4 * i + 2 : bi;
                    bi = v[u].y == m ? 4 * i + 1 : bi;
                    bi = v[u].x == m ? 4 * i : bi;
                }
            }
        }
    }
    for (int i = nvec * 4 + threadIdx.x; i < cols; i += kArgmaxThreads) argmax_take(row[i], i, best, bi);
    // the wave's winner by exchanges between lanes, the block's through LDS
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) argmax_take(__shfl_xor(best, d), __shfl_xor(bi, d), best, bi);
    if ((threadIdx.x & 63) == 0) sv[threadIdx.x >> 6] = best, si[threadIdx.x >> 6] = bi;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kArgmaxThreads / 64; w++) argmax_take(sv[w], si[w], best, bi);
        out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
    }
}

__global__ __launch_bounds__(kLlmThreads) void embed_f16_kernel(const __half *__restrict__ table, const int32_t *__restrict__ ids,
                                                               __half *__restrict__ out, int rows, int hidden, int vocab) {
    const int gid = blockIdx.x * kLlmThreads + threadIdx.x;
    if (gid >= rows * hidden) return;
    const int r = gid / hidden, c = gid - r * hidden;
    const int id = min(max(ids[r], 0), vocab - 1);
    out[gid] = table[(size_t)id * hidden + c];
}

__global__ void add_i32_kernel(int32_t *x, int n, int32_t delta) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] += delta;
}

} // namespace nnhip

using namespace nnhip;

extern "C" int nncase_hip_w8a16_destroy(nncase_hip_ctx_t *ctx, nncase_hip_w8a16_t *w) {
    NNHIP_CHECK_CTX(ctx);
    if (!w) return 0;
    NNHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (w->d_packed) (void)hipFree(w->d_packed);
    if (w->d_scale) (void)hipFree(w->d_scale);
    if (w->d_bias) (void)hipFree(w->d_bias);
    delete w;
    return 0;
}

extern "C" int nncase_hip_w8a16_prepack(nncase_hip_ctx_t *ctx, const int8_t *w_host, const float *scale_host,
                                        const float *bias_host, int32_t k, int32_t n, nncase_hip_w8a16_t **out) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, w_host && scale_host && out, -EINVAL, "w8a16_prepack: null argument");
    *out = nullptr;
    NNHIP_REQUIRE(ctx, k > 0 && n > 0 && k % 64 == 0 && n % 16 == 0, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "w8a16_prepack: k = %d must be a multiple of 64 and n = %d a multiple of 16", k, n);
    nncase_hip_w8a16 *w = new (std::nothrow) nncase_hip_w8a16();
    NNHIP_REQUIRE(ctx, w, -ENOMEM, "w8a16_prepack: out of host memory");
    w->k = k, w->n = n, w->ntiles = n / 16, w->ksteps = k / 64;
    const size_t bytes = (size_t)n * k;
    std::vector<uint8_t> packed(bytes);
    for (int t = 0; t < w->ntiles; t++)
        for (int ks = 0; ks < w->ksteps; ks++)
            for (int l = 0; l < 64; l++) {
                const int i = l & 15, kg = l >> 4;
                const int8_t *src = w_host + (size_t)(t * 16 + i) * k + ks * 64 + kg * 16;
                uint8_t *dst = &packed[(((size_t)t * w->ksteps + ks) * 64 + l) * 16];
                for (int b = 0; b < 16; b++) dst[b] = (uint8_t)src[b] ^ 0x80u;
            }
    auto cleanup = [&](int rc) {
        (void)nncase_hip_w8a16_destroy(ctx, w);
        return rc;
    };
    if (hipMalloc(&w->d_packed, bytes) != hipSuccess || hipMalloc((void **)&w->d_scale, sizeof(float) * n) != hipSuccess)
        return cleanup(fail(ctx, -ENOMEM, "w8a16_prepack: out of device memory"));
    if (bias_host && hipMalloc((void **)&w->d_bias, sizeof(float) * n) != hipSuccess)
        return cleanup(fail(ctx, -ENOMEM, "w8a16_prepack: out of device memory"));
    if (hipMemcpy(w->d_packed, packed.data(), bytes, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(w->d_scale, scale_host, sizeof(float) * n, hipMemcpyHostToDevice) != hipSuccess ||
        (bias_host && hipMemcpy(w->d_bias, bias_host, sizeof(float) * n, hipMemcpyHostToDevice) != hipSuccess))
        return cleanup(fail(ctx, -EFAULT, "w8a16_prepack: upload failed"));
    *out = w;
    return 0;
}

static W8Product w8_product(const nncase_hip_w8a16_t *w, int m, bool glu) { return W8Product{m, w->k, glu ? w->ntiles / 2 : w->ntiles, glu}; }

// Whether the q / k / v projection of this geometry can rotate and append in its own epilogue (else the caller runs
// the projection and the rope kernel one after the other).
static bool rope_epilogue_fits(const nncase_hip_ctx_t *ctx, const nncase_hip_w8a16_t *w, int m, const RopeArgs &r) {
    return rows_take_split(w8_product(w, m, false), ctx->compute_units) && r.d % 32 == 0 && w->n == (r.hq + 2 * r.hkv) * r.d && w->k <= 1024;
}

template <int G, int KS, bool NORM, int R, int PIECES, bool ROPE>
static int launch_tile(nncase_hip_ctx_t *ctx, const GemmArgs &a, int tiles) {
    const size_t lds = R > 0 ? (size_t)16 * rows_in_lds_pitch(a.k) : 0;
    if (lds + G * kGemmWaves * 4 * kRedPitch * sizeof(float) > 48 * 1024) NNHIP_HIP(ctx, (raise_dynamic_lds<w8a16_tile_kernel<G, KS, NORM, R, PIECES, ROPE>>(ctx->device, 96 * 1024)));
    hipLaunchKernelGGL((w8a16_tile_kernel<G, KS, NORM, R, PIECES, ROPE>), dim3(tiles, (a.m + 15) / 16), dim3(kGemmThreads), lds, ctx->stream, a);
    NNHIP_LAUNCH_CHECK(ctx, "w8a16_tile_kernel");
    return 0;
}
// (kernels for the k-steps that a wave has: what is asked for past its share is read again)
template <int G, bool NORM, bool ROPE> static int launch_tile_rows(nncase_hip_ctx_t *ctx, const GemmArgs &a, int tiles) {
    auto by_rows = [&](auto steps) { // (a row per wave, or two)
        constexpr int S = decltype(steps)::value;
        return a.m <= kGemmWaves ? launch_tile<G, S, NORM, 1, S, ROPE>(ctx, a, tiles) : launch_tile<G, S, NORM, 2, S, ROPE>(ctx, a, tiles);
    };
    static_assert(kRowsPieces == 4, "a piece of a row is a k-step of each wave");
    if (a.k <= 512) return by_rows(std::integral_constant<int, 1>());
    if (a.k <= 1024) return by_rows(std::integral_constant<int, 2>());
    if constexpr (ROPE) return -EINVAL; // (see rope_epilogue_fits)
    else return a.k <= 1536 ? by_rows(std::integral_constant<int, 3>()) : by_rows(std::integral_constant<int, 4>());
}
template <int G> static int launch_tile_long(nncase_hip_ctx_t *ctx, const GemmArgs &a, int tiles) {
    const int share = (a.ksteps + kGemmWaves - 1) / kGemmWaves;
    if (share <= 4) return launch_tile<G, 4, false, 0, 0, false>(ctx, a, tiles);
    if (share <= 5) return launch_tile<G, 5, false, 0, 0, false>(ctx, a, tiles);
    if (share <= 6) return launch_tile<G, 6, false, 0, 0, false>(ctx, a, tiles);
    if (share <= 8) return launch_tile<G, 8, false, 0, 0, false>(ctx, a, tiles);
    return launch_tile<G, kTileMaxK / 512, false, 0, 0, false>(ctx, a, tiles);
}

static int launch_w8a16_gemm(nncase_hip_ctx_t *ctx, const void *a_dev, const nncase_hip_w8a16_t *w, void *out_dev, int32_t m,
                             int32_t mode, const void *residual_dev, int32_t out_dtype, const void *ln_weight_dev, float ln_eps,
                             const RopeArgs *rope = nullptr) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, a_dev && w && out_dev, -EINVAL, "w8a16_gemm: null argument");
    NNHIP_REQUIRE(ctx, (reinterpret_cast<uintptr_t>(ln_weight_dev) & 15u) == 0, -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION,
                  "w8a16_gemm: normalisation weights must be 16-byte aligned");
    NNHIP_REQUIRE(ctx, m > 0 && m <= kMaxRows, -NNCASE_HIP_ERR_SHAPE_MISMATCH, "w8a16_gemm: %d token rows (1..%d supported)", m, kMaxRows);
    NNHIP_REQUIRE(ctx, mode == NNCASE_HIP_GEMM_PLAIN || mode == NNCASE_HIP_GEMM_SWIGLU, -EINVAL, "w8a16_gemm: unknown mode %d", mode);
    NNHIP_REQUIRE(ctx, out_dtype == NNCASE_HIP_DT_F16 || out_dtype == NNCASE_HIP_DT_F32, -NNCASE_HIP_ERR_DATATYPE_MISMATCH,
                  "w8a16_gemm: output type 0x%x", out_dtype);
    NNHIP_REQUIRE(ctx, mode != NNCASE_HIP_GEMM_SWIGLU || w->ntiles % 2 == 0, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "w8a16_gemm: SwiGLU needs gate and up halves of equal size");
    NNHIP_REQUIRE(ctx, ((reinterpret_cast<uintptr_t>(a_dev) | reinterpret_cast<uintptr_t>(out_dev)) & 15u) == 0,
                  -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION, "w8a16_gemm: buffers must be 16-byte aligned");
    NNHIP_REQUIRE(ctx, (reinterpret_cast<uintptr_t>(residual_dev) & 7u) == 0, -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION,
                  "w8a16_gemm: the residual must be 8-byte aligned");
    GemmArgs a;
    memset(&a, 0, sizeof(a));
    a.a = (const uint16_t *)a_dev;
    a.w = (const lu32x4 *)w->d_packed;
    a.scale = w->d_scale, a.bias = w->d_bias;
    a.residual = (const uint16_t *)residual_dev;
    a.ln_w = (const uint16_t *)ln_weight_dev;
    a.ln_eps = ln_eps;
    a.out = out_dev;
    a.m = m, a.k = w->k, a.ksteps = w->ksteps, a.out_f32 = out_dtype == NNCASE_HIP_DT_F32;
    const int out_tiles = mode == NNCASE_HIP_GEMM_SWIGLU ? w->ntiles / 2 : w->ntiles;
    a.up_tile_offset = out_tiles;
    a.n_out = out_tiles * 16;
    const int mt = (m + 15) / 16;
    const bool glu = mode == NNCASE_HIP_GEMM_SWIGLU;
    if (rope) { // (the caller has checked rope_epilogue_fits) a block per pair of tiles d / 2 channels apart
        a.rope = *rope;
        a.up_tile_offset = rope->d / 32;
        return a.ln_w ? launch_tile_rows<2, true, true>(ctx, a, w->ntiles / 2) : launch_tile_rows<2, false, true>(ctx, a, w->ntiles / 2);
    }
    const W8Product product = w8_product(w, m, glu);
    const W8Form form = choose_w8_form(product, a.ln_w != nullptr, ctx->compute_units);
    if (form == W8Form::kTileLong) return glu ? launch_tile_long<2>(ctx, a, out_tiles) : launch_tile_long<1>(ctx, a, out_tiles);
    if (form == W8Form::kTile) {
        if (a.ln_w) return glu ? launch_tile_rows<2, true, false>(ctx, a, out_tiles) : launch_tile_rows<1, true, false>(ctx, a, out_tiles);
        return glu ? launch_tile_rows<2, false, false>(ctx, a, out_tiles) : launch_tile_rows<1, false, false>(ctx, a, out_tiles);
    }
    if (form == W8Form::kSmallTile) {
        hipLaunchKernelGGL((w8a16_small_tile_kernel<kTileMaxK / 1024>), dim3(out_tiles * 2, (m + 7) / 8), dim3(kGemmThreads), 0, ctx->stream, a);
        NNHIP_LAUNCH_CHECK(ctx, "w8a16_small_tile_kernel");
        return 0;
    }
    const bool split = form == W8Form::kSplit;
    const bool paired = split && sums_in_pairs(product, ctx->compute_units);
    const dim3 grid(split ? out_tiles : (out_tiles + kGemmWaves - 1) / kGemmWaves), block(kGemmThreads);
    if (form == W8Form::kRowsInLds) {
        const int mt_built = mt <= 1 ? 1 : (mt == 2 ? 2 : 4);
        const size_t rows_lds = (size_t)mt_built * 16 * rows_in_lds_pitch(w->k);
        const bool short_rows = w->k <= 1024; // rows of two 512-element pieces (a lane keeps a row's pieces in registers)
        // (at most two blocks per compute unit, each walking several groups of eight tiles: what a block repeats -- the
        // rows' trip and their normalisation -- is then paid twice per compute unit, not once per group)
        const dim3 rgrid(std::min((out_tiles + kGemmWaves - 1) / kGemmWaves, 2 * ctx->compute_units)), rblock(kGemmThreads);
        // (eight k-steps of weights per request: asking for a whole 14-step reduction at once costs registers that the
        // vocabulary head needs for occupancy -- 50.7 against 43.9 us when it still ran as 1187 one-group blocks)
#define NNHIP_ROWS_LAUNCH_KB(MTV, GV, KBV, PV)                                                                                 \
    do {                                                                                                                       \
        if (rows_lds > 47 * 1024) NNHIP_HIP(ctx, (raise_dynamic_lds<w8a16_gemm_rows_in_lds_kernel<MTV, GV, KBV, PV>>(ctx->device, 128 * 1024))); \
        hipLaunchKernelGGL((w8a16_gemm_rows_in_lds_kernel<MTV, GV, KBV, PV>), rgrid, rblock, rows_lds, ctx->stream, a); \
    } while (0)
#define NNHIP_ROWS_LAUNCH(MTV, GV)                                                                                             \
    do {                                                                                                                       \
        if (short_rows) NNHIP_ROWS_LAUNCH_KB(MTV, GV, kRowsBatch, 2);                                                          \
        else NNHIP_ROWS_LAUNCH_KB(MTV, GV, kRowsBatch, kRowsPieces);                                                           \
    } while (0)
        if (glu) {
            if (mt_built == 1) NNHIP_ROWS_LAUNCH(1, 2);
            else if (mt_built == 2) NNHIP_ROWS_LAUNCH(2, 2);
            else NNHIP_ROWS_LAUNCH(4, 2);
        } else {
            if (mt_built == 1) NNHIP_ROWS_LAUNCH(1, 1);
            else if (mt_built == 2) NNHIP_ROWS_LAUNCH(2, 1);
            else NNHIP_ROWS_LAUNCH(4, 1);
        }
#undef NNHIP_ROWS_LAUNCH_KB
#undef NNHIP_ROWS_LAUNCH
        NNHIP_LAUNCH_CHECK(ctx, "w8a16_gemm_rows_in_lds_kernel");
        return 0;
    }
#define NNHIP_GEMM_LAUNCH(MTV)                                                                                                 \
    do {                                                                                                                       \
        if (glu && split) hipLaunchKernelGGL((w8a16_gemm_kernel<MTV, 2, true>), grid, block, 0, ctx->stream, a);              \
        else if (glu) hipLaunchKernelGGL((w8a16_gemm_kernel<MTV, 2, false>), grid, block, 0, ctx->stream, a);                 \
        else if (split) hipLaunchKernelGGL((w8a16_gemm_kernel<MTV, 1, true>), grid, block, 0, ctx->stream, a);                \
        else hipLaunchKernelGGL((w8a16_gemm_kernel<MTV, 1, false>), grid, block, 0, ctx->stream, a);                          \
    } while (0)
    if (paired) hipLaunchKernelGGL((w8a16_gemm_kernel<1, 1, true, true>), grid, block, 0, ctx->stream, a); // (one token tile)
    else if (mt == 1) NNHIP_GEMM_LAUNCH(1);
    else if (mt == 2) NNHIP_GEMM_LAUNCH(2);
    else NNHIP_GEMM_LAUNCH(4);
#undef NNHIP_GEMM_LAUNCH
    NNHIP_LAUNCH_CHECK(ctx, "w8a16_gemm_kernel");
    return 0;
}

bool nnhip::w8a16_weight_fetch(const nncase_hip_ctx *ctx, const nncase_hip_w8a16_t *w, int m, int mode, bool normalises,
                               const nncase_hip_paged_attn_args_t *rope, WeightFetch *f) {
    const bool glu = mode == NNCASE_HIP_GEMM_SWIGLU;
    f->packed = w->d_packed;
    f->steps = (uint32_t)w->ksteps;
    if (rope) {
        RopeArgs r;
        memset(&r, 0, sizeof(r));
        r.hq = rope->num_q_heads, r.hkv = rope->num_kv_heads, r.d = rope->head_dim;
        if (rope_epilogue_fits(ctx, w, m, r)) {
            f->blocks = (uint32_t)w->ntiles / 2, f->off = (uint32_t)r.d / 32, f->per_block = 2;
            return true;
        }
    }
    const W8Form form = choose_w8_form(w8_product(w, m, glu), normalises, ctx->compute_units);
    if (form == W8Form::kRowsInLds || form == W8Form::kPerWave) return false;
    // (kSmallTile: two blocks a tile, on the die that a block per tile would be on)
    f->blocks = f->off = (uint32_t)(glu ? w->ntiles / 2 : w->ntiles);
    f->per_block = glu ? 2 : 1;
    return true;
}

extern "C" int nncase_hip_w8a16_gemm(nncase_hip_ctx_t *ctx, const void *a_dev, const nncase_hip_w8a16_t *w, void *out_dev,
                                     int32_t m, int32_t mode, const void *residual_dev, int32_t out_dtype) {
    return launch_w8a16_gemm(ctx, a_dev, w, out_dev, m, mode, residual_dev, out_dtype, nullptr, 0.f);
}

extern "C" int nncase_hip_rmsnorm_w8a16_gemm(nncase_hip_ctx_t *ctx, const void *x_dev, const void *ln_weight_dev, float eps,
                                             const nncase_hip_w8a16_t *w, void *out_dev, int32_t m, int32_t mode,
                                             const void *residual_dev, int32_t out_dtype) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, ln_weight_dev, -EINVAL, "rmsnorm_w8a16_gemm: null normalisation weights");
    return launch_w8a16_gemm(ctx, x_dev, w, out_dev, m, mode, residual_dev, out_dtype, ln_weight_dev, eps);
}

extern "C" int nncase_hip_rmsnorm_f16(nncase_hip_ctx_t *ctx, const void *x_dev, const void *weight_dev, void *out_dev, int32_t rows,
                                      int32_t hidden, float eps) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, x_dev && weight_dev && out_dev && rows > 0 && hidden > 0, -EINVAL, "rmsnorm_f16: bad argument");
    hipLaunchKernelGGL(rmsnorm_f16_kernel, dim3((rows + 3) / 4), dim3(kLlmThreads), 0, ctx->stream, (const __half *)x_dev,
                       (const __half *)weight_dev, (__half *)out_dev, rows, hidden, eps);
    NNHIP_LAUNCH_CHECK(ctx, "rmsnorm_f16_kernel");
    return 0;
}

static int make_rope_args(nncase_hip_ctx_t *ctx, const void *qkv_dev, void *q_out_dev, void *k_cache_dev, void *v_cache_dev,
                          const int32_t *block_table_dev, const int32_t *ctx_lens_dev, const nncase_hip_paged_attn_args_t *p,
                          float rope_theta, RopeArgs *out) {
    NNHIP_REQUIRE(ctx, q_out_dev && k_cache_dev && v_cache_dev && block_table_dev && ctx_lens_dev && p, -EINVAL,
                  "rope_kv_append: null argument");
    NNHIP_REQUIRE(ctx, p->batch > 0 && p->num_q_heads > 0 && p->num_kv_heads > 0 && p->head_dim > 0 && p->head_dim % 2 == 0 &&
                           p->block_size > 0 && p->max_blocks_per_seq > 0 && p->num_blocks > 0 && rope_theta > 0.f,
                  -EINVAL, "rope_kv_append: bad geometry");
    RopeArgs &a = *out;
    a.qkv = (const __half *)qkv_dev, a.q_out = (__half *)q_out_dev, a.k_cache = (__half *)k_cache_dev, a.v_cache = (__half *)v_cache_dev;
    a.block_table = block_table_dev, a.ctx_lens = ctx_lens_dev;
    a.batch = p->batch, a.hq = p->num_q_heads, a.hkv = p->num_kv_heads, a.d = p->head_dim, a.block_size = p->block_size;
    a.max_blocks = p->max_blocks_per_seq, a.num_blocks = p->num_blocks, a.theta = rope_theta;
    return 0;
}

extern "C" int nncase_hip_rope_kv_append(nncase_hip_ctx_t *ctx, const void *qkv_dev, void *q_out_dev, void *k_cache_dev,
                                         void *v_cache_dev, const int32_t *block_table_dev, const int32_t *ctx_lens_dev,
                                         const nncase_hip_paged_attn_args_t *p, float rope_theta) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, qkv_dev, -EINVAL, "rope_kv_append: null argument");
    RopeArgs a;
    const int rc = make_rope_args(ctx, qkv_dev, q_out_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, p, rope_theta, &a);
    if (rc) return rc;
    const int64_t total = (int64_t)a.batch * (a.hq + 2 * a.hkv) * (a.d / 2);
    NNHIP_REQUIRE(ctx, total < ((int64_t)1 << 31), -EINVAL, "rope_kv_append: too large");
    hipLaunchKernelGGL(rope_append_kernel, dim3((unsigned)((total + kLlmThreads - 1) / kLlmThreads)), dim3(kLlmThreads), 0, ctx->stream, a);
    NNHIP_LAUNCH_CHECK(ctx, "rope_append_kernel");
    return 0;
}

extern "C" int nncase_hip_w8a16_gemm_rope_kv_append(nncase_hip_ctx_t *ctx, const void *x_dev, const void *ln_weight_dev, float eps,
                                                    const nncase_hip_w8a16_t *w, void *qkv_dev, void *q_out_dev, void *k_cache_dev,
                                                    void *v_cache_dev, const int32_t *block_table_dev, const int32_t *ctx_lens_dev,
                                                    const nncase_hip_paged_attn_args_t *p, float rope_theta) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, x_dev && w && qkv_dev, -EINVAL, "w8a16_gemm_rope_kv_append: null argument");
    RopeArgs r;
    int rc = make_rope_args(ctx, qkv_dev, q_out_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, p, rope_theta, &r);
    if (rc) return rc;
    NNHIP_REQUIRE(ctx, w->n == (r.hq + 2 * r.hkv) * r.d, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "w8a16_gemm_rope_kv_append: the matrix has %d output channels, the heads need %d", w->n, (r.hq + 2 * r.hkv) * r.d);
    if (rope_epilogue_fits(ctx, w, r.batch, r))
        return launch_w8a16_gemm(ctx, x_dev, w, qkv_dev, r.batch, NNCASE_HIP_GEMM_PLAIN, nullptr, NNCASE_HIP_DT_F16, ln_weight_dev, eps, &r);
    // other geometries: the projection into qkv_dev, then the rope kernel (the same values: the epilogue above rounds to
    // fp16 where this path stores fp16)
    rc = launch_w8a16_gemm(ctx, x_dev, w, qkv_dev, r.batch, NNCASE_HIP_GEMM_PLAIN, nullptr, NNCASE_HIP_DT_F16, ln_weight_dev, eps);
    if (rc) return rc;
    return nncase_hip_rope_kv_append(ctx, qkv_dev, q_out_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, p, rope_theta);
}

extern "C" int nncase_hip_argmax_f32(nncase_hip_ctx_t *ctx, const float *x_dev, int32_t *out_dev, int32_t rows, int32_t cols) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, x_dev && out_dev && rows > 0 && cols > 0, -EINVAL, "argmax_f32: bad argument");
    hipLaunchKernelGGL(argmax_f32_kernel, dim3(rows), dim3(kArgmaxThreads), 0, ctx->stream, x_dev, out_dev, cols);
    NNHIP_LAUNCH_CHECK(ctx, "argmax_f32_kernel");
    return 0;
}

extern "C" int nncase_hip_embedding_f16(nncase_hip_ctx_t *ctx, const void *table_dev, const int32_t *ids_dev, void *out_dev,
                                        int32_t rows, int32_t hidden, int32_t vocab) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, table_dev && ids_dev && out_dev && rows > 0 && hidden > 0 && vocab > 0, -EINVAL, "embedding_f16: bad argument");
    const int64_t total = (int64_t)rows * hidden;
    NNHIP_REQUIRE(ctx, total < ((int64_t)1 << 31), -EINVAL, "embedding_f16: too large");
    hipLaunchKernelGGL(embed_f16_kernel, dim3((unsigned)((total + kLlmThreads - 1) / kLlmThreads)), dim3(kLlmThreads), 0, ctx->stream,
                       (const __half *)table_dev, ids_dev, (__half *)out_dev, rows, hidden, vocab);
    NNHIP_LAUNCH_CHECK(ctx, "embed_f16_kernel");
    return 0;
}

extern "C" int nncase_hip_add_i32(nncase_hip_ctx_t *ctx, int32_t *x_dev, int32_t count, int32_t delta) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, x_dev && count > 0, -EINVAL, "add_i32: bad argument");
    hipLaunchKernelGGL(add_i32_kernel, dim3((count + 255) / 256), dim3(256), 0, ctx->stream, x_dev, count, delta);
    NNHIP_LAUNCH_CHECK(ctx, "add_i32_kernel");
    return 0;
}
