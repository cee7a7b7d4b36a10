// Paged-attention decode: one query token per sequence against a block-paged
// fp16 KV cache.  HBM-bound (every cached K and V element is read once per
// step, ~7 flop per byte), so the kernel is organised around the KV stream and
// keeps the arithmetic on the matrix cores:
//
//   grid = (sequences x kv heads, splits).  A block owns one kv head of one
//   sequence and a contiguous range of cached tokens, and serves ALL query
//   heads that share the kv head, so K and V cross the memory system once
//   however many query heads there are (GQA).  Each of its waves owns a
//   contiguous run of 16-token tiles and issues the loads of ALL its K and V
//   tiles before any arithmetic (up to 16 KiB of K + 16 KiB of V in flight per wave).
//
//   Logits: S^T[token, head] = K[token, :] . Q^T[:, head] with K rows as the
//   MFMA A operand (one 16-byte load per lane straight from the cache) and the
//   query heads, padded to 16, as B.  The accumulator layout of S^T (lane =
//   head, 4 consecutive tokens per lane) IS the A-operand layout of the
//   product P.V, so probabilities never move between lanes.  V is cached
//   d-major ([block][kv head][d][token]) so that a lane's B operand
//   (consecutive tokens of one d) is one load.  P is split into two fp16
//   terms (p = hi + lo), which keeps the P.V product at fp32-level accuracy.
//
//   Every wave keeps its own (max, sum, unnormalised output); the block merges
//   its waves through LDS and writes one partial per split.  The block
//   that finishes last for a (sequence, kv head) - found with one atomic
//   counter per pair, which it resets for the next call - merges the splits
//   and writes the output, so there is a single launch per call.
#include "attn_rules.hpp"
#include "common.hpp"

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace nnhip {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t au32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t au32x2 __attribute__((ext_vector_type(2)));

constexpr int kAttnHeads = 16; // query heads per kv head, padded to the MFMA tile
constexpr float kLog2e = 1.4426950408889634f;
// Probabilities enter P.V times 2^14, up to 16 384: their second fp16 term ends at 2^-24, an eighth of a millionth of a probability of
// a half, and the small ones of a long run lost bits there.
constexpr float kProbScale = 16384.f;

// Keys and values of this many bytes are not found in any cache when the next step comes back to them (the memory side's holds
// 256 MiB): values are then read past the caches, 6.8 TB/s against 6.0 (48 sequences of up to 6000, 8 heads of 128: 135.2 -> 119.6
// us; of 268 MB, half of it in use: 30.8 -> 33.1).  By the capacity, whatever is in use of it: of 805 MB, 48 sequences of 300 / 700 /
// 1000 / 2000 / 8192 tokens 13.3 -> 12.4, 23.4 -> 24.6, 31.2 -> 32.7, 65.3 -> 56.9, 280 -> 254.  Not the keys, whose loads take 64 of a
// line's 128 bytes at a time: they are read twice then (133.9).
constexpr int64_t kStreamedBytes = 512000000;
constexpr int kStreamWaves = 4;

struct AttnArgs {
    const uint16_t *q, *k_cache, *v_cache;
    const int32_t *block_table, *ctx_lens;
    float *part_o;  // [batch][q heads][splits][D], unnormalised, relative to the split's max
    float *part_ml; // [batch][q heads][splits][2]: max of (logit * scale * log2 e), sum of 2^(. - max)
    uint32_t *done; // [batch][kv heads] blocks finished; zero between calls
    void *out;
    int batch, hq, hkv, group, d, block_size, max_blocks, num_blocks, splits, split_tokens, len_offset;
    FastDiv d_block, d_hkv;
    float scale_log2e;
    int out_f16;
    AttnRunRule rule; // (this and the next of the kernel that goes through its split)
    int rotate;       // a mask on the split: by how many pairs its blocks are moved on
};
// A launch that fetches weights beside its own work.  (A type of its own, and with it kernels of their own: the longer arguments and
// the branch cost a launch 1.8 %, 8.69 -> 8.85 us at 24 x 64 x 2820 tokens.)
struct AttnFetchArgs : AttnArgs {
    WeightFetches fetch;
};

// two neighbouring floats at an 8-byte aligned address
__device__ __forceinline__ uint64_t coherent_load2(const float *p) {
    return __hip_atomic_load(reinterpret_cast<const uint64_t *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void coherent_store2(float *p, float v0, float v1) {
    __hip_atomic_store(reinterpret_cast<uint64_t *>(p), (uint64_t)__float_as_uint(v0) | (uint64_t)__float_as_uint(v1) << 32, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
// outputs i and i + 1 (i even)
__device__ __forceinline__ void store_pair(const AttnArgs &a, size_t i, float v0, float v1) {
    if (a.out_f16) *reinterpret_cast<__half2 *>(reinterpret_cast<__half *>(a.out) + i) = __halves2half2(__float2half_rn(v0), __float2half_rn(v1));
    else *reinterpret_cast<float2 *>(reinterpret_cast<float *>(a.out) + i) = float2{v0, v1};
}

// bytes of dynamic LDS of a block of W waves: the waves' unnormalised outputs, maxima and sums
constexpr size_t attn_lds_bytes(int d, int waves) { return (size_t)waves * kAttnHeads * (d + 2) * sizeof(float); }

// Merges ns partials of G query heads (rows row0 + head * splits) into outputs out0 ...; every thread of the block calls it.
// A thread merges two neighbouring outputs over every GR-th run of U splits: their (max, sum) and (value, value) pairs are
// requested together, one memory round trip per GR * U splits (a trip per eight splits was 8 of the 12 us of one sequence of
// 16 000 tokens); runs combine under a running maximum, the GR partial results through LDS.
template <int D, int U>
__device__ __forceinline__ void merge_splits(const AttnArgs &a, int ns, int G, size_t row0, size_t out0, float *part, int threads) {
    const int pairs = G * D / 2;
    int GR = 1, gr = 0;
    if (U == 8) {
        while (GR < 4 && (GR + 1) * pairs <= threads && GR * U < ns) GR++;
        for (int q = 1; q < GR; q++) gr += (int)threadIdx.x >= q * pairs;
        if ((int)threadIdx.x >= GR * pairs && GR > 1) gr = GR;
    }
    for (int p0 = gr < GR ? (int)threadIdx.x - gr * pairs : pairs; p0 < pairs; p0 += threads) { // (more than one turn only with GR = 1)
        const int h = p0 * 2 / D, e = p0 * 2 % D;
        const size_t rowh = row0 + (size_t)h * a.splits;
        float m = -INFINITY, den = 0.f, n0 = 0.f, n1 = 0.f;
        for (int sp0 = gr * U; sp0 < ns; sp0 += GR * U) {
            uint64_t ml[U], vv[U];
#pragma unroll
            for (int k = 0; k < U; k++) {
                const size_t row = rowh + min(sp0 + k, ns - 1);
                ml[k] = coherent_load2(a.part_ml + row * 2);
                vv[k] = coherent_load2(a.part_o + row * D + e);
            }
            auto pm = [&](int k) { return __uint_as_float((uint32_t)ml[k]); };
            float mc = m;
#pragma unroll
            for (int k = 0; k < U; k++) mc = fmaxf(mc, pm(k)); // a repeated last split does not change the max
            const float f = __builtin_amdgcn_exp2f(m - mc);      // 0 on the first run (m = -inf)
            float s0 = 0.f, s1 = 0.f, sd = 0.f; // (the run's own sums first: one rounding of the total a run)
#pragma unroll
            for (int k = 0; k < U; k++) {
                const float w = sp0 + k < ns ? __builtin_amdgcn_exp2f(pm(k) - mc) : 0.f;
                s0 += w * __uint_as_float((uint32_t)vv[k]);
                s1 += w * __uint_as_float((uint32_t)(vv[k] >> 32));
                sd += w * __uint_as_float((uint32_t)(ml[k] >> 32));
            }
            n0 = n0 * f + s0, n1 = n1 * f + s1, den = den * f + sd;
            m = mc;
        }
        if (GR > 1) *reinterpret_cast<f32x4 *>(part + ((size_t)gr * pairs + p0) * 4) = f32x4{m, den, n0, n1};
        else store_pair(a, out0 + (size_t)h * D + e, n0 / den, n1 / den);
    }
    if (GR == 1) return;
    __syncthreads();
    for (int p0 = threadIdx.x; p0 < pairs; p0 += threads) {
        float m = part[(size_t)p0 * 4];
        for (int q = 1; q < GR; q++) m = fmaxf(m, part[((size_t)q * pairs + p0) * 4]);
        float den = 0.f, n0 = 0.f, n1 = 0.f;
        for (int q = 0; q < GR; q++) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(part + ((size_t)q * pairs + p0) * 4);
            const float w = __builtin_amdgcn_exp2f(t[0] - m);
            den += w * t[1], n0 += w * t[2], n1 += w * t[3];
        }
        store_pair(a, out0 + (size_t)p0 * 2, n0 / den, n1 / den);
    }
}

// What the blocks of the grid's second and further planes do: bring fragments of the weights that the next products read into the
// L2 of the die whose blocks will ask for them; the loads' results are dropped.  While the blocks of the first plane wait for one
// memory round trip after another, the memory would be idle: one sequence of 700 tokens, a decode layer with its 14.9 MB of
// weights fetched 24.8 -> 22.9 us.  (Fetched by the products' own launches instead, or by them too, it takes 23.7 to 26.7.)
// A wave has one batch of fragments, all of them under way at once.
constexpr int kFetchBatch = 8;
template <int W> __device__ __forceinline__ void fetch_weights(const AttnFetchArgs &a) {
    const uint32_t pairs = a.hkv * a.batch, block = ((uint32_t)blockIdx.z * a.splits + blockIdx.y) * pairs + blockIdx.x;
    const uint32_t x = block % kXcds, p = (block - pairs * a.splits) / kXcds; // (every eight consecutive blocks have one on each die)
    const uint32_t lane = threadIdx.x & 63, u0 = p * W + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), stride = (uint32_t)a.fetch.blocks * W;
    uint32_t n = 0;
    for (int i = 0; i < a.fetch.count; i++) n += fetch_fragments(a.fetch.f[i], x);
    if (p >= (uint32_t)a.fetch.blocks || u0 >= n) return;
    au32x4 v[kFetchBatch];
#pragma unroll
    for (int k = 0; k < kFetchBatch; k++) v[k] = reinterpret_cast<const au32x4 *>(fetch_address(a.fetch, x, min(u0 + k * stride, n - 1)))[lane];
#pragma unroll
    for (int k = 0; k < kFetchBatch; k++) asm volatile("" ::"v"(v[k]));
}

// The end of a block, given every wave's maximum, sum (of head j, the same in all g) and unnormalised output of the tokens that it
// went through: the waves merge through LDS, and the last block of the (sequence, kv head) to get here merges the splits.
template <int D, int W>
__device__ __forceinline__ void finish_block(const AttnArgs &a, int b, int kvh, int split, int ns, int wave, int j, int g, float m_w, float l_w,
                                             const f32x4 (&o)[D / 16]) {
    constexpr int kAttnWaves = W, kAttnThreads = W * 64, DT = D / 16;
    extern __shared__ __align__(16) float attn_smem[];
    float(*red)[kAttnHeads][D] = reinterpret_cast<float(*)[kAttnHeads][D]>(attn_smem);                            // [W][heads][D]
    float(*smax)[kAttnHeads] = reinterpret_cast<float(*)[kAttnHeads]>(attn_smem + (size_t)W * kAttnHeads * D);    // [W][heads]
    float(*ssum)[kAttnHeads] = smax + W;                                                                            // [W][heads]
    __shared__ uint32_t s_last;
    const int G = a.group;
    // ---- merge the waves ----------------------------------------------------------------
    // One barrier: the waves' outputs meet under their own maxima, and a thread takes the exponents of its head along with two
    // neighbouring columns (before, the waves scaled their outputs ahead of a second barrier and a thread took the exponents for one
    // column: one sequence of 700 tokens, 7 heads of 64 on one, 6.3 -> 5.8 us, 64 of 1000 9.65 -> 9.1, 200 of 100 with 4 of 128 14.5 ->
    // 13.5).
    if (g == 0) {
        // (never -inf, of no tokens or of logits of -inf alone: the merges take exponents relative to the largest of these.  Here it is
        // one instruction, at each exponent short contexts took up to 6 % longer: 36 sequences of 32 tokens, 16 heads on one, 5.5 -> 5.2 us)
        smax[wave][j] = fmaxf(m_w, -FLT_MAX);
        ssum[wave][j] = l_w;
    }
    // o[dt][r] belongs to head 4g + r, column dt*16 + j
#pragma unroll
    for (int r = 0; r < 4; r++)
        if (g * 4 + r < G) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++) red[wave][g * 4 + r][dt * 16 + j] = o[dt][r];
        }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * (D / 2); idx += kAttnThreads) {
        const int h = idx / (D / 2), e = idx % (D / 2) * 2;
        float m = smax[0][h];
#pragma unroll
        for (int w = 1; w < kAttnWaves; w++) m = fmaxf(m, smax[w][h]);
        float v0 = 0.f, v1 = 0.f, l = 0.f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; w++) {
            const float f = __builtin_amdgcn_exp2f(smax[w][h] - m); // 0 for a wave without tokens
            const float2 t = *reinterpret_cast<const float2 *>(&red[w][h][e]);
            v0 += t.x * f, v1 += t.y * f;
            l += ssum[w][h] * f;
        }
        if (ns == 1) { // the whole context was in this block
            store_pair(a, ((size_t)b * a.hq + kvh * G + h) * D + e, v0 / l, v1 / l);
        } else {
            const size_t row = ((size_t)b * a.hq + kvh * G + h) * a.splits + split;
            coherent_store2(a.part_o + row * D + e, v0, v1);
            if (e == 0) coherent_store2(a.part_ml + row * 2, m, l);
        }
    }
    if (ns == 1) return;

    // ---- the last block of the (sequence, kv head) to finish merges the splits -------------------
    // The partials are written and read with device-scope accesses, which go through to the
    // memory side instead of staying in the L2 of the XCD that issued them; waiting for this
    // thread's stores and then for the block makes them globally visible before the count.
    // (A device-scope fence would do the same by writing back and invalidating the whole L2,
    // once per block - an order of magnitude slower here.)
    uint32_t *done = a.done + (size_t)b * a.hkv + kvh;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0)
        s_last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(ns - 1);
    __syncthreads();
    if (!s_last) return;
    const size_t row0 = ((size_t)b * a.hq + kvh * G) * a.splits, out0 = ((size_t)b * a.hq + kvh * G) * D;
    float *const part = attn_smem; // (the waves' outputs have been read)
    if (ns <= 4) merge_splits<D, 4>(a, ns, G, row0, out0, part, kAttnThreads);
    else merge_splits<D, 8>(a, ns, G, row0, out0, part, kAttnThreads);
    if (threadIdx.x == 0) // ready for the next call on this stream
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// NT = 16-token tiles per wave (even); W = waves per block (a block owns W * NT * 16 tokens).
template <int D, int NT, int W, class Args> __global__ __launch_bounds__(W * 64, W <= 8 ? 2 : 1) void paged_attn_kernel(const Args a) {
    constexpr int kAttnWaves = W, kAttnThreads = W * 64;
    constexpr int KS = D / 32; // 32-deep steps of the logit product
    constexpr int DT = D / 16; // 16-wide column tiles of the output
    constexpr int WAVE_TOKENS = NT * 16;
    constexpr int SPLIT = kAttnWaves * WAVE_TOKENS;

    if constexpr (std::is_same_v<Args, AttnFetchArgs>)
        if (blockIdx.z != 0) { // (a branch on an argument would put its load's trip in front of the others')
            fetch_weights<W>(a);
            return;
        }
    // kv head fastest, then sequence, then split: consecutive workgroups go to different XCDs, so
    // every XCD gets the same mix of early (always present) and late (long contexts only) splits
    const int b = (int)fastdiv(blockIdx.x, a.d_hkv), kvh = (int)blockIdx.x - b * a.hkv, split = blockIdx.y;
    const int tok0 = split * SPLIT;
    const int G = a.group;
    const int lane = threadIdx.x & 63;
    // the wave index as a scalar, so that everything derived from it (tile positions, block-table
    // lookups, cache base addresses) stays on the scalar unit
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int wave_tok0 = tok0 + wave * WAVE_TOKENS;
    // The block-table entries of this wave's tiles do not depend on the context length, so they
    // are fetched together with it (one scalar-memory round trip instead of two).  A tile past
    // the end of the context may get any entry of the table; its block id is clamped into the
    // cache, its logits are masked and its V operand is zeroed.
    const int32_t *table = a.block_table + (size_t)b * a.max_blocks;
    int pbs[NT], inb[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) {
        const int tt = wave_tok0 + t * 16;
        const uint32_t lb = fastdiv((uint32_t)tt, a.d_block);
        inb[t] = tt - (int)lb * a.block_size;
        pbs[t] = table[min((int)lb, a.max_blocks - 1)];
    }
    const int ctx = min(a.ctx_lens[b] + a.len_offset, a.max_blocks * a.block_size);
    if (ctx <= 0) { // empty context: zeros, written by the first block of the pair
        if (split == 0)
            for (int idx = threadIdx.x; idx < G * D; idx += kAttnThreads) {
                const size_t oi = ((size_t)b * a.hq + kvh * G) * D + idx;
                if (a.out_f16) reinterpret_cast<__half *>(a.out)[oi] = __float2half_rn(0.f);
                else reinterpret_cast<float *>(a.out)[oi] = 0.f;
            }
        return;
    }
    if (tok0 >= ctx) return; // uniform for the block
    const int ns = (ctx + SPLIT - 1) / SPLIT; // blocks of this (sequence, kv head) that get here

    float m_w = -INFINITY, l_w = 0.f;
    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (wave_tok0 < ctx) { // uniform for the wave
        // ---- issue every load of this wave ----------------------------------------------
        // Every K and V load back to back (the block-table entries are already here: a lookup
        // between two tiles' loads would wait for the earlier tile's data as well).
        au32x4 kf[NT][KS];
        au32x2 vf[NT][DT];
        const uint32_t koff = (uint32_t)(j * D + g * 8) * 2u;            // bytes, the same for every tile
        const uint32_t voff = (uint32_t)(j * a.block_size + g * 4) * 2u;
        const size_t vstep = (size_t)a.block_size * 32;                  // 16 rows of d
#pragma unroll
        for (int t = 0; t < NT; t++) {
            // a block id outside the cache would fault; read block 0 instead (undefined result, no fault)
            const int pb = min(max(pbs[t], 0), a.num_blocks - 1);
            const size_t head_base = ((size_t)pb * a.hkv + kvh) * (size_t)a.block_size * D;
            const char *kb = reinterpret_cast<const char *>(a.k_cache) + (head_base + (size_t)inb[t] * D) * 2;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kf[t][ks] = *reinterpret_cast<const au32x4 *>(kb + ks * 64 + koff);
            const char *vb = reinterpret_cast<const char *>(a.v_cache) + (head_base + (size_t)inb[t]) * 2;
#pragma unroll
            for (int dt = 0; dt < DT; dt++) vf[t][dt] = *reinterpret_cast<const au32x2 *>(vb + dt * vstep + voff);
        }
        // query heads of the group as the B operand (columns past the group are zero)
        f16x8 qf[KS];
        {
            const uint16_t *qp = a.q + ((size_t)b * a.hq + kvh * G + min(j, G - 1)) * D + g * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                au32x4 raw = *reinterpret_cast<const au32x4 *>(qp + ks * 32);
                if (j >= G) raw = au32x4{0u, 0u, 0u, 0u};
                __builtin_memcpy(&qf[ks], &raw, 16);
            }
        }

        // keep every load above the arithmetic (the scheduler would otherwise sink the V loads
        // below the logit products to save registers, exposing a second memory round trip)
        __builtin_amdgcn_sched_barrier(0);

        // ---- logits, scaled to base-2 exponents -------------------------------------------
        float s[NT][4];
        float m_lane = -INFINITY;
#pragma unroll
        for (int t = 0; t < NT; t++) {
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                f16x8 kk;
                __builtin_memcpy(&kk, &kf[t][ks], 16);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk, qf[ks], acc, 0, 0, 0);
            }
            const int left = ctx - (wave_tok0 + t * 16 + g * 4); // valid tokens among this lane's four
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float v = acc[r] * a.scale_log2e;
                s[t][r] = r < left ? v : -INFINITY;
                m_lane = fmaxf(m_lane, s[t][r]);
            }
        }
        m_w = fmaxf(m_lane, __shfl_xor(m_lane, 16));
        m_w = fmaxf(m_w, __shfl_xor(m_w, 32)); // finite: the wave's first token is valid for every head

        // ---- probabilities and P.V, two token tiles per 16x16x32 product ----------------------
        float l_lane = 0.f;
#pragma unroll
        for (int t = 0; t < NT; t += 2) {
            f16x8 ph, pl;
            uint32_t keep[2][2];
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int left = ctx - (wave_tok0 + (t + u) * 16 + g * 4);
                keep[u][0] = (left > 0 ? 0x0000ffffu : 0u) | (left > 1 ? 0xffff0000u : 0u);
                keep[u][1] = (left > 2 ? 0x0000ffffu : 0u) | (left > 3 ? 0xffff0000u : 0u);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = __builtin_amdgcn_exp2f(s[t + u][r] - m_w);
                    l_lane += p;
                    const _Float16 hi = (_Float16)p;
                    ph[u * 4 + r] = hi;
                    pl[u * 4 + r] = (_Float16)(p - (float)hi);
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                // k slot (g, e): token 4g + e of tile t for e < 4, of tile t+1 otherwise - the same in both operands
                const au32x4 raw = au32x4{vf[t][dt].x & keep[0][0], vf[t][dt].y & keep[0][1],
                                          vf[t + 1][dt].x & keep[1][0], vf[t + 1][dt].y & keep[1][1]};
                f16x8 vv;
                __builtin_memcpy(&vv, &raw, 16);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, vv, o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, vv, o[dt], 0, 0, 0);
            }
        }
        l_w = l_lane + __shfl_xor(l_lane, 16);
        l_w += __shfl_xor(l_w, 32);
    }

    finish_block<D, W>(a, b, kvh, split, ns, wave, j, g, m_w, l_w, o);
}

// Tokens per split, chosen from the lengths of all sequences (at most 256): the same in every block.  `first`: the lane's sequence's.
// (The capacity says nothing of a server's contexts, whose cache holds the longest that the model takes.  With splits by the capacity
// 32 pairs of 1000 / 3400 tokens took 13.7 / 29.4 us in one of 16 384, and take 9.3 / 15.3; full ones 49.8 -> 50.1, 300 tokens 7.5 -> 7.7.
// A few shapes whose lengths are spread evenly up to the capacity lost: 32 pairs of one head 34.5 -> 36.9, 48 of four 29.0 -> 31.0, where
// the blocks without work stay a little longer and more of those with work share a compute unit.)
__device__ __forceinline__ int run_of_launch(const AttnArgs &a, int lane, int capacity, int32_t first) {
    uint32_t total = 0, longest = 0;
    auto add = [&](int i, int32_t len) __attribute__((always_inline)) {
        const uint32_t n = (uint32_t)max(min(len + a.len_offset, capacity), 0);
        total += i < a.batch ? n : 0, longest = max(longest, n);
    };
    add(lane, first);
    if (a.batch > 64) {
        int32_t more[3];
#pragma unroll
        for (int k = 0; k < 3; k++) more[k] = a.ctx_lens[min(lane + 64 * (k + 1), a.batch - 1)];
#pragma unroll
        for (int k = 0; k < 3; k++) add(lane + 64 * (k + 1), more[k]);
    }
#define NNHIP_STEP(CTRL, ROWS)                                                                  \
    total += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)total, CTRL, ROWS, 0xf, false); \
    longest = max(longest, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)longest, CTRL, ROWS, 0xf, false));
    NNHIP_STEP(0x111, 0xf) NNHIP_STEP(0x112, 0xf) NNHIP_STEP(0x114, 0xf) NNHIP_STEP(0x118, 0xf) // row_shr:1, 2, 4, 8
    NNHIP_STEP(0x142, 0xa) NNHIP_STEP(0x143, 0xc)                                               // row_bcast:15, 31
#undef NNHIP_STEP
    return attn_run(a.rule, (uint32_t)__builtin_amdgcn_readlane((int)longest, 63), (uint32_t)__builtin_amdgcn_readlane((int)total, 63));
}

// A wave goes through its share of the split 32 tokens at a time (the block's waves in turn: a split that the context ends in is
// shared by all of them), under a running maximum.  The next 32 keys are requested as soon as these have met the queries, the next
// values when these have met the probabilities, so the memory is never waited for with nothing under way, and what a block does once
// -- lengths, queries, the merge of its waves, the partials and the count -- is paid once per split instead of once per 128 to 512
// tokens.  Bound by the memory from some 50 MB on: 48 sequences of up to 6000 tokens, 8 heads of 128, 146.7 -> 125.7 us (5.4 TB/s).
template <int D, int W, bool NT, bool BY_LENS, class Args> __global__ __launch_bounds__(W * 64, 3) void paged_attn_stream_kernel(const Args a) {
    constexpr int KS = D / 32, DT = D / 16;
    if constexpr (std::is_same_v<Args, AttnFetchArgs>)
        if (blockIdx.z != 0) { // (a branch on an argument would put its load's trip in front of the others')
            fetch_weights<W>(a);
            return;
        }
    const int split = blockIdx.y;
    int pair = blockIdx.x;
    if (BY_LENS) {
        pair += split & a.rotate;
        if (pair >= a.batch * a.hkv) pair -= a.batch * a.hkv;
    }
    const int b = (int)fastdiv((uint32_t)pair, a.d_hkv), kvh = pair - b * a.hkv;
    const int G = a.group;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    const int32_t *table = a.block_table + (size_t)b * a.max_blocks;
    struct Place {
        int pb[2], in_block[2];
    };
    auto look_up = [&](int tok) {
        Place p;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint32_t lb = fastdiv((uint32_t)(tok + u * 16), a.d_block);
            p.in_block[u] = tok + u * 16 - (int)lb * a.block_size;
            p.pb[u] = table[min((int)lb, a.max_blocks - 1)]; // (a tile past the context: any entry, masked below)
        }
        return p;
    };
    // Every length, the block's own and its first pages in one trip (the pages as for splits of split_tokens: right for the first
    // split, and for all where the contexts fill the cache).
    int32_t first_len = 0;
    if (BY_LENS) {
        first_len = a.ctx_lens[min(lane, a.batch - 1)];
        __builtin_amdgcn_sched_barrier(0);
    }
    int tok0 = split * a.split_tokens, run = a.split_tokens;
    Place at = look_up(tok0 + wave * 32);
    const int capacity = a.max_blocks * a.block_size, ctx = min(a.ctx_lens[b] + a.len_offset, capacity);
    if (BY_LENS) {
        __builtin_amdgcn_sched_barrier(0); // (all requested above the wait for the lengths)
        run = run_of_launch(a, lane, capacity, first_len);
    }
    if (ctx <= 0) { // empty context: zeros, written by the first block of the pair
        if (split == 0)
            for (int idx = threadIdx.x; idx < G * D; idx += W * 64) {
                const size_t oi = ((size_t)b * a.hq + kvh * G) * D + idx;
                if (a.out_f16) reinterpret_cast<__half *>(a.out)[oi] = __float2half_rn(0.f);
                else reinterpret_cast<float *>(a.out)[oi] = 0.f;
            }
        return;
    }
    if (split * run >= ctx) return; // uniform for the block
    if (BY_LENS && split > 0 && run != a.split_tokens) {
        tok0 = split * run;
        at = look_up(tok0 + wave * 32);
    }
    int tok = tok0 + wave * 32;
    const int end = min(ctx, tok0 + run);

    // The 32 tokens are dealt to the products so that a lane's eight of P.V, (g, e), are eight neighbours, 8 g + e: one 16-byte load of
    // values.  Row 4 g + r of the u-th logit product is token 8 g + 4 u + r, so its rows come from both tiles.
    const uint32_t koff = (uint32_t)(((j >> 2 & 1) * 8 + (j & 3)) * D + g * 8) * 2u, voff = (uint32_t)(j * a.block_size + (g & 1) * 8) * 2u;
    const size_t vstep = (size_t)a.block_size * 32;
    au32x4 kf[2][KS], vf[DT];
    auto head_base = [&](int pb) { // a block id outside the cache would fault; read block 0 instead (undefined result, no fault)
        return ((size_t)min(max(pb, 0), a.num_blocks - 1) * a.hkv + kvh) * (size_t)a.block_size * D;
    };
    auto request_keys = [&](const Place &p) {
        const size_t b0 = head_base(p.pb[0]) + (size_t)p.in_block[0] * D, b1 = head_base(p.pb[1]) + (size_t)p.in_block[1] * D;
        const char *kb = reinterpret_cast<const char *>(a.k_cache) + (j < 8 ? b0 : b1) * 2 + koff;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int ks = 0; ks < KS; ks++) kf[u][ks] = *reinterpret_cast<const au32x4 *>(kb + u * (4 * D * 2) + ks * 64);
    };
    auto request_values = [&](const Place &p) {
        const size_t b0 = head_base(p.pb[0]) + (size_t)p.in_block[0], b1 = head_base(p.pb[1]) + (size_t)p.in_block[1];
        const char *vb = reinterpret_cast<const char *>(a.v_cache) + (g < 2 ? b0 : b1) * 2 + voff;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const au32x4 *const at = reinterpret_cast<const au32x4 *>(vb + dt * vstep);
            vf[dt] = NT ? __builtin_nontemporal_load(at) : *at;
        }
    };
    float m_w = -INFINITY, l_lane = 0.f;
    f32x4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (tok < end) { // uniform for the wave
        f16x8 qf[KS];
        {
            const uint16_t *qp = a.q + ((size_t)b * a.hq + kvh * G + min(j, G - 1)) * D + g * 8;
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                au32x4 raw = *reinterpret_cast<const au32x4 *>(qp + ks * 32);
                if (j >= G) raw = au32x4{0u, 0u, 0u, 0u};
                __builtin_memcpy(&qf[ks], &raw, 16);
            }
        }
        request_keys(at);
        __builtin_amdgcn_sched_barrier(0);
        request_values(at);
        __builtin_amdgcn_sched_barrier(0);
        // One step; LAST: the context may end in it, and nothing follows it.
        auto step = [&](auto last_c) __attribute__((always_inline)) {
            constexpr bool LAST = decltype(last_c)::value;
            Place next = at;
            if (!LAST) next = look_up(tok + W * 32);
            __builtin_amdgcn_sched_barrier(0);
            float s[2][4], m = -INFINITY;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ks++) {
                    f16x8 kk;
                    __builtin_memcpy(&kk, &kf[t][ks], 16);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kk, qf[ks], acc, 0, 0, 0);
                }
                const int left = ctx - (tok + g * 8 + t * 4); // valid tokens among this lane's four
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[t][r] = acc[r];
                    if (!LAST || r < left) m = fmaxf(m, acc[r] * a.scale_log2e);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!LAST) request_keys(next);
            __builtin_amdgcn_sched_barrier(0);
            m = fmaxf(m, __shfl_xor(m, 16));
            m = fmaxf(m, __shfl_xor(m, 32)); // (the first of the 32 is valid for every head: -inf only where the logits are)
            if (__any(m > m_w)) {            // (uniform; seldom after the first few steps)
                // (from the first step's maximum on by whole numbers, where a float has room for them: the factors are powers of two
                // and round nothing)
                const float up = m_w + ceilf(m - m_w), to = m > m_w ? (up >= m && up - m <= 1.f ? up : m) : m_w;
                const float f = m > m_w ? __builtin_amdgcn_exp2f(m_w - to) : 1.f; // 0 on the first step
                m_w = to, l_lane *= f;
#pragma unroll
                for (int r = 0; r < 4; r++) { // o[dt][r] belongs to head 4g + r
                    const float fr = __shfl(f, g * 4 + r);
#pragma unroll
                    for (int dt = 0; dt < DT; dt++) o[dt][r] *= fr;
                }
            }
            const float base = m_w == -INFINITY ? 0.f : m_w; // (logits of -inf alone so far: probabilities of 0)
            // One rounding of the exponent: two were most of a large logit's error.  Of a logit whose float has steps of whole numbers
            // the product is rounded as it was for the maximum, which would not be its own exponent's base otherwise.
            float scale = a.scale_log2e;
            if (__any(fabsf(base) > 65536.f)) {
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++) s[u][r] *= scale;
                scale = 1.f;
            }
            const int left = ctx - (tok + g * 8); // valid tokens among this lane's eight
            f16x8 ph, pl;
            float sum[2] = {0.f, 0.f}; // (a long run's sum takes one addition a step)
#pragma unroll
            for (int u = 0; u < 2; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][r], scale, -base));
                    if (LAST && left <= u * 4 + r) p = 0.f;
                    sum[u] += p;
                    const float ps = p * kProbScale;
                    const _Float16 hi = (_Float16)ps;
                    ph[u * 4 + r] = hi;
                    pl[u * 4 + r] = (_Float16)(ps - (float)hi);
                }
            l_lane += sum[0] + sum[1];
            au32x4 keep; // (what lies in a cache slot past the context may be anything)
#pragma unroll
            for (int d = 0; d < 4; d++) keep[d] = (left > 2 * d ? 0x0000ffffu : 0u) | (left > 2 * d + 1 ? 0xffff0000u : 0u);
#pragma unroll
            for (int dt = 0; dt < DT; dt++) {
                const au32x4 raw = LAST ? vf[dt] & keep : vf[dt];
                f16x8 vv;
                __builtin_memcpy(&vv, &raw, 16);
                // (the step's sum first: one rounding of the run's sum a step)
                const f32x4 lo = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, vv, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                o[dt] += __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, vv, lo, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!LAST) request_values(next);
            __builtin_amdgcn_sched_barrier(0);
            at = next;
        };
#pragma clang loop unroll(disable)
        for (; tok + W * 32 < end; tok += W * 32) step(std::integral_constant<bool, false>());
        step(std::integral_constant<bool, true>());
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] *= 1.f / kProbScale;
    }
    float l_w = l_lane + __shfl_xor(l_lane, 16);
    l_w += __shfl_xor(l_w, 32);
    const int ns = D == 128 ? (int)(((uint32_t)ctx + run - 1) / (uint32_t)run) : 1; // blocks of this (sequence, kv head) that get here
    finish_block<D, W>(a, b, kvh, split, ns, wave, j, g, m_w, l_w, o);
}

// Sets `count` 32-bit words to zero (counter areas are cleared with a kernel, not a memset node, so
// the call may sit inside a captured graph).
__global__ void attn_zero_u32_kernel(uint32_t *p, size_t count) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

// ---- static device scratch of the entry point that allocates nothing -------------------------
// One copy per GPU, held until the process ends: completion counters first, split partials after.
constexpr size_t kScratchCounterBytes = 64u << 10;  // 16384 (sequence, kv head) pairs
constexpr size_t kScratchPartialBytes = 8u << 20;   // batch * query heads * splits * (head_dim + 2) floats
static __device__ __align__(256) unsigned char scratch[kScratchCounterBytes + kScratchPartialBytes];

// Every GPU holds its own copy of the array at its own address: a context takes the address of its device's copy when
// it is created (ctx.hip) and the entry point uses that pointer, never the array's name.
hipError_t attn_static_scratch_address(void **ptr) { return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch)); }

// Everything a launch needs except the buffers: checked geometry, split plan, sizes of the scratch areas.
struct AttnPlan {
    AttnArgs a;
    int nt = 2, waves = 8;               // of the kernel that has a block's whole share under way at once, or
    bool stream = false, stream_values = false, by_lens = false; // the one that goes through it
    size_t partial_bytes = 0, counter_bytes = 0;
};

static int attn_plan(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *p, AttnPlan *plan, size_t most_partial_bytes = SIZE_MAX) {
    NNHIP_REQUIRE(ctx, p->batch > 0 && p->num_q_heads > 0 && p->num_kv_heads > 0 && p->max_blocks_per_seq > 0 &&
                           p->num_blocks > 0,
                  -EINVAL, "paged_attention_decode: non-positive dimension");
    NNHIP_REQUIRE(ctx, p->head_dim == 64 || p->head_dim == 128, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "paged_attention_decode: head_dim %d (64 or 128 supported)", p->head_dim);
    NNHIP_REQUIRE(ctx, p->num_q_heads % p->num_kv_heads == 0 && p->num_q_heads / p->num_kv_heads <= kAttnHeads,
                  -NNCASE_HIP_ERR_SHAPE_MISMATCH, "paged_attention_decode: %d query heads per kv head unsupported (max %d)",
                  p->num_q_heads / p->num_kv_heads, kAttnHeads);
    NNHIP_REQUIRE(ctx, p->block_size > 0 && p->block_size % 16 == 0, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "paged_attention_decode: block_size %d must be a multiple of 16", p->block_size);
    NNHIP_REQUIRE(ctx, (int64_t)p->max_blocks_per_seq * p->block_size < (int64_t(1) << 31), -EINVAL,
                  "paged_attention_decode: context capacity exceeds 2^31 tokens");
    NNHIP_REQUIRE(ctx, p->out_dtype == NNCASE_HIP_DT_F16 || p->out_dtype == NNCASE_HIP_DT_F32,
                  -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "paged_attention_decode: output type 0x%x", p->out_dtype);
    NNHIP_REQUIRE(ctx, (int64_t)p->batch * p->num_kv_heads < (int64_t(1) << 31), -EINVAL, "paged_attention_decode: grid too large");

    AttnArgs &a = plan->a;
    memset(&a, 0, sizeof(a));
    a.batch = p->batch;
    a.hq = p->num_q_heads;
    a.hkv = p->num_kv_heads;
    a.group = p->num_q_heads / p->num_kv_heads;
    a.d = p->head_dim;
    a.block_size = p->block_size;
    a.max_blocks = p->max_blocks_per_seq;
    a.num_blocks = p->num_blocks;
    a.len_offset = p->ctx_len_offset;
    const int64_t max_tokens = (int64_t)p->max_blocks_per_seq * p->block_size;
    const int64_t pairs = (int64_t)p->batch * p->num_kv_heads;
    const int longest = p->head_dim == 64 ? 1024 : 512; // tokens per split that a capacity is accepted for
    const int run = choose_attn_run(p->head_dim, pairs, max_tokens, ctx->compute_units);
    const AttnBlock block = choose_attn_block(p->head_dim, pairs, max_tokens, ctx->compute_units);
    int nt = block.tiles, waves = block.waves;
    for (;;) { // (longer runs where there would be too many splits, for the merge or for the scratch there is)
        a.split_tokens = waves * nt * 16;
        a.splits = (int)std::min<int64_t>((max_tokens + a.split_tokens - 1) / a.split_tokens, INT32_MAX);
        plan->partial_bytes = (size_t)a.batch * a.hq * a.splits * (a.d + 2) * sizeof(float);
        if (a.splits <= kAttnMaxSplits && plan->partial_bytes <= most_partial_bytes) break;
        if (nt == 2) nt = 4;
        else if (waves == 4) waves = 8;
        else if (p->head_dim == 64 && nt == 4) nt = 8;
        else break;
    }
    plan->nt = nt;
    plan->waves = waves;
    plan->stream = plan->stream_values = plan->by_lens = false;
    NNHIP_REQUIRE(ctx, a.splits <= kAttnMaxSplits, -EINVAL,
                  "paged_attention_decode: context capacity of %lld tokens exceeds %d (head_dim %d)", (long long)max_tokens,
                  kAttnMaxSplits * a.split_tokens, p->head_dim);
    if (run > 0) {
        auto bytes = [&](int64_t splits) { return (size_t)(a.batch * a.hq * splits * (a.d + 2) * (int64_t)sizeof(float)); };
        const int64_t splits = (max_tokens + run - 1) / run;
        // (what is refused for want of scratch does not depend on which kernel it would be)
        const size_t needed = bytes(std::max(splits, (max_tokens + longest - 1) / longest));
        if (splits <= kAttnMaxSplits && needed <= most_partial_bytes) {
            a.split_tokens = run, a.splits = (int)splits, plan->partial_bytes = needed, plan->stream = true;
            plan->stream_values = pairs * max_tokens * a.d * 4 >= kStreamedBytes;
            // (with more pairs than compute units the capacity's run is at most 1024 tokens, and many blocks would read many lengths)
            if (a.d == 128 && pairs <= ctx->compute_units) {
                const int64_t room = (int64_t)std::min(most_partial_bytes / bytes(1), (size_t)kAttnMaxSplits);
                const int64_t most = std::max(splits, std::min(attn_most_splits(pairs, max_tokens, run), room));
                a.splits = (int)most, plan->partial_bytes = std::max(needed, bytes(most)), plan->by_lens = true;
                a.rule = attn_run_rule(a.batch, a.hkv, ctx->compute_units, most);
                // Splits of one sequence of few heads on all dies, where the launch's shape would put them on the same few: 32
                // sequences of one head, one of 16 384 tokens and 31 of 400: 32.1 -> 17.7 us.
                a.rotate = a.hkv % kXcds ? 15 : 0;
            }
        }
    }
    a.d_block = make_fastdiv((uint32_t)p->block_size);
    a.d_hkv = make_fastdiv((uint32_t)p->num_kv_heads);
    a.scale_log2e = p->scale * kLog2e;
    a.out_f16 = p->out_dtype == NNCASE_HIP_DT_F16;
    plan->counter_bytes = (size_t)a.batch * a.hkv * sizeof(uint32_t);
    return 0;
}

template <class Args> static bool attn_launch_kernel(nncase_hip_ctx *ctx, const AttnPlan &plan, dim3 grid, int waves, const Args &a) {
    const dim3 block(waves * 64);
    const size_t lds = attn_lds_bytes(a.d, waves);
    bool launched = false;
    auto go = [&](auto kernel) {
        if (lds > 65536) { // more than 64 KiB of dynamic LDS has to be asked for (cheap: a field of the function's record)
            if (hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) return;
        }
        hipLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, a);
        launched = true;
    };
    if (plan.stream) {
        if (a.d == 64) {
            if constexpr (std::is_same_v<Args, AttnArgs>) go(paged_attn_stream_kernel<64, kStreamWaves, false, false, Args>); // (one split)
        } else if (plan.stream_values) {
            if (plan.by_lens) go(paged_attn_stream_kernel<128, kStreamWaves, true, true, Args>);
            else go(paged_attn_stream_kernel<128, kStreamWaves, true, false, Args>);
        } else {
            if (plan.by_lens) go(paged_attn_stream_kernel<128, kStreamWaves, false, true, Args>);
            else go(paged_attn_stream_kernel<128, kStreamWaves, false, false, Args>);
        }
        return launched;
    }
#define NNHIP_ATTN_CASE(DV, NTV, WV) \
    if (!launched && a.d == DV && plan.nt == NTV && waves == WV) go(paged_attn_kernel<DV, NTV, WV, Args>);
    NNHIP_ATTN_CASE(64, 2, 4) NNHIP_ATTN_CASE(64, 4, 4) NNHIP_ATTN_CASE(64, 2, 8) NNHIP_ATTN_CASE(64, 4, 8) NNHIP_ATTN_CASE(64, 8, 8)
    NNHIP_ATTN_CASE(128, 2, 4) NNHIP_ATTN_CASE(128, 4, 4) NNHIP_ATTN_CASE(128, 2, 8) NNHIP_ATTN_CASE(128, 4, 8)
#undef NNHIP_ATTN_CASE
    return launched;
}

static int attn_launch(nncase_hip_ctx *ctx, AttnPlan &plan, const void *q_dev, const void *k_cache_dev, const void *v_cache_dev,
                       const int32_t *block_table_dev, const int32_t *ctx_lens_dev, void *out_dev, void *partials, void *counters,
                       const WeightFetches *fetch = nullptr) {
    AttnArgs &a = plan.a;
    a.q = (const uint16_t *)q_dev;
    a.k_cache = (const uint16_t *)k_cache_dev;
    a.v_cache = (const uint16_t *)v_cache_dev;
    a.block_table = block_table_dev;
    a.ctx_lens = ctx_lens_dev;
    a.out = out_dev;
    a.done = reinterpret_cast<uint32_t *>(counters);
    a.part_o = reinterpret_cast<float *>(partials);
    a.part_ml = a.part_o + (size_t)a.batch * a.hq * a.splits * a.d;
    const int waves = plan.stream ? kStreamWaves : plan.waves;
    dim3 grid(a.hkv * a.batch, a.splits);
    const int64_t own = (int64_t)grid.x * grid.y, busy = (int64_t)grid.x * (((int64_t)a.max_blocks * a.block_size + a.split_tokens - 1) / a.split_tokens);
    // Weights are fetched beside launches that merge splits (one that does not is over before they are here: 8 sequences of 100
    // tokens, a decode layer 25.2 -> 25.5 us) and that leave memory idle (64 sequences of 2048, 1152 blocks: 49.3 -> 49.7; 32 of
    // them, 576 blocks: 39.8 -> 39.5; one of 700, 12 blocks: 24.8 -> 22.9).
    bool launched;
    if (fetch && fetch->count > 0 && a.splits > 1 && busy <= 3 * ctx->compute_units) {
        AttnFetchArgs f;
        static_cast<AttnArgs &>(f) = a;
        f.fetch = *fetch;
        uint32_t fragments = 0; // of die 0, which has the most
        for (int i = 0; i < fetch->count; i++) fragments += fetch_fragments(fetch->f[i], 0);
        f.fetch.blocks = (int)((fragments + waves * kFetchBatch - 1) / (waves * kFetchBatch));
        grid.z = 1 + (unsigned)(((int64_t)f.fetch.blocks * kXcds + own - 1) / own);
        launched = attn_launch_kernel(ctx, plan, grid, waves, f);
    } else {
        launched = attn_launch_kernel(ctx, plan, grid, waves, a);
    }
    NNHIP_REQUIRE(ctx, launched, -EINVAL, "paged_attention_decode: no kernel for head_dim %d, %d tiles per wave, %d waves", a.d, plan.nt, waves);
    NNHIP_LAUNCH_CHECK(ctx, "paged_attn_kernel");
    return 0;
}

// Makes the context's split workspace and counters large enough for this geometry.  Growth frees the
// old areas, so it is refused while a captured graph holds their addresses (-EBUSY) and while the
// context's stream is capturing (an allocation and a synchronisation would invalidate the capture):
// resident functions reserve when the operator is recorded, before any capture.
static bool attn_fits(const nncase_hip_ctx *ctx, const AttnPlan &plan) {
    return ctx->attn_ws_bytes >= plan.partial_bytes && ctx->attn_done_bytes >= plan.counter_bytes;
}
// The plan for a call on the context's workspace: where that cannot grow and longer runs per block (fewer splits) make
// the call fit, those are taken.
static int attn_plan_on_context(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *p, AttnPlan *plan) {
    int rc = attn_plan(ctx, p, plan);
    if (rc || attn_fits(ctx, *plan)) return rc;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (ctx->attn_pins == 0 && hipStreamIsCapturing(ctx->stream, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) return 0;
    AttnPlan small;
    if (attn_plan(ctx, p, &small, ctx->attn_ws_bytes) == 0 && attn_fits(ctx, small)) *plan = small;
    return 0;
}

int attn_reserve(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *p) {
    AttnPlan plan;
    const int rc = attn_plan_on_context(ctx, p, &plan);
    if (rc) return rc;
    if (attn_fits(ctx, plan)) return 0;
    NNHIP_REQUIRE(ctx, ctx->attn_pins == 0, -EBUSY,
                  "paged_attention_decode: the split workspace would have to grow (%zu -> %zu bytes) while %d captured "
                  "function(s) refer to it; record the larger operator before capturing",
                  ctx->attn_ws_bytes, plan.partial_bytes, ctx->attn_pins);
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    NNHIP_HIP(ctx, hipStreamIsCapturing(ctx->stream, &cs));
    NNHIP_REQUIRE(ctx, cs == hipStreamCaptureStatusNone, -EBUSY,
                  "paged_attention_decode: the split workspace cannot be allocated while the stream is capturing");
    NNHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->attn_ws_bytes < plan.partial_bytes) {
        if (ctx->attn_ws) NNHIP_HIP(ctx, hipFree(ctx->attn_ws));
        ctx->attn_ws = nullptr;
        ctx->attn_ws_bytes = 0;
        NNHIP_HIP(ctx, hipMalloc(&ctx->attn_ws, plan.partial_bytes));
        ctx->attn_ws_bytes = plan.partial_bytes;
    }
    if (ctx->attn_done_bytes < plan.counter_bytes) {
        if (ctx->attn_done) NNHIP_HIP(ctx, hipFree(ctx->attn_done));
        ctx->attn_done = nullptr;
        ctx->attn_done_bytes = 0;
        const size_t cap = (plan.counter_bytes + 4095) / 4096 * 4096;
        NNHIP_HIP(ctx, hipMalloc(&ctx->attn_done, cap));
        ctx->attn_done_bytes = cap;
        // zero before the first launch; every launch leaves the counters it used at zero again
        hipLaunchKernelGGL(attn_zero_u32_kernel, dim3(4), dim3(256), 0, ctx->stream, (uint32_t *)ctx->attn_done, cap / 4);
        NNHIP_LAUNCH_CHECK(ctx, "attn_zero_u32_kernel");
        NNHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    }
    return 0;
}

int attn_scratch_sizes(nncase_hip_ctx *ctx, const nncase_hip_paged_attn_args_t *p, size_t *partial_bytes, size_t *counter_bytes) {
    AttnPlan plan;
    const int rc = attn_plan(ctx, p, &plan);
    if (rc) return rc;
    *partial_bytes = plan.partial_bytes, *counter_bytes = plan.counter_bytes;
    return 0;
}

int attn_decode_on(nncase_hip_ctx *ctx, const void *q_dev, const void *k_cache_dev, const void *v_cache_dev, const int32_t *block_table_dev,
                   const int32_t *ctx_lens_dev, void *out_dev, const nncase_hip_paged_attn_args_t *p, void *partials,
                   size_t partial_bytes, void *counters, size_t counter_bytes, const WeightFetches *fetch) {
    AttnPlan plan;
    const int rc = attn_plan(ctx, p, &plan);
    if (rc) return rc;
    NNHIP_REQUIRE(ctx, partials && counters && plan.partial_bytes <= partial_bytes && plan.counter_bytes <= counter_bytes, -ENOSPC,
                  "paged_attention_decode: the scratch areas brought along hold %zu and %zu bytes, the geometry needs %zu and %zu",
                  partial_bytes, counter_bytes, plan.partial_bytes, plan.counter_bytes);
    return attn_launch(ctx, plan, q_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, out_dev, partials, counters, fetch);
}

int attn_decode_on_context(nncase_hip_ctx *ctx, const void *q_dev, const void *k_cache_dev, const void *v_cache_dev,
                           const int32_t *block_table_dev, const int32_t *ctx_lens_dev, void *out_dev,
                           const nncase_hip_paged_attn_args_t *p, const WeightFetches *fetch) {
    AttnPlan plan;
    int rc = attn_plan_on_context(ctx, p, &plan);
    if (rc) return rc;
    if (!attn_fits(ctx, plan)) {
        rc = attn_reserve(ctx, p);
        if (rc) return rc;
    }
    return attn_launch(ctx, plan, q_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, out_dev, ctx->attn_ws,
                       ctx->attn_done, fetch);
}

} // namespace nnhip

using namespace nnhip;

extern "C" int nncase_hip_paged_attention_decode(nncase_hip_ctx_t *ctx, const void *q_dev, const void *k_cache_dev,
                                                 const void *v_cache_dev, const int32_t *block_table_dev,
                                                 const int32_t *ctx_lens_dev, void *out_dev,
                                                 const nncase_hip_paged_attn_args_t *p) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, q_dev && k_cache_dev && v_cache_dev && block_table_dev && ctx_lens_dev && out_dev && p, -EINVAL,
                  "paged_attention_decode: null argument");
    return attn_decode_on_context(ctx, q_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, out_dev, p, nullptr);
}

extern "C" int nncase_hip_paged_attention_decode_noalloc(nncase_hip_ctx_t *ctx, const void *q_dev, const void *k_cache_dev,
                                                         const void *v_cache_dev, const int32_t *block_table_dev,
                                                         const int32_t *ctx_lens_dev, void *out_dev,
                                                         const nncase_hip_paged_attn_args_t *p) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, q_dev && k_cache_dev && v_cache_dev && block_table_dev && ctx_lens_dev && out_dev && p, -EINVAL,
                  "paged_attention_decode_noalloc: null argument");
    AttnPlan plan;
    const int rc = attn_plan(ctx, p, &plan, kScratchPartialBytes);
    if (rc) return rc;
    NNHIP_REQUIRE(ctx, plan.partial_bytes <= kScratchPartialBytes && plan.counter_bytes <= kScratchCounterBytes, -ENOSPC,
                  "paged_attention_decode_noalloc: needs %zu bytes of split partials and %zu of counters; the static "
                  "scratch holds %zu and %zu (use nncase_hip_paged_attention_decode)",
                  plan.partial_bytes, plan.counter_bytes, kScratchPartialBytes, kScratchCounterBytes);
    NNHIP_REQUIRE(ctx, ctx->attn_static, -ENOMEM, "paged_attention_decode_noalloc: the context has no address for the static scratch");
    unsigned char *base = reinterpret_cast<unsigned char *>(ctx->attn_static);
    // The array keeps the previous call's contents: the counters this launch uses must start at zero.
    hipLaunchKernelGGL(attn_zero_u32_kernel, dim3(1), dim3(256), 0, ctx->stream, (uint32_t *)base, plan.counter_bytes / 4);
    NNHIP_LAUNCH_CHECK(ctx, "attn_zero_u32_kernel");
    return attn_launch(ctx, plan, q_dev, k_cache_dev, v_cache_dev, block_table_dev, ctx_lens_dev, out_dev,
                       base + kScratchCounterBytes, base);
}
