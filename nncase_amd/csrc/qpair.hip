// Two pointwise (1x1, stride 1, no padding) quantized convolutions, the second reading the first's result, as one
// launch:  y1 = conv_a(x) [table] [+ residual],  y2 = conv_b(y1) [table].
//
// A linear-bottleneck network alternates a projection (many -> few channels, src/Nncase.Importer/TFLite/Conv2D.cs:17-69
// imports each as its own Conv2D) with the next block's expansion (few -> many).  At small batches the two are
// launch-latency-bound kernels of a few microseconds; here the few-channel tensor between them stays in LDS (it is
// also stored: a later residual add reads it), and the second product starts as soon as the first's tile exists.
//
// Work split: a workgroup owns 16 pixels (8 or 4 behind a depthwise convolution) and a range of conv_b's channel tiles.  It computes ALL of conv_a for its
// pixels (every workgroup of a pixel tile repeats that: the reduction is the cheap side of the pair and recomputing
// keeps enough workgroups alive on 7x7 and 14x14 maps), requantises it exactly as nncase_hip_qconv2d does, and
// multiplies the LDS tile with its range of conv_b.  Results are bit-identical to the two nncase_hip_qconv2d calls.
//
// Weights are re-packed for this kernel: [channel tile][k-step][64 lanes][16 bytes], lane (i, g) holding
// w[16 t + i][64 ks + 16 g ..] - 128 as s8 (zero past the real extents), so that one 16-byte load per lane is an MFMA
// operand and lane (j, g) of the result holds channels 16 t + 4 g .. + 3 of pixel j: four neighbours, one dword.
//
// The second stage alone is the few-pixel path of nncase_hip_qconv2d (qpointwise_rows_kernel, further down): one dense
// 1x1 convolution over few pixels (rows_shapes_ok), optionally behind a global average pool computed by the same launch.
#include "qconv.hpp"
#include "qconv_rules.hpp"

#include <new>
#include <vector>

using namespace nnhip;

struct nncase_hip_qpair {
    const nncase_hip_weights *first = nullptr, *second = nullptr;
    int k1 = 0, n1 = 0, n2 = 0;     // x channels, y1 channels, y2 channels
    int ks1 = 0, ks2 = 0;           // k-steps of 64 of the two reductions
    int t1 = 0, t2 = 0;             // 16-channel tiles of the two results
    uint8_t *d_wa = nullptr, *d_wb = nullptr;
    int32_t *d_wsum_a = nullptr, *d_wsum_b = nullptr; // sum_k (w - 128) per output channel (padded to whole tiles)
    int32_t *d_bias_a = nullptr, *d_bias_b = nullptr; // bias, padded to whole tiles
};

namespace nnhip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPairMaxK1 = 1024;  // x channels
constexpr int kPairMaxN1 = 512;   // y1 channels
constexpr int kPairMaxPixelTiles = 1024; // (of 16: four to a compute unit, see pair_pays)
constexpr int kRowPad = 16;       // bytes between LDS rows beyond the padded reduction (spreads the 16 rows over the banks)

// bytes of an LDS row: the reduction rounded up to whole chunks of `chunk` k-steps, and the pad
__host__ __device__ constexpr int pair_row_bytes(int ksteps, int chunk) { return (ksteps + chunk - 1) / chunk * chunk * 64 + kRowPad; }

struct PairArgs {
    const uint8_t *x;
    uint8_t *y0;           // of the depthwise convolution, where its result is stored too
    uint8_t *y1, *y2;
    const uint8_t *wa, *wb;
    const int32_t *bias_a, *wsum_a, *bias_b, *wsum_b;
    const uint32_t *lut_a, *lut_b;
    int m;                 // pixels
    int ldy, y_coff;       // bytes between pixels of y2, and where its channels begin (n2 and 0 but for one convolution alone)
    int k1, n1, n2;
    int ks1, ks2, t1, t2;
    FastDiv d_pieces;      // 16-byte pieces per LDS row of x
    int tiles_per_block;   // conv_b channel tiles per workgroup (blockIdx.y selects the range)
    int zxa, zwa, zxb, zwb; // zero points - 128
    Epilogue ep_a, ep_b;
    ResidualEpilogue rep_a;
    // with a 3x3 depthwise convolution in front (the DW kernels): x is ITS input [batch, in_h, in_w, k1], and the pixel
    // tile the first convolution multiplies is computed here instead of loaded
    const int16_t *dw_w;             // [9][k1]  w - zw
    const int32_t *dw_bias, *dw_wsum; // [k1]; sum over the taps of w - zw
    int in_h, in_w, out_w, out_hw, stride, pad_h, pad_w;
    FastDiv d_out_hw, d_out_w;
    FastDiv d_quads;       // four channels of k1
    int dw_groups;         // pixels that the workgroup's threads cover at a time, or 0: fewer threads than quads
    int dw_zx;
    Epilogue ep_dw;
    // the second convolution alone (qpointwise_rows_kernel): x holds ITS input rows [m][n1]; its result may leave as the
    // float32 value of the u8 code, and its rows may be the global average of x [m][pool_hw][n1]
    int parts, part_steps; // waves that share a channel tile's reduction, and the k-steps of each (whole chunks)
    FastDiv d_tiles;       // tiles_per_block
    ResidualEpilogue rep_b;
    int deq, deq_zero;
    float deq_scale;
    int pool_hw;
    float pool_zx, pool_sx, pool_zy, pool_sy;
};

__device__ __forceinline__ uint32_t table4(const uint8_t *t, uint32_t v) {
    return (uint32_t)t[v & 0xffu] | ((uint32_t)t[(v >> 8) & 0xffu] << 8) | ((uint32_t)t[(v >> 16) & 0xffu] << 16) |
           ((uint32_t)t[v >> 24] << 24);
}

// What a wave fetches from global memory for one channel tile ahead of multiplying it: the first KC weight fragments,
// and the constants of the tile's epilogue (bias, weight sums and, for the first convolution, the residual bytes).
template <int KC> struct TileLoads {
    v4i frag[KC];
    v4i bias, wsum;
    uint32_t res;
};

// Loads KC weight fragments of one tile from k-step ks0 on; past the tile's last k-step the last one is loaded again
// (the activation tile is zero there, so what such a fragment holds does not matter, and no lane branches).
template <int KC> __device__ __forceinline__ void load_chunk(v4i (&f)[KC], const uint8_t *w, int tile, int ks0, int ksteps, int lane) {
    const v4i *src = reinterpret_cast<const v4i *>(w) + (size_t)tile * ksteps * 64 + lane;
#pragma unroll
    for (int c = 0; c < KC; c++) f[c] = src[min(ks0 + c, ksteps - 1) * 64];
}

template <int KC, bool FIRST>
__device__ __forceinline__ void load_tile(TileLoads<KC> &l, const PairArgs &a, int tile, int ks0, int lane, int p) {
    load_chunk<KC>(l.frag, FIRST ? a.wa : a.wb, tile, ks0, FIRST ? a.ks1 : a.ks2, lane);
    const int ch = tile * 16 + (lane >> 4) * 4;
    l.bias = *reinterpret_cast<const v4i *>((FIRST ? a.bias_a : a.bias_b) + ch);
    l.wsum = *reinterpret_cast<const v4i *>((FIRST ? a.wsum_a : a.wsum_b) + ch);
    l.res = 0;
    if (FIRST && a.rep_a.res && p < a.m && ch < a.n1) l.res = *reinterpret_cast<const uint32_t *>(a.rep_a.res + (size_t)p * a.n1 + ch);
}

// A tile's accumulators to its results: `sum` is the sum of this lane's pixel's row (the same in every lane of it).
// ALONE: of one convolution by itself, which may add a residual.  row: of the lane's pixel in `ys`; live: it is a pixel of the tensor, and
// this lane the one to store it.
template <bool FIRST, bool ALONE = false>
__device__ __forceinline__ void finish_tile(const PairArgs &a, int t, const v4i &acc, int32_t sum, const v4i &bias, const v4i &ws, uint32_t rv, uint8_t *ys,
                                            int sy, const uint8_t *lut, int lane, int row, int p, bool live, bool store_y1) {
    const int g = lane >> 4;
    const int zx = FIRST ? a.zxa : a.zxb, zw = FIRST ? a.zwa : a.zwb;
    const Epilogue &ep = FIRST ? a.ep_a : a.ep_b;
    const int32_t kzz = (FIRST ? a.k1 : a.n1) * zx * zw;
    const int ch = t * 16 + g * 4;
    const int32_t nrs = -zw * sum;
    int32_t v[4];
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = acc[r] + (bias[r] - zx * ws[r] + kzz) + nrs;
    uint32_t q = requant4_u8_packed(v, ep);
    if (lut) q = table4(lut, q);
    if constexpr (FIRST) {
        if (ch < a.n1) {
            if (a.rep_a.res) q = residual4_packed(q, rv, a.rep_a);
            *reinterpret_cast<uint32_t *>(ys + row * sy + ch) = q ^ 0x80808080u;
            if (store_y1 && live) *reinterpret_cast<uint32_t *>(a.y1 + (size_t)p * a.n1 + ch) = q;
        }
    } else if (ch < a.n2 && live) {
        if (ALONE && a.rep_b.res) q = residual4_packed(q, rv, a.rep_b);
        if (ALONE && a.deq) { // the Dequantize behind the convolution: one float per channel
            u32x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = __float_as_uint((float)((int)((q >> (8 * r)) & 0xffu) - a.deq_zero) * a.deq_scale);
            *reinterpret_cast<u32x4 *>(reinterpret_cast<float *>(a.y2) + (size_t)p * a.n2 + ch) = o;
        } else {
            *reinterpret_cast<uint32_t *>(a.y2 + (size_t)p * a.ldy + a.y_coff + ch) = q;
        }
    }
}

// One convolution of the pair for this wave's channel tiles first, first + step, ... below end.  `rows` is the LDS
// activation tile ([16][stride] s8); `cur` holds the loads of the first tile already.  FIRST: results go to the LDS tile
// `ys` as s8 (and to y1 when store_y1); else to y2.  The sum of a row, which
// the weight zero point multiplies, is a second product of the same operands with ones, beside the first (by itself, before it, it
// was 0.3 us of a launch).
template <int KC, bool FIRST>
__device__ __forceinline__ void run_stage(const PairArgs &a, const uint8_t *rows, int stride, uint8_t *ys, int sy, const uint8_t *lut, int first,
                                          int step, int end, TileLoads<KC> &cur, int lane, int p, bool store_y1) {
    const int j = lane & 15, g = lane >> 4;
    const int ksteps = FIRST ? a.ks1 : a.ks2;
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const uint8_t *row = rows + j * stride + g * 16;
    v4i bias = cur.bias, ws = cur.wsum; // the constants of a tile arrive with its first chunk and are used after its last
    uint32_t rv = cur.res;
#pragma unroll 1
    for (int t = first; t < end; t += step) {
        v4i acc = {0, 0, 0, 0}, rs = {0, 0, 0, 0};
#pragma unroll 1
        for (int ks0 = 0; ks0 < ksteps; ks0 += KC) {
            // what follows this chunk (the tile's next one, else the next tile's first) travels while this one multiplies;
            // one wave-uniform branch around all of it: behind the last chunk nothing is requested, so nothing is waited for
            const bool more = ks0 + KC < ksteps;
            TileLoads<KC> nxt;
            if (more || t + step < end) load_tile<KC, FIRST>(nxt, a, more ? t : t + step, more ? ks0 + KC : 0, lane, p);
            if (!more) bias = cur.bias, ws = cur.wsum, rv = cur.res;
#pragma unroll
            for (int c = 0; c < KC; c++) {
                const v4i xf = *reinterpret_cast<const v4i *>(row + (ks0 + c) * 64);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.frag[c], xf, acc, 0, 0, 0);
                rs = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xf, rs, 0, 0, 0);
            }
            cur = nxt;
        }
        finish_tile<FIRST>(a, t, acc, rs[0], bias, ws, rv, ys, sy, lut, lane, j, p, p < a.m, store_y1);
    }
}

// The nine input dwords (four channels from c4) of output pixel `px`'s window; taps outside the image read as the
// zero point, whose share the accumulator's start value takes back out (addresses are clamped into the image, so the
// loads need no branch).
__device__ __forceinline__ void dw_fetch(uint32_t (&buf)[9], const PairArgs &a, int px, int c4) {
    px = min(px, a.m - 1);
    const int n = (int)fastdiv((uint32_t)px, a.d_out_hw), rem = px - n * a.out_hw;
    const int oy = (int)fastdiv((uint32_t)rem, a.d_out_w), ox = rem - oy * a.out_w;
    const int iy0 = oy * a.stride - a.pad_h, ix0 = ox * a.stride - a.pad_w;
    const uint32_t zx4 = (uint32_t)a.dw_zx * 0x01010101u;
#pragma unroll
    for (int ky = 0; ky < 3; ky++) {
        const int iy = iy0 + ky, iyc = min(max(iy, 0), a.in_h - 1);
        const uint8_t *rowp = a.x + (size_t)(n * a.in_h + iyc) * a.in_w * a.k1 + c4;
#pragma unroll
        for (int kx = 0; kx < 3; kx++) {
            const int ix = ix0 + kx, ixc = min(max(ix, 0), a.in_w - 1);
            const uint32_t v = *reinterpret_cast<const uint32_t *>(rowp + (size_t)ixc * a.k1);
            buf[ky * 3 + kx] = (iy == iyc && ix == ixc) ? v : zx4;
        }
    }
}

// The depthwise convolution's 16 pixels x k1 channels, requantised, into the LDS tile as s8.  A thread keeps the
// weights of four channels and walks the pixels pg, pg + pgs, ...: the next pixel's window is requested before this
// one is multiplied.
__device__ __forceinline__ void dw_stage(const PairArgs &a, uint8_t *xs, int sx, int p0, int tid, int threads) {
    const int quads = a.k1 >> 2;
    const bool wide = threads >= quads;            // a thread per channel quad, and pixel groups of them
    const int pgs = wide ? threads / quads : 1, pg = wide ? tid / quads : 0;
    if (pg >= pgs) return;
#pragma unroll 1
    for (int q = wide ? tid - pg * quads : tid; q < quads; q += wide ? quads : threads) {
        const int c4 = q * 4;
        uint32_t cur[9], w01[9], w23[9];
        dw_fetch(cur, a, p0 + pg, c4);
#pragma unroll
        for (int t = 0; t < 9; t++) {
            const uint2 wv = *reinterpret_cast<const uint2 *>(a.dw_w + (size_t)t * a.k1 + c4);
            w01[t] = wv.x, w23[t] = wv.y;
        }
        const v4i bias = *reinterpret_cast<const v4i *>(a.dw_bias + c4), ws = *reinterpret_cast<const v4i *>(a.dw_wsum + c4);
        int32_t ct[4];
#pragma unroll
        for (int c = 0; c < 4; c++) ct[c] = bias[c] - a.dw_zx * ws[c];
#pragma unroll 1
        for (int r = pg; r < 16; r += pgs) {
            uint32_t nxt[9];
            if (r + pgs < 16) dw_fetch(nxt, a, p0 + r + pgs, c4);
            int32_t acc[4] = {ct[0], ct[1], ct[2], ct[3]};
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const uint32_t x01 = __builtin_amdgcn_perm(0, cur[t], 0x0c010c00u), x23 = __builtin_amdgcn_perm(0, cur[t], 0x0c030c02u);
                acc[0] = mad16_lo(x01, w01[t], acc[0]);
                acc[1] = mad16_hi(x01, w01[t], acc[1]);
                acc[2] = mad16_lo(x23, w23[t], acc[2]);
                acc[3] = mad16_hi(x23, w23[t], acc[3]);
            }
            uint32_t code = requant4_u8_packed(acc, a.ep_dw);
            if (p0 + r >= a.m) code = 0x80808080u; // rows past the tensor read as zero
            *reinterpret_cast<uint32_t *>(xs + r * sx + c4) = code ^ 0x80808080u;
#pragma unroll
            for (int t = 0; t < 9; t++) cur[t] = nxt[t];
        }
    }
}

// KA / KB: weight fragments a wave requests at a time for the first / second convolution (each twice in registers).
// MAXW: most waves a workgroup is launched with; OCC: waves per SIMD the register budget is held to.
// DW: a 3x3 depthwise convolution produces the pixel tile (dw_stage).
template <int KA, int KB, int MAXW, int OCC, bool DW>
__global__ __launch_bounds__(MAXW * 64, OCC) void qpointwise_pair_kernel(const PairArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    // rows hold whole chunks of k-steps, zero past the real reduction
    const int sx = pair_row_bytes(a.ks1, KA), sy = pair_row_bytes(a.ks2, KB);
    uint8_t *xs = smem;              // [16][sx]  x - 128
    uint8_t *ys = xs + 16 * sx;      // [16][sy]  y1 - 128
    uint8_t *lut_a = ys + 16 * sy;   // 256 bytes each
    uint8_t *lut_b = lut_a + 256;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, threads = blockDim.x, waves = threads >> 6;
    const int p0 = blockIdx.x * 16, p = p0 + (lane & 15);
    const int b_first = blockIdx.y * a.tiles_per_block;
    const int b_end = min(a.t2, b_first + a.tiles_per_block);

    // the first tiles' weights and constants travel while the pixel tile is staged
    TileLoads<KA> la;
    TileLoads<KB> lb;
    if (wave < a.t1) load_tile<KA, true>(la, a, wave, 0, lane, p);
    if (b_first + wave < b_end) load_tile<KB, false>(lb, a, b_first + wave, 0, lane, p);

    // x tile as s8 (x - 128); rows past the tensor and bytes past K read as zero
    const int pieces = (sx - kRowPad) / 16; // 16-byte pieces per row
    if constexpr (DW) {
        dw_stage(a, xs, sx, p0, tid, threads);
        const int first = a.k1 / 16, extra = pieces - first;
        for (int e = tid; e < 16 * extra; e += threads) {
            const int r = e / extra, c = first + (e - r * extra);
            *reinterpret_cast<u32x4 *>(xs + r * sx + c * 16) = u32x4{0u, 0u, 0u, 0u};
        }
    } else {
        const u32x4 none = {0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
        constexpr int U = KA > 4 ? 2 : 1;
#pragma unroll 1
        for (int e0 = tid; e0 < 16 * pieces; e0 += U * threads) {
            u32x4 v[U];
            uint32_t at[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t e = (uint32_t)(e0 + u * threads), r = fastdiv(e, a.d_pieces), c = e - r * (uint32_t)pieces;
                at[u] = r * sx + c * 16;
                v[u] = none;
                if (r < 16 && p0 + (int)r < a.m && (int)c * 16 < a.k1) v[u] = *reinterpret_cast<const u32x4 *>(a.x + (size_t)(p0 + (int)r) * a.k1 + c * 16);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (e0 + u * threads < 16 * pieces) *reinterpret_cast<u32x4 *>(xs + at[u]) = v[u] ^ 0x80808080u;
        }
    }
    for (int e = tid; e < 4 * sy; e += threads) reinterpret_cast<uint32_t *>(ys)[e] = 0; // channels past N1 stay zero
    for (int e = tid; e < 128; e += threads) {
        if (e < 64) {
            if (a.lut_a) reinterpret_cast<uint32_t *>(lut_a)[e] = a.lut_a[e];
        } else if (a.lut_b) {
            reinterpret_cast<uint32_t *>(lut_b)[e - 64] = a.lut_b[e - 64];
        }
    }
    __syncthreads();
    // the first convolution over the whole of its channels, into LDS (and, from the first channel range, into y1)
    if (wave < a.t1) run_stage<KA, true>(a, xs, sx, ys, sy, a.lut_a ? lut_a : nullptr, wave, waves, a.t1, la, lane, p, blockIdx.y == 0);
    __syncthreads();
    // the second: this workgroup's channel tiles from the LDS tile
    if (b_first + wave < b_end) run_stage<KB, false>(a, ys, sy, nullptr, 0, a.lut_b ? lut_b : nullptr, b_first + wave, waves, b_end, lb, lane, p, false);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pair_resource(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// The kernel's arguments that its epilogues take, loaded where this is called and all together.  With what a launch needs at its start
// there are more than scalar registers: left to itself the compiler loads everything first and puts it in lanes of vector registers and
// out again, eight scalar round trips in front of the first request; or, kept from that, each where a branch first uses it.
__device__ __forceinline__ void gather(Epilogue &to, const Epilogue &ep) {
    to.mult = ep.mult, to.sy = ep.sy, to.rsy = ep.rsy, to.zy = ep.zy, to.qlo = ep.qlo, to.qhi = ep.qhi, to.c1 = ep.c1, to.c2 = ep.c2;
    to.fast = ep.fast, to.full = ep.full;
}
template <bool FRONT> __device__ __forceinline__ PairArgs gather_epilogues() {
    auto p = (const __attribute__((address_space(4))) PairArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    const PairArgs &a = *(const PairArgs *)p;
    PairArgs l; // (what is not assigned here is not used)
    if constexpr (FRONT) { // the depthwise stage's
        gather(l.ep_dw, a.ep_dw);
        l.dw_zx = a.dw_zx, l.y0 = a.y0;
        asm volatile("" ::"s"(l.ep_dw.mult), "s"(l.ep_dw.sy), "s"(l.ep_dw.rsy), "s"(l.ep_dw.zy), "s"(l.ep_dw.qlo), "s"(l.ep_dw.qhi), "s"(l.ep_dw.c1),
                     "s"(l.ep_dw.c2), "s"(l.ep_dw.fast), "s"(l.ep_dw.full), "s"(l.dw_zx), "s"(l.y0));
    } else {
        gather(l.ep_a, a.ep_a), gather(l.ep_b, a.ep_b), gather(l.rep_a.sum, a.rep_a.sum);
        l.rep_a.res = a.rep_a.res, l.rep_a.zy = a.rep_a.zy, l.rep_a.sy = a.rep_a.sy, l.rep_a.zr = a.rep_a.zr, l.rep_a.sr = a.rep_a.sr;
        l.y1 = a.y1, l.y2 = a.y2, l.k1 = a.k1, l.n1 = a.n1, l.n2 = a.n2, l.ldy = a.ldy, l.y_coff = a.y_coff;
        l.zxa = a.zxa, l.zwa = a.zwa, l.zxb = a.zxb, l.zwb = a.zwb;
        asm volatile("" ::"s"(l.ep_a.mult), "s"(l.ep_a.sy), "s"(l.ep_a.rsy), "s"(l.ep_a.zy), "s"(l.ep_a.qlo), "s"(l.ep_a.qhi), "s"(l.ep_a.c1), "s"(l.ep_a.c2),
                     "s"(l.ep_a.fast), "s"(l.ep_a.full), "s"(l.rep_a.sum.sy), "s"(l.rep_a.sum.rsy), "s"(l.rep_a.sum.zy), "s"(l.rep_a.sum.qlo),
                     "s"(l.rep_a.sum.qhi), "s"(l.rep_a.res), "s"(l.rep_a.zy), "s"(l.rep_a.sy), "s"(l.rep_a.zr), "s"(l.rep_a.sr), "s"(l.y1), "s"(l.zxa), "s"(l.zwa));
        asm volatile("" ::"s"(l.ep_b.mult), "s"(l.ep_b.sy), "s"(l.ep_b.rsy), "s"(l.ep_b.zy), "s"(l.ep_b.qlo), "s"(l.ep_b.qhi), "s"(l.ep_b.c1), "s"(l.ep_b.c2),
                     "s"(l.ep_b.fast), "s"(l.ep_b.full), "s"(l.y2), "s"(l.n2), "s"(l.zxb), "s"(l.zwb), "s"(l.ldy), "s"(l.y_coff));
    }
    return l;
}

// A window of the depthwise convolution as dw_fetch's, in two halves: the requests, and the taps outside the image.  (The input is less
// than 2 GiB.)
struct DwWindow {
    uint32_t x[9];
    bool in_y[3], in_x[3];
};
__device__ __forceinline__ void dw_request(DwWindow &w, const PairArgs &a, int px, int c4) {
    px = min(px, a.m - 1);
    const int n = (int)fastdiv((uint32_t)px, a.d_out_hw), rem = px - n * a.out_hw;
    const int oy = (int)fastdiv((uint32_t)rem, a.d_out_w), ox = rem - oy * a.out_w;
    const int iy0 = oy * a.stride - a.pad_h, ix0 = ox * a.stride - a.pad_w;
    int iy[3], ix[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        iy[k] = min(max(iy0 + k, 0), a.in_h - 1), w.in_y[k] = iy[k] == iy0 + k;
        ix[k] = min(max(ix0 + k, 0), a.in_w - 1), w.in_x[k] = ix[k] == ix0 + k;
    }
    const uint32_t pitch = (uint32_t)a.in_w * (uint32_t)a.k1;
    uint32_t ro[3], co[3]; // (a clamped position is the last one's or one further: one multiplication each, which takes four times an addition)
    ro[0] = (uint32_t)(n * a.in_h + iy[0]) * pitch, co[0] = (uint32_t)ix[0] * (uint32_t)a.k1 + (uint32_t)c4;
#pragma unroll
    for (int k = 1; k < 3; k++) ro[k] = ro[k - 1] + (iy[k] != iy[k - 1] ? pitch : 0u), co[k] = co[k - 1] + (ix[k] != ix[k - 1] ? (uint32_t)a.k1 : 0u);
#pragma unroll
    for (int t = 0; t < 9; t++) w.x[t] = *reinterpret_cast<const uint32_t *>(a.x + (size_t)(ro[t / 3] + co[t % 3]));
}
struct DwTaps {
    uint32_t w01[9], w23[9];
    v4i bias, ws;
};
__device__ __forceinline__ void dw_request_taps(DwTaps &d, const PairArgs &a, int c4) {
#pragma unroll
    for (int t = 0; t < 9; t++) {
        const uint2 wv = *reinterpret_cast<const uint2 *>(a.dw_w + (uint32_t)(t * a.k1 + c4));
        d.w01[t] = wv.x, d.w23[t] = wv.y;
    }
    d.bias = *reinterpret_cast<const v4i *>(a.dw_bias + c4), d.ws = *reinterpret_cast<const v4i *>(a.dw_wsum + c4);
}
__device__ __forceinline__ uint32_t dw_codes(const DwWindow &w, const DwTaps &d, const PairArgs &a) {
    const uint32_t zx4 = (uint32_t)a.dw_zx * 0x01010101u;
    int32_t acc[4];
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = d.bias[c] - a.dw_zx * d.ws[c];
#pragma unroll
    for (int t = 0; t < 9; t++) {
        const uint32_t x = w.in_y[t / 3] && w.in_x[t % 3] ? w.x[t] : zx4;
        const uint32_t x01 = __builtin_amdgcn_perm(0, x, 0x0c010c00u), x23 = __builtin_amdgcn_perm(0, x, 0x0c030c02u);
        acc[0] = mad16_lo(x01, d.w01[t], acc[0]);
        acc[1] = mad16_hi(x01, d.w01[t], acc[1]);
        acc[2] = mad16_lo(x23, d.w23[t], acc[2]);
        acc[3] = mad16_hi(x23, d.w23[t], acc[3]);
    }
    return requant4_u8_packed(acc, a.ep_dw);
}

// The same where no wave has more than one tile of either convolution and KA and KB fragments hold their reductions.  Such a launch is
// bound by its chain of waits and by the instructions between them, so a wave's requests come first, in the order in which they are
// needed, and where a wave has none of a kind it skips them as a whole (a load past the end of a buffer resource fetches nothing, but
// holds up the loads behind it like any other: a wave's spare fragments are few).
//
// PT: pixels of a workgroup, 16, 8 or 4.  The matrix instruction's 16 columns hold them 16 / PT times over; what is saved is the
// depthwise stage, which is vector work on one compute unit, by leaving it to more of them.  us from the first wave's start to the last
// store, in a MobileNetV2 step of one image, before / now: 192 -> 32 -> 192 of 784 pixels with the stage 4.6 / 3.3, 192 -> 64 -> 384 of 196
// 4.5 / 3.2, without it 384 -> 64 -> 384 3.5 / 2.9; a launch of its own for 384 channels' stage, 1.4 us and a gap of 1.6, is now 0.8 us of
// the pair's.  The step: 160.9 -> 125.7.
template <int KA, int KB, int MAXW, int OCC, bool DW, int PT>
__global__ __launch_bounds__(MAXW * 64, OCC) void qpointwise_pair_once_kernel(const PairArgs a) {
    static_assert(DW || PT == 16, "smaller tiles are for the depthwise stage");
    extern __shared__ __align__(16) uint8_t smem[];
    const int ks1 = a.ks1, ks2 = a.ks2, k1 = a.k1, n1 = a.n1;
    const int sx = pair_row_bytes(ks1, 1), sy = pair_row_bytes(ks2, 1);
    uint8_t *const xs = smem;              // [PT][sx]  x - 128
    uint8_t *const ys = xs + PT * sx;      // [PT][sy]  y1 - 128
    uint8_t *const lut_a = ys + PT * sy;   // 256 bytes each
    uint8_t *const lut_b = lut_a + 256;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x, waves = threads >> 6;
    const int g = lane >> 4, row = lane & (PT - 1);
    const int p0 = (int)blockIdx.x * PT, p = p0 + row, pixels = min(PT, a.m - p0);
    const bool live = (lane & 15) < PT && p < a.m;
    const int tile_b = (int)blockIdx.y * a.tiles_per_block + wave;
    const bool works_a = wave < a.t1, works_b = wave < a.tiles_per_block && tile_b < a.t2; // uniform
    const bool has_lut_a = a.lut_a != nullptr, has_lut_b = a.lut_b != nullptr;

    // ---- requests: a wave's weights and constants of the first convolution ---------------------------------
    v4i fa[KA], fb[KB], bias_a, wsum_a, bias_b, wsum_b;
    uint32_t rv = 0;
    const int ch_a = wave * 16 + g * 4, ch_b = tile_b * 16 + g * 4;
    auto request_a = [&]() __attribute__((always_inline)) { // (where works_a; k-steps past the reduction: past the end)
        const auto w = pair_resource(a.wa + (size_t)wave * ks1 * 1024, (uint32_t)ks1 * 1024u);
#pragma unroll
        for (int c = 0; c < KA; c++) fa[c] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w, lane * 16 + c * 1024, 0, 0));
        bias_a = *reinterpret_cast<const v4i *>(a.bias_a + ch_a), wsum_a = *reinterpret_cast<const v4i *>(a.wsum_a + ch_a);
        const auto residual = pair_resource(a.rep_a.res + (a.rep_a.res ? (size_t)p0 * n1 : 0), a.rep_a.res ? (uint32_t)(pixels * n1) : 0u);
        rv = __builtin_amdgcn_raw_buffer_load_b32(residual, row * n1 + ch_a, 0, 0); // (of channels past N1: the next pixel's, unused)
    };
    // ... and of the second, behind the pixels: there is the first convolution's time for them
    uint32_t ta, tb;
    auto request_b = [&]() __attribute__((always_inline)) {
        const auto w = pair_resource(a.wb + (size_t)(works_b ? tile_b : 0) * ks2 * 1024, works_b ? (uint32_t)ks2 * 1024u : 0u);
#pragma unroll
        for (int c = 0; c < KB; c++) fb[c] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w, lane * 16 + c * 1024, 0, 0));
        const uint32_t bytes_b = works_b ? (uint32_t)a.t2 * 64u : 0u;
        bias_b = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(pair_resource(a.bias_b, bytes_b), ch_b * 4, 0, 0));
        wsum_b = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(pair_resource(a.wsum_b, bytes_b), ch_b * 4, 0, 0));
        __builtin_amdgcn_sched_barrier(0);
    };
    ta = __builtin_amdgcn_raw_buffer_load_b32(pair_resource(a.lut_a, wave == 0 && has_lut_a ? 256u : 0u), lane * 4, 0, 0);
    tb = __builtin_amdgcn_raw_buffer_load_b32(pair_resource(a.lut_b, wave == waves - 1 && has_lut_b ? 256u : 0u), lane * 4, 0, 0);

    // ---- the pixel tile as s8 (x - 128); bytes past K are zero --------------------------------------------
    if constexpr (DW) {
        // A thread per window of four channels, in the last waves: the first ones bring the first convolution's weights in.
        const int quads = k1 >> 2, ftid = threads - 1 - tid, fwave = waves - 1 - wave;
        int pg = 0, quad = ftid;
        if (a.dw_groups > 0) pg = (int)fastdiv((uint32_t)ftid, a.d_quads), quad = ftid - pg * quads;
        bool mine = a.dw_groups > 0 ? pg < a.dw_groups : ftid < quads;
        const bool fronts = fwave * 64 < quads * max(a.dw_groups, 1); // uniform
        DwWindow win;
        DwTaps taps;
        if (fronts) {
            const int c4 = mine ? quad * 4 : 0;
            dw_request(win, a, p0 + pg, c4);
            dw_request_taps(taps, a, c4);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (works_a) request_a();
        const PairArgs later = gather_epilogues<true>(); // (the trip beside the others')
        for (int q = quad, r = pg; fronts;) { // (one turn where there is a thread per window)
            const uint32_t code = dw_codes(win, taps, later);
            if (mine) {
                *reinterpret_cast<uint32_t *>(xs + r * sx + q * 4) = (p0 + r < a.m ? code : 0x80808080u) ^ 0x80808080u;
                if (later.y0 && blockIdx.y == 0 && p0 + r < a.m) *reinterpret_cast<uint32_t *>(later.y0 + (size_t)(p0 + r) * k1 + q * 4) = code;
            }
            r += max(a.dw_groups, 1);
            bool more = r < PT;
            if (a.dw_groups == 0 && !more) q += threads, r = 0, more = q < quads, mine = more;
            if (!__any(mine && more)) break;
            mine = mine && more;
            const int c4 = mine ? q * 4 : 0;
            dw_request(win, a, p0 + min(r, PT - 1), c4);
            if (a.dw_groups == 0) dw_request_taps(taps, a, c4);
        }
        request_b();
        for (int r = wave; r < PT && k1 < ks1 * 64; r += waves)
            if (k1 + lane * 4 < ks1 * 64) *reinterpret_cast<uint32_t *>(xs + r * sx + k1 + lane * 4) = 0u;
    } else {
        constexpr int U = KA > 8 ? 2 : 1; // pieces of 16 bytes that a thread brings in at once
        const int pieces = ks1 * 4;       // ... of a row, past K as well
        const auto rows = pair_resource(a.x + (size_t)p0 * k1, (uint32_t)(pixels * k1));
        u32x4 v[U];
        auto request_x = [&](int e0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t e = (uint32_t)(e0 + u * threads), r = fastdiv(e, a.d_pieces), c = e - r * (uint32_t)pieces;
                v[u] = __builtin_amdgcn_raw_buffer_load_b128(rows, (int)(r * (uint32_t)k1 + c * 16u), 0, 0);
            }
        };
        auto put_x = [&](int e0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t e = (uint32_t)(e0 + u * threads), r = fastdiv(e, a.d_pieces), c = e - r * (uint32_t)pieces;
                if (r < 16) *reinterpret_cast<u32x4 *>(xs + r * sx + c * 16) = (int)c * 16 < k1 ? v[u] ^ 0x80808080u : u32x4{0u, 0u, 0u, 0u};
            }
        };
        request_x(tid);
        __builtin_amdgcn_sched_barrier(0);
        if (works_a) { // (each with the pixels' first turn: behind a join the wait for them would be one for the weights too)
            request_a();
            __builtin_amdgcn_sched_barrier(0);
            put_x(tid);
        } else {
            put_x(tid);
        }
#pragma unroll 1
        for (int e0 = tid + U * threads; e0 - tid < 16 * pieces; e0 += U * threads) request_x(e0), put_x(e0);
        request_b();
    }
    const PairArgs later = gather_epilogues<false>();
    for (int r = wave; r < PT && n1 < ks2 * 64; r += waves)
        if (n1 + lane * 4 < ks2 * 64) *reinterpret_cast<uint32_t *>(ys + r * sy + n1 + lane * 4) = 0u;
    if (wave == 0 && has_lut_a) reinterpret_cast<uint32_t *>(lut_a)[lane] = ta;
    if (wave == waves - 1 && has_lut_b) reinterpret_cast<uint32_t *>(lut_b)[lane] = tb;
    __syncthreads();

    // ---- products: the first over the whole of its channels into LDS (and, from the first channel range, into y1), then the second ----
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    if (works_a) {
        const uint8_t *from = xs + row * sx + g * 16;
        v4i acc = {0, 0, 0, 0}, rs = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < KA; c++)
            if (c < ks1) { // uniform
                const v4i xf = *reinterpret_cast<const v4i *>(from + c * 64);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[c], xf, acc, 0, 0, 0);
                rs = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xf, rs, 0, 0, 0);
            }
        finish_tile<true>(later, wave, acc, rs[0], bias_a, wsum_a, rv, ys, sy, has_lut_a ? lut_a : nullptr, lane, row, p, live, blockIdx.y == 0);
    }
    __syncthreads();
    if (works_b) {
        const uint8_t *from = ys + row * sy + g * 16;
        v4i acc = {0, 0, 0, 0}, rs = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < KB; c++)
            if (c < ks2) { // uniform
                const v4i xf = *reinterpret_cast<const v4i *>(from + c * 64);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[c], xf, acc, 0, 0, 0);
                rs = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xf, rs, 0, 0, 0);
            }
        finish_tile<false>(later, tile_b, acc, rs[0], bias_b, wsum_b, 0u, nullptr, 0, has_lut_b ? lut_b : nullptr, lane, row, p, live, false);
    }
}

// One dense 1x1 convolution over a few rows (pixels): the second stage of the pair kernel alone.  A workgroup stages 16
// rows as s8 in LDS and takes a range of the channel tiles, the weights straight from global memory
// into MFMA operands with the first chunk requested before the rows are staged.  Against the tiled kernels, which
// stream k-step by k-step through LDS with a barrier each, a launch is one memory round trip long, not one per k-step.
// A tile's reduction is shared by a.parts waves, a chunk each where there are enough (us with one wave that takes its chunks one after the
// other and stages the rows by itself / so: 1 row of 1280 -> 1000 6.5 / 3.8, 16 rows 9.1 / 4.6, 25 of 576 -> 96 6.7 / 3.7).
// POOL: the rows are global averages over pool_hw pixels, computed here (global_avgpool4, a thread per four channels).
constexpr int kRowsChunk = 8, kRowsWaves = 12;
constexpr int kRowsShareBytes = 64 * 5 * 4; // what a wave hands over: 4 accumulators and the row sum per lane
template <bool POOL> __global__ __launch_bounds__(kRowsWaves * 64, 3) void qpointwise_rows_kernel(const PairArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int sy = pair_row_bytes(a.ks2, kRowsChunk);
    uint8_t *ys = smem;              // [16][sy]  rows - 128
    uint8_t *lut_b = ys + 16 * sy;   // 256 bytes
    uint8_t *shares = lut_b + 256;   // [parts - 1][tiles_per_block][64 lanes] x 16 bytes, then as many dwords
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), threads = blockDim.x;
    const int p0 = blockIdx.x * 16, p = p0 + (lane & 15);
    const int part = (int)fastdiv((uint32_t)wave, a.d_tiles), slot = wave - part * a.tiles_per_block;
    const int tile = blockIdx.y * a.tiles_per_block + slot;
    const int first = part * a.part_steps, last = min(a.ks2, first + a.part_steps);
    const bool works = part < a.parts && tile < a.t2;
    TileLoads<kRowsChunk> cur;
    uint32_t rv = 0;
    if (works) {
        load_tile<kRowsChunk, false>(cur, a, tile, first, lane, p);
        const int ch = tile * 16 + (lane >> 4) * 4;
        if (a.rep_b.res && part == 0 && p < a.m && ch < a.n2) rv = *reinterpret_cast<const uint32_t *>(a.rep_b.res + (size_t)p * a.n2 + ch);
    }
    const int pieces = (sy - kRowPad) / 16;
    if constexpr (POOL) {
        const int quads = a.n1 >> 2;
#pragma unroll 1
        for (int e = tid; e < 16 * quads; e += threads) {
            const int r = e / quads, c4 = (e - r * quads) * 4;
            uint32_t code = 0x80808080u; // rows past the tensor read as zero
            if (p0 + r < a.m) code = global_avgpool4(a.x + (size_t)(p0 + r) * a.pool_hw * a.n1 + c4, a.pool_hw, a.n1, a.pool_zx, a.pool_sx, a.pool_zy, a.pool_sy);
            *reinterpret_cast<uint32_t *>(ys + r * sy + c4) = code ^ 0x80808080u;
        }
        const int real = a.n1 / 16, extra = pieces - real; // pieces past the real reduction
        for (int e = tid; e < 16 * extra; e += threads) {
            const int r = e / extra, c = real + (e - r * extra);
            *reinterpret_cast<u32x4 *>(ys + r * sy + c * 16) = u32x4{0u, 0u, 0u, 0u};
        }
    } else {
        constexpr int U = 4;
#pragma unroll 1
        for (int e0 = tid; e0 < 16 * pieces; e0 += U * threads) {
            u32x4 v[U];
            uint32_t at[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const uint32_t e = (uint32_t)(e0 + u * threads), r = fastdiv(e, a.d_pieces), c = e - r * (uint32_t)pieces;
                at[u] = r * sy + c * 16;
                v[u] = u32x4{0x80808080u, 0x80808080u, 0x80808080u, 0x80808080u};
                if (r < 16 && p0 + (int)r < a.m && (int)c * 16 < a.n1) v[u] = *reinterpret_cast<const u32x4 *>(a.x + (size_t)(p0 + (int)r) * a.n1 + c * 16);
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (e0 + u * threads < 16 * pieces) *reinterpret_cast<u32x4 *>(ys + at[u]) = v[u] ^ 0x80808080u;
        }
    }
    if (a.lut_b)
        for (int e = tid; e < 64; e += threads) reinterpret_cast<uint32_t *>(lut_b)[e] = a.lut_b[e];
    __syncthreads();
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101}, bias = cur.bias, ws = cur.wsum;
    v4i acc = {0, 0, 0, 0}, rs = {0, 0, 0, 0};
    if (works) {
        const uint8_t *row = ys + (lane & 15) * sy + (lane >> 4) * 16;
#pragma unroll 1
        for (int ks0 = first; ks0 < last; ks0 += kRowsChunk) {
            v4i nxt[kRowsChunk];
            const bool more = ks0 + kRowsChunk < last;
            if (more) load_chunk<kRowsChunk>(nxt, a.wb, tile, ks0 + kRowsChunk, a.ks2, lane);
#pragma unroll
            for (int c = 0; c < kRowsChunk; c++) {
                const v4i xf = *reinterpret_cast<const v4i *>(row + (ks0 + c) * 64);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur.frag[c], xf, acc, 0, 0, 0);
                rs = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xf, rs, 0, 0, 0);
            }
            if (more) {
#pragma unroll
                for (int c = 0; c < kRowsChunk; c++) cur.frag[c] = nxt[c];
            }
        }
    }
    if (a.parts > 1) { // (uniform for the launch)
        const int spare = (a.parts - 1) * a.tiles_per_block;
        v4i *const accs = reinterpret_cast<v4i *>(shares);
        int32_t *const sums = reinterpret_cast<int32_t *>(shares + (size_t)spare * 64 * 16);
        if (works && part > 0) {
            const int at = ((part - 1) * a.tiles_per_block + slot) * 64 + lane;
            accs[at] = acc, sums[at] = rs[0];
        }
        __syncthreads();
        if (works && part == 0)
            for (int q = 0; q < a.parts - 1; q++) {
                const int at = (q * a.tiles_per_block + slot) * 64 + lane;
                acc += accs[at], rs[0] += sums[at];
            }
    }
    if (works && part == 0) finish_tile<false, true>(a, tile, acc, rs[0], bias, ws, rv, nullptr, 0, a.lut_b ? lut_b : nullptr, lane, lane & 15, p, p < a.m, false);
}

// [tile][k-step][lane][16] s8 of w - 128, zero beyond the real channels / reduction
static void pack_pair_weights(std::vector<uint8_t> &out, std::vector<int32_t> &wsum, const uint8_t *w_oihw, int n, int k, int tiles, int ksteps) {
    out.assign((size_t)tiles * ksteps * 1024, 0);
    wsum.assign((size_t)tiles * 16, 0);
    for (int ch = 0; ch < n; ch++) {
        int32_t s = 0;
        for (int kk = 0; kk < k; kk++) {
            const uint8_t raw = w_oihw[(size_t)ch * k + kk];
            s += (int32_t)raw - 128;
            const int t = ch >> 4, i = ch & 15, ks = kk >> 6, g = (kk >> 4) & 3, b = kk & 15;
            out[(((size_t)t * ksteps + ks) * 64 + g * 16 + i) * 16 + b] = raw ^ 0x80;
        }
        wsum[ch] = s;
    }
}

static void free_pair(nncase_hip_qpair *pr) {
    if (!pr) return;
    if (pr->d_wa) (void)hipFree(pr->d_wa);
    if (pr->d_wb) (void)hipFree(pr->d_wb);
    if (pr->d_wsum_a) (void)hipFree(pr->d_wsum_a);
    if (pr->d_wsum_b) (void)hipFree(pr->d_wsum_b);
    if (pr->d_bias_a) (void)hipFree(pr->d_bias_a);
    if (pr->d_bias_b) (void)hipFree(pr->d_bias_b);
    delete pr;
}

static bool pair_shapes_ok(int k1, int n1, int n2) {
    return k1 > 0 && n1 > 0 && n2 > 0 && k1 % 16 == 0 && n1 % 4 == 0 && n2 % 4 == 0 && k1 <= kPairMaxK1 && n1 <= kPairMaxN1;
}

static int upload(nncase_hip_ctx *ctx, void **dst, const void *src, size_t bytes) {
    NNHIP_HIP(ctx, hipMalloc(dst, bytes));
    NNHIP_HIP(ctx, hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice));
    return 0;
}

static bool pointwise_weights(const nncase_hip_weights *w) {
    return w && w->kind == nncase_hip_weights::kIgemm && w->groups == 1 && w->kernel_h == 1 && w->kernel_w == 1;
}

} // namespace nnhip

extern "C" int nncase_hip_qpointwise_pair_supported(int32_t in_channels, int32_t mid_channels, int32_t out_channels) {
    return pair_shapes_ok(in_channels, mid_channels, out_channels) ? 1 : 0;
}

extern "C" int nncase_hip_qpointwise_pair_create(nncase_hip_ctx_t *ctx, const nncase_hip_weights_t *first,
                                                 const uint8_t *first_oihw_host, const nncase_hip_weights_t *second,
                                                 const uint8_t *second_oihw_host, nncase_hip_qpair_t **pair) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, first && first_oihw_host && second && second_oihw_host && pair, -EINVAL, "qpointwise_pair_create: null argument");
    *pair = nullptr;
    NNHIP_REQUIRE(ctx, pointwise_weights(first) && pointwise_weights(second), -EINVAL,
                  "qpointwise_pair_create: both convolutions must be dense 1x1 convolutions");
    NNHIP_REQUIRE(ctx, first->out_channels == second->in_channels, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "qpointwise_pair_create: the first convolution has %d output channels, the second reads %d", first->out_channels,
                  second->in_channels);
    NNHIP_REQUIRE(ctx, pair_shapes_ok(first->in_channels, first->out_channels, second->out_channels), -EINVAL,
                  "qpointwise_pair_create: channels %d -> %d -> %d unsupported (first a multiple of 16 up to %d, second a multiple of 4 "
                  "up to %d, third a multiple of 4)",
                  first->in_channels, first->out_channels, second->out_channels, kPairMaxK1, kPairMaxN1);
    nncase_hip_qpair *pr = new (std::nothrow) nncase_hip_qpair();
    NNHIP_REQUIRE(ctx, pr, -ENOMEM, "qpointwise_pair_create: out of host memory");
    pr->first = first, pr->second = second;
    pr->k1 = first->in_channels, pr->n1 = first->out_channels, pr->n2 = second->out_channels;
    pr->ks1 = (pr->k1 + 63) / 64, pr->ks2 = (pr->n1 + 63) / 64;
    pr->t1 = (pr->n1 + 15) / 16, pr->t2 = (pr->n2 + 15) / 16;
    NNHIP_HIP(ctx, hipSetDevice(ctx->device));
    std::vector<uint8_t> packed;
    std::vector<int32_t> wsum, bias;
    int rc = 0;
    auto side = [&](const nncase_hip_weights *w, const uint8_t *host, int n, int k, int tiles, int ksteps, uint8_t **d_w, int32_t **d_wsum,
                    int32_t **d_bias) -> int {
        pack_pair_weights(packed, wsum, host, n, k, tiles, ksteps);
        bias.assign((size_t)tiles * 16, 0);
        NNHIP_HIP(ctx, hipMemcpy(bias.data(), w->d_bias, sizeof(int32_t) * n, hipMemcpyDeviceToHost));
        int r = upload(ctx, (void **)d_w, packed.data(), packed.size());
        if (!r) r = upload(ctx, (void **)d_wsum, wsum.data(), wsum.size() * sizeof(int32_t));
        if (!r) r = upload(ctx, (void **)d_bias, bias.data(), bias.size() * sizeof(int32_t));
        return r;
    };
    rc = side(first, first_oihw_host, pr->n1, pr->k1, pr->t1, pr->ks1, &pr->d_wa, &pr->d_wsum_a, &pr->d_bias_a);
    if (!rc) rc = side(second, second_oihw_host, pr->n2, pr->n1, pr->t2, pr->ks2, &pr->d_wb, &pr->d_wsum_b, &pr->d_bias_b);
    if (rc) {
        free_pair(pr);
        return rc;
    }
    *pair = pr;
    return 0;
}

extern "C" int nncase_hip_qpointwise_pair_destroy(nncase_hip_ctx_t *ctx, nncase_hip_qpair_t *pair) {
    NNHIP_CHECK_CTX(ctx);
    if (!pair) return 0;
    NNHIP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    free_pair(pair);
    return 0;
}

// ---- the few-pixel path of one dense 1x1 convolution ----------------------------------------------------------------
namespace nnhip {
constexpr int kRowsMaxK = 2048;                 // reduction length (an LDS row: 16 of them stay below 64 KiB)
constexpr int64_t kRowsStreamLimit = 4 << 20;   // weight bytes all pixel tiles stream between them
constexpr int64_t kRowsMaxPixels = 32;
// Past two pixel tiles: reductions long enough that a wave per chunk of them is a shorter chain than the tiled kernels' steps, while
// what the tiles stream between them stays small (us, tiled / so: 49 pixels of 512 -> 512 4.1 / 3.3, 400 of them 4.2 / 3.7, 400 of 960 ->
// 160 5.0 / 4.0, 1600 of 512 -> 128 4.2 / 3.7; shorter reductions 400 of 160 -> 960 3.8 / 3.9, 1600 of 64 -> 256 3.6 / 4.0; more to stream
// 784 of 1024 -> 512, 26 MB, 5.0 / 5.3, 1600 of 1536 -> 256, 39 MB, 5.6 / 7.7).  Past 1600 pixels what streams little still gains and
// the rest does not (2500 of 512 -> 64, 5 MB, 4.3 / 3.7, 4900 of them 4.4 / 4.0; 2500 of 960 -> 160, 24 MB, 5.4 / 5.3, 3136 of them
// 5.5 / 7.6; 1936 of 256 -> 128, 4 MB, 3.6 / 3.7, 4900 of them 4.5 / 4.9).
constexpr int kManyRowsMinK = 256;
constexpr int64_t kManyRowsStreamLimit = 14000000, kManyRowsMaxPixels = 1600;

bool rows_shapes_ok(int in_channels, int out_channels, int64_t pixels) {
    if (pixels <= 0 || pixels > kManyRowsMaxPixels || in_channels % 16 != 0 || out_channels % 4 != 0 || in_channels > kRowsMaxK) return false;
    const int64_t stream = (pixels + 15) / 16 * (int64_t)in_channels * out_channels;
    return pixels <= kRowsMaxPixels ? stream <= kRowsStreamLimit : in_channels >= kManyRowsMinK && stream <= kManyRowsStreamLimit;
}
bool pool_rows_ok(int in_channels, int out_channels, int64_t rows) { return rows <= kRowsMaxPixels && rows_shapes_ok(in_channels, out_channels, rows); }

// Every workgroup of the pooled launch pools its (up to 16) rows itself, on one compute unit: beyond this many values
// per workgroup the separate pool kernel, which spreads over the device, is the faster one.
bool pool_front_pays(int rows, int hw, int channels) { return (int64_t)std::min(rows, 16) * hw * channels <= (128 << 10); }

// Also of what may become half of a pair with the operator recorded next to it (launch_joined_convs), up to the pixels where one pays.
bool rows_wanted(const nncase_hip_weights *w) {
    if (!pointwise_weights(w)) return false;
    const bool pair_half = w->pixels_hint > 0 && w->pixels_hint <= 16 * kPairMaxPixelTiles && w->in_channels % 16 == 0 && w->out_channels % 4 == 0 &&
                           w->in_channels <= kPairMaxK1;
    return pair_half || rows_shapes_ok(w->in_channels, w->out_channels, w->pixels_hint);
}

// A block per channel tile: the tile's fragments as pack_pair_weights lays them out, its weight sums and its bias.
constexpr int kRowsPackWaves = 4;
__global__ __launch_bounds__(kRowsPackWaves * 64) void rows_pack_kernel(RawWeights raw, const int32_t *bias_in, int n, int k, int ksteps, uint8_t *dst, int32_t *wsum,
                                                                        int32_t *bias) {
    __shared__ int32_t sums[kRowsPackWaves][16];
    const int t = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, i = lane & 15, ch = t * 16 + i;
    int32_t sum = 0;
    for (int ks = wave; ks < ksteps; ks += kRowsPackWaves) {
        const int k0 = ks * 64 + (lane >> 4) * 16;
        u32x4 d = {0u, 0u, 0u, 0u};
        if (ch < n && k0 < k) { // (k is whole pieces)
#pragma unroll
            for (int b = 0; b < 16; b++) {
                const uint32_t v = raw.ptr[(int64_t)ch * raw.oc_stride + (int64_t)(k0 + b) * raw.ic_stride];
                sum += (int32_t)v - 128;
                d[b / 4] |= (v ^ 0x80u) << (8 * (b & 3));
            }
        }
        *reinterpret_cast<u32x4 *>(dst + (((size_t)t * ksteps + ks) * 64 + lane) * 16) = d;
    }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (lane < 16) sums[wave][i] = sum;
    __syncthreads();
    if (threadIdx.x < 16) {
        int32_t s = 0;
        for (int w = 0; w < kRowsPackWaves; w++) s += sums[w][i];
        wsum[ch] = s, bias[ch] = ch < n ? bias_in[ch] : 0;
    }
}

// `raw`: the weights on the device; w->d_bias is on its way on the context's stream.
int rows_prepack(nncase_hip_ctx *ctx, nncase_hip_weights *w, const RawWeights &raw) {
    nncase_hip_qpair *pr = new (std::nothrow) nncase_hip_qpair();
    NNHIP_REQUIRE(ctx, pr, -ENOMEM, "qconv2d_prepack: out of host memory");
    pr->second = w;
    pr->n1 = w->in_channels, pr->n2 = w->out_channels;
    pr->ks2 = (pr->n1 + 63) / 64, pr->t2 = (pr->n2 + 15) / 16;
    w->rows_pack = pr; // (released with the weights, also if what follows fails)
    NNHIP_HIP(ctx, hipMalloc((void **)&pr->d_wb, (size_t)pr->t2 * pr->ks2 * 1024));
    NNHIP_HIP(ctx, hipMalloc((void **)&pr->d_wsum_b, (size_t)pr->t2 * 16 * sizeof(int32_t)));
    NNHIP_HIP(ctx, hipMalloc((void **)&pr->d_bias_b, (size_t)pr->t2 * 16 * sizeof(int32_t)));
    hipLaunchKernelGGL(rows_pack_kernel, dim3(pr->t2), dim3(kRowsPackWaves * 64), 0, ctx->stream, raw, w->d_bias, pr->n2, pr->n1, pr->ks2, pr->d_wb,
                       pr->d_wsum_b, pr->d_bias_b);
    NNHIP_LAUNCH_CHECK(ctx, "rows_pack_kernel");
    return 0;
}

void rows_free(nncase_hip_weights *w) {
    if (w && w->rows_pack) free_pair(w->rows_pack);
    if (w) w->rows_pack = nullptr;
}

bool rows_path_taken(const nncase_hip_weights *w, const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    if (!w->rows_pack) return false;
    // (a pixel's channels leave as dwords: a wider tensor's have to lie at such addresses)
    if (((c->out_channel_stride | c->out_channel_offset) & 3) != 0 || c->out_channel_offset < 0 ||
        (c->out_channel_stride ? (int64_t)c->out_channel_offset + w->out_channels > c->out_channel_stride : c->out_channel_offset != 0))
        return false;
    if (!(c->stride_h == 1 && c->stride_w == 1 && c->pad_h_before == 0 && c->pad_w_before == 0 && out_h == c->in_h && out_w == c->in_w)) return false;
    // (u8 codes, or their float32 values: the entry point turns the latter into a u8 call with the flag set)
    if (!(c->out_dtype == NNCASE_HIP_DT_U8 || (c->out_dtype == NNCASE_HIP_DT_F32 && c->dequantize_output != 0))) return false;
    return rows_shapes_ok(w->in_channels, w->out_channels, (int64_t)c->batch * out_h * out_w);
}

// Fills in how the launch is split, and launches.
static int launch_rows(nncase_hip_ctx *ctx, PairArgs &a, bool pool) {
    // pixel tiles x ranges of channel tiles, enough workgroups to spread the weights over the device; a wave per tile and chunk of
    // the reduction, up to the waves there are
    const int ptiles = (a.m + 15) / 16;
    int ranges = (a.t2 + kRowsWaves - 1) / kRowsWaves;
    const int want = std::max(1, 2 * ctx->compute_units / ptiles);
    int per = std::max(1, (a.t2 + want - 1) / want); // tiles per workgroup when as many workgroups as wanted
    if (pool) per = std::max(per, 4);                 // (every workgroup repeats the pooling)
    per = std::min(per, kRowsWaves);
    ranges = (a.t2 + per - 1) / per;
    a.tiles_per_block = per;
    const int chunks = (a.ks2 + kRowsChunk - 1) / kRowsChunk, most = std::min(chunks, kRowsWaves / per);
    a.part_steps = (chunks + most - 1) / most * kRowsChunk;
    a.parts = (a.ks2 + a.part_steps - 1) / a.part_steps;
    a.d_tiles = make_fastdiv((uint32_t)per);
    const int sy = pair_row_bytes(a.ks2, kRowsChunk);
    a.d_pieces = make_fastdiv((uint32_t)(sy - kRowPad) / 16);
    int waves = std::max(4, per * a.parts); // (four stage the rows in fewer trips than one)
    if (pool) waves = kRowsWaves; // the pooling has a thread per four channels
    const size_t lds = 16 * (size_t)sy + 256 + (size_t)(a.parts - 1) * per * kRowsShareBytes;
    NNHIP_HIP(ctx, hipSetDevice(ctx->device));
    if (pool) hipLaunchKernelGGL(qpointwise_rows_kernel<true>, dim3(ptiles, ranges), dim3(waves * 64), lds, ctx->stream, a);
    else hipLaunchKernelGGL(qpointwise_rows_kernel<false>, dim3(ptiles, ranges), dim3(waves * 64), lds, ctx->stream, a);
    NNHIP_LAUNCH_CHECK(ctx, "qpointwise_rows_kernel");
    return 0;
}

int launch_qconv_rows(nncase_hip_ctx *ctx, const uint8_t *x, const nncase_hip_weights *w, void *y, const nncase_hip_conv2d_args_t *c,
                      const PoolFront *pool) {
    const nncase_hip_qpair *pr = w->rows_pack;
    const int64_t m64 = (int64_t)c->batch * c->in_h * c->in_w;
    NNHIP_REQUIRE(ctx, m64 > 0 && m64 < ((int64_t)1 << 30), -EINVAL, "qconv2d: %lld output pixels unsupported", (long long)m64);
    NNHIP_REQUIRE(ctx, (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0,
                  -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION, "qconv2d: activation buffers must be 16-byte aligned");
    PairArgs a;
    memset(&a, 0, sizeof(a));
    a.x = x, a.y2 = reinterpret_cast<uint8_t *>(y);
    a.wb = pr->d_wb, a.bias_b = pr->d_bias_b, a.wsum_b = pr->d_wsum_b;
    a.lut_b = w->d_post_lut;
    a.m = (int)m64;
    a.n1 = pr->n1, a.n2 = pr->n2, a.ks2 = pr->ks2, a.t2 = pr->t2;
    a.zxb = c->x_qp.zero_point - 128, a.zwb = w->zw - 128;
    const int rc = make_epilogue(ctx, &a.ep_b, c->x_qp.scale, w->sw, c->y_qp, c->clamp_min, c->clamp_max, NNCASE_HIP_DT_U8, "qconv2d");
    if (rc) return rc;
    const int res = make_residual_epilogue(ctx, &a.rep_b, c, w);
    if (res) return res;
    a.ldy = c->out_channel_stride ? c->out_channel_stride : w->out_channels, a.y_coff = c->out_channel_offset;
    NNHIP_REQUIRE(ctx, m64 * a.ldy < ((int64_t)1 << 40), -EINVAL, "qconv2d: output too large");
    if (c->dequantize_output != 0) {
        const nncase_hip_quant_param_t last = c->residual_dev ? c->sum_qp : (w->d_post_lut ? w->post_lut_qp : c->y_qp);
        a.deq = 1, a.deq_zero = last.zero_point, a.deq_scale = last.scale;
    }
    if (pool) {
        NNHIP_REQUIRE(ctx, pool->hw > 0 && (int64_t)m64 * pool->hw * pr->n1 < ((int64_t)1 << 31), -EINVAL, "qglobal_avgpool_qconv2d: input too large");
        a.pool_hw = pool->hw;
        a.pool_zx = (float)pool->x_qp.zero_point, a.pool_sx = pool->x_qp.scale;
        a.pool_zy = (float)c->x_qp.zero_point, a.pool_sy = c->x_qp.scale;
    }
    return launch_rows(ctx, a, pool != nullptr);
}
} // namespace nnhip

void nnhip::describe_pair(const nncase_hip_ctx *ctx, const nncase_hip_qpair *pr, const nncase_hip_conv2d_args_t *first, bool dw, char *buf, size_t cap) {
    const bool apart = split_pair((int64_t)first->batch * first->in_h * first->in_w, pr->k1, pr->n1, pr->n2, dw, ctx->compute_units).apart;
    snprintf(buf, cap, "%s", apart ? "qpointwise_rows+qpointwise_rows" : dw ? "dw3x3+qpointwise_pair_kernel" : "qpointwise_pair_kernel");
}

// dw / da: the depthwise convolution in front and its arguments, or null; y0_dev: where its result is stored too, or null
static int launch_pair(nncase_hip_ctx *ctx, const char *who, const uint8_t *x_dev, const nncase_hip_weights *dw,
                       const nncase_hip_conv2d_args_t *da, const nncase_hip_qpair *pr, uint8_t *y1_dev, uint8_t *y2_dev,
                       const nncase_hip_conv2d_args_t *fa, const nncase_hip_conv2d_args_t *sa, uint8_t *y0_dev = nullptr) {
    NNHIP_REQUIRE(ctx, x_dev && pr && y1_dev && y2_dev && fa && sa, -EINVAL, "%s: null argument", who);
    NNHIP_REQUIRE(ctx, fa->batch > 0 && fa->in_h > 0 && fa->in_w > 0, -EINVAL, "%s: non-positive input shape", who);
    NNHIP_REQUIRE(ctx, sa->batch == fa->batch && sa->in_h == fa->in_h && sa->in_w == fa->in_w, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                  "%s: the second convolution reads [%d,%d,%d], the first writes [%d,%d,%d]", who, sa->batch, sa->in_h, sa->in_w, fa->batch,
                  fa->in_h, fa->in_w);
    for (const nncase_hip_conv2d_args_t *c : {fa, sa}) {
        NNHIP_REQUIRE(ctx, c->stride_h == 1 && c->stride_w == 1 && c->pad_h_before == 0 && c->pad_h_after == 0 && c->pad_w_before == 0 &&
                               c->pad_w_after == 0,
                      -EINVAL, "%s: stride 1 and no padding only for the 1x1 convolutions", who);
    }
    for (const nncase_hip_conv2d_args_t *c : {fa, sa, da}) {
        if (!c) continue;
        NNHIP_REQUIRE(ctx, c->out_dtype == NNCASE_HIP_DT_U8 && c->dequantize_output == 0, -NNCASE_HIP_ERR_DATATYPE_MISMATCH, "%s: u8 results only",
                      who);
        NNHIP_REQUIRE(ctx, c->out_channel_stride == 0 && c->out_channel_offset == 0, -EINVAL, "%s: dense results only", who);
        NNHIP_REQUIRE(ctx, c->x_qp.zero_point >= 0 && c->x_qp.zero_point <= 255, -EINVAL, "%s: input zero point %d outside u8", who,
                      c->x_qp.zero_point);
        NNHIP_REQUIRE(ctx, c->y_qp.scale > 0.f && std::isfinite(c->y_qp.scale) && c->y_qp.zero_point >= 0 && c->y_qp.zero_point <= 255, -EINVAL,
                      "%s: output quantisation outside u8", who);
    }
    NNHIP_REQUIRE(ctx, !sa->residual_dev, -EINVAL, "%s: only the first 1x1 convolution takes a residual", who);
    if (fa->residual_dev)
        NNHIP_REQUIRE(ctx, fa->sum_qp.scale > 0.f && std::isfinite(fa->sum_qp.scale) && fa->sum_qp.zero_point >= 0 && fa->sum_qp.zero_point <= 255,
                      -EINVAL, "%s: sum quantisation outside u8", who);
    const int64_t m64 = (int64_t)fa->batch * fa->in_h * fa->in_w;
    NNHIP_REQUIRE(ctx, m64 < ((int64_t)1 << 30), -EINVAL, "%s: %lld pixels unsupported", who, (long long)m64);
    NNHIP_REQUIRE(ctx, ((reinterpret_cast<uintptr_t>(x_dev) | reinterpret_cast<uintptr_t>(y1_dev) | reinterpret_cast<uintptr_t>(y2_dev)) & 15u) == 0,
                  -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION, "%s: activation buffers must be 16-byte aligned", who);

    PairArgs a;
    memset(&a, 0, sizeof(a));
    a.x = x_dev, a.y0 = y0_dev, a.y1 = y1_dev, a.y2 = y2_dev;
    a.wa = pr->d_wa, a.wb = pr->d_wb;
    a.bias_a = pr->d_bias_a, a.wsum_a = pr->d_wsum_a, a.bias_b = pr->d_bias_b, a.wsum_b = pr->d_wsum_b;
    a.lut_a = pr->first->d_post_lut, a.lut_b = pr->second->d_post_lut;
    a.m = (int)m64;
    a.k1 = pr->k1, a.n1 = pr->n1, a.n2 = pr->n2;
    a.ldy = a.n2;
    a.ks1 = pr->ks1, a.ks2 = pr->ks2, a.t1 = pr->t1, a.t2 = pr->t2;
    a.zxa = fa->x_qp.zero_point - 128, a.zwa = pr->first->zw - 128;
    a.zxb = sa->x_qp.zero_point - 128, a.zwb = pr->second->zw - 128;
    int rc = make_epilogue(ctx, &a.ep_a, fa->x_qp.scale, pr->first->sw, fa->y_qp, fa->clamp_min, fa->clamp_max, NNCASE_HIP_DT_U8, who);
    if (!rc) rc = make_epilogue(ctx, &a.ep_b, sa->x_qp.scale, pr->second->sw, sa->y_qp, sa->clamp_min, sa->clamp_max, NNCASE_HIP_DT_U8, who);
    if (!rc) rc = make_residual_epilogue(ctx, &a.rep_a, fa, pr->first);
    if (rc) return rc;
    if (dw) {
        NNHIP_REQUIRE(ctx, da, -EINVAL, "%s: null argument", who);
        NNHIP_REQUIRE(ctx, dw->kind == nncase_hip_weights::kDepthwise && dw->kernel_h == 3 && dw->kernel_w == 3 && dw->out_channels == pr->k1, -EINVAL,
                      "%s: the convolution in front must be a 3x3 depthwise convolution over the first 1x1 convolution's %d channels", who, pr->k1);
        NNHIP_REQUIRE(ctx, !dw->d_post_lut && !da->residual_dev, -EINVAL, "%s: the depthwise convolution takes no table or residual", who);
        NNHIP_REQUIRE(ctx, da->stride_h == da->stride_w && (da->stride_h == 1 || da->stride_h == 2) && da->dilation_h == 1 && da->dilation_w == 1,
                      -EINVAL, "%s: depthwise stride 1 or 2, no dilation", who);
        NNHIP_REQUIRE(ctx, da->pad_h_before >= 0 && da->pad_h_after >= 0 && da->pad_w_before >= 0 && da->pad_w_after >= 0, -EINVAL,
                      "%s: negative padding", who);
        NNHIP_REQUIRE(ctx, da->in_h > 0 && da->in_w > 0, -EINVAL, "%s: non-positive input shape", who);
        const int out_h = windowed_output_size(da->in_h, 3, da->stride_h, 1, da->pad_h_before, da->pad_h_after);
        const int out_w = windowed_output_size(da->in_w, 3, da->stride_w, 1, da->pad_w_before, da->pad_w_after);
        NNHIP_REQUIRE(ctx, da->batch == fa->batch && out_h == fa->in_h && out_w == fa->in_w, -NNCASE_HIP_ERR_SHAPE_MISMATCH,
                      "%s: the depthwise convolution writes [%d,%d,%d], the first 1x1 convolution reads [%d,%d,%d]", who, da->batch, out_h, out_w,
                      fa->batch, fa->in_h, fa->in_w);
        NNHIP_REQUIRE(ctx, da->y_qp.zero_point == fa->x_qp.zero_point && da->y_qp.scale == fa->x_qp.scale, -EINVAL,
                      "%s: the first 1x1 convolution must read the depthwise result with the quantisation it is written with", who);
        NNHIP_REQUIRE(ctx, (int64_t)da->batch * da->in_h * da->in_w * pr->k1 < ((int64_t)1 << 31), -EINVAL, "%s: input of 2 GiB or more", who);
        a.dw_w = reinterpret_cast<const int16_t *>(dw->d_packed), a.dw_bias = dw->d_bias, a.dw_wsum = dw->d_wsum;
        a.in_h = da->in_h, a.in_w = da->in_w, a.out_w = out_w, a.out_hw = out_h * out_w;
        a.stride = da->stride_h, a.pad_h = da->pad_h_before, a.pad_w = da->pad_w_before;
        a.d_out_hw = make_fastdiv((uint32_t)a.out_hw), a.d_out_w = make_fastdiv((uint32_t)out_w);
        a.dw_zx = da->x_qp.zero_point;
        rc = make_epilogue(ctx, &a.ep_dw, da->x_qp.scale, dw->sw, da->y_qp, da->clamp_min, da->clamp_max, NNCASE_HIP_DT_U8, who);
        if (rc) return rc;
    }

    const PairSplit split = split_pair(a.m, pr->k1, pr->n1, pr->n2, dw != nullptr, ctx->compute_units);
    a.tiles_per_block = split.tiles_per_block;
    const int waves = split.waves;
    const bool small = split.small;
    NNHIP_HIP(ctx, hipSetDevice(ctx->device));
    if (split.apart) {
        PairArgs one = a;
        one.ldy = a.n1, one.y2 = y1_dev, one.wb = a.wa, one.bias_b = a.bias_a, one.wsum_b = a.wsum_a, one.lut_b = a.lut_a;
        one.n1 = a.k1, one.n2 = a.n1, one.ks2 = a.ks1, one.t2 = a.t1, one.zxb = a.zxa, one.zwb = a.zwa, one.ep_b = a.ep_a, one.rep_b = a.rep_a;
        rc = launch_rows(ctx, one, false);
        if (rc) return rc;
        a.x = y1_dev;
        return launch_rows(ctx, a, false);
    }
    const int pt = split.pixels;
    const dim3 grid((a.m + pt - 1) / pt, split.ranges), block(waves * 64);
    if (dw) {
        a.d_quads = make_fastdiv((uint32_t)pr->k1 / 4);
        a.dw_groups = std::min(waves * 64 / (pr->k1 / 4), pt);
    }
    auto go = [&](auto kernel, int ka, int kb) { // (rows of whole chunks)
        const int sx = pair_row_bytes(a.ks1, ka), sy = pair_row_bytes(a.ks2, kb);
        a.d_pieces = make_fastdiv((uint32_t)(sx - kRowPad) / 16);
        hipLaunchKernelGGL(kernel, grid, block, pt * (size_t)(sx + sy) + 512, ctx->stream, a);
    };
    if (split.once) {
#define NNHIP_PAIR_CASE(KA, KB, MAXW, OCC)                                               \
    do {                                                                                 \
        if (!dw) go(qpointwise_pair_once_kernel<KA, KB, MAXW, OCC, false, 16>, 1, 1);    \
        else if (pt == 16) go(qpointwise_pair_once_kernel<KA, KB, MAXW, OCC, true, 16>, 1, 1); \
        else if (pt == 8) go(qpointwise_pair_once_kernel<KA, KB, MAXW, OCC, true, 8>, 1, 1);   \
        else go(qpointwise_pair_once_kernel<KA, KB, MAXW, OCC, true, 4>, 1, 1);          \
    } while (0)
        if (small) NNHIP_PAIR_CASE(4, 2, 16, 4);
        else if (a.ks1 <= 8 && a.ks2 <= 2) NNHIP_PAIR_CASE(8, 2, 12, 3);
        else if (a.ks1 <= 8) NNHIP_PAIR_CASE(8, 4, 12, 3);
        else if (a.ks1 <= 12) NNHIP_PAIR_CASE(12, 4, 12, 3);
        else NNHIP_PAIR_CASE(16, 4, 12, 3);
#undef NNHIP_PAIR_CASE
    } else if (small) {
        dw ? go(qpointwise_pair_kernel<4, 2, 16, 4, true>, 4, 2) : go(qpointwise_pair_kernel<4, 2, 16, 4, false>, 4, 2);
    } else {
        dw ? go(qpointwise_pair_kernel<8, 4, 12, 3, true>, 8, 4) : go(qpointwise_pair_kernel<8, 4, 12, 3, false>, 8, 4);
    }
    NNHIP_LAUNCH_CHECK(ctx, "qpointwise_pair_kernel");
    return 0;
}

// ---- operators recorded one behind the other, as one launch ---------------------------------------------------------------
namespace nnhip {
struct Range {
    const uint8_t *p;
    size_t bytes;
};
static bool apart(Range a, Range b) { return !a.p || !b.p || a.p + a.bytes <= b.p || b.p + b.bytes <= a.p; }

static bool plain_u8(const nncase_hip_conv2d_args_t &c) { // what launch_pair would refuse stays with the operators' own entry points
    auto fits = [](const nncase_hip_quant_param_t &q) { return q.scale > 0.f && std::isfinite(q.scale) && q.zero_point >= 0 && q.zero_point <= 255; };
    return c.out_dtype == NNCASE_HIP_DT_U8 && c.dequantize_output == 0 && c.out_channel_stride == 0 && c.out_channel_offset == 0 && c.batch > 0 &&
           c.in_h > 0 && c.in_w > 0 && fits(c.x_qp) && fits(c.y_qp) && (!c.residual_dev || fits(c.sum_qp));
}
static int64_t pixels_of(const nncase_hip_conv2d_args_t &c) { return (int64_t)c.batch * c.in_h * c.in_w; }

// Two convolutions as a pair over the fragments that each of them carries for its few-pixel kernel.
static bool as_pair(const nncase_hip_ctx *ctx, const JoinedConv &first, const JoinedConv &second, nncase_hip_qpair *pr) {
    for (const JoinedConv *j : {&first, &second}) {
        const nncase_hip_conv2d_args_t &c = *j->args;
        if (!j->weights->rows_pack || !plain_u8(c) || c.stride_h != 1 || c.stride_w != 1 || c.pad_h_before || c.pad_h_after || c.pad_w_before ||
            c.pad_w_after)
            return false;
    }
    const nncase_hip_conv2d_args_t &fa = *first.args, &sa = *second.args;
    const int k1 = first.weights->in_channels, n1 = first.weights->out_channels, n2 = second.weights->out_channels;
    if (second.x != first.y || second.weights->in_channels != n1 || sa.residual_dev || sa.batch != fa.batch || sa.in_h != fa.in_h || sa.in_w != fa.in_w ||
        !nncase_hip_qpointwise_pair_supported(k1, n1, n2))
        return false;
    const int64_t m = pixels_of(fa);
    if (m >= ((int64_t)1 << 30) || !pair_pays(m, k1, n1, n2, ctx->compute_units) || split_pair(m, k1, n1, n2, false, ctx->compute_units).apart) return false;
    // (every range of the second convolution reads the pixels and the residual again, while others store)
    const Range x{first.x, (size_t)m * k1}, res{reinterpret_cast<const uint8_t *>(fa.residual_dev), (size_t)m * n1}, y1{first.y, (size_t)m * n1},
        y2{second.y, (size_t)m * n2};
    if (!apart(x, y1) || !apart(x, y2) || !apart(res, y1) || !apart(res, y2) || !apart(y1, y2)) return false;
    const nncase_hip_qpair *a = first.weights->rows_pack, *b = second.weights->rows_pack;
    pr->first = first.weights, pr->second = second.weights;
    pr->k1 = k1, pr->n1 = n1, pr->n2 = n2, pr->ks1 = a->ks2, pr->ks2 = b->ks2, pr->t1 = a->t2, pr->t2 = b->t2;
    pr->d_wa = a->d_wb, pr->d_wsum_a = a->d_wsum_b, pr->d_bias_a = a->d_bias_b, pr->d_wb = b->d_wb, pr->d_wsum_b = b->d_wsum_b, pr->d_bias_b = b->d_bias_b;
    return true;
}

// Whether the depthwise convolution joins the launch of the pair that reads its result.
static bool front_joins(const nncase_hip_ctx *ctx, const JoinedConv &dw, const nncase_hip_qpair &pr, const JoinedConv &first, const JoinedConv &second) {
    const nncase_hip_conv2d_args_t &da = *dw.args, &fa = *first.args;
    const nncase_hip_weights &w = *dw.weights;
    if (w.kind != nncase_hip_weights::kDepthwise || w.kernel_h != 3 || w.kernel_w != 3 || w.out_channels != pr.k1 || w.d_post_lut || !plain_u8(da) ||
        da.residual_dev || da.stride_h != da.stride_w || (da.stride_h != 1 && da.stride_h != 2) || da.dilation_h != 1 || da.dilation_w != 1 ||
        da.pad_h_before < 0 || da.pad_h_after < 0 || da.pad_w_before < 0 || da.pad_w_after < 0)
        return false;
    if (first.x != dw.y || !plain_u8(fa) || !plain_u8(*second.args) || da.batch != fa.batch ||
        windowed_output_size(da.in_h, 3, da.stride_h, 1, da.pad_h_before, da.pad_h_after) != fa.in_h ||
        windowed_output_size(da.in_w, 3, da.stride_w, 1, da.pad_w_before, da.pad_w_after) != fa.in_w ||
        da.y_qp.zero_point != fa.x_qp.zero_point || da.y_qp.scale != fa.x_qp.scale)
        return false;
    const int64_t m = pixels_of(fa), in_bytes = pixels_of(da) * pr.k1;
    if (in_bytes >= ((int64_t)1 << 31) || m >= ((int64_t)1 << 30) || (reinterpret_cast<uintptr_t>(dw.x) & 15u) != 0 ||
        !front_pays(m, pr.k1, pr.n1, pr.n2, ctx->compute_units))
        return false;
    const Range x{dw.x, (size_t)in_bytes}, mid{dw.y, (size_t)m * pr.k1}, res{reinterpret_cast<const uint8_t *>(fa.residual_dev), (size_t)m * pr.n1},
        y1{first.y, (size_t)m * pr.n1}, y2{second.y, (size_t)m * pr.n2};
    return apart(x, mid) && apart(x, y1) && apart(x, y2) && apart(mid, res) && apart(mid, y1) && apart(mid, y2);
}

int launch_joined_convs(nncase_hip_ctx *ctx, const JoinedConv *dw, const nncase_hip_qpair *pair, const JoinedConv &first, const JoinedConv &second, bool *taken) {
    *taken = false;
    nncase_hip_qpair made; // (borrows what it points to)
    if (!pair) {
        if (!as_pair(ctx, first, second, &made)) return 0;
        pair = &made;
    }
    if (dw && !front_joins(ctx, *dw, *pair, first, second)) return 0;
    const uint8_t *const x = dw ? dw->x : first.x;
    for (const uint8_t *p : {x, (const uint8_t *)first.y, (const uint8_t *)second.y})
        if ((reinterpret_cast<uintptr_t>(p) & 15u) != 0) return 0;
    *taken = true;
    return launch_pair(ctx, dw ? "qdepthwise_pointwise_pair" : "qpointwise_pair", x, dw ? dw->weights : nullptr, dw ? dw->args : nullptr, pair, first.y,
                       second.y, first.args, second.args, dw ? dw->y : nullptr);
}
} // namespace nnhip

extern "C" int nncase_hip_qpointwise_pair(nncase_hip_ctx_t *ctx, const uint8_t *x_dev, const nncase_hip_qpair_t *pair, uint8_t *y1_dev,
                                          uint8_t *y2_dev, const nncase_hip_conv2d_args_t *first_args,
                                          const nncase_hip_conv2d_args_t *second_args) {
    NNHIP_CHECK_CTX(ctx);
    return launch_pair(ctx, "qpointwise_pair", x_dev, nullptr, nullptr, pair, y1_dev, y2_dev, first_args, second_args);
}

extern "C" int nncase_hip_qdepthwise_pointwise_pair(nncase_hip_ctx_t *ctx, const uint8_t *x_dev, const nncase_hip_weights_t *depthwise,
                                                    const nncase_hip_conv2d_args_t *depthwise_args, const nncase_hip_qpair_t *pair,
                                                    uint8_t *y1_dev, uint8_t *y2_dev, const nncase_hip_conv2d_args_t *first_args,
                                                    const nncase_hip_conv2d_args_t *second_args) {
    NNHIP_CHECK_CTX(ctx);
    NNHIP_REQUIRE(ctx, depthwise && depthwise_args, -EINVAL, "qdepthwise_pointwise_pair: null argument");
    return launch_pair(ctx, "qdepthwise_pointwise_pair", x_dev, depthwise, depthwise_args, pair, y1_dev, y2_dev, first_args, second_args);
}
