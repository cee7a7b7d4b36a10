// u8/u8 convolution over a window to codes or float32, with the input of a two-dimensional tile of output pixels in LDS.
//
// The implicit-GEMM kernels fetch, re-bias and sum an activation once per tap of the window: nine times for 3x3, a hundred
// instructions of a wave per k-step against eight products, and an instruction of a wave that is alone on its SIMD takes eight
// to nine cycles.  Here a block brings the input under its tile of output pixels into LDS once (re-biased, the padding filled
// with the zero point) and every tap is an LDS read at another offset; the sum of x over a window, which the weight zero
// point multiplies, is the sum of per-pixel channel sums taken on the way in.  What is left of a k-step is RG + 1 LDS reads
// (operands and where the next tap lies), T loads of packed weights straight into registers, four k-steps ahead, and the
// products: no barrier, no staging.  A wave owns RG * 16 pixels x T * 16 channels; a block is WM x WN waves.
//   * weights come from L2 through the vector L1 (64 bytes per clock): with 64 x 32 outputs per wave a k-step of four waves
//     takes 8 KiB of them for 128 clocks of matrix work, so waves share pixels rather than channels where they can;
//   * blocks start the reduction at different k-steps (integer sums do not care): otherwise all of them wait for the same
//     weights to come from memory at the same time, step after step;
//   * results leave through LDS as whole pixel rows, whose bytes of a residual are asked for before the sums meet;
//   * what a block does before its first request and after its last product counts as much as the reduction: all arguments of the
//     requests in one trip and those of the stores in another, a thread that keeps its piece of a pixel (two multiply-adds an address,
//     short divisions), a channel's terms asked for first.  Start to end of a block, 6400 pixels 64 -> 64 3x3 with a residual 4.6 us ->
//     3.7 (before the first request 0.6 -> 0.4, requests 0.5 -> 0.3, results 1.1 -> 0.5), 409 600 pixels 32 -> 32 21.8 -> 19.2 a launch.
//   * a launch of few blocks splits each one's k-steps between groups of waves, which meet once: up to four k-steps of every group are on
//     their way when the first product starts, where the ring of qconv_wide_kernel goes through a barrier for each.  In a chain, us there /
//     here: 128 -> 128 3x3 of 1600 pixels 5.3 / 4.0, 256 -> 256 of 400 6.8 / 4.7, 512 -> 512 of 400 11.0 / 7.9.
//   * float32 results leave the same way, four pieces for sixteen channels (116 layers of 8 to 640 channels 1.38 times as quick in the
//     mean as by the ring; 441 -> 29 3x3 stride 2 of 2601 pixels 13.0 / 6.1, 80 -> 12 5x5 of 54 675 16.0 / 9.4); int32 stays there.
// Arithmetic, weight packing and the bytes of the result are those of qconv_igemm.hpp.
#pragma once

#include "qconv_rules.hpp"
#include "qconv_wide.hpp"

namespace nnhip {

__device__ __forceinline__ int tile_div(int p, uint32_t mul) { return (int)(__umul24((uint32_t)p, mul) >> 20); } // make_tile_div

// LDS for the sums of `units` results of each wave that the groups of a split reduction pass on.
constexpr int tile_part_bytes(int units, int waves, int groups) { return units * (groups - 1) * waves * 1024; }

struct TileArgs {
    int th, tw;                    // output tile
    int hr, hc;                    // input rows / columns under it
    int half;                      // input columns per column phase (stride 2: column c lies at (c & 1) * half + c / 2, so that
                                   // neighbouring output pixels read neighbouring LDS pixels)
    int pitch, row_pitch;          // bytes of an LDS pixel (an odd number of 16-byte pieces: eight lanes, eight banks) / row
    int pieces;                    // 16-byte pieces per pixel
    int apart, dc, dr;             // whole pixels that a block's threads cover at once, and that as a step in (column, row)
    int row_bytes;                 // of the tensor
    int tile_off;
    int ragged;                    // channels of a group that are no multiple of 16
    uint32_t d_pieces, d_hc, d_tw; // of make_tile_div
    FastDiv d_tx, d_txy, d_nchunks, d_rest;
};

// Pixels x channels of a block; by n: its k-steps shared by n groups of waves.
enum TileShape {
    kTile128x32, kTile64x32, kTile32x64, kTile128x128, kTile64x128,
    kTile32x32by2, kTile32x32by4, kTile16x32by4, kTile32x64by2, kTile32x64by4, kTile16x64by4,
    kTileNone
};

struct TilePlan {
    TileShape shape = kTileNone;
    TileArgs t;
    int tiles; // of the whole batch
    size_t lds;
};

// The plan of a call (the same for every group of a grouped layer); shape kTileNone: not a layer of this kernel.
TilePlan plan_qconv_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, bool ragged, int tiles, int nchunks);
int launch_qconv_tile(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks);
int launch_tile_ragged(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks); // (qconv_tile_ragged.hip)

// A launch's results: codes; codes whose requantisation is the one-instruction form without a clamp of its own (Epilogue::fast and ::full);
// float32.
enum TileOut { kTileCodes, kTileFastCodes, kTileFloats };

// What a launch's last stage takes of the arguments, in one trip: fetched ahead, the values would be spilled while the reduction runs,
// and a request of the first stage would wait behind them.
template <TileOut OUT> __device__ __forceinline__ IgemmArgs gather_store_args() {
    auto p = (const __attribute__((address_space(4))) IgemmArgs *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    const IgemmArgs &a = *(const IgemmArgs *)p;
    IgemmArgs l; // (what is not assigned here is not used)
    if constexpr (OUT == kTileFloats) {
        l.ep.mult = a.ep.mult, l.ep.lo = a.ep.lo, l.ep.hi = a.ep.hi;
        l.y = a.y, l.n = a.n, l.ldy = a.ldy, l.y_coff = a.y_coff, l.zwp = a.zwp, l.m = a.m, l.d_ohow.div = a.d_ohow.div, l.d_ow.div = a.d_ow.div;
        asm volatile("" ::"s"(l.ep.mult), "s"(l.ep.lo), "s"(l.ep.hi), "s"(l.y), "s"(l.n), "s"(l.ldy), "s"(l.y_coff), "s"(l.zwp), "s"(l.m),
                     "s"(l.d_ohow.div), "s"(l.d_ow.div));
        return l;
    }
    l.ep.c1 = a.ep.c1, l.ep.c2 = a.ep.c2;
    if constexpr (OUT == kTileCodes) {
        l.ep.mult = a.ep.mult, l.ep.sy = a.ep.sy, l.ep.rsy = a.ep.rsy, l.ep.zy = a.ep.zy, l.ep.qlo = a.ep.qlo, l.ep.qhi = a.ep.qhi;
        l.ep.fast = a.ep.fast, l.ep.full = a.ep.full;
        asm volatile("" ::"s"(l.ep.mult), "s"(l.ep.sy), "s"(l.ep.rsy), "s"(l.ep.zy), "s"(l.ep.qlo), "s"(l.ep.qhi), "s"(l.ep.fast), "s"(l.ep.full));
    }
    l.rep.res = a.rep.res, l.rep.zy = a.rep.zy, l.rep.sy = a.rep.sy, l.rep.zr = a.rep.zr, l.rep.sr = a.rep.sr;
    l.rep.sum.sy = a.rep.sum.sy, l.rep.sum.rsy = a.rep.sum.rsy, l.rep.sum.zy = a.rep.sum.zy, l.rep.sum.qlo = a.rep.sum.qlo, l.rep.sum.qhi = a.rep.sum.qhi;
    l.y = a.y, l.m = a.m, l.n = a.n, l.ldy = a.ldy, l.y_coff = a.y_coff, l.ldr = a.ldr, l.r_coff = a.r_coff, l.zwp = a.zwp, l.lut = a.lut;
    l.d_ohow.div = a.d_ohow.div, l.d_ow.div = a.d_ow.div;
    asm volatile("" ::"s"(l.ep.c1), "s"(l.ep.c2), "s"(l.rep.res), "s"(l.rep.zy), "s"(l.rep.sy), "s"(l.rep.zr), "s"(l.rep.sr), "s"(l.rep.sum.sy), "s"(l.rep.sum.rsy),
                 "s"(l.rep.sum.zy), "s"(l.rep.sum.qlo), "s"(l.rep.sum.qhi), "s"(l.y), "s"(l.m), "s"(l.n), "s"(l.ldy), "s"(l.y_coff), "s"(l.ldr), "s"(l.r_coff),
                 "s"(l.zwp), "s"(l.lut), "s"(l.d_ohow.div), "s"(l.d_ow.div));
    return l;
}

// KG > 1: KG groups of WM x WN waves share the reduction, every KG-th k-step each, and add their sums up at the end.
// RAGGED: channels that are no multiple of 16, at any byte (qconv_igemm.hip packs the weights such that what else a piece holds adds nothing).
template <int T, int RG, int WM, int WN, int KG, TileOut OUT, bool RAGGED>
__global__ __launch_bounds__(WM * WN * KG * 64, 4) void qconv_tile_kernel(const IgemmArgs a, const TileArgs t) {
    constexpr int THREADS = WM * WN * KG * 64, PIX = WM * RG * 16, TB = T * WN;
    constexpr int D = 4;                                             // k-steps of weights in flight
    constexpr int UNITS = RG * T, EACH = (UNITS + KG - 1) / KG;      // results of a wave, 16 pixels x 16 channels; those that a group finishes
    static_assert(TB * 16 <= THREADS && THREADS <= kTileDivMost, "a thread per channel, tile_div");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    int32_t *cterm = reinterpret_cast<int32_t *>(smem);              // [TB * 16]
    int32_t *sums = cterm + TB * 16;                                 // [KG][PIX] sum of x' over a group's share of a pixel's window
    uint8_t *lutl = reinterpret_cast<uint8_t *>(sums + KG * PIX);    // [256]
    v4i *parts = reinterpret_cast<v4i *>(lutl + 256);                // [UNITS][KG - 1][waves of a group][64] sums on their way to the group that finishes them
    int32_t *taps = reinterpret_cast<int32_t *>(lutl + 256 + tile_part_bytes(UNITS, WM * WN, KG)); // [KS + 2 KG][4] LDS offset of a piece of the reduction
    uint8_t *tile = smem + t.tile_off;

    // (what the requests need, in one trip; see gather_store_args for the rest)
    asm volatile("" ::"s"(a.x), "s"(a.x_bytes), "s"(a.wpk), "s"(a.bias), "s"(a.wsum), "s"(a.lut), "s"(a.ksteps), "s"(a.ldx), "s"(a.x_coff), "s"(a.in_h), "s"(a.in_w),
                 "s"(a.stride_h), "s"(a.stride_w), "s"(a.pad_h), "s"(a.pad_w), "s"(a.num_mtiles), "s"(a.n));
    asm volatile("" ::"s"(t.th), "s"(t.tw), "s"(t.hr), "s"(t.hc), "s"(t.half), "s"(t.pitch), "s"(t.row_pitch), "s"(t.pieces), "s"(t.apart), "s"(t.dc), "s"(t.dr),
                 "s"(t.row_bytes), "s"(t.d_pieces), "s"(t.d_hc), "s"(t.d_txy.mul), "s"(t.d_txy.shift), "s"(t.d_txy.div), "s"(t.d_tx.mul), "s"(t.d_tx.shift),
                 "s"(t.d_tx.div), "s"(t.d_nchunks.mul), "s"(t.d_nchunks.shift), "s"(t.d_nchunks.div));

    // as in qconv_wide_kernel: channel chunks of a tile back to back, a contiguous eighth of the tiles per XCD
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
    const int turn = (int)fastdiv((uint32_t)seq, t.d_nchunks), chunk = seq - turn * (int)t.d_nchunks.div;
    const int per = (a.num_mtiles + 7) >> 3;
    const int mt = xcd * per + turn;
    if (turn >= per || mt >= a.num_mtiles) return;

    const int tid = threadIdx.x, lane = tid & 63;
    const int bwave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = KG == 1 ? 0 : bwave / (WM * WN), wave = bwave - kg * (WM * WN);
    const int wm = wave % WM, wn = wave / WM;
    const int j = lane & 15, gq = lane >> 4;
    const int KS = a.ksteps;
    const int ch_base = chunk * (TB * 16);
    const bool two = a.stride_w == 2;

    // ---- a channel's terms and the byte table: asked for first, needed last ----
    int32_t bias = 0, wsum = 0;
    uint32_t table = 0;
    if (ch_base + tid < a.n && tid < TB * 16) bias = a.bias[ch_base + tid], wsum = a.wsum[ch_base + tid];
    if (a.lut && tid < 64) table = a.lut[tid];

    // ---- the input tile: requested in batches of U pieces per thread, the next before one is stored.  A thread keeps its piece of
    // a pixel and goes through the pixels t.apart at a time ----
    const uint32_t img = fastdiv((uint32_t)mt, t.d_txy);
    const uint32_t in_img = (uint32_t)mt - img * t.d_txy.div;
    const uint32_t tyi = fastdiv(in_img, t.d_tx);
    const int oy0 = (int)tyi * t.th, ox0 = (int)(in_img - tyi * t.d_tx.div) * t.tw;
    const int iy0 = oy0 * a.stride_h - a.pad_h, ix0 = ox0 * a.stride_w - a.pad_w;
    const int base = ((int)img * a.in_h + iy0) * t.row_bytes + ix0 * a.ldx + a.x_coff; // (may be negative at a border)
    const __amdgpu_buffer_rsrc_t xres = wide_rsrc(a.x, RAGGED ? ((uint32_t)a.x_bytes + 3) & ~3u : (uint32_t)a.x_bytes);
    // (ragged: the last piece of the tensor's last pixels reaches past it)
    const bool near_end = RAGGED && (int64_t)base + (int64_t)(t.hr - 1) * t.row_bytes + (t.hc - 1) * a.ldx + t.pieces * 16 > (int64_t)a.x_bytes;
    constexpr int U = 4;
    struct Batch {
        wide_u32x4 v[U];
        int dst[U];        // where the piece goes in LDS; its bit 0: the pixel lies in the padding
    };
    const int n = t.hr * t.hc; // pixels
    const bool inside = iy0 >= 0 && ix0 >= 0 && iy0 + t.hr <= a.in_h && ix0 + t.hc <= a.in_w; // no padding under this tile
    int r, c;  // row and column of this thread's next pixel
    int owned; // its pixels are those of t.apart, 2 t.apart, ... below this
    int q16;   // its piece
    {
        const int p0 = tile_div(tid, t.d_pieces);
        q16 = (tid - __mul24(p0, t.pieces)) * 16;
        r = tile_div(p0, t.d_hc);
        c = p0 - __mul24(r, t.hc);
        owned = p0 < t.apart ? n - p0 : 0; // (threads past the last whole pixel: none)
    }
    // (a thread past the tile's last pixel reads what follows it in the tensor, or 0 past its end, and drops it)
    int off[RAGGED ? U : 1];
    auto request_piece = [&](Batch &f, int u, bool in_c) __attribute__((always_inline)) {
        const int goff = __mul24(r, t.row_bytes) + (__mul24(c, a.ldx) + q16);
        f.dst[u] = __mul24(r, t.row_pitch) + (__mul24(two ? (c & 1) * t.half + (c >> 1) : c, t.pitch) + q16);
        if constexpr (RAGGED) {
            const bool in = in_c || ((unsigned)(iy0 + r) < (unsigned)a.in_h && (unsigned)(ix0 + c) < (unsigned)a.in_w);
            off[u] = in ? base + goff : 0;
            f.v[u] = load_ragged(a.x, (int)a.x_bytes, off[u]);
            f.dst[u] |= in ? 0 : 1;
        } else if (in_c) {
            f.v[u] = __builtin_amdgcn_raw_buffer_load_b128(xres, goff, base, 0);
        } else {
            const bool in = (unsigned)(iy0 + r) < (unsigned)a.in_h && (unsigned)(ix0 + c) < (unsigned)a.in_w;
            f.v[u] = __builtin_amdgcn_raw_buffer_load_b128(xres, in ? (uint32_t)(base + goff) : 0xffffffffu, 0, 0);
            f.dst[u] |= in ? 0 : 1;
        }
        c += t.dc;
        const bool carry = c >= t.hc;
        c -= carry ? t.hc : 0;
        r += t.dr + (carry ? 1 : 0);
    };
    auto request = [&](Batch &f, int i0) __attribute__((always_inline)) {
        if (inside) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * t.apart >= n) break;
                request_piece(f, u, true);
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * t.apart >= n) break;
                request_piece(f, u, false);
            }
        }
        if constexpr (RAGGED) {
            if (!near_end) return;
            bool past = false;
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * t.apart >= n) break;
                past = past || (i0 + u * t.apart < owned && off[u] > (int)a.x_bytes - 16);
            }
            if (!__any(past)) return;
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * t.apart >= n) break;
                f.v[u] = load_ragged_end(xres, off[u]);
            }
        }
    };
    auto keep = [&](const Batch &f, int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + u * t.apart;
            if (i >= n) break;
            if (i < owned) {
                const uint32_t fill = (f.dst[u] & 1) ? a.zx_splat : 0u;
                wide_u32x4 w;
#pragma unroll
                for (int d = 0; d < 4; d++) { // (a piece of the padding was read as 0; ragged: as whatever lies at 0)
                    const uint32_t x = RAGGED && (f.dst[u] & 1) ? 0u : f.v[u][d];
                    w[d] = (inside ? x : x | fill) ^ 0x80808080u;
                }
                *reinterpret_cast<wide_u32x4 *>(tile + (f.dst[u] & ~1)) = w;
            }
        }
    };
    Batch fa;
    request(fa, 0);

    // ---- weights: D k-steps ahead.  The last k-step, which may end past the reduction, comes first, the others follow from
    // where this block starts; group kg takes the kg-th of that order and every KG-th from there ----
    const __amdgpu_buffer_rsrc_t wres = wide_rsrc(a.wpk + (size_t)chunk * KS * TB * 1024, (uint32_t)KS * TB * 1024);
    const int rest = KS - 1;
    const int ks0 = rest == 0 ? 0 : seq - (int)fastdiv((uint32_t)seq, t.d_rest) * rest;
    const int w_end = rest * TB * 1024, w_lane = wn * T * 1024 + lane * 16;
    int w_off = w_end; // of the next k-step to request
    auto load_w = [&](v4i (&dst)[T]) __attribute__((always_inline)) {
#pragma unroll
        for (int nt = 0; nt < T; nt++) dst[nt] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wres, w_lane + nt * 1024, w_off, 0));
    };
    auto advance = [&](int ksteps) __attribute__((always_inline)) { // (of at most `rest`: choose_tile)
        w_off += ksteps * (TB * 1024);
        w_off -= w_off >= w_end ? w_end : 0;
    };
    auto load_next = [&](v4i (&dst)[T]) __attribute__((always_inline)) {
        load_w(dst);
        advance(KG);
    };
    v4i wf[D][T];
    if (KG == 1 || kg == 0) {
        load_w(wf[0]);
        w_off = ks0 * TB * 1024;
        if (KG > 1) advance(KG - 1);
    } else {
        w_off = ks0 * TB * 1024;
        advance(kg - 1);
        load_next(wf[0]);
    }
#pragma unroll
    for (int d = 1; d < D; d++) load_next(wf[d]);

    // ---- tables ----
    for (int e = tid; e < (KS + 2 * KG) * 4; e += THREADS) { // in the order of this block's k-steps
        const int s = e >> 2;
        int ks = s == 0 ? rest : ks0 + s - 1;
        ks -= s > 0 && ks >= rest ? rest : 0;
        const int kk = ks * 64 + (e & 3) * 16;
        int off = 0; // (past the reduction: any place, its weights are 0)
        if (kk < a.k && s < KS) {
            const uint32_t tap = fastdiv((uint32_t)kk, a.d_gic);
            const uint32_t ky = fastdiv(tap, a.d_kw);
            const int dx = ((int)tap - (int)ky * a.kw) * a.dil_w;
            off = (int)ky * a.dil_h * t.row_pitch + (two ? (dx & 1) * t.half + (dx >> 1) : dx) * t.pitch + kk - (int)tap * a.g_ic;
        }
        taps[e] = off;
    }
    // this lane's pixels: pixel (wm RG + rg) * 16 + j of the tile, in rows of tw
    auto lds_of = [&](int group) __attribute__((always_inline)) {
        const int p = (wm * RG + group) * 16 + j;
        int ty = tile_div(p, t.d_tw);
        int tx = p - __mul24(ty, t.tw);
        if (ty >= t.th) ty = tx = 0; // (surplus of the block: not stored)
        return __mul24(ty, a.stride_h * t.row_pitch) + __mul24(tx, t.pitch);
    };
    // the sum of x' of a pixel group comes from a product with ones; waves that share the pixels share that work
    constexpr int SG = (RG + WN - 1) / WN; // groups per wave
    int xbase[RG], xsum[SG];
#pragma unroll
    for (int rg = 0; rg < RG; rg++) xbase[rg] = lds_of(rg);
#pragma unroll
    for (int i = 0; i < SG; i++) xsum[i] = WN == 1 ? xbase[i] : lds_of(min(wn * SG + i, RG - 1));
    if (tid < TB * 16) cterm[tid] = bias - a.zxp * wsum + a.k * a.zxp * a.zwp;
    if (tid < 64) reinterpret_cast<uint32_t *>(lutl)[tid] = table;
    {
        int i0 = 0;
        for (; i0 + U * t.apart < n; i0 += U * t.apart) {
            Batch fb;
            request(fb, i0 + U * t.apart);
            keep(fa, i0);
            fa = fb;
        }
        keep(fa, i0);
    }
    const IgemmArgs late = gather_store_args<OUT>();
    __syncthreads();

    // ---- the reduction ----
    const int ch0 = gq * (4 * TB) + wn * (4 * T);
    v4i acc[RG][T], rs[SG];
    v4i xf[2][RG], xs[2][SG]; // (a wave reads the operand it sums by itself: which of xf that is depends on the wave)
    const int32_t *tap = taps + kg * 4 + gq; // of the k-step whose operands are read next
    int toff = tap[0];
    auto operands = [&](v4i (&dst)[RG], v4i (&dsts)[SG], int ahead) __attribute__((always_inline)) {
#pragma unroll
        for (int rg = 0; rg < RG; rg++) dst[rg] = *reinterpret_cast<const v4i *>(tile + xbase[rg] + toff);
#pragma unroll
        for (int i = 0; i < SG; i++) dsts[i] = WN == 1 ? dst[i] : *reinterpret_cast<const v4i *>(tile + xsum[i] + toff);
        toff = tap[ahead * (4 * KG)];
    };
    operands(xf[0], xs[0], 1);
    operands(xf[1], xs[1], 2);
    tap += 2 * (4 * KG);
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    {
        const int one = kg > 0 || rest * 64 + gq * 16 < a.k ? 0x01010101 : 0; // (pieces past the reduction)
        const v4i ones_last = {one, one, one, one}, zero = {0, 0, 0, 0};
#pragma unroll
        for (int nt = 0; nt < T; nt++) {
            v4i ct = *reinterpret_cast<const v4i *>(cterm + ch0 + nt * 4);
            if (KG > 1 && kg > 0) ct = zero;
#pragma unroll
            for (int rg = 0; rg < RG; rg++) acc[rg][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[0][nt], xf[0][rg], ct, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < SG; i++) rs[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones_last, xs[0][i], zero, 0, 0, 0);
    }
    load_next(wf[0]);
    // (whole groups of D k-steps without a branch between them: behind one, a wait for one k-step's weights waits for all)
    auto kstep = [&](auto u_c) __attribute__((always_inline)) {
        constexpr int u = decltype(u_c)::value, b = u % D;
        operands(xf[(u + 1) & 1], xs[(u + 1) & 1], u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nt = 0; nt < T; nt++)
#pragma unroll
            for (int rg = 0; rg < RG; rg++) acc[rg][nt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[b][nt], xf[u & 1][rg], acc[rg][nt], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < SG; i++) rs[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, xs[u & 1][i], rs[i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_next(wf[b]);
    };
    int left = KG == 1 ? rest : (rest - kg) / KG;
#pragma clang loop unroll(disable)
    for (; left >= D; left -= D) {
        static_for<1, D + 1>(kstep);
        tap += D * (4 * KG);
    }
    static_for<1, D>([&](auto u_c) __attribute__((always_inline)) {
        if (decltype(u_c)::value <= left) kstep(u_c);
    });

    // ---- epilogue ----
    // whole pixel rows: TB threads per pixel, 16 channels each.  Their bytes of the residual are asked for before the sums meet.
    // (floats: four pieces for every sixteen channels)
    constexpr int ES = OUT == kTileFloats ? 4 : 1, PIECES = TB * ES;
    constexpr int PPT = THREADS / PIECES < PIX ? THREADS / PIECES : PIX, PASSES = PIX / PPT; // pixels of a pass
    static_assert(PIX % PPT == 0, "whole passes");
    const int oh_img = (int)late.d_ohow.div, ow = (int)late.d_ow.div;
    const int cb = (tid % PIECES) * (16 / ES), ch = ch_base + cb;
    const bool whole = ch + 16 / ES <= late.n, wide_y = OUT == kTileFloats || ((late.ldy | late.y_coff) & 3) == 0;
    int px[PASSES]; // pixel index of the tensor, late.m where there is none
    u32x4 rv[PASSES];
#pragma unroll
    for (int it = 0; it < PASSES; it++) {
        const int p = it * PPT + tid / PIECES;
        const int ty = tile_div(p, t.d_tw);
        const int oy = oy0 + ty, ox = ox0 + p - __mul24(ty, t.tw);
        const int at = __mul24(oy, ow) + ox;
        px[it] = p < PIX && ty < t.th && ox < ow && at < oh_img && ch < late.n ? (int)img * oh_img + at : late.m;
    }
    if (OUT != kTileFloats && late.rep.res) {
        const bool wide_r = ((late.ldr | late.r_coff) & 3) == 0;
#pragma unroll
        for (int it = 0; it < PASSES; it++) {
            rv[it] = u32x4{0, 0, 0, 0};
            if (px[it] >= late.m) continue;
            const uint8_t *ro = late.rep.res + (size_t)px[it] * late.ldr + late.r_coff + ch;
            if (whole && wide_r) {
                const u32x4_a4 r4 = *reinterpret_cast<const u32x4_a4 *>(ro);
                rv[it] = u32x4{r4[0], r4[1], r4[2], r4[3]};
            } else {
#pragma unroll
                for (int b = 0; b < 16; b++)
                    if (ch + b < late.n) rv[it][b / 4] |= (uint32_t)ro[b] << (8 * (b & 3));
            }
        }
    }
    if (gq == 0) {
#pragma unroll
        for (int i = 0; i < SG; i++)
            if (wn * SG + i < RG) sums[kg * PIX + (wm * RG + wn * SG + i) * 16 + j] = rs[i][0];
    }
    // (unit u of a wave: pixel group u / T, channel tile u % T; group u / EACH finishes it)
    auto part = [&](int u, int from) __attribute__((always_inline)) { return parts + ((u * (KG - 1) + from) * (WM * WN) + wave) * 64 + lane; };
    if constexpr (KG > 1) {
        static_for<0, UNITS>([&](auto u_c) __attribute__((always_inline)) {
            constexpr int u = decltype(u_c)::value, by = u / EACH;
            if (kg != by) *part(u, kg - (kg > by ? 1 : 0)) = acc[u / T][u % T];
        });
    }
    __syncthreads(); // the sums are there, and every wave is through with the tile: its place takes the result
    constexpr int kOutPitch = TB * 16 * ES + 16;
    auto finish = [&](auto first_c) __attribute__((always_inline)) { // the EACH units from there on
        constexpr int first = decltype(first_c)::value, count = KG == 1 ? UNITS : (UNITS - first < EACH ? UNITS - first : EACH);
        int32_t owed[RG];
#pragma unroll
        for (int rg = first / T; rg <= (first + count - 1) / T; rg++) {
            int32_t sum = sums[(wm * RG + rg) * 16 + j];
#pragma unroll
            for (int g = 1; g < KG; g++) sum += sums[g * PIX + (wm * RG + rg) * 16 + j];
            owed[rg] = -late.zwp * sum;
        }
        uint32_t packed[count];
        if constexpr (KG > 1) {
            v4i others[count][KG - 1];
#pragma unroll
            for (int u = 0; u < count; u++)
#pragma unroll
                for (int from = 0; from < KG - 1; from++) others[u][from] = *part(first + u, from);
#pragma unroll
            for (int u = 0; u < count; u++)
#pragma unroll
                for (int from = 0; from < KG - 1; from++) acc[(first + u) / T][(first + u) % T] += others[u][from];
        }
#pragma unroll
        for (int u = 0; u < count; u++) {
            const int rg = (first + u) / T, nt = (first + u) % T;
            int32_t v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = acc[rg][nt][r] + owed[rg];
            if constexpr (OUT == kTileFloats) {
                u32x4 o;
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = __float_as_uint(clamp_ref((float)v[r] * late.ep.mult, late.ep.lo, late.ep.hi));
                *reinterpret_cast<u32x4 *>(tile + ((wm * RG + rg) * 16 + j) * kOutPitch + (ch0 + nt * 4) * 4) = o;
            } else {
                packed[u] = OUT == kTileFastCodes ? requant4_u8_packed_direct(v, late.ep) : requant4_u8_packed(v, late.ep);
            }
        }
        if constexpr (OUT == kTileFloats) return;
        if (late.lut) { // (every byte is asked for before the first is used)
            uint32_t b[count][4];
#pragma unroll
            for (int u = 0; u < count; u++)
#pragma unroll
                for (int r = 0; r < 4; r++) b[u][r] = lutl[(packed[u] >> (8 * r)) & 0xffu];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < count; u++) packed[u] = b[u][0] | (b[u][1] << 8) | (b[u][2] << 16) | (b[u][3] << 24);
        }
#pragma unroll
        for (int u = 0; u < count; u++)
            *reinterpret_cast<uint32_t *>(tile + ((wm * RG + (first + u) / T) * 16 + j) * kOutPitch + ch0 + (first + u) % T * 4) = packed[u];
    };
    if constexpr (KG == 1) {
        finish(std::integral_constant<int, 0>());
    } else {
        static_for<0, (UNITS + EACH - 1) / EACH>([&](auto g_c) __attribute__((always_inline)) {
            if (kg == decltype(g_c)::value) finish(std::integral_constant<int, decltype(g_c)::value * EACH>());
        });
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < PASSES; it++) {
        if (px[it] >= late.m) continue;
        u32x4 v = *reinterpret_cast<const u32x4 *>(tile + (it * PPT + tid / PIECES) * kOutPitch + cb * ES);
        if constexpr (OUT == kTileFloats) {
            uint32_t *const yo = reinterpret_cast<uint32_t *>(late.y) + (size_t)px[it] * late.ldy + late.y_coff + ch;
            if (whole) {
                *reinterpret_cast<u32x4_a4 *>(yo) = u32x4_a4{v[0], v[1], v[2], v[3]};
            } else {
#pragma unroll
                for (int b = 0; b < 4; b++)
                    if (ch + b < late.n) yo[b] = v[b];
            }
            continue;
        }
        if (late.rep.res) {
#pragma unroll
            for (int d = 0; d < 4; d++) v[d] = residual4_packed(v[d], rv[it][d], late.rep);
        }
        uint8_t *yo = reinterpret_cast<uint8_t *>(late.y) + (size_t)px[it] * late.ldy + late.y_coff + ch;
        if (whole && wide_y) {
            *reinterpret_cast<u32x4_a4 *>(yo) = u32x4_a4{v[0], v[1], v[2], v[3]};
        } else if (whole) {
#pragma unroll
            for (int d = 0; d < 4; d++) reinterpret_cast<U32Unaligned *>(yo + d * 4)->v = v[d];
        } else {
#pragma unroll
            for (int b = 0; b < 16; b++)
                if (ch + b < late.n) yo[b] = (uint8_t)(v[b / 4] >> (8 * (b & 3)));
        }
    }
}

template <int T, int RG, int WM, int WN, int KG, TileOut OUT, bool RAGGED> int launch_tile_f(nncase_hip_ctx *ctx, const IgemmArgs &args, const TilePlan &plan, int nchunks) {
    if (plan.lds > 65536) NNHIP_HIP(ctx, (raise_dynamic_lds<qconv_tile_kernel<T, RG, WM, WN, KG, OUT, RAGGED>>(ctx->device, 160 * 1024)));
    hipLaunchKernelGGL((qconv_tile_kernel<T, RG, WM, WN, KG, OUT, RAGGED>), dim3(ceil_div(args.num_mtiles, 8) * 8 * nchunks), dim3(WM * WN * KG * 64), plan.lds, ctx->stream, args,
                       plan.t);
    NNHIP_LAUNCH_CHECK(ctx, "qconv_tile_kernel");
    return 0;
}
template <bool RAGGED, int T, int RG, int WM, int WN, int KG = 1> int launch_tile_t(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks) {
    IgemmArgs args = a;
    args.num_mtiles = plan.tiles;
    if (a.ep.out_mode != kOutU8) return launch_tile_f<T, RG, WM, WN, KG, kTileFloats, RAGGED>(ctx, args, plan, nchunks);
    return a.ep.fast && a.ep.full ? launch_tile_f<T, RG, WM, WN, KG, kTileFastCodes, RAGGED>(ctx, args, plan, nchunks)
                                  : launch_tile_f<T, RG, WM, WN, KG, kTileCodes, RAGGED>(ctx, args, plan, nchunks);
}

template <bool RAGGED> int launch_tile_shape(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks) {
    switch (plan.shape) {
    case kTile128x32: return launch_tile_t<RAGGED, 2, 4, 2, 1>(ctx, a, plan, nchunks);
    case kTile64x32: return launch_tile_t<RAGGED, 2, 2, 2, 1>(ctx, a, plan, nchunks);
    case kTile32x64: return launch_tile_t<RAGGED, 2, 2, 1, 2>(ctx, a, plan, nchunks);
    case kTile128x128: return launch_tile_t<RAGGED, 2, 4, 2, 4>(ctx, a, plan, nchunks);
    case kTile64x128: return launch_tile_t<RAGGED, 2, 2, 2, 4>(ctx, a, plan, nchunks);
    case kTile32x32by2: return launch_tile_t<RAGGED, 2, 2, 1, 1, 2>(ctx, a, plan, nchunks);
    case kTile32x32by4: return launch_tile_t<RAGGED, 2, 2, 1, 1, 4>(ctx, a, plan, nchunks);
    case kTile16x32by4: return launch_tile_t<RAGGED, 2, 1, 1, 1, 4>(ctx, a, plan, nchunks);
    case kTile32x64by2: return launch_tile_t<RAGGED, 2, 2, 1, 2, 2>(ctx, a, plan, nchunks);
    case kTile32x64by4: return launch_tile_t<RAGGED, 2, 2, 1, 2, 4>(ctx, a, plan, nchunks);
    case kTile16x64by4: return launch_tile_t<RAGGED, 2, 1, 1, 2, 4>(ctx, a, plan, nchunks);
    case kTileNone: break;
    }
    return fail(ctx, -EINVAL, "qconv2d: not a layer of the tile kernel");
}

} // namespace nnhip
