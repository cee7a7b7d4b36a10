// Which launches the window kernel of qconv_tile.hpp takes, with which block, and the launches for channels that are multiples of 16.
#include "qconv_tile.hpp"

namespace nnhip {

namespace {
// The plan of a kernel with `pix` pixels and `tb` 16-channel tiles per block; `groups` of waves, whose sums take `parts` bytes, share its k-steps.
TilePlan plan_tile(const IgemmArgs &a, int pix, int tb, int threads, int nchunks, int groups, int parts) {
    const int ow = (int)a.d_ow.div, oh = (int)a.d_ohow.div / ow, batch = a.m / (int)a.d_ohow.div;
    const OutputTile o = choose_output_tile(oh, ow, pix, a.stride_h, a.stride_w, (a.kh - 1) * a.dil_h + 1, (a.kw - 1) * a.dil_w + 1);
    TilePlan p;
    p.tiles = batch * o.across * o.down;
    TileArgs &t = p.t;
    t.th = o.th, t.tw = o.tw, t.hr = o.in_rows, t.hc = o.in_cols;
    t.half = ceil_div(t.hc, a.stride_w);
    t.pieces = a.g_ic / 16;
    t.pitch = (t.pieces | 1) * 16;
    t.row_pitch = a.stride_w * t.half * t.pitch;
    t.row_bytes = a.in_w * a.ldx;
    t.d_pieces = make_tile_div(t.pieces), t.d_hc = make_tile_div(t.hc), t.d_tw = make_tile_div(t.tw);
    t.d_tx = make_fastdiv((uint32_t)o.across), t.d_txy = make_fastdiv((uint32_t)(o.across * o.down));
    t.d_nchunks = make_fastdiv((uint32_t)nchunks), t.d_rest = make_fastdiv((uint32_t)std::max(1, a.ksteps - 1));
    t.tile_off = (tb * 16 + groups * pix + (a.ksteps + 2 * groups) * 4) * 4 + 256 + parts;
    t.apart = threads / t.pieces, t.dc = t.apart % t.hc, t.dr = t.apart / t.hc;
    p.lds = t.tile_off + std::max((size_t)t.hr * t.row_pitch, (size_t)pix * (tb * 16 * (a.ep.out_mode == kOutU8 ? 1 : 4) + 16));
    return p;
}

template <int T, int RG, int WM, int WN, int KG = 1> TilePlan plan_shape(const IgemmArgs &a, int nchunks) {
    return plan_tile(a, WM * RG * 16, T * WN, WM * WN * KG * 64, nchunks, KG, tile_part_bytes(RG * T, WM * WN, KG));
}

// A launch of few blocks: the smallest tile first, four groups before two.
template <int T, int RG, int WM, int WN, int KG> bool split_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, int nchunks, TilePlan *plan) {
    if (a.ksteps <= KG || (long long)ceil_div(a.m, WM * RG * 16) * nchunks * WM * WN * KG > split_window_waves(ctx->compute_units)) return false;
    *plan = plan_shape<T, RG, WM, WN, KG>(a, nchunks);
    return plan->t.apart > 0 && split_window_pays(TileLaunch{a.stride_w, a.ksteps, a.g_ic, WM * RG * 16, WM * WN * KG, plan->lds, plan->tiles, nchunks, a.m}, ctx->compute_units);
}
TileShape choose_split_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, int tiles, int nchunks, TilePlan *plan) {
    if (tiles == 4) {
        if (a.ksteps < 7) return kTileNone; // (five or six: 32 -> 100 3x3 of 400 pixels 3.9 by the k-steps' ring, 4.1 so)
        if (split_tile<2, 1, 1, 2, 4>(ctx, a, nchunks, plan)) return kTile16x64by4;
        if (split_tile<2, 2, 1, 2, 4>(ctx, a, nchunks, plan)) return kTile32x64by4;
        if (split_tile<2, 2, 1, 2, 2>(ctx, a, nchunks, plan)) return kTile32x64by2;
    } else if (tiles == 2) {
        if (a.ksteps < 5) return kTileNone;
        if (split_tile<2, 1, 1, 1, 4>(ctx, a, nchunks, plan)) return kTile16x32by4;
        if (split_tile<2, 2, 1, 1, 4>(ctx, a, nchunks, plan)) return kTile32x32by4;
        if (split_tile<2, 2, 1, 1, 2>(ctx, a, nchunks, plan)) return kTile32x32by2;
    }
    return kTileNone;
}

// Which block, if any, by the packed chunk (`tiles` of 16 channels) and the waves the launch has (byte results, windows,
// strides of 1 and 2).  Measured us, implicit GEMM / here, byte table behind the convolution:
//   * eight waves share the staging of a 128-channel chunk: 25 600 pixels 128 -> 128 3x3 11.7 / 9.7 with 128 pixels per block
//     (10.4 with 64), 6400 pixels 256 -> 256 11.8 / 9.2 with 64 (11.4 with 128: fewer blocks than compute units); three blocks of
//     128 pixels for four compute units are enough (asked for twice as many, 750 windows lose 7 % where it makes a difference);
//   * one wave row of 32 pixels for 64 channels: 102 400 pixels 64 -> 64 12.7 / 11.5 (13.9 with 128 pixels, 12.3 with 64);
//   * 32 channels: 409 600 pixels 32 -> 32 21.9 / 15.6, 1 638 400 pixels 16 -> 32 41.4 / 36.7; two k-steps and fewer are the
//     epilogue's work alone and stay (802 816 pixels 16 -> 32 2x2 14.9 / 18.6);
//   * the k-steps it takes: whole_window_ksteps;
//   * and what tile_kernel_pays asks of the launch.
TileShape choose_whole_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, bool ragged, int tiles, int nchunks, TilePlan *plan) {
    if (a.ksteps < whole_window_ksteps(a.stride_w, tiles, ragged)) return kTileNone;
    TileShape shape = kTileNone;
    int waves = 2, pix = 64;
    // (the smaller tile too where the larger one is not half full of an image's pixels)
    auto enough = [&](int blocks) { return (long long)plan->tiles * nchunks >= blocks && 2ll * a.m >= (long long)plan->tiles * 128; };
    switch (tiles) {
    case 2:
        *plan = plan_shape<2, 4, 2, 1>(a, nchunks), shape = kTile128x32, pix = 128;
        if (!enough(3 * ctx->compute_units)) *plan = plan_shape<2, 2, 2, 1>(a, nchunks), shape = kTile64x32, pix = 64;
        break;
    case 4: *plan = plan_shape<2, 2, 1, 2>(a, nchunks), shape = kTile32x64, pix = 32; break;
    case 8:
        *plan = plan_shape<2, 4, 2, 4>(a, nchunks), shape = kTile128x128, waves = 8, pix = 128;
        if (!enough(3 * ctx->compute_units / 4)) *plan = plan_shape<2, 2, 2, 4>(a, nchunks), shape = kTile64x128, pix = 64;
        // (a sixth of surplus pixels: 334 -> 360 3x3 of 47 images of 14 x 14 24.6 by the ring, 27.0 so)
        if (ragged && 20ll * a.m < 17ll * plan->tiles * pix) return kTileNone;
        break;
    default: return kTileNone;
    }
    return plan->t.apart > 0 && tile_kernel_pays(TileLaunch{a.stride_w, a.ksteps, a.g_ic, pix, waves, plan->lds, plan->tiles, nchunks, a.m}, ctx->compute_units) ? shape : kTileNone;
}
TileShape choose_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, bool ragged, int tiles, int nchunks, TilePlan *plan) {
    if (a.kh * a.kw == 1 || a.g_ic % 16 != 0 || a.x_bytes < 16 || a.kc_mask != -1 || a.stride_w > 2 || (int64_t)a.in_w * a.ldx >= (1 << 23)) return kTileNone;
    // Fewer than ten k-steps are split where one group is no choice (three waves for two compute units and more: 64 -> 64 of 6400 pixels
    // 4.2 / 4.0, 48 -> 32 of 25 600 4.5 / 4.2, 32 -> 48 of 12 800 4.1 / 4.2).
    if (a.ksteps >= 10) {
        const TileShape split = choose_split_tile(ctx, a, tiles, nchunks, plan);
        if (split != kTileNone) return split;
    }
    const TileShape whole = choose_whole_tile(ctx, a, ragged, tiles, nchunks, plan);
    return whole != kTileNone || a.ksteps >= 10 ? whole : choose_split_tile(ctx, a, tiles, nchunks, plan);
}
} // namespace

const char *tile_kernel_block(const nncase_hip_ctx *ctx, const nncase_hip_weights *w, const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    static const char *const names[] = {"128x32", "64x32", "32x64", "128x128", "64x128", "32x32,KG=2", "32x32,KG=4", "16x32,KG=4", "32x64,KG=2",
                                        "32x64,KG=4", "16x64,KG=4", nullptr};
    if (c->dequantize_output || c->out_dtype == NNCASE_HIP_DT_I32) return nullptr;
    IgemmArgs a;
    memset(&a, 0, sizeof(a));
    a.ep.out_mode = c->out_dtype == NNCASE_HIP_DT_U8 ? kOutU8 : kOutF32;
    a.m = (int)std::min<int64_t>((int64_t)c->batch * out_h * out_w, 1 << 30);
    a.d_ohow = make_fastdiv((uint32_t)(out_h * out_w)), a.d_ow = make_fastdiv((uint32_t)out_w);
    a.kh = w->kernel_h, a.kw = w->kernel_w, a.stride_h = c->stride_h, a.stride_w = c->stride_w, a.dil_h = c->dilation_h, a.dil_w = c->dilation_w;
    a.g_ic = w->tap_ic, a.in_w = c->in_w, a.ldx = w->in_channels, a.x_bytes = (size_t)c->batch * c->in_h * c->in_w * w->in_channels, a.ksteps = w->ksteps, a.kc_mask = w->fold ? 1 : -1;
    TilePlan plan;
    return names[choose_tile(ctx, a, w->ragged, w->tiles, w->nchunks, &plan)];
}

TilePlan plan_qconv_tile(const nncase_hip_ctx *ctx, const IgemmArgs &a, bool ragged, int tiles, int nchunks) {
    TilePlan plan;
    const TileShape shape = !a.deq && a.ep.out_mode != kOutI32 ? choose_tile(ctx, a, ragged, tiles, nchunks, &plan) : kTileNone;
    plan.shape = shape;
    plan.t.ragged = ragged;
    return plan;
}

int launch_qconv_tile(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks) {
    return plan.t.ragged ? launch_tile_ragged(ctx, a, plan, nchunks) : launch_tile_shape<false>(ctx, a, plan, nchunks);
}

} // namespace nnhip
