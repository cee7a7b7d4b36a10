// Host side of the implicit-GEMM convolution: weight pre-packing into MFMA
// operand order, the tiling plan, and the launch dispatch.
#include "qconv_rules.hpp"
#include "qconv_tile.hpp"

#include <algorithm>
#include <vector>

namespace nnhip {

static const int kAllowedTiles[] = {1, 2, 3, 4, 5, 6, 8, 9, 10, 12, 16};

static int round_tiles(int t) {
    for (int v : kAllowedTiles)
        if (v >= t) return v;
    return 16;
}

// Chooses the channel-chunk width T (in 16-channel tiles), the number of chunks and the
// LDS staging depth for a reduction of `ksteps` k-steps.  Wide chunks reuse every
// activation fragment for more output channels; narrow ones give more blocks.  With a
// pixel-count hint the widest chunk that still yields about two blocks per compute unit
// (at the smallest pixel tile) is taken; without one, the widest that fits the LDS budget.
static void plan_igemm(int g_oc, int ksteps, int64_t pixels_hint, int compute_units, int *tiles, int *nchunks,
                       int *kc_steps) {
    const int tt = ceil_div(g_oc, 16);
    const long long target = 2LL * compute_units;
    int best_t = 1, best_kc = std::min(ksteps, kLdsFrags);
    for (int nc = 1; nc <= tt; nc++) {
        if (ceil_div(tt, nc) > 16) continue; // more tiles than the widest kernel
        const int t = round_tiles(ceil_div(tt, nc));
        int kc;
        if (ksteps * t <= kLdsFrags) kc = ksteps;              // whole reduction resident
        else if (ksteps > 12 && t <= 4) kc = kLdsFrags / t;     // long reduction: staged in pieces
        else continue;
        best_t = t;
        best_kc = kc;
        if (pixels_hint <= 0 || t == 1) break;
        if ((long long)ceil_div((int)std::min<int64_t>(pixels_hint, 1 << 30), kWaves * 16) * ceil_div(tt, t) >= target) break;
    }
    *tiles = best_t;
    *nchunks = ceil_div(tt, best_t);
    *kc_steps = best_kc;
}

int igemm_plan(nncase_hip_ctx *ctx, nncase_hip_weights *w, const int32_t *bias) {
    const int taps = w->kernel_h * w->kernel_w;
    NNHIP_REQUIRE(ctx, (int64_t)taps * w->g_ic < 65536, -EINVAL,
                  "qconv2d_prepack: reduction length %lld would overflow the int32 accumulator",
                  (long long)taps * w->g_ic);
    w->tap_ic = w->g_ic;
    if (w->g_ic % 16 != 0 && ragged_pays(w->g_ic, taps, w->g_oc, w->pixels_hint)) w->ragged = true, w->tap_ic = ceil_div(w->g_ic, 16) * 16;
    w->k = taps * w->tap_ic;
    w->ksteps = ceil_div(w->k, 64);
    plan_igemm(w->g_oc, w->ksteps, w->pixels_hint, ctx->compute_units, &w->tiles, &w->nchunks, &w->kc_steps);
    // Long reductions over many pixels and more than 64 channels are bound by the matrix cores: they take the
    // wide-tile kernels (a wave owns 64 pixels x 64 or 128 channels) when the launch has a 256-pixel block for every
    // compute unit; smaller launches keep the small tiles, whose larger wave count fills the device better.  (Up to 64
    // channels the 128 x 64 blocks below are quicker at any size: 200 704 pixels 64 -> 64 3x3 20.6 us against 25.6.)
    {
        const long long ptiles = ceil_div((int)std::min<int64_t>(std::max<int64_t>(w->pixels_hint, 0), 1 << 30), 256);
        // 256-channel chunks (two waves side by side share the block's activations) where that still fills the device; rows
        // that the DMA kernel moves itself, from dword addresses (1x1 windows): by dma_pays
        const bool dma = taps == 1 && (!w->ragged || w->g_ic % 4 == 0);
        const bool fills = dma ? dma_pays(std::max<int64_t>(w->pixels_hint, 0), w->g_oc, w->ksteps, ctx->compute_units)
                               : !w->ragged && w->g_oc > 128 && ptiles * ceil_div(w->g_oc, 256) >= ctx->compute_units;
        const int wide_tiles = fills ? 16 : 8;
        w->wide = w->tap_ic % 16 == 0 && w->ksteps >= kWideMinKsteps && w->g_oc > 64 &&
                  (wide_tiles == 16 || ptiles * ceil_div(w->g_oc, 128) >= ctx->compute_units);
        if (w->wide) {
            w->tiles = wide_tiles;
            w->nchunks = ceil_div(w->g_oc, w->tiles * 16);
            w->kc_steps = std::min(w->ksteps, kLdsFrags / w->tiles);
        }
    }
    // Reductions of five k-steps and more over fewer pixels, and some shorter ones, take the same kernel with blocks of 8192 or
    // 2048 outputs: against the small tiles' per-lane loads of 16 pixels' slices, the row-order fetch through LDS needs a
    // quarter of the requests to the vector L1, which is what such launches are bound by.
    if (!w->wide && (w->ragged || (w->g_ic % 16 == 0 && small_wide_pays(w->g_oc, w->ksteps, w->tiles)))) {
        w->wide = 2;
        // (2048 outputs per block while the larger ones would leave more than half of the compute units without a block:
        // the 512 x 1024 x 1024 product takes 7.0 us with them, 9.2 us with 64 blocks of 8192)
        const long long blocks = (long long)ceil_div((int)std::min<int64_t>(std::max<int64_t>(w->pixels_hint, 1), 1 << 30), 128) * ceil_div(w->g_oc, 64);
        const bool small = w->g_oc <= 32 || (w->pixels_hint > 0 && 2 * blocks < ctx->compute_units);
        // A block that is wide in channels stages and re-biases half the activations per product (6400 pixels 256 -> 256 3x3:
        // 17.4 -> 16.1 us; 400 pixels: 14.5 -> 12.3 us), unless that rounds the channel count up by more than an eighth.
        auto rounded = [&](int chunk) { return ceil_div(w->g_oc, chunk) * chunk; };
        const int narrow = small ? 32 : 64;
        const bool flat = w->g_oc > narrow && 8 * rounded(2 * narrow) <= 9 * rounded(narrow);
        w->small_shape = small ? (flat ? kBlock32x64 : kBlock64x32) : (flat ? kBlock64x128 : kBlock128x64);
        w->tiles = (flat ? 2 * narrow : narrow) / 16;
        w->nchunks = ceil_div(w->g_oc, w->tiles * 16);
        w->kc_steps = std::min(w->ksteps, kLdsFrags / w->tiles);
    }
    // -(zw - 128) has to be an s8 value
    w->fold = !w->ragged && w->ksteps == 1 && w->k <= 32 && w->zw >= 1;
    w->packed_bytes = (size_t)w->nchunks * w->ksteps * w->tiles * 1024 * w->groups;
    w->bias_absmax = 0;
    if (bias)
        for (int i = 0; i < w->out_channels; i++) w->bias_absmax = std::max<long long>(w->bias_absmax, std::llabs((long long)bias[i]));
    return 0;
}

size_t igemm_const_bytes(const nncase_hip_weights *w) { return w->packed_bytes + 2 * sizeof(int32_t) * (size_t)w->out_channels; }

void igemm_place(nncase_hip_weights *w, void *block) {
    w->d_packed = block;
    w->d_wsum = reinterpret_cast<int32_t *>(reinterpret_cast<uint8_t *>(block) + w->packed_bytes);
    w->d_bias = w->d_wsum + w->out_channels;
}

// What pack_group does, on the device: a block packs one 16-channel tile of a chunk, its waves taking the k-steps in turn
// (lane = 16-byte piece of the fragment), and adds up the tile's sums on the way.  Bound by the byte gather (a piece of a
// windowed layer reads 16 bytes `taps` apart); 110 KB of 3x3 weights take 4 us where the host loops took 250.
struct PackArgs {
    RawWeights raw;
    uint8_t *dst;
    int32_t *wsum;
    size_t group_bytes; // of the packed result
    int g_oc, g_ic, tap_ic, k, ksteps, tiles;
    int zw, fold_value; // fold_value: 0 = no fold
};
constexpr int kPackWaves = 8;
__global__ __launch_bounds__(kPackWaves * 64) void igemm_pack_kernel(const PackArgs a) {
    __shared__ int32_t sums[kPackWaves][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = lane & 15, kg = lane >> 4;
    const int chunk = blockIdx.x / a.tiles, nt = blockIdx.x - chunk * a.tiles, g = blockIdx.y;
    const int oc = chunk * 16 * a.tiles + (i / 4) * 4 * a.tiles + nt * 4 + (i % 4);
    const uint8_t *const src = a.raw.ptr + g * a.raw.group_bytes + oc * a.raw.oc_stride;
    int32_t sum = 0;
    for (int ks = wave; ks < a.ksteps; ks += kPackWaves) {
        const int kk0 = ks * 64 + kg * 16;
        int tap = kk0 / a.tap_ic, ic = kk0 - tap * a.tap_ic;
        uint32_t v[16];
#pragma unroll
        for (int b = 0; b < 16; b++) { // every load is requested before the first is used
            const bool real = oc < a.g_oc && kk0 + b < a.k;
            v[b] = a.zw;
            if (real && ic < a.g_ic) v[b] = src[ic * a.raw.ic_stride + tap];
            v[b] = real ? v[b] : 0x80u;
            if (++ic == a.tap_ic) ic = 0, tap++;
        }
        u32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < 16; b++) {
            const uint32_t x = v[b] ^ 0x80u;
            sum += (int32_t)(int8_t)x;
            const bool folded = a.fold_value != 0 && kk0 + b >= 32 && kk0 + b - 32 < a.k;
            d[b / 4] |= (folded ? (uint32_t)a.fold_value & 0xffu : x) << (8 * (b & 3));
        }
        *reinterpret_cast<u32x4 *>(a.dst + g * a.group_bytes + (((size_t)chunk * a.ksteps + ks) * a.tiles + nt) * 1024 + lane * 16) = d;
    }
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (kg == 0) sums[wave][i] = sum;
    __syncthreads();
    if (threadIdx.x < 16 && oc < a.g_oc) {
        int32_t s = 0;
        for (int w = 0; w < kPackWaves; w++) s += sums[w][i];
        a.wsum[g * a.g_oc + oc] = s;
    }
}

int igemm_pack(nncase_hip_ctx *ctx, nncase_hip_weights *w, const RawWeights &raw) {
    PackArgs a;
    a.raw = raw;
    a.dst = reinterpret_cast<uint8_t *>(w->d_packed), a.wsum = w->d_wsum;
    a.group_bytes = w->packed_bytes / w->groups;
    a.g_oc = w->g_oc, a.g_ic = w->g_ic, a.tap_ic = w->tap_ic, a.k = w->k, a.ksteps = w->ksteps, a.tiles = w->tiles;
    a.zw = w->zw, a.fold_value = w->fold ? 128 - w->zw : 0;
    if (w->fold && a.fold_value == 0) a.fold_value = 256; // (the low byte is what is stored)
    hipLaunchKernelGGL(igemm_pack_kernel, dim3(w->nchunks * w->tiles, w->groups), dim3(kPackWaves * 64), 0, ctx->stream, a);
    NNHIP_LAUNCH_CHECK(ctx, "igemm_pack_kernel");
    return 0;
}

int igemm_pixel_groups(const nncase_hip_ctx *ctx, const nncase_hip_weights *w, int m) {
    return choose_rg(ctx, w->tiles, w->nchunks, m);
}

static bool igemm_is_pointwise(const nncase_hip_weights *w, const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    return w->kernel_h == 1 && w->kernel_w == 1 && c->stride_h == 1 && c->stride_w == 1 && c->pad_h_before == 0 && c->pad_w_before == 0 &&
           out_h == c->in_h && out_w == c->in_w;
}

// Strided 1x1 windows packed for the DMA kernel: it moves whole pixels, wherever they lie (the plan, which does not know the stride, has
// counted on its blocks' heights).  us, with 8 tiles / by the window's taps in blocks of 256 x 256 / so: 16 000 pixels 640 -> 512 14.9 / 19.2 /
// 12.5, 2048 of 4096 -> 4096 55.8 / 63.5 / 41.0, 15 488 of 2240 -> 364 28.7 / 41.9 / 25.0, 12 288 of 1536 -> 1024 - / 32.9 / 26.2.
static bool igemm_rows_apart(const nncase_hip_weights *w, const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    return w->wide == 1 && w->tiles == 16 && w->kernel_h == 1 && w->kernel_w == 1 && !igemm_is_pointwise(w, c, out_h, out_w) && c->pad_h_before == 0 &&
           c->pad_w_before == 0 && (int64_t)(out_h - 1) * c->stride_h < c->in_h && (int64_t)(out_w - 1) * c->stride_w < c->in_w;
}

int igemm_load_mode(const nncase_hip_weights *w, const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    const bool pointwise = igemm_is_pointwise(w, c, out_h, out_w) || igemm_rows_apart(w, c, out_h, out_w);
    if (w->g_ic % 16 == 0) return pointwise ? kRows16 : kVec16;
    if (w->g_ic % 8 != 0) return kVec4;
    // (the row loader reads 16 bytes at a time: the tensor has to hold that many)
    return pointwise && (int64_t)c->batch * c->in_h * c->in_w * w->in_channels >= 16 ? kRows8 : kVec8; // (anything else is ragged)
}

int launch_qconv_igemm(nncase_hip_ctx *ctx, const uint8_t *x, const nncase_hip_weights *w, void *y,
                       const nncase_hip_conv2d_args_t *c, int out_h, int out_w) {
    const int64_t m64 = (int64_t)c->batch * out_h * out_w;
    const int64_t in_bytes = (int64_t)c->batch * c->in_h * c->in_w * w->in_channels;
    const int out_es = c->out_dtype == NNCASE_HIP_DT_U8 && !c->dequantize_output ? 1 : 4;
    NNHIP_REQUIRE(ctx, m64 > 0 && m64 < ((int64_t)1 << 30), -EINVAL, "qconv2d: %lld output pixels unsupported",
                  (long long)m64);
    NNHIP_REQUIRE(ctx, in_bytes < ((int64_t)1 << 31), -EINVAL, "qconv2d: input of %lld bytes exceeds 2 GiB",
                  (long long)in_bytes);
    NNHIP_REQUIRE(ctx, m64 * w->out_channels * out_es < ((int64_t)1 << 40), -EINVAL, "qconv2d: output too large");
    NNHIP_REQUIRE(ctx, (reinterpret_cast<uintptr_t>(x) & 15u) == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0,
                  -NNCASE_HIP_ERR_INVALID_MEMORY_LOCATION, "qconv2d: activation buffers must be 16-byte aligned");

    IgemmArgs a;
    memset(&a, 0, sizeof(a));
    a.x = x;
    a.y = y;
    a.m = (int)m64;
    a.n = w->g_oc;
    a.k = w->k;
    a.ksteps = w->ksteps;
    a.kc_steps = w->kc_steps;
    a.ldx = w->in_channels;
    a.x_bytes = (size_t)c->batch * c->in_h * c->in_w * w->in_channels;
    a.ldy = c->out_channel_stride ? c->out_channel_stride : w->out_channels;
    a.ldr = w->out_channels;
    NNHIP_REQUIRE(ctx, c->out_channel_stride >= 0 && c->out_channel_offset >= 0 &&
                           (c->out_channel_stride ? c->out_channel_offset + w->out_channels <= c->out_channel_stride : c->out_channel_offset == 0),
                  -EINVAL, "qconv2d: %d output channels at offset %d do not fit a pixel stride of %d", w->out_channels, c->out_channel_offset,
                  c->out_channel_stride);
    NNHIP_REQUIRE(ctx, m64 * a.ldy * out_es < ((int64_t)1 << 40), -EINVAL, "qconv2d: output too large");
    a.g_ic = w->tap_ic;
    a.in_h = c->in_h;
    a.in_w = c->in_w;
    a.kh = w->kernel_h;
    a.kw = w->kernel_w;
    a.stride_h = c->stride_h;
    a.stride_w = c->stride_w;
    a.dil_h = c->dilation_h;
    a.dil_w = c->dilation_w;
    a.pad_h = c->pad_h_before;
    a.pad_w = c->pad_w_before;
    a.d_ohow = make_fastdiv((uint32_t)(out_h * out_w));
    a.d_ow = make_fastdiv((uint32_t)out_w);
    a.d_kw = make_fastdiv((uint32_t)w->kernel_w);
    a.d_gic = make_fastdiv((uint32_t)w->tap_ic);
    a.zxp = c->x_qp.zero_point - 128;
    a.zwp = w->zw - 128;
    a.zwp_rows = w->fold ? 0 : a.zwp;
    a.kc_mask = w->fold ? 1 : -1;
    a.zx_splat = (uint32_t)(c->x_qp.zero_point & 0xff) * 0x01010101u;
    {
        const int rc = make_epilogue(ctx, &a.ep, c->x_qp.scale, w->sw, c->y_qp, c->clamp_min, c->clamp_max, c->out_dtype, "qconv2d");
        if (rc) return rc;
    }

    {
        const int rc = make_residual_epilogue(ctx, &a.rep, c, w);
        if (rc) return rc;
    }
    // every accumulator, the zero-point terms included, is at most |bias| + 4 K 128^2 in magnitude
    a.magic_ok = a.ep.magic && a.ep.full && w->bias_absmax + 4ll * w->k * 16384 <= a.ep.magic_limit;
    a.lut = c->out_dtype == NNCASE_HIP_DT_U8 ? w->d_post_lut : nullptr;
    if (c->dequantize_output != 0) { // (out_dtype is u8 here: the entry point has turned the call into its u8 form)
        const nncase_hip_quant_param_t last = c->residual_dev ? c->sum_qp : (w->d_post_lut ? w->post_lut_qp : c->y_qp);
        a.deq = 1, a.deq_zero = last.zero_point, a.deq_scale = last.scale;
    }
    const int mode = igemm_load_mode(w, c, out_h, out_w);
    a.apart = igemm_rows_apart(w, c, out_h, out_w);

    const TilePlan tile = plan_qconv_tile(ctx, a, w->ragged, w->tiles, w->nchunks);
    const size_t group_bytes = (size_t)w->nchunks * w->ksteps * w->tiles * 1024;
    for (int g = 0; g < w->groups; g++) {
        a.wpk = reinterpret_cast<const uint8_t *>(w->d_packed) + g * group_bytes;
        a.wsum = w->d_wsum + (size_t)g * w->g_oc;
        a.bias = w->d_bias + (size_t)g * w->g_oc;
        a.x_coff = g * w->g_ic;
        a.y_coff = g * w->g_oc + c->out_channel_offset;
        a.r_coff = g * w->g_oc;
        int rc;
        if (tile.shape != kTileNone) {
            rc = launch_qconv_tile(ctx, a, tile, w->nchunks);
            if (rc) return rc;
            continue;
        }
        if (w->ragged) {
            const bool rows = a.apart || igemm_is_pointwise(w, c, out_h, out_w);
            rc = w->wide == 2 ? launch_wide_small_ragged(ctx, a, rows, w->small_shape, w->nchunks) : launch_wide_ragged(ctx, a, rows, w->tiles, w->nchunks);
            if (rc) return rc;
            continue;
        }
        if (w->wide == 2) {
            rc = mode == kRows16 ? launch_wide_small_rows16(ctx, a, w->small_shape, w->nchunks) : launch_wide_small_vec16(ctx, a, w->small_shape, w->nchunks);
            if (rc) return rc;
            continue;
        }
        if (w->wide) {
            rc = mode == kRows16 ? launch_wide_rows16(ctx, a, w->tiles, w->nchunks) : launch_wide_vec16(ctx, a, w->tiles, w->nchunks);
            if (rc) return rc;
            continue;
        }
        const int rg = choose_rg(ctx, w->tiles, w->nchunks, a.m);
        switch (mode) {
        case kRows16: rc = launch_igemm_rows16(ctx, a, w->tiles, w->nchunks, rg); break;
        case kVec16: rc = launch_igemm_vec16(ctx, a, w->tiles, w->nchunks, rg); break;
        case kVec4: rc = launch_igemm_vec4(ctx, a, w->tiles, w->nchunks, rg); break;
        case kVec8: rc = launch_igemm_vec8(ctx, a, w->tiles, w->nchunks, rg); break;
        default: rc = launch_igemm_rows8(ctx, a, w->tiles, w->nchunks, rg); break;
        }
        if (rc) return rc;
    }
    return 0;
}

} // namespace nnhip
