// Instantiations of the wide-tile implicit-GEMM kernels for channel counts that are no multiple of 16.
#include "qconv_wide.hpp"

namespace nnhip {
int launch_wide_ragged(nncase_hip_ctx *ctx, const IgemmArgs &a, bool rows, int tiles, int nchunks) {
    return rows ? launch_wide_lm<kWideRagRows>(ctx, a, tiles, nchunks) : launch_wide_lm<kWideRagWindow>(ctx, a, tiles, nchunks);
}
int launch_wide_small_ragged(nncase_hip_ctx *ctx, const IgemmArgs &a, bool rows, int shape, int nchunks) {
    return rows ? launch_wide_small_lm<kWideRagRows>(ctx, a, shape, nchunks) : launch_wide_small_lm<kWideRagWindow>(ctx, a, shape, nchunks);
}
} // namespace nnhip
