// The window kernel of qconv_tile.hpp for channels that are no multiple of 16.
#include "qconv_tile.hpp"

namespace nnhip {

int launch_tile_ragged(nncase_hip_ctx *ctx, const IgemmArgs &a, const TilePlan &plan, int nchunks) {
    return launch_tile_shape<true>(ctx, a, plan, nchunks);
}

} // namespace nnhip
