// Packed weights brought into the L2 caches ahead of the products that read them: which 1 KiB fragments the blocks of an XCD
// will ask for.  Plain arithmetic for host and device, so that a test can hold it to every fragment once and to its bounds
// without a device.
#pragma once

#include <cstddef>
#include <cstdint>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define NNHIP_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define NNHIP_HOST_DEVICE inline
#endif

namespace nnhip {

constexpr int kXcds = 8;             // dies with an L2 of their own; block i of a launch runs on die i % 8
constexpr size_t kMaxFetchBytes = 20u << 20; // of the 32 MiB the dies' caches hold, beside the cached keys and values under way
constexpr int kMaxWeightFetches = 4; // products behind one attention operator: output, gate / up, down, the next q / k / v

// A product whose block b reads the tiles (b / off) * 2 off + b % off and, with two tiles a block, the one `off` further
// (one tile a block: off = tiles, which makes that b).
struct WeightFetch {
    const void *packed; // [tiles][steps] fragments of 1 KiB
    uint32_t blocks, steps, off, per_block; // per_block: 1 or 2 tiles
};

// fragments that the blocks of die x read
NNHIP_HOST_DEVICE uint32_t fetch_fragments(const WeightFetch &f, uint32_t x) {
    return (f.blocks + kXcds - 1 - x) / kXcds * (f.per_block * f.steps);
}
// position of die x's u-th fragment (u < fetch_fragments), in fragments
NNHIP_HOST_DEVICE uint32_t fetch_position(const WeightFetch &f, uint32_t x, uint32_t u) {
    const uint32_t per = f.per_block * f.steps, turn = u / per, rest = u - turn * per;
    const uint32_t b = x + kXcds * turn, second = rest >= f.steps;
    const uint32_t tile = b / f.off * (2 * f.off) + b % f.off + second * f.off;
    return tile * f.steps + (rest - second * f.steps);
}

// What an attention launch fetches beside its own work.
struct WeightFetches {
    WeightFetch f[kMaxWeightFetches];
    int count;
    int blocks; // that fetch, on each die
};

// die x's u-th fragment of all the products, one behind the other (u < the sum of fetch_fragments)
NNHIP_HOST_DEVICE const char *fetch_address(const WeightFetches &s, uint32_t x, uint32_t u) {
    for (int i = 0;; i++) {
        const uint32_t n = fetch_fragments(s.f[i], x);
        if (u < n) return (const char *)s.f[i].packed + (size_t)fetch_position(s.f[i], x, u) * 1024;
        u -= n;
    }
}

// Whether an attention brings weights into the caches for the products behind it where its function has lanes that run side by side:
// another lane's products are then using the memory that the attention leaves idle, and two lanes' weights and rows do not fit the
// caches together.  Beyond eight rows a lane it costs more than it gives, and where a lane's keys and values are some 30 MB (a decode step of 24 layers as two lanes, us a step without / with: rows a lane x context 4 x 700 753 / 731, 8 x 700
// 793 / 790, 8 x 4096 901 / 890, 8 x 8192 963 / 998, 12 x 1500 880 / 901, 16 x 700 869 / 885, 16 x 2048 909 / 953, 16 x 4096 1037 / 1069,
// 32 x 2048 1138 / 1180; as four lanes 8 x 700 1668 / 1643, 16 x 2048 1962 / 1992).  With one lane 1 x 700 655 / 602, 16 x 2048 817 /
// 814, 32 x 700 895 / 886, 32 x 4096 1057 / 1068.
inline bool fetch_beside_lanes(int lanes, int rows, int64_t kv_bytes) { return lanes <= 1 || (rows <= 8 && kv_bytes <= 25000000); }

} // namespace nnhip
