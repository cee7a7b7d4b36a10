// How the paged attention splits a context over blocks: plain host arithmetic, so that a test can hold the choice against the
// measured times without a device.
#pragma once

#include <cstdint>

namespace nnhip {

struct AttnBlock {
    int tiles, waves; // a block owns tiles * waves * 16 tokens
};

// Tokens per block, as waves of 16-token tiles, from the capacity (the kernel cannot know the real lengths on the host) and the
// launch's pairs of sequence and kv head.  Four waves of four tiles where they serve: a block of eight holds twice the registers
// or, at head_dim 128, half the compute unit's LDS, and its phases (requests, products, merge) then have one other block to
// overlap with.  us as 2 x 4 / 4 x 4 / 2 x 8 / 4 x 8 (tiles x waves):
//   * up to 128 tokens one block of 2 x 4, no merge (8 pairs of 64, 112 tokens 4.2 / 4.4 / 4.3 / 4.6), up to 256 one of 2 x 8 (8
//     pairs of 128, 208 tokens 7.7 / 7.4 / 7.0 / 7.7) unless there is more than one per compute unit; up to 1024, eight blocks,
//     which are merged in one memory round trip, 2 x 4 (8 pairs of 128, 512 tokens 7.9 / 9.6 / 9.1 / 10.5)
//   * head_dim 128 past that: 2 x 8 while that is at most three blocks per compute unit (8 pairs, 4096 tokens 14.1 / 12.4 / 11.0 /
//     13.0), 4 x 8 for a few very long contexts (8 pairs of 16 000 41.0 / 26.8 / 22.4 / 20.1)
//   * head_dim 64: 4 x 8 where its blocks, two of which a compute unit holds, make one round of the device and a little (64 pairs
//     of 4064 tokens 16.4 / 13.8 / 14.8 / 12.9), and for long contexts up to three of them per compute unit (16 pairs of 16 000
//     41.1 / 26.1 / 24.7 / 19.0)
// (Of 908 launches the choice is 1.3 % behind the best of these in the mean.)
inline AttnBlock choose_attn_block(int head_dim, int64_t pairs, int64_t max_tokens, int compute_units) {
    auto blocks = [&](int64_t tokens) { return pairs * ((max_tokens + tokens - 1) / tokens); };
    if (max_tokens <= 128) return {2, 4};
    if (max_tokens <= 256) return pairs <= compute_units ? AttnBlock{2, 8} : AttnBlock{4, 4};
    if (max_tokens <= 1024) return {2, 4};
    if (head_dim == 128) {
        if (max_tokens >= 10000 && pairs <= 8) return {4, 8};
        return blocks(256) <= 3ll * compute_units ? AttnBlock{2, 8} : AttnBlock{4, 4};
    }
    const int64_t per_ten_units = 10 * blocks(512) / compute_units;
    if (max_tokens >= 3200 && per_ten_units >= 17 && per_ten_units <= 23) return {4, 8};
    if (max_tokens >= 6500 && 4 * blocks(512) >= compute_units && blocks(512) <= 3ll * compute_units) return {4, 8};
    return {4, 4};
}

} // namespace nnhip
