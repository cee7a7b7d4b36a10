// How the paged attention splits a context over blocks: plain host arithmetic, so that a test can hold the choice against the
// measured times without a device.
#pragma once

#include <algorithm>
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

// Tokens per split of the kernel that goes through a split 128 tokens at a time, or 0 where the one above is taken (us, that one's
// best block / in steps):
//   * 64-wide heads, 257 to 512 tokens, from 24 pairs: one split, no merge (24 pairs of 265 tokens 5.8 / 5.3, 60 of 459 6.6 / 6.2, 240
//     of 384 7.8 / 5.9; 12 of 433 6.2 / 6.4).  Longer contexts come out even with that (12 pairs of 13 658 13.9 / 12.7, 84 of 4759
//     16.4 / 17.9, 132 of 14 756 50.7 / 52.1)
//   * 128-wide heads from 50 MB of keys and values on (48 pairs of 1851 15.2 / 13.8, 36 of 6028 22.3 / 17.9, 104 of 9746 107 / 80, 656 of
//     4073 267 / 229; below, 64 of 1205 12.1 / 13.0 and 8 of 4387 12.3 / 14.0), which few pairs reach with long contexts only, and too
//     many splits (8 of 12 668 18.4 / 20.0).
// There one split up to 384 tokens, else as many as make one round of the device, a block per compute unit: fewer leave units idle, a
// second round costs as much as the first (with runs of 256 / 512 / 1024 / 2048: 32 of 3425 12.6 11.3 15.3 23.9, 80 of 2220 19.0 18.8
// 16.8 25.2).  Where splits of 2048 tokens would still be more than that: 512 tokens, which even the rounds out (152 of 10 998 82.7
// 77.6 82.4 91.1), or 1024 where that is the whole context or with nine rounds and more (1600 of 1500 136 126 117 119).
inline int choose_attn_run(int head_dim, int64_t pairs, int64_t max_tokens, int compute_units) {
    auto even = [&](int64_t splits) { return (int)(((max_tokens + splits - 1) / splits + 127) / 128 * 128); };
    if (head_dim == 64) return max_tokens > 256 && max_tokens <= 512 && pairs >= 24 ? even(1) : 0;
    if (pairs < 16 || pairs * max_tokens < 98304) return 0;
    if (max_tokens <= 384) return even(1);
    const int64_t one_round = compute_units / pairs;
    if (one_round >= 1 && even(one_round) <= 2048) return std::max(even(one_round), 256);
    if (max_tokens <= 1024) return 1024;
    return pairs * ((max_tokens + 1023) / 1024) >= 9ll * compute_units ? 1024 : 512;
}

} // namespace nnhip
