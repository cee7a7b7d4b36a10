// How the paged attention splits a context over blocks: plain arithmetic, so that a test can hold the choice against the measured
// times without a device.
#pragma once

#include "weight_fetch.hpp"

#include <algorithm>
#include <cstdint>

namespace nnhip {

constexpr int kAttnMaxSplits = 1024; // splits of one sequence (bounds the merge loop and the workspace)

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

// Division by a small number as a multiplication: exact up to 2^21 + 1024 (the longest context that is gone through in steps) for
// divisors up to 1024, at most one more above that.
struct AttnDivisor {
    uint32_t divisor, mul;
};
inline AttnDivisor attn_divisor(int64_t d) { return {(uint32_t)d, (uint32_t)(((int64_t(1) << 32) + d - 1) / d)}; }
NNHIP_HOST_DEVICE uint32_t attn_divide(uint32_t n, const AttnDivisor &d) { return d.divisor == 1 ? n : (uint32_t)((uint64_t)n * d.mul >> 32); }

// What does not change with the lengths.
struct AttnRunRule {
    uint32_t batch, nine_rounds; // nine_rounds: splits of each pair that are nine rounds of the device and more
    bool has_round;              // a round holds a split of each pair
    AttnDivisor round, two_rounds, most; // splits of each pair that make one round, splits of one head of all sequences that make two,
                                         // splits of a pair that there is room for
};
inline AttnRunRule attn_run_rule(int64_t batch, int64_t kv_heads, int compute_units, int64_t most) {
    const int64_t pairs = batch * kv_heads, round = compute_units / pairs;
    return {(uint32_t)batch, (uint32_t)((9ll * compute_units + pairs - 1) / pairs), round > 0, attn_divisor(std::max<int64_t>(round, 1)),
            attn_divisor(std::max<int64_t>(2 * compute_units / kv_heads, 1)), attn_divisor(most)};
}

// Tokens per split of the kernel that goes through a split 128 tokens at a time, for sequences of `total` tokens the longest of which
// has `longest`: one split up to 512 tokens, without a merge (24 sequences of one head of up to 439 tokens 8.9 us, 10.9 as two; 13 of 4 of
// 468 8.4 / 9.2), else as many as make one round of the device, a block per compute unit: fewer leave units idle, a second round
// costs as much as the first (us with runs of 256 / 512 / 1024 / 2048: 32 pairs of 3425 tokens 12.6 11.3 15.3 23.9, 80 of 2220 19.0
// 18.8 16.8 25.2).  Where splits of 2048 tokens would still be more than that: 512 tokens, which even the rounds
// out (152 of 10 998 82.7 77.6 82.4 91.1), or 1024 where that is the whole context or with nine rounds and more (1600 of 1500 136 126
// 117 119).
//   * Sequences that together are less than a quarter of what they would be at the longest's length: two rounds, of 256 to 512
//     tokens, are there in the long ones alone, and a block that goes through 2048 tokens would outlast all others (16 sequences of
//     8 heads, one of 4096 tokens and 15 of 400: 18.3 25.4 30.1 29.2; 32 of one head, one of 16 384: 15.9 16.4 19.4 23.7).
NNHIP_HOST_DEVICE int attn_run(const AttnRunRule &r, uint32_t longest, uint32_t total) {
    auto steps = [](uint32_t tokens) { return (tokens + 127) / 128 * 128; };
    const uint32_t least = steps(attn_divide(longest + r.most.divisor - 1, r.most));
    const uint32_t even = steps(attn_divide(longest + r.round.divisor - 1, r.round));
    uint32_t run;
    if (longest <= 512) run = steps(longest);
    else if (total * 4 < longest * r.batch) run = std::min(std::max(steps(attn_divide(total, r.two_rounds)), 256u), 512u);
    else if (r.has_round && even <= 2048) run = std::max(even, 256u);
    else if (longest <= 1024) run = 1024;
    else run = (longest + 1023) / 1024 >= r.nine_rounds ? 1024 : 512;
    return (int)std::max(run, least);
}

// The same where every context fills the capacity, or 0 where the kernel above is taken (us, that one's best block / in steps):
//   * 64-wide heads, 257 to 512 tokens, from 24 pairs: one split, no merge (24 pairs of 265 tokens 5.8 / 5.3, 60 of 459 6.6 / 6.2, 240
//     of 384 7.8 / 5.9; 12 of 433 6.2 / 6.4).  Longer contexts come out even with that (12 pairs of 13 658 13.9 / 12.7, 84 of 4759
//     16.4 / 17.9, 132 of 14 756 50.7 / 52.1)
//   * 128-wide heads from 50 MB of keys and values on (48 pairs of 1851 15.2 / 13.8, 36 of 6028 22.3 / 17.9, 104 of 9746 107 / 80, 656 of
//     4073 267 / 229; below, 64 of 1205 12.1 / 13.0 and 8 of 4387 12.3 / 14.0), which few pairs reach with long contexts only, and too
//     many splits (8 of 12 668 18.4 / 20.0); not in a step or less a wave (1616 of 64 8.5 / 10.4, 8192 of 16 28.9 / 38.1, 4096 of 112 17.9 /
//     19.1; 192 of 512 level), nor where one split a pair is a block more for a few of the compute units (272 of 711 15.5 / 17.5, 260 of
//     984 22.4 / 26.2, 288 of 670 16.1 / 18.6; 308 of 690 20.7 / 19.0, 332 of 606 19.5 / 17.2, 436 of 622 24.2 / 20.1).  By the capacity: short
//     contexts in a large cache take it too, and are no slower for it (32 pairs of 300 / 1000 tokens in one of 16 384: 9.3 / 7.7 and 9.7 / 9.3).
inline int choose_attn_run(int head_dim, int64_t pairs, int64_t max_tokens, int compute_units) {
    if (head_dim == 64) return max_tokens > 256 && max_tokens <= 512 && pairs >= 24 ? (int)((max_tokens + 127) / 128 * 128) : 0;
    if (pairs < 16 || max_tokens <= 128 || pairs * max_tokens < 98304 || max_tokens > kAttnMaxSplits * 2048) return 0;
    if (max_tokens > 512 && max_tokens <= 1024 && pairs > compute_units && 6 * pairs <= 7ll * compute_units) return 0;
    return attn_run(attn_run_rule(1, pairs, compute_units, kAttnMaxSplits), (uint32_t)max_tokens, (uint32_t)max_tokens);
}

// Splits of a pair that a launch makes room for where the lengths are to choose the run, up to splits of 256 tokens: those that no
// sequence has cost a block each that reads the lengths and leaves.  2048 blocks of which most leave are not seen in the time (128 pairs,
// capacity 4096, one sequence of that length, the rest 400: 20.9 us with 2048, 25.7 with 1024; all 300: 8.4, 8.3); 9216 of them are (384 pairs of 300 14.1 -> 19.5).
inline int64_t attn_most_splits(int64_t pairs, int64_t max_tokens, int run) {
    return std::max((max_tokens + run - 1) / run, std::min((max_tokens + 255) / 256, std::min<int64_t>(2048 / pairs, kAttnMaxSplits)));
}

} // namespace nnhip
