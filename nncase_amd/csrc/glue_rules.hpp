// What the glue kernels are built for, as plain host arithmetic that a test can reach without a device.
#pragma once

namespace nnhip {

// A window's values are asked for in turns of up to five before the first is compared.  How many a turn takes: the window spread
// evenly over its turns, since what a turn asks for past the window's end is loaded all the same (16 x 112 x 112 by 64 at stride 1,
// us, value by value / in turns of five / evenly: 2 x 2 8.9 / 10.6 / 7.6, 3 x 3 13.7 / 13.2 / 10.5, 5 x 5 26.3 / 18.8 / 18.8, 7 x 7
// 44.7 / 39.3 / 33.1).
constexpr int kMostLoadsPerTurn = 5;
inline int loads_per_turn(int window) {
    const int turns = (window + kMostLoadsPerTurn - 1) / kMostLoadsPerTurn;
    return (window + turns - 1) / turns;
}

} // namespace nnhip
