// What is asked of the runtime once per kernel and device, as plain host code that a test can reach without a device.
#pragma once

#include <mutex>

namespace nnhip {

constexpr int kMostDevices = 16;

// ask() for the first caller per device, its result for every later one: a refusal stays one.  The kernel is part of the type (kernels
// with the same arguments are pointers of the same type, and would share the record).
template <auto Kernel, class F> auto once_per_kernel(int device, F &&ask) -> decltype(ask()) {
    static std::once_flag asked[kMostDevices];
    static decltype(ask()) result[kMostDevices];
    const int at = device & (kMostDevices - 1);
    std::call_once(asked[at], [&] { result[at] = ask(); });
    return result[at];
}

} // namespace nnhip
