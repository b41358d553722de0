// Launch bookkeeping of the kernels (ss2_kernels.hip), host only.
#pragma once

#include <algorithm>
#include <array>
#include <atomic>
#include <cstdint>

namespace vqm::ss2 {

// What `query` says of `Kernel` on `device`, asked once of each and kept while
// it is not 0. The kernel is part of the type, not an argument: kernels of one
// signature share every type they are passed by.
template <auto Kernel, typename Query>
uint32_t OncePerKernel(int device, Query&& query) {
    static std::array<std::atomic<uint32_t>, 64> known{};
    if (device < 0 || device >= static_cast<int>(known.size())) return query();
    uint32_t value = known[device].load(std::memory_order_relaxed);
    if (value == 0) known[device].store(value = query(), std::memory_order_relaxed);
    return value;
}

// The most blocks of `threads` threads a launch may have: HIP takes fewer than
// 2^32 threads. A multiple of 8, the XCDs.
constexpr uint32_t MaxBlocks(uint32_t threads) { return 0xFFFFFFFFu / threads / 8 * 8; }

// Launches `count` units, at most `most` at a time, in order:
// launch(first, n, last) for each run, until one fails.
template <typename Launch>
auto InRuns(uint32_t count, uint32_t most, Launch&& launch) {
    for (uint32_t first = 0;; first += most) {
        const uint32_t n = std::min(count - first, most);
        const bool last = n == count - first;
        const auto e = launch(first, n, last);
        if (last || e != decltype(e){}) return e;
    }
}

}  // namespace vqm::ss2
