// Launch bookkeeping of the kernels (ss2_kernels.hip), host only.
#pragma once

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

}  // namespace vqm::ss2
