// ss2_launch.h: kernels of one signature keep their own values in OncePerKernel,
// so do devices, and each is asked once; and launches of 2^32 threads or more
// (1,000,000 pairs' reduce, 5,000 1080p pairs in the scale kernel's block form)
// are cut into runs that HIP takes, in order and whole.
#include <cstdio>

#include "ss2_launch.h"

using namespace vqm::ss2;

namespace {
template <int N>
void Kernel(const float*, uint32_t) {}
int asked = 0;

template <auto K>
uint32_t Value(int device, uint32_t value) {
    return OncePerKernel<K>(device, [&] { return ++asked, value; });
}
}  // namespace

int main() {
    int failures = 0;
    failures += Value<&Kernel<0>>(0, 1024) != 1024;
    failures += Value<&Kernel<1>>(0, 2560) != 2560;  // the same signature, other occupancy
    failures += Value<&Kernel<0>>(1, 128) != 128;
    failures += asked != 3;
    failures += Value<&Kernel<0>>(0, 1) != 1024 || Value<&Kernel<1>>(0, 1) != 2560 || Value<&Kernel<0>>(1, 1) != 128;
    failures += asked != 3;
    // A device past the table and a value of 0 are asked again.
    failures += Value<&Kernel<0>>(64, 7) != 7 || Value<&Kernel<0>>(-1, 8) != 8;
    failures += Value<&Kernel<2>>(0, 0) != 0 || Value<&Kernel<2>>(0, 9) != 9;
    failures += asked != 7;

    for (uint32_t threads : {64u, 128u, 256u, 512u, 1024u}) {
        failures += MaxBlocks(threads) % 8 != 0 || static_cast<uint64_t>(MaxBlocks(threads)) * threads >= 1ull << 32;
        failures += (static_cast<uint64_t>(MaxBlocks(threads)) + 8) * threads < (1ull << 32) - threads;
    }
    struct Case {
        uint32_t count, unit, threads;  // blocks a unit
    };
    for (const Case c : {Case{1, 18, 256}, {932067, 18, 256}, {932068, 18, 256}, {1000000, 18, 256}, {4000000, 18, 256},
                         {5000, 1752, 512}, {4789, 1752, 512}, {9000000, 1, 512}, {0x7FFFFFFFu, 1, 512}}) {
        uint64_t next = 0;
        uint32_t lasts = 0;
        const uint32_t most = MaxBlocks(c.threads) / c.unit;
        failures += InRuns(c.count, most, [&](uint32_t first, uint32_t n, bool last) {
                        failures += first != next || n == 0 || n > most || lasts != 0;
                        failures += static_cast<uint64_t>(n) * c.unit * c.threads >= 1ull << 32;
                        next += n;
                        lasts += last;
                        return 0;
                    }) != 0;
        failures += next != c.count || lasts != 1;
    }
    // The first failure ends them.
    int runs = 0;
    failures += InRuns(10, 3, [&](uint32_t, uint32_t, bool) { return ++runs == 2 ? 5 : 0; }) != 5 || runs != 2;
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    else std::printf("launch ok\n");
    return failures != 0;
}
