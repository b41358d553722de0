// OncePerKernel (ss2_launch.h): kernels of one signature keep their own values,
// so do devices, and each is asked once.
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
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    else std::printf("launch ok\n");
    return failures != 0;
}
