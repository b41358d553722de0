// A pooled workspace (PooledWorkspace, ss2_host.h) takes no more than the
// planes of uncut strips, one partial sum a strip and 1,024 bytes, whichever
// parts the shape is cut into, so that a budget counted that way holds it.
// Prints the bytes of a 1024x1024 pair counted so.
#include <cstdio>

#include "ss2_host.h"

using namespace vqm::ss2;

namespace {
uint64_t Up(uint64_t v) { return (v + 255) / 256 * 256; }
uint64_t Counted(const Plan& p) { return Up(2 * p.image_bytes) + Up(p.items * 48ull) + 1024; }
}  // namespace

int main() {
    int failures = 0;
    const uint32_t sizes[][2] = {{8, 8},     {13, 9},      {64, 64},     {129, 97},   {512, 512}, {853, 479},
                                 {1024, 1024}, {1920, 1080}, {3840, 2160}, {8, 20000}, {20000, 8}};
    for (auto [w, h] : sizes)
        for (PlaneFormat format : {kPlaneF32, kPlaneU16})
            for (uint32_t cols : {0u, 64u, 128u})
                for (uint64_t pairs : {1ull, 8ull, 300ull})
                    for (uint32_t fixed : {0u, 8u, 64u}) {
                        const uint32_t rows = fixed ? fixed : DefaultStripRows(w, h, format, cols, pairs, 256);
                        const uint64_t counted = Counted(FillPlan(w, h, format, rows, cols));
                        for (uint32_t parts : {0u, 1u, 2u, 4u}) {
                            if (parts != 0 && rows % (kSumBlockRows * parts) != 0) continue;
                            const GeometryPlan g = BuildPlan(w, h, format, rows, cols, parts);
                            if (parts == 0 && cols != 0) continue;  // not taken
                            if (PooledWorkspace(LayoutWorkspace(g)).total > counted && failures++ < 20)
                                std::fprintf(stderr, "%ux%u format %d rows %u cols %u parts %u\n", w, h,
                                             static_cast<int>(format), rows, cols, parts);
                        }
                    }
    std::printf("%llu\n", static_cast<unsigned long long>(Counted(FillPlan(1024, 1024, kPlaneF32, 64))));
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    return failures != 0;
}
