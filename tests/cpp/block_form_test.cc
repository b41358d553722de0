// The block form's plans (row_parts 0, ss2_host.cc): every output pixel of
// every stored plane lies in exactly one block, a block's loads stay inside
// the padded plane, and its pair takes no more memory than the strip form's.
#include <cstdio>
#include <vector>

#include "ss2_host.h"

using namespace vqm::ss2;

int main() {
    int failures = 0;
    const uint32_t sizes[][2] = {{8, 8}, {13, 9}, {64, 32}, {65, 33}, {127, 63}, {129, 97}, {300, 200}, {853, 479}, {1920, 1080}};
    for (auto [w, h] : sizes)
        for (PlaneFormat format : {kPlaneF32, kPlaneU16}) {
            const GeometryPlan g = BuildPlan(w, h, format, 0, 0, 0);
            const Plan& p = g.plan;
            if (!g.block_form || p.part_shift != 0 || p.part_h != kBlockRows || p.strip_w != 64) ++failures;
            std::vector<std::vector<uint8_t>> cover(kMaxScales * kChannels);
            for (uint32_t l = 0; l < p.levels; ++l)
                for (int c = 0; c < kChannels; ++c) cover[l * 3 + c].assign(static_cast<size_t>(p.w[l]) * p.h[l], 0);
            for (const ScaleItem& it : g.items) {
                const uint32_t W = p.w[it.level], H = p.h[it.level];
                const uint32_t out = std::min(kBlockRows, H - it.y0);
                // The horizontal passes read whole steps of four rows and 78
                // columns from x0 (two of padding, 64 and the halo).
                const uint32_t rows = (out + 2 * kRadius + 3) / 4 * 4;
                failures += it.x0 >= W || it.y0 >= H || it.y0 + rows > p.rows[it.level] || it.x0 + 78 > p.pitch[it.level];
                for (uint32_t y = it.y0; y < it.y0 + out; ++y)
                    for (uint32_t x = it.x0; x < std::min(it.x0 + 64, W); ++x)
                        ++cover[it.level * 3 + it.channel][static_cast<size_t>(y) * W + x];
            }
            for (uint32_t l = 0; l < p.levels; ++l)
                for (int c = 0; c < kChannels; ++c)
                    if (p.mask[l] & (1u << c))
                        for (uint8_t n : cover[l * 3 + c]) failures += n != 1;
            const uint32_t rows = SinglePairStripRows(w, h, format, 0, 0);
            const GeometryPlan strips = BuildPlan(w, h, format, rows, 0, RowParts(w, h, format, rows, 0, 1, 256));
            failures += LayoutWorkspace(g).total > LayoutWorkspace(strips).total;
        }
    // The rule's two sides, and explicit shapes.
    failures += SinglePairRowParts(96, 64, kPlaneF32, 0, 0) != 0;
    failures += SinglePairRowParts(1920, 1080, kPlaneF32, 0, 0) != 0;
    failures += SinglePairRowParts(1920, 1080, kPlaneU16, 0, 0) == 0;
    failures += SinglePairRowParts(3840, 2160, kPlaneF32, 0, 0) == 0;
    failures += SinglePairRowParts(96, 64, kPlaneF32, 0, 64) == 0;
    failures += SinglePairRowParts(96, 64, kPlaneF32, 16, 0) != 1;
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    else std::printf("block form ok\n");
    return failures != 0;
}
