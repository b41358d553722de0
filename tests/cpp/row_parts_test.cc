// RowParts and the parts of a plan (ss2_host.cc): every output pixel of every
// stored plane lies in exactly one part, and a part's source rows, rounded up
// to steps of four, stay inside the padded plane.
#include <cstdio>
#include <vector>

#include "ss2_host.h"

using namespace vqm::ss2;

int main() {
    int failures = 0;
    const uint32_t sizes[][2] = {{8, 8}, {13, 9}, {64, 64}, {65, 71}, {96, 64}, {129, 97}, {300, 200}, {512, 512}, {853, 479}, {1920, 1080}};
    for (auto [w, h] : sizes)
        for (uint32_t rows : {8u, 16u, 24u, 32u, 64u, 104u, 192u})
            for (uint32_t cols : {64u, 128u})
                for (uint64_t pairs : {1ull, 16ull, 300ull}) {
                    const uint32_t bands = RowParts(w, h, kPlaneF32, rows, cols, pairs, 256);
                    const GeometryPlan g = BuildPlan(w, h, kPlaneF32, rows, cols, bands);
                    const Plan& p = g.plan;
                    if (p.part_h * bands != rows || p.part_h % kSumBlockRows != 0 ||
                        (1u << p.part_shift) != bands * (cols / 64)) {
                        std::fprintf(stderr, "%ux%u %u rows: %u bands of %u\n", w, h, rows, bands, p.part_h);
                        ++failures;
                        continue;
                    }
                    std::vector<std::vector<uint8_t>> cover(kMaxScales * kChannels);
                    for (uint32_t l = 0; l < p.levels; ++l)
                        for (int c = 0; c < kChannels; ++c) cover[l * 3 + c].assign(static_cast<size_t>(p.w[l]) * p.h[l], 0);
                    for (uint32_t part = 0; part < g.parts(); ++part) {
                        const ScaleItem& it = g.items[part >> p.part_shift];
                        const uint32_t sub = part & ((1u << p.part_shift) - 1), wide = p.strip_w / 128;
                        const uint32_t x0 = it.x0 + 64 * (sub & wide), y0 = it.y0 + (sub >> wide) * p.part_h;
                        if (x0 >= p.w[it.level] || y0 >= p.h[it.level]) continue;
                        const uint32_t out = std::min(p.part_h, p.h[it.level] - y0);
                        const uint32_t last_row = y0 + (out + 2 * kRadius + 3) / 4 * 4 - 1;
                        if (last_row >= p.rows[it.level] || x0 + 2 + 64 + 2 * kRadius > p.pitch[it.level]) ++failures;
                        for (uint32_t y = y0; y < y0 + out; ++y)
                            for (uint32_t x = x0; x < std::min(x0 + 64, p.w[it.level]); ++x)
                                ++cover[it.level * 3 + it.channel][static_cast<size_t>(y) * p.w[it.level] + x];
                    }
                    for (uint32_t l = 0; l < p.levels; ++l)
                        for (int c = 0; c < kChannels; ++c)
                            if (p.mask[l] & (1u << c))
                                for (uint8_t n : cover[l * 3 + c]) failures += n != 1;
                }
    // One 96x64 pair is one wave's chain of steps: shorter bands; 300 1080p
    // pairs fill the device: whole strips.
    failures += RowParts(96, 64, kPlaneF32, 16, 0, 1, 256) != 2;
    failures += RowParts(1920, 1080, kPlaneF32, 192, 0, 300, 256) != 1;
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    else std::printf("row parts ok\n");
    return failures != 0;
}
