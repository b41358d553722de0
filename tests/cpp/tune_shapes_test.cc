// The autotuner's candidates (TuneShapes, ss2_host.cc) hold the shape that a
// launch takes where none is set, alone or beside others, and every shape that
// a caller can set, those first.
#include <algorithm>
#include <cstdio>
#include <set>

#include "ss2_host.h"

using namespace vqm::ss2;

int main() {
    int failures = 0;
    std::set<uint32_t> seen;  // row_parts
    const uint32_t sizes[][2] = {{8, 8}, {96, 64}, {512, 512}, {853, 479}, {1920, 1080}, {3840, 2160}, {200, 5000}};
    for (auto [w, h] : sizes)
        for (PlaneFormat format : {kPlaneF32, kPlaneF16, kPlaneU16})
            for (uint64_t pairs : {1ull, 2ull, 8ull, 64ull, 512ull})
                for (uint32_t cus : {256u, 32u}) {
                    const std::vector<ScaleShape> shapes = TuneShapes(w, h, format, pairs, cus);
                    for (bool blocks : {false, true}) {
                        const ScaleShape d = DefaultShape(w, h, format, 0, pairs, cus, blocks);
                        seen.insert(d.row_parts);
                        // The tuner names the default width.
                        const bool in = std::any_of(shapes.begin(), shapes.end(), [&](const ScaleShape& s) {
                            return s.rows == d.rows && s.row_parts == d.row_parts &&
                                   (s.cols == d.cols || s.cols == kDefaultStripCols);
                        });
                        if (!in && failures++ < 20)
                            std::fprintf(stderr, "%ux%u format %d, %llu pairs: %u rows, %u parts\n", w, h,
                                         static_cast<int>(format), static_cast<unsigned long long>(pairs), d.rows,
                                         d.row_parts);
                        BuildPlan(w, h, format, d.rows, d.cols, d.row_parts);
                    }
                    for (size_t k = 0; k < kTuneSettable; ++k)
                        failures += shapes[k].row_parts != 1 || shapes[k].cols == 0 || shapes[k].rows % 8 != 0;
                    for (const ScaleShape& s : shapes) BuildPlan(w, h, format, s.rows, s.cols, s.row_parts);
                }
    failures += kTuneSettable != 12 || !seen.count(0) || !seen.count(1) || !seen.count(2);
    // One pair's default shape is a pipeline's.
    failures += DefaultShape(96, 64, kPlaneF32, 0, 1, 256, true).row_parts != SinglePairRowParts(96, 64, kPlaneF32, 0, 0);
    failures += DefaultShape(3840, 2160, kPlaneF32, 0, 1, 256, true).row_parts !=
                SinglePairRowParts(3840, 2160, kPlaneF32, 0, 0);
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    else std::printf("tune shapes ok\n");
    return failures != 0;
}
