// The sizes the allocation-free entry point takes (PlanNoAlloc, ss2_host.cc):
// they are those whose items, one partial sum a strip and planes fit 128 MiB,
// whatever parts a strip is cut into, and all of them fit the scratch. The
// sizes lie along the limit, over aspect ratios from 8 columns to 8 rows.
#include <cmath>
#include <cstdio>

#include "ss2_host.h"

using namespace vqm::ss2;

namespace {
int failures = 0;
unsigned taken = 0, refused = 0;

uint64_t Up(uint64_t v) { return (v + 255) / 256 * 256; }

void Check(uint32_t w, uint32_t h, PlaneFormat format, uint32_t rows, uint32_t cols) {
    const Plan p = FillPlan(w, h, format, SinglePairStripRows(w, h, format, rows, cols), cols);
    const uint64_t need = Up(Up(2048 + p.items * sizeof(ScaleItem)) + p.items * 48ull) + 2 * p.image_bytes;
    const bool fits = need <= 128ull << 20;
    bool ok = true;
    try {
        const NoAllocPlan n = PlanNoAlloc(w, h, format, rows, cols);
        const uint32_t parts = SinglePairRowParts(w, h, format, rows, cols);
        ok = fits && n.block_form == (parts == 0) &&
             n.parts == static_cast<uint64_t>(n.plan.items) << n.plan.part_shift &&
             n.partials_at >= kNoAllocItemsAt + n.plan.items * sizeof(ScaleItem) &&
             n.planes_at >= n.partials_at + n.parts * 48 && n.partials_at % 256 == 0 && n.planes_at % 256 == 0 &&
             n.planes_at + 2 * n.plan.image_bytes <= kNoAllocScratchBytes;
        ++taken;
    } catch (const Error& e) {
        ok = !fits && e.status == VQM_INVALID_ARGUMENT;
        ++refused;
    }
    if (!ok && failures++ < 20)
        std::fprintf(stderr, "%ux%u format %d rows %u cols %u: needs %llu\n", w, h, static_cast<int>(format), rows, cols,
                     static_cast<unsigned long long>(need));
}
}  // namespace

int main() try {
    for (PlaneFormat format : {kPlaneF32, kPlaneU16}) {
        // Taken before a strip was cut into parts.
        for (auto [w, h] : {std::pair{1692u, 5271u}, {4874u, 1868u}, {5281u, 1745u}, {5762u, 1540u}, {6798u, 2770u}, {1666u, 5251u}})
            Check(w, h, format, 0, 0);
        for (auto [rows, cols] : {std::pair{0u, 0u}, {0u, 64u}, {0u, 128u}, {8u, 0u}, {8u, 64u}, {64u, 128u}, {1024u, 0u}})
            for (double x = std::log(8.0); x < std::log(1 << 20); x += 0.017) {
                const auto w = static_cast<uint32_t>(std::exp(x) + 0.5);
                uint32_t low = 8, high = 1u << 20;  // the tallest pair of this width that is taken, near enough
                while (high - low > 1) {
                    const uint32_t mid = low + (high - low) / 2;
                    bool below = false;  // nor where the plan itself overflows
                    try {
                        below = 2 * FillPlan(w, mid, format, rows, cols).image_bytes <= 128ull << 20;
                    } catch (const Error&) {
                    }
                    (below ? low : high) = mid;
                }
                for (int d = -40; d <= 8; ++d) {
                    const int64_t h = static_cast<int64_t>(low) + d * std::max<int64_t>(1, low / 2000);
                    if (h >= 8 && h <= 1 << 20) Check(w, static_cast<uint32_t>(h), format, rows, cols);
                }
            }
    }
    std::printf("%u taken, %u refused\n", taken, refused);
    if (taken < 1000 || refused < 1000) ++failures;
    if (failures) std::fprintf(stderr, "%d failures\n", failures);
    return failures != 0;
} catch (const Error& e) {
    std::fprintf(stderr, "%s\n", e.message.c_str());
    return 1;
}
