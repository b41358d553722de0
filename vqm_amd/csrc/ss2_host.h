// Host-side logic of the SSIMULACRA 2.1 path: scale plan, taps, pruning,
// score mapping, input validation, decode table and the per-geometry work
// plan the kernels consume. No GPU calls here.
#pragma once

#include <array>
#include <cstddef>
#include <cstdint>
#include <iterator>
#include <map>
#include <string>
#include <vector>

#include "ss2_common.h"
#include "vqm_ss2.h"

namespace vqm::ss2 {

// Thrown by host logic; the C ABI maps each to its status code.
struct Error {
    int status;
    std::string message;
};

[[noreturn]] void Fail(int status, std::string message);

struct ScalePlan {
    uint32_t count = 0;
    std::array<uint32_t, kMaxScales> w{}, h{};
};

// pipeline.cc:28-48.
ScalePlan PlanScales(uint32_t width, uint32_t height);

// pipeline.cc:274-291: 13 FP32 taps of exp(-0.5 (k/1.5)^2) normalised in FP64.
std::array<float, kTaps> GaussianTaps();

// score.cc:103-114.
bool ChannelPruned(uint32_t channel, uint32_t scale, uint32_t scales);

// score.cc:118-163. Throws Error{VQM_INVALID_ARGUMENT} on more than six
// scales, nonfinite norms or an overflowing mapping.
double Score(uint32_t scales, const double* norms);

// The u8 sRGB decode table the prepare kernel reads: FP32 decode scale
// (input.cc:714-757) and the IEC 61966-2-1 EOTF (color.glsl:135-137).
std::array<float, 256> SrgbTable();

// vqm_image.h:122-133 and input.cc:114-145,244-255: packed planes, each
// starting on a 4-byte boundary.
uint64_t RequiredBytes(const vqm_image_format& format, uint32_t width, uint32_t height);

// input.cc:152-240: the image matches the geometry, its format is one the
// reference accepts, and its byte length is RequiredBytes. Throws
// Error{VQM_INVALID_ARGUMENT}.
void CheckImage(const vqm_image_desc& image, uint32_t width, uint32_t height,
                const char* name);

// image_view.cc:16-45 (DescribeImageView): a non-empty size, a format the
// reference accepts, a pointer and a stride of at least one row for every
// present plane, and a last row whose end is addressable. Returns the
// packed byte length. Throws Error{VQM_INVALID_ARGUMENT} or
// Error{VQM_OVERFLOW}.
uint64_t CheckView(const vqm_host_view& view);

// image_view.cc:47-77 (PackImageView): copies a checked view into the
// packed layout at `dst` (CheckView's length), zeroing the at most three
// bytes that pad each plane to a 4-byte boundary.
void PackView(const vqm_host_view& view, uint8_t* dst);

// Per-geometry plan: level sizes, padded plane geometry, plane offsets per
// image, the scale work items and their per-(level, channel) ranges.
struct GeometryPlan {
    Plan plan{};
    std::vector<ScaleItem> items;
    uint64_t plane_bytes_per_image = 0;  // padded plane storage
    PlaneFormat format = kPlaneF32;
    uint32_t prep_tiles = 0;             // prepare blocks per image
    bool block_form = false;             // the scale kernel's form (RowParts)
    uint32_t parts() const { return plan.items << plan.part_shift; }  // scale blocks per pair
};

// strip_rows: output rows per scale work item, a multiple of 8 up to 1024
// (0 = 64; launches pick theirs with DefaultStripRows); strip_cols: its
// width, 64 or 128 columns (0 = 128); row_parts: 1, 2 or 4 bands of a
// multiple of 8 rows a strip is cut into, one wave each (RowParts), or 0: the
// scale kernel's block form, whose strips are kBlockRows rows by 64 columns
// whatever the other two are.
GeometryPlan BuildPlan(uint32_t width, uint32_t height, PlaneFormat format,
                       uint32_t strip_rows, uint32_t strip_cols = 0, uint32_t row_parts = 1);

// The plan alone, without the item table (ItemAt enumerates the items):
// nothing is allocated.
Plan FillPlan(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_rows,
              uint32_t strip_cols = 0, uint32_t row_parts = 1);

// The default strip height of a scale launch over `pairs` pairs of this
// geometry on a device of `cus` compute units: 192 rows when their work
// items fill every wave slot of the device (8 per CU) four times over, else
// 128 when theirs fill every slot once, else the tallest of 64 and 32 rows
// whose items give each SIMD one (4 per CU), else 16. Taller strips blur
// each strip's 12 halo rows over more output rows; shorter ones keep a
// narrow launch (one pair, a small batch) wide.
uint32_t DefaultStripRows(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_cols,
                          uint64_t pairs, uint32_t cus);

// The strip height of a single-pair pipeline (and of the allocation-free
// entry point): `strip_rows` when set, else DefaultStripRows for one pair on
// a whole MI355X (256 CUs), a function of the geometry alone so that the
// memory plan, which needs no device, predicts it (16 rows at 1080p, 64 at
// 4K).
uint32_t SinglePairStripRows(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_rows,
                             uint32_t strip_cols);

// The bands a default strip height is cut into (1, 2 or 4), by the scale
// launch's modelled time on a device of `cus` compute units: a wave takes a
// band in steps of four rows, three of them for the 12 halo rows, so short
// bands repeat more work and tall ones leave a small launch waiting for one
// wave's chain of steps. An explicit height is one band, so that equal
// heights give equal sums whatever the launch.
uint32_t RowParts(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_rows, uint32_t strip_cols,
                  uint64_t pairs, uint32_t cus);

// Whether a scale launch of `pairs` pairs of this geometry alone takes the
// block form.
bool PrefersBlocks(uint32_t width, uint32_t height, PlaneFormat format, uint64_t pairs, uint32_t cus);

// A scale launch's shape: FillPlan's strip_rows, strip_cols (0: the default
// width) and row_parts.
struct ScaleShape {
    uint32_t rows = 64, cols = 0, row_parts = 1;
    bool operator==(const ScaleShape&) const = default;
};

// The shape that a launch of `pairs` pairs of this geometry takes where none is
// set: DefaultStripRows cut by RowParts, or the block form where PrefersBlocks
// and `blocks` (the geometry alone, one block a part, no strip width set).
ScaleShape DefaultShape(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_cols, uint64_t pairs,
                        uint32_t cus, bool blocks);

// The shapes the autotuner times: first those that a caller can set, every
// height of kTuneRows in both widths, then the default shape of such a launch
// where it is another (cut strips) and the block form.
inline constexpr uint32_t kTuneRows[] = {16, 32, 64, 128, 192, 256};
inline constexpr uint32_t kTuneCols[] = {64, 128};
inline constexpr size_t kTuneSettable = std::size(kTuneRows) * std::size(kTuneCols);
std::vector<ScaleShape> TuneShapes(uint32_t width, uint32_t height, PlaneFormat format, uint64_t pairs, uint32_t cus);

// RowParts of a single-pair pipeline's default height (of the geometry
// alone, as SinglePairStripRows), or 0 for the block form, where neither
// `strip_rows` nor `strip_cols` is set; 1 when `strip_rows` is set.
uint32_t SinglePairRowParts(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_rows,
                            uint32_t strip_cols);

// Bytes of one pair's workspace: planes of both images and partials, each
// rounded to 256 bytes.
struct WorkspaceLayout {
    uint64_t planes = 0, partials = 0, total = 0;
};
WorkspaceLayout LayoutWorkspace(const GeometryPlan& plan);

// What a pair's workspace holds in the pools of batches and servers: its
// planes. The partials of the pairs in flight are their lane's (a strip's
// parts have up to eight times the sums of a strip, so that workspaces with
// them would not fit a budget that held them with one sum a strip).
inline WorkspaceLayout PooledWorkspace(const WorkspaceLayout& layout) { return {layout.planes, 0, layout.planes}; }

// The allocation-free entry point's pairs. It takes a pair whose regions of
// fixed size, items, one partial sum a strip and planes of both images fit
// kNoAllocPairBytes, whichever form of the scale kernel runs. Its scratch is
// larger: a strip has up to eight parts, of 48 bytes each, and the planes
// under a part (8 rows or more by 64 columns, two images of two bytes a sample
// or more) hold 2,048 bytes or more, so the parts of such a pair take at most
// 48 / 2048 of kNoAllocPairBytes, 3 MiB.
inline constexpr uint64_t kNoAllocPairBytes = 128ull << 20;
inline constexpr uint64_t kNoAllocScratchBytes = 132ull << 20;
inline constexpr uint64_t kNoAllocItemsAt = 2048;  // behind the regions of fixed size
struct NoAllocPlan {
    Plan plan{};
    bool block_form = false;
    uint64_t parts = 0;                       // scale blocks
    uint64_t partials_at = 0, planes_at = 0;  // scratch offsets
};
// The plan of a single-pair pipeline of this geometry, so that both give the
// same sums. Throws Error{VQM_INVALID_ARGUMENT} for a pair that it does not
// take.
NoAllocPlan PlanNoAlloc(uint32_t width, uint32_t height, PlaneFormat format, uint32_t strip_rows,
                        uint32_t strip_cols);

// Offset bookkeeping of a device arena: ranges of a fixed capacity handed
// out in 256-byte multiples by first fit over an address-ordered free list,
// neighbours merged on release.
class RangeAllocator {
public:
    static constexpr uint64_t kAlign = 256;
    explicit RangeAllocator(uint64_t capacity);
    // Offset of a new range of `bytes`, or ~0 when no free range fits.
    uint64_t Alloc(uint64_t bytes);
    void Free(uint64_t offset, uint64_t bytes);
    uint64_t capacity() const { return capacity_; }
    uint64_t free_bytes() const;
    size_t free_ranges() const { return free_.size(); }
    static constexpr uint64_t kNone = ~0ull;

private:
    uint64_t capacity_;
    std::map<uint64_t, uint64_t> free_;  // offset -> length
};

// Algorithmic HBM bytes of one pair: both u8 inputs read once, every stored
// plane element written once and read once per image.
uint64_t AlgorithmicBytes(const GeometryPlan& plan);

}  // namespace vqm::ss2
