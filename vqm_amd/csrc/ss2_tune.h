// Launch-shape autotuner: picks the scale launch's shape (TuneShapes) and the
// batch chunk count for a geometry, plane format and batch size by timing
// every candidate on the device. No shape changes a pixel's arithmetic or an
// FP32 block sum; only the order of the FP64 strip partials follows the
// strips, so the choice is free to follow the measurement. Choices are cached per (width,
// height, format, map form, batch-size class) for the process.
#pragma once

#include <cstdint>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "ss2_common.h"
#include "ss2_host.h"

namespace vqm::ss2 {

struct TuneChoice {
    // The fastest shape that a caller can set.
    uint32_t strip_rows = 64;
    uint32_t strip_cols = kDefaultStripCols;
    uint32_t chunks = 1;
    float ms_per_launch = 0.0f;  // best candidate, milliseconds per launch
    float default_ms = 0.0f;     // the default shape (64 rows, 128 columns, 1 chunk)
    uint32_t candidates = 0;     // shapes timed
    bool cached = false;
    // What a batch takes: the fastest of all shapes, and of all strips (a
    // launch of several geometries, a persistent one).
    struct Launch {
        ScaleShape shape;
        uint32_t chunks = 1;
    };
    Launch any, strips;
};

class Tuner {
public:
    static Tuner& Get();
    // Chunk counts tried.
    static constexpr uint32_t kChunks[] = {1, 2, 4, 8};
    // The batch-size class a pair count falls in: the next power of two,
    // capped at 512.
    static uint32_t SizeClass(uint32_t pairs);
    TuneChoice Choose(uint32_t width, uint32_t height, PlaneFormat format, MapForm map, uint32_t pairs);

private:
    std::mutex mu_;
    std::map<std::tuple<uint32_t, uint32_t, uint32_t, uint32_t, uint32_t>, TuneChoice> cache_;
};

}  // namespace vqm::ss2
