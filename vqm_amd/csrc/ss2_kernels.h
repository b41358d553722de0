// Host-side launch API of the SSIMULACRA 2.1 kernels (ss2_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ss2_common.h"

namespace vqm::ss2 {

// A flat work list entry: pair index in the batch and the local work index
// (prepare: tile | image << 31; scale: part). Used when a batch mixes
// geometries; a batch of one geometry indexes blocks arithmetically.
struct WorkRef {
    uint32_t pair;
    uint32_t index;
};

// sRGB decode table and taps live in device memory owned by the caller.
// All launches are asynchronous on `stream`. `done` (null: none) is an event
// that the kernel's own dispatch sets as it ends. Three events recorded behind
// the kernels, as packets of their own, held the next kernel back 5.6 us each:
// a 96x64 pair took 61.0 us against 44.4, a 1080p pair 91.5 against 72.5. An
// event for a kernel's start is not given: it made the launch itself slower
// (51 us for the three kernels, against 13).

// Builds every stored plane of both images of each pair.
// Uniform geometry: blocks = pairs * 2 * tiles_per_image, work = nullptr.
// src0/src1, when not null, replace every pair's inputs (single-pair use).
// general: some image of the launch has a SourceDesc of kind 1 (formats
// other than 8-bit sRGB RGB); the table-only kernel ignores descriptors.
// `persistent`: launch only as many blocks as stay resident at once, each
// looping over the work items (the grid otherwise covers them, one each).
// `map` picks the arithmetic form of the XYB transform (MapForm).
hipError_t LaunchPrepare(PlaneFormat format, MapForm map, bool general, const PairDesc* pairs,
                         const WorkRef* work, uint32_t blocks, uint32_t tiles_per_image, const float* lut,
                         const uint8_t* src0, const uint8_t* src1, hipStream_t stream,
                         bool persistent = false, hipEvent_t done = nullptr);

// One 64-lane wave per part of a scale work item (level, channel, 64 columns
// by Plan::part_h rows). Uniform geometry: blocks = pairs * parts_per_pair,
// work = nullptr; else work[].index is a part. `blur` picks the kernel: kBlurSampled (13-tap sampled Gaussian)
// or kBlurRecursive (the recursive Gaussian's 9-tap truncated-cosine
// kernel); `map` the SSIM' map's form, which must be the one the planes were
// prepared with. block_form: the plans are of that form (GeometryPlan), a
// block of 512 threads per item; not with `persistent`.
hipError_t LaunchScale(PlaneFormat format, uint32_t blur, MapForm map, const PairDesc* pairs, const WorkRef* work,
                       uint32_t blocks, uint32_t parts_per_pair, bool block_form, hipStream_t stream,
                       bool persistent = false, hipEvent_t done = nullptr);

// Sums each (level, channel) norm's partials in FP64 and writes the 108 norms
// (device or pinned host memory).
hipError_t LaunchReduce(const PairDesc* pairs, uint32_t pairs_count, hipStream_t stream, hipEvent_t done = nullptr);

// Device-to-device copy of `bytes` (a multiple of 16) by a plain kernel.
hipError_t LaunchCopy(void* dst, const void* src, uint64_t bytes, hipStream_t stream);

// Counters of the cube-root self-check; `first_mismatch` starts at
// 0xFFFFFFFF and the others at 0.
struct CbrtCheck {
    unsigned long long mismatches;
    unsigned long long near;
    unsigned long long max_h_bits;
    uint32_t first_mismatch;
    uint32_t pad;
};

// Compares the reference form's cube root (hardware-seeded) with the one of
// IEEE steps only for every float with bits in [first, end), adding to `out`.
hipError_t LaunchCbrtCheck(uint32_t first, uint32_t end, CbrtCheck* out, hipStream_t stream);

// Counters of the division self-check; `first_mismatch` starts at
// 0xFFFFFFFF and the others at 0.
struct DivCheck {
    unsigned long long mismatches;
    unsigned long long rcp_mismatches;
    uint32_t first_mismatch;
    uint32_t pad;
};

// Compares the map's division with the IEEE quotient for b significands
// [mb_first, mb_first + rows) against every a significand, and the hardware
// reciprocal's exponent invariance for those b, adding to `out`.
hipError_t LaunchDivCheck(uint32_t mb_first, uint32_t rows, DivCheck* out, hipStream_t stream);

}  // namespace vqm::ss2
