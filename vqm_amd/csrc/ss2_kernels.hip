// SSIMULACRA 2.1 kernels for CDNA4 (gfx950), wave64.
//
//   prepare  u8 sRGB -> linear (256-entry table) -> XYB, plus the 2x2 box
//            pyramid of the linear planes, writing only the (level, channel)
//            planes whose maps survive pruning (prepare.comp:170-232).
//   scale    one wave per 64-column part of a strip of one (level, channel):
//            the 13-tap blurs of the map's quantities, the SSIM' and edge
//            maps, and six map sums, FP32 over 8-row blocks then FP64
//            (scale.comp:335-437). Rows stream through the wave four at a
//            time: staged in LDS, blurred horizontally (lane = row and four
//            columns), turned in LDS to lane = column, and added to the
//            partial sums of the output rows that wait for them. No map ever
//            reaches HBM.
//   reduce   FP64 sum of each norm's per-strip partials, 1-norm means and
//            4-norm fourth roots (reduce.comp:21-63, vulkan.cc:545-583).
//
// Two arithmetic forms (MapForm) share the kernels: the reference form
// (prepare.comp and scale.comp in their own operation order, correctly
// rounded cube roots, five blurred quantities) and the difference form (the
// SSIM' map from four blurred quantities, rearranged to avoid a cancellation).
//
// Arithmetic contract. Every FP32 operation below is an IEEE add, multiply,
// fused multiply-add (written explicitly), division, min/max, abs or an
// integer/float conversion, with contraction switched off, so the CPU
// oracle's FP32 forms (ref for the reference form, dev for the difference
// form) reproduce each pixel's values bit for bit. The blur runs horizontal
// pass first with taps in ascending order, as scale.comp:149-301 does.
//
// Memory access. Descriptors (pairs, plans, work items) are read through
// constant-address-space pointers so that their uniform fields become scalar
// loads; images and planes through global-address-space pointers.

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "ss2_cbrt.h"
#include "ss2_common.h"
#include "ss2_kernels.h"
#include "ss2_launch.h"

#pragma clang fp contract(off)

namespace vqm::ss2 {
namespace {

template <typename T> using ConstAS = __attribute__((address_space(4))) const T;
template <typename T> using GlobalAS = __attribute__((address_space(1))) T;

// Builtin vector types for wide loads and stores through qualified pointers.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ ConstAS<T>* as_const(const T* p) {
    return (ConstAS<T>*)p;
}
template <typename T>
__device__ __forceinline__ GlobalAS<T>* as_global(T* p) {
    return (GlobalAS<T>*)p;
}

// The tap tables SampledTaps and CosineTaps live in ss2_common.h.

// XYB constants of prepare.comp:40-54 rounded to FP32.
constexpr float kM00 = 0x1.333334p-2f, kM01 = 0x1.3e76c8p-1f, kM02 = 0x1.3f7ceep-4f;
constexpr float kM10 = 0x1.d70a3ep-3f, kM11 = 0x1.624dd2p-1f, kM12 = 0x1.3f7ceep-4f;
constexpr float kM20 = 0x1.f28798p-3f, kM21 = 0x1.a35d1ep-3f, kM22 = 0x1.1a86d2p-1f;
constexpr float kOpsinBias = 0x1.f12a6cp-9f;
constexpr float kCbrtBias = 0x1.3f64eap-3f;
constexpr float kC2 = 0.0009f;            // scale.comp:87

__device__ __forceinline__ float fma_(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
}

// fma(w, x, c) for a constant w into a register of its own: the compiler
// forms it in c's register and copies that away where c's name changes.
__device__ __forceinline__ float fma_move(float w, float x, float c) {
    float r;
    asm("v_fmamk_f32 %0, %1, %3, %2" : "=v"(r) : "v"(x), "v"(c), "i"(__builtin_bit_cast(int, w)));
    return r;
}

// Smallest normal float: the XYB mixes are clamped to it instead of 0, so the
// cube roots never see zero or a denormal. Its root, 2^-42, vanishes in every
// sum it enters (all are at least ~1e-2 away from it), as a zero root would:
// 2^-42 minus the cube-root bias rounds to minus the bias.
constexpr float kMinNormal = 0x1p-126f;

// 1 / x correctly rounded, for x a positive normal float in [2^-24, 2^24):
// the hardware reciprocal and one Newton step r += r (1 - x r), 3
// instructions. vqm_ss2_check_div checks it against the IEEE quotient for
// every significand and the hardware reciprocal's invariance under scaling
// by 2^e, e in [-24, 24) (the Newton step scales exactly).
__device__ __forceinline__ float rcp_rn(float x) {
    const float r = __builtin_amdgcn_rcpf(x);
    return fma_(fma_(-x, r, 1.0f), r, r);
}

// a / b correctly rounded (the IEEE quotient), for the map's quotients: b a
// positive normal float in [2^-24, 2^24) and a either 0.0f (never -0.0f) or
// |a| >= 2^-100, with |a / b| inside [2^-100, 2^100]. The hardware
// reciprocal, one Newton step (the reciprocal correctly rounded), the
// product, and one residual correction (Markstein's): 6 instructions, where
// the compiler's `a / b` takes 11 (two corrections, operand scaling and a
// special-value fix-up). vqm_ss2_check_div compares it with the IEEE
// quotient on the device: over every pair of significands (a, b in [1, 2),
// 2^46 pairs, about 30 s) it differs nowhere, and the hardware reciprocal of
// m 2^e is that of m scaled by 2^-e for every e in [-24, 24); the fused
// steps scale exactly, so the whole domain follows. The map's operands stay
// in it: denominators are at least c2 - 2^-22 or 1 and at most a few units,
// and numerators are 0.0f (an exact difference of equal values rounds to
// +0) or multiples of 2^-82.
__device__ __forceinline__ float div_rn(float a, float b) {
    const float r = rcp_rn(b);
    const float q = a * r;
    return fma_(fma_(-b, q, a), r, q);
}

// The two arithmetic forms of the path (MapForm):
//
//   Reference form (Ref = true): prepare.comp:81-98 and scale.comp:130-142,
//   305-333 in their own operation order. The cube roots are correctly
//   rounded (cube_roots), the five quantities a, b, a*a, b*b and a*b are
//   blurred, and the SSIM' map subtracts the squared means from the blurred
//   second moments directly, with IEEE divisions.
//
//   Difference form (Ref = false): the cube-root bias cancelled where it
//   cancels exactly, the fast cube root (cbrt_fast), and the SSIM' map from
//   four blurred quantities a, b, (a - b)^2 and a*b (see scale_item).
//
// XYB of one linear sample, only the channels in `mask` (bit 0 X, 1 Y, 2 B).
// With c_i = cbrt(m_i) - bias, the reference computes X = (0.5 (c0 - c1)) 14
// + 0.42, Y = 0.5 (c0 + c1) + 0.01 and B = (c2 - 0.5 (c0 + c1)) + 0.55. The
// difference form takes them from the roots directly:
// X = 7 (cbrt0 - cbrt1) + 0.42, Y = (cbrt0 + cbrt1)/2 + (0.01 - bias) and
// B = cbrt2 - (cbrt0 + cbrt1)/2 + 0.55 (three subtractions fewer, no
// rounding of c_i).
constexpr float kYOffset = 0.01f - kCbrtBias;  // rounded once


// The cube roots of K mixes, in place. The reference form takes every root's
// fast part first, so that the roots' instruction chains share a basic block
// and interleave, and settles the rare near-midpoint roots in one branch for
// all of them. Any: the mixes may be any positive normal float, else they lie
// in cbrt_rn_near_f32's range.
template <bool Ref, bool Any, int K>
__device__ __forceinline__ void cube_roots(float (&m)[K]) {
    if constexpr (!Ref) {
#pragma unroll
        for (int k = 0; k < K; ++k) m[k] = cbrt_fast(m[k]);
    } else {
        float c[K];
        bool unsettled[K], any = false;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            c[k] = cbrt_rn_near_f32(m[k], &unsettled[k]);
            if constexpr (Any) unsettled[k] |= __float_as_uint(m[k]) - kCbrtF32First >= kCbrtF32Count;
            any |= unsettled[k];
        }
        if (any) {
            // One copy of the exact root, the roots passing through it in
            // turn; those that no lane has to settle pass by it.
            uint32_t which = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) which |= (__builtin_amdgcn_ballot_w64(unsettled[k]) != 0u ? 1u : 0u) << k;
#pragma unroll 1
            for (int k = 0; k < K; ++k) {
                const float x = m[0];
                float y = c[0];
                if ((which >> k) & 1u) {
                    if constexpr (Any) {
                        bool n;
                        y = cbrt_rn_near_hw(x, &n);
                    }
                    y = cbrt_round_exact(x, y);
                }
#pragma unroll
                for (int i = 0; i + 1 < K; ++i) m[i] = m[i + 1], c[i] = c[i + 1];
                m[K - 1] = x;
                c[K - 1] = y;
            }
        }
#pragma unroll
        for (int k = 0; k < K; ++k) m[k] = c[k];
    }
}

// Roots taken together: those of two pixels. Measured at 92 registers: one 4K
// pair's prepare 38.5 us against 38.9 with four pixels' (94 registers, and
// their `unsettled` masks spill).
constexpr int kRootBatch = 4;

// N pixels (px[j] = linear r, g, b): put(channel, values) for the channels in
// `mask`. Clamp: the mixes may fall below the smallest normal float (samples
// decoded from a general format); table-decoded samples lie in [0, 1], whose
// mixes are at least the bias.
template <bool Ref, int N, bool Clamp, typename Put>
__device__ __forceinline__ void xyb_group(const float (*px)[3], uint32_t mask, Put&& put) {
    auto mix = [](const float* p, float k0, float k1, float k2) {
        const float m = fma_(k0, p[0], fma_(k1, p[1], fma_(k2, p[2], kOpsinBias)));
        return Clamp ? fmaxf(m, kMinNormal) : m;
    };
    float c[2 * N], v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
        c[2 * j] = mix(px[j], kM00, kM01, kM02);
        c[2 * j + 1] = mix(px[j], kM10, kM11, kM12);
    }
#pragma unroll
    for (int j = 0; j < 2 * N; j += kRootBatch) {
        float batch[kRootBatch < 2 * N ? kRootBatch : 2 * N];
        constexpr int n = sizeof(batch) / sizeof(float);
#pragma unroll
        for (int i = 0; i < n; ++i) batch[i] = c[j + i];
        cube_roots<Ref, Clamp>(batch);
#pragma unroll
        for (int i = 0; i < n; ++i) c[j + i] = batch[i];
    }
    if constexpr (Ref) {
#pragma unroll
        for (int j = 0; j < 2 * N; ++j) c[j] = c[j] - kCbrtBias;
    }
    if (mask & 1u) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            v[j] = Ref ? fma_(0.5f * (c[2 * j] - c[2 * j + 1]), 14.0f, 0.42f)
                       : fma_(c[2 * j] - c[2 * j + 1], 7.0f, 0.42f);
        put(0u, v);
    }
    if (mask & 2u) {
#pragma unroll
        for (int j = 0; j < N; ++j)
            v[j] = Ref ? 0.5f * (c[2 * j] + c[2 * j + 1]) + 0.01f : fma_(0.5f, c[2 * j] + c[2 * j + 1], kYOffset);
        put(1u, v);
    }
    if (mask & 4u) {
        float b[N];
#pragma unroll
        for (int j = 0; j < N; ++j) b[j] = mix(px[j], kM20, kM21, kM22);
        cube_roots<Ref, Clamp>(b);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float sum = c[2 * j] + c[2 * j + 1];
            v[j] = Ref ? (b[j] - kCbrtBias - 0.5f * sum) + 0.55f : fma_(-0.5f, sum, b[j]) + 0.55f;
        }
        put(2u, v);
    }
}

// ---- plane element formats ------------------------------------------------

// A format loads two adjacent elements as Raw bits (or one element) and
// unpacks them to FP32 only where they are consumed, so that the wait for a prefetched row lands
// one row later instead of right behind the load.
struct F32 {
    using E = float;
    using Raw4 = f32x4;
    static __device__ __forceinline__ Raw4 load4(GlobalAS<const E>* p) {
        return Raw4{p[0], p[1], p[2], p[3]};
    }
    static __device__ __forceinline__ void unpack4(Raw4 v, float out[4]) {
        for (int i = 0; i < 4; ++i) out[i] = v[i];
    }
    static __device__ __forceinline__ float load1(GlobalAS<const E>* p) { return *p; }
    static __device__ __forceinline__ void store1(GlobalAS<E>* p, float v) { *p = v; }
    static __device__ __forceinline__ void store2(GlobalAS<E>* p, float a, float b) {
        *reinterpret_cast<GlobalAS<f32x2>*>(p) = f32x2{a, b};
    }
    static __device__ __forceinline__ void store4(GlobalAS<E>* p, const float v[4]) {
        *reinterpret_cast<GlobalAS<f32x4>*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    }
};

// FP32 -> FP16, round to nearest even, written out in integer operations so
// that every value (ties included) rounds exactly as IEEE 754 specifies and
// as the oracle's restatement does.
__device__ __forceinline__ uint16_t to_f16(float v) {
    const uint32_t x = __float_as_uint(v);
    const uint32_t sign = (x >> 16) & 0x8000u;
    const uint32_t a = x & 0x7FFFFFFFu;
    if (a >= 0x477FF000u)  // rounds to infinity (65520 and up), or NaN
        return static_cast<uint16_t>(sign | (a > 0x7F800000u ? 0x7E00u : 0x7C00u));
    if (a < 0x38800000u)   // below 2^-14: a multiple of 2^-24, exact product
        return static_cast<uint16_t>(sign | static_cast<uint32_t>(__builtin_rintf(__uint_as_float(a) * 0x1p24f)));
    uint32_t r = a - 0x38000000u;  // rebias the exponent from 127 to 15
    r += 0xFFFu + ((r >> 13) & 1u);
    return static_cast<uint16_t>(sign | (r >> 13));
}
__device__ __forceinline__ float from_f16(uint16_t v) {
    return static_cast<float>(__builtin_bit_cast(_Float16, v));
}
__device__ __forceinline__ uint16_t to_bf16(float v) {
    uint32_t bits = __float_as_uint(v);
    bits += 0x7FFFu + ((bits >> 16) & 1u);
    return static_cast<uint16_t>(bits >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t v) {
    return __uint_as_float(static_cast<uint32_t>(v) << 16);
}

template <uint16_t (*To)(float), float (*From)(uint16_t)>
struct Narrow {
    using E = uint16_t;
    using Raw4 = u32x2;
    static __device__ __forceinline__ Raw4 load4(GlobalAS<const E>* p) {
        GlobalAS<const uint32_t>* w = reinterpret_cast<GlobalAS<const uint32_t>*>(p);
        return Raw4{w[0], w[1]};
    }
    static __device__ __forceinline__ void unpack4(Raw4 v, float out[4]) {
        for (int i = 0; i < 2; ++i) {
            out[2 * i] = From(static_cast<uint16_t>(v[i] & 0xFFFFu));
            out[2 * i + 1] = From(static_cast<uint16_t>(v[i] >> 16));
        }
    }
    static __device__ __forceinline__ float load1(GlobalAS<const E>* p) { return From(*p); }
    static __device__ __forceinline__ void store1(GlobalAS<E>* p, float v) { *p = To(v); }
    static __device__ __forceinline__ void store2(GlobalAS<E>* p, float a, float b) {
        *reinterpret_cast<GlobalAS<uint32_t>*>(p) =
            static_cast<uint32_t>(To(a)) | (static_cast<uint32_t>(To(b)) << 16);
    }
    static __device__ __forceinline__ void store4(GlobalAS<E>* p, const float v[4]) {
        *reinterpret_cast<GlobalAS<u32x2>*>(p) =
            u32x2{static_cast<uint32_t>(To(v[0])) | (static_cast<uint32_t>(To(v[1])) << 16),
                  static_cast<uint32_t>(To(v[2])) | (static_cast<uint32_t>(To(v[3])) << 16)};
    }
};
// FP32 -> unsigned 16-bit fixed point q / 65536, round to nearest even,
// clamped to 0 .. 65535 (NaN and negatives to 0). The XYB values of linear
// RGB in [0, 1] lie in [0, 0.94]: the step is a uniform 2^-16 and zero, the
// plane borders' value, is exact. Scaling by 2^16 and back is exact.
__device__ __forceinline__ uint16_t to_unorm16(float v) {
    const float s = fminf(fmaxf(v * 65536.0f, 0.0f), 65535.0f);
    return static_cast<uint16_t>(__builtin_rintf(s));
}
__device__ __forceinline__ float from_unorm16(uint16_t v) {
    return static_cast<float>(v) * (1.0f / 65536.0f);
}

using F16 = Narrow<to_f16, from_f16>;
using BF16 = Narrow<to_bf16, from_bf16>;
using U16 = Narrow<to_unorm16, from_unorm16>;

// The element format of every stored plane, and RoundLinear: the linear box
// averages of levels >= 1 are rounded to the element format too, before
// their XYB and before the next level averages them -- the reference's
// half-plane build (prepare.comp:100-111, ssimu2_common.glsl:84-96), which
// FP16 planes reproduce.
template <typename FmtT, bool RoundLinear = false>
struct Layout {
    using Fmt = FmtT;
    static constexpr bool kRoundLinear = RoundLinear;
};
using LayoutF32 = Layout<F32>;
using LayoutF16 = Layout<F16, true>;
using LayoutBF16 = Layout<BF16>;
using LayoutU16 = Layout<U16>;

// A level's linear box average as the layout hands it on.
template <typename Lay>
__device__ __forceinline__ float linear_sample(float v) {
    if constexpr (Lay::kRoundLinear) {
        return from_f16(to_f16(v));
    } else {
        return v;
    }
}

// Element pointer of a plane: planes of one image start at `base` and
// `offset` is in bytes.
template <typename Fmt>
__device__ __forceinline__ GlobalAS<typename Fmt::E>* plane_at(GlobalAS<uint8_t>* base, uint64_t offset) {
    return reinterpret_cast<GlobalAS<typename Fmt::E>*>(base + offset);
}

// Workgroup b runs on XCD b % 8. Renumber so each XCD receives a contiguous
// run of logical work items: neighbouring strips and tiles, which share halo
// rows and input cache lines, then share one L2.
__device__ __forceinline__ uint32_t xcd_remap(uint32_t b, uint32_t n) {
    constexpr uint32_t kXcds = 8;
    const uint32_t xcd = b % kXcds, idx = b / kXcds;
    const uint32_t per = n / kXcds, rem = n % kXcds;
    return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// Four bytes at any alignment.
struct __attribute__((packed, aligned(1))) Bytes4 {
    uint32_t v;
};

// ---- general input decode -----------------------------------------------------
//
// Images that are not 8-bit sRGB RGB are decoded per pixel from their
// SourceDesc, in the stage order of color.glsl:447-541: raw sample with the
// range/depth scale and offset, chroma upsampling, the matrix (or the
// constant-luminance or ICtCp op), alpha, the transfer curve, and the
// primaries matrix to linear BT.709. Powers and exponentials go through the
// hardware base-2 logarithm and exponential (as a shader's pow does), and
// the stages are held to the A/B tolerances of the input tests, not bit
// parity.

namespace decode {

// x^y for x >= 0 from v_log_f32 and v_exp_f32 (about one ulp each): relative
// error about |y log2 x| 2^-23 plus one ulp, some 150 instructions fewer than
// the library powf. Inputs below the smallest normal float are taken as it
// (their powers are 0 to FP32 precision for y >= 1; the curves with y < 1
// map them to 0 after their own offsets).
__device__ __forceinline__ float pow_hw(float x, float y) {
    const float power = __builtin_amdgcn_exp2f(y * __builtin_amdgcn_logf(fmaxf(x, 0x1p-126f)));
    return x <= 0.0f ? 0.0f : power;  // no branch: the powers of several samples interleave
}
// e^x and 10^x through v_exp_f32.
__device__ __forceinline__ float exp_hw(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
__device__ __forceinline__ float exp10_hw(float x) { return __builtin_amdgcn_exp2f(x * 3.32192809488736235f); }

constexpr float kRec709Alpha = 1.09929682680944f;
constexpr float kRec709Beta = 0.018053968510807f;

__device__ float raw_sample(ConstAS<SourceDesc>* d, GlobalAS<const uint8_t>* src, uint32_t plane,
                            uint32_t x, uint32_t y) {
    const uint64_t index = static_cast<uint64_t>(y) * d->plane_w[plane] + x;
    GlobalAS<const uint8_t>* base = src + d->plane_off[plane];
    float v;
    switch (d->type) {
        case 0: v = static_cast<float>(base[index]); break;
        case 1: v = static_cast<float>(reinterpret_cast<GlobalAS<const uint16_t>*>(base)[index]); break;
        case 2: v = static_cast<float>(reinterpret_cast<GlobalAS<const _Float16>*>(base)[index]); break;
        default: v = reinterpret_cast<GlobalAS<const float>*>(base)[index]; break;
    }
    // Sample class: 2 alpha, 1 the chroma planes of YUV, 0 luma or RGB.
    const uint32_t cls = plane == 3 ? 2u : (plane != 0 && d->family == 2 ? 1u : 0u);
    return v * d->scale[cls] + d->offset[cls];
}

// BT.709 inverse OETF (the CL op and the xvYCC / BT.1361 extensions).
__device__ float rec709_inverse_oetf(float x) {
    x = fmaxf(x, 0.0f);
    return x < 4.5f * kRec709Beta ? x / 4.5f
                                  : pow_hw((x + (kRec709Alpha - 1.0f)) / kRec709Alpha, 1.0f / 0.45f);
}

// IEC 61966-2-1.
__device__ float srgb_eotf(float v) {
    return v <= 0.04045f ? v / 12.92f : pow_hw((v + 0.055f) / 1.055f, 2.4f);
}

// SMPTE ST 2084, normalised to 10000 cd/m^2, of each of N samples, times
// `scale`.
// A sample at a time, with a branch for zero and one for the division each,
// the samples' chains of transcendentals could not interleave: 4K 10-bit 4:2:0
// prepared in 136.5 us; in 123.0 with six samples together, 121.4 with a
// pixel's three.
template <int N>
__device__ __forceinline__ void pq_eotf(float scale, float (&v)[N]) {
    float num[N], den[N], q[N];
    bool past = false;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float p = pow_hw(v[i], 1.0f / 78.84375f);
        num[i] = fmaxf(p - 0.8359375f, 0.0f);
        den[i] = fmaxf(18.8515625f - 18.6875f * p, 1.17549435e-38f);
        // num is 0 or at least 2^-26 and den, but for samples far past the
        // curve's range, at least 2^-3: inside div_rn's domain, whose quotient
        // is the IEEE one.
        q[i] = div_rn(num[i], den[i]);
        past |= den[i] < 0x1p-20f;
    }
    if (past) {
#pragma unroll 1
        for (int k = 0; k < N; ++k) {  // one copy of the division, the samples passing through it
            const float n = num[0], d = den[0], exact = d < 0x1p-20f ? n / d : q[0];
#pragma unroll
            for (int i = 0; i + 1 < N; ++i) num[i] = num[i + 1], den[i] = den[i + 1], q[i] = q[i + 1];
            num[N - 1] = n;
            den[N - 1] = d;
            q[N - 1] = exact;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float y = pow_hw(q[i], 1.0f / 0.1593017578125f);
        v[i] = scale * (v[i] <= 0.0f ? 0.0f : y);
    }
}

// ARIB STD-B67 inverse OETF (scene light).
__device__ float hlg_inverse_oetf(float x) {
    x = fmaxf(x, 0.0f);
    return x <= 0.5f ? (x * x) * (1.0f / 3.0f) : (exp_hw((x - 0.55991073f) / 0.17883277f) + 0.28466892f) / 12.0f;
}

// The decode curve `id` of every sample of four pixels: one branch for the
// twelve, so that their chains interleave.
__device__ __forceinline__ void curves(uint32_t id, float scale, float3 (&px)[4]) {
    auto each = [&](auto&& f) {
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j] = make_float3(f(px[j].x), f(px[j].y), f(px[j].z));
    };
    auto power = [&](float y) { each([y](float v) { return pow_hw(v, y); }); };
    switch (id) {
        case kCurvePow24: power(2.4f); break;
        case kCurvePow22: power(2.2f); break;
        case kCurvePow28: power(2.8f); break;
        case kCurveSrgb: each([](float v) { return srgb_eotf(v); }); break;
        case kCurveLog100: each([](float v) { return v <= 0.0f ? 0.01f : exp10_hw(2.0f * (v - 1.0f)); }); break;
        case kCurveLog316: each([](float v) { return v <= 0.0f ? 0.00316227766f : exp10_hw(2.5f * (v - 1.0f)); }); break;
        case kCurveXvycc:
            each([](float v) {
                if (v >= 0.0f && v <= 1.0f) return pow_hw(v, 2.4f);
                return v < 0.0f ? -rec709_inverse_oetf(-v) : rec709_inverse_oetf(v);
            });
            break;
        case kCurveBt1361:
            each([](float v) {
                if (v >= 0.0f && v <= 1.0f) return pow_hw(v, 2.4f);
                return v >= 0.0f ? rec709_inverse_oetf(v) : -rec709_inverse_oetf(-4.0f * v) / 4.0f;
            });
            break;
        case kCurvePq:
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float v[3] = {px[j].x, px[j].y, px[j].z};
                pq_eotf(scale, v);
                px[j] = make_float3(v[0], v[1], v[2]);
            }
            break;
        case kCurveSt428: each([](float v) { return v < 0.0f ? 0.0f : (52.37f / 48.0f) * pow_hw(v, 2.6f); }); break;
        default: break;
    }
}

__device__ float3 apply(ConstAS<float>* m, float3 v) {
    return make_float3(m[0] * v.x + m[1] * v.y + m[2] * v.z, m[3] * v.x + m[4] * v.y + m[5] * v.z,
                       m[6] * v.x + m[7] * v.y + m[8] * v.z);
}

// Constant-luminance Y'CbCr to linear RGB through the BT.709 curve.
__device__ float3 cl_to_rgb(ConstAS<SourceDesc>* d, float3 e) {
    const float u = e.y, v = e.z;
    const float b_minus_y = u * 2.0f * (u < 0.0f ? d->cl[0] : d->cl[1]);
    const float r_minus_y = v * 2.0f * (v < 0.0f ? d->cl[2] : d->cl[3]);
    const float b = rec709_inverse_oetf(b_minus_y + e.x);
    const float r = rec709_inverse_oetf(r_minus_y + e.x);
    const float luma = rec709_inverse_oetf(e.x);
    return make_float3(r, (luma - d->kr * r - d->kb * b) / d->kg, b);
}

// Resampling kernels: triangle, Catmull-Rom (B = 0, C = 0.5), Lanczos-3.
__device__ float sinc(float x) {
    const float pix = 3.14159265358979323846f * x;
    return x == 0.0f ? 1.0f : sinf(pix) / pix;
}
__device__ float filter_weight(uint32_t filter, float x) {
    x = fabsf(x);
    if (filter == 0) return fmaxf(1.0f - x, 0.0f);
    if (filter == 1) {
        if (x < 1.0f) return 1.0f + x * x * (-2.5f + x * 1.5f);
        if (x < 2.0f) return 2.0f + x * (-4.0f + x * (2.5f - 0.5f * x));
        return 0.0f;
    }
    return x < 3.0f ? sinc(x) * sinc(x / 3.0f) : 0.0f;
}

// Rounds half up such that round(x - 1) == round(x) - 1.
__device__ float round_halfup(float x) { return x < 0.0f ? floorf(x + 0.5f) : floorf(x + 0.49999997f); }

// A tap position mirrored once at the plane edges, then clamped.
__device__ uint32_t mirror(float pos, uint32_t dim) {
    const float extent = static_cast<float>(dim);
    const float m = pos < 0.0f ? -pos : (pos >= extent ? 2.0f * extent - pos : pos);
    return static_cast<uint32_t>(fminf(fmaxf(m, 0.0f), extent - 1.0f));
}

constexpr int kMaxTaps = 6;

__device__ __forceinline__ int tap_count(uint32_t filter) { return filter == 0 ? 2 : filter == 1 ? 4 : 6; }

// Chroma position of output sample `out` on one axis: (out + 0.5) / ratio
// + shift.
__device__ __forceinline__ float chroma_pos(uint32_t out, uint32_t sub, float shift) {
    return (static_cast<float>(out) + 0.5f) * __builtin_ldexpf(1.0f, -static_cast<int>(sub)) + shift;
}

// The first tap's sample index before mirroring, round(pos - taps / 2): an
// integer-valued float, non-decreasing in pos.
__device__ __forceinline__ float first_tap(int taps, float pos) {
    return round_halfup(pos - 0.5f * static_cast<float>(taps));
}

// The weights of one axis for output sample `out`, taps centred half a
// sample past the first tap. Bilinear weights are 1 - t and t (their sum is
// exactly one); the others are normalised by their sum. Returns the tap
// count; *first is the first tap's unmirrored index. Bilinear (filter 0)
// callers set Bilinear, so the tap loops unroll and the weights stay in
// registers.
template <bool Bilinear>
__device__ __forceinline__ int axis_weights(uint32_t filter, uint32_t out, uint32_t sub, float shift,
                                            float (&w)[Bilinear ? 2 : kMaxTaps], int* first) {
    const int taps = Bilinear ? 2 : tap_count(filter);
    const float pos = chroma_pos(out, sub, shift);
    const float n0 = first_tap(taps, pos);
    const float base = n0 + 0.5f;
    if (Bilinear || filter == 0) {
        const float t = pos - base;
        w[0] = 1.0f - t;
        w[1] = t;
    } else {
        float total = 0.0f;
        for (int j = 0; j < taps; ++j) total += filter_weight(filter, base + static_cast<float>(j) - pos);
        for (int j = 0; j < taps; ++j) w[j] = filter_weight(filter, base + static_cast<float>(j) - pos) / total;
    }
    *first = static_cast<int>(n0);
    return taps;
}

// Sample index of unmirrored tap index n: the tap's centre n + 0.5 mirrored
// once at the plane edges, then clamped.
__device__ __forceinline__ uint32_t tap_index(int n, uint32_t dim) {
    return mirror(static_cast<float>(n) + 0.5f, dim);
}

// The chroma samples a tile's pixels read, staged in LDS: both chroma planes
// (scaled and offset) interleaved as (U, V), rows of `cols` entries from
// unmirrored tap index (x0, y0). Over every subsampling (1x, 2x, 4x per
// axis), siting and filter, a 64 x 32 tile needs at most 69 x 22 = 1518
// entries (Lanczos-3, 2x vertical subsampling only); the bound was found by
// enumerating tile positions on frames up to 3840 x 2160.
constexpr uint32_t kChromaWindow = 1664;
struct ChromaWindow {
    int x0, y0;
    uint32_t cols, rows;
};

// The window of pixels x_first .. x_last by y_first .. y_last; false if it
// does not fit in kChromaWindow entries.
__device__ bool chroma_window(ConstAS<SourceDesc>* d, uint32_t x_first, uint32_t x_last, uint32_t y_first,
                              uint32_t y_last, ChromaWindow* w) {
    const int taps = tap_count(d->filter);
    const int x0 = static_cast<int>(first_tap(taps, chroma_pos(x_first, d->sub_w, d->shift_x)));
    const int x1 = static_cast<int>(first_tap(taps, chroma_pos(x_last, d->sub_w, d->shift_x)));
    const int y0 = static_cast<int>(first_tap(taps, chroma_pos(y_first, d->sub_h, d->shift_y)));
    const int y1 = static_cast<int>(first_tap(taps, chroma_pos(y_last, d->sub_h, d->shift_y)));
    w->x0 = x0;
    w->y0 = y0;
    w->cols = static_cast<uint32_t>(x1 - x0 + taps);
    w->rows = static_cast<uint32_t>(y1 - y0 + taps);
    return w->cols * w->rows <= kChromaWindow;
}

// Block-wide: thread `tid` of `threads` loads every threads-th entry of the
// window.
__device__ void stage_chroma(ConstAS<SourceDesc>* d, GlobalAS<const uint8_t>* src, const ChromaWindow& w,
                             uint32_t tid, uint32_t threads, float2* window) {
    const uint32_t n = w.cols * w.rows;
    for (uint32_t i = tid; i < n; i += threads) {
        const uint32_t r = i / w.cols, c = i - r * w.cols;
        const uint32_t ix = tap_index(w.x0 + static_cast<int>(c), d->plane_w[1]);
        const uint32_t iy = tap_index(w.y0 + static_cast<int>(r), d->plane_h[1]);
        window[i] = make_float2(raw_sample(d, src, 1, ix, iy), raw_sample(d, src, 2, ix, iy));
    }
}

// The weights of a tile's columns and rows (Rows of them), staged in LDS for the
// filters of more than two taps. Formed for each pixel (24 sines a pixel for
// Lanczos-3) a 4K 4:2:0 pair took 1,183 us with Lanczos-3 and 500 with
// Catmull-Rom, now 503 and 344, a 1080p pair 367 and 176, now 184 and 135; and
// the registers of the sums spilled six values of the four-row form, in all
// formats (4K 8-bit bilinear 97.1 us of prepare, now 93.0).
template <uint32_t Rows>
struct ChromaWeights {
    float x[kPrepTileW][kMaxTaps], y[Rows][kMaxTaps];
};

// Block-wide, as stage_chroma: thread `tid` forms every threads-th column or
// row from pixel (x0, y0).
template <uint32_t Rows>
__device__ void stage_weights(ConstAS<SourceDesc>* d, uint32_t x0, uint32_t y0, uint32_t tid, uint32_t threads,
                              ChromaWeights<Rows>& weights) {
    for (uint32_t i = tid; i < kPrepTileW + Rows; i += threads) {
        const bool column = i < kPrepTileW;
        const uint32_t at = column ? i : i - kPrepTileW;
        float w[kMaxTaps] = {};
        int first;
        axis_weights<false>(d->filter, (column ? x0 : y0) + at, column ? d->sub_w : d->sub_h,
                            column ? d->shift_x : d->shift_y, w, &first);
        float* const out = column ? weights.x[at] : weights.y[at];
#pragma unroll
        for (int j = 0; j < kMaxTaps; ++j) out[j] = w[j];
    }
}

// Both chroma samples of pixel (x, y): the two chroma planes share their
// size and siting, so one set of taps serves both. Rows are summed first,
// then weighted by the vertical taps. With a staged window the samples come
// from LDS (the same values, in the same order), else from the planes.
// Bilinear: the descriptor's filter is 0; else staged_x and staged_y are the
// staged weights of x and y.
template <bool Bilinear>
__device__ __forceinline__ float2 chroma_samples(ConstAS<SourceDesc>* d, GlobalAS<const uint8_t>* src,
                                                 const float2* window, const ChromaWindow& cw, uint32_t x, uint32_t y,
                                                 const float* staged_x, const float* staged_y) {
    float wx[Bilinear ? 2 : kMaxTaps], wy[Bilinear ? 2 : kMaxTaps];
    int fx, fy, tx, ty;
    if constexpr (Bilinear) {
        tx = axis_weights<true>(0u, x, d->sub_w, d->shift_x, wx, &fx);
        ty = axis_weights<true>(0u, y, d->sub_h, d->shift_y, wy, &fy);
    } else {
        tx = ty = tap_count(d->filter);
        fx = static_cast<int>(first_tap(tx, chroma_pos(x, d->sub_w, d->shift_x)));
        fy = static_cast<int>(first_tap(ty, chroma_pos(y, d->sub_h, d->shift_y)));
#pragma unroll
        for (int k = 0; k < kMaxTaps; ++k) wx[k] = staged_x[k], wy[k] = staged_y[k];
    }
    float sum_u = 0.0f, sum_v = 0.0f;
    if (window != nullptr) {
        // The first taps are non-decreasing in x and y, so they lie within
        // the window; the clamp only guards the LDS bounds.
        const uint32_t cx = min(static_cast<uint32_t>(fx - cw.x0), cw.cols - static_cast<uint32_t>(tx));
        const uint32_t cy = min(static_cast<uint32_t>(fy - cw.y0), cw.rows - static_cast<uint32_t>(ty));
        for (int j = 0; j < ty; ++j) {
            const float2* row = window + (cy + static_cast<uint32_t>(j)) * cw.cols + cx;
            float row_u = 0.0f, row_v = 0.0f;
            for (int k = 0; k < tx; ++k) {
                const float2 s = row[k];
                row_u += wx[k] * s.x;
                row_v += wx[k] * s.y;
            }
            sum_u += wy[j] * row_u;
            sum_v += wy[j] * row_v;
        }
    } else {
        for (int j = 0; j < ty; ++j) {
            const uint32_t iy = tap_index(fy + j, d->plane_h[1]);
            float row_u = 0.0f, row_v = 0.0f;
            for (int k = 0; k < tx; ++k) {
                const uint32_t ix = tap_index(fx + k, d->plane_w[1]);
                row_u += wx[k] * raw_sample(d, src, 1, ix, iy);
                row_v += wx[k] * raw_sample(d, src, 2, ix, iy);
            }
            sum_u += wy[j] * row_u;
            sum_v += wy[j] * row_v;
        }
    }
    return make_float2(sum_u, sum_v);
}

// A full-size plane's samples of a lane's four pixels of row y (the columns
// col[], 0 .. 3 on from bx but for clamped ones): one 4- or 8-byte load (at
// any alignment) for byte and word samples inside the row, else one load a
// pixel.
__device__ __forceinline__ void plane4(ConstAS<SourceDesc>* d, GlobalAS<const uint8_t>* src, uint32_t plane,
                                       uint32_t bx, const uint32_t (&col)[4], uint32_t y, uint32_t W, float (&out)[4]) {
    const uint32_t pw = d->plane_w[plane];
    if (d->type <= 1u && bx + 3u < W) {
        const uint64_t index = static_cast<uint64_t>(y) * pw + bx;
        GlobalAS<const uint8_t>* base = src + d->plane_off[plane];
        const uint32_t cls = plane != 0u && d->family == 2u ? 1u : 0u;
        const float scale = d->scale[cls], offset = d->offset[cls];
        if (d->type == 0u) {
            const uint32_t w = reinterpret_cast<GlobalAS<const Bytes4>*>(base + index)->v;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) out[j] = static_cast<float>((w >> (8u * j)) & 255u) * scale + offset;
        } else {
            GlobalAS<const Bytes4>* words = reinterpret_cast<GlobalAS<const Bytes4>*>(base + 2u * index);
            const uint32_t w0 = words[0].v, w1 = words[1].v;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t word = (j < 2u ? w0 : w1) >> (16u * (j & 1u));
                out[j] = static_cast<float>(word & 0xFFFFu) * scale + offset;
            }
        }
    } else {
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) out[j] = raw_sample(d, src, plane, col[j], y);
    }
}

// The columns of a lane's four pixels in the staged window, bilinear: the right
// tap's weight (the left's is one less it) and the left tap's entry in a row.
// They are the same in all four rows; formed again for each, a 1080p 8-bit
// 4:2:0 pair prepared in 33.9 us, without that in 32.7.
struct BilinearColumns {
    float t[4];
    uint32_t at[4];
};
__device__ __forceinline__ BilinearColumns bilinear_columns(ConstAS<SourceDesc>* d, const ChromaWindow& cw,
                                                            const uint32_t (&col)[4]) {
    BilinearColumns c;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float wx[2];
        int fx;
        axis_weights<true>(0u, col[j], d->sub_w, d->shift_x, wx, &fx);
        c.t[j] = wx[1];
        // The first taps are non-decreasing in x and y, so they lie within
        // the window; the clamps only guard the LDS bounds.
        c.at[j] = min(static_cast<uint32_t>(fx - cw.x0), cw.cols - 2u);
    }
    return c;
}

// Both chroma samples of four pixels of row y from the staged window,
// bilinear.
__device__ __forceinline__ void bilinear4(ConstAS<SourceDesc>* d, const float2* window, const ChromaWindow& cw,
                                          const BilinearColumns& columns, uint32_t y, float3 (&e)[4]) {
    float wy[2];
    int fy;
    axis_weights<true>(0u, y, d->sub_h, d->shift_y, wy, &fy);
    const uint32_t cy = min(static_cast<uint32_t>(fy - cw.y0), cw.rows - 2u);
    const float2* const row0 = window + cy * cw.cols;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float w0 = 1.0f - columns.t[j], w1 = columns.t[j];
        const float2* const s0 = row0 + columns.at[j];
        const float2* const s1 = s0 + cw.cols;
        const float2 a = s0[0], b = s0[1], c = s1[0], f = s1[1];
        e[j].y = wy[0] * (w0 * a.x + w1 * b.x) + wy[1] * (w0 * c.x + w1 * f.x);
        e[j].z = wy[0] * (w0 * a.y + w1 * b.y) + wy[1] * (w0 * c.y + w1 * f.y);
    }
}

// Linear BT.709 RGB of a lane's four pixels of row y, each stage over the
// four, so that its branches are taken and its descriptor fields read once
// (a pixel at a time took 18 scalar loads and 123 scalar instructions each).
// Prepare of one pair: 1080p 8-bit 4:2:0 49.7 -> 36.0 us, 4K 10-bit PQ 4:2:0
// 170 -> 149 us. What bounds it now is waiting with four waves a SIMD: they wait
// in 53% of their cycles at 1080p (8-bit), whose 4,080 waves are all resident at
// once, in 45% at 4K and 40% there in PQ, and issue 0.56, 0.80 and 0.85 vector
// instructions a CU-cycle of 1.78; a wave makes some 130 scalar loads and 900
// scalar instructions. Loading the luma of all four rows ahead of the chroma
// gave nothing (and spilled), leaving out every stage that these formats pass by
// 4 us of 123.
// `window` is the tile's staged chroma, or null to read the chroma planes
// directly; `weights` the staged ones of the tile from pixel (X0, Y0).
template <uint32_t Rows>
__device__ __forceinline__ void row4(ConstAS<SourceDesc>* d, GlobalAS<const uint8_t>* src, const float2* window,
                                     const ChromaWindow& cw, const BilinearColumns& columns,
                                     const ChromaWeights<Rows>& weights, uint32_t X0, uint32_t Y0, uint32_t bx,
                                     const uint32_t (&col)[4], uint32_t y, uint32_t W, float (&lin)[4][3]) {
    float3 px[4];
    {
        float first[4];
        plane4(d, src, 0, bx, col, y, W, first);
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j] = make_float3(first[j], first[j], first[j]);
    }
    const uint32_t family = d->family;
    if (family == 2 && (d->sub_w != 0 || d->sub_h != 0)) {
        if (d->filter == 0 && window != nullptr) {
            bilinear4(d, window, cw, columns, y, px);
        } else {
#pragma unroll 1
            for (int k = 0; k < 4; ++k) {
                // One copy of the code, the pixels passing through it in turn.
                const uint32_t x = k == 0 ? col[0] : k == 1 ? col[1] : k == 2 ? col[2] : col[3];
                const float2 uv =
                    d->filter == 0 ? chroma_samples<true>(d, src, window, cw, x, y, nullptr, nullptr)
                                   : chroma_samples<false>(d, src, window, cw, x, y, weights.x[x - X0], weights.y[y - Y0]);
                const float3 p = make_float3(px[0].x, uv.x, uv.y);
                px[0] = px[1];
                px[1] = px[2];
                px[2] = px[3];
                px[3] = p;
            }
        }
    } else if (family != 0) {
        float u[4], v[4];
        plane4(d, src, 1, bx, col, y, W, u);
        plane4(d, src, 2, bx, col, y, W, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j].y = u[j], px[j].z = v[j];
    }
    const uint32_t mode = d->mode;
    if (mode == 1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j] = cl_to_rgb(d, px[j]);
    } else if (!d->identity1) {
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j] = apply(d->m1, px[j]);
    }
    if (d->alpha != 0) {
        const bool premultiplied = d->alpha == 2;
        const float background = d->background;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float alpha = raw_sample(d, src, 3, col[j], y);
            if (premultiplied) {
                const float a = fminf(fmaxf(alpha, 0.0f), 1.0f);
                px[j] = a == 0.0f ? make_float3(0.0f, 0.0f, 0.0f) : make_float3(px[j].x / a, px[j].y / a, px[j].z / a);
            }
            const float target = (1.0f - alpha) * background;
            px[j] = make_float3(alpha * px[j].x + target, alpha * px[j].y + target, alpha * px[j].z + target);
        }
    }
    if (mode != 1) {
        if (d->transfer == kCurveHlg) {
            // Per-channel inverse OETF, then the luminance OOTF and the peak.
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float3 c = make_float3(hlg_inverse_oetf(px[j].x), hlg_inverse_oetf(px[j].y), hlg_inverse_oetf(px[j].z));
                const float luma = fmaxf(d->kr * c.x + d->kg * c.y + d->kb * c.z, 1.17549435e-38f);
                const float k = pow_hw(luma, 0.2f) * d->to_linear_scale;
                px[j] = make_float3(c.x * k, c.y * k, c.z * k);
            }
        } else {
            curves(d->transfer, d->to_linear_scale, px);
        }
    }
    if (!d->identity2) {
#pragma unroll
        for (int j = 0; j < 4; ++j) px[j] = apply(d->m2, px[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        lin[j][0] = px[j].x;
        lin[j][1] = px[j].y;
        lin[j][2] = px[j].z;
    }
}

}  // namespace decode

// ---- prepare ----------------------------------------------------------------

// Orders a wave's LDS accesses: the wave's own are executed in order by the
// hardware, so only the compiler has to keep them apart.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Tile l's image, pair and origin (the launch's work list, or the arithmetic
// order of a uniform batch).
struct TileRef {
    ConstAS<PairDesc>* pdp;
    ConstAS<Plan>* plan;
    uint32_t image, X0, Y0;
};

__device__ __forceinline__ TileRef resolve_tile(uint32_t l, const PairDesc* __restrict__ pairs,
                                                const WorkRef* __restrict__ work, uint32_t tiles_per_image) {
    uint32_t pair_idx, image, tile;
    if (work != nullptr) {
        ConstAS<WorkRef>* w = as_const(work) + l;
        pair_idx = w->pair;
        image = w->index >> 31;
        tile = w->index & 0x7FFFFFFFu;
    } else {
        // One division: l = (pair * 2 + image) * tiles_per_image + tile.
        const uint32_t q = l / tiles_per_image;
        tile = l - q * tiles_per_image;
        image = q & 1u;
        pair_idx = q >> 1;
    }
    TileRef t;
    t.pdp = as_const(pairs) + pair_idx;
    t.plan = as_const(t.pdp->plan);
    t.image = image;
    const uint32_t tiles_x = t.plan->prep_tiles_x;
    const uint32_t ty = tile / tiles_x;
    t.X0 = (tile - ty * tiles_x) * kPrepTileW;
    t.Y0 = ty * kPrepTileH;
    return t;
}

// A wave's share of a 64 x 32 tile is its upper or lower 16 rows; a lane has
// 4 x 4 base pixels of them, and with them four samples of level 1 and one of
// level 2.
constexpr uint32_t kWaveRows = 16;
// Waves of a block: one in the table decode, which needs nothing of the other
// half (and whose LDS addresses are then constants); both in the general
// decode, which shares the tile's chroma window.
template <bool General> constexpr uint32_t kPrepWaves = General ? kPrepTileH / kWaveRows : 1u;

// The 8-bit table path's source bytes of this lane's 4 x 4 pixels: one 32-bit
// word per row and channel, when the row segments are whole (valid).
struct TileWords {
    uint32_t w[4][3];
    bool valid;
};

// Entry `byte J of w` of a table of floats: the byte times four in one
// instruction (the compiler takes two).
template <int J>
__device__ __forceinline__ float table_at(const float* table, uint32_t w) {
    uint32_t offset;
    const uint32_t two = 2u;
    if constexpr (J == 0) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_0" : "=v"(offset) : "v"(two), "v"(w));
    if constexpr (J == 1) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_1" : "=v"(offset) : "v"(two), "v"(w));
    if constexpr (J == 2) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_2" : "=v"(offset) : "v"(two), "v"(w));
    if constexpr (J == 3) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:BYTE_3" : "=v"(offset) : "v"(two), "v"(w));
    return *reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(table) + offset);
}

template <typename Row>
__device__ __forceinline__ TileWords load_tile_words(GlobalAS<const uint8_t>* src, uint64_t plane_stride, uint32_t W,
                                                     uint32_t bx, Row&& row) {
    TileWords out;
    out.valid = bx + 3u < W;
    if (!out.valid) return out;
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
        const uint64_t at = static_cast<uint64_t>(row(r)) * W + bx;
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c)
            out.w[r][c] = reinterpret_cast<GlobalAS<const Bytes4>*>(src + c * plane_stride + at)->v;
    }
    return out;
}

// One wave's LDS: its decode table (filled and read without a barrier), the
// linear samples of levels 2 (16 x 4) and 3 (8 x 2) and the cube roots of
// levels 3 and 4.
struct PrepareLds {
    float lut[256];
    float level2[3][64];
    float level3[3][16];
    float roots[64];
};

// The 2x2 box of column pair 2 i and rows row0, row1 of a wave's level of
// `side` columns, in (0,0), (1,0), (0,1), (1,1) order, the right column
// clamped onto the left one at odd widths (prepare.comp:146-168).
template <typename Lay>
__device__ __forceinline__ float box(const float* level, uint32_t side, uint32_t i, uint32_t row0, uint32_t row1,
                                     bool clamp_x) {
    const float2 top = *reinterpret_cast<const float2*>(level + row0 * side + 2u * i);
    const float2 bottom = *reinterpret_cast<const float2*>(level + row1 * side + 2u * i);
    float s = top.x;
    s = s + (clamp_x ? top.x : top.y);
    s = s + bottom.x;
    s = s + (clamp_x ? bottom.x : bottom.y);
    return linear_sample<Lay>(s * 0.25f);
}

// Levels 3 and 4 of a wave's 64 x 16 pixels: 8 x 2 and 4 x 1 samples, a lane
// per sample and channel (lanes 16 k + sample for channel k of level 3, 48 +
// 4 k + sample for level 4), so that one pass takes all their cube roots.
template <typename Lay, bool Ref, bool Clamp>
__device__ __forceinline__ void prepare_coarse(ConstAS<Plan>* plan, GlobalAS<uint8_t>* planes, uint32_t X0,
                                               uint32_t Y0, uint32_t lane, PrepareLds& lds) {
    using Fmt = typename Lay::Fmt;
    const uint32_t levels = plan->levels;
    const bool coarse = lane >= 48u;
    const uint32_t k = coarse ? (lane - 48u) / 4u : lane / 16u;  // 3: idle
    const uint32_t i = coarse ? lane % 4u : lane % 8u, j = coarse ? 0u : lane / 8u % 2u;
    float v[3] = {0.0f, 0.0f, 0.0f};
    // Level 3, whose samples level 4 needs.
    uint32_t gx = (X0 >> 3) + i, gy = (Y0 >> 3) + j;
    bool inside = !coarse && gx < plan->w[3] && gy < plan->h[3];
    if (!coarse) {
        const bool clamp_x = 2u * gx + 1u >= plan->w[2], clamp_y = 2u * gy + 1u >= plan->h[2];
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) v[c] = box<Lay>(lds.level2[c], 16u, i, 2u * j, 2u * j + (clamp_y ? 0u : 1u), clamp_x);
        if (lane < 16u) {
#pragma unroll
            for (uint32_t c = 0; c < 3; ++c) lds.level3[c][lane] = v[c];
        }
    }
    wave_fence();
    uint32_t mask = plan->mask[3], pitch = plan->pitch[3];
    if (levels > 4u && coarse) {
        gx = (X0 >> 4) + i;
        gy = Y0 >> 4;
        inside = k < 3u && gx < plan->w[4] && gy < plan->h[4];
        const bool clamp_x = 2u * gx + 1u >= plan->w[3], clamp_y = 2u * gy + 1u >= plan->h[3];
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) v[c] = box<Lay>(lds.level3[c], 8u, i, 0u, clamp_y ? 0u : 1u, clamp_x);
        mask = plan->mask[4];
        pitch = plan->pitch[4];
    }
    float m[1] = {fma_(k == 0u ? kM00 : k == 1u ? kM10 : kM20, v[0],
                       fma_(k == 0u ? kM01 : k == 1u ? kM11 : kM21, v[1],
                            fma_(k < 2u ? kM02 : kM22, v[2], kOpsinBias)))};
    static_assert(kM02 == kM12);
    if constexpr (Clamp) m[0] = fmaxf(m[0], kMinNormal);
    cube_roots<Ref, Clamp>(m);
    lds.roots[lane] = Ref ? m[0] - kCbrtBias : m[0];
    wave_fence();
    // This lane's channel from its sample's roots.
    const uint32_t stride = coarse ? 4u : 16u, at0 = lane - k * stride;
    const float c0 = lds.roots[at0], c1 = lds.roots[at0 + stride], c2 = lds.roots[min(at0 + 2u * stride, 63u)];
    float o;
    if constexpr (Ref) {
        const float half_sum = 0.5f * (c0 + c1);
        o = k == 0u ? fma_(0.5f * (c0 - c1), 14.0f, 0.42f) : k == 1u ? half_sum + 0.01f : (c2 - half_sum) + 0.55f;
    } else {
        const float sum = c0 + c1;
        o = k == 0u ? fma_(c0 - c1, 7.0f, 0.42f) : k == 1u ? fma_(0.5f, sum, kYOffset) : fma_(-0.5f, sum, c2) + 0.55f;
    }
    if (inside && ((mask >> k) & 1u) != 0u) {
        const uint64_t plane = plan->plane_off[coarse ? 4 : 3][k];
        Fmt::store1(plane_at<Fmt>(planes, plane) + static_cast<uint64_t>(gy + kPadTop) * pitch + gx + kPadLeft, o);
    }
    wave_fence();  // the next tile reuses the LDS
}

// One wave's half of prepare work item `b`. Waves work alone (no barriers)
// but for the chroma window of the general decode, which the block stages.
template <typename Lay, bool General, bool Ref>
__device__ __forceinline__ void prepare_tile(const TileRef& tr, uint32_t half, const uint8_t* src0,
                                             const uint8_t* src1, PrepareLds& lds) {
    using Fmt = typename Lay::Fmt;
    ConstAS<PairDesc>* pdp = tr.pdp;
    ConstAS<Plan>* plan = tr.plan;
    const uint32_t image = tr.image, X0 = tr.X0;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t Y0 = tr.Y0 + kWaveRows * half;
    const uint32_t W = plan->width, H = plan->height, levels = plan->levels;
    const uint32_t lx = lane % 16u, ly = lane / 16u;
    GlobalAS<uint8_t>* planes = as_global(static_cast<uint8_t*>(pdp->planes)) + (image ? plan->image_bytes : 0);
    // Single-pair launches name their inputs directly; batches use pd.src.
    const uint8_t* src_ptr = image ? (src1 != nullptr ? src1 : pdp->src[1])
                                   : (src0 != nullptr ? src0 : pdp->src[0]);
    GlobalAS<const uint8_t>* src = as_global(src_ptr);
    const uint64_t plane_stride = plan->plane_stride;
    const uint32_t bx = X0 + 4u * lx;
    bool table = true;
    ConstAS<SourceDesc>* sd = nullptr;
    const float2* window = nullptr;
    decode::ChromaWindow cw{0, 0, 0, 0};
    decode::ChromaWeights<kPrepTileH>* weights = nullptr;
    if constexpr (General) {
        __shared__ decode::ChromaWeights<kPrepTileH> staged;
        weights = &staged;
        // Formats other than 8-bit sRGB RGB decode per pixel (block-uniform).
        const SourceDesc* sdp = image ? pdp->source[1] : pdp->source[0];
        if (sdp != nullptr && as_const(sdp)->kind != 0u) {
            table = false;
            sd = as_const(sdp);
            // Subsampled chroma: the block stages the tile's chroma samples
            // in LDS once, instead of each pixel loading its taps from the
            // planes (8 loads a pixel for bilinear 4:2:0, 72 for Lanczos-3).
            __shared__ float2 chroma[decode::kChromaWindow];
            if (sd->family == 2 && (sd->sub_w != 0 || sd->sub_h != 0)) {
                constexpr uint32_t kThreads = 64u * kPrepWaves<General>;
                if (sd->filter != 0) decode::stage_weights(sd, X0, tr.Y0, threadIdx.x, kThreads, *weights);
                if (decode::chroma_window(sd, X0, min(X0 + kPrepTileW - 1u, W - 1u), tr.Y0,
                                          min(tr.Y0 + kPrepTileH - 1u, H - 1u), &cw)) {
                    decode::stage_chroma(sd, src, cw, threadIdx.x, kThreads, chroma);
                    window = chroma;
                }
                __syncthreads();
            }
        }
    }
    if (Y0 >= H) return;  // the image ends above this wave's rows
    TileWords pre{};
    const uint32_t W1 = plan->w[1], H1 = plan->h[1];
    const uint32_t last_row1 = 2u * (H1 - 1u), last_col1 = 2u * (W1 - 1u);
    auto base_row = [&](uint32_t r) -> uint32_t { return min(min(Y0 + 4u * ly + (r & 2u), last_row1) + (r & 1u), H - 1u); };
    auto base_col = [&](uint32_t j) -> uint32_t { return min(min(bx + (j & 2u), last_col1) + (j & 1u), W - 1u); };
    if constexpr (!General) pre = load_tile_words(src, plane_stride, W, bx, base_row);
    wave_fence();  // the decode table, written while the loads above are under way

    // Levels 0 and 1, a base row at a time; boxes are summed in (0,0), (1,0),
    // (0,1), (1,1) order (prepare.comp:100-111). A sample past a level's last
    // row or column is that row or column again (color.glsl:453-462,
    // prepare.comp:146-168): base samples past the image are clamped to it,
    // and those of a level-1 sample past level 1 are the last one's.
    decode::BilinearColumns columns{};
    if constexpr (General) {
        if (window != nullptr && sd->filter == 0) {
            const uint32_t col[4] = {base_col(0), base_col(1), base_col(2), base_col(3)};
            columns = decode::bilinear_columns(sd, cw, col);
        }
    }
    const uint32_t mask0 = plan->mask[0], mask1 = plan->mask[1];
    const uint32_t gx1 = X0 / 2u + 2u * lx, gy1 = Y0 / 2u + 2u * ly;
    float s2[3] = {0.0f, 0.0f, 0.0f};  // level 2's box
    float v1[2][3] = {};
#pragma unroll 1
    for (uint32_t r = 0; r < 4; ++r) {
        const uint32_t y = Y0 + 4u * ly + r, yc = base_row(r);
        float lin[4][3];
        if constexpr (General) {
            if (!table) {
                const uint32_t col[4] = {base_col(0), base_col(1), base_col(2), base_col(3)};
                decode::row4(sd, src, window, cw, columns, *weights, X0, tr.Y0, bx, col, yc, W, lin);
            }
        }
        if (table) {
#pragma unroll
            for (uint32_t c = 0; c < 3; ++c) {
                if (General ? bx + 3u < W : pre.valid) {
                    const uint32_t v =
                        General ? reinterpret_cast<GlobalAS<const Bytes4>*>(src + c * plane_stride +
                                                                            static_cast<uint64_t>(yc) * W + bx)->v
                                : pre.w[0][c];
                    lin[0][c] = table_at<0>(lds.lut, v);
                    lin[1][c] = table_at<1>(lds.lut, v);
                    lin[2][c] = table_at<2>(lds.lut, v);
                    lin[3][c] = table_at<3>(lds.lut, v);
                } else {
                    GlobalAS<const uint8_t>* row = src + c * plane_stride + static_cast<uint64_t>(yc) * W;
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) lin[j][c] = lds.lut[row[base_col(j)]];
                }
                if constexpr (!General) {
                    pre.w[0][c] = pre.w[1][c];
                    pre.w[1][c] = pre.w[2][c];
                    pre.w[2][c] = pre.w[3][c];
                }
            }
        }
        if (mask0 != 0u && y < H) {
            const uint64_t at = static_cast<uint64_t>(y + kPadTop) * plan->pitch[0] + bx + kPadLeft;
            xyb_group<Ref, 4, General>(lin, mask0, [&](uint32_t c, const float (&v)[4]) {
                auto* p = plane_at<Fmt>(planes, plan->plane_off[0][c]) + at;
                if (bx + 3u < W) {
                    Fmt::store4(p, v);
                } else {
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        if (bx + j < W) Fmt::store1(p + j, v[j]);
                }
            });
        }
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
#pragma unroll
            for (uint32_t jj = 0; jj < 2; ++jj) {
                v1[jj][c] = v1[jj][c] + lin[2 * jj][c];
                v1[jj][c] = v1[jj][c] + lin[2 * jj + 1][c];
            }
        }
        if ((r & 1u) == 0u || levels < 2u) continue;
        // The level-1 row of this row and the one above.
        const uint32_t gy = gy1 + r / 2u;
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c)
#pragma unroll
            for (uint32_t jj = 0; jj < 2; ++jj) v1[jj][c] = linear_sample<Lay>(v1[jj][c] * 0.25f);
        if (mask1 != 0u && gy < H1) {
            const uint64_t at = static_cast<uint64_t>(gy + kPadTop) * plan->pitch[1] + gx1 + kPadLeft;
            xyb_group<Ref, 2, General>(v1, mask1, [&](uint32_t c, const float (&v)[2]) {
                auto* p = plane_at<Fmt>(planes, plan->plane_off[1][c]) + at;
                if (gx1 + 1u < W1) {
                    Fmt::store2(p, v[0], v[1]);
                } else if (gx1 < W1) {
                    Fmt::store1(p, v[0]);
                }
            });
        }
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            s2[c] = s2[c] + v1[0][c];
            s2[c] = s2[c] + v1[1][c];
            v1[0][c] = v1[1][c] = 0.0f;
        }
    }
    if (levels < 3u) return;

    // Level 2: one sample a lane.
#pragma unroll
    for (uint32_t c = 0; c < 3; ++c) {
        s2[c] = linear_sample<Lay>(s2[c] * 0.25f);
        lds.level2[c][lane] = s2[c];
    }
    const uint32_t mask2 = plan->mask[2], gx2 = X0 / 4u + lx, gy2 = Y0 / 4u + ly;
    if (mask2 != 0u && gx2 < plan->w[2] && gy2 < plan->h[2]) {
        const uint64_t at = static_cast<uint64_t>(gy2 + kPadTop) * plan->pitch[2] + gx2 + kPadLeft;
        xyb_group<Ref, 1, General>(&s2, mask2, [&](uint32_t c, const float (&v)[1]) {
            Fmt::store1(plane_at<Fmt>(planes, plan->plane_off[2][c]) + at, v[0]);
        });
    }
    if (levels < 4u) return;
    wave_fence();
    prepare_coarse<Lay, Ref, General>(plan, planes, X0, Y0, lane, lds);
}

// What bounds it: VALU issue, of which the cube roots take about half (15
// instructions each, two of them transcendentals at 8.2 cycles; FP32
// instructions take 2.2). With the roots' last step in FP64 (six instructions
// and three conversions at 4.2, values of two registers) and four waves a SIMD
// 300 1080p pairs took 3.80 ms, one 4K pair 44.9 us; 3.56 ms and 41.8 us with
// the FP32 step alone, 3.32 ms and 38.6 us with the fifth wave that its
// registers leave room for (six waves, 80 registers, spill: 4.0 ms).
//
// A lane takes 4 x 4 base pixels, and with them the boxes of levels 1 and 2,
// so that these need no exchange and every lane works at them; a pass over
// the 60 roots of levels 3 and 4 does the rest. Waves meet at no barrier (the
// 64 x 32 tile of a four-wave block met at five, with one or two waves busy
// from level 2 on). Rows pass through one copy of the code: 9.9 KB against
// 25. 300 pairs: 4.07 -> 3.80 ms, of which the shorter root alone gave none
// while the waves waited at barriers; one 4K pair 53.7 -> 45.9 us; 100 pairs
// in the mixed form 0.90 -> 0.86 ms. (Launches of few tiles, whose time is one
// wave's chain of rows, take the split form below.)
//
// Registers: 93 in the table decode's two forms (five waves a SIMD), 127 in the general decode (four).
template <typename Lay, bool General, bool Ref>
__global__ __launch_bounds__(64 * kPrepWaves<General>) __attribute__((amdgpu_waves_per_eu(General ? 4 : 5))) void
prepare_kernel(const PairDesc* __restrict__ pairs, const WorkRef* __restrict__ work, uint32_t tiles,
               uint32_t tiles_per_image, const float* __restrict__ lut_g, const uint8_t* src0, const uint8_t* src1) {
    constexpr uint32_t kWaves = kPrepWaves<General>, kHalves = kPrepTileH / kWaveRows;
    __shared__ __align__(16) PrepareLds lds[kWaves];
    const uint32_t wave = kWaves == 1u ? 0u : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t entry = 4u * (threadIdx.x & 63u);
    *reinterpret_cast<f32x4*>(lds[wave].lut + entry) =
        *reinterpret_cast<GlobalAS<const f32x4>*>(as_global(lut_g) + entry);
    const uint32_t blocks = tiles * (kHalves / kWaves);
    for (uint32_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        const uint32_t l = xcd_remap(b, blocks) * kWaves + wave;
        prepare_tile<Lay, General, Ref>(resolve_tile(l / kHalves, pairs, work, tiles_per_image), l % kHalves, src0,
                                        src1, lds[wave]);
        if constexpr (General) __syncthreads();  // the next tile reuses the chroma window
    }
}

// The prepare kernel's split form, for launches of few tiles, whose time is one
// wave's chain: four waves take a wave's 64 x 16 pixels, wave r the rows
// 4 ly + r, and pass the boxes on through LDS in the same order of additions:
// waves 1 and 3 finish the two level-1 rows, wave 3 level 2, and wave 0 levels
// 3 and 4 meanwhile. The same samples bit for bit. In the general decode the
// block stages the chroma of its 16 rows.
//
// What bounds it: the launch, the reads of the descriptor, the plan and the row
// (2,900 cycles of the other form's 16,700 at 96x64), and the chain of one row's
// roots, where the other form has four rows' and three levels' (13,800). 48
// registers. Prepare of a launch, reference form: one pair of 96x64 9.0 -> 5.1
// us, 512x512 9.2 -> 6.3, 1080p 19.9 -> 17.2, 8 pairs of 853x479 26.0 -> 24.9.
// The exchange and its three barriers are work of their own, so it loses where
// the device is full anyway.
//
// Up to 14 tiles a CU, where the forms met: 3,360 tiles 24.9 us against 26.0,
// 3,600 (2560x1440) 24.1 both, 6,720 40.8 against 39.2, 4K (8,160) 45.4 against
// 41.2; U16 planes 24.5 against 24.9, 22.8 against 23.1, 37.9 against 36.3.
// General decode, up to 4 tiles a CU: 512x512 8-bit 4:2:0 20.2 -> 10.9 us, 10-bit
// PQ 23.3 -> 11.8, 1280x720 (920 tiles) 24.9 -> 21.0 and 31.6 -> 24.4; 1080p
// (2,040) 33.7 against 36.6 and 42.0 against 41.2. 82 registers.
template <bool General> constexpr uint32_t kSplitTiles = (General ? 4 : 14) * 256;

template <typename Lay, bool General, bool Ref>
__global__ __launch_bounds__(256) void prepare_split_kernel(const PairDesc* __restrict__ pairs,
                                                            const WorkRef* __restrict__ work, uint32_t tiles,
                                                            uint32_t tiles_per_image, const float* __restrict__ lut_g,
                                                            const uint8_t* src0, const uint8_t* src1) {
    using Fmt = typename Lay::Fmt;
    constexpr uint32_t kHalves = kPrepTileH / kWaveRows;
    __shared__ __align__(16) PrepareLds lds[4];  // a decode table a wave; the levels in the first
    __shared__ float boxes1[2][2][3][64], boxes2[3][64];  // sums of the rows above
    const uint32_t r = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t entry = 4u * lane;
    const f32x4 table = *reinterpret_cast<GlobalAS<const f32x4>*>(as_global(lut_g) + entry);
    const uint32_t l = xcd_remap(blockIdx.x, tiles * kHalves);
    const TileRef tr = resolve_tile(l / kHalves, pairs, work, tiles_per_image);
    ConstAS<PairDesc>* pdp = tr.pdp;
    ConstAS<Plan>* plan = tr.plan;
    const uint32_t X0 = tr.X0, Y0 = tr.Y0 + kWaveRows * (l % kHalves);
    const uint32_t W = plan->width, H = plan->height, levels = plan->levels;
    if (Y0 >= H) return;  // the image ends above these rows
    const uint32_t lx = lane % 16u, ly = lane / 16u;
    GlobalAS<uint8_t>* planes =
        as_global(static_cast<uint8_t*>(pdp->planes)) + (tr.image ? plan->image_bytes : 0);
    const uint8_t* src_ptr = tr.image ? (src1 != nullptr ? src1 : pdp->src[1])
                                      : (src0 != nullptr ? src0 : pdp->src[0]);
    GlobalAS<const uint8_t>* src = as_global(src_ptr);
    const uint32_t bx = X0 + 4u * lx, W1 = plan->w[1], H1 = plan->h[1];

    // The base row and columns, clamped as in prepare_tile.
    const uint32_t y = Y0 + 4u * ly + r;
    const uint32_t yc = min(min(Y0 + 4u * ly + (r & 2u), 2u * (H1 - 1u)) + (r & 1u), H - 1u);
    auto base_col = [&](uint32_t j) -> uint32_t { return min(min(bx + (j & 2u), 2u * (W1 - 1u)) + (j & 1u), W - 1u); };
    const bool whole = bx + 3u < W;
    float lin[4][3];
    bool from_table = true;
    if constexpr (General) {
        const SourceDesc* sdp = tr.image ? pdp->source[1] : pdp->source[0];
        if (sdp != nullptr && as_const(sdp)->kind != 0u) {
            from_table = false;
            ConstAS<SourceDesc>* sd = as_const(sdp);
            __shared__ float2 chroma[decode::kChromaWindow];
            const float2* window = nullptr;
            decode::ChromaWindow cw{0, 0, 0, 0};
            __shared__ decode::ChromaWeights<kWaveRows> weights;
            if (sd->family == 2 && (sd->sub_w != 0 || sd->sub_h != 0)) {
                if (sd->filter != 0) decode::stage_weights(sd, X0, Y0, threadIdx.x, 256u, weights);
                if (decode::chroma_window(sd, X0, min(X0 + kPrepTileW - 1u, W - 1u), Y0, min(Y0 + kWaveRows - 1u, H - 1u), &cw)) {
                    decode::stage_chroma(sd, src, cw, threadIdx.x, 256u, chroma);
                    window = chroma;
                }
                __syncthreads();
            }
            const uint32_t col[4] = {base_col(0), base_col(1), base_col(2), base_col(3)};
            decode::BilinearColumns columns{};
            if (window != nullptr && sd->filter == 0) columns = decode::bilinear_columns(sd, cw, col);
            decode::row4(sd, src, window, cw, columns, weights, X0, Y0, bx, col, yc, W, lin);
        }
    }
    if (from_table) {
        uint32_t bytes[3] = {};  // a lane's four samples of each channel
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            GlobalAS<const uint8_t>* row =
                src + c * static_cast<uint64_t>(plan->plane_stride) + static_cast<uint64_t>(yc) * W;
            if (whole) {
                bytes[c] = reinterpret_cast<GlobalAS<const Bytes4>*>(row + bx)->v;
            } else {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) bytes[c] |= static_cast<uint32_t>(row[base_col(j)]) << (8u * j);
            }
        }
        *reinterpret_cast<f32x4*>(lds[r].lut + entry) = table;
        wave_fence();
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            lin[0][c] = table_at<0>(lds[r].lut, bytes[c]);
            lin[1][c] = table_at<1>(lds[r].lut, bytes[c]);
            lin[2][c] = table_at<2>(lds[r].lut, bytes[c]);
            lin[3][c] = table_at<3>(lds[r].lut, bytes[c]);
        }
    }
    // The even rows' half of the level-1 boxes, ahead of their roots.
    if ((r & 1u) == 0u) {
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c)
#pragma unroll
            for (uint32_t jj = 0; jj < 2; ++jj) boxes1[r / 2u][jj][c][lane] = (0.0f + lin[2 * jj][c]) + lin[2 * jj + 1][c];
    }
    __syncthreads();
    const uint32_t gx1 = X0 / 2u + 2u * lx, gy1 = Y0 / 2u + 2u * ly + r / 2u;
    float v1[2][3] = {}, s2[3] = {0.0f, 0.0f, 0.0f};
    if ((r & 1u) != 0u) {
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
#pragma unroll
            for (uint32_t jj = 0; jj < 2; ++jj) {
                v1[jj][c] = boxes1[r / 2u][jj][c][lane] + lin[2 * jj][c];
                v1[jj][c] = v1[jj][c] + lin[2 * jj + 1][c];
                v1[jj][c] = linear_sample<Lay>(v1[jj][c] * 0.25f);
            }
            if (r == 1u) boxes2[c][lane] = (0.0f + v1[0][c]) + v1[1][c];
        }
    }
    __syncthreads();
    if (r == 3u) {
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) {
            s2[c] = boxes2[c][lane] + v1[0][c];
            s2[c] = s2[c] + v1[1][c];
            s2[c] = linear_sample<Lay>(s2[c] * 0.25f);
            lds[0].level2[c][lane] = s2[c];
        }
    }
    __syncthreads();

    const uint32_t mask0 = plan->mask[0], mask1 = plan->mask[1], mask2 = plan->mask[2];
    if (mask0 != 0u && y < H) {
        const uint64_t at = static_cast<uint64_t>(y + kPadTop) * plan->pitch[0] + bx + kPadLeft;
        xyb_group<Ref, 4, General>(lin, mask0, [&](uint32_t c, const float (&v)[4]) {
            auto* p = plane_at<Fmt>(planes, plan->plane_off[0][c]) + at;
            if (whole) {
                Fmt::store4(p, v);
            } else {
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    if (bx + j < W) Fmt::store1(p + j, v[j]);
            }
        });
    }
    if ((r & 1u) != 0u && levels >= 2u && mask1 != 0u && gy1 < H1) {
        const uint64_t at = static_cast<uint64_t>(gy1 + kPadTop) * plan->pitch[1] + gx1 + kPadLeft;
        xyb_group<Ref, 2, General>(v1, mask1, [&](uint32_t c, const float (&v)[2]) {
            auto* p = plane_at<Fmt>(planes, plan->plane_off[1][c]) + at;
            if (gx1 + 1u < W1) {
                Fmt::store2(p, v[0], v[1]);
            } else if (gx1 < W1) {
                Fmt::store1(p, v[0]);
            }
        });
    }
    const uint32_t gx2 = X0 / 4u + lx, gy2 = Y0 / 4u + ly;
    if (r == 2u && levels >= 3u && mask2 != 0u && gx2 < plan->w[2] && gy2 < plan->h[2]) {
#pragma unroll
        for (uint32_t c = 0; c < 3; ++c) s2[c] = lds[0].level2[c][lane];
        const uint64_t at = static_cast<uint64_t>(gy2 + kPadTop) * plan->pitch[2] + gx2 + kPadLeft;
        xyb_group<Ref, 1, General>(&s2, mask2, [&](uint32_t c, const float (&v)[1]) {
            Fmt::store1(plane_at<Fmt>(planes, plan->plane_off[2][c]) + at, v[0]);
        });
    }
    if (r == 0u && levels >= 4u) prepare_coarse<Lay, Ref, General>(plan, planes, X0, Y0, lane, lds[0]);
}

// ---- scale ------------------------------------------------------------------

// What bounds it: VALU issue and, at full rate, the clock. A SIMD issues FP32
// adds, multiplies and fused multiply-adds of two waves at once, one per wave
// every 4.5 cycles (5.1 with a literal operand): 2.2 to 2.6 cycles an
// instruction from two waves up, an even number of them (three share as one
// and two: 1.30 against 0.99 ns an instruction). Only one of the two may be a
// min/max, a conversion, a shift or any instruction with an SGPR operand, and
// FP64 and transcendental instructions take both (4.2 and 8.2 cycles). The
// taps are literals: held in VGPRs the instructions read three registers and
// the launch took 4.62 ms against 4.24 (300 1080p pairs).
//
// Hence four waves a SIMD, 128 registers: one column a lane, not two (a
// 13-row ring of five quantities and two columns alone was 130). The ring is
// kept as the partial sums of the 12 output rows that still wait for source
// rows: a step of four rows completes four of them, and the multiply-add that
// takes a sum's next tap also moves it four places on, so the loop needs no
// unrolling by rows (8.7 KB of code against 45; a wave of a 96x64 pair spends
// 17 us against 30, most of it fetching instructions). FP64 sums live in LDS,
// 10,176 bytes a wave, sixteen waves a CU.
//
// Lanes take four columns of one row in the horizontal pass, so a row's 16
// source samples serve four outputs: 16 bytes of LDS reads an output and
// image in 16-byte accesses, and the products formed in registers, against
// 52 bytes a quantity for a column a lane. (An LDS read of 16 bytes a lane
// runs at 245 B/cycle a CU; the pair of 8-byte reads the two-column form
// compiled to, at 125.)
//
// 300 1080p pairs, reference form: 5.45 -> 4.24 ms, 3.37e9 wave instructions
// at 2.4 cycles each per SIMD (3.7 before), at a clock of about 1.9 GHz (2.2
// before: the chip lowers it as the issue rate rises). 60 pairs of 640x360 to
// 4K: 1.71 -> 1.19 ms; one 4K pair: 91 -> 75 us.
constexpr int kStep = 4;             // source rows a wave takes per step
constexpr int kPending = kTaps - 1;  // output rows that wait for more source rows
constexpr int kSrcCols = 64 + 2 * kRadius;
constexpr int kRawRows = kStep + kRadius;  // raw rows kept in LDS: the step's and the six before them

// Blurred quantities by form:
// the reference form blurs a, b, a*a, b*b and a*b (scale.comp:130-142); the
// difference form a, b, (a - b)^2 and a*b.
template <bool Ref> constexpr int kBlurred = Ref ? 5 : 4;

template <int... P, typename F>
__device__ __forceinline__ void unroll(std::integer_sequence<int, P...>, F&& f) {
    (f(std::integral_constant<int, P>{}), ...);
}

// The six map values of one pixel from its blurred quantities `bl` (in the
// form's order) and its raw samples a and b: d, d^4, ring, ring^4, blur,
// blur^4 (scale.comp:305-333).
template <bool Ref>
__device__ __forceinline__ void map_values(const float* bl, float a, float b, float v6[6]) {
    const float mu1 = bl[0], mu2 = bl[1];
    const float det_dist = 1.0f + fabsf(b - mu2);
    const float det_orig = 1.0f + fabsf(a - mu1);
    float d, d1;
    if constexpr (Ref) {
        // scale.comp:305-333 in its order (the multiply-adds fused):
        // num_m = 1 - (mu1 - mu2)^2, num_s = 2 (s12 - mu1 mu2) + c2,
        // den = (s11 - mu1^2) + (s22 - mu2^2) + c2,
        // d = max((den - num_m num_s) / den, 0), d1 = (det_dist - det_orig) / det_orig,
        // with correctly rounded divisions.
        const float t = mu1 - mu2;
        const float num_m = fma_(-t, t, 1.0f);
        const float num_s = fma_(2.0f, fma_(-mu1, mu2, bl[4]), kC2);
        const float den = (fma_(-mu1, mu1, bl[2]) + fma_(-mu2, mu2, bl[3])) + kC2;
        d = fmaxf(div_rn(fma_(-num_m, num_s, den), den), 0.0f);
        d1 = div_rn(det_dist - det_orig, det_orig);
    } else {
        // scale.comp:305-333 rearranged: with e the blurred (a - b)^2 and
        // t = mu1 - mu2, s11 + s22 - mu1^2 - mu2^2 = num_s - c2 + v where
        // v = e - t^2, so den = num_s + v and den - num_m num_s =
        // v + t^2 num_s. The small v replaces the difference of two large
        // second moments (closer to FP64 than the direct form), and
        // identical images give v = t = 0, d = 0 exactly. One reciprocal
        // serves both quotients: q = 1 / (den det_orig), with
        // den >= c2 - rounding > 0 and det_orig >= 1.
        const float t = mu1 - mu2;
        const float num_s = fma_(2.0f, fma_(-mu1, mu2, bl[3]), kC2);
        const float v = fma_(-t, t, bl[2]);
        const float den = num_s + v;
        const float q = rcp_rn(den * det_orig);
        d = fmaxf((fma_(t * t, num_s, v) * det_orig) * q, 0.0f);
        d1 = ((det_dist - det_orig) * den) * q;
    }
    const float dd = d * d;
    const float ring = fmaxf(d1, 0.0f);
    const float blur = fmaxf(-d1, 0.0f);
    const float rr = ring * ring, bb = blur * blur;
    v6[0] = d;
    v6[1] = dd * dd;
    v6[2] = ring;
    v6[3] = rr * rr;
    v6[4] = blur;
    v6[5] = bb * bb;
}

// Adds source columns 4 t .. 4 t + 3 of a row (samples a, b of both images) to
// the horizontal sums of its output columns 0 .. 3, whose taps ascend with the
// source column (scale.comp:187-241).
template <typename TapsT, bool Ref>
__device__ __forceinline__ void blur_quad(int t, f32x4 a, f32x4 b, float (&acc)[kBlurred<Ref>][4]) {
    constexpr int Q = kBlurred<Ref>;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int m = 4 * t + e;
        const float x = a[e], y = b[e];
        float v[Q];
        v[0] = x;
        v[1] = y;
        if constexpr (Ref) {
            v[2] = x * x;
            v[3] = y * y;
            v[4] = x * y;
        } else {
            const float d = x - y;
            v[2] = d * d;
            v[3] = x * y;
        }
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int k = m - c;
                if (k == 0) acc[q][c] = TapsT::w[0] * v[q];
                if (k > 0 && k < kTaps) acc[q][c] = fma_(TapsT::w[k], v[q], acc[q][c]);
            }
    }
}

// One wave's LDS: the raw rows of the last kRawSlots steps, and the
// exchange that turns horizontal results (lane = row and column group) into
// the vertical pass's (lane = column).
struct ScaleLds {
    float raw[2][kRawRows][kSrcCols];
    float turn[kStep][64];
    double sums[6][64];
};

// One wave's part of a scale work item: 64 columns from x0 of the strip
// whose first row is y0, with the plane elements in format Fmt. Leaves the
// six map sums of each column in lds.sums.
template <typename Fmt, typename TapsT, bool Ref>
__device__ __forceinline__ void scale_strip(ConstAS<PairDesc>* pdp, ConstAS<Plan>* plan, uint32_t level,
                                            uint32_t channel, uint32_t x0, uint32_t y0, ScaleLds& lds) {
    using E = typename Fmt::E;
    constexpr int Q = kBlurred<Ref>;
    const uint32_t H = plan->h[level], pitch = plan->pitch[level];
    // The part's output rows stop at the level's last row.
    const int total = static_cast<int>(min(plan->part_h, H - y0)) + 2 * kRadius;

    // Source row r (0 .. total-1) is image row y0 - 6 + r, padded row y0 + r;
    // source column j (0 .. 75) is image column x0 - 6 + j, padded x0 + 2 + j.
    GlobalAS<const uint8_t>* pa =
        as_global(static_cast<const uint8_t*>(pdp->planes)) + plan->plane_off[level][channel] +
        (static_cast<uint64_t>(y0) * pitch + x0 + 2u) * sizeof(E);
    GlobalAS<const uint8_t>* pb = pa + plan->image_bytes;
    auto load = [](GlobalAS<const uint8_t>* p, uint32_t offset) {
        return Fmt::load4(reinterpret_cast<GlobalAS<const E>*>(p + offset));
    };

    // Horizontal roles: lane = source row `r` of the step and four columns
    // from 4 g. The 12 halo columns of the step's rows are three quads a row
    // and image, loaded by lanes 0 .. 11 (a) and 16 .. 27 (b).
    uint32_t lane = threadIdx.x & 63u;
    asm volatile("" : "+v"(lane));  // nothing formed from it is held across items
    const uint32_t r = lane >> 4, g = lane & 15u;
    const bool halo = g < 3u * kStep && lane < 32u;
    const uint32_t hr = (g < 12u ? g : 0u) / 3u, hc = 64u + 4u * (g - 3u * hr);
    const uint32_t at = (r * pitch + 4u * g) * sizeof(E), halo_at = (hr * pitch + hc) * sizeof(E);
    float* const halo_to = &lds.raw[lane < 16u ? 0 : 1][0][hc];

    const bool halo_b = lane >= 16u;
    typename Fmt::Raw4 cur_a = load(pa, at), cur_b = load(pb, at), cur_h = load(halo_b ? pb : pa, halo_at);

    // The vertical pass in flight: partial sums of the 12 output rows that
    // still miss source rows, oldest first.
    float part[Q][kPending];
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int m = 0; m < kPending; ++m) part[q][m] = 0.0f;
    float block[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        block[k] = 0.0f;
        lds.sums[k][lane] = 0.0;
    }
    uint32_t slot = 0;  // the ring row of the step's first row

    for (int i0 = 0; i0 < total; i0 += kStep) {
        // The lane's LDS addresses are formed again each step rather than
        // held: registers are what limits the waves in flight.
        asm("" : "+v"(lane));
        const uint32_t r = lane >> 4, g = lane & 15u;
        // Stage the step's rows.
        auto ring = [&](uint32_t row) { return row >= kRawRows ? row - kRawRows : row; };
        float* const ra = &lds.raw[0][0][0] + (ring(slot + r) * kSrcCols + 4u * g);
        float* const rb = ra + kRawRows * kSrcCols;
        {
            float v[4];
            Fmt::unpack4(cur_a, v);
            *reinterpret_cast<f32x4*>(ra) = f32x4{v[0], v[1], v[2], v[3]};
            Fmt::unpack4(cur_b, v);
            *reinterpret_cast<f32x4*>(rb) = f32x4{v[0], v[1], v[2], v[3]};
            if (halo) {
                Fmt::unpack4(cur_h, v);
                *reinterpret_cast<f32x4*>(halo_to + ring(slot + hr) * kSrcCols) = f32x4{v[0], v[1], v[2], v[3]};
            }
        }
        wave_fence();

        // Horizontal 13-tap pass: columns 4 g .. 4 g + 3 of row r, source
        // columns in ascending order so that every chain's taps ascend
        // (scale.comp:187-241).
        float acc[Q][4];
        {
            f32x4 va = *reinterpret_cast<const f32x4*>(ra), vb = *reinterpret_cast<const f32x4*>(rb);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f32x4 na{}, nb{};
                if (t < 3) {
                    na = *reinterpret_cast<const f32x4*>(ra + 4 * t + 4);
                    nb = *reinterpret_cast<const f32x4*>(rb + 4 * t + 4);
                }
                blur_quad<TapsT, Ref>(t, va, vb, acc);
                va = na;
                vb = nb;
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        // The next step's rows, in flight until its start. (The last step
        // loads its own again: the rows after it may lie past the plane. A
        // branch around the loads lets the compiler sink the sums above past
        // them, which spills.)
        const uint32_t advance = i0 + kStep < total ? kStep * pitch * static_cast<uint32_t>(sizeof(E)) : 0u;
        pa += advance;
        pb += advance;
        cur_a = load(pa, at);
        cur_b = load(pb, at);
        cur_h = load(halo_b ? pb : pa, halo_at);
        __builtin_amdgcn_sched_barrier(0);

        // Turn each quantity's results to lane = column and add the four new
        // rows to the pending output rows, taps ascending with the source
        // row (scale.comp:243-298). Output rows i0 - 12 .. i0 - 9 complete.
        float done[kStep][Q], h[2][kStep];
        auto turn = [&](int q) {
            *reinterpret_cast<f32x4*>(&lds.turn[0][4u * lane]) = f32x4{acc[q][0], acc[q][1], acc[q][2], acc[q][3]};
            wave_fence();
#pragma unroll
            for (int j = 0; j < kStep; ++j) h[q & 1][j] = lds.turn[j][lane];
            wave_fence();
        };
        turn(0);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if (q + 1 < Q) turn(q + 1);  // in flight while this quantity's rows are added
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int m = 0; m < kPending + kStep; ++m) {
                // Output row i0 - 12 + m: new row j is its tap 12 - m + j.
                float v = m < kPending ? part[q][m] : 0.0f;
#pragma unroll
                for (int j = 0; j < kStep; ++j) {
                    const int k = kTaps - 1 - m + j;
                    if (k == 0) v = TapsT::w[0] * h[q & 1][j];
                    if (k > 0 && k < kTaps)
                        v = j == 0 ? fma_move(TapsT::w[k], h[q & 1][j], v) : fma_(TapsT::w[k], h[q & 1][j], v);
                }
                if (m < kStep) done[m][q] = v; else part[q][m - kStep] = v;
            }
            __builtin_amdgcn_sched_barrier(0);
        }

        // The pixels' own samples: source rows i - 6, kStep rows on in the
        // ring (nothing uses them before the first output row).
        float own[kStep][2];
#pragma unroll
        for (int j = 0; j < kStep; ++j) {
            const float* const at_j = &lds.raw[0][0][kRadius] + (ring(slot + kStep + j) * kSrcCols + lane);
            own[j][0] = at_j[0];
            own[j][1] = at_j[kRawRows * kSrcCols];
        }
        unroll(std::make_integer_sequence<int, kStep>{}, [&](auto jc) {
            constexpr int J = decltype(jc)::value;
            if (i0 < 2 * kRadius || i0 + J >= total) return;
            float v6[6];
            map_values<Ref>(done[J], own[J][0], own[J][1], v6);
#pragma unroll
            for (int k = 0; k < 6; ++k) block[k] = block[k] + v6[k];
            __builtin_amdgcn_sched_barrier(0);
        });
        // Rows 8k .. 8k+7 of the level end with every second step; the
        // level's last rows are added after the loop.
        if ((i0 & kStep) == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                lds.sums[k][lane] += static_cast<double>(block[k]);
                block[k] = 0.0f;
            }
        }
        slot = ring(slot + kStep);
        wave_fence();
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) lds.sums[k][lane] += static_cast<double>(block[k]);
}

// v plus lane (l ^ 1)'s, (l ^ 2)'s or (7 - l % 8)'s v, by DPP control.
template <int Ctrl>
__device__ __forceinline__ double add_dpp(double v) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(bits), Ctrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(bits >> 32), Ctrl, 0xF, 0xF, true);
    return v + __builtin_bit_cast(double, static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32 | static_cast<uint32_t>(lo));
}

// The wave's map sums over its first `cols` columns: lanes 8 k .. 8 k + 7
// (k < 6) return map k's, each lane adding every eighth column.
__device__ __forceinline__ double sum_columns(const ScaleLds& lds, uint32_t lane, uint32_t cols) {
    const uint32_t k = min(lane >> 3, 5u);
    double v = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        const uint32_t c = (lane & 7u) + 8u * i;
        v += c < cols ? lds.sums[k][c] : 0.0;
    }
    v = add_dpp<0xB1>(v);   // quad_perm [1, 0, 3, 2]
    v = add_dpp<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    return add_dpp<0x141>(v);  // row_half_mirror
}

// Parts blockIdx.x, blockIdx.x + gridDim.x, ... of `blocks`, one wave each:
// item * parts_per_item + sub, where an item's parts run over its 64-column
// halves, then its part_h-row bands.
template <typename Lay, typename TapsT, bool Ref>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void scale_kernel(
    const PairDesc* __restrict__ pairs, const WorkRef* __restrict__ work, uint32_t blocks, uint32_t parts_per_pair) {
    __shared__ __align__(16) ScaleLds lds;

    for (uint32_t b = blockIdx.x; b < blocks; b += gridDim.x) {
        uint32_t pair_idx, part;
        if (work != nullptr) {
            ConstAS<WorkRef>* w = as_const(work) + xcd_remap(b, blocks);
            pair_idx = w->pair;
            part = w->index;
        } else {
            const uint32_t l = xcd_remap(b, blocks);
            pair_idx = l / parts_per_pair;
            part = l % parts_per_pair;
        }
        ConstAS<PairDesc>* pdp = as_const(pairs) + pair_idx;
        ConstAS<Plan>* plan = as_const(pdp->plan);
        const uint32_t shift = plan->part_shift, wide = plan->strip_w / 128u;
        ConstAS<ScaleItem>* item = as_const(pdp->items) + (part >> shift);
        const uint32_t sub = part & ((1u << shift) - 1u);
        const uint32_t level = item->level, channel = item->channel;
        const uint32_t x0 = item->x0 + 64u * (sub & wide), y0 = item->y0 + (sub >> wide) * plan->part_h;
        const uint32_t W = plan->w[level];
        uint32_t lane = threadIdx.x & 63u;
        double v = 0.0;
        if (x0 < W && y0 < plan->h[level]) {  // else the item's strip ends before this part
            scale_strip<typename Lay::Fmt, TapsT, Ref>(pdp, plan, level, channel, x0, y0, lds);
            asm volatile("" : "+v"(lane));  // the addresses below are formed here, not held through the strip
            wave_fence();
            v = sum_columns(lds, lane, W - x0);
            wave_fence();  // the next part reuses the LDS
        }
        GlobalAS<double>* out = as_global(pdp->partials) + static_cast<uint64_t>(part) * 6u;
        if (lane < 48u && (lane & 7u) == 0u) out[lane >> 3] = v;
    }
}

// The block form of the scale kernel, for launches of few pairs, whose time is
// the chain of one wave's steps: a block of eight waves takes 64 columns by 32
// rows of a level and channel.
//
// The waves blur the block's 44 source rows horizontally, four rows a wave at
// a time as above but from global memory, into LDS; after a barrier each takes
// 8 rows of 32 columns, a lane four rows of a column, down the columns. So a
// wave's chain is one or two horizontal passes and four output rows' vertical
// ones, against five and more steps of both, and the 12 rows above a band are
// blurred once for 32 output rows, not once for each 8 or 16.
//
// What bounds it: at 96x64 that chain, some 10,000 cycles against 22,900 (2,000
// of them the reads of the descriptor, the plan and the item); from 1080p on
// VALU issue. One pair's launch, reference form: 96x64 10.2 -> 5.9 us, 512x512
// 11.7 -> 6.6, 1080p 27.2 -> 23.2, 2560x1440 41.2 -> 38.4; a 4K pair takes 77
// against 71 us (SinglePairRowParts). 78 registers and 69,888 bytes of LDS: two
// blocks a CU.
constexpr int kBlockWaves = 8;
constexpr int kBlockSourceRows = static_cast<int>(kBlockRows) + 2 * kRadius;
constexpr int kBlockPitch = 72;  // floats a row: rows four apart lie 32 banks apart

template <bool Ref>
struct BlockLds {
    float blurred[kBlurred<Ref>][kBlockSourceRows][kBlockPitch];
    float sums[kBlockWaves][6][32];
    double parts[kBlockWaves][6];
};

template <typename Lay, typename TapsT, bool Ref>
__global__ __launch_bounds__(64 * kBlockWaves) __attribute__((amdgpu_waves_per_eu(4))) void scale_block_kernel(
    const PairDesc* __restrict__ pairs, const WorkRef* __restrict__ work, uint32_t blocks, uint32_t items_per_pair) {
    using Fmt = typename Lay::Fmt;
    using E = typename Fmt::E;
    constexpr int Q = kBlurred<Ref>;
    __shared__ __align__(16) BlockLds<Ref> lds;
    const uint32_t l = xcd_remap(blockIdx.x, blocks);
    uint32_t pair_idx, index;
    if (work != nullptr) {
        ConstAS<WorkRef>* w = as_const(work) + l;
        pair_idx = w->pair;
        index = w->index;
    } else {
        pair_idx = l / items_per_pair;
        index = l - pair_idx * items_per_pair;
    }
    ConstAS<PairDesc>* pdp = as_const(pairs) + pair_idx;
    ConstAS<Plan>* plan = as_const(pdp->plan);
    ConstAS<ScaleItem>* item = as_const(pdp->items) + index;
    const uint32_t level = item->level, channel = item->channel, x0 = item->x0, y0 = item->y0;
    const uint32_t W = plan->w[level], pitch = plan->pitch[level];
    const int out = static_cast<int>(min(kBlockRows, plan->h[level] - y0));  // the level ends below them
    const int total = out + 2 * kRadius, units = (total + kStep - 1) / kStep;
    const int wave = static_cast<int>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    const uint32_t lane = threadIdx.x & 63u;

    // Source row r is padded row y0 + r, source column j is padded x0 + 2 + j
    // (as in scale_strip).
    GlobalAS<const uint8_t>* base = as_global(static_cast<const uint8_t*>(pdp->planes)) +
                                    plan->plane_off[level][channel] +
                                    (static_cast<uint64_t>(y0) * pitch + x0 + 2u) * sizeof(E);
    GlobalAS<const E>* pa = reinterpret_cast<GlobalAS<const E>*>(base);
    GlobalAS<const E>* pb = reinterpret_cast<GlobalAS<const E>*>(base + plan->image_bytes);

    // Vertical role: lane = four rows from row0 of column `col`; its own
    // samples are loaded ahead (rows past the block's last are that row).
    const int row0 = 8 * (wave >> 1) + 4 * static_cast<int>(lane >> 5);
    const uint32_t col = 32u * (static_cast<uint32_t>(wave) & 1u) + (lane & 31u);
    float own[kStep][2];
#pragma unroll
    for (int j = 0; j < kStep; ++j) {
        const uint32_t at = static_cast<uint32_t>(min(row0 + j, out - 1) + kRadius) * pitch + kRadius + col;
        own[j][0] = Fmt::load1(pa + at);
        own[j][1] = Fmt::load1(pb + at);
    }

    for (int unit = wave; unit < units; unit += kBlockWaves) {
        const uint32_t r = static_cast<uint32_t>(unit) * kStep + (lane >> 4), g = lane & 15u;
        const uint32_t at = r * pitch + 4u * g;
        typename Fmt::Raw4 ra[4], rb[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            ra[t] = Fmt::load4(pa + at + 4 * t);
            rb[t] = Fmt::load4(pb + at + 4 * t);
        }
        float acc[Q][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            float a[4], b[4];
            Fmt::unpack4(ra[t], a);
            Fmt::unpack4(rb[t], b);
            blur_quad<TapsT, Ref>(t, f32x4{a[0], a[1], a[2], a[3]}, f32x4{b[0], b[1], b[2], b[3]}, acc);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q)
            *reinterpret_cast<f32x4*>(&lds.blurred[q][r][4u * g]) = f32x4{acc[q][0], acc[q][1], acc[q][2], acc[q][3]};
    }
    __syncthreads();

    double v = 0.0;
    if (8 * (wave >> 1) < out) {
        // Taps ascend with the source row (scale.comp:243-298).
        float done[kStep][Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
#pragma unroll
            for (int m = 0; m < kTaps - 1 + kStep; ++m) {
                const float h = lds.blurred[q][row0 + m][col];
#pragma unroll
                for (int j = 0; j < kStep; ++j) {
                    const int k = m - j;
                    if (k == 0) done[j][q] = TapsT::w[0] * h;
                    if (k > 0 && k < kTaps) done[j][q] = fma_(TapsT::w[k], h, done[j][q]);
                }
            }
        }
        // FP32 sums of the level's rows 8 k .. 8 k + 7 in their order: the
        // lower lanes' four rows, then the upper lanes'.
        float v6[kStep][6], sum[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < kStep; ++j) {
            map_values<Ref>(done[j], own[j][0], own[j][1], v6[j]);
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                v6[j][k] = row0 + j < out ? v6[j][k] : 0.0f;
                sum[k] = sum[k] + v6[j][k];
            }
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            sum[k] = __int_as_float(
                __builtin_amdgcn_ds_bpermute(static_cast<int>(4u * (lane & 31u)), __float_as_int(sum[k])));
#pragma unroll
            for (int j = 0; j < kStep; ++j) sum[k] = sum[k] + v6[j][k];
            if (lane >= 32u) lds.sums[wave][k][lane - 32u] = sum[k];
        }
        wave_fence();
        // Lanes 8 k .. 8 k + 7 add map k's columns that lie in the level.
        const uint32_t k = min(lane >> 3, 5u);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t c = (lane & 7u) + 8u * i;
            v += x0 + 32u * (static_cast<uint32_t>(wave) & 1u) + c < W ? static_cast<double>(lds.sums[wave][k][c]) : 0.0;
        }
        v = add_dpp<0xB1>(v);
        v = add_dpp<0x4E>(v);
        v = add_dpp<0x141>(v);
    }
    if (lane < 48u && (lane & 7u) == 0u) lds.parts[wave][lane >> 3] = v;
    __syncthreads();
    if (threadIdx.x < 6u) {
        double total_k = 0.0;
#pragma unroll
        for (int w = 0; w < kBlockWaves; ++w) total_k += lds.parts[w][threadIdx.x];
        as_global(pdp->partials)[static_cast<uint64_t>(index) * 6u + threadIdx.x] = total_k;
    }
}

// ---- reduce -----------------------------------------------------------------

// One block per (pair, level, channel): its threads stride over the range's
// parts, each adding the six partial sums of its parts in FP64 (four parts'
// loads in flight at a time), rows of 16 lanes and then six threads add them
// up, and those write the six norms (zeros for a channel that is not stored).
// Latency bound. A launch of one pair took 4.0 (96x64), 7.4 (1080p) and 11.4
// us (4K) in one block of 16 waves a pair, a wave to a range; it takes 3.7, 3.9
// and 5.3 (3.7 is an empty range's time). 8 pairs of 853x479: 5.8 -> 4.1 us;
// 300 of 1080p: 16 -> 18, of 8,100 for all three kernels.
// Norm level*18 + k: k < 6 is channel k/2's SSIM' slot k%2; k >= 6 is
// channel (k-6)/4's edge slot 2 + (k-6)%4 (ring 1-, 4-norm, blur 1-, 4-norm).
constexpr uint32_t kReduceThreads = 256;
constexpr uint32_t kRanges = kMaxScales * kChannels;

__global__ __launch_bounds__(kReduceThreads) void reduce_kernel(const PairDesc* __restrict__ pairs) {
    __shared__ double rows[kReduceThreads / 16][6];
    const uint32_t pair = blockIdx.x / kRanges, range = blockIdx.x % kRanges;
    ConstAS<PairDesc>* pdp = as_const(pairs) + pair;
    ConstAS<Plan>* plan = as_const(pdp->plan);
    const uint32_t level = range / kChannels, c = range % kChannels;
    const bool active = level < plan->levels && (plan->mask[level] & (1u << c)) != 0u;
    if (active) {
        const uint32_t begin = plan->item_begin[level][c] << plan->part_shift;
        const uint32_t count = plan->item_count[level][c] << plan->part_shift;
        GlobalAS<const double>* p = as_global(static_cast<const double*>(pdp->partials)) +
                                    static_cast<uint64_t>(begin) * 6u;
        double sum[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (uint32_t i = threadIdx.x; i < count; i += kReduceThreads)
#pragma unroll
            for (int k = 0; k < 6; ++k) sum[k] += p[static_cast<uint64_t>(i) * 6u + k];
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            sum[k] = add_dpp<0xB1>(sum[k]);   // quad_perm [1, 0, 3, 2]
            sum[k] = add_dpp<0x4E>(sum[k]);   // quad_perm [2, 3, 0, 1]
            sum[k] = add_dpp<0x141>(sum[k]);  // row_half_mirror
            sum[k] = add_dpp<0x140>(sum[k]);  // row_mirror
        }
        if (threadIdx.x % 16u == 0u)
#pragma unroll
            for (int k = 0; k < 6; ++k) rows[threadIdx.x / 16u][k] = sum[k];
    }
    __syncthreads();
    const uint32_t slot = threadIdx.x;
    if (slot >= 6u) return;
    double value = 0.0;
    if (active) {
#pragma unroll
        for (uint32_t r = 0; r < kReduceThreads / 16u; ++r) value += rows[r][slot];
        value *= 1.0 / (static_cast<double>(plan->w[level]) * static_cast<double>(plan->h[level]));
        if (slot & 1u) value = sqrt(sqrt(value));
    }
    const uint32_t k = slot < 2u ? 2u * c + slot : 6u + 4u * c + (slot - 2u);
    // Coherent host memory, or the caller's on the device: seen by the host once
    // it has waited for an event behind this kernel. (System-scope stores took
    // 32 to 42 us for 300 pairs, these 18.)
    as_global(pdp->norms)[level * 18u + k] = value;
}

// A plain streaming copy (16-byte loads and stores): the reference point that
// scales the FETCH_SIZE / WRITE_SIZE counters to bytes.
__global__ __launch_bounds__(256) void copy_kernel(const uint4* __restrict__ src,
                                                   uint4* __restrict__ dst, uint64_t n) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        dst[i] = src[i];
}

// Self-check of the reference form's cube root over the floats with bits in
// [first, end): cbrt_rn_near_hw settled by cbrt_round_exact, and on its range
// cbrt_rn_near_f32 settled the same way, against cbrt_rn (IEEE steps only).
// Counts the inputs where they differ and those where the FP64 step took the
// exact one, and keeps the smallest differing input and the largest
// |1 - x r^3| of the hardware seed r (as FP64 bits: non-negative doubles
// order as their bits). One atomic per wave and counter.
__global__ __launch_bounds__(256) void cbrt_check_kernel(uint32_t first, uint32_t end, CbrtCheck* out) {
    unsigned long long bad = 0, near = 0, h_bits = 0;
    uint32_t first_bad = 0xFFFFFFFFu;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t u = first + static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; u < end; u += stride) {
        const float x = __uint_as_float(static_cast<uint32_t>(u));
        bool n;
        const float rounded = cbrt_rn_near_hw(x, &n);
        const float got = n ? cbrt_round_exact(x, rounded) : rounded;
        near += n ? 1u : 0u;
        const float want = cbrt_rn(x);
        bool differs = got != want;
        if (static_cast<uint32_t>(u) - kCbrtF32First < kCbrtF32Count) {
            bool unsettled;
            float root = cbrt_rn_near_f32(x, &unsettled);
            if (unsettled) root = cbrt_round_exact(x, root);
            differs |= root != want;
        }
        if (differs) {
            ++bad;
            first_bad = min(first_bad, static_cast<uint32_t>(u));
        }
        const double r = cbrt_seed_hw(x);
        const double h = fabs(fma_(-static_cast<double>(x), (r * r) * r, 1.0));
        h_bits = max(h_bits, static_cast<unsigned long long>(__double_as_longlong(h)));
    }
    for (int offset = 32; offset > 0; offset >>= 1) {
        bad += __shfl_xor(bad, offset, 64);
        near += __shfl_xor(near, offset, 64);
        h_bits = max(h_bits, __shfl_xor(h_bits, offset, 64));
        first_bad = min(first_bad, __shfl_xor(first_bad, offset, 64));
    }
    if (threadIdx.x % 64u == 0u) {
        atomicAdd(&out->mismatches, bad);
        atomicAdd(&out->near, near);
        atomicMax(&out->max_h_bits, h_bits);
        atomicMin(&out->first_mismatch, first_bad);
    }
}

// Self-check of div_rn over the significand pairs a = 1.ma, b = 1.mb with
// mb in [mb_first, mb_first + rows) and every ma, against the IEEE quotient;
// of rcp_rn(b) against 1 / b; and of the hardware reciprocal's exponent
// invariance for those b over 2^e, e in [-24, 24). One atomic per wave and
// counter.
__global__ __launch_bounds__(256) void div_check_kernel(uint32_t mb_first, uint32_t rows, DivCheck* out) {
    unsigned long long bad = 0, rcp_bad = 0;
    uint32_t first_bad = 0xFFFFFFFFu;
    const uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t lane0 = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t k = 0; k < rows; ++k) {
        const uint32_t mb = mb_first + k;
        const float b = __uint_as_float(0x3F800000u | mb);
        for (uint32_t ma = lane0; ma < (1u << 23); ma += stride) {
            const float a = __uint_as_float(0x3F800000u | ma);
            if (__float_as_uint(div_rn(a, b)) != __float_as_uint(a / b)) {
                ++bad;
                first_bad = min(first_bad, mb);
            }
        }
        if (lane0 < 48u) {
            const int e = static_cast<int>(lane0) - 24;
            const float want = __builtin_ldexpf(__builtin_amdgcn_rcpf(b), -e);
            if (__float_as_uint(__builtin_amdgcn_rcpf(__builtin_ldexpf(b, e))) != __float_as_uint(want)) ++rcp_bad;
        } else if (lane0 == 48u) {
            // The refined reciprocal is the correctly rounded 1 / b.
            if (__float_as_uint(rcp_rn(b)) != __float_as_uint(1.0f / b)) ++rcp_bad;
        }
    }
    for (int offset = 32; offset > 0; offset >>= 1) {
        bad += __shfl_xor(bad, offset, 64);
        rcp_bad += __shfl_xor(rcp_bad, offset, 64);
        first_bad = min(first_bad, __shfl_xor(first_bad, offset, 64));
    }
    if (threadIdx.x % 64u == 0u) {
        atomicAdd(&out->mismatches, bad);
        atomicAdd(&out->rcp_mismatches, rcp_bad);
        atomicMin(&out->first_mismatch, first_bad);
    }
}

// Blocks of `kernel` the device holds resident at once: occupancy per
// compute unit x compute units, rounded down to a multiple of 8 (at least
// 8). A persistent launch uses min(work items, this) blocks, each looping
// over its share; 0 when the runtime cannot say.
uint32_t ResidentGrid(const void* kernel, int device, int block_threads) {
    int per_cu = 0;
    hipDeviceProp_t prop{};
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block_threads, 0) != hipSuccess ||
        hipGetDeviceProperties(&prop, device) != hipSuccess || per_cu <= 0 || prop.multiProcessorCount <= 0)
        return 0;
    const uint64_t resident = static_cast<uint64_t>(per_cu) * static_cast<uint64_t>(prop.multiProcessorCount);
    return static_cast<uint32_t>(std::min<uint64_t>(std::max<uint64_t>(8, resident / 8 * 8), 0x7FFFFFF8u));
}

// The grid of a kernel whose blocks stride over `blocks`: all that a launch may
// have, or the resident ones.
template <auto Kernel>
uint32_t GridOf(int block_threads, uint32_t blocks, bool persistent) {
    blocks = std::min(blocks, MaxBlocks(static_cast<uint32_t>(block_threads)));
    int device = 0;
    if (!persistent || hipGetDevice(&device) != hipSuccess) return blocks;
    const uint32_t resident = OncePerKernel<Kernel>(
        device, [&] { return ResidentGrid(reinterpret_cast<const void*>(Kernel), device, block_threads); });
    return resident == 0 ? blocks : std::min(blocks, resident);
}

// Launches `kernel`, with `done` (null: none) set by its own dispatch.
template <typename... Params, typename... Args>
hipError_t Dispatch(void (*kernel)(Params...), uint32_t grid, uint32_t threads, hipStream_t stream, hipEvent_t done,
                    Args... args) {
    if (done != nullptr)
        hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, stream, nullptr, done, 0,
                              static_cast<Params>(args)...);
    else
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), 0, stream, static_cast<Params>(args)...);
    return hipGetLastError();
}

// A launch of no work: `done` still follows what is queued.
hipError_t Nothing(hipStream_t stream, hipEvent_t done) {
    return done != nullptr ? hipEventRecord(done, stream) : hipSuccess;
}

template <typename Lay, bool General, bool Ref>
hipError_t launch_prepare_g(const PairDesc* pairs, const WorkRef* work, uint32_t blocks, uint32_t tiles,
                            const float* lut, const uint8_t* src0, const uint8_t* src1, bool persistent,
                            hipStream_t stream, hipEvent_t done) {
    if (!persistent && blocks <= kSplitTiles<General>)
        return Dispatch(&prepare_split_kernel<Lay, General, Ref>, blocks * (kPrepTileH / kWaveRows), 256, stream, done,
                        pairs, work, blocks, tiles, lut, src0, src1);
    constexpr uint32_t kThreads = 64 * kPrepWaves<General>, kBlocksPerTile = kPrepTileH / kWaveRows / kPrepWaves<General>;
    const uint32_t grid = GridOf<&prepare_kernel<Lay, General, Ref>>(kThreads, blocks * kBlocksPerTile, persistent);
    return Dispatch(&prepare_kernel<Lay, General, Ref>, grid, kThreads, stream, done, pairs, work, blocks, tiles, lut,
                    src0, src1);
}

template <typename Lay, bool Ref>
hipError_t launch_prepare_m(bool general, const PairDesc* pairs, const WorkRef* work, uint32_t blocks,
                            uint32_t tiles, const float* lut, const uint8_t* src0, const uint8_t* src1,
                            bool persistent, hipStream_t stream, hipEvent_t done) {
    const auto launch = general ? &launch_prepare_g<Lay, true, Ref> : &launch_prepare_g<Lay, false, Ref>;
    return launch(pairs, work, blocks, tiles, lut, src0, src1, persistent, stream, done);
}

template <typename Lay>
hipError_t launch_prepare_t(MapForm map, bool general, const PairDesc* pairs, const WorkRef* work,
                            uint32_t blocks, uint32_t tiles, const float* lut, const uint8_t* src0,
                            const uint8_t* src1, bool persistent, hipStream_t stream, hipEvent_t done) {
    const auto launch = map == kMapReference ? &launch_prepare_m<Lay, true> : &launch_prepare_m<Lay, false>;
    return launch(general, pairs, work, blocks, tiles, lut, src0, src1, persistent, stream, done);
}

template <typename Lay, typename TapsT, bool Ref>
hipError_t launch_scale_g(const PairDesc* pairs, const WorkRef* work, uint32_t blocks, uint32_t parts,
                          bool block_form, bool persistent, hipStream_t stream, hipEvent_t done) {
    if (block_form) {
        // Runs of whole pairs, or of the work list.
        constexpr uint32_t kMost = MaxBlocks(64 * kBlockWaves);
        const uint32_t unit = work != nullptr ? 1u : parts;
        return InRuns(blocks / unit, std::max(kMost / unit, 1u), [&](uint32_t first, uint32_t n, bool last) {
            return Dispatch(&scale_block_kernel<Lay, TapsT, Ref>, n * unit, 64 * kBlockWaves, stream,
                            last ? done : nullptr, work != nullptr ? pairs : pairs + first,
                            work != nullptr ? work + first : nullptr, n * unit, parts);
        });
    }
    const uint32_t grid = GridOf<&scale_kernel<Lay, TapsT, Ref>>(64, blocks, persistent);
    return Dispatch(&scale_kernel<Lay, TapsT, Ref>, grid, 64, stream, done, pairs, work, blocks, parts);
}

template <typename Lay, bool Ref>
hipError_t launch_scale_m(uint32_t blur, const PairDesc* pairs, const WorkRef* work, uint32_t blocks,
                          uint32_t parts, bool block_form, bool persistent, hipStream_t stream, hipEvent_t done) {
    return blur == kBlurRecursive
               ? launch_scale_g<Lay, CosineTaps, Ref>(pairs, work, blocks, parts, block_form, persistent, stream, done)
               : launch_scale_g<Lay, SampledTaps, Ref>(pairs, work, blocks, parts, block_form, persistent, stream, done);
}

template <typename Lay>
hipError_t launch_scale_t(uint32_t blur, MapForm map, const PairDesc* pairs, const WorkRef* work, uint32_t blocks,
                          uint32_t parts, bool block_form, bool persistent, hipStream_t stream, hipEvent_t done) {
    return map == kMapReference
               ? launch_scale_m<Lay, true>(blur, pairs, work, blocks, parts, block_form, persistent, stream, done)
               : launch_scale_m<Lay, false>(blur, pairs, work, blocks, parts, block_form, persistent, stream, done);
}

}  // namespace

hipError_t LaunchCopy(void* dst, const void* src, uint64_t bytes, hipStream_t stream) {
    const uint64_t n = bytes / 16;
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(copy_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream,
                       static_cast<const uint4*>(src), static_cast<uint4*>(dst), n);
    return hipGetLastError();
}

hipError_t LaunchDivCheck(uint32_t mb_first, uint32_t rows, DivCheck* out, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(div_check_kernel, dim3(2048), dim3(256), 0, stream, mb_first, rows, out);
    return hipGetLastError();
}

hipError_t LaunchCbrtCheck(uint32_t first, uint32_t end, CbrtCheck* out, hipStream_t stream) {
    if (end <= first) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((static_cast<uint64_t>(end - first) + 255) / 256, 256 * 64);
    hipLaunchKernelGGL(cbrt_check_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(256), 0, stream, first, end,
                       out);
    return hipGetLastError();
}

hipError_t LaunchPrepare(PlaneFormat format, MapForm map, bool general, const PairDesc* pairs,
                         const WorkRef* work, uint32_t blocks, uint32_t tiles_per_image, const float* lut,
                         const uint8_t* src0, const uint8_t* src1, hipStream_t stream, bool persistent,
                         hipEvent_t done) {
    if (blocks == 0) return Nothing(stream, done);
    if (map > kMapDifference) return hipErrorInvalidValue;
    const uint32_t t = tiles_per_image;
    switch (format) {
        case kPlaneF32:
            return launch_prepare_t<LayoutF32>(map, general, pairs, work, blocks, t, lut, src0, src1, persistent,
                                              stream, done);
        case kPlaneF16:
            return launch_prepare_t<LayoutF16>(map, general, pairs, work, blocks, t, lut, src0, src1, persistent,
                                              stream, done);
        case kPlaneBF16:
            return launch_prepare_t<LayoutBF16>(map, general, pairs, work, blocks, t, lut, src0, src1, persistent,
                                               stream, done);
        case kPlaneU16:
            return launch_prepare_t<LayoutU16>(map, general, pairs, work, blocks, t, lut, src0, src1, persistent,
                                              stream, done);
    }
    return hipErrorInvalidValue;
}

hipError_t LaunchScale(PlaneFormat format, uint32_t blur, MapForm map, const PairDesc* pairs, const WorkRef* work,
                       uint32_t blocks, uint32_t parts_per_pair, bool block_form, hipStream_t stream,
                       bool persistent, hipEvent_t done) {
    if (blocks == 0) return Nothing(stream, done);
    if (block_form && persistent) return hipErrorInvalidValue;
    if (blur > kBlurRecursive || map > kMapDifference) return hipErrorInvalidValue;
    const uint32_t n = parts_per_pair;
    switch (format) {
        case kPlaneF32:
            return launch_scale_t<LayoutF32>(blur, map, pairs, work, blocks, n, block_form, persistent, stream, done);
        case kPlaneF16:
            return launch_scale_t<LayoutF16>(blur, map, pairs, work, blocks, n, block_form, persistent, stream, done);
        case kPlaneBF16:
            return launch_scale_t<LayoutBF16>(blur, map, pairs, work, blocks, n, block_form, persistent, stream, done);
        case kPlaneU16:
            return launch_scale_t<LayoutU16>(blur, map, pairs, work, blocks, n, block_form, persistent, stream, done);
    }
    return hipErrorInvalidValue;
}

hipError_t LaunchReduce(const PairDesc* pairs, uint32_t pairs_count, hipStream_t stream, hipEvent_t done) {
    if (pairs_count == 0) return Nothing(stream, done);
    return InRuns(pairs_count, MaxBlocks(kReduceThreads) / kRanges, [&](uint32_t first, uint32_t n, bool last) {
        return Dispatch(&reduce_kernel, n * kRanges, kReduceThreads, stream, last ? done : nullptr, pairs + first);
    });
}

}  // namespace vqm::ss2
