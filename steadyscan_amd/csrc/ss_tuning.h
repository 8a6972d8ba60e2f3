// ss_tuning.h -- launch variants of the pixel kernels, per pixel precision.
//
// Each of the assembly, line-search and correlation kernels is built in
// kVariants variants of (samples, waves):
//   samples: template samples a thread keeps in flight (the unrolled chunk
//            of rows times the samples per row; a power of two),
//   waves:   minimum waves per SIMD that the kernel's register allocation
//            must allow (more waves hide more gather latency; fewer
//            registers limit how many gathers a wave keeps in flight).
// Variant 0 is the default: the values measured fastest on MI355X for batches
// of 512x512 groups (1000 x 512x512 uint16 in FP64: line search 36.6 ms with
// 4 samples at 5 waves against 46.0 at 4 waves and 40.0 with 8 samples at 3;
// correlation, then in two passes, 10.4 against 11.8 with 8 samples at 3 waves; assembly 20.6
// against 21.2 at 3 waves.  24 uneven groups in FP32: line search 36.3 ms with
// 4 samples at 5 waves against 37.9 with 8 at 4, correlation 8.7 against 9.4).
// One 512x512 group of 50 frames, which does not fill the chip, measures the
// same order.
// The engine's autotuner (off unless asked for) times all variants on a
// group shape's first tick and keeps the fastest per kernel.
// A variant only changes how many rows a thread unrolls and how registers
// are allocated: every thread still accumulates its pixels in the same
// order, so all variants give the same results bit for bit.
#pragma once

namespace ss {

constexpr int kVariants = 3;
enum TuneKernel { TK_ASSEMBLE = 0, TK_LS = 1, TK_CORR = 2, TK_COUNT = 3 };

struct TuneVariant {
    int samples, waves;
};

// [kernel][fp64][variant]
constexpr TuneVariant kTuneTable[TK_COUNT][2][kVariants] = {
    // assembly: FP32, FP64
    {{{8, 4}, {4, 4}, {4, 5}}, {{4, 4}, {4, 3}, {2, 4}}},
    // line search
    {{{4, 5}, {8, 4}, {4, 4}}, {{4, 5}, {8, 3}, {4, 4}}},
    // correlation (one sample per row; a chunk holds at most 8 rows)
    {{{4, 5}, {8, 4}, {4, 6}}, {{4, 4}, {8, 3}, {2, 4}}},
};

template <int KERNEL, typename R, int V>
__host__ __device__ constexpr TuneVariant tune_variant() {
    return kTuneTable[KERNEL][sizeof(R) == 8 ? 1 : 0][V];
}

// the final pass runs once per group: one variant
constexpr int kFinalSamplesF32 = 4, kFinalWavesF32 = 4, kFinalSamplesF64 = 4, kFinalWavesF64 = 4;

}  // namespace ss
