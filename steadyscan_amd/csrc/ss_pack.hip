// ss_pack.hip -- a frame stack's block matrices on the GPU: the packing of
// estimate_displacements (steady_scan.m:229-234, image2blockmatrix,
// steady_scan.m:601-613) and, after the alignment, which blocks of a frame
// have a masked pixel (steady_scan.m:255).  Both only move, convert or test
// values; memory bound.
#include <algorithm>
#include <type_traits>

#include <hip/hip_runtime.h>

#include "ss_pack.h"

namespace {

using ss::kNoPixel;

// Block-matrix element e (row e % fh of block e / fh) of frame blockIdx.y is
// the raw pixel at[e], or 0 where the block is shorter (kNoPixel).  A block
// lists its pixels column by column, so a wave reads runs of consecutive
// lines and writes consecutive elements; the table stays in the L2s.
template <typename T, typename TO>
__global__ __launch_bounds__(256) void k_pack(const uint32_t *__restrict__ at, int nbm, const T *__restrict__ frames,
                                              size_t rawPix, TO *__restrict__ out) {
    const size_t fo = (size_t)blockIdx.y;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < nbm; e += gridDim.x * 256) {
        const uint32_t p = at[e];
        out[fo * nbm + e] = p != kNoPixel ? (TO)frames[fo * rawPix + p] : (TO)0;
    }
}

// used[c] = 1 when column c of the mask (fh rows) has a nonzero byte: one
// wave per column.
__global__ __launch_bounds__(256) void k_used(const uint8_t *__restrict__ mask, int fh, int cols,
                                              uint8_t *__restrict__ used) {
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (c >= cols) return;
    const uint8_t *m = mask + (size_t)c * fh;
    int any = 0;
    for (int r = lane; r < fh && !__any(any); r += 64) any = m[r];
    any = __any(any);
    if (lane == 0) used[c] = any ? 1 : 0;
}

}  // namespace

namespace ss {

int pack_frames(void *stream, const uint32_t *at, int nbm, int esz, bool toFloat, const void *frames, size_t rawPix, int n,
                void *out) {
    const hipStream_t s = (hipStream_t)stream;
    const int gx = std::min((nbm + 255) / 256, 1024);
    for (int f = 0; f < n; f += 65535) {
        const dim3 grid(gx, std::min(n - f, 65535));
        const char *src = (const char *)frames + rawPix * esz * f;
        char *dst = (char *)out + (size_t)nbm * (toFloat ? sizeof(float) : esz) * f;
        auto launch = [&](auto *from, auto *to) {
            using T = std::remove_pointer_t<decltype(from)>;
            using TO = std::remove_pointer_t<decltype(to)>;
            hipLaunchKernelGGL((k_pack<T, TO>), grid, dim3(256), 0, s, at, nbm, (const T *)src, rawPix, (TO *)dst);
        };
        if (toFloat) launch((double *)nullptr, (float *)nullptr);
        else if (esz == 8) launch((uint64_t *)nullptr, (uint64_t *)nullptr);
        else if (esz == 4) launch((uint32_t *)nullptr, (uint32_t *)nullptr);
        else launch((uint16_t *)nullptr, (uint16_t *)nullptr);
    }
    return (int)hipGetLastError();
}

int used_blocks(void *stream, const uint8_t *mask, int fh, int cols, uint8_t *used) {
    hipLaunchKernelGGL(k_used, dim3((cols + 3) / 4), dim3(256), 0, (hipStream_t)stream, mask, fh, cols, used);
    return (int)hipGetLastError();
}

}  // namespace ss
