// ss_prefilter.hip -- the frame preparation and gap filling of steady_scan.m:
// prefilter_foralignment (steady_scan.m:625-643) and imgapfill_leastsquares
// (steady_scan.m:525-560).
//
// prefilter_foralignment blurs each frame with a Gaussian through 2-D FFTs of
// the frame, zero-padded by L pixels on the far sides, and of a wrapped
// Gaussian on the padded grid: a circular convolution.  The wrapped Gaussian
// is separable, g2d(y, x) = g1(y) g2(x) with each factor normalised, so the
// convolution is two circulant matrix products restricted to the H x W
// output: T = C1 D over the rows and U = T C2^T over the columns, in FP64.
// Up to kBlurRadius taps on each side both run in one sweep over the frame
// (k_blur), which leaves out taps below 2^-64 of the centre one; wider kernels,
// frames so small that a wide kernel's taps outnumber their pixels, and frames
// with an infinity run as FP64 tiled GEMMs whose circulant operand is generated
// from g1/g2 on the fly.  Both agree with the FFT to FP64 rounding of the
// frame's largest value.  Of a pixel that lies a factor of 2^60 or more below
// its neighbours only the GEMMs' result holds the far taps' terms.
// The result takes the input's class (integer frames: rounded half away
// from zero and saturated, NaN to 0).  Median normalisation divides each
// frame by its median, found exactly by an 8-pass radix select on the
// order-preserving 64-bit keys of the values.
//
// imgapfill_leastsquares fills the NaN pixels of each frame with the
// minimiser of the summed squared adjacent differences, the known pixels
// fixed: the Dirichlet Laplacian system  deg_i c_i - sum_{missing j~i} c_j =
// sum_{known j~i} a_j  over the missing pixels.  The reference solves it with
// a sparse direct solve; here one workgroup per frame runs conjugate
// gradients in FP64 to a relative residual of 1e-13, with every reduction in
// a fixed order (deterministic).
#include <algorithm>
#include <new>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include <hip/hip_runtime.h>

#include "ss_host.h"
#include "steadyscan.h"

namespace {

constexpr int TM = 64, TN = 64, TK = 16;
// FP64 planes of the frames that the sweep hands to the GEMMs: 32 frames of
// 512x512, 2048 workgroups a launch
constexpr size_t kPlaneBytes = (size_t)64 << 20;
// most frames of a launch whose flags are cleared by the tables' upload
constexpr int kFlagsInTab = 1024;
constexpr int kCgThreads = 1024;

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Assignment of a double into an array of class T (MATLAB's conversion).
template <typename T> __device__ inline T to_class(double v);
template <> __device__ inline double to_class<double>(double v) { return v; }
template <> __device__ inline float to_class<float>(double v) { return (float)v; }
template <> __device__ inline uint16_t to_class<uint16_t>(double v) {
    if (isnan(v)) return 0;
    v = round(v);  // half away from zero
    return (uint16_t)fmin(fmax(v, 0.0), 65535.0);
}
template <> __device__ inline int16_t to_class<int16_t>(double v) {
    if (isnan(v)) return 0;
    v = round(v);
    return (int16_t)fmin(fmax(v, -32768.0), 32767.0);
}

// ---------------------------------------------------------------------------
// blur: both factors of the separable circular convolution in one sweep
// ---------------------------------------------------------------------------
constexpr int kBadNan = 1, kBadInf = 2;

constexpr int kBlurRadius = 64;  // most taps on each side of the centre
constexpr int kBlurRows = 64, kBlurCols = 32, kBlurOut = 8;
constexpr int kBlurMid = kBlurRows + 1;  // doubles per ring column: neighbouring columns in different banks
constexpr int kBlurThreads = 256;
constexpr int kBlurRowLoads = (kBlurRows + 2 * kBlurRadius + 63) / 64;

// the taps, which no kernel writes, come by scalar loads
#define SS_CONST __attribute__((address_space(4)))
// device memory behind a pointer of a struct: global instead of flat loads
#define SS_GLOBAL __attribute__((address_space(1)))

// One axis: the tap at distance d (dlo <= d <= dhi, every residue mod S at
// most once) is g[d - dlo + kBlurOut - 1]; kBlurOut - 1 zeros stand on both
// sides, and more at the end, so that the unrolled loop needs no tests.
struct BlurAxis {
    int n, S, dlo, dhi;  // pixels, padded period, tap range
    int steps;           // inputs the unrolled loop of kBlurOut outputs reads (a multiple of kBlurOut)
    const double *g;
};

// dst = the blurred frame, both as the class's values.  A workgroup takes 64
// rows (consecutive in memory) of a frame and sweeps a segment of its
// columns: 32 columns at a time are loaded with the rows' halo into LDS as
// doubles, convolved along the rows into a ring of columns, and the 32
// columns whose taps the ring now covers are convolved along x and stored.
// A thread makes 8 outputs of one line, so that a value read from LDS feeds
// 8 multiply-adds (the LDS returns one wave's doubles in the time of four
// multiply-adds per SIMD); the taps are wave-uniform and come through the
// scalar cache.  A frame is read once, plus the halo rows of each strip
// (through L2), and written once.  bad[f] reports a frame with a NaN (kBadNan)
// or an infinity (kBadInf), which the full convolution spreads over the whole
// frame, and *anyBad, in host memory, that there is one.
// Bound by the multiply-adds and LDS reads: 500 x 512x512 uint16 take 0.60 ms
// at sigma 1 (9 taps a side; 1.06 ms without the loads a step ahead, 1.46
// with the taps through vector loads) and 3.4 ms at sigma 6.8 (64 taps a side), where
// the two GEMMs take 8.6 ms for any sigma.  The LDS (132 KB at 64 taps a side)
// sets kBlurRadius.
template <typename T>
__global__ __launch_bounds__(kBlurThreads) void k_blur(const T *__restrict__ src, T *__restrict__ dst, BlurAxis Y,
                                                       BlurAxis X, int segCols, int ring, int *__restrict__ bad,
                                                       int *__restrict__ anyBad) {
    extern __shared__ double lds[];
    const int rowsIn = kBlurRows - kBlurOut + Y.steps;  // rows of a loaded column, with the loop's padding
    const int strideIn = rowsIn | 1;                    // odd: columns start in different banks
    double *in = lds, *mid = lds + kBlurCols * strideIn;
    const int H = Y.n, W = X.n;
    const size_t fo = (size_t)blockIdx.y * H * W;
    const T *s = src + fo;
    T *d = dst + fo;
    const int y0 = blockIdx.x * kBlurRows;
    const int x0 = blockIdx.z * segCols, x1 = min(W, x0 + segCols);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int i = tid; i < ring * kBlurMid; i += kBlurThreads) mid[i] = 0.0;
    const int rowsUsed = kBlurRows + Y.dhi - Y.dlo;
    int next = x0 + X.dlo, slot = 0;  // next virtual column of the ring and where it goes
    int first = 0;                    // slot of virtual column x + X.dlo of the outputs at x
    bool finite = true;
    // A step's columns are loaded into registers one step ahead, while the
    // step before is convolved: wave w holds columns w, w + 4, ..., rows lane,
    // lane + 64, ...  Virtual rows and columns wrap at the padded period; the
    // padding is 0.
    constexpr int kColsPerWave = kBlurCols / (kBlurThreads / 64);
    T pre[kColsPerWave][kBlurRowLoads];
    auto fetch = [&](int col, int count) {
#pragma unroll
        for (int k = 0; k < kColsPerWave; k++) {
            const int c = wave + k * (kBlurThreads / 64);
            int cx = (col + c) % X.S;
            cx += cx < 0 ? X.S : 0;
#pragma unroll
            for (int m = 0; m < kBlurRowLoads; m++) {
                const int r = lane + 64 * m;
                int ry = y0 + Y.dlo + r;
                ry += ry < 0 ? Y.S : 0;
                ry -= ry >= Y.S ? Y.S : 0;
                pre[k][m] = (T)0;
                if (c < count && cx < W && r < rowsUsed && ry < H) pre[k][m] = s[(size_t)cx * H + ry];
            }
        }
    };
    // the first step takes what leaves whole blocks of columns for the others
    const int last = x1 + X.dhi;  // one past the last virtual column
    int nc = (min(kBlurCols, x1 - x0) + X.dhi - X.dlo - 1) % kBlurCols + 1;
    fetch(next, nc);
    for (int x = x0; x < x1; x += kBlurCols) {
        const int need = min(x + kBlurCols, x1) + X.dhi;
        while (next < need) {
#pragma unroll
            for (int k = 0; k < kColsPerWave; k++)
#pragma unroll
                for (int m = 0; m < kBlurRowLoads; m++) {
                    const int r = lane + 64 * m;
                    const double v = (double)pre[k][m];
                    if constexpr (std::is_floating_point<T>::value) finite = finite && isfinite(v);
                    if (r < rowsIn) in[(wave + k * (kBlurThreads / 64)) * strideIn + r] = v;
                }
            __syncthreads();
            const int now = nc;
            nc = min(kBlurCols, last - next - now);
            if (nc > 0) fetch(next + now, nc);
            // along the rows: thread = column (tid & 31), 8 rows (tid >> 5)
            {
                const int c = tid & (kBlurCols - 1), r0 = (tid / kBlurCols) * kBlurOut;
                const double *q = in + c * strideIn + r0;
                double acc[kBlurOut] = {};
                for (int i = 0; i < Y.steps; i += kBlurOut) {
                    const SS_CONST double *g = (const SS_CONST double *)Y.g + i;
#pragma unroll
                    for (int u = 0; u < kBlurOut; u++) {
                        const double v = q[i + u];
#pragma unroll
                        for (int j = 0; j < kBlurOut; j++) acc[j] = fma(g[kBlurOut - 1 + u - j], v, acc[j]);
                    }
                }
                if (c < now) {
                    int sl = slot + c;
                    sl -= sl >= ring ? ring : 0;
                    double *m = mid + sl * kBlurMid + r0;
#pragma unroll
                    for (int j = 0; j < kBlurOut; j++) m[j] = acc[j];
                }
            }
            __syncthreads();
            next += now;
            slot += now;
            slot -= slot >= ring ? ring : 0;
        }
        // along x: wave w makes columns x + 8 w .. + 7 of row y0 + lane
        {
            const int xo = wave * kBlurOut;
            int sl = first + xo;
            sl -= sl >= ring ? ring : 0;
            double acc[kBlurOut] = {};
            for (int i = 0; i < X.steps; i += kBlurOut) {
                const SS_CONST double *g = (const SS_CONST double *)X.g + i;
#pragma unroll
                for (int u = 0; u < kBlurOut; u++) {
                    const double v = mid[sl * kBlurMid + lane];
                    sl = sl + 1 == ring ? 0 : sl + 1;
#pragma unroll
                    for (int j = 0; j < kBlurOut; j++) acc[j] = fma(g[kBlurOut - 1 + u - j], v, acc[j]);
                }
            }
            const int y = y0 + lane;
            if (y < H) {
#pragma unroll
                for (int j = 0; j < kBlurOut; j++)
                    if (x + xo + j < x1) d[(size_t)(x + xo + j) * H + y] = to_class<T>(acc[j]);
            }
        }
        first += kBlurCols;
        first -= first >= ring ? ring : 0;
        __syncthreads();
    }
    // which kind, in a second look at the workgroup's own pixels: told apart in
    // the loop, frames without any lose 10% at 56 taps a side
    if constexpr (std::is_floating_point<T>::value) {
        if (__syncthreads_or(!finite)) {
            int kind = 0;
            for (int x = x0 + wave; x < x1; x += kBlurThreads / 64) {
                const double v = y0 + lane < H ? (double)s[(size_t)x * H + y0 + lane] : 0.0;
                kind |= isnan(v) ? kBadNan : isinf(v) ? kBadInf : 0;
            }
            if (kind) {
                atomicOr(&bad[blockIdx.y], kind);
                *anyBad = 1;
            }
        }
    }
}

// The taps of one axis: g1[j] at circular distance j (0 <= j < S) of a period
// of S; the radius keeps every tap of at least 2^-64 of the centre one.
// False if that takes more than kBlurRadius taps on a side.
bool blur_taps(const std::vector<double> &g1, int n, BlurAxis &A, std::vector<double> &taps) {
    const int S = (int)g1.size();
    int r = 0;
    for (int j = 1; j <= S / 2; j++)
        if (g1[j] >= std::ldexp(g1[0], -64)) r = j;
    if (r > kBlurRadius) return false;
    A.n = n;
    A.S = S;
    A.dhi = r;
    A.dlo = -std::min(r, (S - 1) / 2);
    const int nd = A.dhi - A.dlo + 1;
    A.steps = (nd + kBlurOut - 1 + kBlurOut - 1) / kBlurOut * kBlurOut;
    taps.assign(A.steps + kBlurOut, 0.0);
    for (int d = A.dlo; d <= A.dhi; d++) taps[d - A.dlo + kBlurOut - 1] = g1[d < 0 ? d + S : d];
    return true;
}

// Whether the sweep makes no more multiply-adds for a frame than the GEMMs,
// the padding of both included: a wide kernel's taps go round a small frame's
// padded period and outnumber its pixels.  512 uint16 frames, sweep and GEMMs
// (ratio of the multiply-adds): 48x48 at sigma 2 (1.4) 53 and 55 us, at sigma 6
// (2.9) 94 and 56; 100x100 at sigma 4 (1.1) 225 and 156; 129x129 at sigma 4
// (0.7) 367 and 322; 256 of 256x256 at sigma 6.7 (0.7) 519 and 586.  Few
// frames favour the sweep, which is one launch: 8 of 200x48 at sigma 4 (1.2) 53
// and 66 us, 512 of them 239 and 159.  The number of frames is left out all
// the same, so that a frame's result does not depend on its stack.
bool blur_by_sweep(const BlurAxis &Y, const BlurAxis &X) {
    auto whole = [](double n, double tile) { return std::ceil(n / tile) * tile; };
    const double rows = whole(Y.n, kBlurRows);
    const double sweep = rows * (whole(X.n + X.dhi - X.dlo, kBlurCols) * Y.steps + whole(X.n, kBlurCols) * X.steps);
    const double gemms = rows * ((double)X.n * whole(Y.n, TK) + whole(X.n, TN) * whole(X.n, TK));
    return sweep <= gemms;
}

// The sweep's LDS, and the columns of its ring.
size_t blur_lds(const BlurAxis &Y, const BlurAxis &X, int &ring) {
    ring = X.dhi - X.dlo + kBlurCols;
    return 8 * ((size_t)kBlurCols * ((kBlurRows - kBlurOut + Y.steps) | 1) + (size_t)ring * kBlurMid);
}

// Columns of a workgroup's segment, for `strips` strips of rows: a strip may
// be cut into segments of whole column blocks, each of which makes the
// ring's columns before its own again, where that fills the chip.  Taken is
// the least of a segment's multiply-adds times the workgroups that a CU's LDS
// has to take one after the other (and a fifth for those of a launch that
// does not fill the chip).  Cut to 4 workgroups a CU whatever the LDS holds, wide kernels made
// their columns several times: 8 x 512x512 uint16, sigma 6, 186 -> 113 us;
// 64 x 160x160, 178 -> 114 us.
int blur_segment(const BlurAxis &Y, const BlurAxis &X, size_t strips, size_t lds) {
    constexpr size_t kCus = 256, kLdsOfCu = 160 << 10;
    auto whole = [](size_t c) { return (c + kBlurCols - 1) / kBlurCols * kBlurCols; };
    const size_t perCu = std::max<size_t>(1, std::min<size_t>(4, kLdsOfCu / lds));
    const size_t blocks = whole(X.n) / kBlurCols, most = std::min(blocks, std::max<size_t>(1, 4 * kCus / strips));
    size_t best = 0, bestCost = 0;
    for (size_t q = 1; q <= most; q++) {
        const size_t cols = (blocks + q - 1) / q * kBlurCols, used = std::min<size_t>(cols, X.n);
        const size_t work = whole(used + X.dhi - X.dlo) * Y.steps + whole(used) * X.steps;
        const size_t groups = strips * ((X.n + cols - 1) / cols), rounds = (groups + kCus * perCu - 1) / (kCus * perCu);
        const size_t cost = work * (5 * rounds + 1);
        if (!best || cost < bestCost) {
            best = cols;
            bestCost = cost;
        }
    }
    return (int)best;
}

// ---------------------------------------------------------------------------
// the same convolution as GEMMs, for wider kernels, small frames and frames
// with an infinity
// ---------------------------------------------------------------------------
// C(y, x) = sum_k A(y, k) B(k, x), 64 x 64 tile per workgroup, 4 x 4 per thread.
// MODE 0, the frames' columns side by side: A(y, k) = g[(y - k) mod S]
//         (generated), B = src, the class's values (frame f's at listed
//         place list[f]), C = dst, consecutive FP64 planes; M = H, N = W * nf,
//         K = H.
// MODE 1, frame blockIdx.z: A = src, its FP64 plane, B(k, x) = g[(x - k) mod S]
//         (generated), C = dst, the class's values (at its listed place);
//         M = H, N = W, K = W.
// The frames are converted where they are read and written: 8 frames of
// 48x48 take 50 us a call in two launches, 57 us in four.
__device__ __forceinline__ size_t frame_of(const int *list, int f) { return list ? list[f] : f; }

template <int MODE, typename TI, typename TO>
__global__ __launch_bounds__(256) void k_circ_gemm(const TI *__restrict__ src, TO *__restrict__ dst,
                                                   const int *__restrict__ list, const double *__restrict__ g, int S,
                                                   int H, int W, int ncols) {
    __shared__ double As[TK][TM + 1];
    __shared__ double Bs[TK][TN + 1];
    const int M = H;
    const int N = MODE == 0 ? ncols : W;
    const int K = MODE == 0 ? H : W;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
    // the thread's columns of B (MODE 0) or the frame (MODE 1)
    const TI *s[4];
    for (int e = 0; e < 4; e++) {
        const int x = min(n0 + (tid + 256 * e) / TK, N - 1), f = MODE == 0 ? x / W : (int)blockIdx.z;
        s[e] = MODE == 0 ? src + (frame_of(list, f) * W + (x - f * W)) * H : src + (size_t)f * H * W;
    }
    TO *d = MODE == 0 ? dst : dst + frame_of(list, blockIdx.z) * H * W;
    auto tap = [&](int at) { return g[at < 0 ? at + S : at]; };
    // a step's operands are loaded into registers while the step before is computed
    double ra[4], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = tid + 256 * e;
            const int y = m0 + idx % TM, ka = k0 + idx / TM, x = n0 + idx / TK, kb = k0 + idx % TK;
            ra[e] = rb[e] = 0.0;
            if (y < M && ka < K) ra[e] = MODE == 0 ? tap(y - ka) : (double)s[0][(size_t)ka * H + y];
            if (x < N && kb < K) rb[e] = MODE == 0 ? (double)s[e][kb] : tap(x - kb);
        }
    };
    double acc[4][4] = {};
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = tid + 256 * e;
            As[idx / TM][idx % TM] = ra[e];
            Bs[idx % TK][idx / TK] = rb[e];
        }
        __syncthreads();
        if (k0 + TK < K) fetch(k0 + TK);
#pragma unroll
        for (int kk = 0; kk < TK; kk++) {
            double a[4], b[4];
            for (int i = 0; i < 4; i++) a[i] = As[kk][ty + 16 * i];
            for (int j = 0; j < 4; j++) b[j] = Bs[kk][tx + 16 * j];
            for (int i = 0; i < 4; i++)
                for (int j = 0; j < 4; j++) acc[i][j] += a[i] * b[j];
        }
        __syncthreads();
    }
    for (int i = 0; i < 4; i++)
        for (int j = 0; j < 4; j++) {
            const int y = m0 + ty + 16 * i, x = n0 + tx + 16 * j;
            if (y < M && x < N) {
                if constexpr (MODE == 0) d[(size_t)x * H + y] = acc[i][j];
                else d[(size_t)x * H + y] = to_class<TO>(acc[i][j]);
            }
        }
}

template <typename T>
__global__ __launch_bounds__(256) void k_set_nan(T *__restrict__ out, const int *__restrict__ list, size_t np) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < np) out[list[blockIdx.y] * np + i] = (T)__builtin_nan("");
}

__device__ inline unsigned long long order_key(double v) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return (b >> 63) ? ~b : (b | (1ull << 63));
}

__device__ inline double key_value(unsigned long long k) {
    const unsigned long long b = (k >> 63) ? (k & ~(1ull << 63)) : ~k;
    return __longlong_as_double((long long)b);
}

// The rank-th smallest value of the frame (all threads of the workgroup call it).
template <typename T>
__device__ double select_rank(const T *v, int np, int rank, int *hist, unsigned long long *s_prefix,
                              int *s_rank) {
    unsigned long long prefix = 0, pmask = 0;
    for (int pass = 0; pass < 8; pass++) {
        const int shift = 56 - 8 * pass;
        for (int b = threadIdx.x; b < 256; b += blockDim.x) hist[b] = 0;
        __syncthreads();
        for (int i = threadIdx.x; i < np; i += blockDim.x) {
            const unsigned long long k = order_key((double)v[i]);
            if ((k & pmask) == prefix) atomicAdd(&hist[(k >> shift) & 255], 1);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            int acc = 0, d = 0;
            for (d = 0; d < 256; d++) {
                if (acc + hist[d] > rank) break;
                acc += hist[d];
            }
            if (d > 255) d = 255;
            *s_rank = rank - acc;
            *s_prefix = prefix | ((unsigned long long)d << shift);
        }
        __syncthreads();
        rank = *s_rank;
        prefix = *s_prefix;
        pmask |= 255ull << shift;
        __syncthreads();
    }
    return key_value(prefix);
}

// MATLAB median of each frame (NaN if the frame holds a NaN), then the
// division data ./ median in the class's arithmetic.
template <typename T>
__global__ __launch_bounds__(1024) void k_median_divide(T *__restrict__ data, const int *__restrict__ list, int np) {
    __shared__ int hist[256];
    __shared__ unsigned long long s_prefix;
    __shared__ int s_rank, s_nan;
    T *v = data + frame_of(list, blockIdx.x) * np;
    if (threadIdx.x == 0) s_nan = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < np; i += blockDim.x)
        if (isnan((double)v[i])) atomicOr(&s_nan, 1);
    __syncthreads();
    T med;
    if (s_nan) {
        med = (T)__builtin_nan("");
    } else if (np % 2) {
        med = (T)select_rank(v, np, np / 2, hist, &s_prefix, &s_rank);
    } else {
        const T a = (T)select_rank(v, np, np / 2 - 1, hist, &s_prefix, &s_rank);
        const T b = (T)select_rank(v, np, np / 2, hist, &s_prefix, &s_rank);
        med = (T)((a + b) / (T)2);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < np; i += blockDim.x) v[i] = v[i] / med;
}

// ---------------------------------------------------------------------------
// gap filling
// ---------------------------------------------------------------------------
struct FillChunk {
    int th, tw, np;
    int *list;             // B x np: missing pixels, ascending
    int *map;              // B x np: compact index of each missing pixel
    int *nmiss;            // B
    uint2 *code;           // B x np (the first nmiss used, as below): an entry's W and E neighbours,
    uint8_t *meta;         // its degree and whether N and S are missing
    double *x, *r, *p;     // solution, residual and search direction of the entries past the LDS
    int *status;           // B: iterations, or -1 if not converged
    int maxit;
};

// A missing pixel's system: the sum of its known neighbours and its degree
// (in-image neighbours), W N S E (ascending index), the compact indices of
// missing W and E neighbours and whether N and S are missing (entries m - 1
// and m + 1).
constexpr unsigned kAbsent = ~0u;
struct FillEntry {
    double known;
    unsigned deg, w, e;
    bool n, s;
};
template <typename T>
__device__ __forceinline__ FillEntry fill_entry(const T *a, const int *map, int i, int th, int tw) {
#pragma clang fp contract(off)
    FillEntry q{0.0, 0, kAbsent, kAbsent, false, false};
    const int col = i / th, row = i - col * th;
    if (col > 0) {
        const double v = (double)a[i - th];
        q.deg++;
        if (isnan(v)) q.w = (unsigned)map[i - th];
        else q.known += v;
    }
    if (row > 0) {
        const double v = (double)a[i - 1];
        q.deg++;
        q.n = isnan(v);
        if (!q.n) q.known += v;
    }
    if (row + 1 < th) {
        const double v = (double)a[i + 1];
        q.deg++;
        q.s = isnan(v);
        if (!q.s) q.known += v;
    }
    if (col + 1 < tw) {
        const double v = (double)a[i + th];
        q.deg++;
        if (isnan(v)) q.e = (unsigned)map[i + th];
        else q.known += v;
    }
    return q;
}

// The missing (NaN) pixels of a frame in ascending order, and their count:
// tiles of 4 * kCgThreads pixels, 4 consecutive ones per thread, a wave
// scan by shuffles and the wave totals through LDS.
template <typename T>
__global__ __launch_bounds__(kCgThreads) void k_fill_list(FillChunk C, const T *__restrict__ data) {
    constexpr int kW = kCgThreads / 64;
    __shared__ int wsum[kW];
    const int f = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
    const T *a = data + (size_t)f * C.np;
    int *list = C.list + (size_t)f * C.np;
    const int np = C.np;
    int carry = 0;
    for (int base = 0; base < np; base += 4 * kCgThreads) {
        const int i0 = base + 4 * t;
        bool miss[4];
        int own = 0;
        for (int q = 0; q < 4; q++) {
            miss[q] = i0 + q < np && isnan(a[i0 + q]);
            own += miss[q] ? 1 : 0;
        }
        int incl = own;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(incl, off, 64);
            if (lane >= off) incl += y;
        }
        if (lane == 63) wsum[w] = incl;
        __syncthreads();
        int before = 0, tile = 0;
        for (int k = 0; k < kW; k++) {
            const int ws = wsum[k];
            if (k < w) before += ws;
            tile += ws;
        }
        int pos = carry + before + incl - own;
        for (int q = 0; q < 4; q++)
            if (miss[q]) list[pos++] = i0 + q;
        carry += tile;
        __syncthreads();
    }
    if (t == 0) C.nmiss[f] = carry;
}

// Sum over the workgroup of one value per thread: a butterfly in each wave,
// then the 16 wave sums in order.  sp alternates between two buffers from
// call to call, so that one barrier a call is enough.
__device__ __forceinline__ double block_sum(double v, double *sp) {
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < kCgThreads / 64; w++) r += sp[w];
    return r;
}

// Conjugate gradients of a frame in compact form (entry m = the m-th missing
// pixel), one workgroup per frame.  The search direction p takes the
// workgroup's LDS, and thread t keeps the solution and the residual of its
// entries t, t + 1024, ... in registers.  A missing N or S neighbour is entry
// m - 1 or m + 1; the compact indices of W and E (15 bits each) and the two
// flags fill one word.  An absent neighbour reads the zero after the last
// entry, and entries past n hold zeros.  Dot products add every thread's
// entries in order, then the threads as block_sum does.
// Bound by the 10 LDS reads per entry and iteration and by the barriers of
// the two reductions.  128 x 512x512 frames with up to 18300 missing pixels
// and 546 iterations take 5.8 ms (6.0 with one loop for all lengths); with the
// residual in LDS too, which held 8192 entries and left larger frames to a
// kernel in global memory, 25 ms.
constexpr int kFillK = 19;
constexpr int kFillLds = kFillK * kCgThreads;
constexpr unsigned kNoNbr = 0x7fffu, kHasN = 1u << 30, kHasS = 1u << 31;
static_assert(kFillLds < (int)kNoNbr, "compact indices take 15 bits");

// The entries of frame f: neighbours and right-hand side (put(m, known) takes
// the latter); returns the thread's part of its square.
template <typename T, typename Put>
__device__ __forceinline__ double fill_setup(const FillChunk &C, const T *a, size_t fo, int n, Put &&put) {
#pragma clang fp contract(off)
    const SS_GLOBAL int *list = (const SS_GLOBAL int *)C.list + fo;
    int *map = C.map + fo;
    SS_GLOBAL uint32_t *code = (SS_GLOBAL uint32_t *)(C.code + fo);
    SS_GLOBAL uint8_t *meta = (SS_GLOBAL uint8_t *)C.meta + fo;
    for (int m = threadIdx.x; m < n; m += kCgThreads) map[list[m]] = m;
    __syncthreads();
    double part = 0.0;
    for (int m = threadIdx.x; m < n; m += kCgThreads) {
        const FillEntry q = fill_entry(a, map, list[m], C.th, C.tw);
        code[2 * (size_t)m] = q.w;
        code[2 * (size_t)m + 1] = q.e;
        meta[m] = (uint8_t)(q.deg | (q.n ? 8 : 0) | (q.s ? 16 : 0));
        put(m, q.known);
        part += q.known * q.known;
    }
    return part;
}

using Partials = double[kCgThreads / 64];

// K: the most entries a thread has, kFillK or fewer.
template <int K, typename T>
__device__ __forceinline__ void fill_cg_lds(const FillChunk &C, T *__restrict__ data, Partials *sp, double *lp) {
#pragma clang fp contract(off)
    const int f = blockIdx.x, t = threadIdx.x, np = C.np;
    const size_t fo = (size_t)f * np;
    T *a = data + fo;
    const SS_GLOBAL int *list = (const SS_GLOBAL int *)C.list + fo;
    const int n = C.nmiss[f];
    const int nk = (n + kCgThreads - 1) / kCgThreads;
    for (int m = n + t; m < nk * kCgThreads; m += kCgThreads) lp[m] = 0.0;
    if (t == 0) lp[kFillLds] = 0.0;
    double part = fill_setup(C, a, fo, n, [&](int m, double known) { lp[m] = known; });
    const SS_GLOBAL uint32_t *code = (const SS_GLOBAL uint32_t *)(C.code + fo);
    const SS_GLOBAL uint8_t *meta = (const SS_GLOBAL uint8_t *)C.meta + fo;
    double r[K], x[K];
    unsigned nb[K], deg[(K + 9) / 10] = {};  // deg: 3 bits per entry
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int m = t + k * kCgThreads;
        x[k] = r[k] = 0.0;
        nb[k] = kNoNbr | (kNoNbr << 15);
        if (m < n) {
            r[k] = lp[m];
            const unsigned w = code[2 * (size_t)m], e = code[2 * (size_t)m + 1], q = meta[m];
            nb[k] = min(w, kNoNbr) | (min(e, kNoNbr) << 15) | ((q & 8) ? kHasN : 0) | ((q & 16) ? kHasS : 0);
            deg[k / 10] |= (q & 7) << (3 * (k % 10));
        }
    }
    // (A p)_m of entry k, p_m in p.  The word is opaque here: unpacked ahead
    // of the loop its indices would take four registers per entry.
    auto apply = [&](int k, double &p) {
        const int m = t + k * kCgThreads;
        unsigned c = nb[k], d = deg[k / 10];
        asm volatile("" : "+v"(c), "+v"(d));
        const unsigned w = min(c & kNoNbr, (unsigned)kFillLds), e = min((c >> 15) & kNoNbr, (unsigned)kFillLds);
        const unsigned no = (c & kHasN) ? m - 1 : kFillLds, so = (c & kHasS) ? m + 1 : kFillLds;
        p = lp[m];
        double s = 0.0;
        s += lp[w];
        s += lp[no];
        s += lp[so];
        s += lp[e];
        return (double)((d >> (3 * (k % 10))) & 7u) * p - s;
    };
    double rr_ = block_sum(part, sp[0]);  // also orders the direction's writes before the reads
    const double tol2 = 1e-26 * rr_;
    int it = 0;
    // nk, opaque in each phase: kept over the loop, the K tests' results would
    // spill scalar registers (256 frames of 12000 missing pixels 4.65 -> 4.29 ms)
    auto entries = [nk] {
        int v = nk;
        asm volatile("" : "+s"(v));
        return v;
    };
    bool ok = rr_ <= tol2;
    while (!ok && it < C.maxit) {
        it++;
        part = 0.0;
        int nk_ = entries();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (K == 1 || k < nk_) {
                double p;
                const double ap = apply(k, p);
                part += p * ap;
            }
        }
        const double pap = block_sum(part, sp[1]);
        const double alpha = rr_ / pap;
        part = 0.0;
        nk_ = entries();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (K == 1 || k < nk_) {
                double p;
                const double ap = apply(k, p);
                x[k] += alpha * p;
                r[k] -= alpha * ap;
                part += r[k] * r[k];
            }
        }
        const double rn = block_sum(part, sp[0]);  // also orders these reads of p before its writes
        if (rn <= tol2) {
            ok = true;
            break;
        }
        const double beta = rn / rr_;
        rr_ = rn;
        nk_ = entries();
#pragma unroll
        for (int k = 0; k < K; k++) {
            if (K == 1 || k < nk_) {
                const int m = t + k * kCgThreads;
                lp[m] = r[k] + beta * lp[m];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int m = t + k * kCgThreads;
        if (m < n) a[list[m]] = to_class<T>(x[k]);
    }
    if (t == 0) C.status[f] = ok ? it : -1;
}

// The same for larger regions: p of the first kFillLds entries in LDS, the
// rest of it and the other vectors in global memory, at one CU's latency and
// bandwidth: 58 bytes per entry and iteration (neighbours, degree and flags
// twice 9, the solution 16, the residual 24), 32 more for the direction of an
// entry past the LDS, and its neighbours'.  128 frames of which the largest
// misses 20400 pixels take 14 ms; 29 ms through generic pointers with p on the
// image grid.
template <typename T>
__device__ __forceinline__ void fill_cg_stream(const FillChunk &C, T *__restrict__ data, Partials *sp, double *lp) {
#pragma clang fp contract(off)
    const int f = blockIdx.x, t = threadIdx.x, np = C.np;
    const size_t fo = (size_t)f * np;
    T *a = data + fo;
    const SS_GLOBAL int *list = (const SS_GLOBAL int *)C.list + fo;
    const int n = C.nmiss[f];
    const SS_GLOBAL uint32_t *code = (const SS_GLOBAL uint32_t *)(C.code + fo);
    const SS_GLOBAL uint8_t *meta = (const SS_GLOBAL uint8_t *)C.meta + fo;
    SS_GLOBAL double *x = (SS_GLOBAL double *)C.x + fo, *r = (SS_GLOBAL double *)C.r + fo,
                     *gp = (SS_GLOBAL double *)C.p + fo;
    double part = fill_setup(C, a, fo, n, [&](int m, double known) {
        x[m] = 0.0;
        r[m] = known;
        if (m < kFillLds) lp[m] = known;
        else gp[m] = known;
    });
    // Entries [m0, m1) of this thread, four at a time: all loads of the four
    // first, p from LDS where the index lies there.
    auto near = [&](unsigned i) { return lp[min(i, (unsigned)kFillLds - 1)]; };
    auto passes = [&](auto &&body) {
        for (int m0 = t; m0 < n; m0 += 4 * kCgThreads) {
            unsigned w[4], e[4], q[4];
            double p[4], vw[4], vn[4], vs[4], ve[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int m = min(m0 + u * kCgThreads, n - 1);
                w[u] = code[2 * (size_t)m];
                e[u] = code[2 * (size_t)m + 1];
                q[u] = meta[m];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const unsigned m = min(m0 + u * kCgThreads, n - 1);
                p[u] = near(m);
                vw[u] = near(w[u]);
                vn[u] = near(m - 1);
                vs[u] = near(m + 1);
                ve[u] = near(e[u]);
                if (m >= (unsigned)kFillLds) p[u] = gp[m];
                if (m > (unsigned)kFillLds) vn[u] = gp[m - 1];
                if (m + 1 >= (unsigned)kFillLds) vs[u] = gp[min(m + 1, (unsigned)n - 1)];
                if (w[u] != kAbsent && w[u] >= (unsigned)kFillLds) vw[u] = gp[w[u]];
                if (e[u] != kAbsent && e[u] >= (unsigned)kFillLds) ve[u] = gp[e[u]];
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int m = m0 + u * kCgThreads;
                double s = 0.0;
                s += w[u] != kAbsent ? vw[u] : 0.0;
                s += (q[u] & 8) ? vn[u] : 0.0;
                s += (q[u] & 16) ? vs[u] : 0.0;
                s += e[u] != kAbsent ? ve[u] : 0.0;
                if (m < n) body(m, p[u], (double)(q[u] & 7u) * p[u] - s);
            }
        }
    };
    double rr_ = block_sum(part, sp[0]);  // also orders the direction's writes before the reads
    const double tol2 = 1e-26 * rr_;
    int it = 0;
    bool ok = rr_ <= tol2;
    while (!ok && it < C.maxit) {
        it++;
        part = 0.0;
        passes([&](int, double p, double ap) { part += p * ap; });
        const double pap = block_sum(part, sp[1]);
        const double alpha = rr_ / pap;
        part = 0.0;
        passes([&](int m, double p, double ap) {
            x[m] += alpha * p;
            const double rm = r[m] - alpha * ap;
            r[m] = rm;
            part += rm * rm;
        });
        const double rn = block_sum(part, sp[0]);
        if (rn <= tol2) {
            ok = true;
            break;
        }
        const double beta = rn / rr_;
        rr_ = rn;
#pragma unroll 4
        for (int m = t; m < kFillLds; m += kCgThreads) lp[m] = r[m] + beta * lp[m];
#pragma unroll 4
        for (int m = kFillLds + t; m < n; m += kCgThreads) gp[m] = r[m] + beta * gp[m];
        __syncthreads();
    }
    for (int m = t; m < n; m += kCgThreads) a[list[m]] = to_class<T>(x[m]);
    if (t == 0) C.status[f] = ok ? it : -1;
}

// Frames by their entries per thread: the loop over kFillK entries costs
// every iteration 19 tests a phase, so that smaller frames take loops of
// their own length.  4000 x 16x16 frames of 31 missing pixels 1.58 -> 1.21
// ms, 2000 x 64x64 frames of 127, 0.88 -> 0.67 ms, 256 frames of 8000, 2.79 ->
// 2.14 ms.  (In kernels of their own the frames of one would wait for those of
// the other: 128 x 512x512 frames 6.1 -> 7.9 ms.)
template <typename T>
__global__ __launch_bounds__(kCgThreads) void k_fill_cg(FillChunk C, T *__restrict__ data) {
    __shared__ Partials sp[2];
    __shared__ double lp[kFillLds + 1];
    const int n = C.nmiss[blockIdx.x];
    if (n == 0 || n == C.np) {  // nothing to fill, or no known pixel (left as NaN)
        if (threadIdx.x == 0) C.status[blockIdx.x] = 0;
    } else if (n <= kCgThreads) {
        fill_cg_lds<1>(C, data, sp, lp);
    } else if (n <= 2 * kCgThreads) {
        fill_cg_lds<2>(C, data, sp, lp);
    } else if (n <= 4 * kCgThreads) {
        fill_cg_lds<4>(C, data, sp, lp);
    } else if (n <= 8 * kCgThreads) {
        fill_cg_lds<8>(C, data, sp, lp);
    } else if (n <= kFillLds) {
        fill_cg_lds<kFillK>(C, data, sp, lp);
    } else {
        fill_cg_stream(C, data, sp, lp);
    }
}

size_t esize(ss_dtype t) { return t == SS_F64 ? 8 : t == SS_F32 ? 4 : 2; }

template <typename F>
void dispatch(ss_dtype t, F &&f) {
    switch (t) {
    case SS_F64: f((double *)nullptr); break;
    case SS_F32: f((float *)nullptr); break;
    case SS_U16: f((uint16_t *)nullptr); break;
    default: f((int16_t *)nullptr); break;
    }
}

}  // namespace

#define PCHK(expr)                                                                            \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return ss::handle_fail(h, e_ == hipErrorOutOfMemory ? SS_ERR_OUT_OF_MEMORY : SS_ERR_DEVICE, \
                                   std::string(#expr) + ": " + hipGetErrorString(e_));        \
    } while (0)

extern "C" ss_status ss_prefilter(ss_handle *h, ss_dtype type, const void *in, void *out, int32_t height,
                                  int32_t width, int32_t n_frames, double pregauss, int32_t mednorm,
                                  int32_t on_device) try {
    if (!h) return SS_ERR_INVALID_ARGUMENT;
    if (!in || !out || height < 1 || width < 1 || n_frames < 1 || !(pregauss >= 0) || !std::isfinite(pregauss) ||
        type < SS_F64 || type > SS_I16)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "prefilter: bad arguments");
    if (mednorm && (type == SS_U16 || type == SS_I16))
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT,
                               "prefilter: median normalisation of integer frames is not supported");
    if ((double)height * width > 2.0e9)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "prefilter: frame too large");
    const int H = height, W = width;
    const size_t np = (size_t)H * W, es = esize(type);
    std::vector<double> g1, g2;
    int S1 = H, S2 = W;
    if (pregauss > 0) {
        // L = ceil(sqrt((2 gsd^2) log(10000 / (sqrt(2 pi) gsd)))) (steady_scan.m:628)
        const double gsd = pregauss;
        const int L = (int)std::ceil(std::sqrt((2 * gsd * gsd) * std::log(10000 / (std::sqrt(2 * 3.14159265358979323846) * gsd))));
        S1 = H + L;
        S2 = W + L;
        auto make = [&](int S, std::vector<double> &g) {
            g.resize(S);
            double sum = 0;
            for (int j = 0; j < S; j++) {
                const double d = std::min(j, S - j);
                g[j] = std::exp(-(d * d) / (2 * gsd * gsd));
                sum += g[j];
            }
            for (double &v : g) v /= sum;
        };
        make(S1, g1);
        make(S2, g2);
    }
    BlurAxis Y{}, X{};
    std::vector<double> taps1, taps2;
    const bool sweep = pregauss > 0 && blur_taps(g1, H, Y, taps1) && blur_taps(g2, W, X, taps2) && blur_by_sweep(Y, X);
    const bool isFloat = type == SS_F64 || type == SS_F32;
    // the GEMMs need an FP64 plane per frame (the sweep only for frames with
    // an infinity, as many at a time as fill the chip); the sweep reads and
    // writes different buffers
    const bool inPlace = on_device && in == out;
    const size_t plane = align256(np * 8);
    const size_t perFrame = (sweep || !(pregauss > 0) ? 0 : plane) + (on_device ? 0 : align256(np * es)) +
                            (sweep && (!on_device || inPlace) ? align256(np * es) : 0) + 256;
    // work memory: half of what is free on the device or already held by the handle
    PCHK(hipSetDevice(ss::handle_device(h)));
    size_t freeB = 0, totalB = 0;
    PCHK(hipMemGetInfo(&freeB, &totalB));
    const size_t budget = std::max<size_t>((size_t)1 << 30, (freeB + ss::handle_scratch_held(h)) / 2);
    // frames of a launch: the grid's limit and, for the GEMMs, 31 bits of columns
    const size_t most = sweep ? 65535 : std::min<size_t>(65535, (INT32_MAX - TN) / W);
    const int B = (int)std::max<size_t>(1, std::min<size_t>({(size_t)n_frames, budget / perFrame, most}));
    const size_t G = !(pregauss > 0) ? 0 : !sweep ? B : !isFloat ? 0 : std::min<size_t>(B, std::max<size_t>(1, kPlaneBytes / plane));
    ss_status rc;
    // the tables, in one upload: the sweep's taps, the whole kernels where the
    // GEMMs may run, and the first launch's flags (0)
    std::vector<double> tab;
    if (sweep) {
        tab = taps1;
        tab.insert(tab.end(), taps2.begin(), taps2.end());
    }
    const size_t oG = tab.size();
    if (G) {
        tab.insert(tab.end(), g1.begin(), g1.end());
        tab.insert(tab.end(), g2.begin(), g2.end());
    }
    const size_t oBad = tab.size();
    const bool flagsInTab = sweep && isFloat && B <= kFlagsInTab;
    if (flagsInTab) tab.resize(oBad + ((size_t)B + 1) / 2, 0.0);
    const size_t tableBytes = align256(8 * tab.size()) + align256(4 * (size_t)B) * 2 + (sweep ? plane * G : 0);
    char *base = (char *)ss::handle_scratch(h, tableBytes + perFrame * B, &rc);
    if (!base) return rc;
    hipStream_t s = ss::handle_stream(h);
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = base + off;
        off += align256(bytes);
        return (void *)p;
    };
    double *dtab = (double *)take(8 * tab.size()), *dg = dtab + oG;
    int *dbad = (int *)take(4 * (size_t)B), *dlist = (int *)take(4 * (size_t)B);
    if (flagsInTab) dbad = (int *)(dtab + oBad);
    double *dT = G ? (double *)take(np * 8 * G) : nullptr;
    int *anyBad = nullptr;
    if (sweep && isFloat && !(anyBad = ss::handle_host_flag(h, &rc))) return rc;
    char *dio = on_device ? nullptr : (char *)take(es * np * B);
    char *dcopy = sweep && (!on_device || inPlace) ? (char *)take(es * np * B) : nullptr;
    if (!tab.empty()) PCHK(hipMemcpyAsync(dtab, tab.data(), 8 * tab.size(), hipMemcpyHostToDevice, s));
    size_t lds = 0;
    int ring = 0;
    if (sweep) {
        Y.g = dtab;
        X.g = dtab + taps1.size();
        lds = blur_lds(Y, X, ring);
    }
    const unsigned gx = (unsigned)((np + 255) / 256);
    // nf frames of class values (or the listed ones) at `from`, blurred by the
    // GEMMs to the same places at `work`
    auto gemms = [&](const char *from, char *work, const int *list, int nf) {
        dispatch(type, [&](auto *tp) {
            using T = std::remove_pointer_t<decltype(tp)>;
            hipLaunchKernelGGL((k_circ_gemm<0, T, double>), dim3((W * nf + TN - 1) / TN, (H + TM - 1) / TM, 1), dim3(256),
                               0, s, (const T *)from, dT, list, dg, S1, H, W, W * nf);
            hipLaunchKernelGGL((k_circ_gemm<1, double, T>), dim3((W + TN - 1) / TN, (H + TM - 1) / TM, nf), dim3(256), 0,
                               s, dT, (T *)work, list, dg + S1, S2, H, W, 0);
        });
    };
    auto median = [&](char *work, const int *list, int nf) {
        if (type == SS_F64)
            hipLaunchKernelGGL(k_median_divide<double>, dim3(nf), dim3(1024), 0, s, (double *)work, list, (int)np);
        else
            hipLaunchKernelGGL(k_median_divide<float>, dim3(nf), dim3(1024), 0, s, (float *)work, list, (int)np);
    };
    std::vector<int> bad, list;
    for (int f0 = 0; f0 < n_frames; f0 += B) {
        const int nb = std::min(B, n_frames - f0);
        const size_t cnt = np * nb;
        const char *src = (const char *)in + es * np * f0;
        char *dst = (char *)out + es * np * f0;
        char *work = on_device ? dst : dio;
        const char *from = src;  // the sweep's input
        if (sweep) {
            if (dcopy) {
                PCHK(hipMemcpyAsync(dcopy, src, es * cnt, on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, s));
                from = dcopy;
            }
            if (isFloat) {
                if (f0 > 0 || !flagsInTab) PCHK(hipMemsetAsync(dbad, 0, 4 * (size_t)nb, s));
                *anyBad = 0;
            }
            const int strips = (H + kBlurRows - 1) / kBlurRows, segCols = blur_segment(Y, X, (size_t)strips * nb, lds);
            const dim3 grid(strips, nb, (W + segCols - 1) / segCols);
            hipError_t le = hipSuccess;
            dispatch(type, [&](auto *tp) {
                using T = std::remove_pointer_t<decltype(tp)>;
                le = hipFuncSetAttribute((const void *)k_blur<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                hipLaunchKernelGGL(k_blur<T>, grid, dim3(kBlurThreads), lds, s, (const T *)from, (T *)work, Y, X, segCols,
                                   ring, dbad, anyBad);
            });
            PCHK(le);
        } else {
            if (!on_device) PCHK(hipMemcpyAsync(work, src, es * cnt, hipMemcpyHostToDevice, s));
            else if (src != dst && !(pregauss > 0))
                PCHK(hipMemcpyAsync(work, src, es * cnt, hipMemcpyDeviceToDevice, s));
            if (pregauss > 0) gemms(on_device ? src : work, work, nullptr, nb);
        }
        if (mednorm) median(work, nullptr, nb);
        PCHK(hipGetLastError());
        if (!on_device) PCHK(hipMemcpyAsync(dst, work, es * cnt, hipMemcpyDeviceToHost, s));
        PCHK(hipStreamSynchronize(s));
        if (!anyBad || !*(volatile int *)anyBad) continue;
        // Frames with a NaN become NaN throughout: every output of the full
        // convolution has it as a term.  Frames with an infinity go through the GEMMs.
        // 500 x 512x512 float32 frames with a NaN each take 0.78 ms, with an
        // infinity each 7.7 ms; blurred by the GEMMs one by one, 106 ms.
        bad.resize(nb);
        PCHK(hipMemcpy(bad.data(), dbad, 4 * (size_t)nb, hipMemcpyDeviceToHost));
        list.clear();
        for (int f = 0; f < nb; f++)
            if (bad[f] & kBadNan) list.push_back(f);
        const size_t nans = list.size();
        for (int f = 0; f < nb; f++)
            if (bad[f] == kBadInf) list.push_back(f);
        PCHK(hipMemcpyAsync(dlist, list.data(), 4 * list.size(), hipMemcpyHostToDevice, s));
        if (nans) {
            const dim3 grid(gx, (unsigned)nans);
            if (type == SS_F64) hipLaunchKernelGGL(k_set_nan<double>, grid, dim3(256), 0, s, (double *)work, dlist, np);
            else hipLaunchKernelGGL(k_set_nan<float>, grid, dim3(256), 0, s, (float *)work, dlist, np);
        }
        for (size_t k = nans; k < list.size(); k += G) {
            const int n = (int)std::min(G, list.size() - k);
            gemms(from, work, dlist + k, n);
            if (mednorm) median(work, dlist + k, n);
        }
        PCHK(hipGetLastError());
        if (!on_device) PCHK(hipMemcpyAsync(dst, work, es * cnt, hipMemcpyDeviceToHost, s));
        PCHK(hipStreamSynchronize(s));
    }
    return SS_OK;
} catch (const std::bad_alloc &) {
    return SS_ERR_OUT_OF_MEMORY;  // host memory; C callers never see an exception
} catch (...) {
    return SS_ERR_DEVICE;
}

extern "C" ss_status ss_fill_gaps(ss_handle *h, ss_dtype type, const void *in, void *out, int32_t height,
                                  int32_t width, int32_t n_frames, int32_t on_device) try {
    if (!h) return SS_ERR_INVALID_ARGUMENT;
    if (!in || !out || height < 1 || width < 1 || n_frames < 1 || (type != SS_F64 && type != SS_F32))
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "fill_gaps: bad arguments (float32 or float64 frames)");
    if ((double)height * width > 2.0e9)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "fill_gaps: frame too large");
    const int H = height, W = width;
    const size_t np = (size_t)H * W, es = esize(type);
    const size_t perFrame = align256(np * 8) * 4 + align256(np * 4) * 2 + align256(np) + align256(8) * 2 +
                            (on_device ? 0 : align256(np * es));
    // work memory: half of what is free on the device or already held by the handle
    PCHK(hipSetDevice(ss::handle_device(h)));
    size_t freeB = 0, totalB = 0;
    PCHK(hipMemGetInfo(&freeB, &totalB));
    const size_t budget = std::max<size_t>((size_t)1 << 30, (freeB + ss::handle_scratch_held(h)) / 2);
    const int B = (int)std::max<size_t>(1, std::min<size_t>({(size_t)n_frames, budget / perFrame, (size_t)65535}));
    ss_status rc;
    char *base = (char *)ss::handle_scratch(h, perFrame * B, &rc);
    if (!base) return rc;
    hipStream_t s = ss::handle_stream(h);
    PCHK(hipSetDevice(ss::handle_device(h)));
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = base + off;
        off += align256(bytes);
        return (void *)p;
    };
    FillChunk C{};
    C.th = H;
    C.tw = W;
    C.np = (int)np;
    C.maxit = 200000;
    C.x = (double *)take(np * 8 * B);
    C.r = (double *)take(np * 8 * B);
    C.p = (double *)take(np * 8 * B);
    C.code = (uint2 *)take(np * 8 * B);
    C.meta = (uint8_t *)take(np * B);
    C.map = (int *)take(np * 4 * B);
    C.list = (int *)take(np * 4 * B);
    C.nmiss = (int *)take(4 * (size_t)B);
    C.status = (int *)take(4 * (size_t)B);
    char *dio = on_device ? nullptr : (char *)take(es * np * B);
    std::vector<int> status(B);
    for (int f0 = 0; f0 < n_frames; f0 += B) {
        const int nb = std::min(B, n_frames - f0);
        const size_t cnt = np * nb;
        const char *src = (const char *)in + es * np * f0;
        char *dst = (char *)out + es * np * f0;
        // only the missing pixels are written: the frames are filled in place
        char *work = on_device ? dst : dio;
        if (!on_device) PCHK(hipMemcpyAsync(dio, src, es * cnt, hipMemcpyHostToDevice, s));
        else if (src != dst) PCHK(hipMemcpyAsync(dst, src, es * cnt, hipMemcpyDeviceToDevice, s));
        auto fill = [&](auto *frames) {
            using T = std::remove_pointer_t<decltype(frames)>;
            hipLaunchKernelGGL(k_fill_list<T>, dim3(nb), dim3(kCgThreads), 0, s, C, (const T *)frames);
            hipLaunchKernelGGL(k_fill_cg<T>, dim3(nb), dim3(kCgThreads), 0, s, C, frames);
        };
        if (type == SS_F64) fill((double *)work);
        else fill((float *)work);
        PCHK(hipGetLastError());
        PCHK(hipMemcpyAsync(status.data(), C.status, 4 * nb, hipMemcpyDeviceToHost, s));
        if (!on_device) PCHK(hipMemcpyAsync(dst, dio, es * cnt, hipMemcpyDeviceToHost, s));
        PCHK(hipStreamSynchronize(s));
        if (const char *e = std::getenv("SS_FILL_STATS"); e && e[0] == '1') {
            std::vector<int> nm(nb);
            PCHK(hipMemcpy(nm.data(), C.nmiss, 4 * (size_t)nb, hipMemcpyDeviceToHost));
            long sum = 0, msum = 0;
            int mx = 0, nf = 0, inLds = 0, mmax = 0;
            for (int f = 0; f < nb; f++) {
                msum += nm[f];
                mmax = std::max(mmax, nm[f]);
                inLds += nm[f] <= kFillLds;
                if (status[f] > 0) {
                    sum += status[f];
                    mx = std::max(mx, status[f]);
                    nf++;
                }
            }
            std::fprintf(stderr,
                         "[fill] chunk of %d frames: %d filled, CG iterations mean %.1f max %d; missing pixels "
                         "mean %.0f max %d, %d frames in LDS\n",
                         nb, nf, nf ? (double)sum / nf : 0.0, mx, (double)msum / nb, mmax, inLds);
        }
        for (int f = 0; f < nb; f++)
            if (status[f] < 0)
                return ss::handle_fail(h, SS_ERR_NUMERICAL,
                                       "fill_gaps: frame " + std::to_string(f0 + f) +
                                           ": conjugate gradients did not converge");
    }
    return SS_OK;
} catch (const std::bad_alloc &) {
    return SS_ERR_OUT_OF_MEMORY;  // host memory; C callers never see an exception
} catch (...) {
    return SS_ERR_DEVICE;
}
