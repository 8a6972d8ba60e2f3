// ss_resample.hip -- corrected frames: resample_frame + pushgrid
// (steady_scan.m:562-599) on the GPU.
//
// pushgrid splats every in-bounds data pixel onto the 4 template pixels of
// its cell with bilinear weights, through MATLAB indexed assignments
// z(ind) = z(ind) + v.  With repeated indices such an assignment keeps the
// value of the LAST occurrence, so for each template pixel and each of the
// four corner offsets exactly one data pixel contributes: the one with the
// largest (column-major) pixel index.  All four corners of a cell see the
// same data pixels, so the winner is a property of the cell.  The GPU form is
//   pass 0: the launch's table of cell winners is set to -1 (a fill kernel,
//           so that the pass also runs under stream capture);
//   pass 1: per frame and data pixel, atomicMax of the pixel index into its
//           cell (an integer maximum: order-independent, deterministic);
//   pass 2: per frame and tile of template pixels, the cells' winners are
//           evaluated once into LDS, and every template pixel accumulates its
//           <= 4 in single precision in the statement order of pushgrid.
// Positions are computed in FP64 without contraction, as MATLAB does.
// 200 x 512x512 uint16, device to device: 0.62 ms, of which the winners take
// 0.23 (bound by the atomics, which gfx950 performs behind the L2s) and the
// gather 0.32 (its chain of dependent loads); 8.2 ms with an atomicMax per
// corner, winners evaluated by each corner and a host-built geometry table.
//
// All frames of a launch share the pixel geometry; grid.y is the frame, or
// kWinFrames of them in the winners' pass.
// ss_resample tables each pixel's knot and fraction once per call on the GPU
// (k_scan_table).  The work memory (tables, knots, winners and the staging of
// host frames and host output) is the handle's, kept across calls, and
// everything runs on the handle's stream with one synchronisation at the end
// of the call.
//
// ss_resample_noalloc runs the same three passes with no allocation at all:
// the kernels compute each pixel's geometry from the scan formulas
// (ss_scan.h) instead of reading a table, and the knots and winner tables
// live in a fixed static device array (kNoAllocBytes per device).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include <hip/hip_runtime.h>

#include "ss_host.h"
#include "ss_scan.h"
#include "steadyscan.h"

namespace {

struct PixGeo {
    double bx, by, tf;
    int k;  // prevknotind - 1
    int pad;
};

__global__ __launch_bounds__(256) void k_fill_minus1(int *__restrict__ p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = -1;
}

// Pixel geometry from the call's tables: 12 bytes per pixel (3 MB at 512x512,
// within an XCD's L2), the base coordinates per column and row.
struct TableGeo {
    const double *tf, *bx, *by;
    const int *k;
    int hc;
    __device__ __forceinline__ PixGeo at(int i) const {
        const int jc = i / hc;
        return PixGeo{bx[jc], by[i - jc * hc], tf[i], k[i], 0};
    }
};

// Pixel geometry computed from the scan formulas (the same functions that
// build the table on the host, so the same doubles); kt: the knot times.
struct ScanGeo {
    ss::ScanParams s;
    const double *kt;
    __device__ __forceinline__ PixGeo at(int i) const {
        const int ic = i % s.Hc, jc = i / s.Hc;  // cropped (row, column), column-major
        const double t = ss::scan_cropped_time(s, ic, jc);
        // t lies in (0, 1) and the knot times run from 0 to 1, so the bin is
        // 1 .. nknots - 1; the clamp only guards the knot reads
        const int k = min(max(ss::scan_bin(kt, s.nknots, t), 1), s.nknots - 1);
        return PixGeo{ss::scan_base_x(s, jc), ss::scan_base_y(s, ic), ss::scan_tfrac(kt, k, t), k - 1, 0};
    }
};

// The tables of TableGeo, by the formulas of ScanGeo (one thread per pixel).
__global__ __launch_bounds__(256) void k_scan_table(ScanGeo geo, int npix, double *__restrict__ tf, int *__restrict__ k,
                                                    double *__restrict__ bx, double *__restrict__ by) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npix) return;
    const PixGeo q = geo.at(i);
    tf[i] = q.tf;
    k[i] = q.k;
    const int jc = i / geo.s.Hc, ic = i - jc * geo.s.Hc;
    if (ic == 0) bx[jc] = q.bx;
    if (jc == 0) by[ic] = q.by;
}

// Knots of the launch's frames: frame f's x knots at kx + f * stride, its y
// knots at ky + f * stride.
struct FrameKnots {
    const double *kx, *ky;
    size_t stride;
};

// Frames per thread of the winners pass: a pixel's geometry is loaded once
// for all of them, and their knots are loaded together.
constexpr int kWinFrames = 4;

template <typename Geo>
__global__ __launch_bounds__(256) void k_splat_winners(Geo geo, int npix, FrameKnots kn, int nf, int th, int tw,
                                                       int *__restrict__ win) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npix) return;
    const PixGeo q = geo.at(i);
    const double tc = 1.0 - q.tf;
    const int f0 = blockIdx.y * kWinFrames;
    double x[kWinFrames], y[kWinFrames];
#pragma unroll
    for (int j = 0; j < kWinFrames; j++) {
        const size_t o = (size_t)min(f0 + j, nf - 1) * kn.stride + q.k;
        x[j] = q.bx + kn.kx[o] * tc + kn.kx[o + 1] * q.tf;
        y[j] = q.by + kn.ky[o] * tc + kn.ky[o + 1] * q.tf;
    }
#pragma unroll
    for (int j = 0; j < kWinFrames; j++) {
        const bool in = x[j] >= 1.0 && x[j] < (double)tw && y[j] >= 1.0 && y[j] < (double)th && f0 + j < nf;
        if (!in) continue;
        const int xi = (int)floor(x[j]), yi = (int)floor(y[j]);
        atomicMax(&win[(size_t)(f0 + j) * th * tw + (yi - 1) + th * (xi - 1)], i);
    }
}

// Tile of the gather: 64 rows (consecutive in memory) x 16 columns of template
// pixels, from the 65 x 17 cells that they are corners of.  A cell's winner
// is evaluated once instead of by each of its four corners.
constexpr int kTileR = 64, kTileC = 16, kCellR = kTileR + 1, kCells = kCellR * (kTileC + 1);

template <typename TD, typename Geo>
__global__ __launch_bounds__(256) void k_splat_gather(Geo geo, const TD *__restrict__ data, size_t framePix, int hc,
                                                      int nl, int cl, int cb, FrameKnots kn, int th, int tw,
                                                      const int *__restrict__ win, float *__restrict__ out) {
#pragma clang fp contract(off)
    // a cell's contribution to its corners 0, 1, th, th+1: the weighted value
    // and the weight; 0 without a winner, which leaves the sums as they are
    __shared__ float2 sw[4][kCells];
    const size_t tp = (size_t)th * tw;
    const int f = blockIdx.y;
    const int tilesR = (th + kTileR - 1) / kTileR;
    const int r0 = (blockIdx.x % tilesR) * kTileR, c0 = (blockIdx.x / tilesR) * kTileC;
    const double *kx = kn.kx + (size_t)f * kn.stride, *ky = kn.ky + (size_t)f * kn.stride;
    const int *wf = win + (size_t)f * tp;
    const TD *df = data + framePix * f;
    // a thread's cells go through the dependent loads (winner, geometry and
    // data, knots) together
    constexpr int kPer = (kCells + 255) / 256;
    int win_[kPer];
    PixGeo geo_[kPer];
    double d_[kPer], k_[kPer][4];
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int q = threadIdx.x + 256 * j;
        const int qc = q / kCellR, r = r0 - 1 + q - qc * kCellR, c = c0 - 1 + qc;
        win_[j] = q < kCells && r >= 0 && c >= 0 && r < th && c < tw ? wf[(size_t)c * th + r] : -1;
    }
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = max(win_[j], 0);
        geo_[j] = geo.at(i);
        const int jc = i / hc, ic = i - jc * hc;  // cropped (row, column)
        d_[j] = (double)df[(size_t)(jc + cl) * nl + (ic + cb)];
    }
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int k = geo_[j].k;
        k_[j][0] = kx[k];
        k_[j][1] = kx[k + 1];
        k_[j][2] = ky[k];
        k_[j][3] = ky[k + 1];
    }
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int q = threadIdx.x + 256 * j;
        if (q >= kCells) break;
        const double tf = geo_[j].tf, tc = 1.0 - tf;
        const double x = geo_[j].bx + k_[j][0] * tc + k_[j][1] * tf, y = geo_[j].by + k_[j][2] * tc + k_[j][3] * tf;
        const double xf = x - floor(x), yf = y - floor(y);
        // corner offsets 0, 1, th, th+1 <-> weights (steady_scan.m:589-592)
        const double ws[4] = {(1 - xf) * (1 - yf), (1 - xf) * yf, xf * (1 - yf), xf * yf};
#pragma unroll
        for (int s = 0; s < 4; s++)
            sw[s][q] = win_[j] >= 0 ? make_float2((float)(ws[s] * d_[j]), (float)ws[s]) : make_float2(0.f, 0.f);
    }
    __syncthreads();
    for (int o = threadIdx.x; o < kTileR * kTileC; o += 256) {
        const int lc = o / kTileR, lr = o - lc * kTileR;
        const int r = r0 + lr, c = c0 + lc;
        if (r >= th || c >= tw) continue;
        // the cells whose corner 0, 1, th, th+1 this pixel is
        const int base = (lc + 1) * kCellR + lr + 1;
        const float2 w0 = sw[0][base], w1 = sw[1][base - 1], w2 = sw[2][base - kCellR], w3 = sw[3][base - kCellR - 1];
        // z statements in order: offsets 0, 1, th, th+1 (steady_scan.m:589-592)
        float z = 0.f + w0.x;
        z = z + w1.x;
        z = z + w2.x;
        z = z + w3.x;
        // n statements in order: offsets 1, th, 0, th+1 (steady_scan.m:595-598)
        float n = 0.f + w1.y;
        n = n + w2.y;
        n = n + w0.y;
        n = n + w3.y;
        out[(size_t)f * tp + (size_t)c * th + r] = z / n;
    }
}

template <typename TD, typename Geo>
hipError_t launch_frames(hipStream_t s, const Geo &geo, int npix, const void *data, size_t framePix,
                         const ss_geometry_desc &g, int hc, const FrameKnots &kn, int nf, int *win, float *out) {
    const int th = g.template_h, tw = g.template_w;
    const size_t tp = (size_t)th * tw, nwin = (size_t)nf * tp;
    const int fillGrid = (int)std::min<size_t>((nwin + 255) / 256, 8192);
    hipLaunchKernelGGL(k_fill_minus1, dim3(fillGrid), dim3(256), 0, s, win, nwin);
    hipLaunchKernelGGL((k_splat_winners<Geo>), dim3((npix + 255) / 256, (nf + kWinFrames - 1) / kWinFrames), dim3(256), 0,
                       s, geo, npix, kn, nf, th, tw, win);
    hipLaunchKernelGGL((k_splat_gather<TD, Geo>), dim3((unsigned)(((th + kTileR - 1) / kTileR) * ((tw + kTileC - 1) / kTileC)), nf), dim3(256), 0, s, geo,
                       (const TD *)data, framePix, hc, g.nlines, g.cropping[0], g.cropping[2], kn, th, tw, win, out);
    return hipGetLastError();
}

template <typename Geo>
hipError_t launch_typed(ss_dtype type, hipStream_t s, const Geo &geo, int npix, const void *data, size_t framePix,
                        const ss_geometry_desc &g, int hc, const FrameKnots &kn, int nf, int *win, float *out) {
    switch (type) {
    case SS_F64: return launch_frames<double>(s, geo, npix, data, framePix, g, hc, kn, nf, win, out);
    case SS_F32: return launch_frames<float>(s, geo, npix, data, framePix, g, hc, kn, nf, win, out);
    case SS_U16: return launch_frames<uint16_t>(s, geo, npix, data, framePix, g, hc, kn, nf, win, out);
    default: return launch_frames<int16_t>(s, geo, npix, data, framePix, g, hc, kn, nf, win, out);
    }
}

// ---------------------------------------------------------------------------
// the allocation-free variant's work area: one static array per device
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocBytes = (size_t)64 << 20;
constexpr int kNoAllocMaxKnots = 4096;
constexpr int kMaxDevices = 64;

// In host code `scratch` names a host-side stand-in, not device memory: only
// the address that hipGetSymbolAddress returns for a device may be used.
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

std::mutex g_scratchLock;
void *g_scratchPtr[kMaxDevices] = {};
hipError_t g_scratchErr[kMaxDevices] = {};
bool g_scratchDone[kMaxDevices] = {};

}  // namespace

namespace ss {

// Looks up this device's copy of the static work area, once per device, with
// the device current (called from ss_create).
hipError_t resample_scratch_init(int device) {
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratchLock);
    if (!g_scratchDone[device]) {
        void *ptr = nullptr;
        g_scratchErr[device] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        g_scratchPtr[device] = g_scratchErr[device] == hipSuccess ? ptr : nullptr;
        g_scratchDone[device] = true;
    }
    return g_scratchErr[device];
}

}  // namespace ss

extern "C" ss_status ss_resample(ss_handle *h, const ss_resample_in *in, float *out) try {
    if (!h) return SS_ERR_INVALID_ARGUMENT;
    if (!in || !out || !in->geometry || !in->frames || !in->knots_x || !in->knots_y || in->n_frames < 1)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample: NULL argument or no frames");
    if (in->data_type < SS_F64 || in->data_type > SS_I16)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample: invalid data_type");
    const ss_geometry_desc &g = *in->geometry;
    // the validity rules of ss_geometry_size: vertical cropping mis-sizes the
    // default basey (steady_scan.m:799, 822-824)
    ss::ScanParams sp;
    std::vector<double> kt(std::max(2, g.nknots));
    if (!ss::scan_setup(g, sp, kt.data()) || sp.cb + sp.ct != 0)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample: invalid geometry");
    const int hc = sp.Hc, wc = sp.Wc;
    ss_status st = SS_OK;
    const int th = g.template_h, tw = g.template_w, nk = g.nknots, nF = in->n_frames;
    if (th < 2 || tw < 2) return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample: template smaller than 2x2");
    if ((long long)hc * wc >= (1ll << 31) || (long long)th * tw >= (1ll << 31))
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample: frame or template too large");
    if (hipSetDevice(ss::handle_device(h)) != hipSuccess) return ss::handle_fail(h, SS_ERR_DEVICE, "hipSetDevice");
    hipStream_t s = ss::handle_stream(h);
    const int npix = hc * wc;
    // knots of all frames, per frame [x(0..nk-1), y(0..nk-1)]
    std::vector<double> kn((size_t)2 * nk * nF);
    for (int f = 0; f < nF; f++) {
        std::memcpy(kn.data() + (size_t)f * 2 * nk, in->knots_x + (size_t)f * nk, sizeof(double) * nk);
        std::memcpy(kn.data() + (size_t)f * 2 * nk + nk, in->knots_y + (size_t)f * nk, sizeof(double) * nk);
    }
    const size_t tp = (size_t)th * tw;
    const size_t esz = in->data_type == SS_F64 ? 8 : in->data_type == SS_F32 ? 4 : 2;
    const size_t fpix = (size_t)g.nlines * g.linewidth;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    // work memory: geometry tables + knots, then per frame of a launch the
    // winner table and the staging of host frames / host output
    const size_t tables = al(sizeof(double) * npix) + al(sizeof(int) * npix) + al(sizeof(double) * wc) +
                          al(sizeof(double) * hc) + al(sizeof(double) * nk);
    const size_t fixed = tables + al(kn.size() * sizeof(double));
    const size_t perFrame = tp * sizeof(int) + (in->data_on_device ? 0 : esz * fpix) +
                            (in->out_on_device ? 0 : tp * sizeof(float));
    const size_t budget = std::max<size_t>(ss::handle_scratch_held(h), (size_t)256 << 20);
    const int chunk = (int)std::max<size_t>(1, std::min<size_t>(
                                                   {(size_t)nF, (budget > fixed ? budget - fixed : 0) / perFrame, 65535}));
    char *mem = (char *)ss::handle_scratch(h, fixed + al(perFrame * chunk) + 4096, &st);
    if (!mem) return st;
    double *dtf = (double *)mem;
    int *dki = (int *)(mem + al(sizeof(double) * npix));
    double *dbx = (double *)((char *)dki + al(sizeof(int) * npix));
    double *dby = (double *)((char *)dbx + al(sizeof(double) * wc));
    double *dkt = (double *)((char *)dby + al(sizeof(double) * hc));
    double *dk = (double *)(mem + tables);
    int *dwin = (int *)(mem + fixed);
    char *dstage = (char *)dwin + al(tp * sizeof(int) * chunk);
    char *ddata = in->data_on_device ? nullptr : dstage;
    float *dout = in->out_on_device ? nullptr : (float *)(dstage + (in->data_on_device ? 0 : al(esz * fpix * chunk)));
    const TableGeo geo{dtf, dbx, dby, dki, hc};
#define RCHK(expr)                                                                                       \
    do {                                                                                                 \
        hipError_t e_ = (expr);                                                                          \
        if (e_ != hipSuccess) return ss::handle_fail(h, SS_ERR_DEVICE, std::string("resample: ") + #expr + \
                                                                           ": " + hipGetErrorString(e_)); \
    } while (0)
    RCHK(hipMemcpyAsync(dkt, kt.data(), sizeof(double) * nk, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_scan_table, dim3((npix + 255) / 256), dim3(256), 0, s, ScanGeo{sp, dkt}, npix, dtf, dki, dbx, dby);
    RCHK(hipMemcpyAsync(dk, kn.data(), kn.size() * sizeof(double), hipMemcpyHostToDevice, s));
    for (int f0 = 0; f0 < nF; f0 += chunk) {
        const int nf = std::min(chunk, nF - f0);
        const void *src = (const char *)in->frames + esz * fpix * f0;
        if (ddata) {
            RCHK(hipMemcpyAsync(ddata, src, esz * fpix * nf, hipMemcpyHostToDevice, s));
            src = ddata;
        }
        float *o = dout ? dout : out + tp * f0;
        const double *kf = dk + (size_t)2 * nk * f0;
        const FrameKnots fk{kf, kf + nk, (size_t)2 * nk};
        RCHK((launch_typed(in->data_type, s, geo, npix, src, fpix, g, hc, fk, nf, dwin, o)));
        if (dout) RCHK(hipMemcpyAsync(out + tp * f0, dout, sizeof(float) * tp * nf, hipMemcpyDeviceToHost, s));
    }
    RCHK(hipStreamSynchronize(s));
#undef RCHK
    return SS_OK;
} catch (const std::bad_alloc &) {
    return SS_ERR_OUT_OF_MEMORY;  // host memory; C callers never see an exception
} catch (...) {
    return SS_ERR_DEVICE;
}

extern "C" ss_status ss_resample_noalloc(ss_handle *h, const ss_resample_in *in, float *out) try {
    if (!h) return SS_ERR_INVALID_ARGUMENT;
    if (!in || !out || !in->geometry || !in->frames || !in->knots_x || !in->knots_y || in->n_frames < 1)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: NULL argument or no frames");
    if (in->data_type < SS_F64 || in->data_type > SS_I16)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: invalid data_type");
    if (!in->data_on_device || !in->out_on_device)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT,
                               "resample_noalloc: frames and output must be device memory (data_on_device and "
                               "out_on_device set)");
    const ss_geometry_desc &g = *in->geometry;
    if (g.nknots < 2 || g.nknots > kNoAllocMaxKnots)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: nknots must be 2 .. 4096");
    ss::ScanParams sp;
    double kt[kNoAllocMaxKnots];
    // the same validity rules as ss_geometry_size: vertical cropping mis-sizes
    // the default basey (steady_scan.m:799, 822-824)
    if (!ss::scan_setup(g, sp, kt) || sp.cb + sp.ct != 0)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: invalid geometry");
    const int th = g.template_h, tw = g.template_w, nk = g.nknots, nF = in->n_frames;
    if (th < 2 || tw < 2)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: template smaller than 2x2");
    if ((long long)sp.Hc * sp.Wc >= (1ll << 31) || (long long)th * tw >= (1ll << 31))
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT, "resample_noalloc: frame or template too large");
    const int dev = ss::handle_device(h);
    if (hipSetDevice(dev) != hipSuccess) return ss::handle_fail(h, SS_ERR_DEVICE, "hipSetDevice");
    const hipError_t se = ss::resample_scratch_init(dev);  // done by ss_create; cached
    char *base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratchLock);
        base = se == hipSuccess ? (char *)g_scratchPtr[dev] : nullptr;
    }
    if (!base)
        return ss::handle_fail(h, SS_ERR_DEVICE, std::string("resample_noalloc: static work area unavailable: ") +
                                                     hipGetErrorString(se));
    // work area: [knot times][x knots of a launch][y knots][winner tables]
    const size_t tp = (size_t)th * tw;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t fixed = al(sizeof(double) * nk);
    auto need = [&](size_t nf) { return fixed + 2 * al(sizeof(double) * nk * nf) + tp * sizeof(int) * nf; };
    // templates are accepted up to 16 bytes of work area per pixel
    if (need(1) + 3 * tp * sizeof(int) > kNoAllocBytes)
        return ss::handle_fail(h, SS_ERR_INVALID_ARGUMENT,
                               "resample_noalloc: one frame needs " + std::to_string(need(1) + 3 * tp * sizeof(int)) +
                                   " bytes of work memory; the static work area holds " +
                                   std::to_string(kNoAllocBytes) + " bytes (template_h x template_w up to about 4.1 "
                                                                   "million pixels)");
    size_t chunk = std::min<size_t>({(size_t)nF, (kNoAllocBytes - fixed) / (tp * sizeof(int) + 2 * sizeof(double) * nk),
                                     65535});
    while (chunk > 1 && need(chunk) > kNoAllocBytes) chunk--;
    double *dkt = (double *)base;
    double *dkx = (double *)(base + fixed);
    double *dky = (double *)(base + fixed + al(sizeof(double) * nk * chunk));
    int *dwin = (int *)(base + fixed + 2 * al(sizeof(double) * nk * chunk));
    hipStream_t s = ss::handle_stream(h);
    const size_t esz = in->data_type == SS_F64 ? 8 : in->data_type == SS_F32 ? 4 : 2;
    const size_t fpix = (size_t)g.nlines * g.linewidth;
    const int npix = sp.Hc * sp.Wc;
#define NCHK(expr)                                                                                              \
    do {                                                                                                        \
        hipError_t e_ = (expr);                                                                                 \
        if (e_ != hipSuccess) {                                                                                 \
            (void)hipStreamSynchronize(s);                                                                      \
            return ss::handle_fail(h, SS_ERR_DEVICE,                                                            \
                                   std::string("resample_noalloc: ") + #expr + ": " + hipGetErrorString(e_)); \
        }                                                                                                       \
    } while (0)
    NCHK(hipMemcpyAsync(dkt, kt, sizeof(double) * nk, hipMemcpyHostToDevice, s));
    const ScanGeo geo{sp, dkt};
    for (int f0 = 0; f0 < nF; f0 += (int)chunk) {
        const int nf = std::min((int)chunk, nF - f0);
        NCHK(hipMemcpyAsync(dkx, in->knots_x + (size_t)nk * f0, sizeof(double) * nk * nf, hipMemcpyHostToDevice, s));
        NCHK(hipMemcpyAsync(dky, in->knots_y + (size_t)nk * f0, sizeof(double) * nk * nf, hipMemcpyHostToDevice, s));
        const void *src = (const char *)in->frames + esz * fpix * f0;
        const FrameKnots fk{dkx, dky, (size_t)nk};
        NCHK((launch_typed(in->data_type, s, geo, npix, src, fpix, g, sp.Hc, fk, nf, dwin, out + tp * f0)));
    }
    NCHK(hipStreamSynchronize(s));
#undef NCHK
    return SS_OK;
} catch (...) {
    return SS_ERR_DEVICE;
}
