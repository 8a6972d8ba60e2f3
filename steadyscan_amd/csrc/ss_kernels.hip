// ss_kernels.hip -- gfx950 kernels of the align_group_to_template path.
//
// A batch holds any number of alignment groups.  Every group runs its own
// copy of the reference's control flow (Task<T>::alignFrames and
// MainIteration<T>::execute) as a small state machine in device memory
// (GroupCtl), so one host submission ("tick") advances every group by one
// stage without host round trips:
//   k_assemble -> k_solve -> (k_ls_round -> k_ls_decide) x3 -> k_ls_finish
//   -> (the same for the second half-iteration) -> k_corr -> k_corr_finish
//   [-> k_final -> k_final_finish]
// Each kernel skips the groups that are not in its phase.  Without the
// final stages, the next tick's k_assemble and k_solve run the final pass
// and end the groups that stopped.
//
// Pixel work: one workgroup (4 wave64) per line-block column (frame f,
// block b = column c = f * nb + b of the block matrix).  A thread walks runs
// of rows, the lines of one image column of the block, so that neighbouring
// lanes sit on neighbouring scan-line pixels and a wave's template gathers
// touch a few cache lines; frame values come 8 rows at a time in 16-byte
// loads.  A chunk of rows computes its coordinates, issues all its gathers,
// and only then does the arithmetic (sched_fence, pin): left to itself the
// compiler put every sample's gathers under the branch that discards
// unmasked samples, with a wait each.  Per-column partial sums are reduced
// in registers, then across waves through LDS in FP64.  No floating-point
// atomics: every result is run-to-run deterministic.
// What bounds them (1000 x 512x512 uint16, FP64): VALU issue, 61-80% of the
// cycles, next to the L1's 64 bytes a cycle for the gathers.  Global instead
// of flat loads, batched gathers, scalar loads of the group's description,
// line-constant geometry and lane-swap reductions took the full batch's
// first assembly launch from 1269 to 729 us, a line-search launch from 342
// to 193 us and a correlation launch from 624 to 325 us on average.
#include "ss_device.h"
#include "ss_tuning.h"

#include <type_traits>

namespace ss {

constexpr int kWG = 256;       // pixel kernels
constexpr int kSolveWG = 256;  // per-group kernels
constexpr int kCH = 8;         // pixels per unrolled chunk

// Everything a group points to is device memory.  Saying so (address space
// 1) makes the pixel loads global loads; through the generic pointers of
// GroupDev they would be flat loads, which also wait for LDS and cannot be
// counted apart, so that every use waits for all loads in flight.  What no
// kernel of the launch writes (address space 4) is read by scalar loads; of the
// control blocks, the fields that the kernel itself leaves alone.
#define SS_GLOBAL __attribute__((address_space(1)))
#define SS_CONST __attribute__((address_space(4)))
// a group's description in the pixel kernels, which do not write it
using GroupRef = const SS_CONST GroupDev &;

// ---------------------------------------------------------------------------
// precision: pixel arithmetic in R = float (precision 'S') or double ('D');
// every reduction is FP64 in both
// ---------------------------------------------------------------------------
template <typename R>
struct Prec;
template <>
struct Prec<float> {
    static __device__ __forceinline__ const SS_CONST AffineGeo<float> &aff(GroupRef g) { return g.afF; }
    static __device__ __forceinline__ const float4 *geo(GroupRef g) { return g.geo; }
    static __device__ __forceinline__ const float *fnext(GroupRef g) { return g.fnext; }
    static __device__ __forceinline__ const float2 *tp(GroupRef g) { return g.tp; }
    static __device__ __forceinline__ const float2 *gxv(GroupRef g) { return g.gxv; }
    static __device__ __forceinline__ const float2 *gyh(GroupRef g) { return g.gyh; }
};
template <>
struct Prec<double> {
    static __device__ __forceinline__ const SS_CONST AffineGeo<double> &aff(GroupRef g) { return g.afD; }
    static __device__ __forceinline__ const double4 *geo(GroupRef g) { return g.geoD; }
    static __device__ __forceinline__ const double *fnext(GroupRef g) { return g.fnextD; }
    static __device__ __forceinline__ const double2 *tp(GroupRef g) { return g.tpD; }
    static __device__ __forceinline__ const double2 *gxv(GroupRef g) { return g.gxvD; }
    static __device__ __forceinline__ const double2 *gyh(GroupRef g) { return g.gyhD; }
};

__device__ __forceinline__ float mad(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double mad(double a, double b, double c) { return fma(a, b, c); }

template <typename TI>
__host__ __device__ constexpr int img_type() {
    return std::is_same<TI, float>::value      ? IMG_F32
           : std::is_same<TI, uint16_t>::value ? IMG_U16
           : std::is_same<TI, int16_t>::value  ? IMG_I16
                                               : IMG_F64;
}
// true when group g runs in the instantiation <TI, R>
template <typename TI, typename R>
__device__ __forceinline__ bool runs_here(GroupRef g) {
    return g.imgType == img_type<TI>() && g.fp64 == (sizeof(R) == 8 ? 1 : 0);
}

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ const SS_GLOBAL T *as_global(const T *p) {
    return (const SS_GLOBAL T *)p;
}
template <typename T>
__device__ __forceinline__ const SS_CONST T *as_const(const T *p) {
    return (const SS_CONST T *)p;
}
__device__ __forceinline__ GroupRef group_of(const Batch &B, int gi) { return as_const(B.groups)[gi]; }

// The group of frame item i; a batch of one group has no table to wait for.
__device__ __forceinline__ int group_index(const Batch &B, const int *table, int i) {
    return B.nGroups == 1 ? 0 : as_const(table)[i];
}
// The values are loaded by here, in one round: ahead of the conditions on
// some of them that the compiler would wait for first.  (Not in the pixel
// kernels: the registers that hold them cost the FP64 line search 5 to 10% at
// 512x512, and the table's shortcut above as much.)
__device__ __forceinline__ void loaded() {}
template <typename T, typename... Rest>
__device__ __forceinline__ void loaded(T x, Rest... rest) {
    asm volatile("" ::"s"(x));
    loaded(rest...);
}
// native vectors: their loads keep the pointer's address space
using f2v = float __attribute__((ext_vector_type(2)));
using f4v = float __attribute__((ext_vector_type(4)));
using d2v = double __attribute__((ext_vector_type(2)));
using d4v = double __attribute__((ext_vector_type(4)));
using u4v = uint32_t __attribute__((ext_vector_type(4)));
template <typename R>
struct Nat {
    using V2 = f2v;
    using V4 = f4v;
};
template <>
struct Nat<double> {
    using V2 = d2v;
    using V4 = d4v;
};

// The scheduler moves nothing across: the loads of a chunk stay ahead of
// the arithmetic that uses them.
__device__ __forceinline__ void sched_fence() { __builtin_amdgcn_sched_barrier(0); }
// A value the compiler must have at this point: an expression that is only
// selected afterwards (cond ? v : 0) is otherwise moved under a branch
// together with its loads, one wait per sample.
__device__ __forceinline__ void pin(float &v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(double &v) { asm volatile("" : "+v"(v)); }
// A wave-uniform value kept in scalar registers.
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Truncation towards zero, saturated at the int range, 0 for NaN (the
// instruction's own behaviour; the C conversion leaves these undefined).
__device__ __forceinline__ int trunc_int(float v) {
    int r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ int trunc_int(double v) {
    int r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
__device__ __forceinline__ float fraction(float v) { return __builtin_amdgcn_fractf(v); }
__device__ __forceinline__ double fraction(double v) { return __builtin_amdgcn_fract(v); }

// kCH consecutive frame values: in raw form (16-byte loads, four registers
// for 16-bit frames) when the rows are aligned, converted when used.
template <typename TI>
struct Rows8 {
    static constexpr int kVec = kCH * (int)sizeof(TI) / 16;
    u4v q[kVec];
    __device__ __forceinline__ void load(const SS_GLOBAL TI *p) {
        const SS_GLOBAL u4v *v = (const SS_GLOBAL u4v *)p;
#pragma unroll
        for (int i = 0; i < kVec; i++) q[i] = v[i];
    }
    // rows past n read as 0
    __device__ __forceinline__ void load_ragged(const SS_GLOBAL TI *p, int n) {
        TI v[kCH];
#pragma unroll
        for (int i = 0; i < kCH; i++) v[i] = i < n ? p[i] : (TI)0;
        __builtin_memcpy(q, v, sizeof(q));
    }
    template <typename R>
    __device__ __forceinline__ R at(int i) const {
        if constexpr (sizeof(TI) == 2) {
            const uint32_t w = q[0][i >> 1];
            if constexpr (std::is_same<TI, uint16_t>::value) return (R)((i & 1) ? w >> 16 : w & 0xffffu);
            else return (R)((i & 1) ? (int)w >> 16 : (int)(int16_t)(w & 0xffffu));
        } else if constexpr (sizeof(TI) == 4) {
            return (R)__uint_as_float(q[i >> 2][i & 3]);
        } else {
            const uint32_t lo = q[i >> 1][2 * (i & 1)], hi = q[i >> 1][2 * (i & 1) + 1];
            return (R)__longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
        }
    }
};

// Rows per chunk: enough independent template gathers per wave to hide
// their latency, few enough that the unrolled chunk stays in registers
// (the kernel's *_SAMPLES tuning value).
template <typename R>
__host__ __device__ constexpr int chunk_rows(int samplesPerRow, int budget) {
    const int c = budget / samplesPerRow;
    return c < 1 ? 1 : (c > kCH ? kCH : c);
}

// Wave sums of NV per-thread doubles without LDS: two lane-swap steps that
// each add the halves of two values at once (lanes 32 apart, then 16 apart),
// then DPP row shifts by 8, 4, 2, 1.  Every value is added in the order
// ((l + l+32) + (l+16 + l+48)) ..., as a shuffle-down tree adds it; value i's
// sum ends in lane 16 * row(i & 3) of register i >> 2, rows 0 2 1 3.  (A
// column's 19 assembly sums were 228 LDS shuffles a wave and a chain of six
// LDS round trips.)
__device__ __forceinline__ void swap_add(double a, double b, double &out, bool half) {
    const long long ba = __double_as_longlong(a), bb = __double_as_longlong(b);
    const auto lo = half ? __builtin_amdgcn_permlane32_swap((int)ba, (int)bb, false, false)
                         : __builtin_amdgcn_permlane16_swap((int)ba, (int)bb, false, false);
    const auto hi = half ? __builtin_amdgcn_permlane32_swap((int)(ba >> 32), (int)(bb >> 32), false, false)
                         : __builtin_amdgcn_permlane16_swap((int)(ba >> 32), (int)(bb >> 32), false, false);
    const double x = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0]));
    const double y = __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
    out = x + y;
}
template <int CTRL>
__device__ __forceinline__ double row_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return v + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
template <int NV>
__device__ __forceinline__ void wave_sums(const double (&v)[NV], double (&q)[(NV + 3) / 4]) {
    constexpr int N2 = (NV + 1) / 2, N4 = (NV + 3) / 4;
    double h[N2];
#pragma unroll
    for (int i = 0; i < N2; i++) swap_add(v[2 * i], 2 * i + 1 < NV ? v[2 * i + 1] : 0.0, h[i], true);
#pragma unroll
    for (int i = 0; i < N4; i++) {
        swap_add(h[2 * i], 2 * i + 1 < N2 ? h[2 * i + 1] : 0.0, q[i], false);
        q[i] = row_add<0x108>(q[i]);  // row_shl:8: lane l adds lane l + 8 of its row
        q[i] = row_add<0x104>(q[i]);
        q[i] = row_add<0x102>(q[i]);
        q[i] = row_add<0x101>(q[i]);
    }
}

// Sum over the workgroup of NV per-thread doubles; thread i < NV gets sum i
// in out (LDS-backed, returns after a barrier).
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double *out) {
    __shared__ double sh[kWG / 64][(NV + 3) / 4 * 4];
    double q[(NV + 3) / 4];
    wave_sums<NV>(v, q);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if ((lane & 15) == 0) {
        const int row = lane >> 4, which = ((row & 1) << 1) | (row >> 1);
#pragma unroll
        for (int i = 0; i < (NV + 3) / 4; i++) sh[wave][4 * i + which] = q[i];
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kWG / 64; w++) s += sh[w][threadIdx.x];
        out[threadIdx.x] = s;
    }
    __syncthreads();
}

__device__ __forceinline__ int block_min(int v) {
    __shared__ int sh[kWG / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_down(v, off, 64));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    int m = sh[0];
#pragma unroll
    for (int w = 1; w < kWG / 64; w++) m = min(m, sh[w]);
    __syncthreads();
    return m;
}

__device__ __forceinline__ double reduce_pow(double v, double r, int k) {
    for (int i = 0; i < k; i++) v *= r;
    return v;
}

// Geometry of the pixels of one thread's run of rows: affine in the block's
// (column j, line i) coordinates -- the block matrix lists a block's pixels
// column-major, row r = j * L + i -- or read from the per-pixel table.
// FAST (see GroupDev::fast): a run is one image column's L lines, so j is
// fixed and i counts the rows.
template <typename R, bool FAST>
struct GeoRun {
    const SS_CONST AffineGeo<R> &a;
    R byb, fj, fi, Lf, f0, x0, y0;
    int affine, L;
    const SS_GLOBAL typename Nat<R>::V4 *tab;
    __device__ __forceinline__ GeoRun(GroupRef g, int b) : a(Prec<R>::aff(g)) {
        affine = FAST ? 1 : g.affine;
        L = g.L;
        byb = a.gy0 + a.gyb * (R)b;
        if constexpr (!FAST) {
            tab = (const SS_GLOBAL typename Nat<R>::V4 *)Prec<R>::geo(g) + (size_t)b * g.frameH;
            Lf = (R)L;
        }
    }
    __device__ __forceinline__ void start(int run, int r0) {
        fi = (R)0;
        if constexpr (FAST) {
            set_column((R)run);
        } else if (affine) {
            const int j = r0 / L;
            fi = (R)(r0 - j * L);
            set_column((R)j);
        }
    }
    __device__ __forceinline__ void set_column(R j) {
        fj = j;
        f0 = mad(a.fj, fj, a.f0);
        x0 = mad(a.gxj, fj, a.gx0);
        y0 = mad(a.gyj, fj, byb);
    }
    // the next CH rows, from row r on (rows past last repeat it)
    template <int CH>
    __device__ __forceinline__ void rows(int r, int last, R (&bx)[CH], R (&by)[CH], R (&f)[CH], bool (&m)[CH]) {
        if (FAST || affine) {
#pragma unroll
            for (int k = 0; k < CH; k++) {
                f[k] = mad(a.fi, fi, f0);
                bx[k] = mad(a.gxi, fi, x0);
                by[k] = mad(a.gyi, fi, y0);
                m[k] = true;
                fi += (R)1;
                if constexpr (!FAST) {
                    if (fi == Lf) {
                        fi = (R)0;
                        set_column(fj + (R)1);
                    }
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < CH; k++) {
                const typename Nat<R>::V4 q = tab[min(r + k, last)];
                bx[k] = q.x;
                by[k] = q.y;
                f[k] = q.z;
                m[k] = q.w != (R)0;
            }
        }
    }
};

// Two BF16 values packed in 32 bits (low half first) as a float pair.
__device__ __forceinline__ float2 bf16_pair(uint32_t u) {
    return make_float2(__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u));
}

// Bilinear template samples (task_differenceimage.cuh:13-32) from the paired
// layout.  A point outside the mask reads the nearest cell (the caller
// discards the value), so a wave issues all gathers of a chunk before it
// waits on any.  FAST addresses the template by 32-bit byte offsets.
template <typename R>
struct Tap {
    R fx, fy;
    typename Nat<R>::V2 top, bot;
    unsigned t;
};
template <typename R, bool FAST>
struct Template {
    const SS_GLOBAL char *row0, *row1;
    int tw, xl, yl;
    R xmax, ymax;
    __device__ __forceinline__ explicit Template(GroupRef g) {
        tw = g.tw;
        xl = g.tw - 2;
        yl = g.th - 2;
        xmax = (R)g.xmax;
        ymax = (R)g.ymax;
        row0 = (const SS_GLOBAL char *)Prec<R>::tp(g);
        row1 = row0 + (size_t)tw * sizeof(typename Nat<R>::V2);
    }
    __device__ __forceinline__ bool inside(R x, R y) const {
        // non-short-circuit: four compares combined without branches
        return (x >= (R)0) & (x < xmax) & (y >= (R)0) & (y < ymax);
    }
    __device__ __forceinline__ void fetch(R x, R y, Tap<R> &c) const {
        using V2 = typename Nat<R>::V2;
        const int ix = min(max(trunc_int(x), 0), xl), iy = min(max(trunc_int(y), 0), yl);
        c.fx = fraction(x);
        c.fy = fraction(y);
        c.t = __umul24(iy, tw) + ix;
        if constexpr (FAST) {
            const unsigned o = c.t * (unsigned)sizeof(V2);
            c.top = *(const SS_GLOBAL V2 *)(row0 + o);
            c.bot = *(const SS_GLOBAL V2 *)(row1 + o);
        } else {
            const size_t o = (size_t)((long long)iy * tw + ix) * sizeof(V2);
            c.t = (unsigned)(iy * tw + ix);
            c.top = *(const SS_GLOBAL V2 *)(row0 + o);
            c.bot = *(const SS_GLOBAL V2 *)(row1 + o);
        }
    }
};
template <typename R>
__device__ __forceinline__ R bilinear(const Tap<R> &c) {
    const R a = mad(c.fx, c.top.y - c.top.x, c.top.x);
    const R b = mad(c.fx, c.bot.y - c.bot.x, c.bot.x);
    return mad(c.fy, b - a, a);
}

// Template gradients at a sample (task_updategradients.cu): derived from the
// cell corners when they are forward differences, from the BF16 gradient
// pairs in mixed precision, else from the gradient pairs.
enum GradForm { GRAD_FD = 0, GRAD_PAIRS = 1, GRAD_BF16 = 2 };
template <typename R, int GRAD>
struct Grads {
    typename Nat<R>::V2 gx, gy;
    __device__ __forceinline__ void fetch(GroupRef g, const Tap<R> &c) {
        if constexpr (GRAD == GRAD_PAIRS) {
            gx = ((const SS_GLOBAL typename Nat<R>::V2 *)Prec<R>::gxv(g))[(size_t)c.t];
            gy = ((const SS_GLOBAL typename Nat<R>::V2 *)Prec<R>::gyh(g))[(size_t)c.t];
        }
        if constexpr (GRAD == GRAD_BF16) {  // pairs (G[t], G[t + step]) as two BF16 values
            gx.x = __uint_as_float(as_global(g.gxvB)[(size_t)c.t]);
            gy.x = __uint_as_float(as_global(g.gyhB)[(size_t)c.t]);
        }
    }
    __device__ __forceinline__ void eval(const Tap<R> &c, R &wx, R &wy) const {
        if constexpr (GRAD == GRAD_FD) {
            wx = mad(c.fy, (c.bot.y - c.bot.x) - (c.top.y - c.top.x), c.top.y - c.top.x);
            wy = mad(c.fx, (c.bot.y - c.top.y) - (c.bot.x - c.top.x), c.bot.x - c.top.x);
        } else if constexpr (GRAD == GRAD_BF16) {
            const float2 p = bf16_pair(__float_as_uint(gx.x)), q = bf16_pair(__float_as_uint(gy.x));
            wx = mad(c.fy, p.y - p.x, p.x);
            wy = mad(c.fx, q.y - q.x, q.x);
        } else {
            wx = mad(c.fy, gx.y - gx.x, gx.x);
            wy = mad(c.fx, gy.y - gy.x, gy.x);
        }
    }
};

// Knots of a column for candidate k of the line search (or the half-
// iteration start state for k < 0), as x = base_x + a + d * frac.
template <typename R>
struct ColKnots {
    R ax, dx, ay, dy;
    __device__ __forceinline__ R x(R bx, R f) const { return mad(dx, f, bx + ax); }
    __device__ __forceinline__ R y(R by, R f) const { return mad(dy, f, by + ay); }
};
template <typename R>
__device__ __forceinline__ ColKnots<R> make_knots(double lx, double rx, double ly, double ry) {
    return ColKnots<R>{uniform((R)lx), uniform((R)(rx - lx)), uniform((R)ly), uniform((R)(ry - ly))};
}
template <typename R>
__device__ __forceinline__ ColKnots<R> state_knots(GroupRef g, int c, int k) {
    const int N = g.N;
    const SS_CONST double *p0 = as_const(g.p0), *d0 = as_const(g.d0);
    double lx, ly, rx, ry;
    if (k < 0) {  // half-iteration start: p0 with the real right knot
        lx = p0[c];
        ly = p0[c + N];
        rx = p0[c + 1];
        ry = p0[c + 1 + N];
    } else {
        const double r = g.rmult;
        lx = p0[c] + reduce_pow(d0[c], r, k);
        ly = p0[c + N] + reduce_pow(d0[c + N], r, k);
        if (c + 1 == g.fframeW) {  // pnew of the group's last knot is never written
            rx = 1e6;
            ry = 1e6;
        } else {
            rx = p0[c + 1] + reduce_pow(d0[c + 1], r, k);
            ry = p0[c + 1 + N] + reduce_pow(d0[c + 1 + N], r, k);
        }
    }
    return make_knots<R>(lx, rx, ly, ry);
}

// Knots of column c from the current parameter vector p (applyParameters on p).
template <typename R>
__device__ __forceinline__ ColKnots<R> current_knots(GroupRef g, int c) {
    const int N = g.N;
    const SS_CONST double *p = as_const(g.p);
    return make_knots<R>(p[c], p[c + 1], p[c + N], p[c + 1 + N]);
}

template <typename TI>
__device__ __forceinline__ const SS_GLOBAL TI *column_ptr(GroupRef g, int c) {
    return (const SS_GLOBAL TI *)g.img + (size_t)c * g.frameH;
}

// Walks a thread's rows of a column in chunks of CH: body(r, n, I, off) gets
// the first row, the rows of the chunk inside the run (CH when FAST) and
// the frame values (chunk row k is I.at(off + k)).
template <int CH, bool FAST, typename TI, typename Start, typename Body>
__device__ __forceinline__ void walk_rows(GroupRef g, const SS_GLOBAL TI *img, Start &&start, Body &&body) {
    const int L = g.runLen, H = g.frameH;
    for (int run = threadIdx.x; run * L < H; run += kWG) {
        const int rend = min(run * L + L, H);
        start(run, run * L);
        for (int r0 = run * L; r0 < rend; r0 += kCH) {
            Rows8<TI> I;
            if (FAST || (g.vec && rend - r0 >= kCH)) I.load(img + r0);
            else I.load_ragged(img + r0, rend - r0);
#pragma unroll
            for (int q = 0; q < kCH; q += CH) {
                if (!FAST && r0 + q >= rend) break;
                body(r0 + q, FAST ? CH : min(CH, rend - r0 - q), I, q);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// assembly pass: warp + residual + errval terms + J^T J / J^T d partials
// (d_applyParameters, d_createDifferenceImage, d_calcBaseErrval,
//  d_updateGradients, d_fillDiagonals, d_fillJTr in one pass)
// ---------------------------------------------------------------------------
template <typename TI, typename R, int V, bool FAST, int GRAD>
__device__ __forceinline__ void assemble_column_t(GroupRef g, int c) {
    const int b = c % g.nb;
    const ColKnots<R> kn = current_knots<R>(g, c);
    const Template<R, FAST> T(g);
    GeoRun<R, FAST> geo(g, b);
    const SS_GLOBAL R *fnx = FAST || g.fracUniform ? nullptr : as_global(Prec<R>::fnext(g)) + (size_t)b * g.frameH;
    const int last = g.frameH - 1;
    // h[1] = sum I, h[i - 1] = column sum i for i >= CS_AXX; the errval term
    // is accumulated in FP64 per pixel: it decides line-search acceptance
    // against near-equal candidates
    double d2 = 0.0;
    R h[CS_N - 1];
#pragma unroll
    for (int i = 0; i < CS_N - 1; i++) h[i] = (R)0;
    int cnt = 0;
    constexpr int CH = chunk_rows<R>(2, tune_variant<TK_ASSEMBLE, R, V>().samples);
    walk_rows<CH, FAST>(
        g, column_ptr<TI>(g, c), [&](int run, int r0) { geo.start(run, r0); },
        [&](int r, int n, const Rows8<TI> &I, int off) {
            R bx[CH], by[CH], f[CH];
            bool ok[CH];
            Tap<R> tap[CH];
            Grads<R, GRAD> gr[CH];
            geo.template rows<CH>(r, last, bx, by, f, ok);
#pragma unroll
            for (int k = 0; k < CH; k++) {
                const R x = kn.x(bx[k], f[k]), y = kn.y(by[k], f[k]);
                ok[k] = (FAST || (k < n && ok[k])) && T.inside(x, y);
                T.fetch(x, y, tap[k]);
                gr[k].fetch(g, tap[k]);
            }
            sched_fence();
#pragma unroll
            for (int k = 0; k < CH; k++) {
                const R Ik = I.template at<R>(off + k);
                h[CS_SUMI] += Ik;
                R d = Ik - bilinear(tap[k]), wx, wy;
                gr[k].eval(tap[k], wx, wy);
                pin(d);
                pin(wx);
                pin(wy);
                // outside the mask every term below is zero
                d = ok[k] ? d : (R)0;
                wx = ok[k] ? wx : (R)0;
                wy = ok[k] ? wy : (R)0;
                const R fk = f[k];
                const R cf = (R)1 - fk;
                const R xx = wx * wx, yy = wy * wy, xy = wx * wy;
                const R c2 = cf * cf, f2 = fk * fk, fc = fk - f2;
                cnt += ok[k] ? 1 : 0;
                d2 = fma((double)d, (double)d, d2);
                h[CS_AXX - 1] = mad(xx, c2, h[CS_AXX - 1]);
                h[CS_AYY - 1] = mad(yy, c2, h[CS_AYY - 1]);
                h[CS_AXY - 1] = mad(xy, c2, h[CS_AXY - 1]);
                h[CS_BXX - 1] = mad(xx, f2, h[CS_BXX - 1]);
                h[CS_BYY - 1] = mad(yy, f2, h[CS_BYY - 1]);
                h[CS_BXY - 1] = mad(xy, f2, h[CS_BXY - 1]);
                h[CS_CXX - 1] = mad(xx, fc, h[CS_CXX - 1]);
                h[CS_CYY - 1] = mad(yy, fc, h[CS_CYY - 1]);
                h[CS_CXY - 1] = mad(xy, fc, h[CS_CXY - 1]);
                const R dc = d * cf, df = d * fk;
                h[CS_JXA - 1] = mad(dc, wx, h[CS_JXA - 1]);
                h[CS_JYA - 1] = mad(dc, wy, h[CS_JYA - 1]);
                h[CS_JXB - 1] = mad(df, wx, h[CS_JXB - 1]);
                h[CS_JYB - 1] = mad(df, wy, h[CS_JYB - 1]);
                if (!FAST && fnx) {
                    const R fn = fnx[min(r + k, last)];
                    const R n2 = fn * fn;
                    h[CS_QXX - 1] = mad(xx, n2, h[CS_QXX - 1]);
                    h[CS_QYY - 1] = mad(yy, n2, h[CS_QYY - 1]);
                    h[CS_QXY - 1] = mad(xy, n2, h[CS_QXY - 1]);
                }
            }
        });
    double v[CS_N];
    v[CS_D2] = d2;
    v[CS_SUMI] = (double)h[CS_SUMI];
    v[CS_CNT] = (double)cnt;
#pragma unroll
    for (int i = CS_AXX; i < CS_N; i++) v[i] = (double)h[i - 1];
    __shared__ double out[CS_N];
    block_sum<CS_N>(v, out);
    if (threadIdx.x < CS_N) g.colsum[(size_t)c * CS_N + threadIdx.x] = out[threadIdx.x];
}

template <typename TI, typename R, int V>
__device__ __forceinline__ void assemble_column(GroupRef g, int c) {
    if constexpr (sizeof(R) == 4) {
        if (g.gradBF16) {
            if (g.fast) assemble_column_t<TI, R, V, true, GRAD_BF16>(g, c);
            else assemble_column_t<TI, R, V, false, GRAD_BF16>(g, c);
            return;
        }
    }
    if (!g.gradFD) assemble_column_t<TI, R, V, false, GRAD_PAIRS>(g, c);
    else if (g.fast) assemble_column_t<TI, R, V, true, GRAD_FD>(g, c);
    else assemble_column_t<TI, R, V, false, GRAD_FD>(g, c);
}

template <typename TI, typename R>
__device__ __forceinline__ void final_column(GroupRef g, int c);

// The assembly launch also runs the final pass of the groups that stopped
// in the previous tick (phase PH_FINAL), for a tick without final stages.
template <typename TI, typename R, int V>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(tune_variant<TK_ASSEMBLE, R, V>().waves))) void k_assemble(Batch B) {
    for (int item = blockIdx.x; item < B.nItems; item += gridDim.x) {
        const int gi = as_const(B.itemGroup)[item];
        const int phase = as_const(B.ctl)[gi].phase;
        if (phase != PH_ASSEMBLE && phase != PH_FINAL) continue;
        GroupRef g = group_of(B, gi);
        if (!runs_here<TI, R>(g) || g.var[TK_ASSEMBLE] != V) continue;
        if (phase == PH_FINAL) {
            final_column<TI, R>(g, item - g.itemStart);
            continue;
        }
        if ((g.iterTimes || g.funcTimes) && item == g.itemStart && threadIdx.x == 0) {
            GroupCtl &c = B.ctl[gi];  // the first iteration starts (outputs 9 and 10)
            if (c.tIter == 0 || c.tStage == 0) {
                const unsigned long long now = wall_clock64();
                if (c.tIter == 0) c.tIter = now;
                if (c.tStage == 0) c.tStage = now;
            }
        }
        assemble_column<TI, R, V>(g, item - g.itemStart);
    }
}

// ---------------------------------------------------------------------------
// solve: errvals, knot usage, block-tridiagonal normal equations, exact FP64
// solve (partitioned block Thomas + cyclic reduction of the interface
// system), step filter, red/green expansion and line-search set-up.  One
// workgroup per group.
// ---------------------------------------------------------------------------
// level-0 equation of knot i:  O_{i-1} x_{i-1} + D_i x_i + O_i x_{i+1} = g_i,
// with D_i, O_i symmetric 2x2 ([xx xy; xy yy]).
struct Eq0 {
    double b0, b1, b2;  // D
    double c0, c1, c2;  // O (coupling to knot i+1)
    double d0, d1;      // rhs
};

struct M2 {  // general 2x2, row-major
    double a, b, c, d;
};
__device__ __forceinline__ M2 sym(double x0, double x1, double x2) { return M2{x0, x1, x1, x2}; }
__device__ __forceinline__ M2 inv(const M2 &m) {
    const double id = 1.0 / (m.a * m.d - m.b * m.c);
    return M2{m.d * id, -m.b * id, -m.c * id, m.a * id};
}
__device__ __forceinline__ M2 mul(const M2 &x, const M2 &y) {
    return M2{x.a * y.a + x.b * y.c, x.a * y.b + x.b * y.d, x.c * y.a + x.d * y.c,
              x.c * y.b + x.d * y.d};
}
__device__ __forceinline__ M2 add(const M2 &x, const M2 &y) { return M2{x.a + y.a, x.b + y.b, x.c + y.c, x.d + y.d}; }
__device__ __forceinline__ M2 sub(const M2 &x, const M2 &y) { return M2{x.a - y.a, x.b - y.b, x.c - y.c, x.d - y.d}; }
__device__ __forceinline__ M2 neg(const M2 &x) { return M2{-x.a, -x.b, -x.c, -x.d}; }
__device__ __forceinline__ M2 zero2() { return M2{0, 0, 0, 0}; }
__device__ __forceinline__ M2 eye2() { return M2{1, 0, 0, 1}; }
__device__ __forceinline__ double2 mulv(const M2 &m, double2 v) {
    return make_double2(m.a * v.x + m.b * v.y, m.c * v.x + m.d * v.y);
}

// x as an affine function of the neighbouring interface unknowns:
// x = y + V z_prev + W z_own
struct Aff {
    double2 y;
    M2 V, W;
};
__device__ __forceinline__ Aff aff_apply(const M2 &m, const Aff &a) {
    return Aff{mulv(m, a.y), mul(m, a.V), mul(m, a.W)};
}
__device__ __forceinline__ Aff aff_sub(const Aff &a, const Aff &b) {
    return Aff{make_double2(a.y.x - b.y.x, a.y.y - b.y.y), sub(a.V, b.V), sub(a.W, b.W)};
}

struct RedEq {  // reduced (interface) equation, general 2x2 blocks, B inverted
    M2 A, Bi, C;
    double2 d, x;
    double pad;  // neighbouring equations start in different LDS banks
};

struct InteriorRow {  // forward-eliminated interior row: Bh^{-1} and rhs
    M2 Bi;
    Aff R;
};

// The solve kernel's LDS besides the equations: the interface system, before
// it the first interiors' affine forms, after it the filter's partial scans.
struct SolveLds {
    union {
        RedEq red[kSolveWG];
        Aff first[kSolveWG];
        double scan[kSolveWG][4];
    };
    int hasInt[kSolveWG];
    __device__ SolveLds() {}
};

// Solver id 0 (SolverCuSparse::solve, cusparsesolver.cu:41-174): incomplete
// LU with zero fill of the normal equations ordered [x_0..x_{n-1},
// y_0..y_{n-1}] (the compacted COO order; unused knots are decoupled
// identity rows and change nothing), then the unit-lower and upper
// triangular solves.  With this ordering every row of the pattern is known:
// x_i: {x_{i-1}, x_i, x_{i+1}, y_{i-1}, y_i, y_{i+1}}, y_i likewise, so the
// elimination reduces to the recurrences below, applied in column order
// exactly as a row-wise ILU(0) does (separately rounded products).
struct IluRow {
    double lx;                        // x row: l(x_i, x_{i-1})
    double uxx, uxn, uxyp, uxy, uxyn; // u(x_i, x_i), u(x_i, x_{i+1}), u(x_i, y_{i-1}), u(x_i, y_i), u(x_i, y_{i+1})
    double l1, l2, l3, l4;            // y row: l(y_i, x_{i-1}), l(y_i, x_i), l(y_i, x_{i+1}), l(y_i, y_{i-1})
    double uyy, uyn;                  // u(y_i, y_i), u(y_i, y_{i+1})
};
static_assert(sizeof(IluRow) <= sizeof(InteriorRow), "ILU factors reuse the interior-row workspace");

__device__ void ilu0_solve(const Eq0 *E, IluRow *F, double2 *X, int n) {
#pragma clang fp contract(off)
    // x rows: the only lower entry is x_{i-1}
    for (int i = 0; i < n; i++) {
        const Eq0 q = E[i];
        IluRow r;
        r.uxx = q.b0;
        r.uxn = q.c0;
        r.uxy = q.b1;
        r.uxyn = q.c1;
        r.uxyp = 0.0;
        r.lx = 0.0;
        if (i > 0) {
            const Eq0 qp = E[i - 1];
            const IluRow &p = F[i - 1];
            r.uxyp = qp.c1;
            r.lx = qp.c0 / p.uxx;
            r.uxx = r.uxx - r.lx * p.uxn;
            r.uxyp = r.uxyp - r.lx * p.uxy;
            r.uxy = r.uxy - r.lx * p.uxyn;
        }
        F[i] = r;
    }
    // y rows: lower entries x_{i-1}, x_i, x_{i+1}, y_{i-1}
    for (int i = 0; i < n; i++) {
        const Eq0 q = E[i];
        IluRow &r = F[i];
        double ayxp = 0.0, ayx = q.b1, ayxn = q.c1, ayyp = 0.0, ayy = q.b2, ayyn = q.c2;
        r.l1 = r.l3 = r.l4 = 0.0;
        if (i > 0) {
            const IluRow &p = F[i - 1];
            ayxp = E[i - 1].c1;
            ayyp = E[i - 1].c2;
            r.l1 = ayxp / p.uxx;
            ayx = ayx - r.l1 * p.uxn;
            ayyp = ayyp - r.l1 * p.uxy;
            ayy = ayy - r.l1 * p.uxyn;
        }
        r.l2 = ayx / r.uxx;
        ayxn = ayxn - r.l2 * r.uxn;
        ayyp = ayyp - r.l2 * r.uxyp;
        ayy = ayy - r.l2 * r.uxy;
        ayyn = ayyn - r.l2 * r.uxyn;
        if (i + 1 < n) {
            const IluRow &nx = F[i + 1];
            r.l3 = ayxn / nx.uxx;
            ayy = ayy - r.l3 * nx.uxyp;
            ayyn = ayyn - r.l3 * nx.uxy;
        }
        if (i > 0) {
            const IluRow &p = F[i - 1];
            r.l4 = ayyp / p.uyy;
            ayy = ayy - r.l4 * p.uyn;
        }
        r.uyy = ayy;
        r.uyn = ayyn;
    }
    // forward: z = L^{-1} g (z kept in X)
    for (int i = 0; i < n; i++) {
        double zx = E[i].d0;
        if (i > 0) zx = zx - F[i].lx * X[i - 1].x;
        X[i].x = zx;
    }
    for (int i = 0; i < n; i++) {
        const IluRow &r = F[i];
        double zy = E[i].d1;
        if (i > 0) zy = zy - r.l1 * X[i - 1].x;
        zy = zy - r.l2 * X[i].x;
        if (i + 1 < n) zy = zy - r.l3 * X[i + 1].x;
        if (i > 0) zy = zy - r.l4 * X[i - 1].y;
        X[i].y = zy;
    }
    // backward: y rows from the last, then x rows
    for (int i = n - 1; i >= 0; i--) {
        double s = X[i].y;
        if (i + 1 < n) s = s - F[i].uyn * X[i + 1].y;
        X[i].y = s / F[i].uyy;
    }
    for (int i = n - 1; i >= 0; i--) {
        const IluRow &r = F[i];
        double s = X[i].x;
        if (i + 1 < n) s = s - r.uxn * X[i + 1].x;
        if (i > 0) s = s - r.uxyp * X[i - 1].y;
        s = s - r.uxy * X[i].y;
        if (i + 1 < n) s = s - r.uxyn * X[i + 1].y;
        X[i].x = s / r.uxx;
    }
}

// Level-0 equations of knots tid, tid + kSolveWG, ... (d_fillDiagonals /
// d_fillJTr entries, lambda extension) into put(k, equation, used).  Knot
// usage (d_createParameterMask): knot k < n is used when block column k or
// k - 1 reaches its block's minimum point count; knots from n on never are.
// Each knot takes its own and its neighbours' usage from the column counts,
// so that no pass over the flags has to come first, and every load is issued
// before any is used, at clamped indices instead of under a condition: one
// memory latency per knot, and the pointers do not alias, so that the next
// knots' loads overlap it.
template <typename Put>
__device__ __forceinline__ void level0_equations(const SS_GLOBAL double *__restrict__ S,
                                                 const SS_GLOBAL int *__restrict__ minPts, int n, int nb,
                                                 double lambda, int fracUniform, int tid, Put &&put) {
    const int q = fracUniform ? CS_BXX : CS_QXX;
#pragma unroll 4
    for (int k = tid; k < n; k += kSolveWG) {
        const SS_GLOBAL double *s = S + (size_t)k * CS_N;
        const SS_GLOBAL double *sp = k > 0 ? s - CS_N : s, *sn = k + 1 < n ? s + CS_N : s;
        const SS_GLOBAL double *spp = k > 1 ? sp - CS_N : sp;
        // block column of k - 2 .. k + 1
        const int b = k % nb, bp = b > 0 ? b - 1 : nb - 1, bpp = bp > 0 ? bp - 1 : nb - 1, bn = b + 1 < nb ? b + 1 : 0;
        double dxx = s[CS_AXX], dyy = s[CS_AYY], dxy = s[CS_AXY];
        double jx = s[CS_JXA], jy = s[CS_JYA];
        const double cxx = s[CS_CXX], cxy = s[CS_CXY], cyy = s[CS_CYY];
        const double pxx = sp[q], pyy = sp[q + 1], pxy = sp[q + 2], pjx = sp[CS_JXB], pjy = sp[CS_JYB];
        const double cnt = s[CS_CNT], cntP = sp[CS_CNT], cntPP = spp[CS_CNT], cntN = sn[CS_CNT];
        const int mp = minPts[b], mpP = minPts[bp], mpPP = minPts[bpp], mpN = minPts[bn];
        const bool c = cnt >= (double)mp, cP = k > 0 && cntP >= (double)mpP;
        const bool cPP = k > 1 && cntPP >= (double)mpPP, cN = k + 1 < n && cntN >= (double)mpN;
        const bool u = c || cP, up = k > 0 && (cP || cPP), un = k + 1 < n && (cN || c);
        if (k > 0) {
            dxx += pxx;
            dyy += pyy;
            dxy += pxy;
            jx += pjx;
            jy += pjy;
        }
        const double nl = (double)(up ? 1 : 0) + (double)(un ? 1 : 0);
        Eq0 e;
        e.b0 = u ? dxx + lambda * nl : 1.0;
        e.b1 = u ? dxy : 0.0;
        e.b2 = u ? dyy + lambda * nl : 1.0;
        e.c0 = u && un ? cxx - lambda : 0.0;
        e.c1 = u && un ? cxy : 0.0;
        e.c2 = u && un ? cyy - lambda : 0.0;
        e.d0 = u ? jx : 0.0;
        e.d1 = u ? jy : 0.0;
        put(k, e, u);
    }
}

// Where the equations of a group lie.  Few enough: in LDS, in order.  More:
// in memory as 16-byte pieces [row of the partition][piece][thread], so that
// the threads, each walking the rows of its own partition, load and store
// consecutive addresses.
struct LdsRows {
    Eq0 *E;
    int m;
    __device__ __forceinline__ Eq0 load(int t, int r) const { return E[t * m + r]; }
    __device__ __forceinline__ Eq0 knot(int k) const { return E[k]; }
    __device__ __forceinline__ void put(int k, const Eq0 &e) const { E[k] = e; }
    __device__ __forceinline__ void put_rhs(int k, double d0, double d1) const {
        E[k].d0 = d0;
        E[k].d1 = d1;
    }
};
struct MemRows {
    SS_GLOBAL d2v *E;
    int m;
    __device__ __forceinline__ SS_GLOBAL d2v *at(int t, int r) const { return E + (size_t)r * 4 * kSolveWG + t; }
    __device__ __forceinline__ Eq0 load(int t, int r) const {
        const SS_GLOBAL d2v *q = at(t, r);
        const d2v a = q[0], b = q[kSolveWG], c = q[2 * kSolveWG], d = q[3 * kSolveWG];
        return Eq0{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
    }
    __device__ __forceinline__ Eq0 knot(int k) const { return load(k / m, k % m); }
    __device__ __forceinline__ void put(int k, const Eq0 &e) const {
        SS_GLOBAL d2v *q = at(k / m, k % m);
        q[0] = d2v{e.b0, e.b1};
        q[kSolveWG] = d2v{e.b2, e.c0};
        q[2 * kSolveWG] = d2v{e.c1, e.c2};
        q[3 * kSolveWG] = d2v{e.d0, e.d1};
    }
    __device__ __forceinline__ void put_rhs(int k, double d0, double d1) const {
        at(k / m, k % m)[3 * kSolveWG] = d2v{d0, d1};
    }
};
// The solution, in LDS or in memory.
struct Solution {
    double2 *lds;
    SS_GLOBAL d2v *mem;
    bool inLds;
    __device__ __forceinline__ double2 get(int k) const {
        if (inLds) return lds[k];
        const d2v v = mem[k];
        return make_double2(v.x, v.y);
    }
    __device__ __forceinline__ void set(int k, double2 v) const {
        if (inLds) lds[k] = v;
        else mem[k] = d2v{v.x, v.y};
    }
};

// 2x2 products with the rounding fixed: the second product rounded, the first
// fused to it, as the compiler contracts the plain forms above in straight
// code (elsewhere it may pick the other one).
__device__ __forceinline__ M2 mul_f(const M2 &x, const M2 &y) {
    return M2{fma(x.a, y.a, x.b * y.c), fma(x.a, y.b, x.b * y.d), fma(x.c, y.a, x.d * y.c), fma(x.c, y.b, x.d * y.d)};
}
__device__ __forceinline__ double2 mulv_f(const M2 &m, double2 v) {
    return make_double2(fma(m.a, v.x, m.b * v.y), fma(m.c, v.x, m.d * v.y));
}
// ... the first product rounded, the second fused to it
__device__ __forceinline__ M2 mul_s(const M2 &x, const M2 &y) {
    return M2{fma(x.b, y.c, x.a * y.a), fma(x.b, y.d, x.a * y.b), fma(x.d, y.c, x.c * y.a), fma(x.d, y.d, x.c * y.b)};
}
__device__ __forceinline__ double2 mulv_s(const M2 &m, double2 v) {
    return make_double2(fma(m.b, v.y, m.a * v.x), fma(m.d, v.y, m.c * v.x));
}
// ... of an inverse: the off-diagonal product rounded
__device__ __forceinline__ double2 mulv_i(const M2 &m, double2 v) {
    return make_double2(fma(m.a, v.x, m.b * v.y), fma(m.d, v.y, m.c * v.x));
}
__device__ __forceinline__ M2 inv_f(const M2 &m) {
    const double id = 1.0 / fma(m.a, m.d, -(m.b * m.c));
    return M2{m.d * id, -m.b * id, -m.c * id, m.a * id};
}
__device__ __forceinline__ Aff aff_apply_f(const M2 &m, const Aff &a) {
    return Aff{mulv_f(m, a.y), mul_f(m, a.V), mul_f(m, a.W)};
}

// Interface system of the partitioned solve: thread t < P contributes the
// equation of its partition's last knot z_t in terms of z_{t-1} and z_{t+1}
// (its last interior row as lastA, the next partition's first interior row
// as firstAff[t + 1]); cyclic reduction solves it.  Called by all threads;
// returns z_t and z_{t-1} (0 for t = 0).
__device__ __forceinline__ void solve_interfaces(bool interior, const Aff &first, const Aff &lastA, const Eq0 &q,
                                                 const M2 &A, SolveLds &S, int P, int tid, double2 &zo, double2 &zp) {
#pragma clang fp contract(off)
    RedEq *red = S.red;
    if (tid < P) {
        S.hasInt[tid] = interior ? 1 : 0;
        S.first[tid] = first;
    }
    __syncthreads();
    // x_{j+1}: first interior of partition t+1, or z_{t+1}
    Aff F{make_double2(0, 0), zero2(), eye2()};
    if (tid + 1 < P && S.hasInt[tid + 1]) F = S.first[tid + 1];
    __syncthreads();  // the interface system takes the affine forms' memory
    // Cyclic reduction, in place: level l's equation k is that of thread
    // k * 2^l + 2^l - 1.  A thread keeps its own equation in registers and
    // leaves the others what they read of it: the inverse of B, which its
    // back substitution takes too, A, C and d.  (With whole equations read
    // from LDS and both neighbours' B inverted by every reader, the system of
    // 96 knots took 17,000 cycles of a launch's 30,000.)
    M2 B = zero2(), Bi = zero2(), Ai = zero2(), C = zero2();
    double2 d = make_double2(0, 0);
    auto publish = [&]() {
        Bi = inv_f(B);
        red[tid].A = Ai;
        red[tid].Bi = Bi;
        red[tid].C = C;
        red[tid].d = d;
    };
    if (tid < P) {
        const M2 Cn = sym(q.c0, q.c1, q.c2);
        Ai = mul_f(A, lastA.V);
        B = add(add(sym(q.b0, q.b1, q.b2), mul_f(A, lastA.W)), mul_f(Cn, F.V));
        C = mul_f(Cn, F.W);
        const double2 ay = mulv_f(A, lastA.y), cy = mulv_f(Cn, F.y);
        d = make_double2(q.d0 - ay.x - cy.x, q.d1 - ay.y - cy.y);
        if (tid == 0) Ai = zero2();
        publish();
    }
    __syncthreads();
    int nlev = 0;
    for (int mm = P; mm > 1; mm >>= 1) nlev++;
    for (int l = 0; l < nlev; l++) {
        const int st = 1 << l;
        if (tid < P && ((tid + 1) & (2 * st - 1)) == 0) {
            const RedEq em = red[tid - st];
            const M2 al = neg(mul_f(Ai, em.Bi));
            Ai = mul_s(al, em.A);
            B = add(B, mul_s(al, em.C));
            double2 t = mulv_s(al, em.d);
            double2 o = make_double2(d.x + t.x, d.y + t.y);
            if (tid + st < P) {
                const RedEq ep = red[tid + st];
                const M2 ga = neg(mul_f(C, ep.Bi));
                B = add(B, mul_s(ga, ep.A));
                C = mul_s(ga, ep.C);
                t = mulv_s(ga, ep.d);
                o = make_double2(o.x + t.x, o.y + t.y);
            } else {
                C = zero2();
            }
            d = o;
            publish();
        }
        __syncthreads();
    }
    zo = make_double2(0, 0);
    zp = make_double2(0, 0);
    for (int l = nlev; l >= 0; l--) {
        const int st = 1 << l;
        if (tid < P && ((tid + 1) & (2 * st - 1)) == st) {  // eliminated at level l
            double2 r = d;
            if (tid >= st) {
                const double2 t = mulv_f(Ai, red[tid - st].x);
                r.x -= t.x;
                r.y -= t.y;
            }
            if (tid + st < P) {
                const double2 t = mulv_f(C, red[tid + st].x);
                r.x -= t.x;
                r.y -= t.y;
            }
            zo = mulv_i(Bi, r);
            red[tid].x = zo;
        }
        __syncthreads();
    }
    if (tid < P && tid > 0) zp = red[tid - 1].x;
}

// Exact FP64 solve of the level-0 block-tridiagonal system E (knots 0..n-1)
// into X: partitioned block Thomas + cyclic reduction of the interface
// system.  Thread t owns knots [s, e); its interior rows s..e-2 are
// eliminated in terms of the interfaces z_{t-1} = x_{s-1} and z_t = x_{e-1}.
// Called by all threads of the workgroup.
//
// Partitions of at most M knots keep their rows and eliminated rows in
// registers (one round of loads).
template <int M, typename Rows>
__device__ __forceinline__ void exact_solve_reg(const Rows &E, const Solution &X, SolveLds &S, int n, int tid) {
    const int m = (n + kSolveWG - 1) / kSolveWG;
    const int P = (n + m - 1) / m;
    const int s0 = tid * m, e0 = min(n, s0 + m);
    const int len = e0 - s0;
    Eq0 q[M];
    InteriorRow ir[M];
    Eq0 qm{};  // row s0 - 1
    Aff lastA, first;
    Eq0 qj{};  // row e0 - 1
    M2 A = zero2();
    const bool interior = len >= 2;
    if (tid < P) {
#pragma unroll
        for (int r = 0; r < M; r++)
            if (r < len) q[r] = E.load(tid, r);
        if (s0 > 0) qm = E.load(tid - 1, m - 1);
        if (interior) {
            // forward elimination
            M2 BiPrev = zero2();
            Aff Rprev;
#pragma unroll
            for (int r = 0; r < M - 1; r++) {
                if (r > len - 2) continue;
                const Eq0 &qq = q[r];
                M2 Bh = sym(qq.b0, qq.b1, qq.b2);
                Aff R{make_double2(qq.d0, qq.d1), zero2(), zero2()};
                if (r == 0) {
                    if (tid > 0) R.V = neg(sym(qm.c0, qm.c1, qm.c2));
                } else {
                    const Eq0 &qp = q[r - 1];
                    const M2 Ap = sym(qp.c0, qp.c1, qp.c2);  // A_i = O_{i-1}
                    const M2 Lm = mul(Ap, BiPrev);
                    Bh = sub(Bh, mul(Lm, Ap));
                    R = aff_sub(R, aff_apply(Lm, Rprev));
                }
                if (r == len - 2) R.W = neg(sym(qq.c0, qq.c1, qq.c2));
                const M2 Bi = inv(Bh);
                ir[r] = InteriorRow{Bi, R};
                BiPrev = Bi;
                Rprev = R;
            }
            // back substitution of the affine forms
            Aff Xa = aff_apply(BiPrev, Rprev);
            lastA = Xa;
#pragma unroll
            for (int r = M - 3; r >= 0; r--) {
                if (r > len - 3) continue;
                const Eq0 &qq = q[r];
                const Aff t = aff_sub(ir[r].R, aff_apply(sym(qq.c0, qq.c1, qq.c2), Xa));
                Xa = aff_apply(ir[r].Bi, t);
            }
            first = Xa;
        } else {
            lastA = Aff{make_double2(0, 0), eye2(), zero2()};      // x_{e-2} := z_prev
            first = Aff{make_double2(0, 0), zero2(), eye2()};      // unused
        }
        // the interface row j = e0 - 1 and its coupling A = O_{j-1}
        const int j = e0 - 1;
#pragma unroll
        for (int r = 0; r < M; r++)
            if (r == len - 1) qj = q[r];
        if (len >= 2) {
#pragma unroll
            for (int r = 0; r < M - 1; r++)
                if (r == len - 2) A = sym(q[r].c0, q[r].c1, q[r].c2);
        } else if (j > 0) {
            A = sym(qm.c0, qm.c1, qm.c2);
        }
    }
    double2 zo, zp;
    solve_interfaces(interior, first, lastA, qj, A, S, P, tid, zo, zp);
    // interior reconstruction: x_i = Bi_i (R_i(z) - O_i x_{i+1})
    if (tid < P) {
        X.set(e0 - 1, zo);
        double2 xn = zo;
#pragma unroll
        for (int r = M - 2; r >= 0; r--) {
            if (r > len - 2) continue;
            const InteriorRow &iri = ir[r];
            const double2 v = mulv_s(iri.R.V, zp), w = mulv_f(iri.R.W, zo);
            double2 rr = make_double2(iri.R.y.x + v.x + w.x, iri.R.y.y + v.y + w.y);
            if (r < len - 2) {
                const double2 t = mulv_f(sym(q[r].c0, q[r].c1, q[r].c2), xn);
                rr.x -= t.x;
                rr.y -= t.y;
            }
            xn = mulv_f(iri.Bi, rr);
            X.set(s0 + r, xn);
        }
    }
    __threadfence_block();
    __syncthreads();
}

// Longer partitions walk their rows, the next ones loaded while these are
// eliminated, and keep the eliminated rows in IR (workspace, laid out like
// MemRows).  The same arithmetic in the same order.
template <typename Rows>
__device__ __forceinline__ void exact_solve_mem(const Rows &E, SS_GLOBAL d2v *IR, const Solution &X, SolveLds &S, int n,
                                                int tid) {
#pragma clang fp contract(off)
    const int m = (n + kSolveWG - 1) / kSolveWG;
    const int P = (n + m - 1) / m;
    const int s0 = tid * m, e0 = min(n, s0 + m);
    const int len = e0 - s0;
    constexpr int kAhead = 4;
    Aff lastA, first;
    Eq0 qj{};  // row e0 - 1
    M2 A = zero2();
    const bool interior = len >= 2;
    constexpr int kPieces = 7;  // 16-byte pieces of an InteriorRow
    auto irow = [&](int r) { return IR + (size_t)r * kPieces * kSolveWG + tid; };
    struct Row {
        Eq0 q;
        InteriorRow ir;
    };
    auto load_row = [&](int r) {
        const SS_GLOBAL d2v *p = irow(r);
        d2v v[kPieces];
#pragma unroll
        for (int u = 0; u < kPieces; u++) v[u] = p[u * kSolveWG];
        return Row{E.load(tid, r),
                   InteriorRow{M2{v[0].x, v[0].y, v[1].x, v[1].y},
                               Aff{make_double2(v[2].x, v[2].y), M2{v[3].x, v[3].y, v[4].x, v[4].y},
                                   M2{v[5].x, v[5].y, v[6].x, v[6].y}}}};
    };
    // rows top .. 0 in turn, the next ones loaded ahead
    auto rows_down = [&](int top, auto &&body) {
        Row ahead[2];
        ahead[0] = load_row(max(top, 0));
        ahead[1] = load_row(max(top - 1, 0));
        for (int r = top; r >= 0; r--) {
            const Row w = ahead[0];
            ahead[0] = ahead[1];
            ahead[1] = load_row(max(r - 2, 0));
            body(r, w);
        }
    };
    if (tid < P) {
        if (interior) {
            // forward elimination
            M2 BiPrev = zero2();
            Aff Rprev;
            Eq0 qp{}, ahead[kAhead];
            if (tid > 0) qp = E.load(tid - 1, m - 1);
#pragma unroll
            for (int u = 0; u < kAhead; u++) ahead[u] = E.load(tid, min(u, len - 1));
            for (int r = 0; r <= len - 2; r++) {
                const Eq0 qq = ahead[0];
#pragma unroll
                for (int u = 0; u + 1 < kAhead; u++) ahead[u] = ahead[u + 1];
                ahead[kAhead - 1] = E.load(tid, min(r + kAhead, len - 1));
                M2 Bh = sym(qq.b0, qq.b1, qq.b2);
                Aff R{make_double2(qq.d0, qq.d1), zero2(), zero2()};
                if (r == 0) {
                    if (tid > 0) R.V = neg(sym(qp.c0, qp.c1, qp.c2));
                } else {
                    const M2 Ap = sym(qp.c0, qp.c1, qp.c2);  // A_i = O_{i-1}
                    const M2 Lm = mul_f(Ap, BiPrev);
                    Bh = sub(Bh, mul_f(Lm, Ap));
                    R = aff_sub(R, aff_apply_f(Lm, Rprev));
                }
                if (r == len - 2) R.W = neg(sym(qq.c0, qq.c1, qq.c2));
                const M2 Bi = inv_f(Bh);
                SS_GLOBAL d2v *p = irow(r);
                p[0] = d2v{Bi.a, Bi.b};
                p[kSolveWG] = d2v{Bi.c, Bi.d};
                p[2 * kSolveWG] = d2v{R.y.x, R.y.y};
                p[3 * kSolveWG] = d2v{R.V.a, R.V.b};
                p[4 * kSolveWG] = d2v{R.V.c, R.V.d};
                p[5 * kSolveWG] = d2v{R.W.a, R.W.b};
                p[6 * kSolveWG] = d2v{R.W.c, R.W.d};
                BiPrev = Bi;
                Rprev = R;
                qp = qq;
            }
            // back substitution of the affine forms
            Aff Xa = aff_apply_f(BiPrev, Rprev);
            lastA = Xa;
            rows_down(len - 3, [&](int, const Row &w) {
                const Aff t = aff_sub(w.ir.R, aff_apply_f(sym(w.q.c0, w.q.c1, w.q.c2), Xa));
                Xa = aff_apply_f(w.ir.Bi, t);
            });
            first = Xa;
        } else {
            lastA = Aff{make_double2(0, 0), eye2(), zero2()};      // x_{e-2} := z_prev
            first = Aff{make_double2(0, 0), zero2(), eye2()};      // unused
        }
        // the interface row j = e0 - 1 and its coupling A = O_{j-1}
        qj = E.load(tid, len - 1);
        if (e0 - 1 > 0) {
            const Eq0 qp = len >= 2 ? E.load(tid, len - 2) : E.load(tid - 1, m - 1);
            A = sym(qp.c0, qp.c1, qp.c2);
        }
    }
    double2 zo, zp;
    solve_interfaces(interior, first, lastA, qj, A, S, P, tid, zo, zp);
    // interior reconstruction: x_i = Bi_i (R_i(z) - O_i x_{i+1})
    if (tid < P) {
        X.set(e0 - 1, zo);
        double2 xn = zo;
        if (interior)
            rows_down(len - 2, [&](int r, const Row &w) {
                const double2 v = mulv_f(w.ir.R.V, zp), z = mulv_f(w.ir.R.W, zo);
                double2 rr = make_double2(w.ir.R.y.x + v.x + z.x, w.ir.R.y.y + v.y + z.y);
                if (r < len - 2) {
                    const double2 t = mulv_f(sym(w.q.c0, w.q.c1, w.q.c2), xn);
                    rr.x -= t.x;
                    rr.y -= t.y;
                }
                xn = mulv_f(w.ir.Bi, rr);
                X.set(s0 + r, xn);
            });
    }
    __threadfence_block();
    __syncthreads();
}

// knots per partition that stay in registers
constexpr int kSolveRegRows = 8;
// Knots whose level-0 equations the solve keeps in LDS (114 KiB).  Groups of
// more knots keep their solution there instead (four times as many), and the
// knots' usage beside it.  The rest of the 160 KiB holds the interface system.
// One workgroup walks a group's rows, 16 per thread at 4096 knots, so latency
// bounds the launch: with equations and eliminated rows one after the other
// per thread in memory, a launch over groups of up to 4096 knots (10 groups,
// FP32 with refinement) took 199 us; in pieces that a wave loads side by side,
// the next rows ahead, and the solution in LDS, 122 us, and 105 with the
// equations' loads in one round and the reduction in registers.  4096 knots
// without neighbours 131 -> 82 -> 70 us; with the equations in LDS (1600
// knots, FP64) 45 -> 40 -> 33 us; 96 knots 16.8 -> 16 -> 11 us.
constexpr int kSolveLdsRows = 1824, kSolveLdsKnots = 4 * kSolveLdsRows;

// Inlined into the solve kernel: as a called function it would save and
// restore the callee-saved registers it uses (over 200 per call).
template <typename Rows>
__device__ __forceinline__ void exact_solve(const Rows &E, SS_GLOBAL d2v *IR, const Solution &X, SolveLds &S, int n,
                                            int tid) {
    if ((n + kSolveWG - 1) / kSolveWG <= kSolveRegRows)
        exact_solve_reg<kSolveRegRows>(E, X, S, n, tid);
    else
        exact_solve_mem(E, IR, X, S, n, tid);
}

// The exact solve with, in mixed precision, one step of iterative refinement
// in FP64: r = g - H x, H e = r, x += e (the matrix entries stay; each knot's
// right-hand side is replaced by its residual; Xs keeps x).
template <typename Rows>
__device__ __forceinline__ void solve_refined(const Rows &E, SS_GLOBAL d2v *IR, const Solution &X, SS_GLOBAL d2v *Xs,
                                              SolveLds &S, int n, int refine, int tid) {
#pragma clang fp contract(off)
    exact_solve(E, IR, X, S, n, tid);
    if (!refine) return;
    // each thread its partition's rows, loaded four at a time
    const int m = (n + kSolveWG - 1) / kSolveWG;
    const int s0 = tid * m, len = min(n, s0 + m) - s0;
    Eq0 qp{};  // the row before
    if (len > 0 && s0 > 0) qp = E.load(tid - 1, m - 1);
    for (int r0 = 0; r0 < len; r0 += 4) {
        Eq0 q4[4];
#pragma unroll
        for (int u = 0; u < 4; u++) q4[u] = E.load(tid, min(r0 + u, len - 1));
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = s0 + r0 + u;
            if (r0 + u >= len) break;
            const Eq0 q = q4[u];
            const double2 x = X.get(k);
            double r0_ = q.d0 - fma(q.b0, x.x, q.b1 * x.y);
            double r1_ = q.d1 - fma(q.b1, x.x, q.b2 * x.y);
            if (k > 0) {
                const double2 xp = X.get(k - 1);
                r0_ -= fma(qp.c0, xp.x, qp.c1 * xp.y);
                r1_ -= fma(qp.c1, xp.x, qp.c2 * xp.y);
            }
            if (k + 1 < n) {
                const double2 xn = X.get(k + 1);
                r0_ -= fma(q.c0, xn.x, q.c1 * xn.y);
                r1_ -= fma(q.c1, xn.x, q.c2 * xn.y);
            }
            Xs[k] = d2v{x.x, x.y};
            E.put_rhs(k, r0_, r1_);
            qp = q;
        }
    }
    __threadfence_block();
    __syncthreads();
    exact_solve(E, IR, X, S, n, tid);
    for (int k = tid; k < n; k += kSolveWG) {
        const double2 e = X.get(k);
        const d2v x = Xs[k];
        X.set(k, make_double2(x.x + e.x, x.y + e.y));
    }
    __threadfence_block();
    __syncthreads();
}

// Output 10: the device time since the group's last stage end goes to slot
// `slot`.  Called by one thread of a per-group kernel.
template <typename G>
__device__ __forceinline__ void stage_time(G &g, GroupCtl &ctl, int slot) {
    if (!g.funcTimes) return;
    const unsigned long long now = wall_clock64();
    if (ctl.tStage) g.funcTimes[slot] += (double)(now - ctl.tStage) / g.clockHz;
    ctl.tStage = now;
}

__device__ void final_finish(GroupRef g, GroupCtl &ctl);

// The solve launch also ends the groups whose final pass ran in the
// assembly launch before it (phase PH_FINAL).
__global__ __launch_bounds__(kSolveWG) void k_solve(Batch B) {
    const int gi = blockIdx.x;
    GroupCtl &ctl = B.ctl[gi];
    GroupRef g = group_of(B, gi);
    // read ahead; this launch writes the phase
    const SS_GLOBAL GroupCtl &was = as_global(B.ctl)[gi];
    const int phase = was.phase, shift = was.shift;
    const int nF = g.nF, nb = g.nb, N = g.N, n = g.fframeW, G = g.groupSize;
    loaded(phase, shift, nF, nb, N, n, G, g.colsum, g.minPts, g.deltaP, g.p, g.d0, g.p0, g.errval, g.ws, g.lambda,
           g.fracUniform, g.solverId, g.refine, g.funcTimes);
    if (phase == PH_FINAL) {
        final_finish(g, ctl);
        return;
    }
    if (phase != PH_ASSEMBLE) return;
    const int tid = threadIdx.x;
    SS_GLOBAL double *deltaP = (SS_GLOBAL double *)g.deltaP, *d0 = (SS_GLOBAL double *)g.d0,
                     *p0 = (SS_GLOBAL double *)g.p0;
    const SS_GLOBAL double *p = as_global(g.p);
    // filter deactivation after max_filter_iterations (mainiteration.cpp:80-90)
    __shared__ int s_filter;
    if (tid == 0) {
        if (ctl.nFilterIterations != 0 && ctl.iteration > ctl.nFilterIterations) {
            ctl.solverFilter = 0;
            ctl.filterID = 0;
            ctl.nFilterIterations = 0;
        }
        s_filter = ctl.solverFilter;
        stage_time(g, ctl, FT_ASSEMBLY);
    }
    const SS_GLOBAL double *S = as_global(g.colsum);
    const SS_GLOBAL int *minPts = as_global(g.minPts);
    // The loops below load a batch of entries before they use any of it:
    // one thread per frame or knot would otherwise wait out a memory latency
    // per entry.  The additions keep their order.
    constexpr int kBatch = 8;
    // 1. per-frame errval of this shift (d_calcAllGroupErrval): a frame's
    //    columns in batches of 32 (one round of loads for 512x512 frames).
    //    From the last thread on: a small group's equations are the first
    //    waves' work, and the two run beside each other.
    constexpr int kEvBatch = 32;
    SS_GLOBAL double *errval = (SS_GLOBAL double *)g.errval + shift * nF;
    for (int f = kSolveWG - 1 - tid; f < nF; f += kSolveWG) {
        const SS_GLOBAL double *col = S + (size_t)f * nb * CS_N;
        double s = 0.0, c = 0.0;
        for (int b0 = 0; b0 < nb; b0 += kEvBatch) {
            double vs[kEvBatch], vc[kEvBatch];
#pragma unroll
            for (int u = 0; u < kEvBatch; u++) {
                const int bb = min(b0 + u, nb - 1);
                vs[u] = col[(size_t)bb * CS_N + CS_D2];
                vc[u] = col[(size_t)bb * CS_N + CS_CNT];
            }
#pragma unroll
            for (int u = 0; u < kEvBatch; u++) {
                if (b0 + u < nb) {
                    s += vs[u];
                    c += vc[u];
                }
            }
        }
        errval[f] = s / c;
    }
    // The knots' state that step 6 starts from, a batch per thread, ahead of
    // the solve.
    double dv0[kBatch], pv0[kBatch];
    auto load_state = [&](int i0) {
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int idx = min(i0 + u * kSolveWG + tid, 2 * N - 1);
            dv0[u] = deltaP[idx];
            pv0[u] = p[idx];
        }
    };
    load_state(0);
    // 2. knot usage (d_createParameterMask) and level-0 equations
    //    (d_fillDiagonals / d_fillJTr entries, lambda extension); the knots
    //    from n on are never used.
    __shared__ __align__(16) Eq0 sE[kSolveLdsRows];
    __shared__ uint8_t sUsed[kSolveLdsKnots];
    __shared__ SolveLds sS;
    const int m = (n + kSolveWG - 1) / kSolveWG;
    const bool rowsInLds = n <= kSolveLdsRows, usedInLds = n <= kSolveLdsKnots;
    SS_GLOBAL uint8_t *gUsed = (SS_GLOBAL uint8_t *)g.used;
    auto set_used = [&](int k, bool u) {
        if (usedInLds) sUsed[k] = u;
        else gUsed[k] = u;
    };
    auto used = [&](int k) {
        uint8_t u;
        if (usedInLds) u = sUsed[k];
        else u = gUsed[k];
        return u != 0;
    };
    // workspace: [equations][eliminated rows][solution][saved solution]
    const size_t rows = (size_t)n + kSolveWG;
    double *ws = g.ws;
    SS_GLOBAL d2v *IR = (SS_GLOBAL d2v *)(ws + rows * 8);
    double2 *Xmem = reinterpret_cast<double2 *>(ws + rows * (8 + sizeof(InteriorRow) / sizeof(double)));
    SS_GLOBAL d2v *Xs = (SS_GLOBAL d2v *)(Xmem + rows);
    // The solution takes the equations' LDS where they are in memory, and
    // where the exact solve without refinement, its partitions in registers,
    // has read every equation before its first barrier and writes the
    // solution after the last.
    const bool xInLds = rowsInLds ? g.solverId != 0 && !g.refine && m <= kSolveRegRows
                                  : g.solverId != 0 && n <= kSolveLdsKnots;
    const Solution X{reinterpret_cast<double2 *>(sE), (SS_GLOBAL d2v *)Xmem, xInLds};
    auto equations = [&](auto &&put) {
        level0_equations(S, minPts, n, nb, g.lambda, g.fracUniform, tid, [&](int k, const Eq0 &e, bool u) {
            put(k, e);
            set_used(k, u);
        });
        __threadfence_block();
        __syncthreads();
    };
    if (g.solverId == 0) {
        // 4a. solver id 0: ILU(0) in x-then-y order (one thread, the
        //     reference's recurrence order)
        Eq0 *E = rowsInLds ? sE : reinterpret_cast<Eq0 *>(ws);
        equations([&](int k, const Eq0 &e) { E[k] = e; });
        if (tid == 0) ilu0_solve(E, (IluRow *)(ws + rows * 8), Xmem, n);
        __threadfence_block();
        __syncthreads();
    } else if (rowsInLds) {
        const LdsRows E{sE, m};
        equations([&](int k, const Eq0 &e) { E.put(k, e); });
        solve_refined(E, IR, X, Xs, sS, n, g.refine, tid);
    } else {
        const MemRows E{(SS_GLOBAL d2v *)ws, m};
        equations([&](int k, const Eq0 &e) { E.put(k, e); });
        solve_refined(E, IR, X, Xs, sS, n, g.refine, tid);
    }
    // 5. step filter over the used knots, x sequence then y sequence
    //    (SmearingFilter::apply / RangeFilter::apply on the compacted halves)
    const int filterKind = s_filter;
    const double strength = g.strength;
    if (filterKind == 1) {
        double (*sa)[4] = sS.scan;
        const int chunk = (n + kSolveWG - 1) / kSolveWG;
        const int c0 = min(n, tid * chunk), c1 = min(n, c0 + chunk);
        double ax = 1, bx = 0, ay = 1, by = 0;
        for (int k = c0; k < c1; k++) {
            if (!used(k)) continue;
            ax *= strength;
            const double2 x = X.get(k);
            bx = strength * bx + (1 - strength) * x.x;
            ay *= strength;
            by = strength * by + (1 - strength) * x.y;
        }
        sa[tid][0] = ax;
        sa[tid][1] = bx;
        sa[tid][2] = ay;
        sa[tid][3] = by;
        __syncthreads();
        for (int st = 1; st < kSolveWG; st <<= 1) {
            double v0 = 0, v1 = 0, v2 = 0, v3 = 0;
            const bool has = tid >= st;
            if (has) {
                v0 = sa[tid - st][0];
                v1 = sa[tid - st][1];
                v2 = sa[tid - st][2];
                v3 = sa[tid - st][3];
            }
            __syncthreads();
            if (has) {
                const double a0 = sa[tid][0], b0 = sa[tid][1], a1 = sa[tid][2], b1 = sa[tid][3];
                sa[tid][0] = a0 * v0;
                sa[tid][1] = a0 * v1 + b0;
                sa[tid][2] = a1 * v2;
                sa[tid][3] = a1 * v3 + b1;
            }
            __syncthreads();
        }
        double yx = tid > 0 ? sa[tid - 1][1] : 0.0;
        double yy = tid > 0 ? sa[tid - 1][3] : 0.0;
        for (int k = c0; k < c1; k++) {
            if (!used(k)) continue;
            const double2 x = X.get(k);
            yx = yx * strength + x.x * (1 - strength);
            yy = yy * strength + x.y * (1 - strength);
            X.set(k, make_double2(yx, yy));
        }
        __threadfence_block();
        __syncthreads();
    } else if (filterKind == 2) {
        if (tid == 0) {
            for (int axis = 0; axis < 2; axis++) {
                int pv = -1, cu = -1;
                for (int k = 0; k < n; k++) {
                    if (!used(k)) continue;
                    if (pv >= 0 && cu >= 0) {
                        const double2 xm = X.get(pv), xp = X.get(k);
                        double2 xc = X.get(cu);
                        const double vm = axis ? xm.y : xm.x;
                        const double vi = axis ? xc.y : xc.x;
                        const double vp = axis ? xp.y : xp.x;
                        const double tc = (vm + vp) / 2;
                        const double diff = (tc - vm) * strength;
                        bool rep;
                        if (vm < vp) rep = vi > vp + diff || vi < vm - diff;
                        else rep = vi < vp + diff || vi > vm - diff;
                        if (rep) {
                            if (axis) xc.y = tc;
                            else xc.x = tc;
                            X.set(cu, xc);
                        }
                    }
                    pv = cu;
                    cu = k;
                }
            }
        }
        __threadfence_block();
        __syncthreads();
    }
    // 6. d_expandResults (task_expandresults.cu:10-41) and line-search set-up
    for (int i0 = 0; i0 < 2 * N; i0 += kSolveWG * kBatch) {
        if (i0 > 0) load_state(i0);
        double xv[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int idx = min(i0 + u * kSolveWG + tid, 2 * N - 1);
            const int j = idx >= N ? idx - N : idx, jj = min(j, n - 1);
            const bool uj = j < n && used(jj);
            const double2 x = X.get(jj);
            xv[u] = uj ? (idx >= N ? x.y : x.x) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int idx = i0 + u * kSolveWG + tid;
            if (idx < 2 * N) {
                const bool fixed = ((((idx + 1) - (shift * (G >> 1))) % G) == 0);
                const double v = fixed ? dv0[u] : xv[u];
                deltaP[idx] = v;
                d0[idx] = v;
                p0[idx] = pv0[u];
            }
        }
    }
    for (int f = tid; f < nF; f += kSolveWG) {
        g.lsActive[f] = 1;
        g.lsNextK[f] = 0;
        g.lsMk[f] = -1;
        g.lsDk[f] = -1;
    }
    if (tid == 0) {
        ctl.slotRounds = 0;
        ctl.roundsThisLS = 0;
        ctl.K = g.K1;
        ctl.phase = PH_LS;
        stage_time(g, ctl, FT_SOLVE);
    }
}

// ---------------------------------------------------------------------------
// line search: K fused candidates p0 + r^k * delta of every active frame
// (the tries of d_linesearch, task_linesearch.cu:35-106, in one pass), then
// one wave per frame resolves the tries sequentially.  A tick runs kLsSlots
// such rounds per half-iteration; after the last one, one wave per group
// does the rounds' bookkeeping.  Separate kernels, so that no device-scope
// fence is needed: on gfx950 each one writes back and invalidates the XCD's
// L2.  Round `slot` of a tick's half-iteration slots runs K = ctl.K
// candidates in slot 0 (K1 after the solve, Kn when the line search goes on
// from the previous slots) and Kn after it; no round runs past maxRounds.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool ls_round_runs(GroupRef g, int roundsThisLS, int slot) {
    return roundsThisLS + slot < g.maxRounds;
}
template <typename G, typename C>
__device__ __forceinline__ int ls_round_k(G &g, C &ctl, int slot) {
    return slot == 0 ? ctl.K : g.Kn;
}

// Candidates k0 .. k0 + K - 1 of column c; their sums go to the column's
// candidate slots slot0 .. slot0 + K - 1.
template <typename TI, typename R, int V, int K, bool FAST>
__device__ __forceinline__ void ls_column_t(GroupRef g, int c, int b, int k0, int slot0) {
    ColKnots<R> kn[K];
    {
        const int N = g.N;
        const double r = g.rmult;
        const SS_CONST double *p0 = as_const(g.p0), *d0 = as_const(g.d0);
        double dlx = reduce_pow(d0[c], r, k0), dly = reduce_pow(d0[c + N], r, k0);
        double drx = reduce_pow(d0[c + 1], r, k0), dry = reduce_pow(d0[c + 1 + N], r, k0);
        const bool lastKnot = (c + 1 == g.fframeW);
        const double plx = p0[c], ply = p0[c + N], prx = p0[c + 1], pry = p0[c + 1 + N];
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double lx = plx + dlx, ly = ply + dly;
            const double rx = lastKnot ? 1e6 : prx + drx, ry = lastKnot ? 1e6 : pry + dry;
            kn[k] = make_knots<R>(lx, rx, ly, ry);
            dlx *= r;
            dly *= r;
            drx *= r;
            dry *= r;
        }
    }
    const Template<R, FAST> T(g);
    GeoRun<R, FAST> geo(g, b);
    const int last = g.frameH - 1;
    double e2[K];  // FP64: compared against the half-iteration's errval
    int cnt[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        e2[k] = 0.0;
        cnt[k] = 0;
    }
    constexpr int CH = chunk_rows<R>(K, tune_variant<TK_LS, R, V>().samples);
    walk_rows<CH, FAST>(
        g, column_ptr<TI>(g, c), [&](int run, int r0) { geo.start(run, r0); },
        [&](int r, int n, const Rows8<TI> &I, int off) {
            R bx[CH], by[CH], f[CH];
            bool m[CH], ok[CH][K];
            Tap<R> tap[CH][K];
            geo.template rows<CH>(r, last, bx, by, f, m);
#pragma unroll
            for (int q = 0; q < CH; q++)
#pragma unroll
                for (int k = 0; k < K; k++) {
                    const R x = kn[k].x(bx[q], f[q]), y = kn[k].y(by[q], f[q]);
                    ok[q][k] = (FAST || (q < n && m[q])) && T.inside(x, y);
                    T.fetch(x, y, tap[q][k]);
                }
            sched_fence();
#pragma unroll
            for (int q = 0; q < CH; q++) {
                const R Iq = I.template at<R>(off + q);
#pragma unroll
                for (int k = 0; k < K; k++) {
                    R d = Iq - bilinear(tap[q][k]);
                    pin(d);
                    d = ok[q][k] ? d : (R)0;
                    e2[k] = fma((double)d, (double)d, e2[k]);
                    cnt[k] += ok[q][k] ? 1 : 0;
                }
            }
        });
    double v[2 * K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        v[2 * k] = e2[k];
        v[2 * k + 1] = (double)cnt[k];
    }
    __shared__ double out[2 * kMaxCand];
    block_sum<2 * K>(v, out);
    if (threadIdx.x < 2 * K) g.lssum[(size_t)c * 2 * kMaxCand + 2 * slot0 + threadIdx.x] = out[threadIdx.x];
}

template <typename TI, typename R, int V, int K>
__device__ __forceinline__ void ls_column(GroupRef g, int c, int b, int k0, int slot0) {
    if (g.fast) ls_column_t<TI, R, V, K, true>(g, c, b, k0, slot0);
    else ls_column_t<TI, R, V, K, false>(g, c, b, k0, slot0);
}

// split = 2: work item w covers column w % nItems and, of a round of four
// candidates, the two of half w / nItems (each candidate's sums are the
// same whichever workgroup computes them); other rounds run in half 0.
template <typename TI, typename R, int V>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(tune_variant<TK_LS, R, V>().waves))) void k_ls_round(Batch B, int slot, int split) {
    const int nWork = B.nItems * split;
    for (int w = blockIdx.x; w < nWork; w += gridDim.x) {
        const int half = w >= B.nItems ? 1 : 0, item = w - half * B.nItems;
        const int gi = as_const(B.itemGroup)[item];
        const SS_CONST GroupCtl &ctl = as_const(B.ctl)[gi];
        if (ctl.phase != PH_LS) continue;
        GroupRef g = group_of(B, gi);
        if (!runs_here<TI, R>(g) || g.var[TK_LS] != V || !ls_round_runs(g, ctl.roundsThisLS, slot)) continue;
        const int c = item - g.itemStart, f = c / g.nb, b = c % g.nb;
        if (!as_const(g.lsActive)[f]) continue;
        int K = ls_round_k(g, ctl, slot), k0 = as_const(g.lsNextK)[f], slot0 = 0;
        if (split == 2 && K == 4) {
            K = 2;
            k0 += 2 * half;
            slot0 = 2 * half;
        } else if (half) {
            continue;
        }
        switch (K) {
        case 1: ls_column<TI, R, V, 1>(g, c, b, k0, slot0); break;
        case 2: ls_column<TI, R, V, 2>(g, c, b, k0, slot0); break;
        default: ls_column<TI, R, V, 4>(g, c, b, k0, slot0); break;
        }
    }
}

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}
__device__ __forceinline__ double wave_max(double x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off, 64));
    return x;
}
// lane u's value, u the same in all lanes
__device__ __forceinline__ double lane_value(double x, int u) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(x), u), hi = __builtin_amdgcn_readlane(__double2hiint(x), u);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ int wave_or(int x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x |= __shfl_xor(x, off, 64);
    return x;
}

// Sequential resolution of the candidates of frame f (reproduces the
// reference's try / reduce / movement-threshold order) and commit.  One
// wave per frame.
__device__ __forceinline__ void ls_decide_frame(GroupRef g, const SS_CONST GroupCtl &ctl, GroupCtl &out, int f, int K,
                                                int slot) {
    const int nb = g.nb, N = g.N, nF = g.nF;
    const int lane = threadIdx.x;
    const SS_GLOBAL double *d0 = as_global(g.d0) + (size_t)f * nb, *p0 = as_global(g.p0) + (size_t)f * nb;
    const SS_GLOBAL int *minPts = as_global(g.minPts);
    SS_GLOBAL double *errval = (SS_GLOBAL double *)g.errval + ctl.shift * nF;
    // all that the decision and the commit read, before any of it is used
    const int active = as_global(g.lsActive)[f], k0 = as_global(g.lsNextK)[f];
    const double ev = errval[f];
    const double r = g.rmult, thr = g.thr;
    struct Column {
        double d0x, d0y, p0x, p0y;
        int minPts;
        d2v ls[kMaxCand];
    };
    auto column = [&](int bb) {
        const SS_GLOBAL d2v *ls = (const SS_GLOBAL d2v *)g.lssum + (size_t)(f * nb + bb) * kMaxCand;
        Column q{d0[bb], d0[bb + N], p0[bb], p0[bb + N], minPts[bb], {}};
#pragma unroll
        for (int k = 0; k < kMaxCand; k++) q.ls[k] = ls[k];
        return q;
    };
    const Column q0 = column(min(lane, nb - 1));
    asm volatile("" ::"v"(active), "v"(k0), "v"(ev), "v"(q0.p0y), "v"(q0.minPts), "v"(q0.ls[kMaxCand - 1].x));
    if (!active) return;
    double se[kMaxCand], sn[kMaxCand];
#pragma unroll
    for (int k = 0; k < kMaxCand; k++) se[k] = sn[k] = 0.0;
    int pres = 0;  // bit k: some column of candidate k reaches its block's min points
    double dmax = 0.0;
    for (int bb = lane; bb < nb; bb += 64) {
        const Column q = bb < 64 ? q0 : column(bb);
#pragma unroll
        for (int k = 0; k < kMaxCand; k++) {
            if (k < K) {
                se[k] += q.ls[k].x;
                sn[k] += q.ls[k].y;
                if (q.ls[k].y >= (double)q.minPts) pres |= 1 << k;
            }
        }
        dmax = fmax(dmax, fmax(fabs(q.d0x), fabs(q.d0y)));
    }
#pragma unroll
    for (int k = 0; k < kMaxCand; k++) {
        if (k < K) {
            se[k] = wave_sum(se[k]);
            sn[k] = wave_sum(sn[k]);
        }
    }
    pres = wave_or(pres);
    dmax = wave_max(dmax);
    int fin = -1, acc = -1;
    if (lane == 0) {
        double dm = reduce_pow(dmax, r, k0);
        int mk = -1, tries = 0;
        for (int kk = 0; kk < K && fin < 0; kk++) {
            const int k = k0 + kk;
            tries++;
            mk = k;
            if (!((pres >> kk) & 1)) {
                const double dm1 = dm * r;
                if (!(dm1 > thr)) fin = k + 1;
                dm = dm1;
            } else {
                g.lsDk[f] = k;
                double e = 0.0, c = 0.0;
#pragma unroll
                for (int q = 0; q < kMaxCand; q++)
                    if (q == kk) {
                        e = se[q];
                        c = sn[q];
                    }
                e /= c;
                if (e < ev) {
                    acc = k;
                    fin = k;
                    if (f == 0) errval[0] = e;
                } else if (!(dm > thr)) {
                    fin = k;
                } else {
                    dm *= r;
                }
            }
        }
        g.lsMk[f] = mk;
        atomicAdd(&out.tries, tries);
        atomicAdd(&out.lsFramePasses, 1);
        atomicMax(&out.slotRounds, slot + 1);
        if (fin < 0) g.lsNextK[f] = k0 + K;
        else g.lsActive[f] = 0;
    }
    fin = __shfl(fin, 0, 64);
    acc = __shfl(acc, 0, 64);
    if (fin >= 0) {
        SS_GLOBAL double *deltaP = (SS_GLOBAL double *)g.deltaP + (size_t)f * nb, *p = (SS_GLOBAL double *)g.p + (size_t)f * nb;
        for (int bb = lane; bb < nb; bb += 64) {
            double d0x = q0.d0x, d0y = q0.d0y, p0x = q0.p0x, p0y = q0.p0y;
            if (bb >= 64) {
                d0x = d0[bb];
                d0y = d0[bb + N];
                p0x = p0[bb];
                p0y = p0[bb + N];
            }
            deltaP[bb] = reduce_pow(d0x, r, fin);
            deltaP[bb + N] = reduce_pow(d0y, r, fin);
            if (acc >= 0) {
                p[bb] = p0x + reduce_pow(d0x, r, acc);
                p[bb + N] = p0y + reduce_pow(d0y, r, acc);
            }
        }
    }
}

__global__ __launch_bounds__(64) void k_ls_decide(Batch B, int slot) {
    for (int fi = blockIdx.x; fi < B.nFrames; fi += gridDim.x) {
        const int gi = group_index(B, B.frameGroup, fi);
        // the sums and flags that the decisions change are not read here
        const SS_CONST GroupCtl &ctl = as_const(B.ctl)[gi];
        GroupRef g = group_of(B, gi);
        const int phase = ctl.phase, rounds = ctl.roundsThisLS, K = ls_round_k(g, ctl, slot);
        loaded(phase, rounds, K, ctl.shift, g.maxRounds, g.frameStart, g.nb, g.N, g.nF, g.lsActive, g.lsNextK, g.lssum,
               g.errval, g.d0, g.p0, g.minPts);
        if (phase != PH_LS || !ls_round_runs(g, rounds, slot)) continue;
        ls_decide_frame(g, ctl, B.ctl[gi], fi - g.frameStart, K, slot);
    }
}

// After a tick's last line-search slot: the rounds' bookkeeping, and either
// the next slots' frames or the end of the half-iteration (`improved`,
// task_linesearch.cu:117-125) and of MainIteration::execute
// (mainiteration.cpp:103-118).  A half-iteration that ends in an earlier
// slot leaves the later slots with no active frame.
__global__ __launch_bounds__(64) void k_ls_finish(Batch B) {
    const int gi = blockIdx.x;
    GroupCtl &ctl = B.ctl[gi];
    GroupRef g = group_of(B, gi);
    const SS_GLOBAL GroupCtl &was = as_global(B.ctl)[gi];  // read ahead; this launch writes these fields
    const int nF = g.nF, phase = was.phase, shift = was.shift, it0 = was.iteration;
    const int improved = was.improved, nFilterIterations = was.nFilterIterations, slotRounds = was.slotRounds;
    const int rounds = was.rounds + slotRounds, roundsThisLS = was.roundsThisLS + slotRounds;
    const int halfIterations = was.halfIterations + 1;
    loaded(nF, phase, shift, it0, improved, nFilterIterations, rounds, roundsThisLS, halfIterations, g.Kn, g.maxRounds,
           g.errval, g.lsActive, g.rgParams, g.maxIter, g.funcTimes);
    if (phase != PH_LS) return;
    // the frames' error values, 64 at a time, each added in the frames' order
    const SS_GLOBAL double *ev = as_global(g.errval);
    int active = 0;
    double e0 = 0.0, e1 = 0.0;
    for (int f0 = 0; f0 < nF; f0 += 64) {
        const int f = min(f0 + (int)threadIdx.x, nF - 1), in = f0 + (int)threadIdx.x < nF;
        const double v0 = ev[f], v1 = ev[f + nF];
        active += in ? as_global(g.lsActive)[f] : 0;
        const int m = min(64, nF - f0);
#pragma unroll 4
        for (int u = 0; u < m; u++) {
            e0 += lane_value(v0, u);
            e1 += lane_value(v1, u);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) active += __shfl_xor(active, off, 64);
    if (active == 0 && g.rgParams && it0 <= g.maxIter) {  // output 14 (timedmainiteration.cpp:124)
        const int P = 2 * g.N;
        double *dst = g.rgParams + (size_t)P * (size_t)(shift + 2 * (it0 - 1));
        for (int i = threadIdx.x; i < P; i += 64) dst[i] = g.p[i];
    }
    if (threadIdx.x != 0) return;
    stage_time(g, ctl, FT_LINESEARCH);
    ctl.rounds = rounds;
    ctl.roundsThisLS = roundsThisLS;
    ctl.slotRounds = 0;
    if (active > 0) {
        ctl.K = g.Kn;
        if (roundsThisLS >= g.maxRounds) {
            ctl.error = 4;  // SS_ERR_NUMERICAL
            ctl.phase = PH_ERROR;
        }
        return;
    }
    // half-iteration complete
    const int imp = improved & ((shift && e0 > e1) || (!shift && e0 < e1));
    ctl.improved = imp;
    ctl.halfIterations = halfIterations;
    if (shift == 0) {
        ctl.shift = 1;
        ctl.phase = PH_ASSEMBLE;
        return;
    }
    if (!imp && nFilterIterations != 0) {
        ctl.solverFilter = 0;
        ctl.nFilterIterations = 0;
        ctl.improved = 1;  // run this iteration again without the filter
        ctl.shift = 0;
        ctl.phase = PH_ASSEMBLE;
        return;
    }
    ctl.iterImproved = imp;
    ctl.phase = PH_CORR;
}

// ---------------------------------------------------------------------------
// global correlation statistic (hd_globalCorrelation,
// task_correlation.cu:63-99) of every frame's last-tried state; the
// statistic of a column covers its leading run of masked rows only.
// ---------------------------------------------------------------------------
template <typename TI, typename R, int V, bool FAST, bool ONE>
__device__ __forceinline__ void corr_column_t(GroupRef g, int c) {
    const int f = c / g.nb, b = c % g.nb;
    const int mk = as_const(g.lsMk)[f], dk = as_const(g.lsDk)[f];
    const bool same = (mk == dk);
    const ColKnots<R> km = state_knots<R>(g, c, mk);
    const ColKnots<R> kd = state_knots<R>(g, c, dk);
    const SS_GLOBAL TI *img = column_ptr<TI>(g, c);
    const Template<R, FAST> T(g);
    GeoRun<R, FAST> geo(g, b);
    const int last = g.frameH - 1;
    // First row outside the mask of the last-tried state: the moments cover
    // the rows before it.  Where a thread has at most two runs of rows (ONE),
    // it needs no pass of its own for it: it stops at its own first row
    // outside, keeps the moments of its first run, and takes back what lies
    // behind the column's first row outside once all threads are through.
    // 20 groups of 50 512x512 frames, FP64: 166 -> 148 us a launch; FP32, 24
    // uneven groups: 126 -> 121 us.
    int firstOut = g.frameH;
    constexpr int CH = chunk_rows<R>(1, tune_variant<TK_CORR, R, V>().samples);
    const int start2 = (threadIdx.x + kWG) * g.runLen;  // the second run's first row
    if constexpr (!ONE) {
        for (int run = threadIdx.x; run * g.runLen < g.frameH; run += kWG) {
            const int rend = min(run * g.runLen + g.runLen, g.frameH);
            geo.start(run, run * g.runLen);
            for (int r0 = run * g.runLen; r0 < rend && r0 < firstOut; r0 += CH) {
                R bx[CH], by[CH], f1[CH];
                bool m[CH];
                geo.template rows<CH>(r0, last, bx, by, f1, m);
#pragma unroll
                for (int q = 0; q < CH; q++) {
                    const R x = km.x(bx[q], f1[q]), y = km.y(by[q], f1[q]);
                    if ((FAST || r0 + q < rend) && !(m[q] && T.inside(x, y))) firstOut = min(firstOut, r0 + q);
                }
            }
        }
        firstOut = block_min(firstOut);
    }
    double first[CR_N];  // the moments of the first run
    double v[CR_N];
#pragma unroll
    for (int i = 0; i < CR_N; i++) v[i] = first[i] = 0.0;
    walk_rows<CH, FAST>(
        g, img,
        [&](int run, int r0) {
            geo.start(run, r0);
            if (ONE && run >= kWG) {
#pragma unroll
                for (int i = CR_SA; i < CR_N; i++) first[i] = v[i];
            }
        },
        [&](int r, int n, const Rows8<TI> &I, int off) {
            R bx[CH], by[CH], f1[CH];
            bool m[CH], mm[CH], okd[CH];
            Tap<R> tap[CH];
            geo.template rows<CH>(r, last, bx, by, f1, m);
            R xd[CH], yd[CH];
#pragma unroll
            for (int q = 0; q < CH; q++) {
                m[q] = FAST || (q < n && m[q]);
                xd[q] = km.x(bx[q], f1[q]);
                yd[q] = km.y(by[q], f1[q]);
                okd[q] = mm[q] = m[q] && T.inside(xd[q], yd[q]);
            }
            // the difference image holds the last-decided state's residual
            if (!same) {
#pragma unroll
                for (int q = 0; q < CH; q++) {
                    xd[q] = kd.x(bx[q], f1[q]);
                    yd[q] = kd.y(by[q], f1[q]);
                    okd[q] = m[q] && T.inside(xd[q], yd[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < CH; q++) T.fetch(xd[q], yd[q], tap[q]);
            sched_fence();
#pragma unroll
            for (int q = 0; q < CH; q++) {
                const R Iq = I.template at<R>(off + q);
                R d = Iq - bilinear(tap[q]);
                pin(d);
                const R dbuf = okd[q] ? d : (R)0;
                const R w = Iq - dbuf;
                const double Id = FAST || q < n ? (double)Iq : 0.0;
                v[CR_SUMD] += (double)(mm[q] ? w : dbuf);
                v[CR_NMASK] += mm[q] ? 1.0 : 0.0;
                if (ONE && (FAST || q < n) && !mm[q]) firstOut = min(firstOut, r + q);
                const bool lead = r + q < firstOut;  // rows before it are all inside the mask
                const double a = lead ? (double)w : 0.0, bb = lead ? Id : 0.0;
                v[CR_SA] += a;
                v[CR_SAA] += a * a;
                v[CR_SB] += bb;
                v[CR_SBB] += bb * bb;
                v[CR_SAB] += a * bb;
                v[CR_NS] += lead ? 1.0 : 0.0;
            }
        });
    if constexpr (ONE) {
        firstOut = block_min(firstOut);
        const bool none = firstOut <= (int)threadIdx.x * g.runLen, one = start2 < g.frameH && firstOut <= start2;
#pragma unroll
        for (int i = CR_SA; i < CR_N; i++) v[i] = none ? 0.0 : one ? first[i] : v[i];
    }
    __shared__ double out[CR_N];
    block_sum<CR_N>(v, out);
    if (threadIdx.x < CR_N) g.corrsum[(size_t)c * CR_N + threadIdx.x] = out[threadIdx.x];
}

template <typename TI, typename R, int V>
__device__ __forceinline__ void corr_column(GroupRef g, int c) {
    const bool one = g.frameH <= 2 * kWG * g.runLen;
    if (g.fast && one) corr_column_t<TI, R, V, true, true>(g, c);
    else if (g.fast) corr_column_t<TI, R, V, true, false>(g, c);
    else if (one) corr_column_t<TI, R, V, false, true>(g, c);
    else corr_column_t<TI, R, V, false, false>(g, c);
}

template <typename TI, typename R, int V>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(tune_variant<TK_CORR, R, V>().waves))) void k_corr(Batch B) {
    for (int item = blockIdx.x; item < B.nItems; item += gridDim.x) {
        const int gi = as_const(B.itemGroup)[item];
        if (as_const(B.ctl)[gi].phase != PH_CORR) continue;
        GroupRef g = group_of(B, gi);
        if (!runs_here<TI, R>(g) || g.var[TK_CORR] != V) continue;
        corr_column<TI, R, V>(g, item - g.itemStart);
    }
}

// Flag 'c': the frame correlation taken right after the global correlation
// (task.cpp:286-293).  The global correlation swaps every masked pixel to
// image - difference but swaps back only the row-major pixels below its
// grid, fframeW rounded up to 256 (task_correlation.cu:97); the frame
// correlation then swaps every masked pixel once more
// (task_correlation.cu:176-178).  Sums over all of the column's rows, in
// finalsum's slots (free while the group is in this phase).  A kernel of its
// own, launched only for batches that ask for it, so that the correlation
// kernel's register allocation does not carry it.
template <typename TI, typename R>
__device__ void frame_corr_column(GroupRef g, int c) {
    const int f = c / g.nb, b = c % g.nb;
    const int mk = as_const(g.lsMk)[f], dk = as_const(g.lsDk)[f];
    const bool same = (mk == dk);
    const ColKnots<R> km = state_knots<R>(g, c, mk);
    const ColKnots<R> kd = state_knots<R>(g, c, dk);
    const Template<R, false> T(g);
    GeoRun<R, false> geo(g, b);
    const int last = g.frameH - 1;
    constexpr int CH = chunk_rows<R>(1, sizeof(R) == 8 ? kFinalSamplesF64 : kFinalSamplesF32);
    const long long swapBack = min((long long)((g.fframeW + 255) / 256) * 256, (long long)g.frameH * g.fframeW);
    double w[FC_N];
#pragma unroll
    for (int i = 0; i < FC_N; i++) w[i] = 0.0;
    walk_rows<CH, false>(
        g, column_ptr<TI>(g, c), [&](int run, int r0) { geo.start(run, r0); },
        [&](int r, int n, const Rows8<TI> &I, int off) {
            R bx[CH], by[CH], f1[CH];
            bool m[CH];
            geo.template rows<CH>(r, last, bx, by, f1, m);
#pragma unroll
            for (int q = 0; q < CH; q++) {
                const bool in = q < n && m[q];
                R xd = km.x(bx[q], f1[q]), yd = km.y(by[q], f1[q]);
                const bool mm = in && T.inside(xd, yd);
                bool okd = mm;
                if (!same) {
                    xd = kd.x(bx[q], f1[q]);
                    yd = kd.y(by[q], f1[q]);
                    okd = in && T.inside(xd, yd);
                }
                Tap<R> tap;
                T.fetch(xd, yd, tap);
                const R smp = bilinear(tap);
                const R Ir = q < n ? I.template at<R>(off + q) : (R)0;
                const R dbuf = okd ? Ir - smp : (R)0;
                const bool pre = (long long)(r + q) * g.fframeW + c < swapBack;
                const R d1 = Ir - dbuf;           // the global correlation's swap
                const R d2 = pre ? Ir - d1 : d1;  // its partial swap-back
                const R d3 = mm ? Ir - d2 : dbuf; // the frame correlation's swap
                const double a = mm ? (double)d3 : 0.0, bb = mm ? (double)Ir : 0.0;
                // an unmasked pixel enters the reference's second pass times 0
                // (task_correlation.cu:150-156): NaN or Inf there gives NaN
                const double za = q < n ? (double)d3 * 0.0 : 0.0, zb = (double)Ir * 0.0;
                w[FC_CNT] += mm ? 1.0 : 0.0;
                w[FC_SA] += a;
                w[FC_SAA] += mm ? a * a : za * za;
                w[FC_SB] += bb;
                w[FC_SBB] += mm ? bb * bb : zb * zb;
                w[FC_SAB] += a * bb;
            }
        });
    __shared__ double outF[FC_N];
    block_sum<FC_N>(w, outF);
    if (threadIdx.x < FC_N) g.finalsum[(size_t)c * FS_N + threadIdx.x] = outF[threadIdx.x];
}

template <typename TI, typename R>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(2))) void k_corr_frames(Batch B) {
    for (int item = blockIdx.x; item < B.nItems; item += gridDim.x) {
        const int gi = as_const(B.itemGroup)[item];
        if (as_const(B.ctl)[gi].phase != PH_CORR) continue;
        GroupRef g = group_of(B, gi);
        if (!g.fcIter || !runs_here<TI, R>(g)) continue;
        frame_corr_column<TI, R>(g, item - g.itemStart);
    }
}

// Global correlation of the group and the stop tests of Task::alignFrames
// (task.cpp:281-342).
__global__ __launch_bounds__(kSolveWG) void k_corr_finish(Batch B) {
    const int gi = blockIdx.x;
    GroupCtl &ctl = B.ctl[gi];
    GroupRef g = group_of(B, gi);
    // read ahead: thread 0 advances them
    const SS_GLOBAL GroupCtl &was = as_global(B.ctl)[gi];
    const int phase = was.phase, it = was.iteration, filterID = was.filterID, iterImproved = was.iterImproved;
    const double correlation = was.correlation;
    loaded(phase, it, filterID, iterImproved, g.fframeW, g.corrsum, g.colsum, g.N, g.nF, g.nb, g.fcIter, g.maxIter,
           g.allParams, g.p, g.pLast, g.funcTimes, g.iterCorr, g.iterTimes, g.iterErr, correlation, g.cit, g.fct,
           g.halt);
    if (phase != PH_CORR) return;
    double v[CR_N + 1];
#pragma unroll
    for (int i = 0; i <= CR_N; i++) v[i] = 0.0;
    for (int c = threadIdx.x; c < g.fframeW; c += kSolveWG) {
        for (int i = 0; i < CR_N; i++) v[i] += as_global(g.corrsum)[(size_t)c * CR_N + i];
        v[CR_N] += as_global(g.colsum)[(size_t)c * CS_N + CS_SUMI];  // image over all pixels
    }
    __shared__ double tot[CR_N + 1];
    block_sum<CR_N + 1>(v, tot);
    const int P = 2 * g.N;
    if (g.fcIter && it <= g.maxIter)  // flag 'c' (task.cpp:304-306)
        for (int f = threadIdx.x; f < g.nF; f += kSolveWG) {
            double sf[FC_N];
            for (int i = 0; i < FC_N; i++) sf[i] = 0.0;
            for (int bb = 0; bb < g.nb; bb++)
                for (int i = 0; i < FC_N; i++) sf[i] += g.finalsum[(size_t)(f * g.nb + bb) * FS_N + i];
            const double nn = sf[FC_CNT], mA = sf[FC_SA] / nn, mB = sf[FC_SB] / nn;
            const double assq = sf[FC_SAA] - nn * mA * mA;
            const double bssq = sf[FC_SBB] - nn * mB * mB;
            const double q = sf[FC_SAB] - nn * mA * mB;
            g.fcIter[(size_t)(it - 1) * g.nF + f] = q / sqrt(assq * bssq);
        }
    if (g.allParams && it <= g.maxIter)
        for (int i = threadIdx.x; i < P; i += kSolveWG) g.allParams[(size_t)(it - 1) * P + i] = g.p[i];
    __shared__ int s_copy, s_save;
    if (threadIdx.x == 0) {
        const double nm = tot[CR_NMASK];
        const double mA = tot[CR_N] / nm, mB = tot[CR_SUMD] / nm, ns = tot[CR_NS];
        const double assq = tot[CR_SAA] - 2 * mA * tot[CR_SA] + ns * mA * mA;
        const double bssq = tot[CR_SBB] - 2 * mB * tot[CR_SB] + ns * mB * mB;
        const double q = tot[CR_SAB] - mB * tot[CR_SA] - mA * tot[CR_SB] + ns * mA * mB;
        const double corr = q / sqrt(assq * bssq);
        ctl.corr = corr;
        stage_time(g, ctl, FT_CORRELATION);
        if (g.iterCorr && it <= g.maxIter) g.iterCorr[it - 1] = corr;
        if (g.iterTimes) {  // output 9: this iteration's time
            const unsigned long long now = wall_clock64();
            if (it <= g.maxIter) g.iterTimes[it - 1] = (double)(now - ctl.tIter) / g.clockHz;
            ctl.tIter = now;
        }
        int copy = 0, save = 0;
        if (corr - correlation < g.cit) {
            ctl.retv = 0;  // CorrelationIncreaseThreshold
            ctl.phase = PH_FINAL;
        } else if (corr - correlation < g.fct && filterID != 0) {
            ctl.solverFilter = 0;
            ctl.nFilterIterations = 0;
            ctl.filterID = 0;
            if (it >= g.maxIter) {  // never run past max_iterations
                ctl.retv = 3;
                ctl.phase = PH_FINAL;
            } else {
                ctl.iteration = it + 1;
                ctl.improved = 1;
                ctl.shift = 0;
                ctl.phase = PH_ASSEMBLE;
            }
        } else if (!iterImproved) {
            ctl.retv = 2;  // MovementThreshold
            ctl.phase = PH_FINAL;
        } else if (g.maxIter == it) {
            ctl.retv = 3;  // IterationLimit
            ctl.phase = PH_FINAL;
        } else if (correlation >= g.halt) {
            ctl.retv = 1;  // HaltCorrelationReached
            ctl.phase = PH_FINAL;
        } else {
            ctl.correlation = corr;
            copy = 1;
            save = 1;
            ctl.iteration = it + 1;
            ctl.improved = 1;
            ctl.shift = 0;
            ctl.phase = PH_ASSEMBLE;
        }
        if (ctl.phase == PH_FINAL && it == 1) copy = 1;  // task.cpp:381-383
        s_copy = copy;
        s_save = save;
    }
    __syncthreads();
    if (s_copy)
        for (int i = threadIdx.x; i < P; i += kSolveWG) g.pLast[i] = g.p[i];
    if (s_save && g.iterErr)  // flag 'e': an iteration that continues (task.cpp:362-370)
        for (int f = threadIdx.x; f < g.nF; f += kSolveWG) {
            const size_t o = (size_t)f * 2 * g.maxIter + 2 * (size_t)(it - 1);
            g.iterErr[o] = g.errval[f];
            g.iterErr[o + 1] = g.errval[g.nF + f];
        }
}

// ---------------------------------------------------------------------------
// final state: errvals, frame correlations and mask of the last-tried state
// (hd_calculateGroupErrvals(0) + hd_frameCorrelation, task.cpp:389-405)
// ---------------------------------------------------------------------------
template <typename TI, typename R, bool FAST>
__device__ __forceinline__ void final_column_t(GroupRef g, int c) {
    const int f = c / g.nb, b = c % g.nb;
    const ColKnots<R> kn = state_knots<R>(g, c, as_const(g.lsMk)[f]);
    const Template<R, FAST> T(g);
    GeoRun<R, FAST> geo(g, b);
    const int last = g.frameH - 1;
    SS_GLOBAL uint8_t *mo = g.maskOut ? (SS_GLOBAL uint8_t *)g.maskOut + (size_t)c * g.frameH : nullptr;
    double v[FS_N];
#pragma unroll
    for (int i = 0; i < FS_N; i++) v[i] = 0.0;
    constexpr int CH = chunk_rows<R>(1, sizeof(R) == 8 ? kFinalSamplesF64 : kFinalSamplesF32);
    walk_rows<CH, FAST>(
        g, column_ptr<TI>(g, c), [&](int run, int r0) { geo.start(run, r0); },
        [&](int r, int n, const Rows8<TI> &I, int off) {
            R bx[CH], by[CH], f1[CH];
            bool mm[CH];
            Tap<R> tap[CH];
            geo.template rows<CH>(r, last, bx, by, f1, mm);
#pragma unroll
            for (int q = 0; q < CH; q++) {
                const R x = kn.x(bx[q], f1[q]), y = kn.y(by[q], f1[q]);
                mm[q] = (FAST || (q < n && mm[q])) && T.inside(x, y);
                T.fetch(x, y, tap[q]);
            }
            sched_fence();
            if (mo) {
#pragma unroll
                for (int q = 0; q < CH; q++)
                    if (FAST || q < n) mo[r + q] = mm[q] ? 1 : 0;
            }
#pragma unroll
            for (int q = 0; q < CH; q++) {
                double s = (double)bilinear(tap[q]);
                pin(s);
                const double wI = mm[q] ? s : 0.0, Iq = mm[q] ? (double)I.template at<R>(off + q) : 0.0;
                const double d = Iq - wI;
                v[FS_D2] += d * d;
                v[FS_CNT] += mm[q] ? 1.0 : 0.0;
                v[FS_SA] += wI;
                v[FS_SAA] += wI * wI;
                v[FS_SB] += Iq;
                v[FS_SBB] += Iq * Iq;
                v[FS_SAB] += wI * Iq;
            }
        });
    __shared__ double out[FS_N];
    block_sum<FS_N>(v, out);
    if (threadIdx.x < FS_N) g.finalsum[(size_t)c * FS_N + threadIdx.x] = out[threadIdx.x];
}

template <typename TI, typename R>
__device__ __forceinline__ void final_column(GroupRef g, int c) {
    if (g.fast) final_column_t<TI, R, true>(g, c);
    else final_column_t<TI, R, false>(g, c);
}

template <typename TI, typename R>
__global__ __launch_bounds__(kWG) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 8 ? kFinalWavesF64 : kFinalWavesF32))) void k_final(Batch B) {
    for (int item = blockIdx.x; item < B.nItems; item += gridDim.x) {
        const int gi = as_const(B.itemGroup)[item];
        if (as_const(B.ctl)[gi].phase != PH_FINAL) continue;
        GroupRef g = group_of(B, gi);
        if (!runs_here<TI, R>(g)) continue;
        final_column<TI, R>(g, item - g.itemStart);
    }
}

// Residual RMS and frame correlations of the final state, and the end of
// the group.  Called by every thread of a kSolveWG workgroup.
__device__ void final_finish(GroupRef g, GroupCtl &ctl) {
    for (int f = threadIdx.x; f < g.nF; f += kSolveWG) {
        double s[FS_N];
        for (int i = 0; i < FS_N; i++) s[i] = 0.0;
        for (int bb = 0; bb < g.nb; bb++)
            for (int i = 0; i < FS_N; i++) s[i] += g.finalsum[(size_t)(f * g.nb + bb) * FS_N + i];
        const double nn = s[FS_CNT];
        g.resid[f] = sqrt(s[FS_D2] / nn);
        const double mA = s[FS_SA] / nn, mB = s[FS_SB] / nn;
        const double assq = s[FS_SAA] - nn * mA * mA;
        const double bssq = s[FS_SBB] - nn * mB * mB;
        const double q = s[FS_SAB] - nn * mA * mB;
        // flag 'c': the last iteration's correlations stand (task.cpp:392-394)
        g.fcorr[f] = g.fcIter ? g.fcIter[(size_t)(ctl.iteration - 1) * g.nF + f] : q / sqrt(assq * bssq);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        stage_time(g, ctl, FT_CORRELATION);
        ctl.phase = PH_DONE;
    }
}

__global__ __launch_bounds__(kSolveWG) void k_final_finish(Batch B) {
    const int gi = blockIdx.x;
    GroupCtl &ctl = B.ctl[gi];
    if (ctl.phase != PH_FINAL) return;
    final_finish(group_of(B, gi), ctl);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// one launch per (frame type, precision) present in the batch
#define SS_LAUNCH_ONE(kernel, TI, R, grid, L, s)                                                  \
    do {                                                                                          \
        if ((L).hasType[img_type<TI>() + IMG_NTYPES * (sizeof(R) == 8 ? 1 : 0)])                  \
            hipLaunchKernelGGL((kernel<TI, R>), grid, dim3(kWG), 0, s, (L).b);                   \
    } while (0)
// kernels built in kVariants variants: one launch per variant some group of
// the type and precision uses
#define SS_LAUNCH_VAR_ONE(kernel, TK, TI, R, grid, L, s, ...)                                                 \
    do {                                                                                                      \
        const int m_ = (L).hasVar[TK][img_type<TI>() + IMG_NTYPES * (sizeof(R) == 8 ? 1 : 0)];                \
        if (m_ & 1) hipLaunchKernelGGL((kernel<TI, R, 0>), grid, dim3(kWG), 0, s, (L).b, ##__VA_ARGS__);      \
        if (m_ & 2) hipLaunchKernelGGL((kernel<TI, R, 1>), grid, dim3(kWG), 0, s, (L).b, ##__VA_ARGS__);      \
        if (m_ & 4) hipLaunchKernelGGL((kernel<TI, R, 2>), grid, dim3(kWG), 0, s, (L).b, ##__VA_ARGS__);      \
    } while (0)
#define SS_LAUNCH_VAR(kernel, TK, grid, L, s, ...)                                   \
    do {                                                                             \
        SS_LAUNCH_VAR_ONE(kernel, TK, float, float, grid, L, s, ##__VA_ARGS__);      \
        SS_LAUNCH_VAR_ONE(kernel, TK, uint16_t, float, grid, L, s, ##__VA_ARGS__);   \
        SS_LAUNCH_VAR_ONE(kernel, TK, int16_t, float, grid, L, s, ##__VA_ARGS__);    \
        SS_LAUNCH_VAR_ONE(kernel, TK, double, float, grid, L, s, ##__VA_ARGS__);     \
        SS_LAUNCH_VAR_ONE(kernel, TK, float, double, grid, L, s, ##__VA_ARGS__);     \
        SS_LAUNCH_VAR_ONE(kernel, TK, uint16_t, double, grid, L, s, ##__VA_ARGS__);  \
        SS_LAUNCH_VAR_ONE(kernel, TK, int16_t, double, grid, L, s, ##__VA_ARGS__);   \
        SS_LAUNCH_VAR_ONE(kernel, TK, double, double, grid, L, s, ##__VA_ARGS__);    \
    } while (0)
#define SS_LAUNCH_TYPED(kernel, grid, L, s)                  \
    do {                                                     \
        SS_LAUNCH_ONE(kernel, float, float, grid, L, s);     \
        SS_LAUNCH_ONE(kernel, uint16_t, float, grid, L, s);  \
        SS_LAUNCH_ONE(kernel, int16_t, float, grid, L, s);   \
        SS_LAUNCH_ONE(kernel, double, float, grid, L, s);    \
        SS_LAUNCH_ONE(kernel, float, double, grid, L, s);    \
        SS_LAUNCH_ONE(kernel, uint16_t, double, grid, L, s); \
        SS_LAUNCH_ONE(kernel, int16_t, double, grid, L, s);  \
        SS_LAUNCH_ONE(kernel, double, double, grid, L, s);   \
    } while (0)

hipError_t launch_stage(const LaunchBatch &L, int entry, hipStream_t s) {
    const dim3 items(L.itemGrid), groups(L.b.nGroups);
    const int slot = entry_slot(entry);
    switch (entry_stage(entry)) {
    case ST_ASSEMBLE: SS_LAUNCH_VAR(k_assemble, TK_ASSEMBLE, items, L, s); break;
    case ST_SOLVE: hipLaunchKernelGGL(k_solve, groups, dim3(kSolveWG), 0, s, L.b); break;
    case ST_LS:
        if (slot == 0) SS_LAUNCH_VAR(k_ls_round, TK_LS, items, L, s, slot, 1);
        else SS_LAUNCH_VAR(k_ls_round, TK_LS, dim3(L.lsSplitGrid), L, s, slot, L.lsSplit);
        break;
    case ST_LS_DECIDE:
        hipLaunchKernelGGL(k_ls_decide, dim3(L.frameGrid), dim3(64), 0, s, L.b, slot);
        if (slot == kLsSlots - 1) hipLaunchKernelGGL(k_ls_finish, groups, dim3(64), 0, s, L.b);
        break;
    case ST_CORR:
        SS_LAUNCH_VAR(k_corr, TK_CORR, items, L, s);
        if (L.hasFrameCorr) SS_LAUNCH_TYPED(k_corr_frames, items, L, s);
        break;
    case ST_CORR_FINISH: hipLaunchKernelGGL(k_corr_finish, groups, dim3(kSolveWG), 0, s, L.b); break;
    case ST_FINAL: SS_LAUNCH_TYPED(k_final, items, L, s); break;
    case ST_FINAL_FINISH: hipLaunchKernelGGL(k_final_finish, groups, dim3(kSolveWG), 0, s, L.b); break;
    }
    return hipGetLastError();
}

size_t solve_workspace_bytes(int n) {
    // Eq0 + InteriorRow + solution + the refinement's saved solution per knot
    // and, the last partition's unused rows, per thread
    return ((size_t)n + kSolveWG) * (sizeof(Eq0) + sizeof(InteriorRow) + 2 * sizeof(double2)) + 256;
}

}  // namespace ss
