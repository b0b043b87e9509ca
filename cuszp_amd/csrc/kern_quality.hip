// Reconstruction quality of a decompressed array against its original, on the
// device: the figures of the reference's computePSNR (src/cuSZp_utility.cu:891-950)
// plus the two maxima it tracks, and its windowed SSIM (:761-889), for the
// batched and serving reports.
//
// Per element the arithmetic is the reference's: for f32 data the error
// |dec - ori|, its square, dec * dec and the pointwise relative error are
// float operations, everything is accumulated in double; f64 data is handled
// in double throughout. One launch per report: the workgroups' partial results
// meet in the last workgroup (grid_words.hpp), which writes the sums to pinned
// host memory.
#include <hip/hip_runtime.h>

#include <cmath>
#include <map>
#include <memory>
#include <mutex>

#include "../../include/cuSZp.h"
#include "grid_words.hpp"

namespace cuszp_quality {

constexpr int kThreads = 256;
constexpr unsigned kMaxBlocks = 1024;    // error figures: four workgroups per CU
constexpr unsigned kMaxSsimBlocks = 2048;

// the reference's per-element operations for T = float (float results), and
// their double counterparts for T = double
template <class T>
__device__ __forceinline__ T abs_err(T d, T o) { return d > o ? d - o : o - d; }
__device__ __forceinline__ float max_of(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double max_of(double a, double b) { return fmax(a, b); }

// Count, means and centred sums of pairs (o, d) seen so far.
struct Moments {
    double n, mo, md, oo, dd, od;
};
// Two disjoint sets' moments as one (Chan, Golub and LeVeque's update): the
// centred sums are corrected by the distance of the means, so no large sums
// cancel and one read of the arrays does.
__device__ __forceinline__ Moments merge(const Moments& a, const Moments& b) {
    Moments r;
    r.n = a.n + b.n;
    const double f = r.n > 0 ? b.n / r.n : 0.0;
    const double eo = b.mo - a.mo, ed = b.md - a.md, w = a.n * f;
    r.mo = a.mo + eo * f;
    r.md = a.md + ed * f;
    // w first: it is 0 where either set is empty, and a distance (then a mean) may square to infinity
    r.oo = a.oo + b.oo + eo * w * eo;
    r.dd = a.dd + b.dd + ed * w * ed;
    r.od = a.od + b.od + eo * w * ed;
    return r;
}

// A share's sums (dec^2, err^2), maxima (ori, -ori, err, rel err) and moments.
constexpr int kFigures = 12;
struct Figures {
    double s[2], m[4];
    Moments c;
    __device__ __forceinline__ void init() {
        for (int k = 0; k < 2; ++k) s[k] = 0;
        for (int k = 0; k < 4; ++k) m[k] = k < 2 ? -INFINITY : 0.0;
        c = Moments{0, 0, 0, 0, 0, 0};
    }
    __device__ __forceinline__ void add(const Figures& b) {
        for (int k = 0; k < 2; ++k) s[k] += b.s[k];
        for (int k = 0; k < 4; ++k) m[k] = fmax(m[k], b.m[k]);
        c = merge(c, b.c);
    }
    template <class F>
    __device__ __forceinline__ void each(F&& f) {
        for (int k = 0; k < 2; ++k) f(k, s[k]);
        for (int k = 0; k < 4; ++k) f(2 + k, m[k]);
        f(6, c.n);
        f(7, c.mo);
        f(8, c.md);
        f(9, c.oo);
        f(10, c.dd);
        f(11, c.od);
    }
};

// The workgroup's figures, in thread 0 (sm: kFigures doubles per wave).
__device__ __forceinline__ void block_figures(Figures& f, double* sm) {
    for (int o = 32; o > 0; o >>= 1) {
        Figures g = f;
        g.each([&](int, double& v) { v = __shfl_down(v, o, 64); });
        f.add(g);   // lanes past 64 - o add what is not used
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) f.each([&](int k, double& v) { sm[w * kFigures + k] = v; });
    __syncthreads();
    if (threadIdx.x == 0)
        for (int j = 1; j < kThreads / 64; ++j) {
            Figures g;
            g.each([&](int k, double& v) { v = sm[j * kFigures + k]; });
            f.add(g);
        }
    __syncthreads();
}

// Error figures in one read of both arrays. A thread takes U 16-byte vectors of
// each array at a time (their loads in flight together), centres them on their
// own means and merges the result into its moments. Bound by the read: 21.8 M
// pairs of f32 (175 MB) took 124 us as two passes (means first, then centred
// sums) and 48 us this way, about 10 of them the reductions at the end.
// gw: kFigures values of two words per workgroup; res: the figures.
template <class T>
__global__ void __launch_bounds__(kThreads) figures_kernel(const T* __restrict__ ori, const T* __restrict__ dec,
                                                           uint64_t n, uint64_t steps, const cuszp::GridWords gw,
                                                           double* res) {
    constexpr int V = 16 / (int)sizeof(T), U = 4, E = U * V;
    typedef T VT __attribute__((ext_vector_type(V), aligned(sizeof(T))));   // arrays start at any element
    __shared__ double sm[(kThreads / 64) * kFigures];
    __shared__ bool lost;
    if (threadIdx.x == 0) lost = false;
    Figures f;
    f.init();
    T m[4] = {-INFINITY, -INFINITY, T(0), T(0)};
    auto take = [&](T o, T d) {
        const T err = abs_err(d, o);
        f.s[0] += (double)(T)(d * d);
        f.s[1] += (double)(T)(err * err);
        m[0] = max_of(m[0], o);
        m[1] = max_of(m[1], -o);
        m[2] = max_of(m[2], err);
        if (o != T(0)) m[3] = max_of(m[3], (T)(err / (o < T(0) ? -o : o)));
    };
    for (uint64_t i = blockIdx.x; i < steps; i += gridDim.x) {
        const uint64_t at = (i * U * kThreads + threadIdx.x) * V;
        VT vo[U], vd[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            vo[u] = *(const VT*)(ori + at + (uint64_t)u * kThreads * V);
            vd[u] = *(const VT*)(dec + at + (uint64_t)u * kThreads * V);
        }
        double so = 0, sd = 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                take(vo[u][j], vd[u][j]);
                so += (double)vo[u][j];
                sd += (double)vd[u][j];
            }
        Moments c = {(double)E, so * (1.0 / E), sd * (1.0 / E), 0, 0, 0};
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const double a = (double)vo[u][j] - c.mo, b = (double)vd[u][j] - c.md;
                c.oo += a * a;
                c.dd += b * b;
                c.od += a * b;
            }
        f.c = merge(f.c, c);
    }
    if (blockIdx.x == gridDim.x - 1)   // fewer than one step's elements are left
        for (uint64_t i = steps * kThreads * E + threadIdx.x; i < n; i += kThreads) {
            take(ori[i], dec[i]);
            f.c = merge(f.c, Moments{1, (double)ori[i], (double)dec[i], 0, 0, 0});
        }
    for (int k = 0; k < 4; ++k) f.m[k] = (double)m[k];
    block_figures(f, sm);
    typedef cuszp::Words<double> W;
    if (blockIdx.x != gridDim.x - 1) {
        // word k of every workgroup in a row: the last workgroup's lanes read
        // neighbours (each workgroup's words in a row, 57,000 lines read one by one,
        // cost 12 us of the 60)
        if (threadIdx.x == 0)
            f.each([&](int k, double& v) {
                const W w = W::of(v);
                gw.put((uint64_t)(2 * k) * gridDim.x + blockIdx.x, w.u[0]);
                gw.put((uint64_t)(2 * k + 1) * gridDim.x + blockIdx.x, w.u[1]);
            });
        return;
    }
    if (threadIdx.x != 0) f.init();
    bool ok = true;
    for (unsigned b = threadIdx.x; b + 1 < gridDim.x; b += kThreads) {
        uint32_t u[2 * kFigures];
        ok &= gw.get_n((uint64_t)b, u, gridDim.x);
        Figures g;
        g.each([&](int k, double& v) {
            W w;
            w.u[0] = u[2 * k];
            w.u[1] = u[2 * k + 1];
            v = w.value();
        });
        f.add(g);
    }
    if (!ok) lost = true;
    block_figures(f, sm);
    if (threadIdx.x == 0) {
        f.each([&](int k, double& v) { cuszp::host_store(res + k, v); });
        cuszp::host_store(res + cuszp::kGridResults - 1, lost ? 1.0 : 0.0);
    }
}
static_assert(kFigures < cuszp::kGridResults, "the figures and the flag");

// SSIM over 7x7x7 windows moved by 2 along each axis (src/cuSZp_utility.cu:761-889):
// per window, the original's min and max, both means, both variances and the
// covariance (double sums of the values), then luminance * contrast * structure
// with c1 = (0.01 R)^2, c2 = (0.03 R)^2, c3 = c2 / 2, R the window's original
// range (1 when the range is 0).
constexpr int kWin = 7, kWinStep = 2;

// Smaller and larger of two or three values, one instruction each (fmin would
// quieten its operands first; a window with a NaN has no SSIM whatever its range).
__device__ __forceinline__ float min_of(float a, float b) { asm("v_min_f32 %0, %1, %2" : "=v"(a) : "v"(a), "v"(b)); return a; }
__device__ __forceinline__ double min_of(double a, double b) { asm("v_min_f64 %0, %1, %2" : "=v"(a) : "v"(a), "v"(b)); return a; }
__device__ __forceinline__ float most_of(float a, float b) { asm("v_max_f32 %0, %1, %2" : "=v"(a) : "v"(a), "v"(b)); return a; }
__device__ __forceinline__ double most_of(double a, double b) { asm("v_max_f64 %0, %1, %2" : "=v"(a) : "v"(a), "v"(b)); return a; }
__device__ __forceinline__ float min_of(float a, float b, float c) { asm("v_min3_f32 %0, %1, %2, %3" : "=v"(a) : "v"(a), "v"(b), "v"(c)); return a; }
__device__ __forceinline__ float most_of(float a, float b, float c) { asm("v_max3_f32 %0, %1, %2, %3" : "=v"(a) : "v"(a), "v"(b), "v"(c)); return a; }
__device__ __forceinline__ double min_of(double a, double b, double c) { return min_of(min_of(a, b), c); }
__device__ __forceinline__ double most_of(double a, double b, double c) { return most_of(most_of(a, b), c); }

// Sums, centred sums and range of a set of pairs: a row of a window, a slice, or all of it.
template <class T>
struct WinStats {
    double x, y, xx, yy, xy;
    T lo, hi;
};
// Equal-sized sets (n pairs each) joined one by one. The distances of their
// sums are taken from the first set's, which is one of them: the correction of
// the squares to the joint mean then cancels at most the number of sets, whatever
// the values' offset.
template <class T>
struct Join {
    WinStats<T> s;                   // s.x, s.y: the first set's sums
    double dx, dy, qxx, qyy, qxy;    // sums and squares of the distances
    __device__ __forceinline__ void first(const WinStats<T>& a) {
        s = a;
        dx = dy = qxx = qyy = qxy = 0;
    }
    __device__ __forceinline__ void next(const WinStats<T>& a) {
        const double u = a.x - s.x, v = a.y - s.y;
        dx += u;
        dy += v;
        qxx = fma(u, u, qxx);
        qyy = fma(v, v, qyy);
        qxy = fma(u, v, qxy);
        s.xx += a.xx;
        s.yy += a.yy;
        s.xy += a.xy;
        s.lo = min_of(s.lo, a.lo);
        s.hi = most_of(s.hi, a.hi);
    }
    __device__ __forceinline__ WinStats<T> done(double n) const {
        WinStats<T> r = s;
        const double f = 1.0 / n, ex = dx * (1.0 / kWin), ey = dy * (1.0 / kWin);
        r.x = fma(s.x, (double)kWin, dx);
        r.y = fma(s.y, (double)kWin, dy);
        r.xx = fma(fma(-ex, dx, qxx), f, s.xx);
        r.yy = fma(fma(-ey, dy, qyy), f, s.yy);
        r.xy = fma(fma(-ex, dy, qxy), f, s.xy);
        return r;
    }
};

// Two slices as one set.
constexpr double kSlice = kWin * kWin;   // values of a window's slice
template <class T>
__device__ __forceinline__ WinStats<T> pair_of(const WinStats<T>& a, const WinStats<T>& b) {
    const double u = b.x - a.x, v = b.y - a.y, fu = u * (1 / (2 * kSlice)), fv = v * (1 / (2 * kSlice));
    return {a.x + b.x, a.y + b.y, fma(fu, u, a.xx + b.xx), fma(fv, v, a.yy + b.yy), fma(fu, v, a.xy + b.xy),
            min_of(a.lo, b.lo), most_of(a.hi, b.hi)};
}
// A window's seven slices: three pairs and one more. Distances of sums are
// taken from the first pair's, as in Join.
template <class T>
__device__ __forceinline__ WinStats<T> window_of(const WinStats<T> (&p)[3], const WinStats<T>& d) {
    static_assert(kWin == 7, "three pairs and a slice");
    const double u1 = p[1].x - p[0].x, v1 = p[1].y - p[0].y, u2 = p[2].x - p[0].x, v2 = p[2].y - p[0].y;
    const double du = u1 + u2, dv = v1 + v2, eu = du * (1.0 / 3), ev = dv * (1.0 / 3);
    // the last slice's distance from the pairs' mean, times 6 slices
    const double wu = fma(6.0, fma(-0.5, p[0].x, d.x), -du), wv = fma(6.0, fma(-0.5, p[0].y, d.y), -dv);
    constexpr double f = 1 / (2 * kSlice), g = 1 / (42 * kSlice);
    WinStats<T> r;
    r.x = fma(3.0, p[0].x, du) + d.x;
    r.y = fma(3.0, p[0].y, dv) + d.y;
    r.xx = fma(wu * g, wu, fma(fma(-eu, du, fma(u1, u1, u2 * u2)), f, p[0].xx + p[1].xx + p[2].xx + d.xx));
    r.yy = fma(wv * g, wv, fma(fma(-ev, dv, fma(v1, v1, v2 * v2)), f, p[0].yy + p[1].yy + p[2].yy + d.yy));
    r.xy = fma(wu * g, wv, fma(fma(-eu, dv, fma(u1, v1, u2 * v2)), f, p[0].xy + p[1].xy + p[2].xy + d.xy));
    r.lo = min_of(min_of(p[0].lo, p[1].lo, p[2].lo), d.lo);
    r.hi = most_of(most_of(p[0].hi, p[1].hi, p[2].hi), d.hi);
    return r;
}

// Whether a window's values are finite but its centred sums are not: the squares of
// distances between sums of up to 98 values leave double's range before
// those of the values do (f64 deviations of 1e152 and more).
template <class T>
__device__ __forceinline__ bool overflown(const WinStats<T>& s) {
    return sizeof(T) == 8 && !(s.xx + s.yy + fabs(s.xy) < INFINITY) && fabs(s.x) < INFINITY && fabs(s.y) < INFINITY;
}

template <class T>
__device__ __forceinline__ double ssim_of(const WinStats<T>& s) {
    constexpr double np = kWin * kWin * kWin;
    if constexpr (sizeof(T) == 4) {
        // sums of floats are far from the limits of double: numerators and
        // denominators scaled by the count instead of divided by it, one division
        const double rr = (double)(T)(s.hi - s.lo), q = rr == 0 ? 1.0 : rr * rr;
        const double c1 = (0.01 * 0.01) * (np * np) * q, c2 = (0.03 * 0.03) * np * q, d = s.xx + s.yy + c2;
        if (c2 > 0 && d < INFINITY)
            return fma(2 * s.x, s.y, c1) * fma(2.0, s.xy, c2) / (fma(s.x, s.x, fma(s.y, s.y, c1)) * d);
    }
    const double mx = s.x / np, my = s.y / np, vx = s.xx / np, vy = s.yy / np, vxy = s.xy / np;
    const double rr = (double)(T)(s.hi - s.lo);   // the range in the values' type
    const double c1 = rr == 0 ? 0.01 * 0.01 : 0.01 * 0.01 * rr * rr;
    const double c2 = rr == 0 ? 0.03 * 0.03 : 0.03 * 0.03 * rr * rr;
    const double c3 = c2 / 2;
    const double lum = (2 * mx * my + c1) / (mx * mx + my * my + c1);
    // (2 sx sy + c2) / (vx + vy + c2) * (vxy + c3) / (sx sy + c3), in which 2 sx sy + c2 = 2 (sx sy + c3)
    // cancels unless it is 0 or the variances are not finite
    if (c2 > 0 && vx + vy + c2 < INFINITY) return lum * ((2 * vxy + c2) / (vx + vy + c2));
    const double sx = sqrt(vx), sy = sqrt(vy);
    return lum * ((2 * sx * sy + c2) / (sx * sx + sy * sy + c2)) * ((vxy + c3) / (sx * sy + c3));
}

// The SSIM of the window at (o0, o1, o2) by itself, from its 343 pairs: the means, then centred sums.
template <class T>
__device__ double window_ssim(const T* __restrict__ x, const T* __restrict__ y, uint64_t s1, uint64_t s0,
                              uint64_t o0, uint64_t o1, uint64_t o2) {
    const uint64_t b = o0 + s0 * (o1 + s1 * o2);
    T xmin = x[b], xmax = x[b];
    double xs = 0, ys = 0;
    // Rows one by one, a whole row of x before that of y: lanes' rows lie far apart in the volumes
    // that come here, and what one row's loads bring to the L1 is used before the next one's
    // (f64 7 x 9 x 60005 117 us with the two rows' loads mixed, 97 this way).
    auto rows = [&](auto&& take) {
#pragma unroll 1
        for (int k = 0; k < kWin; ++k)
#pragma unroll 1
            for (int j = 0; j < kWin; ++j) {
                const uint64_t r = b + s0 * ((uint64_t)j + s1 * (uint64_t)k);
                T a[kWin], c[kWin];
#pragma unroll
                for (int i = 0; i < kWin; ++i) a[i] = x[r + i];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < kWin; ++i) c[i] = y[r + i];
#pragma unroll
                for (int i = 0; i < kWin; ++i) take(a[i], c[i]);
            }
    };
    rows([&](T a, T c) {
        xmin = a < xmin ? a : xmin;
        xmax = a > xmax ? a : xmax;
        xs += (double)a;
        ys += (double)c;
    });
    constexpr double np = kWin * kWin * kWin;
    const double mx = xs / np, my = ys / np;
    double vx = 0, vy = 0, vxy = 0;
    rows([&](T o, T d) {
        const double a = (double)o - mx, c = (double)d - my;
        vx += a * a;
        vy += c * c;
        vxy += a * c;
    });
    return ssim_of(WinStats<T>{xs, ys, vx, vy, vxy, xmin, xmax});
}

// Windows of a volume, tiled: TX x TY windows of a tile along x and y, `depth`
// layers of windows along z.
struct SsimPlan {
    uint64_t s0, s1;             // extents along x and y
    uint64_t nw0, nw1, nw2;      // windows along x, y, z
    uint64_t t0, t1, tiles;      // tiles along x and y, and in all
    uint64_t depth;              // layers of windows per tile
};

// Barrier that orders LDS accesses only: loads from global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The mean of all threads' totals over n, to res (sm: a double per wave; lost: set to false before).
__device__ __forceinline__ void grid_mean(double total, double n, double* sm, bool& lost, const cuszp::GridWords& gw, double* res) {
    const int tid = (int)threadIdx.x;
    auto block_sum = [&](double v) -> double {   // in thread 0
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        __syncthreads();
        if ((tid & 63) == 0) sm[tid >> 6] = v;
        __syncthreads();
        double t = 0;
        for (int j = 0; j < kThreads / 64; ++j) t += sm[j];
        return t;
    };
    typedef cuszp::Words<double> W;
    total = block_sum(total);
    if (blockIdx.x != gridDim.x - 1) {
        if (tid == 0) {
            const W w = W::of(total);
            gw.put((uint64_t)blockIdx.x * 2, w.u[0]);
            gw.put((uint64_t)blockIdx.x * 2 + 1, w.u[1]);
        }
        return;
    }
    if (tid != 0) total = 0;
    bool ok = true;
    for (unsigned b = threadIdx.x; b + 1 < gridDim.x; b += kThreads) {
        W w;
        ok &= gw.get_n((uint64_t)b * 2, w.u);
        total += w.value();
    }
    if (!ok) lost = true;
    total = block_sum(total);
    if (tid == 0) {
        cuszp::host_store(res, total / n);
        cuszp::host_store(res + cuszp::kGridResults - 1, lost ? 1.0 : 0.0);
    }
}

// Workgroups per CU that the kernel is built for (registers, and LDS of 44 or 61 KB).
template <class T> constexpr int kSsimPerCu = sizeof(T) == 4 ? 3 : 2;

// One workgroup per tile (then the tile gridDim.x further on). It walks down
// the tile's slices. The values of a slice come to LDS by way of registers, read
// while the slice before is worked on; from there threads first make the
// statistics of the rows of seven values that windows start with (2 TY + 5 rows,
// TX per row), then each thread, one window column, joins seven of them to its
// slice of 7 x 7 and those to pairs; three pairs and a slice are a window.
// A value is read once and takes part in 3.5 rows, 3.5 x 3.5 slices... through
// these sums, where a window by itself reads 343 pairs twice. Bound by the f64
// arithmetic, about 80 operations per value, and the waits between its steps.
// 2.5 M windows of f32: 784 us as one thread per window, 190 us with rows read
// from memory as they are needed and 6 layers per tile, 156 us with LDS and deep
// tiles, 131 us with the rows of two windows made together.
template <class T, int TX>
__global__ void __launch_bounds__(kThreads, kSsimPerCu<T>) ssim_kernel(const T* __restrict__ x, const T* __restrict__ y,
                                                        const SsimPlan p, const cuszp::GridWords gw, double* res) {
    constexpr int TY = kThreads / TX, ROWS = kWinStep * TY + kWin - kWinStep, COLS = kWinStep * TX + kWin - kWinStep;
    constexpr int STRIDE = (COLS + 1) / 2 * 2, NV = (ROWS * COLS + kThreads - 1) / kThreads;   // values per thread
    typedef T V2 __attribute__((ext_vector_type(2)));
    __shared__ __align__(16) double rs[5][ROWS][TX];
    __shared__ __align__(16) T rlo[ROWS][TX], rhi[ROWS][TX];
    __shared__ V2 raw[2][ROWS][STRIDE / 2];
    __shared__ double sm[kThreads / 64];
    __shared__ bool lost;
    const int tid = (int)threadIdx.x, tx = tid % TX, ty = tid / TX;
    if (tid == 0) lost = false;
    double total = 0;
    for (uint64_t tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
        const uint64_t wx0 = tile % p.t0 * TX, r = tile / p.t0;
        const uint64_t wy0 = r % p.t1 * TY, wz0 = r / p.t1 * p.depth;
        const uint64_t layers = p.nw2 - wz0 < p.depth ? p.nw2 - wz0 : p.depth;
        const bool mine = wx0 + tx < p.nw0 && wy0 + ty < p.nw1;
        // this thread's values of a slice; past the extents the last ones again (in windows that count nothing)
        uint64_t at[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int i = tid + k * kThreads < ROWS * COLS ? tid + k * kThreads : ROWS * COLS - 1;
            uint64_t yy = kWinStep * wy0 + i / COLS, xx = kWinStep * wx0 + i % COLS;
            yy = yy < p.s1 ? yy : p.s1 - 1;
            xx = xx < p.s0 ? xx : p.s0 - 1;
            at[k] = (kWinStep * wz0 * p.s1 + yy) * p.s0 + xx;
        }
        T vx[NV], vy[NV];
        auto load = [&]() {   // and on to the next slice
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                vx[k] = x[at[k]];
                vy[k] = y[at[k]];
                at[k] += p.s0 * p.s1;
            }
        };
        auto slice = [&](bool more) -> WinStats<T> {   // this thread's 7 x 7 of the slice in vx, vy; loads the next
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int i = tid + k * kThreads;
                if (i < ROWS * COLS) {
                    ((T*)raw[0][i / COLS])[i % COLS] = vx[k];
                    ((T*)raw[1][i / COLS])[i % COLS] = vy[k];
                }
            }
            if (more) load();
            lds_barrier();   // also: the rows of the slice before have been read
#pragma unroll 1
            for (int i = tid; i < ROWS * TX / 2; i += kThreads) {   // the rows of two windows, values 0-6 and 2-8
                const int row = i / (TX / 2), wx = i % (TX / 2) * 2;
                T a[kWin + 2], c[kWin + 2];
#pragma unroll
                for (int j = 0; j < (kWin + 2) / 2; ++j) {
                    const V2 va = raw[0][row][wx + j], vc = raw[1][row][wx + j];
                    a[2 * j] = va[0];
                    a[2 * j + 1] = va[1];
                    c[2 * j] = vc[0];
                    c[2 * j + 1] = vc[1];
                }
                a[kWin + 1] = raw[0][row][wx + (kWin + 1) / 2][0];
                c[kWin + 1] = raw[1][row][wx + (kWin + 1) / 2][0];
                // distances from value 4, a member of both rows: the correction to
                // their own mean cancels at most the number of values
                const double ra = (double)a[4], rc = (double)c[4];
                double u[kWin + 2], v[kWin + 2], su = 0, sv = 0, uu = 0, vv = 0, uv = 0;
#pragma unroll
                for (int j = 0; j < kWin + 2; ++j) {
                    u[j] = (double)a[j] - ra;
                    v[j] = (double)c[j] - rc;
                }
                auto add = [&](int j, double& su, double& sv, double& uu, double& vv, double& uv) {
                    su += u[j];
                    sv += v[j];
                    uu = fma(u[j], u[j], uu);
                    vv = fma(v[j], v[j], vv);
                    uv = fma(u[j], v[j], uv);
                };
                for (int j : {2, 3, 5, 6}) add(j, su, sv, uu, vv, uv);
                const T lo = min_of(min_of(a[2], a[3], a[4]), a[5], a[6]), hi = most_of(most_of(a[2], a[3], a[4]), a[5], a[6]);
                typedef double D2 __attribute__((ext_vector_type(2)));
                D2 o[5];
                V2 ol, oh;
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    double s1 = su, s2 = sv, q1 = uu, q2 = vv, q3 = uv;
                    const int e = w ? kWin : 0;   // the two values that are this row's alone
                    add(e, s1, s2, q1, q2, q3);
                    add(e + 1, s1, s2, q1, q2, q3);
                    const double e1 = s1 * (1.0 / kWin), e2 = s2 * (1.0 / kWin);
                    o[0][w] = fma((double)kWin, ra, s1);
                    o[1][w] = fma((double)kWin, rc, s2);
                    o[2][w] = fma(-e1, s1, q1);
                    o[3][w] = fma(-e2, s2, q2);
                    o[4][w] = fma(-e1, s2, q3);
                    ol[w] = min_of(lo, a[e], a[e + 1]);
                    oh[w] = most_of(hi, a[e], a[e + 1]);
                }
#pragma unroll
                for (int k = 0; k < 5; ++k) *(D2*)&rs[k][row][wx] = o[k];
                *(V2*)&rlo[row][wx] = ol;
                *(V2*)&rhi[row][wx] = oh;
            }
            lds_barrier();
            auto at_row = [&](int row) -> WinStats<T> {
                return WinStats<T>{rs[0][row][tx], rs[1][row][tx], rs[2][row][tx], rs[3][row][tx], rs[4][row][tx],
                                   rlo[row][tx], rhi[row][tx]};
            };
            Join<T> q;
            q.first(at_row(kWinStep * ty));
#pragma unroll
            for (int j = 1; j < kWin; ++j) q.next(at_row(kWinStep * ty + j));
            return q.done((double)kWin);
        };
        // 2 * layers + 5 slices in pairs; from the fourth pair on the first slice of each completes a layer
        load();
        WinStats<T> ring[3];
        for (int k = 0; k < 3; ++k) ring[k] = WinStats<T>{0, 0, 0, 0, 0, T(0), T(0)};
#pragma unroll 1
        for (uint64_t l = 0; l < layers + 3; ++l) {
            const bool last = l == layers + 2;
            const WinStats<T> d = slice(!last);
            if (l >= 3 && mine) {
                const WinStats<T> w = window_of(ring, d);
                if (overflown(w))
                    total += window_ssim(x, y, p.s1, p.s0, kWinStep * (wx0 + tx), kWinStep * (wy0 + ty), kWinStep * (wz0 + l - 3));
                else
                    total += ssim_of(w);
            }
            if (last) break;
            ring[0] = ring[1];
            ring[1] = ring[2];
            ring[2] = pair_of(d, slice(true));
        }
    }
    grid_mean(total, (double)(p.nw0 * p.nw1 * p.nw2), sm, lost, gw, res);
}

// One thread per window: every window reads its own pairs, twice. For volumes
// of few windows along two axes, most of whose tiles' lanes would have no window
// (window_by_window).
template <class T>
__global__ void __launch_bounds__(kThreads) windows_kernel(const T* __restrict__ x, const T* __restrict__ y, const SsimPlan p,
                                                           const cuszp::GridWords gw, double* res) {
    __shared__ double sm[kThreads / 64];
    __shared__ bool lost;
    if (threadIdx.x == 0) lost = false;
    const uint64_t n = p.nw0 * p.nw1 * p.nw2;
    double total = 0;
    for (uint64_t w = (uint64_t)blockIdx.x * kThreads + threadIdx.x; w < n; w += (uint64_t)gridDim.x * kThreads) {
        const uint64_t w0 = w % p.nw0, w1 = (w / p.nw0) % p.nw1, w2 = w / (p.nw0 * p.nw1);
        total += window_ssim(x, y, p.s1, p.s0, w0 * kWinStep, w1 * kWinStep, w2 * kWinStep);
    }
    grid_mean(total, (double)n, sm, lost, gw, res);
}

struct State {
    cuszp::GridState g;
    std::mutex mu;
};
constexpr uint64_t kWords = (uint64_t)kMaxBlocks * kFigures * 2;
static_assert(kWords >= (uint64_t)kMaxSsimBlocks * 2, "words of either kernel");
std::mutex g_mu;
std::map<std::pair<int, hipStream_t>, std::unique_ptr<State>> g_state;

#define Q_HIP(call)                                    \
    do {                                               \
        hipError_t e_ = (call);                        \
        if (e_ != hipSuccess) return CUSZP_ERROR_HIP;  \
    } while (0)

State& state_for(int dev, hipStream_t st) {
    std::lock_guard<std::mutex> lk(g_mu);
    auto& s = g_state[{dev, st}];
    if (!s) s.reset(new State());
    return *s;
}

template <class T>
int run(const T* ori, const T* dec, size_t n, double* out, hipStream_t st) {
    int dev = 0;
    Q_HIP(hipGetDevice(&dev));
    State& s = state_for(dev, st);
    std::lock_guard<std::mutex> lk(s.mu);
    Q_HIP(cuszp::grid_state_init(s.g, kWords, st));
    cuszp::GridWords gw;
    Q_HIP(cuszp::grid_next_tag(s.g, kWords, st, gw));
    const uint64_t steps = n / (64 / sizeof(T) * kThreads);   // 64 bytes of each array per thread and step
    const unsigned blocks = steps < 1 ? 1 : (steps < kMaxBlocks ? (unsigned)steps : kMaxBlocks);
    hipLaunchKernelGGL(figures_kernel<T>, dim3(blocks), dim3(kThreads), 0, st, ori, dec, (uint64_t)n, steps, gw,
                       s.g.h_res);
    Q_HIP(hipGetLastError());
    Q_HIP(hipStreamSynchronize(st));
    const double* r = s.g.h_res;
    if (r[cuszp::kGridResults - 1] != 0.0) return CUSZP_ERROR_INTERNAL;
    const double N = (double)n;
    const double mse = r[1] / N, range = r[2] + r[3];            // r[3]: max of -ori
    out[0] = mse;                                                // src/cuSZp_utility.cu:937-946
    out[1] = range;
    out[2] = 20 * log10(range) - 10 * log10(mse);
    out[3] = sqrt(r[1]);
    out[4] = sqrt(r[1]) / sqrt(r[0]);
    out[5] = sqrt(mse) / range;
    out[6] = r[4];                                               // max |dec - ori|
    out[7] = r[5];                                               // max |dec - ori| / |ori| over ori != 0
    out[8] = (r[11] / N) / sqrt(r[9] / N) / sqrt(r[10] / N);     // correlation (acEff)
    return CUSZP_SUCCESS;
}

// Whether a volume of n windows, nw0 along x, is faster with a thread per window than with
// tiles, whose workgroups go through `slices` slices in a row. A slice takes about 3 us once
// every CU has its workgroups, whatever share of their lanes has windows; a thread per window
// 30-50 us in all while the chip is not full, then 0.3 ns a window (f64 0.6), and more where
// there is one window along x and lanes read rows far apart. us a call, tiles and thread per
// window: f32 7 x 7 x 60005 298 and 62, 13 x 13 x 8755 78 and 50, 13 x 13 x 37505 190 and 111,
// 600005 x 7 x 7 272 and 116; f64 13 x 13 x 37505 224 and 222, 7 x 21 x 75005 444 and 577.
template <class T>
bool window_by_window(uint64_t slices, uint64_t n, uint64_t nw0) {
    constexpr uint64_t kPerSlice = sizeof(T) == 4 ? 9000 : 3900, kPerSliceFar = sizeof(T) == 4 ? 6000 : 1560;
    return slices > 9 + (n <= 65536 ? 0 : n / (nw0 > 1 ? kPerSlice : kPerSliceFar));
}

template <class T>
int run_ssim(const T* x, const T* y, cuszp_dims_t d, double* out, hipStream_t st) {
    if (d.x < (unsigned)kWin || d.y < (unsigned)kWin || d.z < (unsigned)kWin) return CUSZP_ERROR_INVALID_DIMS;
    int dev = 0;
    Q_HIP(hipGetDevice(&dev));
    State& s = state_for(dev, st);
    std::lock_guard<std::mutex> lk(s.mu);
    Q_HIP(cuszp::grid_state_init(s.g, kWords, st));
    cuszp::GridWords gw;
    Q_HIP(cuszp::grid_next_tag(s.g, kWords, st, gw));
    SsimPlan p;
    p.s0 = d.x;
    p.s1 = d.y;
    p.nw0 = (d.x - kWin) / kWinStep + 1;
    p.nw1 = (d.y - kWin) / kWinStep + 1;
    p.nw2 = (d.z - kWin) / kWinStep + 1;
    // tiles of 32 x 8 windows, or 8 x 32 where that leaves fewer lanes idle
    const uint64_t wide = (p.nw0 + 31) / 32 * ((p.nw1 + 7) / 8), tall = (p.nw0 + 7) / 8 * ((p.nw1 + 31) / 32);
    const bool narrow = tall < wide;
    const uint64_t tx = narrow ? 8 : 32, ty = kThreads / tx;
    p.t0 = (p.nw0 + tx - 1) / tx;
    p.t1 = (p.nw1 + ty - 1) / ty;
    // Layers per tile: a tile goes through 2 * depth + 5 slices, so deep tiles do
    // less work, but the chip works on kResident tiles at a time and the last
    // round should be full: the depth with the fewest slices in a row.
    constexpr uint64_t kResident = 256 * kSsimPerCu<T>;
    uint64_t best = ~0ull, depth;
    for (uint64_t chunks = 1; chunks <= p.nw2 && chunks <= 4 * kResident; chunks = depth > 1 ? (p.nw2 + depth - 2) / (depth - 1) : ~0ull) {
        depth = (p.nw2 + chunks - 1) / chunks;   // and on to the fewest chunks that are less deep
        const uint64_t tiles = p.t0 * p.t1 * ((p.nw2 + depth - 1) / depth);
        const uint64_t cost = (tiles + kResident - 1) / kResident * (kWinStep * depth + kWin - kWinStep);
        if (cost < best) {
            best = cost;
            p.depth = depth;
            p.tiles = tiles;
        }
        if (tiles > 4 * kResident) break;   // only more work from here on
    }
    const uint64_t n = p.nw0 * p.nw1 * p.nw2;
    const bool single = window_by_window<T>(best, n, p.nw0);
    const uint64_t work = single ? (n + kThreads - 1) / kThreads : p.tiles;
    // A thread per window: two or four workgroups per CU. Where lanes read rows far apart (f64, or one window
    // along x) more of them only push each other's lines out of the L1: f32 7 x 9 x 2000005 3047 us with
    // four, 2100 with two; 4000005 x 7 x 7 628 with four, 960 with two.
    const unsigned cap = !single ? kMaxSsimBlocks : (sizeof(T) == 8 || p.nw0 == 1 ? 512 : 1024), blocks = work < cap ? (unsigned)work : cap;
    if (single)
        hipLaunchKernelGGL(windows_kernel<T>, dim3(blocks), dim3(kThreads), 0, st, x, y, p, gw, s.g.h_res);
    else if (narrow)
        hipLaunchKernelGGL((ssim_kernel<T, 8>), dim3(blocks), dim3(kThreads), 0, st, x, y, p, gw, s.g.h_res);
    else
        hipLaunchKernelGGL((ssim_kernel<T, 32>), dim3(blocks), dim3(kThreads), 0, st, x, y, p, gw, s.g.h_res);
    Q_HIP(hipGetLastError());
    Q_HIP(hipStreamSynchronize(st));
    if (s.g.h_res[cuszp::kGridResults - 1] != 0.0) return CUSZP_ERROR_INTERNAL;
    *out = s.g.h_res[0];
    return CUSZP_SUCCESS;
}

}  // namespace cuszp_quality

extern "C" int cuSZp_ssim(const void* d_oriData, const void* d_decData, cuszp_dims_t dims, cuszp_type_t type,
                          double* ssim, hipStream_t stream) {
    if (!d_oriData || !d_decData || !ssim) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (type == CUSZP_TYPE_FLOAT)
        return cuszp_quality::run_ssim((const float*)d_oriData, (const float*)d_decData, dims, ssim, stream);
    if (type == CUSZP_TYPE_DOUBLE)
        return cuszp_quality::run_ssim((const double*)d_oriData, (const double*)d_decData, dims, ssim, stream);
    return CUSZP_ERROR_INVALID_ARGUMENT;
}

extern "C" int cuSZp_quality(const void* d_oriData, const void* d_decData, size_t nbEle, cuszp_type_t type,
                             double* metrics, hipStream_t stream) {
    if (!d_oriData || !d_decData || !nbEle || !metrics) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (type == CUSZP_TYPE_FLOAT)
        return cuszp_quality::run((const float*)d_oriData, (const float*)d_decData, nbEle, metrics, stream);
    if (type == CUSZP_TYPE_DOUBLE)
        return cuszp_quality::run((const double*)d_oriData, (const double*)d_decData, nbEle, metrics, stream);
    return CUSZP_ERROR_INVALID_ARGUMENT;
}
