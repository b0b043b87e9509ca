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
    r.oo = a.oo + b.oo + eo * eo * w;
    r.dd = a.dd + b.dd + ed * ed * w;
    r.od = a.od + b.od + eo * ed * w;
    return r;
}

// A share's sums (ori, dec, dec^2, err^2), maxima (ori, -ori, err, rel err) and moments.
constexpr int kFigures = 14;
struct Figures {
    double s[4], m[4];
    Moments c;
    __device__ __forceinline__ void init() {
        for (int k = 0; k < 4; ++k) {
            s[k] = 0;
            m[k] = k < 2 ? -INFINITY : 0.0;
        }
        c = Moments{0, 0, 0, 0, 0, 0};
    }
    __device__ __forceinline__ void add(const Figures& b) {
        for (int k = 0; k < 4; ++k) {
            s[k] += b.s[k];
            m[k] = fmax(m[k], b.m[k]);
        }
        c = merge(c, b.c);
    }
    template <class F>
    __device__ __forceinline__ void each(F&& f) {
        for (int k = 0; k < 4; ++k) f(k, s[k]);
        for (int k = 0; k < 4; ++k) f(4 + k, m[k]);
        f(8, c.n);
        f(9, c.mo);
        f(10, c.md);
        f(11, c.oo);
        f(12, c.dd);
        f(13, c.od);
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
// sums) and 60 us this way.
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
        f.s[2] += (double)(T)(d * d);
        f.s[3] += (double)(T)(err * err);
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
        f.s[0] += so;
        f.s[1] += sd;
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
            f.s[0] += (double)ori[i];
            f.s[1] += (double)dec[i];
            f.c = merge(f.c, Moments{1, (double)ori[i], (double)dec[i], 0, 0, 0});
        }
    for (int k = 0; k < 4; ++k) f.m[k] = (double)m[k];
    block_figures(f, sm);
    typedef cuszp::Words<double> W;
    if (blockIdx.x != gridDim.x - 1) {
        if (threadIdx.x == 0)
            f.each([&](int k, double& v) {
                const W w = W::of(v);
                gw.put(((uint64_t)blockIdx.x * kFigures + k) * 2, w.u[0]);
                gw.put(((uint64_t)blockIdx.x * kFigures + k) * 2 + 1, w.u[1]);
            });
        return;
    }
    if (threadIdx.x != 0) f.init();
    bool ok = true;
    for (unsigned b = threadIdx.x; b + 1 < gridDim.x; b += kThreads) {
        uint32_t u[2 * kFigures];
        ok &= gw.get_n((uint64_t)b * kFigures * 2, u);
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
        s.lo = a.lo < s.lo ? a.lo : s.lo;
        s.hi = a.hi > s.hi ? a.hi : s.hi;
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

template <class T>
__device__ __forceinline__ double ssim_of(const WinStats<T>& s) {
    constexpr double np = kWin * kWin * kWin;
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

// Windows of a volume, tiled: TX x TY windows of a tile along x and y, `depth`
// layers of windows along z.
struct SsimPlan {
    uint64_t s0, s1;             // extents along x and y
    uint64_t nw0, nw1, nw2;      // windows along x, y, z
    uint64_t t0, t1, tiles;      // tiles along x and y, and in all
    uint64_t depth;              // layers of windows per tile
};

// One workgroup per tile (then the tile gridDim.x further on). It walks down
// the tile's slices; for each, threads first make the statistics of the rows of
// seven values that windows start with (2 TY + 5 rows, TX per row), then each
// thread, one window column, joins seven of them to its slice of 7 x 7 and keeps
// the last seven slices in registers; every second slice completes a layer.
// A value takes part in 3.5 rows, 3.5 x 3.5 slices... through these sums and is
// read 3.5 times (from L1), where a window by itself reads 343 pairs twice.
// Bound by the f64 arithmetic: about 100 operations per value. 2.5 M windows of
// f32 took 784 us as one thread per window, 190 us this way.
template <class T, int TX>
__global__ void __launch_bounds__(kThreads, sizeof(T) == 4 ? 3 : 2) ssim_kernel(const T* __restrict__ x, const T* __restrict__ y,
                                                        const SsimPlan p, const cuszp::GridWords gw, double* res) {
    constexpr int TY = kThreads / TX, ROWS = kWinStep * TY + kWin - kWinStep;
    typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    __shared__ double rs[5][ROWS][TX];
    __shared__ T rlo[ROWS][TX], rhi[ROWS][TX];
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
        // threads past the last window read the last one's values and count nothing
        const uint64_t cx = kWinStep * (wx0 + tx < p.nw0 ? wx0 + tx : p.nw0 - 1);
        WinStats<T> ring[kWin];
        auto slice = [&](uint64_t z) -> WinStats<T> {   // this thread's 7 x 7 of slice z
            __syncthreads();                            // the previous slice's rows have been read
#pragma unroll 1
            for (int r0 = 0; r0 < ROWS; r0 += TY) {
                const int row = r0 + ty;
                if (row < ROWS) {
                    uint64_t yy = kWinStep * wy0 + row;
                    yy = yy < p.s1 ? yy : p.s1 - 1;
                    const uint64_t at = (z * p.s1 + yy) * p.s0 + cx;
                    T a[kWin], c[kWin];
#pragma unroll
                    for (int i = 0; i < kWin / 2; ++i) {
                        const V2 va = *(const V2*)(x + at + 2 * i), vc = *(const V2*)(y + at + 2 * i);
                        a[2 * i] = va[0];
                        a[2 * i + 1] = va[1];
                        c[2 * i] = vc[0];
                        c[2 * i + 1] = vc[1];
                    }
                    a[kWin - 1] = x[at + kWin - 1];
                    c[kWin - 1] = y[at + kWin - 1];
                    double sx = 0, sy = 0;
                    T lo = a[0], hi = a[0];
#pragma unroll
                    for (int i = 0; i < kWin; ++i) {
                        sx += (double)a[i];
                        sy += (double)c[i];
                        lo = a[i] < lo ? a[i] : lo;
                        hi = a[i] > hi ? a[i] : hi;
                    }
                    const double mx = sx * (1.0 / kWin), my = sy * (1.0 / kWin);
                    double xx = 0, yy2 = 0, xy = 0;
#pragma unroll
                    for (int i = 0; i < kWin; ++i) {
                        const double u = (double)a[i] - mx, v = (double)c[i] - my;
                        xx = fma(u, u, xx);
                        yy2 = fma(v, v, yy2);
                        xy = fma(u, v, xy);
                    }
                    rs[0][row][tx] = sx;
                    rs[1][row][tx] = sy;
                    rs[2][row][tx] = xx;
                    rs[3][row][tx] = yy2;
                    rs[4][row][tx] = xy;
                    rlo[row][tx] = lo;
                    rhi[row][tx] = hi;
                }
            }
            __syncthreads();
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
        // 2 * layers + 5 slices: one, then pairs; from the third pair on each completes a layer
        const uint64_t z0 = kWinStep * wz0;
        for (int k = 0; k < kWin; ++k) ring[k] = WinStats<T>{0, 0, 0, 0, 0, T(0), T(0)};
        ring[kWin - 3] = slice(z0);
#pragma unroll 1
        for (uint64_t l = 0; l < layers + 2; ++l) {
#pragma unroll
            for (int k = kWin - 2; k < kWin; ++k) ring[k] = slice(z0 + 2 * l + (uint64_t)(k - (kWin - 3)));
            if (l >= 2 && mine) {
                Join<T> q;
                q.first(ring[0]);
#pragma unroll
                for (int k = 1; k < kWin; ++k) q.next(ring[k]);
                total += ssim_of(q.done((double)(kWin * kWin)));
            }
#pragma unroll
            for (int k = 0; k < kWin - 2; ++k) ring[k] = ring[k + 2];
        }
    }
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
        cuszp::host_store(res, total / (double)(p.nw0 * p.nw1 * p.nw2));
        cuszp::host_store(res + cuszp::kGridResults - 1, lost ? 1.0 : 0.0);
    }
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
    const double mse = r[3] / N, range = r[4] + r[5];            // r[5]: max of -ori
    out[0] = mse;                                                // src/cuSZp_utility.cu:937-946
    out[1] = range;
    out[2] = 20 * log10(range) - 10 * log10(mse);
    out[3] = sqrt(r[3]);
    out[4] = sqrt(r[3]) / sqrt(r[2]);
    out[5] = sqrt(mse) / range;
    out[6] = r[6];                                               // max |dec - ori|
    out[7] = r[7];                                               // max |dec - ori| / |ori| over ori != 0
    out[8] = (r[13] / N) / sqrt(r[11] / N) / sqrt(r[12] / N);    // correlation (acEff)
    return CUSZP_SUCCESS;
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
    // Layers per tile: a tile reads 5 slices before its first layer, so few and
    // deep tiles do less work, but the chip holds kMaxSsimBlocks workgroups and
    // needs about that many; at least 4 layers.
    uint64_t chunks = (kMaxSsimBlocks + p.t0 * p.t1 - 1) / (p.t0 * p.t1);
    if (chunks > (p.nw2 + 3) / 4) chunks = (p.nw2 + 3) / 4;
    p.depth = (p.nw2 + chunks - 1) / chunks;
    p.tiles = p.t0 * p.t1 * ((p.nw2 + p.depth - 1) / p.depth);
    const unsigned blocks = p.tiles < kMaxSsimBlocks ? (unsigned)p.tiles : kMaxSsimBlocks;
    if (narrow)
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
