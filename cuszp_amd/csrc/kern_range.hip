// Value range of a device array and the relative error bound derived from it,
// the step before compression when the bound is relative: the reference CLI
// computes it on the host (examples/cuSZp.cpp:176-210): min and max over the
// array (comparisons, so NaNs are skipped unless the first element is NaN,
// which makes both NaN), then errorBound = rel * (max - min) in float
// arithmetic; for f64 arrays the difference is taken in double and rounded to
// float first.
//
// One launch reads the array once: each workgroup reduces a strided share with
// 16-byte loads and publishes its (min, max) pair; the last workgroup reduces
// the pairs (grid_words.hpp) and writes the result to pinned host memory.
#include <hip/hip_runtime.h>

#include <cmath>
#include <map>
#include <memory>
#include <mutex>

#include "../../include/cuSZp.h"
#include "grid_words.hpp"

namespace cuszp_range {

constexpr int kThreads = 256;
// Bound by the read. Four workgroups per CU with eight 16-byte loads in flight
// per lane cover the memory latency.
constexpr unsigned kMaxBlocks = 1024;
constexpr int kInFlight = 8;

template <class T>
struct Vec;
template <>
struct Vec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    static constexpr int N = 4;
};
template <>
struct Vec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    static constexpr int N = 2;
};

template <class T>
__device__ __forceinline__ void take(T v, T& mn, T& mx) {
    mn = v < mn ? v : mn;   // NaN compares false: skipped
    mx = v > mx ? v : mx;
}

template <class T>
__device__ __forceinline__ void block_reduce(T& mn, T& mx, T* smn, T* smx) {
    for (int o = 32; o > 0; o >>= 1) {
        const T a = __shfl_xor(mn, o, 64);
        const T b = __shfl_xor(mx, o, 64);
        mn = a < mn ? a : mn;
        mx = b > mx ? b : mx;
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smn[w] = mn;
        smx[w] = mx;
    }
    __syncthreads();
    mn = smn[0];
    mx = smx[0];
    for (int i = 1; i < kThreads / 64; ++i) {
        mn = smn[i] < mn ? smn[i] : mn;
        mx = smx[i] > mx ? smx[i] : mx;
    }
}

// x: the array; head: elements before the first 16-byte boundary; nv: whole
// vectors after it. gw: 2 values' words per workgroup; res: {min, max}, and in
// res[kGridResults - 1] whether a workgroup's words never came.
template <class T>
__global__ void __launch_bounds__(kThreads) range_kernel(const T* __restrict__ x, uint64_t n, uint64_t head,
                                                         uint64_t nv, const cuszp::GridWords gw, double* res) {
    typedef typename Vec<T>::type V;
    typedef cuszp::Words<T> W;
    constexpr int N = Vec<T>::N;
    __shared__ T smn[kThreads / 64], smx[kThreads / 64];
    __shared__ bool lost;
    if (threadIdx.x == 0) lost = false;
    T mn = INFINITY, mx = -INFINITY;
    const V* __restrict__ xv = (const V*)(x + head);
    const uint64_t stride = (uint64_t)gridDim.x * kThreads;
    uint64_t i = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
    for (; i < nv; i += kInFlight * stride) {   // past the end: the last vector again
        V v[kInFlight];
#pragma unroll
        for (int k = 0; k < kInFlight; ++k) {
            const uint64_t j = i + k * stride;
            v[k] = xv[j < nv ? j : nv - 1];
        }
#pragma unroll
        for (int k = 0; k < kInFlight; ++k) {
#pragma unroll
            for (int j = 0; j < N; ++j) take((T)v[k][j], mn, mx);
        }
    }
    if (blockIdx.x == 0) {   // elements before the first vector and after the last
        const uint64_t tail0 = head + nv * N;
        if (threadIdx.x < head) take(x[threadIdx.x], mn, mx);
        for (uint64_t t = tail0 + threadIdx.x; t < n; t += kThreads) take(x[t], mn, mx);
    }
    block_reduce(mn, mx, smn, smx);
    const bool last = blockIdx.x == gridDim.x - 1;
    if (!last) {
        if (threadIdx.x == 0) {
            const W a = W::of(mn), b = W::of(mx);
#pragma unroll
            for (int k = 0; k < W::N; ++k) {
                gw.put((uint64_t)blockIdx.x * 2 * W::N + k, a.u[k]);
                gw.put((uint64_t)blockIdx.x * 2 * W::N + W::N + k, b.u[k]);
            }
        }
        return;
    }
    bool ok = true;
    for (unsigned b = threadIdx.x; b + 1 < gridDim.x; b += kThreads) {
        uint32_t u[2 * W::N];
        ok &= gw.get_n(b * 2 * W::N, u);
        W a, c;
#pragma unroll
        for (int k = 0; k < W::N; ++k) {
            a.u[k] = u[k];
            c.u[k] = u[W::N + k];
        }
        const T va = a.value(), vc = c.value();
        mn = va < mn ? va : mn;
        mx = vc > mx ? vc : mx;
    }
    __syncthreads();   // smn/smx are reused
    if (!ok) lost = true;
    block_reduce(mn, mx, smn, smx);
    if (threadIdx.x == 0) {
        const T x0 = x[0];
        const bool nan0 = x0 != x0;   // the reference's loop starts from element 0
        cuszp::host_store(res, (double)(nan0 ? x0 : mn));
        cuszp::host_store(res + 1, (double)(nan0 ? x0 : mx));
        cuszp::host_store(res + cuszp::kGridResults - 1, lost ? 1.0 : 0.0);
    }
}

struct State {
    cuszp::GridState g;
    std::mutex mu;
};
constexpr uint64_t kWords = (uint64_t)kMaxBlocks * 2 * 2;   // (min, max) of two words each
std::mutex g_mu;
std::map<std::pair<int, hipStream_t>, std::unique_ptr<State>> g_state;

#define RANGE_HIP(call)                                \
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
int run(const T* x, size_t n, double* mn, double* mx, hipStream_t st) {
    int dev = 0;
    RANGE_HIP(hipGetDevice(&dev));
    State& s = state_for(dev, st);
    std::lock_guard<std::mutex> lk(s.mu);
    RANGE_HIP(cuszp::grid_state_init(s.g, kWords, st));
    cuszp::GridWords gw;
    RANGE_HIP(cuszp::grid_next_tag(s.g, kWords, st, gw));
    constexpr int N = Vec<T>::N;
    const uint64_t mis = (uint64_t)((uintptr_t)x % 16) / sizeof(T);
    uint64_t head = mis ? (uint64_t)N - mis : 0;
    if (head > n) head = n;
    const uint64_t nv = (n - head) / N;
    uint64_t blocks = (nv + (uint64_t)kInFlight * kThreads - 1) / ((uint64_t)kInFlight * kThreads);
    if (blocks < 1) blocks = 1;
    if (blocks > kMaxBlocks) blocks = kMaxBlocks;
    hipLaunchKernelGGL(range_kernel<T>, dim3((unsigned)blocks), dim3(kThreads), 0, st, x, (uint64_t)n, head, nv, gw,
                       s.g.h_res);
    RANGE_HIP(hipGetLastError());
    RANGE_HIP(hipStreamSynchronize(st));
    if (s.g.h_res[cuszp::kGridResults - 1] != 0.0) return CUSZP_ERROR_INTERNAL;
    *mn = s.g.h_res[0];
    *mx = s.g.h_res[1];
    return CUSZP_SUCCESS;
}

}  // namespace cuszp_range

extern "C" {

int cuSZp_value_range(const void* d_data, size_t nbEle, cuszp_type_t type, double* min_val, double* max_val,
                      hipStream_t stream) {
    if (!d_data || !nbEle || !min_val || !max_val) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (type == CUSZP_TYPE_FLOAT) return cuszp_range::run((const float*)d_data, nbEle, min_val, max_val, stream);
    if (type == CUSZP_TYPE_DOUBLE) return cuszp_range::run((const double*)d_data, nbEle, min_val, max_val, stream);
    return CUSZP_ERROR_INVALID_ARGUMENT;
}

int cuSZp_rel_error_bound(const void* d_data, size_t nbEle, cuszp_type_t type, float rel, float* errorBound,
                          hipStream_t stream) {
    if (!errorBound) return CUSZP_ERROR_INVALID_ARGUMENT;
    double mn = 0, mx = 0;
    const int rc = cuSZp_value_range(d_data, nbEle, type, &mn, &mx, stream);
    if (rc) return rc;
    // examples/cuSZp.cpp:186 (f32: float subtraction) and :207 (f64: double, then float)
    const float range = type == CUSZP_TYPE_FLOAT ? (float)mx - (float)mn : (float)(mx - mn);
    *errorBound = rel * range;
    return CUSZP_SUCCESS;
}

}  // extern "C"
