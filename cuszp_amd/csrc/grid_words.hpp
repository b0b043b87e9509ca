// Reduction of a grid's per-workgroup partial results inside one launch.
//
// Every workgroup publishes its partials as 64-bit words {tag, 32 value bits}
// with relaxed agent-scope stores; the last workgroup of the grid reads each
// word until it carries the launch's tag and reduces them. The tag travels in
// the same word as the value, so nothing has to be ordered: no release or
// acquire (which on this chip write back and invalidate the XCD's L2, per
// workgroup) and no counter that all workgroups increment (about 12 ns each).
// Measured on 64 MiB of f32 (value range, 2048 workgroups): 77-95 us with an
// acquire-release ticket per workgroup, 17 us this way.
//
// Only the last workgroup waits, and no workgroup waits for it, so the grid
// drains whatever the dispatch order; the polls are bounded all the same.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cuszp {

constexpr uint32_t kWordPolls = 1u << 22;   // far above any legitimate wait

struct GridWords {
    unsigned long long* w;   // nw words per workgroup
    uint32_t tag;            // of this launch; words of earlier launches carry others

    __device__ __forceinline__ void put(uint64_t i, uint32_t v) const {
        __hip_atomic_store(w + i, ((unsigned long long)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // N words from word i on, `stride` apart, their loads in flight together, until all of them
    // carry the tag; false if they did not within the bound.
    template <int N>
    __device__ __forceinline__ bool get_n(uint64_t i, uint32_t (&v)[N], uint64_t stride = 1) const {
        for (uint32_t p = 0; p < kWordPolls; ++p) {
            unsigned long long x[N];
#pragma unroll
            for (int k = 0; k < N; ++k) x[k] = __hip_atomic_load(w + i + k * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            bool ok = true;
#pragma unroll
            for (int k = 0; k < N; ++k) {
                v[k] = (uint32_t)x[k];
                ok &= (uint32_t)(x[k] >> 32) == tag;
            }
            if (ok) return true;
            __builtin_amdgcn_s_sleep(1);
        }
        return false;
    }
};

// A value as 32-bit words.
template <class T>
struct Words {
    static constexpr int N = sizeof(T) / 4;
    uint32_t u[N];
    __device__ __forceinline__ static Words of(T v) {
        Words r;
        __builtin_memcpy(r.u, &v, sizeof(T));
        return r;
    }
    __device__ __forceinline__ T value() const {
        T v;
        __builtin_memcpy(&v, u, sizeof(T));
        return v;
    }
};

// Results that the host reads after the stream is synchronised, in pinned
// coherent host memory.
__device__ __forceinline__ void host_store(double* p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Host side: the words and the pinned results of one (device, stream).
struct GridState {
    unsigned long long* d_words = nullptr;
    double* h_res = nullptr;   // pinned, written by the kernels
    uint32_t tag = 0;
};
constexpr int kGridResults = 16;   // doubles at h_res; the last one is a kernel's "gave up waiting" flag

// Buffers of `words` words (called with the state's lock held); a failed
// allocation leaves the state empty, and the next call allocates again.
inline hipError_t grid_state_init(GridState& s, uint64_t words, hipStream_t st) {
    if (s.d_words) return hipSuccess;
    unsigned long long* w = nullptr;
    double* h = nullptr;
    hipError_t e = hipMalloc((void**)&w, words * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipHostMalloc((void**)&h, kGridResults * sizeof(double), hipHostMallocCoherent);
    if (e == hipSuccess) e = hipMemsetAsync(w, 0, words * sizeof(unsigned long long), st);
    if (e != hipSuccess) {
        if (w) (void)hipFree(w);
        if (h) (void)hipHostFree(h);
        return e;
    }
    s.d_words = w;
    s.h_res = h;
    return hipSuccess;
}
// Tag of the next launch. Tags repeat only after 2^32 launches; the words are cleared then.
inline hipError_t grid_next_tag(GridState& s, uint64_t words, hipStream_t st, GridWords& g) {
    if (++s.tag == 0) {
        const hipError_t e = hipMemsetAsync(s.d_words, 0, words * sizeof(unsigned long long), st);
        if (e != hipSuccess) return e;
        s.tag = 1;
    }
    g.w = s.d_words;
    g.tag = s.tag;
    return hipSuccess;
}

}  // namespace cuszp
