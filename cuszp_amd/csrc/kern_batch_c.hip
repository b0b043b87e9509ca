// Batched compress: launcher and the kernel of 4-wave workgroups (that of 8
// waves is a translation unit of its own, kern_batch_c8.hip: each holds every
// variant and takes the longest of all to compile).
#include "launch.hpp"

namespace cuszp {

// Advances the scan epoch of a batched plan; runs (one thread) before every
// compress launch, also inside captured graphs. (A decode kernel advances the
// epoch of its offset pass itself; the server's epochs come with its items.)
__global__ void bump_epoch_kernel(unsigned long long* epoch) {
    if (threadIdx.x == 0) epoch[0] = epoch[0] + 1;
}

hipError_t launch_compress_batch(int waves, int window, const Item* items, uint32_t nitems, uint64_t ntiles,
                                 const ScanCtx& sc, const unsigned long long* epoch, hipStream_t st) {
    if (!ntiles) return hipSuccess;
    if ((waves != 4 && waves != 8) || (window != 2 && window != 4)) return hipErrorInvalidValue;
    if (waves == 8) return launch_compress_batch8(window, items, nitems, ntiles, sc, epoch, st);
    return launch_tiles(compress_batch_kernel<4>, 4 * kWaveSize, ntiles, st, items, nitems, sc, epoch, window);
}

hipError_t launch_bump_epoch(unsigned long long* epoch, hipStream_t st) {
    hipLaunchKernelGGL(bump_epoch_kernel, dim3(1), dim3(64), 0, st, epoch);
    return hipGetLastError();
}

}  // namespace cuszp
