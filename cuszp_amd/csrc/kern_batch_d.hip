// Batched decompress: launcher and the kernel of 4-wave workgroups (that of 8
// waves: kern_batch_d8.hip).
#include "launch.hpp"

namespace cuszp {

hipError_t launch_decompress_batch(int waves, int window, const Item* items, uint32_t nitems, uint64_t ntiles,
                                   const ScanCtx& sc, const unsigned long long* epoch, hipStream_t st) {
    if (!ntiles) return hipSuccess;
    if ((waves != 4 && waves != 8) || (window != 2 && window != 4)) return hipErrorInvalidValue;
    if (waves == 8) return launch_decompress_batch8(window, items, nitems, ntiles, sc, epoch, st);
    return launch_tiles(decompress_batch_kernel<4>, 4 * kWaveSize, ntiles, st, items, nitems, sc, epoch, window);
}

}  // namespace cuszp
