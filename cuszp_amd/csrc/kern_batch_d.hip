// Batched decompress: launchers, the offset pass and the kernel of 4-wave
// workgroups (that of 8 waves: kern_batch_d8.hip).
#include "launch.hpp"

namespace cuszp {

hipError_t launch_decompress_batch(int waves, const Item* items, uint32_t nitems, uint64_t ntiles,
                                   const unsigned long long* offs, unsigned long long* bump, hipStream_t st) {
    if (!ntiles) return hipSuccess;
    if (waves != 4 && waves != 8) return hipErrorInvalidValue;
    if (waves == 8) return launch_decompress_batch8(items, nitems, ntiles, offs, bump, st);
    return launch_tiles(decompress_batch_kernel<4>, 4 * kWaveSize, ntiles, st, items, nitems, offs, bump);
}

hipError_t launch_offsets_batch(int waves, const Item* items, uint32_t nitems, uint64_t nseg, unsigned long long* offs,
                                const ScanCtx& sc, const unsigned long long* epoch, hipStream_t st) {
    return launch_tiles(waves == 8 ? unit_offsets_batch_kernel<8> : unit_offsets_batch_kernel<4>, kWaveSize, nseg, st, items,
                        nitems, offs, sc, epoch);
}

}  // namespace cuszp
