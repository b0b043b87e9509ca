// Batched compress kernel of 8-wave workgroups (see kern_batch_c.hip).
#include "launch.hpp"

namespace cuszp {

hipError_t launch_compress_batch8(int window, const Item* items, uint32_t nitems, uint64_t ntiles, const ScanCtx& sc,
                                  const unsigned long long* epoch, hipStream_t st) {
    return launch_tiles(compress_batch_kernel<8>, 8 * kWaveSize, ntiles, st, items, nitems, sc, epoch, window);
}

}  // namespace cuszp
