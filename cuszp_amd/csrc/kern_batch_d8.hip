// Batched decompress kernel of 8-wave workgroups (see kern_batch_d.hip).
#include "launch.hpp"

namespace cuszp {

hipError_t launch_decompress_batch8(const Item* items, uint32_t nitems, uint64_t ntiles,
                                    const unsigned long long* offs, unsigned long long* bump, hipStream_t st) {
    return launch_tiles(decompress_batch_kernel<8>, 8 * kWaveSize, ntiles, st, items, nitems, offs, bump);
}

}  // namespace cuszp
