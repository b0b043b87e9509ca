// Host-side launch interface between the C ABI (cuszp_api.cpp, cuszp_batch.cpp)
// and the kernel instantiations (kern_f32.hip, kern_f64.hip, kern_batch_*.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cuszp_kernels.hpp"

namespace cuszp {

// Tile plan: waves per workgroup (4 or 8), chunks per wave and the number of
// tiles (tile shape: tile_groups).
// CUSZP_WAVES in the environment overrides the choice (tuning experiments).
struct TilePlan {
    int waves;
    int kc;
    uint64_t ntiles;
};
TilePlan plan_tiles(int dim, int type, const Geom& g);
// Tiles up to which a shape short of the largest is taken, by its waves.
constexpr uint64_t shape_tiles(int waves) { return waves == 4 ? 256 : 384; }

// Single-array launches; item.param is 0.5/eb (compress) or eb (decompress).
hipError_t launch_compress_f32(int dim, int mode, int waves, const Item& item, const ScanCtx& sc, hipStream_t st);
hipError_t launch_compress_f64(int dim, int mode, int waves, const Item& item, const ScanCtx& sc, hipStream_t st);
// Single-array decompression reads each wave's payload offset from `offs`,
// which launch_unit_offsets_* fills first on the same stream; a null `offs`
// (headers of at most kDirectHeader bytes) has every workgroup sum them up.
hipError_t launch_decompress_f32(int dim, int mode, int waves, const Item& item, const unsigned long long* offs,
                                 hipStream_t st);
hipError_t launch_decompress_f64(int dim, int mode, int waves, const Item& item, const unsigned long long* offs,
                                 hipStream_t st);
// Offset table of a single-array decompression (unit_offsets_kernel): offs[u]
// for the nunits decode waves of `item`'s plan, from the header bytes of the
// stream at item.src; sc's status words serve the pass's own scan (one per
// segment of prefix_seg_bytes header bytes).
hipError_t launch_unit_offsets_f32(int dim, int mode, const Item& item, uint64_t nunits, unsigned long long* offs,
                                   const ScanCtx& sc, hipStream_t st);
hipError_t launch_unit_offsets_f64(int dim, int mode, const Item& item, uint64_t nunits, unsigned long long* offs,
                                   const ScanCtx& sc, hipStream_t st);
// Blocks one decode wave handles.
constexpr uint64_t unit_blocks(int dim, bool f64, int kc = 0) { return tile_groups(f64, 1, kc) * (dim == 1 ? 2 : 1); }
// The pass of a single array takes every wave for a full one (unit_blocks without kc,
// the kernels' UB). It runs for headers above kDirectHeader only, and those make more
// groups (1D two blocks each) than the longest array of a shorter shape has.
constexpr bool pass_takes_full_tiles(bool f64) {
    return kDirectHeader / 2 >= tile_groups(f64, 8, (f64 ? kChunksOf<double> : kChunksOf<float>) / 2) * shape_tiles(8);
}
static_assert(pass_takes_full_tiles(false) && pass_takes_full_tiles(true), "the offset pass needs full tiles");
// Segments of the offset pass over `nunits` units.
inline uint64_t unit_segments(int dim, bool f64, uint64_t nunits) {
    const uint64_t header = nunits * unit_blocks(dim, f64), seg = prefix_seg_bytes(prefix_threads(header));
    return (header + seg - 1) / seg;
}

// Batched launches over a device table of items (ordered by tile0), one
// workgroup per tile; the scan tag is read from *epoch when the kernel starts
// (graph-replay safe). waves: 4 or 8 per workgroup; window: lookback words per
// lane, 2 or 4 (128 or 256 predecessors per round trip).
hipError_t launch_compress_batch(int waves, int window, const Item* items, uint32_t nitems, uint64_t ntiles,
                                 const ScanCtx& sc, const unsigned long long* epoch, hipStream_t st);
hipError_t launch_compress_batch8(int window, const Item* items, uint32_t nitems, uint64_t ntiles, const ScanCtx& sc,
                                  const unsigned long long* epoch, hipStream_t st);
// Batched decompression: offs[ntiles * waves], filled by launch_offsets_batch on
// the same stream, or null where no array's header is longer than kBatchDirectHeader;
// bump (may be null): an epoch word to advance, for the next pass.
hipError_t launch_decompress_batch(int waves, const Item* items, uint32_t nitems, uint64_t ntiles,
                                   const unsigned long long* offs, unsigned long long* bump, hipStream_t st);
hipError_t launch_decompress_batch8(const Item* items, uint32_t nitems, uint64_t ntiles,
                                    const unsigned long long* offs, unsigned long long* bump, hipStream_t st);
// The offset pass over nseg segments in all (items ordered by seg0, batch_segments
// each), whose waves have whole threads' header bytes (unit_blocks % kPrefixBytes == 0).
hipError_t launch_offsets_batch(int waves, const Item* items, uint32_t nitems, uint64_t nseg, unsigned long long* offs,
                                const ScanCtx& sc, const unsigned long long* epoch, hipStream_t st);
static_assert(unit_blocks(2, false, 4) % kPrefixBytes == 0 && unit_blocks(2, true, 4) % kPrefixBytes == 0,
              "4 chunks per wave, the fewest under a pass, are whole threads' header bytes");
inline uint64_t batch_segments(int dim, bool f64, int kc, uint64_t nunits) {
    return (nunits * unit_blocks(dim, f64, kc) + kBatchSegBytes - 1) / kBatchSegBytes;
}
// Increments *epoch (one thread); runs before each compress launch of a plan.
hipError_t launch_bump_epoch(unsigned long long* epoch, hipStream_t st);
// Largest grid of a tile launch; arrays with more tiles take several launches.
constexpr uint64_t kMaxGrid = 1ull << 22;

// Launches with one workgroup per tile: tile = base + blockIdx.x, in launches
// of up to kMaxGrid tiles. Tiles are numbered in launch order, so the
// predecessors a tile waits on normally belong to workgroups that started
// earlier; the lookback's stealing covers any order.
template <class Kernel, class... Args>
hipError_t launch_tiles(Kernel kernel, int threads, uint64_t ntiles, hipStream_t st, Args... args) {
    for (uint64_t base = 0; base < ntiles; base += kMaxGrid) {
        const uint64_t n = ntiles - base < kMaxGrid ? ntiles - base : kMaxGrid;
        hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(threads), 0, st, args..., base);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace cuszp
