// Kernel instantiations for float: {1D,2D,3D} x {fixed,plain,outlier}, compress and decompress.
#include "launch.hpp"

namespace cuszp {

template <int D, int M, int W>
static hipError_t launch_c(const Item& item, const ScanCtx& sc, hipStream_t st) {
    if (D == 1 || item.geo.runs)
        return launch_tiles(compress_kernel<D, M, float, W, true>, W * kWaveSize, item.geo.ntiles, st, item, sc);
    return launch_tiles(compress_kernel<D, M, float, W, D == 1>, W * kWaveSize, item.geo.ntiles, st, item, sc);
}
template <int D, int M, int W>
static hipError_t launch_d(const Item& item, const unsigned long long* offs, hipStream_t st) {
    if (D == 1 || item.geo.runs)
        return launch_tiles(decompress_kernel<D, M, float, W, true>, W * kWaveSize, item.geo.ntiles, st, item, offs);
    return launch_tiles(decompress_kernel<D, M, float, W, D == 1>, W * kWaveSize, item.geo.ntiles, st, item, offs);
}

// offset pass: S bytes per plane (1D 4, 2D/3D 8), UB blocks per decode wave
template <int M, int S, int UB>
static hipError_t launch_o(const Item& item, uint64_t nunits, unsigned long long* offs, const ScanCtx& sc,
                           hipStream_t st) {
    const uint64_t limit = S == 4 ? item.geo.H : item.geo.nblocks;   // 2D/3D header pad bytes hold no block
    const int threads = prefix_threads(nunits * UB);
    const uint64_t seg = prefix_seg_bytes(threads), nseg = (nunits * UB + seg - 1) / seg;
    return launch_tiles(threads == 256 ? unit_offsets_kernel<M, S, UB, 256> : unit_offsets_kernel<M, S, UB, 1024>, threads, nseg,
                        st, (const uint8_t*)item.src, limit, item.geo.H, nunits, offs, sc);
}

#include "dispatch.inc"

hipError_t launch_compress_f32(int dim, int mode, int waves, const Item& item, const ScanCtx& sc, hipStream_t st) {
    CUSZP_DISPATCH(launch_c, item, sc, st)
}

hipError_t launch_decompress_f32(int dim, int mode, int waves, const Item& item, const unsigned long long* offs,
                                 hipStream_t st) {
    CUSZP_DISPATCH(launch_d, item, offs, st)
}

hipError_t launch_unit_offsets_f32(int dim, int mode, const Item& item, uint64_t nunits, unsigned long long* offs,
                                   const ScanCtx& sc, hipStream_t st) {
    static_assert(kChunksOf<float> * kChunkElems == 128 * 32 && kChunksOf<float> * kChunkElems == 64 * 64, "decode wave units");
    switch ((dim == 1 ? 0 : 3) + mode) {
        case 0: return launch_o<kFixed, 4, 128>(item, nunits, offs, sc, st);
        case 1: return launch_o<kPlain, 4, 128>(item, nunits, offs, sc, st);
        case 2: return launch_o<kOutlier, 4, 128>(item, nunits, offs, sc, st);
        case 3: return launch_o<kFixed, 8, 64>(item, nunits, offs, sc, st);
        case 4: return launch_o<kPlain, 8, 64>(item, nunits, offs, sc, st);
        case 5: return launch_o<kOutlier, 8, 64>(item, nunits, offs, sc, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace cuszp
