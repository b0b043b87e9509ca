// Fused error-bounded compress / decompress kernels for gfx950 (MI355X).
//
// One compress kernel and one decompress kernel, templated over
// {1D, 2D, 3D} x {fixed, plain, outlier} x {f32, f64}. They replace the 36
// per-variant kernels of cuSZp (src/cuSZp_kernels_{1D,2D,3D}_f{32,64}.cu) and
// produce/consume the same byte stream.
//
// Work decomposition (wave64-native; see the repository's design notes):
//   * a "group" is 64 consecutive elements of cuSZp block order: two 32-element
//     blocks in 1D, one 8x8 (2D) or 4x4x4 (3D) block otherwise. A "chunk" is 8
//     groups, 512 elements: a wave holds one, a lane two quads of four
//     consecutive elements (QuadLane);
//   * a workgroup is WAVES waves and handles one tile: each wave owns
//     Geom::kc chunks. The grid has one workgroup per tile (tile = launch base +
//     blockIdx.x). No ticket atomics: one hot device-scope atomic serialises at
//     about 12 ns per operation on MI355X;
//   * sign and magnitude bits travel as byte slices of a quad, as many as the
//     chunk's largest rate needs (one for 7 bits), which a transpose across
//     eight lanes turns into plane words in the bit order of cuSZp's sign/plane
//     bytes (to_planes); decompression runs the inverse;
//   * a block's rate is the bit length of its largest residual; every lane
//     keeps its own block's books in compression, and in decompression one lane
//     per block, once per wave;
//   * the inter-tile exclusive scan of compressed bytes (compress tiles, and the
//     pass over a long header that precedes decompression) is a single-pass
//     decoupled lookback: one 64-bit status word per tile packs
//     {epoch, flag, value}, is read 128 or 256 predecessors at a time by one
//     wave, and
//     needs only relaxed agent-scope atomics (no fences: the value travels in
//     the same word as its flag). Forward progress does not rely on every
//     workgroup being resident: a wave that has waited too long for a
//     predecessor claims it and recomputes that tile's byte count itself;
//   * the batched kernels run the same per-variant loops over a table of
//     arrays; each array's tiles form their own scan segment.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace cuszp {

constexpr int kWaveSize = 64;

enum : int { kFixed = 0, kPlain = 1, kOutlier = 2 };

// Tile status word: [63:40] epoch tag, [39:38] flag, [37:0] byte count.
// Flags: 1 = aggregate of the tile, 2 = inclusive prefix, 3 = claimed by a
// waiting wave that is computing the aggregate; 0 = nothing yet.
constexpr int kEpochShift = 40;
constexpr uint64_t kEpochMask = (1ull << 24) - 1;
constexpr uint64_t kFlagAgg = 1ull << 38;
constexpr uint64_t kFlagPrefix = 2ull << 38;
constexpr uint64_t kFlagClaim = 3ull << 38;
constexpr uint64_t kFlagMask = 3ull << 38;
constexpr uint64_t kValueMask = (1ull << 38) - 1;
constexpr uint64_t kTagMask = ~(kFlagMask | kValueMask);

// Bits of the sticky error words.
constexpr uint32_t kErrOverflow = 1u;    // compressed stream exceeds output capacity
constexpr uint32_t kErrTruncated = 2u;   // stream shorter than its header describes
constexpr uint32_t kErrStall = 4u;       // a lookback gave up waiting (internal error; output invalid)
constexpr uint32_t kInfoStolen = 8u;     // a waiting wave computed a predecessor's byte count (not an error)
constexpr uint32_t kWarnLossy = 16u;     // a 2D/3D outlier block has rate byte 32, which decoders read as rate 0
constexpr uint32_t kErrMask = 7u;

// Item flags. kItemStreamNt: compress writes the stream with nontemporal
// stores. Set for arrays of at least kStreamNtBytes: their streams outgrow the
// memory-side cache at typical ratios, and dirty stream lines left there
// would be written back during the next kernel. A smaller stream is stored
// normally and stays cached for its next reader.
constexpr uint32_t kItemStreamNt = 1u;
constexpr uint64_t kStreamNtBytes = 1ull << 30;

// Bound on lookback polls (each polls the status words once): far above any
// legitimate wait, it guarantees that every wave of a launch exits even if a
// predecessor tile never publishes.
constexpr uint32_t kSpinLimit = 1u << 18;
// A wait longer than this (s_memrealtime ticks: 100 us at the 100 MHz
// reference clock) makes the waiting wave compute pending predecessors itself.
constexpr uint64_t kStealTicks = 10000;

// Tile shape. A wave works through up to kChunksOf<T> chunks of 512 elements
// (16 KiB of values), or fewer where an array would not fill the chip
// (Geom::kc); a tile is WAVES * kc chunks, for compress and decompress alike.
constexpr int kChunkElems = 512;
template <class T> constexpr int kChunksOf = sizeof(T) == 4 ? 8 : 4;
__host__ __device__ constexpr uint64_t tile_groups(bool f64, int waves, int kc = 0) {   // groups of 64 elements
    return (uint64_t)waves * (kc ? kc : (f64 ? kChunksOf<double> : kChunksOf<float>)) * (kChunkElems / 64);
}

struct Geom {
    uint64_t n;         // elements
    uint64_t nblocks;   // cuSZp blocks
    uint64_t H;         // header bytes
    uint64_t ntiles;    // tiles of the array
    uint64_t XY;        // X*Y
    uint32_t X, Y, Z;
    uint32_t Bx, By;    // blocks along x and y (2D/3D)
    uint32_t kc;        // chunks per wave of a tile (at most kChunksOf)
    uint32_t runs;      // every chunk's blocks lie inside the array, 2D/3D consecutive along x (extents multiples
                        // of the block, Bx of a chunk's 8 blocks), and their places fit 32-bit offsets
    uint32_t near;      // 2D/3D: the places of a chunk's blocks fit 32-bit offsets from the first one's
};

// Launch-wide scan state.
struct ScanCtx {
    unsigned long long* status;     // tile status words, one per tile of the launch
    unsigned int* err;              // sticky error bits of the launch (kErrStall, kInfoStolen)
    unsigned long long* diag;       // [0] first stalled tile + 1, [1] its missing predecessor, [2] word seen;
                                    // with `stats`: [4] polls that found a window unresolved, [5] lookbacks
                                    // that polled, [6] predecessors claimed, [7] clock ticks spent waiting
    unsigned long long* mark;       // as Item::mark
    unsigned long long tag;         // epoch << kEpochShift
    uint32_t steal_ticks;           // wait (s_memrealtime ticks) before a pending predecessor is claimed
    uint32_t hold_every;            // scan stress: tile t with t % hold_every == hold_every - 1 waits
    uint32_t hold_ticks;            //   hold_ticks before it publishes anything (0: off)
    uint32_t stats;                 // nonzero: accumulate the lookback counters into diag[4..7]
};

// One array of a launch. The single-array kernels take it as an argument; the
// batched kernels read a table of them.
struct Item {
    const void* src;                // compress: values; decompress: stream
    void* dst;                      // compress: stream; decompress: values
    uint64_t limit;                 // compress: stream capacity; decompress: stream length
    unsigned long long* total;      // out: stream length, written by the last tile (may be null)
    unsigned long long* host_total; // the same once more, in pinned host memory (may be null)
    unsigned int* err;              // sticky error bits of this array (kErrOverflow, kErrTruncated)
    unsigned long long* mark;       // pinned host word set to 1 with every bit of an err word (may be null)
    double param;                   // compress: 0.5/eb, decompress: eb (exact in the array's type)
    uint64_t tile0;                 // first tile of the array in the launch (its scan segment start)
    uint64_t seg0;                  // batched decompress: its first segment in the launch's offset pass
    uint32_t variant;               // type * 9 + (dim - 1) * 3 + mode
    uint32_t flags;                 // kItemStreamNt
    Geom geo;                       // geo.ntiles: tiles of this array
};

// Sets a bit of a sticky error word. The words stay in device memory, where all
// workgroups meet; the mark tells the host, which would otherwise copy them back
// after every call, that there is anything to read.
__device__ __forceinline__ void raise_bit(unsigned int* err, uint32_t bit, unsigned long long* mark) {
    atomicOr(err, bit);
    if (mark) __hip_atomic_store(mark, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// wave64 primitives
// ---------------------------------------------------------------------------
// Lanes whose source is outside the row/wave read 0. With every row and bank
// enabled that is bound_ctrl (no old value to materialise); masked rows/banks
// keep the old value 0.
template <int CTRL, int ROWS = 0xf, int BANKS = 0xf>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
    if constexpr (ROWS == 0xf && BANKS == 0xf)
        return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, ROWS, BANKS, true);
    else
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, BANKS, false);
}
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114, kDppRowShr8 = 0x118;
constexpr int kDppWaveShr1 = 0x138, kDppHalfMirror = 0x141;
constexpr int kDppRowRor8 = 0x128;
constexpr int kDppBcast15 = 0x142, kDppBcast31 = 0x143;
constexpr int kDppQuadSwap1 = 0xB1;   // quad_perm [1,0,3,2]
constexpr int kDppQuadSwap2 = 0x4E;   // quad_perm [2,3,0,1]
constexpr int kDppQuadShr1 = 0x90;    // quad_perm [0,0,1,2]
constexpr int kDppQuadShr2 = 0x40;    // quad_perm [0,0,0,1]
constexpr int kDppRowNewBcast0 = 0x150;   // lane 0 of each row to the whole row

__device__ __forceinline__ uint32_t rdlane(uint32_t v, uint32_t l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
// A value the compiler cannot prove wave-uniform but that is (kept in SGPRs,
// so that uniform-base + 32-bit-offset addressing applies).
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32)) << 32);
}

template <int J>
__device__ __forceinline__ uint32_t swizzle_xor(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x1f | (J << 10));
}
// (m & a) | (~m & b) in one v_bfi_b32 (the compiler otherwise emits and + and_or)
__device__ __forceinline__ uint32_t bfi(uint32_t m, uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}

// ---------------------------------------------------------------------------
// Byte slices and plane words.
//
// A lane holds four consecutive elements (a quad) of a 32-element half, which
// eight lanes hold together: lane k = lane & 7 has elements 4k .. 4k+3. Slice t
// of a quad is a word with byte t of its four elements (element 3 - j in byte
// j). to_planes turns a slice that the eight lanes hold into the plane words of
// bits 8t .. 8t+7 of the half, one per lane: lane k gets plane
// 8t + plane_of_lane(k). In the stream, element e of a half sits at bit e^7 of
// its plane word (byte e/8, bit 7-e%8); that order comes out by itself.
//
// The slice is transposed as 8x8 bits over lane pairs (two exchanges inside the
// word, one of nibbles with lane ^ 1), then as 4x4 bytes over the four pairs
// (lane ^ 2, lane ^ 4): 15 VALU operations for 32 elements' eight planes, where
// one element per lane and a 32x32 transpose took 16 for any number of planes
// of 64 elements, i.e. 4 times as many for the one slice that most data need.
// from_planes is the inverse.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t plane_of_lane(uint32_t k) { return 4 * (k & 1) + 2 * ((k >> 2) & 1) + ((k >> 1) & 1); }
struct PlaneConsts {
    uint32_t rot, msk, sel2, sel4;
    // dec: for from_planes
    __device__ __forceinline__ void init(int lane, bool dec) {
        const bool odd = lane & 1;
        rot = odd != dec ? 4 : 28;                             // bits to the right: 28 is 4 to the left
        msk = odd != dec ? 0x0f0f0f0fu : 0xf0f0f0f0u;
        sel2 = !(lane & 2) ? 0x06020400u : 0x03070105u;        // [x0,y0,x2,y2] | [y1,x1,y3,x3]
        sel4 = !(lane & 4) ? 0x05040100u : 0x03020706u;        // [x0,x1,y0,y1] | [y2,y3,x2,x3]
    }
};
// Exchanges inside the word: bit 0 (1) of the byte's number with bit 0 (1) of the bit's number.
__device__ __forceinline__ uint32_t swap_bits1(uint32_t x) {
    const uint32_t t = (x ^ (x >> 7)) & 0x00AA00AAu;
    return x ^ t ^ (t << 7);
}
__device__ __forceinline__ uint32_t swap_bits2(uint32_t x) {
    const uint32_t t = (x ^ (x >> 14)) & 0x0000CCCCu;
    return x ^ t ^ (t << 14);
}
// N slices at a time, so that the cross-lane reads of a stage are in flight together.
template <int N>
__device__ __forceinline__ void to_planes(uint32_t (&x)[N], const PlaneConsts& c) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = swap_bits2(swap_bits1(x[i]));
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = bfi(c.msk, __builtin_amdgcn_alignbit(x[i], x[i], c.rot), dpp<kDppQuadSwap1>(x[i]));
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_perm(dpp<kDppQuadSwap2>(x[i]), x[i], c.sel2);
    uint32_t t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = swizzle_xor<4>(x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_perm(t[i], x[i], c.sel4);
}
template <int N>
__device__ __forceinline__ void from_planes(uint32_t (&x)[N], const PlaneConsts& c) {
    uint32_t t[N];
#pragma unroll
    for (int i = 0; i < N; ++i) t[i] = swizzle_xor<4>(x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_perm(t[i], x[i], c.sel4);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = __builtin_amdgcn_perm(dpp<kDppQuadSwap2>(x[i]), x[i], c.sel2);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = bfi(c.msk, __builtin_amdgcn_alignbit(x[i], x[i], c.rot), dpp<kDppQuadSwap1>(x[i]));
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = swap_bits1(swap_bits2(x[i]));
}

// Four elements' residuals as byte slices of sign | magnitude: NS slices hold
// 8 NS - 1 magnitude bits and, in the top bit of the last slice, the sign.
template <int NS>
__device__ __forceinline__ void slices_of(const uint32_t (&d)[4], uint32_t (&w)[NS]) {
    static_assert(NS == 1 || NS == 2 || NS == 4, "7, 15 or 31 magnitude bits");
    if constexpr (NS == 4) {
        uint32_t x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int32_t v = (int32_t)d[i], n = (int32_t)(0u - d[i]);
            x[i] = bfi(0x80000000u, d[i], (uint32_t)(v > n ? v : n));
        }
        const uint32_t a = __builtin_amdgcn_perm(x[2], x[3], 0x05010400u), b = __builtin_amdgcn_perm(x[2], x[3], 0x07030602u);
        const uint32_t e = __builtin_amdgcn_perm(x[0], x[1], 0x05010400u), f = __builtin_amdgcn_perm(x[0], x[1], 0x07030602u);
        w[0] = __builtin_amdgcn_perm(e, a, 0x05040100u);
        w[1] = __builtin_amdgcn_perm(e, a, 0x07060302u);
        w[2] = __builtin_amdgcn_perm(f, b, 0x05040100u);
        w[3] = __builtin_amdgcn_perm(f, b, 0x07060302u);
    } else {
        const uint32_t p01 = __builtin_amdgcn_perm(d[1], d[0], 0x05040100u);    // low halves
        const uint32_t p23 = __builtin_amdgcn_perm(d[3], d[2], 0x05040100u);
        if constexpr (NS == 1) {
            const uint32_t v = __builtin_amdgcn_perm(p01, p23, 0x04060002u);    // low bytes, element 3 first
            const uint32_t m = __builtin_amdgcn_perm(p01, p23, 0x0a0b0809u);    // their signs: 0xff or 0
            const uint32_t a = (v ^ m) + (m & 0x01010101u);                     // |d|: no byte carries (|d| <= 127)
            w[0] = bfi(0x80808080u, m, a);
        } else {
            typedef short s2 __attribute__((ext_vector_type(2)));
            uint32_t x[2] = {p01, p23};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                s2 v, n, a;
                __builtin_memcpy(&v, &x[i], 4);
                n = (s2)0 - v;
                a = __builtin_elementwise_max(v, n);
                uint32_t u;
                __builtin_memcpy(&u, &a, 4);
                x[i] = bfi(0x80008000u, x[i], u);
            }
            w[0] = __builtin_amdgcn_perm(x[0], x[1], 0x04060002u);
            w[1] = __builtin_amdgcn_perm(x[0], x[1], 0x05070103u);
        }
    }
}

// Dot products of four signed bytes (two halves) with a constant, plus an
// accumulator: sums of neighbouring residuals in one operation.
__device__ __forceinline__ uint32_t dot4(uint32_t v, uint32_t m, uint32_t acc) {
    return (uint32_t)__builtin_amdgcn_sdot4((int)v, (int)m, (int)acc, false);
}
__device__ __forceinline__ uint32_t dot2(uint32_t v, uint32_t m, uint32_t acc) {
    typedef short s2 __attribute__((ext_vector_type(2)));
    s2 a, b;
    __builtin_memcpy(&a, &v, 4);
    __builtin_memcpy(&b, &m, 4);
    return (uint32_t)__builtin_amdgcn_sdot2(a, b, (int)acc, false);
}

// A quad's residuals as they come back from NS slices: signed bytes (element
// 3 - j in byte j), signed halves ([0]: elements 1, 0; [1]: elements 3, 2, the
// later one low) or words (element i in [i]).
template <int NS>
struct Residuals {
    static constexpr int N = NS == 1 ? 1 : (NS == 2 ? 2 : 4);
    uint32_t v[N];
    // w: slices of sign | magnitude. A sign without a magnitude (element 0 of
    // an outlier-selected block) counts as 0. s0: element 0's sign, 0 or ~0.
    __device__ __forceinline__ void from_slices(const uint32_t (&w)[NS], uint32_t& s0) {
        if constexpr (NS == 1) {
            const uint32_t a = w[0] & 0x7f7f7f7fu;
            const uint32_t s = (a + 0x7f7f7f7fu) & w[0] & 0x80808080u;   // negative and not 0
            const uint32_t t = s >> 7;
            v[0] = (a ^ ((s << 1) - t)) + t;
            s0 = (uint32_t)((int32_t)w[0] >> 31);
        } else if constexpr (NS == 2) {
            typedef short s2 __attribute__((ext_vector_type(2)));
            const uint32_t x[2] = {__builtin_amdgcn_perm(w[1], w[0], 0x07030602u), __builtin_amdgcn_perm(w[1], w[0], 0x05010400u)};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t a = x[i] & 0x7fff7fffu;
                s2 h, m, y;
                __builtin_memcpy(&h, &x[i], 4);
                m = h >> 15;
                uint32_t mu;
                __builtin_memcpy(&mu, &m, 4);
                const uint32_t z = a ^ mu;
                __builtin_memcpy(&y, &z, 4);
                y = y - m;
                __builtin_memcpy(&v[i], &y, 4);
            }
            s0 = (uint32_t)((int32_t)x[0] >> 31);
        } else {
            const uint32_t e = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u), a = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u);
            const uint32_t f = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u), b = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u);
            const uint32_t x[4] = {__builtin_amdgcn_perm(f, e, 0x07060302u), __builtin_amdgcn_perm(f, e, 0x05040100u),
                                   __builtin_amdgcn_perm(b, a, 0x07060302u), __builtin_amdgcn_perm(b, a, 0x05040100u)};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t m = (uint32_t)((int32_t)x[i] >> 31);
                v[i] = ((x[i] & 0x7fffffffu) ^ m) - m;
            }
            s0 = (uint32_t)((int32_t)x[0] >> 31);
        }
    }
    // element I by itself
    template <int I>
    __device__ __forceinline__ uint32_t at() const {
        if constexpr (NS == 1) return (uint32_t)(((int32_t)(v[0] << (8 * I))) >> 24);
        else if constexpr (NS == 2) return (uint32_t)(((int32_t)(v[I / 2] << (16 * (I % 2)))) >> 16);
        else return v[I];
    }
    // acc plus the elements of MASK (bit i: element i)
    template <int MASK>
    __device__ __forceinline__ uint32_t sum(uint32_t acc) const {
        if constexpr (NS == 1) {
            constexpr uint32_t m = ((MASK & 1) ? 0x01000000u : 0) | ((MASK & 2) ? 0x010000u : 0) | ((MASK & 4) ? 0x0100u : 0) |
                                   ((MASK & 8) ? 1u : 0);
            return dot4(v[0], m, acc);
        } else if constexpr (NS == 2) {
            constexpr uint32_t m01 = ((MASK & 1) ? 0x10000u : 0) | ((MASK & 2) ? 1u : 0);
            constexpr uint32_t m23 = ((MASK & 4) ? 0x10000u : 0) | ((MASK & 8) ? 1u : 0);
            if constexpr (m01 != 0) acc = dot2(v[0], m01, acc);
            if constexpr (m23 != 0) acc = dot2(v[1], m23, acc);
            return acc;
        } else {
            if constexpr (MASK & 1) acc += v[0];
            if constexpr (MASK & 2) acc += v[1];
            if constexpr (MASK & 4) acc += v[2];
            if constexpr (MASK & 8) acc += v[3];
            return acc;
        }
    }
    // acc plus element 0 in lanes where `on` is ~0
    __device__ __forceinline__ uint32_t first(uint32_t on, uint32_t acc) const {
        if constexpr (NS == 1) return dot4(v[0], on & 0x01000000u, acc);
        else if constexpr (NS == 2) return dot2(v[0], on & 0x10000u, acc);
        else return acc + (v[0] & on);
    }
};

// Inclusive prefix sums (wrapping u32).
__device__ __forceinline__ uint32_t scan_row16(uint32_t v) {
    v += dpp<kDppRowShr1>(v);
    v += dpp<kDppRowShr2>(v);
    v += dpp<kDppRowShr4>(v);
    v += dpp<kDppRowShr8>(v);
    return v;
}
__device__ __forceinline__ uint32_t scan_seg32(uint32_t v) {
    v = scan_row16(v);
    v += dpp<kDppBcast15, 0xa>(v);
    return v;
}
__device__ __forceinline__ uint32_t scan_wave(uint32_t v) {
    v = scan_seg32(v);
    v += dpp<kDppBcast31, 0xc>(v);
    return v;
}

__device__ __forceinline__ uint32_t bitlen(uint32_t v) { return 32u - (uint32_t)__builtin_clzg(v, 32); }
// Hides a lane constant's origin: the compiler otherwise turns its uses into
// compares and selects of their own.
__device__ __forceinline__ void opaque(uint32_t& v) { asm("" : "+v"(v)); }
// The same for a value that is to be computed where it is used, not once
// before a loop in a register of its own.
__device__ __forceinline__ void opaque_here(uint32_t& v) { asm volatile("" : "+v"(v)); }

// ---------------------------------------------------------------------------
// quantisation: t = RN(x*r); s = (t >= -0.5 ? 0 : 1); q = sat_trunc(RN(t+0.5)) - s
// (src/cuSZp_kernels_1D_f32.cu:3-20, src/cuSZp_kernels_1D_f64.cu:3-8).
// The kernels are built with -ffp-contract=off so mul and add round separately;
// v_cvt_i32_f{32,64} truncates, saturates and maps NaN to 0 like cvt.rzi.s32.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int32_t cvt_i32_sat(float y) {
    int32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(y));
    return r;
}
__device__ __forceinline__ int32_t cvt_i32_sat(double y) {
    int32_t r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(y));
    return r;
}
template <class T>
__device__ __forceinline__ uint32_t quantize(T x, T r) {
    const T t = x * r;
    const uint32_t s = (t >= T(-0.5)) ? 0u : 1u;
    const T y = t + T(0.5);
    return (uint32_t)cvt_i32_sat(y) - s;
}

// ---------------------------------------------------------------------------
// block-byte bookkeeping (decoder view of a header byte; cuSZp's decoders
// src/cuSZp_kernels_1D_f32.cu:1705-1711 for outlier, :837-843 otherwise)
// ---------------------------------------------------------------------------
struct BlockView {
    uint32_t sel, nb, R, size, head;
};
template <int MODE, int S>
__device__ __forceinline__ BlockView view_of(uint32_t byte) {
    BlockView v;
    if constexpr (MODE == kOutlier) {
        v.sel = byte >> 7;
        v.nb = ((byte >> 5) & 3) + 1;
        v.R = byte & 0x1f;
        v.size = v.sel ? S + S * v.R + v.nb : (v.R ? S + S * v.R : 0);
        v.head = v.sel ? v.nb : 0;
    } else {
        v.sel = 0;
        v.nb = 0;
        v.R = byte;
        v.size = v.R ? S + S * v.R : 0;
        v.head = 0;
    }
    return v;
}

// Header byte of a block from its rate over all elements (fr1), over elements
// e >= 1 (fr2) and the bit length of element 0's magnitude (outlier mode).
// src/cuSZp_kernels_1D_f32.cu:1165-1183 (outlier), :641 (fixed/plain).
template <int MODE, int S>
__device__ __forceinline__ uint32_t rate_byte(uint32_t fr1, uint32_t fr2, uint32_t o_bits) {
    if constexpr (MODE != kOutlier) {
        return fr1;
    } else {
        const uint32_t nb = (o_bits + 7) / 8;
        const uint32_t ofs1 = fr1 ? S + fr1 * S : 0;
        const uint32_t ofs2 = fr2 ? S + fr2 * S + nb : S + nb;
        return (ofs1 <= ofs2) ? fr1 : ((fr2 | 0x80u | ((nb - 1) << 5)) & 0xffu);
    }
}

// The outlier header byte and its decoder view in one step, for fr1, fr2 <= 31
// (no block of 32 planes). There view_of(rate_byte(fr1, fr2, o_bits)) is the
// encoder's own choice: a selected block has an element-0 residual, so nb is
// 1..4 and the byte's fields [4:0] = fr2, [6:5] = nb - 1 decode back exactly;
// an unselected byte fr1 <= 31 decodes to R = fr1 and size ofs1.
template <int S>
__device__ __forceinline__ BlockView outlier_code(uint32_t fr1, uint32_t fr2, uint32_t o_bits, uint32_t& byte) {
    const uint32_t nb = (o_bits + 7) >> 3;
    const uint32_t ofs1 = fr1 ? S + fr1 * S : 0;
    const uint32_t ofs2 = S + fr2 * S + nb;
    const bool sel = ofs1 > ofs2;
    byte = sel ? (fr2 | 0x80u | ((nb - 1) << 5)) : fr1;
    BlockView v;
    v.sel = sel;
    v.nb = nb;
    v.R = sel ? fr2 : fr1;
    v.size = sel ? ofs2 : ofs1;
    v.head = sel ? nb : 0;
    return v;
}

// LDS byte pointers and unaligned LDS words (gfx950 accesses LDS unaligned).
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(3))) uint32_t __attribute__((aligned(1))) lds_u32u;
__device__ __forceinline__ void store_u32u(uint8_t* p, uint32_t v) {
    typedef uint32_t __attribute__((aligned(1))) u32u;
    *(u32u*)p = v;
}

// ---------------------------------------------------------------------------
// decoupled lookback (single pass, wave-parallel, segmented, stealing)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t ld_status(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_status(unsigned long long* p, uint64_t v) {
    __hip_atomic_store(p, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t cas_status(unsigned long long* p, uint64_t expect, uint64_t desired) {
    unsigned long long e = expect;
    __hip_atomic_compare_exchange_strong(p, &e, (unsigned long long)desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return e;   // value seen (== expect on success)
}
__device__ __forceinline__ uint64_t rdlane64(uint64_t v, uint32_t l) {
    return (uint64_t)rdlane((uint32_t)v, l) | ((uint64_t)rdlane((uint32_t)(v >> 32), l) << 32);
}

// Sum over the wave of per-lane values below 2^40: two 20-bit halves are
// reduced with DPP adds (no LDS round trips) and recombined.
__device__ __forceinline__ uint64_t wave_sum_u40(uint64_t v) {
    const uint32_t lo = scan_wave((uint32_t)v & 0xfffffu);
    const uint32_t hi = scan_wave((uint32_t)(v >> 20));
    return (uint64_t)rdlane(lo, kWaveSize - 1) + ((uint64_t)rdlane(hi, kWaveSize - 1) << 20);
}

__device__ __forceinline__ bool status_ready(uint64_t w, uint64_t tag) {
    const uint64_t f = w & kFlagMask;
    return ((w & kTagMask) == tag) && f != 0 && f != kFlagClaim;
}

// Exclusive prefix of `tile` within its segment (tiles first .. tile-1), run by
// one whole wave (no workgroup barriers inside).
//
// The wave publishes the tile's aggregate (the segment's first tile publishes
// its inclusive prefix and returns 0), then reads predecessors a window of
// 64 * K at a time: lane j, word k reads position p = 64k + j, i.e. tile
// tile - 1 - p (the K loads of a window are issued back to back: one round
// trip). A window is resolved once every position up to the nearest published
// inclusive prefix P is ready; the values at positions <= P sum to the
// exclusive prefix (with no prefix in the window, the window's sum carries
// into the next one). The wave then publishes the tile's inclusive prefix.
// Positions before the segment read words of an earlier segment or of the
// guard in front of the status array (kStatusGuard words) and count as an
// inclusive prefix of 0.
//
// Tiles are numbered in launch order, so a predecessor normally belongs to a
// workgroup that started earlier. Forward progress does not depend on that:
// when a window stays unresolved for sc.steal_ticks (kStealTicks unless a test
// lowers it), the wave claims the farthest
// pending predecessor of the window (CAS from the word it saw to CLAIM),
// computes that tile's aggregate with agg_of(tile) and publishes it. A claim is
// held only by a running wave that computes without waiting, so every wait
// ends; the owner's later store of the same aggregate (or of its inclusive
// prefix) is harmless.
//
// pre (with has_pre): the window's first read, issued earlier by the caller
// with lookback_window(); its words may be stale (pending ones are read again).
template <int K>
struct LookbackWindow {
    uint64_t w[K];
};
template <int K>
__device__ __forceinline__ LookbackWindow<K> lookback_window(const ScanCtx& sc, uint64_t tile, int lane) {
    LookbackWindow<K> pw;
    const unsigned long long* const wp = sc.status + ((int64_t)tile - 1 - lane);
#pragma unroll
    for (int k = 0; k < K; ++k) pw.w[k] = ld_status(wp - 64 * k);
    return pw;
}
template <int K, class AggF>
__device__ __forceinline__ uint64_t wave_lookback(const ScanCtx& sc, uint64_t tile, uint64_t first, uint64_t agg,
                                                  int lane, AggF&& agg_of, const LookbackWindow<K> pre = {},
                                                  bool has_pre = false) {
    constexpr int WIN = 64 * K;
    const uint64_t tag = sc.tag;
    if (sc.hold_every && tile % sc.hold_every == sc.hold_every - 1) {
        // scan stress (tests): this tile publishes late, so its successors
        // claim it and compute its aggregate themselves; the wait is bounded
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        while (__builtin_amdgcn_s_memrealtime() - t0 < sc.hold_ticks) __builtin_amdgcn_s_sleep(8);
    }
    if (tile == first) {
        if (lane == 0) st_status(sc.status + tile, tag | kFlagPrefix | agg);
        return 0;
    }
    if (lane == 0) st_status(sc.status + tile, tag | kFlagAgg | agg);
    uint64_t excl = 0;
    int64_t hi = (int64_t)tile;
    uint32_t spins = 0;
    const uint64_t t_wait = __builtin_amdgcn_s_memrealtime();
    bool stalled = false;
    int64_t claimed = -1;   // a predecessor this wave claimed and must compute
    for (;;) {
        if (claimed >= 0) {   // computed with no window words live; the window is then re-read
            const uint64_t a = agg_of((uint64_t)claimed);
            if (lane == 0) {
                cas_status(sc.status + claimed, tag | kFlagClaim, tag | kFlagAgg | a);
                raise_bit(sc.err, kInfoStolen, sc.mark);
                if (sc.stats) atomicAdd(sc.diag + 6, 1ull);
            }
            claimed = -1;
        }
        const unsigned long long* const wp = sc.status + (hi - 1 - lane);   // position 64k + lane: wp - 64k
        const int64_t rel = hi - 1 - lane - (int64_t)first;                 // before the segment iff rel < 64k
        uint64_t w[K];
        if (has_pre) {   // the first window, read before (only once: a claim re-reads)
#pragma unroll
            for (int k = 0; k < K; ++k) w[k] = pre.w[k];
            has_pre = false;
        } else {
#pragma unroll
            for (int k = 0; k < K; ++k) w[k] = ld_status(wp - 64 * k);
        }
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (rel < 64 * k) w[k] = tag | kFlagPrefix;
        int P;
        for (;;) {
            P = WIN;
            int N = WIN;
            uint64_t nr[K];
#pragma unroll
            for (int k = K - 1; k >= 0; --k) {
                const bool rd = status_ready(w[k], tag);
                const uint64_t pm = ballot(rd && (w[k] & kFlagMask) == kFlagPrefix);
                if (pm) P = 64 * k + __builtin_ctzll(pm);
                nr[k] = ballot(!rd);
                if (nr[k]) N = 64 * k + __builtin_ctzll(nr[k]);
            }
            if (N > P || N == WIN) break;   // every position up to P is ready
            ++spins;
            // farthest pending position at or below P: (sk, sl)
            int sk = 0, sl = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int lo = 64 * k;
                const uint64_t m = P < lo ? 0ull : (P < lo + 63 ? nr[k] & ((2ull << (P - lo)) - 1) : nr[k]);
                if (m) { sk = k; sl = 63 - __builtin_clzll(m); }
            }
            uint64_t pend = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) if (k == sk) pend = rdlane64(w[k], sl);
            const int64_t pidx = hi - 1 - (64 * sk + sl);
            if (spins >= kSpinLimit ||
                ((spins & 1023) == 0 &&
                 (__hip_atomic_load(sc.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kErrStall))) {
                // last-resort watchdog: record the stuck predecessor and give up
                // (the output is reported invalid; publishing below unblocks successors)
                stalled = true;
                if (lane == 0) {
                    raise_bit(sc.err, kErrStall, sc.mark);
                    if (atomicCAS(sc.diag, 0ull, tile + 1) == 0ull) {
                        sc.diag[1] = (uint64_t)pidx;
                        sc.diag[2] = pend;
                    }
                }
                break;
            }
            if (__builtin_amdgcn_s_memrealtime() - t_wait > sc.steal_ticks &&
                !(((pend & kTagMask) == tag) && ((pend & kFlagMask) == kFlagClaim))) {
                uint64_t seen = 0;
                if (lane == 0) seen = cas_status(sc.status + pidx, pend, tag | kFlagClaim);
                if (rdlane64(seen, 0) == pend) {
                    claimed = pidx;
                    break;
                }
            }
            __builtin_amdgcn_s_sleep(1);
            // re-read the pending words (all loads first; a ready word stays ready)
#pragma unroll
            for (int k = 0; k < K; ++k)
                if ((nr[k] >> lane) & 1) w[k] = ld_status(wp - 64 * k);
        }
        if (claimed >= 0) continue;
        uint64_t part = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) part += (64 * k + lane <= P) ? (w[k] & kValueMask) : 0;
        excl += wave_sum_u40(part);
        if (P < WIN || stalled) break;
        hi -= WIN;
    }
    if (lane == 0) {
        st_status(sc.status + tile, tag | kFlagPrefix | (excl + agg));
        if (sc.stats && spins) {
            atomicAdd(sc.diag + 4, (unsigned long long)spins);
            atomicAdd(sc.diag + 5, 1ull);
            atomicAdd(sc.diag + 7, (unsigned long long)(__builtin_amdgcn_s_memrealtime() - t_wait));
        }
    }
    return excl;
}

// wave_lookback with a window of 128 (2) or 256 (4 words per lane) predecessors.
template <class AggF>
__device__ __forceinline__ uint64_t lookback(const ScanCtx& sc, uint64_t tile, uint64_t first, uint64_t agg, int lane,
                                             int window, AggF&& agg_of) {
    return window == 2 ? wave_lookback<2>(sc, tile, first, agg, lane, agg_of)
                       : wave_lookback<4>(sc, tile, first, agg, lane, agg_of);
}

// ---------------------------------------------------------------------------
// Block walking for 2D/3D: wave-uniform block coordinates advanced by +1 block.
// Block order: b = z*By*Bx + by*Bx + bx (src/cuSZp_kernels_2D_f32.cu:69-73).
// ---------------------------------------------------------------------------
struct Walker {
    uint64_t b;
    uint32_t bx, by, bz;
    __device__ __forceinline__ void init(uint64_t b0, const Geom& g) {
        b = b0;
        const uint64_t t = b0 / g.Bx;
        bx = (uint32_t)(b0 - t * g.Bx);
        by = (uint32_t)(t % g.By);
        bz = (uint32_t)(t / g.By);
    }
    __device__ __forceinline__ void next(const Geom& g) {
        ++b;
        if (++bx == g.Bx) {
            bx = 0;
            if (++by == g.By) { by = 0; ++bz; }
        }
    }
    // advance by n <= Bx blocks (crosses at most one row end)
    __device__ __forceinline__ void step(const Geom& g, uint32_t n) {
        b += n;
        bx += n;
        if (bx >= g.Bx) {
            bx -= g.Bx;
            if (++by == g.By) { by = 0; ++bz; }
        }
    }
};

// Per-lane geometry of an element of a group (natural element order e = lane).
template <int DIM>
struct LaneGeo;

template <>
struct LaneGeo<1> {
    __device__ __forceinline__ void init(int, const Geom&) {}
};
template <>
struct LaneGeo<2> {
    uint32_t r, c;
    uint64_t off;
    __device__ __forceinline__ void init(int e, const Geom& g) {
        r = (uint32_t)e >> 3;
        c = (uint32_t)e & 7;
        off = (uint64_t)r * g.X + c;
    }
};
template <>
struct LaneGeo<3> {
    uint32_t zz, yy, xx;
    uint64_t off;
    __device__ __forceinline__ void init(int e, const Geom& g) {
        zz = (uint32_t)e >> 4;
        yy = ((uint32_t)e >> 2) & 3;
        xx = (uint32_t)e & 3;
        off = (uint64_t)zz * g.XY + (uint64_t)yy * g.X + xx;
    }
};

// Element index and validity of lane `e` of the current group.
template <int DIM>
__device__ __forceinline__ bool elem_of(const Geom& g, const LaneGeo<DIM>& lg, const Walker& wk,
                                        uint64_t grp, int e, uint64_t& idx) {
    if constexpr (DIM == 1) {
        idx = grp * 64 + (uint64_t)e;
        return idx < g.n;
    } else if constexpr (DIM == 2) {
        const uint32_t y = wk.by * 8 + lg.r, x = wk.bx * 8 + lg.c;
        idx = ((uint64_t)wk.bz * g.Y + (uint64_t)wk.by * 8) * g.X + (uint64_t)wk.bx * 8 + lg.off;
        return (wk.b < g.nblocks) & (y < g.Y) & (x < g.X);
    } else {
        const uint32_t z = wk.bz * 4 + lg.zz, y = wk.by * 4 + lg.yy;
        idx = ((uint64_t)wk.bz * 4 * g.Y + (uint64_t)wk.by * 4) * g.X + (uint64_t)wk.bx * 4 + lg.off;
        return (wk.b < g.nblocks) & (z < g.Z) & (y < g.Y);
    }
}

// Element index of the first element of the walker's block (2D/3D).
template <int DIM>
__device__ __forceinline__ uint64_t block_origin(const Geom& g, const Walker& wk) {
    if constexpr (DIM == 2) return ((uint64_t)wk.bz * g.Y + (uint64_t)wk.by * 8) * g.X + (uint64_t)wk.bx * 8;
    else return ((uint64_t)wk.bz * 4 * g.Y + (uint64_t)wk.by * 4) * g.X + (uint64_t)wk.bx * 4;
}

// Predecessor lane of element e in the block's Lorenzo chain (-1: none).
template <int DIM>
__device__ __forceinline__ int pred_lane(int e) {
    if constexpr (DIM == 1) {
        return (e & 31) ? e - 1 : -1;
    } else if constexpr (DIM == 2) {
        return (e & 7) ? e - 1 : ((e >> 3) ? e - 8 : -1);
    } else {
        return (e & 3) ? e - 1 : (((e >> 2) & 3) ? e - 4 : ((e >> 4) ? e - 16 : -1));
    }
}

// ---------------------------------------------------------------------------
// Quads: a lane's four consecutive elements. A chunk is 512 elements, two sets
// of 64 quads; a 1D block is 8 lanes (eight blocks per set), a 2D/3D block a
// DPP row of 16 lanes (four blocks per set; a quad is half a row of an 8x8
// block or a row of a 4x4x4 one). Extents along x are multiples of 4, so a quad
// of a 2D/3D array lies inside the array or outside it as a whole.
// ---------------------------------------------------------------------------
template <int DIM>
struct QuadLane {
    static constexpr int BL = (DIM == 1) ? 8 : 16;   // lanes per block
    static constexpr int SB = 64 / BL;               // blocks per set
    static constexpr int NB = 2 * SB;                // blocks per chunk
    static constexpr int BW = (DIM == 2) ? 8 : 4;    // extent of a 2D/3D block along x (and y)
    uint32_t k;       // lane within its 32-element half
    uint32_t h;       // 2D/3D: which half
    uint32_t blk;     // block within the set
    uint32_t x, y, z; // 2D/3D: the quad's place in its block
    uint32_t e0;      // ~0 in the lane that holds the block's element 0
    uint32_t p1, p2;  // masks of the two candidates for element 0's predecessor (prev_code)
    bool second;      // the lane is in the second half of its block's lanes
    __device__ __forceinline__ void init(int lane) {
        const uint32_t m = (uint32_t)lane % BL;
        k = (uint32_t)lane & 7;
        h = (DIM == 1) ? 0u : m >> 3;
        blk = (uint32_t)lane / BL;
        e0 = m == 0 ? ~0u : 0u;
        if constexpr (DIM == 1) {
            x = y = z = 0;
            p1 = k ? ~0u : 0u;
            p2 = 0;
        } else if constexpr (DIM == 2) {
            x = 4 * (m & 1);
            y = m >> 1;
            z = 0;
            p1 = (m & 1) ? ~0u : 0u;
            p2 = !(m & 1) && m ? ~0u : 0u;
        } else {
            x = 0;
            y = m & 3;
            z = m >> 2;
            p1 = y ? ~0u : 0u;
            p2 = !y && z ? ~0u : 0u;
        }
        second = (lane & (BL / 2)) != 0;
        opaque(e0);
        opaque(p1);
        opaque(p2);
    }
    // Code of the predecessor of the quad's element 0 in the block's Lorenzo
    // chain (0: none): 1D the previous lane's last code; 2D that one, or in
    // column 0 the first code of the row above; 3D the first code of the row
    // before, or in the first row of a slice that of the slice before.
    __device__ __forceinline__ uint32_t prev_code(const uint32_t (&q)[4]) const {
        if constexpr (DIM == 1) return dpp<kDppRowShr1>(q[3]) & p1;
        else if constexpr (DIM == 2) return (dpp<kDppRowShr1>(q[3]) & p1) | (dpp<kDppRowShr2>(q[0]) & p2);
        else return (dpp<kDppRowShr1>(q[0]) & p1) | (dpp<kDppRowShr4>(q[0]) & p2);
    }
    // Both sets' bookkeeping at once: the first half of a block's lanes does it
    // for their block of set 0, the second half for that of set 1. The halves
    // meet in one DPP move (kMeet), which a bank mask confines to either.
    static constexpr int kMeet = (DIM == 1) ? kDppHalfMirror : kDppRowRor8;
    static constexpr int kFirst = (DIM == 1) ? 0x5 : 0x3, kSecond = (DIM == 1) ? 0xa : 0xc;
    // Maxima over the block's lanes of N values per set (0 where absent), in
    // the half that keeps the set's books.
    template <int N>
    __device__ __forceinline__ void block_max(const uint32_t (&v0)[N], const uint32_t (&v1)[N], uint32_t (&r)[N]) const {
        auto mx = [](uint32_t a, uint32_t b) { return a > b ? a : b; };
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = second ? v1[i] : v0[i];
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = mx(r[i], dpp<kMeet, 0xf, kFirst>(v0[i]));
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = mx(r[i], dpp<kMeet, 0xf, kSecond>(v1[i]));
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = mx(r[i], dpp<kDppQuadSwap1>(r[i]));
#pragma unroll
        for (int i = 0; i < N; ++i) r[i] = mx(r[i], dpp<kDppQuadSwap2>(r[i]));
        if constexpr (DIM != 1) {
#pragma unroll
            for (int i = 0; i < N; ++i) r[i] = mx(r[i], dpp<kDppHalfMirror>(r[i]));
        }
    }
    // A value of the books of set 0 (1) in all lanes of the block.
    __device__ __forceinline__ static uint32_t of_set(uint32_t v, int s) {
        return s == 0 ? (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, kMeet, 0xf, kSecond, false)
                      : (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, kMeet, 0xf, kFirst, false);
    }
    // Inclusive sums over the set's blocks of a value that is the same in all lanes of a block.
    __device__ __forceinline__ static uint32_t scan_blocks(uint32_t v) {
        if constexpr (DIM == 1) v += dpp<kDppRowShr8>(v);
        v += dpp<kDppBcast15, 0xa>(v);
        v += dpp<kDppBcast31, 0xc>(v);
        return v;
    }
    // Byte offset of plane p's word of this lane's half in a block's payload
    // after any prefix (the sign word is where plane -1 would be); 2D/3D blocks
    // interleave the halves' words (src/cuSZp_kernels_2D_f32.cu:896-903).
    __device__ __forceinline__ uint32_t plane_offset(uint32_t p) const { return DIM == 1 ? 4 + 4 * p : 8 + 8 * p + 4 * h; }
    // Codes from residuals; r0 is added to element 0 of the block (its
    // magnitude where it travels in the prefix), only in lane e0.
    template <int NS>
    __device__ __forceinline__ void codes(const Residuals<NS>& r, uint32_t r0, uint32_t (&q)[4]) const {
        if constexpr (DIM == 1) {
            const uint32_t t = r.template sum<15>(r0);
            uint32_t s = scan_row16(t);   // two blocks per DPP row: the second starts over
            s -= dpp_newbcast7_hi(s);
            q[0] = r.template sum<1>(s - t + r0);
        } else if constexpr (DIM == 2) {
            // element 0 of a row adds up over the rows, the rest along its row
            const uint32_t col = scan_row16(r.first(~p1, r0));
            q[0] = r.first(p1, col + (dpp<kDppRowShr1>(r.template sum<14>(0u)) & p1));
        } else {
            // element 0 of a slice adds up over the slices, of a row over the slice's rows
            const uint32_t sl = scan_row16(r.first(~p1, r0));
            uint32_t row = r.first(p1, 0u);   // 0 in the slice's first row
            row += dpp<kDppQuadShr1>(row);
            row += dpp<kDppQuadShr2>(row);
            q[0] = sl + row;
        }
        q[1] = r.template sum<2>(q[0]);
        q[2] = r.template sum<4>(q[1]);
        q[3] = r.template sum<8>(q[2]);
    }
    // Lane 7's value of each DPP row in lanes 8..15, 0 in lanes 0..7.
    __device__ __forceinline__ static uint32_t dpp_newbcast7_hi(uint32_t v) { return dpp<kDppRowNewBcast0 + 7, 0xf, 0xc>(v); }
};

// Four consecutive elements, from any element-aligned address.
template <bool NT, class T>
__device__ __forceinline__ void load_quad(const T* p, T (&x)[4]) {
    constexpr int V = 16 / (int)sizeof(T);
    typedef T VT __attribute__((ext_vector_type(V), aligned(sizeof(T))));
#pragma unroll
    for (int i = 0; i < 4 / V; ++i) {
        const VT v = NT ? __builtin_nontemporal_load((const VT*)p + i) : ((const VT*)p)[i];
#pragma unroll
        for (int j = 0; j < V; ++j) x[V * i + j] = v[j];
    }
}
template <bool NT, class T>
__device__ __forceinline__ void store_quad(T* p, const T (&x)[4]) {
    constexpr int V = 16 / (int)sizeof(T);
    typedef T VT __attribute__((ext_vector_type(V), aligned(sizeof(T))));
#pragma unroll
    for (int i = 0; i < 4 / V; ++i) {
        VT v;
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = x[V * i + j];
        if constexpr (NT) __builtin_nontemporal_store(v, (VT*)p + i);
        else ((VT*)p)[i] = v;
    }
}

// Raw buffer resources (gfx9): word 3 of the descriptor, and an offset that is
// always past a resource's range (the range of one wave's payload is < 2^31).
constexpr int kBufferWord3 = 0x00020000;
constexpr uint32_t kAbsent = 0x80000000u;
// How a fast wave's values are loaded and stored: in pieces of 16 bytes per
// lane, such that an instruction covers whole 128-byte lines (loads that do not
// fetch the rest later, nontemporal stores that do not reach 2.3 TB/s instead of
// 6.1). Quads of 1D f32 (1 KiB in a row) and 2D f32 (rows of 128 bytes) are such
// pieces. Four blocks of 3D f32 give rows of 64 bytes only, and a quad of f64 is
// two pieces: there the lanes whose bit 3 is set trade pieces with those whose
// bit 3 is clear (trade_codes on the codes, 32 bits in either type), so that
// one instruction holds the first ones' rows or lines and the other the rest.
// A lane's piece is at a wave-uniform address plus lane_off bytes (Geom::runs
// bounds it): set s's at p + s * kSetOff, its second half (f64) hi_off further;
// of 3D f32 the second piece hi_off further than the first.
template <int DIM, class T>
struct Pieces {
    static constexpr bool kTrade = sizeof(T) == 8 || DIM == 3;
    static constexpr uint64_t kSetOff = (DIM == 1) ? 256 : QuadLane<DIM>::SB * QuadLane<DIM>::BW;
    uint32_t lane_off;   // bytes
    uint64_t hi_off;     // elements
    __device__ __forceinline__ void init(const QuadLane<DIM>& ql, const Geom& g, int lane) {
        const uint32_t b3 = ((uint32_t)lane >> 3) & 1;
        constexpr uint32_t half = sizeof(T) == 8 ? 2 : (uint32_t)kSetOff;
        if constexpr (DIM == 1) {
            lane_off = kTrade ? 4 * (uint32_t)(lane & ~8) + half * b3 : 4 * (uint32_t)lane;
            hi_off = 32;
        } else if constexpr (DIM == 2) {
            lane_off = (kTrade ? ql.y & 3 : ql.y) * g.X + ql.x + ql.blk * 8 + (kTrade ? half * b3 : 0u);
            hi_off = 4 * (uint64_t)g.X;
        } else {
            lane_off = (ql.z & 1) * (uint32_t)g.XY + ql.y * g.X + ql.blk * 4 + half * b3;
            hi_off = 2 * g.XY;
        }
        lane_off *= (uint32_t)sizeof(T);
        opaque(lane_off);
    }
    // Set s's share of a chunk at the wave-uniform p; no memory access and
    // zeros unless `there` (wave-uniform).
    template <bool NT>
    __device__ __forceinline__ void load(const T* p, bool there, int s, T (&x)[4]) const {
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
        constexpr int kAux = NT ? 2 : 0;   // nt
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc((void*)uniform64((uint64_t)p), 0, there ? 0x7fffffff : 0, kBufferWord3);
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off, (uint32_t)((s * kSetOff + j * hi_off) * 8), kAux);
                __builtin_memcpy(&x[2 * j], &v, 16);
            }
        } else {
            const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off, (uint32_t)(s * (kTrade ? hi_off : kSetOff) * 4), kAux);
            __builtin_memcpy(&x[0], &v, 16);
        }
    }
    __device__ __forceinline__ void store(T* p, int s, const T (&x)[4]) const {   // nontemporal
        typedef T V2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const V2 v = {x[2 * j], x[2 * j + 1]};
                __builtin_nontemporal_store(v, (V2*)((char*)(p + s * kSetOff + j * hi_off) + lane_off));
            }
        } else {
            store_quad<true>((T*)((char*)(p + s * (kTrade ? hi_off : kSetOff)) + lane_off), x);
        }
    }
};
// Codes of pieces to codes of quads, and back.
template <int DIM, class T>
__device__ __forceinline__ void trade_codes(uint32_t (&q)[2][4]) {
    auto trade = [](uint32_t& a, uint32_t& b) {   // lanes 8..15 of a row: a from b; lanes 0..7: b from a
        const uint32_t na = (uint32_t)__builtin_amdgcn_update_dpp((int)a, (int)b, kDppRowRor8, 0xf, 0xc, false);
        const uint32_t nb = (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, kDppRowRor8, 0xf, 0x3, false);
        a = na;
        b = nb;
    };
    if constexpr (sizeof(T) == 8) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 2; ++i) trade(q[s][i], q[s][2 + i]);
    } else if constexpr (DIM == 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) trade(q[0][i], q[1][i]);
    }
}

// The quads of the chunks of an array whose extents are not multiples (Geom::near):
// a chunk's 8 blocks follow each other along x, past the end of the row they go
// on in the next one. Most chunks lie inside one row of whole blocks, and every
// lane's place is then the same number of bytes from the chunk's origin. Quads outside the array get an offset past
// every buffer range: loads give zeros, stores do nothing. (Two 64-bit offsets
// per lane and chunk and predicated accesses before: compress kernels of
// 3000 x 1999 x 16 f32 outlier 152 -> 146 us, 600 x 450 x 152 f32 plain 71 -> 69,
// 300 x 450 x 152 f64 outlier 70 -> 64; what is left is arithmetic, and lines that
// two chunks share: 137 us with rows of 3008.)
template <int DIM, class T>
struct RaggedQuads {
    static constexpr uint32_t BW = QuadLane<DIM>::BW, SB = QuadLane<DIM>::SB, kSet = SB * BW * (uint32_t)sizeof(T);
    Walker wk;
    uint64_t end;        // first block that is not the wave's (or the array's): its chunks are not loaded ahead
    uint64_t org;        // the next chunk's origin
    uint32_t lane_off;   // bytes
    __device__ __forceinline__ void init(const Geom& g, const QuadLane<DIM>& ql, uint64_t b0, uint64_t b1) {
        end = b1 < g.nblocks ? b1 : g.nblocks;
        wk.init(b0, g);
        org = block_origin<DIM>(g, wk);
        lane_off = ((DIM == 3 ? ql.z * (uint32_t)g.XY : 0u) + ql.y * g.X + ql.x + ql.blk * BW) * (uint32_t)sizeof(T);
        opaque(lane_off);
    }
    // The next chunk: its origin (elements), its quads' offsets from there (bytes);
    // true if all of them lie inside the array.
    __device__ __forceinline__ bool next(const Geom& g, uint64_t& base, uint32_t (&vo)[2]) {
        base = org;
        vo[0] = lane_off;
        vo[1] = lane_off + kSet;
        auto lane_place = [] {   // made anew where it is needed: nothing of it in registers across the chunk's work
            uint32_t l = __lane_id();
            opaque_here(l);
            QuadLane<DIM> q;
            q.init((int)l);
            return q;
        };
        bool whole = false;
        if (g.Bx < 8) {   // block by block
            const QuadLane<DIM> q = lane_place();
            const uint32_t blk = q.blk, x = q.x, y = q.y, z = q.z;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t o = kAbsent;
#pragma unroll 1
                for (uint32_t i = 0; i < SB; ++i) {
                    bool v = (wk.b < end) & (wk.by * BW + y < g.Y) & (blk == i);
                    if constexpr (DIM == 2) v &= wk.bx * BW + x < g.X;
                    else v &= wk.bz * 4 + z < g.Z;
                    o = v ? (uint32_t)(block_origin<DIM>(g, wk) - base) * (uint32_t)sizeof(T) + lane_off - blk * (BW * (uint32_t)sizeof(T)) : o;
                    wk.next(g);
                }
                vo[s] = o;
            }
            org = block_origin<DIM>(g, wk);
        } else {   // blocks of two rows at most; selects, no branches: the wave's registers stay scalar
            whole = ((wk.bx + 8) * BW <= g.X) & ((wk.by + 1) * BW <= g.Y) & (DIM == 2 || (wk.bz + 1) * 4 <= g.Z) &
                    (wk.b + 8 <= end);
            const uint32_t left = g.Bx - wk.bx;   // blocks of the chunk in its first row
            const bool last_row = wk.by + 1 == g.By;
            Walker w1 = wk;                       // the row after it
            w1.bx = 0;
            w1.by = last_row ? 0u : wk.by + 1;
            w1.bz = wk.bz + (last_row ? 1u : 0u);
            const uint64_t o1 = block_origin<DIM>(g, w1);
            if (!whole) {
                const QuadLane<DIM> q = lane_place();
                const uint32_t blk = q.blk, x = q.x, y = q.y, z = q.z;
                const uint32_t jump = (uint32_t)(o1 - org - (uint64_t)left * BW) * (uint32_t)sizeof(T);
                const uint32_t y0 = g.Y - wk.by * BW, y1 = g.Y - w1.by * BW;
                const uint32_t z0 = g.Z - wk.bz * 4, z1 = g.Z - w1.bz * 4;   // 3D
                const uint64_t nb = wk.b < end ? end - wk.b : 0;
                const uint32_t blocks = nb < 8 ? (uint32_t)nb : 8u;
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const uint32_t i = blk + s * SB;
                    const bool in0 = i < left;
                    bool v = (i < blocks) & (y < (in0 ? y0 : y1));
                    if constexpr (DIM == 2) v &= (in0 ? wk.bx + i : i - left) * BW + x < g.X;
                    else v &= z < (in0 ? z0 : z1);
                    vo[s] = v ? vo[s] + (in0 ? 0u : jump) : kAbsent;
                }
            }
            const bool on = left > 8;   // the next chunk starts in the same row
            org = on ? org + 8 * BW : o1 + (uint64_t)(8 - left) * BW;
            wk.b += 8;
            wk.bx = on ? wk.bx + 8 : 8 - left;
            wk.by = on ? wk.by : w1.by;
            wk.bz = on ? wk.bz : w1.bz;
        }
        return whole;
    }
    static __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const T* p) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)uniform64((uint64_t)p), 0, 0x7fffffff, kBufferWord3);
    }
    static __device__ __forceinline__ void load(const T* p, uint32_t vo, T (&x)[4]) {
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < (int)sizeof(T) / 4; ++j) {
            const v4u v = __builtin_amdgcn_raw_buffer_load_b128(rsrc(p), vo, 16 * j, 0);
            __builtin_memcpy((char*)&x[0] + 16 * j, &v, 16);
        }
    }
    static __device__ __forceinline__ void store(T* p, uint32_t vo, const T (&x)[4]) {
        typedef uint32_t v4u __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int j = 0; j < (int)sizeof(T) / 4; ++j) {
            v4u v;
            __builtin_memcpy(&v, (const char*)&x[0] + 16 * j, 16);
            __builtin_amdgcn_raw_buffer_store_b128(v, rsrc(p), vo, 16 * j, 0);
        }
    }
};

// Where the quads of a 2D/3D chunk lie, for any extents: 64-bit offsets, blocks
// one by one.
template <int DIM>
struct ChunkQuads {
    uint64_t off[2];   // element offset of set s's quad (0 where outside)
    bool ok[2];        // it lies inside the array
    // The quads of the chunk at wk, which moves on to the next chunk.
    __device__ __forceinline__ void locate(const Geom& g, const QuadLane<DIM>& ql, Walker& wk) {
        constexpr uint32_t BW = QuadLane<DIM>::BW, SB = QuadLane<DIM>::SB;
        uint32_t blk = ql.blk, x = ql.x, y = ql.y, z = ql.z;
        opaque_here(blk);   // nothing of this in registers across the chunk's work
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            ok[s] = false;
            off[s] = 0;
#pragma unroll 1
            for (uint32_t i = 0; i < SB; ++i) {
                bool v = (wk.b < g.nblocks) & (wk.by * BW + y < g.Y);
                if constexpr (DIM == 2) v &= wk.bx * BW + x < g.X;
                else v &= wk.bz * 4 + z < g.Z;
                const uint64_t o = block_origin<DIM>(g, wk);
                ok[s] = blk == i ? v : ok[s];
                off[s] = blk == i ? o : off[s];
                wk.next(g);
            }
        }
        const uint64_t lane_off = (uint64_t)z * g.XY + (uint64_t)y * g.X + x;
#pragma unroll
        for (int s = 0; s < 2; ++s) off[s] = ok[s] ? off[s] + lane_off : 0;
    }
};

// The arrays of a batched launch: descriptors in device memory, ordered by
// tile0; a tile belongs to the last array whose tile0 is not above it.
struct ItemTable {
    const Item* items;
    uint32_t count;
    // last item whose first tile (or segment: FIRST) is not past `tile`
    template <uint64_t Item::*FIRST = &Item::tile0>
    __device__ __forceinline__ uint32_t locate(uint64_t tile) const {
        uint32_t lo = 0, hi = count;   // answer in [lo, hi)
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (items[mid].*FIRST <= tile) lo = mid;
            else hi = mid;
        }
        return lo;
    }
    __device__ __forceinline__ Item get(uint32_t i) const { return items[i]; }
    __device__ __forceinline__ uint32_t variant(uint32_t i) const { return items[i].variant; }
};

// ---------------------------------------------------------------------------
// Aggregates recomputed by a waiting wave (see wave_lookback).
// ---------------------------------------------------------------------------
// OR of v over each 32-lane half (every lane of the half gets the result).
__device__ __forceinline__ uint32_t or_half(uint32_t v) {
    v |= swizzle_xor<16>(v);
    v |= swizzle_xor<8>(v);
    v |= swizzle_xor<4>(v);
    v |= swizzle_xor<2>(v);
    v |= swizzle_xor<1>(v);
    return v;
}

// Payload bytes of local tile `lt` of a compress item, by one wave. Same block
// sizes as pass 1 of compress_tile: a block's rate is the bit length of the OR of
// its magnitudes (the highest non-zero plane), 1D ranks |-2^31| as 0.
template <int DIM, int MODE, class T, int WAVES>
__device__ uint64_t compress_tile_bytes(const T* __restrict__ in, const Geom& geo, T r, uint64_t lt, int lane) {
    const int G = (int)geo.kc * (kChunkElems / 64);   // groups per wave
    constexpr int S = (DIM == 1) ? 4 : 8;
    LaneGeo<DIM> lg;
    lg.init(lane, geo);
    const int pl = pred_lane<DIM>(lane);
    const int pl_src = pl < 0 ? lane : pl;
    const bool e0 = (DIM == 1) ? ((lane & 31) == 0) : (lane == 0);
    const uint64_t g0 = lt * WAVES * G;
    Walker wk;
    if constexpr (DIM != 1) wk.init(g0, geo);
    uint64_t sum = 0;
    for (int i = 0; i < WAVES * G; ++i) {
        uint64_t idx;
        const bool valid = elem_of<DIM>(geo, lg, wk, g0 + i, lane, idx);
        const T x = valid ? in[idx] : T(0);
        const uint32_t q = quantize<T>(x, r);
        uint32_t d;
        if constexpr (MODE == kFixed) {
            d = q;
        } else if constexpr (DIM == 1) {
            uint32_t qp = dpp<kDppWaveShr1>(q);
            qp = (lane & 31) ? qp : 0u;
            d = q - qp;
        } else {
            uint32_t qp = (uint32_t)__builtin_amdgcn_ds_bpermute(pl_src << 2, (int)q);
            qp = (pl >= 0) ? qp : 0u;
            d = q - qp;
        }
        d = valid ? d : 0u;
        const uint32_t a = ((int32_t)d < 0) ? 0u - d : d;
        const uint32_t a1 = (DIM == 1) ? (a & 0x7fffffffu) : a;
        const uint32_t o1 = or_half(a1);
        const uint32_t o2 = (MODE == kOutlier) ? or_half(e0 ? 0u : a1) : 0u;
        if constexpr (DIM == 1) {
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const uint32_t byte = rate_byte<MODE, S>(bitlen(rdlane(o1, 32 * hh)), bitlen(rdlane(o2, 32 * hh)),
                                                         bitlen(rdlane(a, 32 * hh)));
                sum += view_of<MODE, S>(byte).size;
            }
        } else {
            const uint32_t byte = rate_byte<MODE, S>(bitlen(rdlane(o1, 0) | rdlane(o1, 32)),
                                                     bitlen(rdlane(o2, 0) | rdlane(o2, 32)), bitlen(rdlane(a, 0)));
            sum += view_of<MODE, S>(byte).size;
            wk.next(geo);
        }
    }
    return sum;
}

// Payload bytes that header bytes describe, four at a time: sums over the bytes
// of a word with v_sad_u8, counts of the non-zero ones with v_bcnt.
template <int MODE, int S>
struct HeaderSum {
    uint32_t r = 0, n = 0, p = 0;   // rates, blocks with payload, prefix bytes
    __device__ __forceinline__ void add(uint32_t x) {
        const uint32_t rates = (MODE == kOutlier) ? x & 0x1f1f1f1fu : x;
        r = __builtin_amdgcn_sad_u8(rates, 0u, r);
        // bit 7 of a byte: it is not 0 (outlier: its rate is not 0, or it is a selected block's)
        n += __builtin_popcount((((rates & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x) & 0x80808080u);
        if constexpr (MODE == kOutlier) {
            const uint32_t sel = (x >> 7) & 0x01010101u;
            p = __builtin_amdgcn_sad_u8((x >> 5) & (sel | (sel << 1)), 0u, p) + __builtin_popcount(sel);
        }
    }
    __device__ __forceinline__ uint32_t bytes() const { return S * (r + n) + p; }
};
// This lane's share of the bytes that the first b1 header bytes (a multiple of
// 16) describe; lanes i of n take every n-th 16 bytes.
template <int MODE, int S>
__device__ __forceinline__ uint32_t header_share(const uint8_t* __restrict__ cmp, uint64_t b1, uint32_t i, uint32_t n) {
    typedef uint32_t v4uu __attribute__((ext_vector_type(4), aligned(1)));
    constexpr int U = 4;   // loads in flight
    HeaderSum<MODE, S> h;
    for (uint64_t b = 16 * (uint64_t)i; b < b1; b += 16 * U * (uint64_t)n) {
        v4uu w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t at = b + 16 * u * (uint64_t)n;
            w[u] = *(const v4uu*)(cmp + (at < b1 ? at : b));
            if (at >= b1) w[u] = 0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int k = 0; k < 4; ++k) h.add(w[u][k]);
    }
    return h.bytes();
}

// Lookback window of a tile: 64 * kLookbackWords predecessors per round trip.
constexpr int kLookbackWords = 4;
// Words in front of every status array (window reads before tile 0 land there).
constexpr uint64_t kStatusGuard = 64 * kLookbackWords;

// ---------------------------------------------------------------------------
// Offset table of a single-array decompression: before any block is decoded,
// a pass over the header bytes alone writes the stream offset of every
// decode wave's payload (a "unit": the UB consecutive blocks one wave
// decodes). The decode waves then start from their own offset, with no
// lookback and no workgroup barrier; the header is 1/32 (1D) or 1/64 (2D/3D)
// of the values' bytes, so the pass reads little.
//
// The pass is itself one single-pass decoupled-lookback scan, over segments of
// one workgroup's threads x kPrefixBytes header bytes: thread t of segment s sums
// the block sizes of header bytes [(s * threads + t) * kPrefixBytes, +kPrefixBytes).
// Few bytes per thread: the pass is bound by its latency, not by the read (128
// bytes per thread, one by one, took 12.5 us for the 2 MiB header of 512^3
// values, this 6.5). Small workgroups start and publish sooner, large ones make
// fewer segments to look back over: a header of 32 MiB
// (4 GiB of f32) took 36 us with 256 threads per workgroup, 23 with 1024.
// ---------------------------------------------------------------------------
// Longest header whose sums every workgroup takes by itself (single arrays,
// arrays of a batch). The sums cost the number of tiles times the length, the
// offset pass and its launch 3-4 us: 1D f32 with 128 KiB of header 13.2 against
// 15.8 us, 256 KiB 14.8 against 15.7, 512 KiB 25.6 against 21.5; 1D f64 with
// 128 KiB 11.5 against 13.0, 256 KiB 20.0 either way, 512 KiB 46.6 against 32.3.
constexpr uint64_t kDirectHeader = 256 << 10;
constexpr uint64_t kBatchDirectHeader = 16 << 10;
__host__ __device__ constexpr int prefix_threads(uint64_t header) { return header >= (4ull << 20) ? 1024 : 256; }
constexpr int kPrefixBytes = 32;
__host__ __device__ constexpr uint64_t prefix_seg_bytes(int threads) { return (uint64_t)threads * kPrefixBytes; }

// Payload bytes of the header bytes [b0, b0 + kPrefixBytes); bytes at or past
// `limit` (2D/3D: the block count, so header pad bytes count nothing) are
// blocks without payload.
template <int MODE, int S>
__device__ __forceinline__ uint32_t thread_bytes(const uint8_t* __restrict__ cmp, uint64_t b0, uint64_t limit) {
    typedef uint32_t v4uu __attribute__((ext_vector_type(4), aligned(1)));
    constexpr int V = kPrefixBytes / 16;
    HeaderSum<MODE, S> h;
    if (b0 + kPrefixBytes <= limit) {
        v4uu w[V];
#pragma unroll
        for (int i = 0; i < V; ++i) w[i] = *((const v4uu*)(cmp + b0) + i);
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) h.add(w[i][k]);
    } else {
        for (int i = 0; i < kPrefixBytes / 4; ++i) {
            uint32_t v = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint64_t b = b0 + 4 * i + k;
                v |= (b < limit ? (uint32_t)cmp[b] : 0u) << (8 * k);
            }
            h.add(v);
        }
    }
    return h.bytes();
}

// Payload bytes of segment `seg`, by one wave (a waiting wave's recomputation
// of a predecessor it claimed; see wave_lookback).
template <int MODE, int S, int THREADS>
__device__ uint64_t segment_bytes(const uint8_t* __restrict__ cmp, uint64_t limit, uint64_t seg, int lane) {
    uint64_t sum = 0;
    constexpr uint32_t n = prefix_seg_bytes(THREADS);
    for (uint32_t i = (uint32_t)lane; i < n; i += kWaveSize) {
        const uint64_t b = seg * n + i;
        sum += view_of<MODE, S>(b < limit ? (uint32_t)cmp[b] : 0u).size;
    }
    return wave_sum_u40(sum);
}

// offs[u] = H + payload bytes of units 0 .. u-1, for u < nunits; segment =
// base + blockIdx.x.
template <int MODE, int S, int UB, int THREADS>
__global__ void __launch_bounds__(THREADS)
unit_offsets_kernel(const uint8_t* __restrict__ cmp, const uint64_t limit, const uint64_t H, const uint64_t nunits,
                    unsigned long long* __restrict__ offs, const ScanCtx sc, const uint64_t base) {
    static_assert(UB % kPrefixBytes == 0 && prefix_seg_bytes(THREADS) % UB == 0, "units of whole threads in segments of whole units");
    constexpr int NW = THREADS / kWaveSize;
    __shared__ uint32_t wsum[NW];
    __shared__ uint64_t excl;
    const uint64_t seg = base + blockIdx.x;
    const int t = (int)threadIdx.x, lane = (int)__lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint64_t th = seg * THREADS + (uint64_t)t;
    const uint32_t tot = thread_bytes<MODE, S>(cmp, th * kPrefixBytes, limit);
    const uint32_t incl = scan_wave(tot);   // < 2^32: a segment holds at most 2^15 blocks of <= 2 KiB
    if (lane == kWaveSize - 1) wsum[wave] = incl;
    // wave 0's first lookback read overlaps the other waves' sums
    LookbackWindow<kLookbackWords> pre = {};
    if (wave == 0 && seg != 0) pre = lookback_window<kLookbackWords>(sc, seg, lane);
    __syncthreads();
    uint32_t wex = 0, stot = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        const uint32_t v = wsum[w];
        wex += (w < wave) ? v : 0u;
        stot += v;
    }
    if (wave == 0) {
        const uint64_t e = wave_lookback<kLookbackWords>(sc, seg, 0, stot, lane, [&](uint64_t p) {
            return segment_bytes<MODE, S, THREADS>(cmp, limit, p, lane);
        }, pre, true);
        if (lane == 0) excl = e;
    }
    __syncthreads();
    if (t % (UB / kPrefixBytes) == 0) {   // the unit's first thread
        const uint64_t u = th / (UB / kPrefixBytes);
        if (u < nunits) offs[u] = H + excl + wex + (incl - tot);
    }
}

// The pass for a batch: one wave per segment of kBatchSegBytes header bytes, each
// array's segments a scan of their own; offs[w] for wave w of the launch's tiles.
// Without it the decode tiles looked back themselves, between their header and
// payload reads, and those waits set the pace: 256 arrays of 1 Ki to 16 Mi values,
// 2.2 GB, 694 us a call with tiles looking back, 488 with this pass (20 us of it).
constexpr uint64_t kBatchSegBytes = kWaveSize * kPrefixBytes;
template <int WAVES>
__global__ void __launch_bounds__(kWaveSize)
unit_offsets_batch_kernel(const Item* __restrict__ items, uint32_t nitems,
                          unsigned long long* __restrict__ offs, ScanCtx sc,
                          const unsigned long long* __restrict__ epoch, const uint64_t base) {
    sc.tag = (epoch[0] & kEpochMask) << kEpochShift;
    const ItemTable src{items, nitems};
    const uint64_t seg = base + blockIdx.x;
    const Item cur = src.get(src.locate<&Item::seg0>(seg));
    const int lane = (int)__lane_id();
    const uint8_t* const cmp = (const uint8_t*)cur.src;
    const bool one_d = cur.variant % 9 < 3, outlier = cur.variant % 3 == kOutlier;
    const uint64_t limit = one_d ? cur.geo.H : cur.geo.nblocks;
    auto bytes = [&](uint64_t s) -> uint32_t {   // of this lane's header bytes of segment s
        const uint64_t b0 = (s - cur.seg0) * kBatchSegBytes + (uint64_t)lane * kPrefixBytes;
        if (one_d) return outlier ? thread_bytes<kOutlier, 4>(cmp, b0, limit) : thread_bytes<kPlain, 4>(cmp, b0, limit);
        return outlier ? thread_bytes<kOutlier, 8>(cmp, b0, limit) : thread_bytes<kPlain, 8>(cmp, b0, limit);
    };
    const uint32_t tot = bytes(seg);
    const uint32_t incl = scan_wave(tot);   // < 2^32: a segment holds 2^11 blocks of <= 2 KiB
    const uint64_t e = wave_lookback<kLookbackWords>(sc, seg, cur.seg0, rdlane(incl, kWaveSize - 1), lane,
                                                     [&](uint64_t p) { return wave_sum_u40(bytes(p)); });
    const uint32_t per = cur.geo.kc * (kChunkElems / (one_d ? 32 : 64)) / kPrefixBytes;   // lanes per unit
    const uint64_t th = (seg - cur.seg0) * kWaveSize + (uint64_t)lane;
    if (th % per == 0 && th / per < cur.geo.ntiles * WAVES)
        offs[cur.tile0 * WAVES + th / per] = cur.geo.H + e + (incl - tot);
}

// ---------------------------------------------------------------------------
// one tile per workgroup pass
// ---------------------------------------------------------------------------

// Compressed bytes a compress wave stages in LDS. A wave's chunks past that
// (compression ratio below about 2.7 on its share of the tile) run twice.
constexpr uint32_t kStageBytes = 6144;
// Payload bytes of a chunk, at most: 16 blocks of 32 planes in 1D, 8 in 2D/3D.
constexpr uint32_t kMaxChunkBytes = 16 * (4 + 32 * 4 + 4);
static_assert(kMaxChunkBytes >= 8 * (8 + 32 * 8 + 4) && kMaxChunkBytes <= kStageBytes, "a chunk fits the staging area");
// Waves per SIMD the compress kernels are built for (the register budget): three
// 8-wave workgroups of about 49 KB of LDS fit one CU's 160 KB. 8 waves per SIMD
// with 4,960-byte staging areas: 1D the same, 2D/3D 12-30 % slower (64 VGPRs spill).
constexpr int kCompressWavesPerSimd = 6;
// Waves per SIMD the decompress kernels are built for: 8 needs at most 64
// VGPRs and few enough SGPRs for eight waves' scalar files.
constexpr int kDecompressWavesPerSimd = 8;
// Largest chunk payload (from its 4-byte-aligned start) read with dense loads
// into the LDS buffer of a decompress wave.
constexpr int kDenseBytes = 2048;
// The LDS buffer of a decompress wave: the wave's whole payload, read in one
// burst of up to four 16-byte-per-lane loads where it fits; otherwise one
// chunk's payload at a time (kDenseBytes). 4032 bytes keep four 8-wave
// workgroups within a CU's 160 KiB of LDS.
constexpr int kWaveBuf = 4032;
static_assert(kWaveBuf >= kDenseBytes && kWaveBuf % 16 == 0, "wave buffer");

// Shared memory of a compress workgroup.
template <int WAVES>
struct SmemC {
    uint64_t wtot[WAVES];                      // per-wave byte counts
    uint64_t excl;                             // the tile's exclusive prefix (wave 0's lookback)
    uint32_t hdr[WAVES][32];                   // header bytes of the wave's blocks, stored after its chunks
    uint4 stage[WAVES][kStageBytes / 16 + 1];  // the wave's payload, as it will appear in the stream (+ a spare word)
};

// Shared memory of a decompress workgroup.
// Per-block metadata of a decompress wave, in LDS (one 8-byte entry per block
// of the wave, written once by the wave's bookkeeping):
//   a:  byte offset of the block's sign word within the wave's payload (past any
//       outlier prefix)
//   nb: [31:24] 0 for a block without payload (or past the array), else R + 1
//       (33 for 32 planes); [8] outlier-selected; [13:9] bits of the prefix - 1
// A lane carries the word of plane p iff p + 1 < R + 1, the sign word iff
// 0 < R + 1: its key, as lane_key, is below nb whatever nb's low flag bits.
struct DMeta {
    uint32_t a, nb;
    __device__ __forceinline__ uint32_t off() const { return a; }
    __device__ __forceinline__ bool sel() const { return (nb >> 8) & 1; }
    __device__ __forceinline__ uint32_t prefix_bits() const { return ((nb >> 9) & 31) + 1; }   // 8, 16, 24 or 32
    // Payload offset of the lane's word, wo bytes into the block, or kAbsent.
    __device__ __forceinline__ uint32_t word_at(uint32_t keyx, uint32_t wo) const {
        return keyx < nb ? a + wo : kAbsent;
    }
};
template <int MODE>
__device__ __forceinline__ DMeta make_dmeta(uint32_t off, const BlockView& v, bool nz) {
    DMeta m;
    m.a = off + v.head;
    m.nb = nz ? (v.R + 1u) << 24 : 0u;
    if constexpr (MODE == kOutlier) m.nb |= nz ? (v.sel << 8) | ((8 * v.nb - 1) << 9) : 0u;
    return m;
}
__device__ __forceinline__ uint32_t lane_key(uint32_t key) { return (key << 24) | 0xffffffu; }

// Blocks of metadata per decompress wave (its KC * blocks-per-chunk).
constexpr int kMetaPerWave = 128;
template <int WAVES>
struct SmemD {
    uint64_t wtot[WAVES];             // per-wave byte counts
    uint32_t before[WAVES];           // per-wave shares of the payload before the tile
    DMeta meta[WAVES][kMetaPerWave];  // per-block metadata of the wave's blocks
    uint4 payload[WAVES][kWaveBuf / 16];  // stream words, loaded densely and read per lane: the wave's or one chunk's
    uint32_t zero[WAVES][2];          // two zero words per wave (read by lanes without a word)
};

// Chunks (of kc) of a wave at group wgrp0 that end within `end` groups (round: the
// groups by which the last one may go past it).
__device__ __forceinline__ int chunks_of(int kc, uint64_t wgrp0, uint64_t end, uint64_t round) {
    if (wgrp0 >= end) return 0;
    const uint64_t n = (end - wgrp0 + round) / (kChunkElems / 64);
    return n < (uint64_t)kc ? (int)n : kc;
}

// Compresses tile `tile` of array `cur` (every wave of the workgroup calls it).
// Each wave runs its KC chunks of 512 elements in turn, a quad per lane and set:
//   1. loads (16 bytes per lane and instruction for f32; the next chunk's are
//      issued as this chunk's values are quantised);
//   2. quantise, Lorenzo residuals: inside the quad, and one DPP read for its
//      first element. The block's rate is the bit length of its largest
//      residual: minimum and maximum over the quad, then over the block's lanes;
//   3. bookkeeping in every lane for its own block of either set: size, and the
//      offset from one scan of both sets' sizes packed into 16 bits each;
//   4. byte slices (as many as the chunk's largest rate needs), their transpose
//      to plane words, and the words into the wave's LDS staging area exactly
//      as they will appear in the stream.
// The wave totals then combine in LDS, wave 0 runs the lookback (publishing
// the tile's byte count first, then its inclusive prefix), and every wave
// copies its staged payload to the stream with 16-byte stores. Chunks that did
// not fit the wave's staging area any more are only counted at first; once the
// offset is known the wave runs them again, staging and copying by turns.
//
// RUNS: 1D, or 2D/3D with every chunk a run of whole blocks along x
// (Geom::runs), whose place is wave-uniform. Otherwise every quad is located
// by itself.
template <int DIM, int MODE, class T, int WAVES, bool RUNS>
__device__ __forceinline__ void compress_tile(const Item& cur, const uint64_t tile, const ScanCtx& sc,
                                              SmemC<WAVES>& sm, const int window) {
    typedef QuadLane<DIM> QL;
    static_assert(DIM != 1 || RUNS, "1D chunks are runs");
    constexpr int G = kChunkElems / 64;          // groups per chunk
    constexpr int S = (DIM == 1) ? 4 : 8;        // bytes per plane
    constexpr int SB = QL::SB, NB = QL::NB;      // blocks per set, per chunk
    constexpr bool NT = DIM == 1;                // 1D loads stream; 2D/3D quads share lines with the other set

    const int lane = (int)__lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const Geom& geo = cur.geo;
    const int KC = (int)geo.kc;
    const T r = (T)cur.param;
    const uint64_t lt = tile - cur.tile0;
    uint8_t* __restrict__ const dst = (uint8_t*)cur.dst;
    const T* __restrict__ const in = (const T*)cur.src;
    const uint64_t wgrp0 = (lt * WAVES + (uint64_t)wave) * (uint64_t)(KC * G);   // this wave's first group

    QL ql;
    ql.init(lane);
    PlaneConsts pc;
    pc.init(lane, false);
    // LDS addresses of the wave's staging area and of the spare word past it,
    // where lanes without a word write
    lds_u8* const sbase = (lds_u8*)sm.stage[wave];
    const uint32_t s0 = (uint32_t)(size_t)sbase, spare = s0 + kStageBytes;
    // This lane's plane of slice 0, its word's place in a block, and where its
    // block's header byte goes. Ragged chunks leave no registers for them: they are
    // made anew for each chunk (a spilled one's reload would wait for the next
    // chunk's loads, which are issued before).
    constexpr bool kKept = RUNS;
    const uint32_t pl = kKept ? plane_of_lane(ql.k) : 0u, po = kKept ? ql.plane_offset(pl) : 0u;
    lds_u8* const hbase = (lds_u8*)sm.hdr[wave] + (kKept ? ql.blk + (ql.second ? SB : 0) : 0);
    auto fresh = [] {
        uint32_t l = __lane_id();
        opaque_here(l);
        QL q;
        q.init((int)l);
        return q;
    };
    auto plane_word = [&](uint32_t& p, uint32_t& o) {
        const QL q = fresh();
        p = plane_of_lane(q.k);
        o = q.plane_offset(p);
    };

    uint64_t excl = 0, wexcl = 0, ttot = 0;
    uint32_t wave_tot = 0;   // the wave's payload so far, of which `copied` bytes have left the staging area
    uint32_t copied = 0, staged = 0;
    int c_over = KC;         // first chunk that did not fit; `staged` bytes come before it
    bool lossy = false;      // a 2D/3D outlier block got rate byte 32 (see kWarnLossy)

    // Processes chunk c from xv; roll(s) runs right after set s's values are
    // consumed (the next chunk's loads into xv[s] go there). PIECES: xv holds
    // pieces (see Pieces), all inside the array; else quads, all inside the array
    // or (!whole, wave-uniform) those elements whose bits 4s + i of vm are set.
    auto process = [&](auto piecesc, int c, T (&xv)[2][4], const bool whole, const uint32_t vm, auto&& roll) {
        constexpr bool PIECES = decltype(piecesc)::value;
        uint32_t q[2][4], d[2][4];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < 4; ++i) q[s][i] = quantize<T>(xv[s][i], r);   // x = 0 outside the array (q = -1 if r = inf: masked below)
            roll(s);
        }
        if constexpr (PIECES) trade_codes<DIM, T>(q);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            if constexpr (MODE == kFixed) {
#pragma unroll
                for (int i = 0; i < 4; ++i) d[s][i] = q[s][i];
            } else {
                d[s][0] = q[s][0] - ql.prev_code(q[s]);
#pragma unroll
                for (int i = 1; i < 4; ++i) d[s][i] = q[s][i] - q[s][i - 1];
            }
            if (!PIECES && !whole) {   // codes and residuals of padding are 0
#pragma unroll
                for (int i = 0; i < 4; ++i) d[s][i] = ((vm >> (4 * s + i)) & 1) ? d[s][i] : 0u;
            }
        }

        // ---- rates ----------------------------------------------------------
        // [0]: the block's largest magnitude (outlier: of elements e >= 1),
        // [1] (outlier): element 0's
        constexpr int NV = (MODE == kOutlier) ? 2 : 1;
        uint32_t v0[NV], v1[NV], bm[NV];
        auto mx = [](int32_t a, int32_t b) { return a > b ? a : b; };
        auto mn = [](int32_t a, int32_t b) { return a < b ? a : b; };
        auto extremes = [&](const uint32_t (&e)[4], uint32_t (&v)[NV]) {
            const int32_t f0 = (int32_t)(MODE == kOutlier ? e[0] & ~ql.e0 : e[0]);
            const int32_t f1 = (int32_t)e[1], f2 = (int32_t)e[2], f3 = (int32_t)e[3];
            const uint32_t hi = (uint32_t)mx(mx(mx(f0, f1), f2), mx(f3, 0));
            const uint32_t lo = 0u - (uint32_t)mn(mn(mn(f0, f1), f2), mn(f3, 0));
            v[0] = hi > lo ? hi : lo;
            if constexpr (MODE == kOutlier) {
                const uint32_t z = e[0] & ql.e0;
                v[NV - 1] = (uint32_t)mx((int32_t)z, (int32_t)(0u - z));   // 2^31 stays 2^31
            }
        };
        extremes(d[0], v0);
        extremes(d[1], v1);
        ql.template block_max<NV>(v0, v1, bm);
        const uint32_t all = (MODE == kOutlier) ? bm[0] | bm[NV - 1] : bm[0];
        const bool rare = ballot((int32_t)all < 0) != 0;   // a residual of magnitude 2^31 (only from saturated or wrapped codes)
        if (DIM == 1 && rare) {   // 1D ranks |-2^31| as 0 (signed running maximum, src/cuSZp_kernels_1D_f32.cu:552)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t o = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t v = (MODE == kOutlier && i == 0) ? d[s][0] & ~ql.e0 : d[s][i];
                    const uint32_t a = ((int32_t)v < 0 ? 0u - v : v) & 0x7fffffffu;
                    o = o > a ? o : a;
                }
                (s ? v1 : v0)[0] = o;
            }
            ql.template block_max<NV>(v0, v1, bm);
        }

        // ---- the books: planes + 1 (0: no payload), bytes, header byte, prefix bytes
        uint32_t b, sz, hb, nb = 0;
        if constexpr (MODE == kOutlier) {
            const uint32_t a0 = (DIM == 1) ? bm[1] & 0x7fffffffu : bm[1];
            const uint32_t m1 = bm[0] > a0 ? bm[0] : a0;
            BlockView v;
            if (DIM != 1 && rare) {
                hb = rate_byte<MODE, S>(bitlen(m1), bitlen(bm[0]), bitlen(bm[1]));
                v = view_of<MODE, S>(hb);
                // R1 = 32 is kept as the plain byte 32, which every outlier
                // decoder reads as rate 0 (written by
                // src/cuSZp_kernels_2D_f32.cu:1494-1505, masked with 0x1f by the
                // decoder at :2320): the block decodes to zeros, so the call
                // reports it
                lossy |= ballot(hb == 32u) != 0;
            } else {
                v = outlier_code<S>(bitlen(m1), bitlen(bm[0]), bitlen(bm[1]), hb);
            }
            nb = v.head;
            sz = v.size;
            b = (v.sel || v.R) ? v.R + 1 : 0u;
        } else {
            hb = bitlen(bm[0]);
            b = hb + (hb < 1u ? hb : 1u);
            sz = S * b;
        }
        // header bytes go to the stream after the wave's chunks: no global
        // store inside the chunk loop, whose waits for the rolling loads would
        // otherwise also wait for those stores
        if constexpr (kKept) {
            hbase[c * NB] = (uint8_t)hb;
        } else {
            const QL f = fresh();
            hbase[c * NB + f.blk + (f.second ? SB : 0)] = (uint8_t)hb;
        }   // the same from all lanes that keep the block's books
        const uint64_t over7 = ballot(b > 8), over15 = ballot(b > 16);
        const uint32_t info = sz | (b << 16) | (nb << 24);
        const uint32_t inf0 = QL::of_set(info, 0), inf1 = QL::of_set(info, 1);
        // both sets' sizes in one scan (a set's are below 2^16 in all)
        const uint32_t both = __builtin_amdgcn_perm(inf1, inf0, 0x05040100u);
        const uint32_t incl = QL::scan_blocks(both);
        const uint32_t tot = rdlane(incl, kWaveSize - 1);
        const uint32_t ctot = (tot & 0xffffu) + (tot >> 16);
        const uint32_t ex = incl - both;
        const uint32_t at0 = wave_tot - copied;
        uint32_t off[2] = {at0 + (ex & 0xffffu), at0 + (tot & 0xffffu) + (ex >> 16)};   // in the staging area
        if (c < c_over && at0 + ctot > kStageBytes) {
            c_over = c;
            staged = wave_tot;
        }
        wave_tot += ctot;
        if (c >= c_over) return;

        // ---- the words ------------------------------------------------------
        const uint32_t bs[2] = {(inf0 >> 16) & 0xffu, (inf1 >> 16) & 0xffu};
        uint32_t sign0[2] = {0, 0};   // in bit 31, of an element 0 that travels in the prefix
        if constexpr (MODE == kOutlier) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t pre = (s ? inf1 : inf0) >> 24;
                const bool drop = (pre & ql.e0) != 0;
                if (drop) {
                    // |d| of element 0, little-endian: 4 bytes, of which the
                    // sign word written next covers what is past the prefix
                    *(lds_u32u*)(sbase + off[s]) = (s ? v1 : v0)[NV - 1];
                }
                off[s] += pre;
                sign0[s] = drop ? d[s][0] : 0u;
                d[s][0] = drop ? 0u : d[s][0];
            }
        }
        // a word of either half's payload; lanes without one write the spare word
        auto word = [&](int s, bool has, uint32_t o, uint32_t w) {
            const uint32_t at = has ? off[s] + (s0 + o) : spare;
            *(lds_u32u*)(size_t)at = w;
        };
        // the words of N sets from s on
        auto emit = [&](auto nsc, auto nc, int s) {
            constexpr int NS = decltype(nsc)::value, N = decltype(nc)::value;
            uint32_t w[N * NS];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                uint32_t t[NS];
                slices_of<NS>(d[s + j], t);
                if constexpr (MODE == kOutlier) t[NS - 1] |= sign0[s + j] & 0x80000000u;
#pragma unroll
                for (int i = 0; i < NS; ++i) w[j * NS + i] = t[i];
            }
            to_planes<N * NS>(w, pc);
            uint32_t pk = 0, pp = 0;
            if constexpr (!kKept) plane_word(pk, pp);
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                // plane p is there if p + 1 < b, the sign word if 0 < b
                uint32_t k = kKept ? pl : pk, p = kKept ? po : pp;
                opaque_here(k);
                opaque_here(p);
                const bool sign = i == NS - 1 && k == 7;
                uint32_t key = sign ? 0u : 8 * i + 1 + k, o = sign ? p - 8 * S : p + 8 * S * i;   // the sign word is 8 planes in front of plane 7
                opaque_here(key);
                opaque_here(o);
#pragma unroll
                for (int j = 0; j < N; ++j) word(s + j, key < bs[s + j], o, w[j * NS + i]);
            }
        };
        typedef std::integral_constant<int, 1> one;
        typedef std::integral_constant<int, 2> two;
        if (!over7 && !rare) {
            emit(one{}, two{}, 0);
        } else if (!over15 && !rare) {
            emit(two{}, two{}, 0);
        } else if (DIM == 1 || !rare) {
            emit(std::integral_constant<int, 4>{}, one{}, 0);   // one set at a time: fewer registers
            emit(std::integral_constant<int, 4>{}, one{}, 1);
        } else {
            // blocks of 32 planes: all 32 bits are planes and the sign words go separately
            uint32_t k = ql.k, p = pl, o = po;
            if constexpr (!kKept) plane_word(p, o);
            opaque_here(k);
            opaque_here(p);
            opaque_here(o);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t w[4], a[4], sg = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t neg = d[s][i] >> 31;
                    a[i] = neg ? 0u - d[s][i] : d[s][i];
                    sg |= (i == 0 ? neg | (sign0[s] >> 31) : neg) << (7 - 4 * (k & 1) - i);   // element e at bit e^7
                }
                sg <<= 8 * (k >> 1);
                sg |= dpp<kDppQuadSwap1>(sg);
                sg |= dpp<kDppQuadSwap2>(sg);
                sg |= dpp<kDppHalfMirror>(sg);
                word(s, bs[s] != 0, o - 8 * p - 8, sg);   // the same from the half's eight lanes
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    w[t] = ((a[3] >> (8 * t)) & 0xff) | (((a[2] >> (8 * t)) & 0xff) << 8) |
                           (((a[1] >> (8 * t)) & 0xff) << 16) | (((a[0] >> (8 * t)) & 0xff) << 24);
                to_planes<4>(w, pc);
#pragma unroll
                for (int i = 0; i < 4; ++i) word(s, 8 * i + p + 1 < bs[s], o + 8 * S * i, w[i]);
            }
        }
    };

    // Runs the wave's chunks from c0 on; before(c) runs first for each. A chunk
    // past the array's groups is all zero: rate bytes 0 in every mode and no
    // payload.
    const uint64_t gvalid = (DIM == 1) ? (geo.n + 63) / 64 : geo.nblocks;   // groups holding elements
    const int nch = chunks_of(KC, wgrp0, gvalid, G - 1);                    // chunks with elements
    auto run = [&](int c0, auto&& before) {
        if constexpr (RUNS) {
            const int nfull = (DIM == 1) ? chunks_of(KC, wgrp0, geo.n / 64, 0) : nch;   // whole chunks
            if (c0 < nfull) {
                Walker wkn;   // 2D/3D: the chunk whose loads are issued next
                if constexpr (DIM != 1) wkn.init(wgrp0 + (uint64_t)c0 * G, geo);
                Pieces<DIM, T> pcs;
                pcs.init(ql, geo, lane);
                // chunk c's loads of set s; c only goes up (2D/3D: all sets of a chunk first)
                auto load = [&](int c, int s, T (&x)[4]) {
                    const T* p;
                    if constexpr (DIM == 1) p = in + (wgrp0 + (uint64_t)c * G) * 64;
                    else p = in + block_origin<DIM>(geo, wkn);
                    pcs.template load<NT>(p, c < nfull, s, x);
                    if (DIM != 1 && s == 1) wkn.step(geo, G);
                };
                T xv[2][4];
#pragma unroll
                for (int s = 0; s < 2; ++s) load(c0, s, xv[s]);
#pragma unroll 1
                for (int c = c0; c < nfull; ++c) {
                    // a set's next loads follow as soon as its values are coded
                    before(c);
                    process(std::true_type{}, c, xv, true, 0u, [&](int s) { load(c + 1, s, xv[s]); });
                }
            }
            if (DIM == 1 && nfull < nch) {   // the array's last elements
                before(nfull);
                T xv[2][4];
                uint32_t vm = 0;
                const uint64_t e = (wgrp0 + (uint64_t)nfull * G) * 64 + 4 * (uint64_t)lane;
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint64_t at = e + 256 * s + i;
                        const bool v = at < geo.n;
                        xv[s][i] = v ? in[at] : T(0);
                        vm |= (uint32_t)v << (4 * s + i);
                    }
                process(std::false_type{}, nfull, xv, false, vm, [](int) {});
            }
        } else if (c0 < nch) {
            const bool near = geo.near != 0;
            RaggedQuads<DIM, T> rq;
            rq.init(geo, ql, wgrp0 + (uint64_t)c0 * G, wgrp0 + (uint64_t)KC * G);
            const T* p = in;          // the chunk's origin
            uint32_t vo[2] = {kAbsent, kAbsent};
            auto locate = [&]() -> bool {
                uint64_t base;
                const bool whole = rq.next(geo, base, vo);
                p = in + base;
                return whole;
            };
            auto inside = [&]() -> uint32_t { return ((int32_t)vo[0] >= 0 ? 0xfu : 0u) | ((int32_t)vo[1] >= 0 ? 0xf0u : 0u); };
            T xv[2][4];
            bool whole = false;
            if (near) whole = locate();
#pragma unroll
            for (int s = 0; s < 2; ++s) RaggedQuads<DIM, T>::load(p, vo[s], xv[s]);
            uint32_t vm = inside();
            bool next_whole = false;
            if (near) next_whole = locate();
#pragma unroll 1
            for (int c = c0; c < nch; ++c) {
                before(c);
                if (!near) {   // rows (2D) or slices (3D) of tens of millions of values: no loads ahead
                    ChunkQuads<DIM> cq;
                    cq.locate(geo, ql, rq.wk);
                    vm = (cq.ok[0] ? 0xfu : 0u) | (cq.ok[1] ? 0xf0u : 0u);
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        load_quad<false>(in + cq.off[s], xv[s]);   // quads outside the array read its first one
#pragma unroll
                        for (int i = 0; i < 4; ++i) xv[s][i] = cq.ok[s] ? xv[s][i] : T(0);
                    }
                }
                process(std::false_type{}, c, xv, whole, vm, [&](int s) { RaggedQuads<DIM, T>::load(p, vo[s], xv[s]); });
                // the chunk after the next, while the next one's loads are under way
                whole = next_whole;
                vm = inside();
                if (near) next_whole = locate();
            }
        }
    };
    run(0, [](int) {});
    for (int c = nch; c < KC; ++c)   // 1D header padding, 2D/3D pad bytes below H
        if (lane < NB / 4) sm.hdr[wave][c * (NB / 4) + lane] = 0;

    // ---- the wave's header bytes (their positions do not depend on the
    // offset); 2D/3D pad bytes [nblocks, H) are 0. Both H and the wave's first
    // block are multiples of 4 -------------------------------------------------
    {
        const int NW = KC * NB / 4;
        static_assert(NB % 4 == 0 && kChunksOf<T> * NB / 4 <= 32, "header words of a wave");
        __builtin_amdgcn_wave_barrier();
        const uint64_t b = ((DIM == 1) ? 2 * wgrp0 : wgrp0) + 4 * (uint64_t)lane;
        if (lane < NW && b < geo.H) store_u32u(dst + b, sm.hdr[wave][lane]);
    }

    // ---- the tile's offset (wave 0) ---------------------------------------------
    if (lane == 0) {
        sm.wtot[wave] = wave_tot;
        if (lossy) raise_bit(cur.err, kWarnLossy, cur.mark);
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const uint64_t t = sm.wtot[w];
        wexcl += (w < wave) ? t : 0;
        ttot += t;
    }
    if (wave == 0) {
        const uint64_t e = lookback(sc, tile, cur.tile0, ttot, lane, window, [&](uint64_t p) {
            return compress_tile_bytes<DIM, MODE, T, WAVES>((const T*)cur.src, geo, r, p - cur.tile0, lane);
        });
        if (lane == 0) {
            sm.excl = e;
            if (lt == geo.ntiles - 1) {
                const unsigned long long bytes = geo.H + e + ttot;
                if (cur.total) *cur.total = bytes;
                if (cur.host_total) __hip_atomic_store(cur.host_total, bytes, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
    __syncthreads();
    excl = sm.excl;
    if (geo.H + excl + ttot > cur.limit) {   // never write past the caller's buffer
        if (wave == 0 && lane == 0) raise_bit(cur.err, kErrOverflow, cur.mark);
        return;
    }
    // ---- copy the staged payload: 16 bytes per lane, then the tail bytes ---------
    uint8_t* const obase = dst + uniform64(geo.H + excl + wexcl);
    auto copy_out = [&](uint32_t upto) {   // staged bytes [copied, upto) of the wave's payload
        typedef uint32_t v4uu __attribute__((ext_vector_type(4), aligned(1)));
        typedef uint32_t v4ul __attribute__((ext_vector_type(4)));
        uint8_t* const o = obase + copied;
        const uint32_t n = upto - copied;
        if (cur.flags & kItemStreamNt) {
            // Nontemporal stores at 16-byte-aligned addresses (the staged bytes
            // are then read at any offset), single bytes at the ends: a
            // compute-free kernel that reads 4 GiB and writes 3,564 bytes per 16
            // KiB took 0.887 ms with stores from each wave's own start, 0.852 ms
            // this way.
            uint32_t head = (0u - (uint32_t)(uintptr_t)o) & 15u;
            head = head < n ? head : n;
            const uint32_t body = (n - head) & ~15u, tail = n - head - body;
            for (uint32_t i = 16u * (uint32_t)lane; i < body; i += 16u * kWaveSize) {
                const lds_u8* const q = sbase + head + i;
                const v4ul v = {*(const lds_u32u*)q, *(const lds_u32u*)(q + 4), *(const lds_u32u*)(q + 8), *(const lds_u32u*)(q + 12)};
                __builtin_nontemporal_store(v, (v4ul*)(o + head + i));
            }
            if ((uint32_t)lane < head) o[lane] = sbase[lane];
            if ((uint32_t)lane < tail) o[head + body + lane] = sbase[head + body + lane];
        } else {
            const uint32_t n16 = n & ~15u;
            for (uint32_t i = 16u * (uint32_t)lane; i < n16; i += 16u * kWaveSize)
                *(v4uu*)(o + i) = *(const v4ul*)&sm.stage[wave][i / 16];
            if ((uint32_t)lane < (n & 15u)) o[n16 + lane] = sbase[n16 + lane];
        }
        copied = upto;
    };
    if (c_over == KC) {
        copy_out(wave_tot);
        return;
    }
    // the rest of the chunks: staged as before, copied whenever the next one may not fit
    wave_tot = staged;
    const int c0 = c_over;
    c_over = KC;
    run(c0, [&](int) {
        if (wave_tot - copied + kMaxChunkBytes > kStageBytes) {
            __builtin_amdgcn_wave_barrier();
            copy_out(wave_tot);
            __builtin_amdgcn_wave_barrier();
        }
    });
    __builtin_amdgcn_wave_barrier();
    copy_out(wave_tot);
}

// Decompresses tile `tile` of array `cur` (every wave of the workgroup calls
// it); the tile has the compress tile's shape (KC chunks of 512 elements per
// wave):
//   1. each wave reads the header bytes of its blocks (one or two per lane),
//      scans their sizes once and writes every block's metadata (offset within
//      the wave's payload, planes) to LDS;
//   2. the wave's payload offset;
//   3. each wave works through its chunks: every lane reads the plane words of
//      its lane number from the payload (one per set and byte slice; as many
//      slices as the chunk's largest rate needs), transposes them back to its
//      quad's residuals, sums those along the Lorenzo chains (dot products inside
//      the quad, one scan of DPP adds across the block's lanes) and stores
//      (T)q * eb * 2.
//
// The wave's payload offset is the sum of the block sizes before it: with an
// offset table `offs` (unit_offsets_kernel, unit_offsets_batch_kernel) the entry
// of the launch's wave, and every wave runs on its own, without a barrier; else
// (short headers) the workgroup sums the header bytes in front of its tile
// itself: a read that hits in cache, and no pass.
template <int DIM, int MODE, class T, int WAVES, bool RUNS>
__device__ __forceinline__ void decompress_tile(const Item& cur, const uint64_t tile, SmemD<WAVES>& sm,
                                                const unsigned long long* __restrict__ offs) {
    typedef QuadLane<DIM> QL;
    constexpr int G = kChunkElems / 64;
    constexpr int S = (DIM == 1) ? 4 : 8;
    constexpr int SB = QL::SB, NB = QL::NB;             // blocks per set, per chunk
    constexpr int NBX = kChunksOf<T> * NB;              // blocks per wave, at most
    constexpr int BPL = (NBX + kWaveSize - 1) / kWaveSize;   // blocks per bookkeeping lane
    static_assert(NBX <= 2 * kWaveSize && NBX <= kMetaPerWave, "a wave's blocks: at most two per lane");

    const int lane = (int)__lane_id();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const Geom& geo = cur.geo;
    const int KC = (int)geo.kc, NBW = KC * NB;          // blocks per wave
    const uint8_t* __restrict__ cmp = (const uint8_t*)cur.src;
    const uint64_t lt = tile - cur.tile0;
    const uint64_t wgrp0 = (lt * WAVES + (uint64_t)wave) * (uint64_t)(KC * G);   // this wave's first group
    const uint64_t wb0 = (DIM == 1) ? 2 * wgrp0 : wgrp0;               // and first block

    // ---- bookkeeping: lane j holds blocks BPL*j .. BPL*j + BPL-1 of the wave ------
    BlockView v[BPL];
    uint32_t sz[BPL];
    bool okb[BPL];
    uint32_t lsum = 0, rmax = 0;
#pragma unroll
    for (int k = 0; k < BPL; ++k) {
        const int j = BPL * lane + k;
        const uint64_t b = wb0 + (uint64_t)j;
        okb[k] = j < NBW && (DIM == 1 || b < geo.nblocks);
        const uint32_t byte = okb[k] ? (uint32_t)cmp[b] : 0u;
        v[k] = view_of<MODE, S>(byte);
        sz[k] = okb[k] ? v[k].size : 0u;
        lsum += sz[k];
        rmax = rmax > v[k].R ? rmax : v[k].R;
    }
    const uint32_t incl = scan_wave(lsum);                 // < 2^32; a cross-lane scan: all lanes
    const uint32_t wtot = rdlane(incl, kWaveSize - 1);
    const uint32_t excl0 = incl - lsum;                    // offset of this lane's first block
    {
        uint32_t off = excl0;                              // offsets within the wave's payload
#pragma unroll
        for (int k = 0; k < BPL; ++k) {
            const int j = BPL * lane + k;
            // every entry is written: blocks past the array carry no words
            if (j < NBW) sm.meta[wave][j] = make_dmeta<MODE>(off, v[k], okb[k] && sz[k] != 0);
            off += sz[k];
        }
    }
    // lanes whose blocks need more than one byte slice, or more than two, or
    // hold 32 planes (2D/3D: the sign words move in front of all planes)
    const uint64_t over7 = ballot(rmax > 7), over15 = ballot(rmax > 15);
    const uint64_t over31 = (MODE == kOutlier) ? 0ull : ballot(rmax > 31);

    uint64_t wave_base;
    if (offs) {
        wave_base = uniform64(offs[tile * WAVES + (uint64_t)wave]);
        __builtin_amdgcn_wave_barrier();   // the metadata in LDS is this wave's own
    } else {
        const uint64_t before = lt * WAVES * (uint64_t)NBW;   // header bytes in front of the tile: a multiple of 16
        const uint32_t share = header_share<MODE, S>(cmp, before, threadIdx.x, WAVES * kWaveSize);
        const uint32_t sum = rdlane(scan_wave(share), kWaveSize - 1);   // < 2^32: at most kDirectHeader blocks
        if (lane == 0) {
            sm.wtot[wave] = wtot;
            sm.before[wave] = sum;
        }
        __syncthreads();
        uint64_t wexcl = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) wexcl += sm.before[w] + ((w < wave) ? (uint64_t)sm.wtot[w] : 0);
        wave_base = geo.H + uniform64(wexcl);
    }
    const uint8_t* const wbase = cmp + uniform64(wave_base);
    const bool intact = wave_base + wtot <= cur.limit;
    if (!intact && lane == 0) raise_bit(cur.err, kErrTruncated, cur.mark);
    // The wave's stream words go through a buffer resource over its payload:
    // 32-bit offsets, and an offset past the range (bit 31 set) reads 0, so
    // lanes without a word need no address select and no masking; a truncated
    // stream gets an empty range (every word reads 0).
    const uint64_t span = cur.limit - wave_base;
    const int nrec = __builtin_amdgcn_readfirstlane(intact ? (int)(span < 0x7fffffffull ? span : 0x7fffffffull) : 0);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)wbase, 0, nrec, kBufferWord3);

    QL ql;
    ql.init(lane);
    PlaneConsts pc;
    pc.init(lane, true);
    const uint32_t pl = plane_of_lane(ql.k), po = ql.plane_offset(pl);   // this lane's plane of slice 0, its word in a block
    T* __restrict__ out = (T*)cur.dst;
    const T eb = (T)cur.param;
    const uint64_t gvalid = (DIM == 1) ? (geo.n + 63) / 64 : geo.nblocks;   // groups holding elements
    // chunks with elements of the array, and (1D) whole ones
    const int nch = chunks_of(KC, wgrp0, gvalid, G - 1);
    const int nfull = (DIM == 1) ? chunks_of(KC, wgrp0, geo.n / 64, 0) : nch;
    Walker wkc;   // 2D/3D: the chunk being stored
    RaggedQuads<DIM, T> rq;
    if constexpr (DIM != 1) {
        if (!RUNS && geo.near) rq.init(geo, ql, wgrp0, wgrp0 + (uint64_t)KC * G);
        else wkc.init(wgrp0, geo);
    }

    typedef uint32_t v4u __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) v4u lds_v4u;
    lds_u8* const buf = (lds_u8*)sm.payload[wave];
    const lds_u8* const zw = (const lds_u8*)&sm.zero[wave][0];
    if (lane < 2) sm.zero[wave][lane] = 0;

    // values of codes (a block without payload, or of a truncated stream,
    // decoded all-zero words: q = 0)
    auto value_of = [&](uint32_t q) -> T { return (T)(int32_t)q * eb * T(2); };   // src/cuSZp_kernels_1D_f32.cu:490

    Pieces<DIM, T> pcs;
    if constexpr (RUNS) pcs.init(ql, geo, lane);
    // Stores a chunk's codes as values. Where chunks are runs of blocks, the
    // output is written once and nontemporally (in pieces that fill lines): dirty
    // lines of it left in L2 and the last-level cache would cost the next kernel
    // their write-back.
    auto store_chunk = [&](int c, uint32_t (&q)[2][4]) {
        if (RUNS && (DIM != 1 || c < nfull)) {
            T* o;
            if constexpr (DIM == 1) {
                o = out + (wgrp0 + (uint64_t)c * G) * 64;
            } else {
                o = out + block_origin<DIM>(geo, wkc);
                wkc.step(geo, G);
            }
            trade_codes<DIM, T>(q);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                T x[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = value_of(q[s][i]);
                pcs.store(o, s, x);
            }
        } else if constexpr (DIM == 1) {   // the array's last elements
            const uint64_t e = (wgrp0 + (uint64_t)c * G) * 64 + 4 * (uint64_t)lane;
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (e + 256 * s + i < geo.n) out[e + 256 * s + i] = value_of(q[s][i]);
        } else {
            // every quad by its own place; plain stores, which meet in L2
            if (geo.near) {
                uint64_t base;
                uint32_t vo[2];
                rq.next(geo, base, vo);
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    T x[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[i] = value_of(q[s][i]);
                    RaggedQuads<DIM, T>::store(out + base, vo[s], x);
                }
                return;
            }
            ChunkQuads<DIM> cq;
            cq.locate(geo, ql, wkc);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                T x[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) x[i] = value_of(q[s][i]);
                if (cq.ok[s]) store_quad<false>(out + cq.off[s], x);
            }
        }
    };

    // Decodes chunk c; fetch(o) reads the payload word at byte offset o of the
    // wave's payload, or 0 for o = kAbsent.
    constexpr int LPC = NB / BPL;   // bookkeeping lanes per chunk
    static_assert(LPC * BPL == NB, "whole lanes per chunk");
    auto decode_chunk = [&](int c, auto&& fetch, uint32_t (&q)[2][4]) {
        DMeta mt[2];
#pragma unroll
        for (int s = 0; s < 2; ++s) mt[s] = sm.meta[wave][c * NB + s * SB + ql.blk];
        const uint64_t cl = ((1ull << LPC) - 1) << (c * LPC);
        // |d| of element 0 of a selected block: up to 4 bytes in front of its sign
        // word; the planes' bits of that element (bits 0-30 of byte 3 of the
        // lane's slices) are ignored (src/cuSZp_kernels_1D_f32.cu:1887)
        uint32_t e0[2] = {0, 0}, keep[2] = {~0u, ~0u};
        if constexpr (MODE == kOutlier) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const uint32_t nbits = mt[s].prefix_bits();
                const bool own = mt[s].sel() && ql.e0;
                const uint32_t w = fetch(own ? mt[s].off() - (nbits >> 3) : kAbsent);
                keep[s] = own ? 0x00ffffffu : ~0u;
                e0[s] = (w << (32 - nbits)) >> (32 - nbits);
            }
        }
        auto decode = [&](auto nsc) {
            constexpr int NS = decltype(nsc)::value;
            uint32_t w[2 * NS];
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                uint32_t k = pl, p = po;
                opaque_here(k);
                opaque_here(p);
                const bool sign = i == NS - 1 && k == 7;
                uint32_t key = lane_key(sign ? 0u : 8 * i + 1 + k), o = sign ? p - 8 * S : p + 8 * S * i;   // the sign word is 8 planes in front of plane 7
                opaque_here(key);
                opaque_here(o);
#pragma unroll
                for (int s = 0; s < 2; ++s) w[s * NS + i] = fetch(mt[s].word_at(key, o));
            }
            from_planes<2 * NS>(w, pc);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint32_t t[NS], s0;
#pragma unroll
                for (int i = 0; i < NS; ++i) {
                    t[i] = w[s * NS + i];
                    if constexpr (MODE == kOutlier) t[i] &= i == NS - 1 ? keep[s] | 0x80000000u : keep[s];
                }
                Residuals<NS> rs;
                rs.from_slices(t, s0);
                const uint32_t r0 = (MODE == kOutlier) ? (e0[s] ^ s0) - s0 : 0u;   // 0 except in lane e0 of a selected block
                if constexpr (MODE == kFixed) {
                    q[s][0] = rs.template at<0>();
                    q[s][1] = rs.template at<1>();
                    q[s][2] = rs.template at<2>();
                    q[s][3] = rs.template at<3>();
                } else {
                    ql.codes(rs, r0, q[s]);
                }
            }
        };
        if (!(over7 & cl)) {
            decode(std::integral_constant<int, 1>{});
        } else if (!(over15 & cl)) {
            decode(std::integral_constant<int, 2>{});
        } else if (DIM == 1 || MODE == kOutlier || !(over31 & cl)) {
            decode(std::integral_constant<int, 4>{});
        } else {
            // 2D/3D blocks of 32 planes among the chunk's: all 32 bits are
            // magnitude, the signs come from the sign words by themselves
            uint32_t w[8], sg[2], k = ql.k, p = pl, o = po;
            opaque_here(k);
            opaque_here(p);
            opaque_here(o);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                sg[s] = fetch(mt[s].word_at(lane_key(0), o - 8 * p - 8));
#pragma unroll
                for (int i = 0; i < 4; ++i) w[4 * s + i] = fetch(mt[s].word_at(lane_key(8 * i + p + 1), o + 8 * S * i));
            }
            from_planes<8>(w, pc);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                Residuals<4> rs;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int b = 8 * (3 - i);   // element i in byte 3 - i of the slices
                    const uint32_t a = ((w[4 * s] >> b) & 0xff) | (((w[4 * s + 1] >> b) & 0xff) << 8) |
                                       (((w[4 * s + 2] >> b) & 0xff) << 16) | (((w[4 * s + 3] >> b) & 0xff) << 24);
                    const uint32_t neg = (sg[s] >> (8 * (k >> 1) + 7 - 4 * (k & 1) - i)) & 1;   // element e at bit e^7
                    rs.v[i] = neg ? 0u - a : a;
                }
                if constexpr (MODE == kFixed) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[s][i] = rs.v[i];
                } else {
                    ql.codes(rs, 0u, q[s]);
                }
            }
        }
    };

    // Where the words come from. A chunk's payload is contiguous: where every
    // chunk of the wave spans at most kDenseBytes from its 4-byte-aligned start,
    // it is read with one or two dense 16-byte-per-lane loads into the wave's
    // LDS buffer and each lane reads its words from there (lanes without a word
    // read a zero word). Loads with some lanes past the buffer range cost far
    // more memory-pipeline time than dense ones. Otherwise each lane loads its
    // own words from global memory.
    auto chunk_start = [&](int c) -> uint32_t { return c < KC ? rdlane(excl0, (uint32_t)(c * LPC)) : wtot; };   // in the wave's payload
    // Buffer loads check their range per dword, so the dwords holding the
    // payload's last bytes must lie inside it: an outlier stream whose length
    // is not a multiple of 4 ends inside a dword, and its last wave keeps the
    // per-lane loads (a truncated stream has an empty range: the same).
    const bool whole = ((wtot + 3u) & ~3u) <= (uint32_t)nrec;   // every payload dword inside the range
    // The wave's whole payload in one burst of loads before its first chunk,
    // where it fits the wave's buffer. A compute-free kernel with the 1D
    // decode's traffic (2^30 f32 written, 0.94 GB read) ran 2.5-4 % faster with
    // each wave's reads in one burst than with a read per chunk.
    const bool burst = whole && wtot <= (uint32_t)kWaveBuf;
    bool dense = whole;
    if (!burst)
        for (int c = 0; c < KC; ++c) dense &= chunk_start(c + 1) - (chunk_start(c) & ~3u) <= (uint32_t)kDenseBytes;
    auto fetch_lds = [&](uint32_t origin) {
        return [=](uint32_t o) -> uint32_t {
            const lds_u8* const p = (int32_t)o < 0 ? zw : buf + (o - origin);
            if constexpr (MODE != kOutlier) return *(const __attribute__((address_space(3))) uint32_t*)p;   // whole 4-byte words
            else return *(const lds_u32u*)p;   // prefixes shift later blocks by 1-3 bytes
        };
    };
    if (burst) {
        constexpr int NL = (kWaveBuf + 1023) / 1024;
        v4u P[NL];
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            // 1 KiB per load; none past the payload; lanes past the buffer read nothing
            const uint32_t o = 1024u * (uint32_t)k + 16u * (uint32_t)lane;
            P[k] = __builtin_amdgcn_raw_buffer_load_b128(
                rsrc, (1024u * (uint32_t)k < wtot && o < (uint32_t)kWaveBuf) ? o : kAbsent, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < NL; ++k)
            if (1024 * k + 16 * lane < kWaveBuf) ((lds_v4u*)buf)[64 * k + lane] = P[k];
        __builtin_amdgcn_wave_barrier();
#pragma unroll 1
        for (int c = 0; c < nch; ++c) {
            uint32_t q[2][4];
            decode_chunk(c, fetch_lds(0), q);
            store_chunk(c, q);
        }
    } else if (dense) {
        // Chunk by chunk, one chunk ahead: a chunk's loads are issued after the
        // stores of the one before the last, so that waiting for them (loads
        // and stores retire in order on this GPU) waits for no later store.
        auto load_chunk = [&](int c, v4u (&P)[2]) {
            // from the chunk's aligned start; the second KiB only when needed
            // (else an offset past every range: no memory access)
            const uint32_t a0 = chunk_start(c) & ~3u, a1 = chunk_start(c + 1);
            P[0] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, c < nch ? a0 + 16u * (uint32_t)lane : kAbsent, 0, 0);
            P[1] = __builtin_amdgcn_raw_buffer_load_b128(
                rsrc, c < nch && a1 - a0 > 1024u ? a0 + 1024u + 16u * (uint32_t)lane : kAbsent, 0, 0);
        };
        v4u P[2];
        uint32_t q[2][4];
        load_chunk(0, P);
#pragma unroll 1
        for (int c = 0; c <= nch; ++c) {
            if (c) store_chunk(c - 1, q);
            if (c == nch) break;
            __builtin_amdgcn_wave_barrier();   // the previous chunk's reads of the buffer come first
            ((lds_v4u*)buf)[lane] = P[0];
            ((lds_v4u*)buf)[64 + lane] = P[1];
            __builtin_amdgcn_wave_barrier();
            load_chunk(c + 1, P);
            decode_chunk(c, fetch_lds(chunk_start(c) & ~3u), q);
        }
    } else {
#pragma unroll 1
        for (int c = 0; c < nch; ++c) {
            uint32_t q[2][4];
            decode_chunk(c, [&](uint32_t o) -> uint32_t { return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc, o, 0, 0); }, q);
            store_chunk(c, q);
        }
    }
}

// ---------------------------------------------------------------------------
// single-array kernels: one workgroup per tile, tile = base + blockIdx.x (tiles
// are numbered in launch order; arrays of more than one grid's tiles take
// several launches)
// ---------------------------------------------------------------------------
template <int DIM, int MODE, class T, int WAVES, bool RUNS>
__global__ void __launch_bounds__(WAVES * kWaveSize, kCompressWavesPerSimd)
compress_kernel(const Item item, const ScanCtx sc, const uint64_t base) {
    __shared__ SmemC<WAVES> sm;
    // a compress tile's predecessors have mostly published by the time its
    // payload is staged: the 128-tile window (2 words per lane) is enough, or
    // one window for all tiles of a short array
    compress_tile<DIM, MODE, T, WAVES, RUNS>(item, base + blockIdx.x, sc, sm, item.geo.ntiles <= 64 * kLookbackWords ? kLookbackWords : 2);
}

// Waves take their payload offsets from `offs` (unit_offsets_kernel, launched
// before on the same stream), or sum them up where it is null (arrays of at most
// kDirectHeader header bytes).
template <int DIM, int MODE, class T, int WAVES, bool RUNS>
__global__ void __launch_bounds__(WAVES * kWaveSize, kDecompressWavesPerSimd)
decompress_kernel(const Item item, const unsigned long long* __restrict__ offs, const uint64_t base) {
    __shared__ SmemD<WAVES> sm;
    decompress_tile<DIM, MODE, T, WAVES, RUNS>(item, base + blockIdx.x, sm, offs);
}

// ---------------------------------------------------------------------------
// batched kernels: the arrays of a table, of any variant, in one launch with
// one workgroup per tile of the concatenated tile space. A tile's array is
// found by binary search on tile0, and each array's tiles (compress) or header
// segments (decompress) form a lookback segment of their own, so every array's
// stream is exactly its single-array stream.
// ---------------------------------------------------------------------------
#define CUSZP_BATCH_CASES(RUN)                                                        \
    case 0: RUN(1, kFixed, float); break;                                             \
    case 1: RUN(1, kPlain, float); break;                                             \
    case 2: RUN(1, kOutlier, float); break;                                           \
    case 3: RUN(2, kFixed, float); break;                                             \
    case 4: RUN(2, kPlain, float); break;                                             \
    case 5: RUN(2, kOutlier, float); break;                                           \
    case 6: RUN(3, kFixed, float); break;                                             \
    case 7: RUN(3, kPlain, float); break;                                             \
    case 8: RUN(3, kOutlier, float); break;                                           \
    case 9: RUN(1, kFixed, double); break;                                            \
    case 10: RUN(1, kPlain, double); break;                                           \
    case 11: RUN(1, kOutlier, double); break;                                         \
    case 12: RUN(2, kFixed, double); break;                                           \
    case 13: RUN(2, kPlain, double); break;                                           \
    case 14: RUN(2, kOutlier, double); break;                                         \
    case 15: RUN(3, kFixed, double); break;                                           \
    case 16: RUN(3, kPlain, double); break;                                           \
    case 17: RUN(3, kOutlier, double); break;                                         \
    default: break;

template <int WAVES>
__global__ void __launch_bounds__(WAVES * kWaveSize, kCompressWavesPerSimd)
compress_batch_kernel(const Item* __restrict__ items, uint32_t nitems, ScanCtx sc,
                      const unsigned long long* __restrict__ epoch, const int window, const uint64_t base) {
    __shared__ SmemC<WAVES> sm;
    sc.tag = (epoch[0] & kEpochMask) << kEpochShift;
    const ItemTable src{items, nitems};
    const uint64_t tile = base + blockIdx.x;
    const Item cur = src.get(src.locate(tile));
#define CUSZP_RUN_C(D, M, T)                                                          \
    if (D == 1 || cur.geo.runs) compress_tile<D, M, T, WAVES, true>(cur, tile, sc, sm, window); \
    else compress_tile<D, M, T, WAVES, D == 1>(cur, tile, sc, sm, window)
    switch (cur.variant) { CUSZP_BATCH_CASES(CUSZP_RUN_C) }
#undef CUSZP_RUN_C
}

template <int WAVES>
__global__ void __launch_bounds__(WAVES * kWaveSize, kDecompressWavesPerSimd)
decompress_batch_kernel(const Item* __restrict__ items, uint32_t nitems,
                        const unsigned long long* __restrict__ offs, unsigned long long* bump, const uint64_t base) {
    __shared__ SmemD<WAVES> sm;
    // the pass that read this epoch has finished: no kernel of its own for that (2 us and a gap)
    if (bump && base + blockIdx.x == 0 && threadIdx.x == 0) *bump += 1;
    const ItemTable src{items, nitems};
    const uint64_t tile = base + blockIdx.x;
    const Item cur = src.get(src.locate(tile));
#define CUSZP_RUN_D(D, M, T)                                                            \
    if (D == 1 || cur.geo.runs) decompress_tile<D, M, T, WAVES, true>(cur, tile, sm, offs); \
    else decompress_tile<D, M, T, WAVES, D == 1>(cur, tile, sm, offs)
    switch (cur.variant) { CUSZP_BATCH_CASES(CUSZP_RUN_D) }
#undef CUSZP_RUN_D
}

}  // namespace cuszp
