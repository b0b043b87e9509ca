// Batched C ABI: many arrays in one launch (compress or decompress) with one
// workgroup per tile of the concatenated arrays,
// optionally held as a captured hipGraph, with a launch-shape autotuner.
//
// A plan validates every array once (the same checks as cuSZp_compress_ex /
// cuSZp_decompress_ex), lays the arrays' tiles end to end, uploads one Item
// descriptor per non-empty array and owns the scan state: tile status words,
// an epoch word bumped on the device for each launch (so replays of a captured
// graph never see the previous run's status words as current), the offset table
// of a decompression, a launch-wide error word and one error word and one stream length per array.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "common.hpp"

using namespace cuszp;

struct cuszp_batch_plan_s {
    int dev = 0;
    int dir = CUSZP_BATCH_COMPRESS;
    int flags = 0;
    // launch shape (choose_shape, or the tuner's): waves per workgroup, chunks per
    // wave at most (a type's own limit holds), lookback words per lane (2 or 4)
    int waves = 8, kc = kChunksOf<float>, window = kLookbackWords;
    bool pass = false;             // decompress: some header is too long for the tiles to sum up
    std::vector<cuszp_batch_item_t> src;
    std::vector<Item> items;      // non-empty arrays, in caller order
    uint64_t ntiles = 0;
    uint64_t nseg = 0;            // decompress: segments of the offset pass, 0 without it
    bool built = false;           // the device table, scan state and offsets fit `items`
    bool epoch_used = false;            // an offset pass took the epoch and the decode kernel that advances it was not launched
    Item* d_items = nullptr;
    size_t cap_items = 0;
    unsigned long long* d_status = nullptr;
    uint64_t cap_status = 0;
    unsigned long long* d_offs = nullptr;   // decompress: payload offset of every decode wave
    uint64_t cap_offs = 0;
    unsigned long long* d_misc = nullptr;   // kMiscWords: [0] epoch, [2] launch bits, [4..7] diagnostics, [8..11] counters
    unsigned int* d_err = nullptr;          // per array
    unsigned long long* d_sizes = nullptr;  // per array (compress)
    unsigned long long* h_res = nullptr;    // pinned, written by the kernels: the mark (Item::mark), then a stream length per array
    hipStream_t cap_stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    unsigned info = 0;                      // information bits harvested since the last scan report
};

namespace {

#define BATCH_HIP(call)                                \
    do {                                               \
        hipError_t e_ = (call);                        \
        if (e_ != hipSuccess) return CUSZP_ERROR_HIP;  \
    } while (0)

// Pinned words that the kernels write. Allocating and freeing pinned memory takes about 33 us, as
// much as the rest of a plan's creation and a third of a one-shot call on small arrays, so the
// words of a destroyed plan wait for the next plan on that GPU: at most kKeptBuffers of kKeptWords
// per GPU (256 KiB). More of them, and those of plans of more arrays, are freed at once. A
// buffer comes back only when its GPU is idle, and is cleared for the next plan.
constexpr size_t kKeptBuffers = 4, kKeptWords = 8192;
std::mutex g_words_mu;
auto& g_words = *new std::map<int, std::vector<unsigned long long*>>;   // per GPU, idle; never destroyed, plans may be at exit

unsigned long long* take_words(int dev, size_t n) {
    unsigned long long* w = nullptr;
    if (n <= kKeptWords) {
        std::lock_guard<std::mutex> lk(g_words_mu);
        auto& kept = g_words[dev];
        if (!kept.empty()) {
            w = kept.back();
            kept.pop_back();
        }
    }
    if (!w && hipHostMalloc((void**)&w, std::max(n, kKeptWords) * sizeof(unsigned long long), hipHostMallocCoherent) != hipSuccess)
        return nullptr;
    std::memset(w, 0, n * sizeof(unsigned long long));
    return w;
}
// idle: no kernel writes the words any more
void return_words(int dev, unsigned long long* w, size_t n, bool idle) {
    if (!w) return;
    if (n <= kKeptWords && idle) {
        std::lock_guard<std::mutex> lk(g_words_mu);
        auto& kept = g_words[dev];
        if (kept.size() < kKeptBuffers) {
            kept.push_back(w);
            return;
        }
    }
    hipHostFree(w);
}

int check_item(const cuszp_batch_item_t& it, int dir, Geom& g) {
    const int dim = it.dim, type = it.type, mode = it.mode;
    if (bad_enums(dim, type, mode) || bad_eb(it.errorBound, type)) return CUSZP_ERROR_INVALID_ARGUMENT;
    int rc = make_geom(dim, it.nbEle, it.dims, g);
    if (rc) return rc;
    if (it.nbEle == 0) return CUSZP_SUCCESS;
    if (!it.d_in || !it.d_out) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (max_stream_bytes(dim, g) > kMaxStream) return CUSZP_ERROR_TOO_LARGE;
    if (it.capacity < g.H) return dir == CUSZP_BATCH_COMPRESS ? CUSZP_ERROR_OUTPUT_TOO_SMALL : CUSZP_ERROR_CORRUPT_STREAM;
    return CUSZP_SUCCESS;
}

int chunks(const cuszp_batch_item_t& s, int kc) {
    return std::min(kc, s.type == CUSZP_TYPE_DOUBLE ? kChunksOf<double> : kChunksOf<float>);
}
uint64_t tiles(const cuszp_batch_item_t& s, const Geom& g, int waves, int kc) {
    const uint64_t groups = (s.dim == CUSZP_DIM_1D) ? g.H / 2 : g.nblocks;
    const uint64_t per_tile = tile_groups(s.type == CUSZP_TYPE_DOUBLE, waves, chunks(s, kc));
    return (groups + per_tile - 1) / per_tile;
}

// The shape of a plan that is not tuned: as a single array's (plan_tiles), with
// the tiles of all arrays together, and at least 4 chunks per wave under an
// offset pass (a thread of the pass takes 32 header bytes). 256 arrays of 1 Ki to
// 16 Mi values, 2.2 GB: 4 waves 522 / 429 us (compress / decompress), 8 waves
// 471 / 417; 16 arrays of up to 256 Ki values, 30 / 27 us with full waves, 22 / 19
// with the rule's (4, 2).
void choose_shape(cuszp_batch_plan_s& p) {
    typedef std::vector<std::pair<int, int>> Ladder;   // (waves, chunks)
    for (const auto& shape : p.pass ? Ladder{{4, 4}, {8, 4}} : Ladder{{4, 1}, {4, 2}, {8, 2}, {8, 4}}) {
        p.waves = shape.first;
        p.kc = shape.second;
        // counted up to the limit only: some hundred arrays at most, however many there are (4,000 arrays,
        // counted in full for each shape, took 40 us of a plan's creation)
        const uint64_t limit = shape_tiles(p.waves);
        uint64_t n = 0;
        for (size_t i = 0; i < p.src.size() && n <= limit; ++i) {
            const cuszp_batch_item_t& s = p.src[i];
            Geom g;
            make_geom(s.dim, s.nbEle, s.dims, g);
            if (s.nbEle) n += tiles(s, g, p.waves, p.kc);
        }
        if (n <= limit) return;
    }
    p.waves = 8;
    p.kc = kChunksOf<float>;
}

// Lay out the tiles of every non-empty array for the plan's shape and upload the
// descriptors (grows device buffers as needed).
int build_table(cuszp_batch_plan_s& p, hipStream_t st) {
    p.built = false;   // until all of it is there: nothing may be launched on part of it
    p.items.clear();
    uint64_t tile0 = 0, seg0 = 0;
    for (size_t i = 0; i < p.src.size(); ++i) {
        const cuszp_batch_item_t& s = p.src[i];
        if (s.nbEle == 0) continue;
        Geom g;
        make_geom(s.dim, s.nbEle, s.dims, g);
        g.kc = chunks(s, p.kc);
        g.ntiles = tiles(s, g, p.waves, p.kc);
        const bool c = p.dir == CUSZP_BATCH_COMPRESS;
        Item it = make_item(s.d_in, s.d_out, s.capacity, c ? p.d_sizes + i : nullptr, p.d_err + i,
                            c ? compress_param(s.errorBound, s.type) : decompress_param(s.errorBound, s.type),
                            s.dim, s.type, s.mode, g);
        it.mark = p.h_res;
        if (c) it.host_total = p.h_res + 1 + i;
        it.tile0 = tile0;
        tile0 += g.ntiles;
        it.seg0 = seg0;
        seg0 += batch_segments(s.dim, s.type == CUSZP_TYPE_DOUBLE, (int)g.kc, g.ntiles * (uint64_t)p.waves);
        p.items.push_back(it);
    }
    p.ntiles = tile0;
    p.nseg = p.pass ? seg0 : 0;
    // Growing a buffer: the old one is released before the new one is
    // allocated, and the capacity drops to 0 in between, so a failed
    // allocation leaves no buffer that a later call would take as large enough
    // (every launch of the plan has finished: the table is built only between
    // synchronised calls).
    if (p.items.size() > p.cap_items) {
        if (p.d_items) BATCH_HIP(hipFree(p.d_items));
        p.d_items = nullptr;
        p.cap_items = 0;
        BATCH_HIP(hipMalloc((void**)&p.d_items, p.items.size() * sizeof(Item)));
        p.cap_items = p.items.size();
    }
    const uint64_t words = p.dir == CUSZP_BATCH_COMPRESS ? p.ntiles : p.nseg;
    const uint64_t need = words ? words : 1;   // an empty table still gets a (cleared) status array
    if (need > p.cap_status) {
        if (p.d_status) BATCH_HIP(hipFree(p.d_status));
        p.d_status = nullptr;
        p.cap_status = 0;
        // kStatusGuard words in front (lookback windows of first tiles read there)
        BATCH_HIP(scan_state_alloc(&p.d_status, (kStatusGuard + need) * sizeof(unsigned long long)));
        p.cap_status = need;
    }
    const uint64_t units = p.nseg ? p.ntiles * (uint64_t)p.waves : 0;
    if (units > p.cap_offs) {
        if (p.d_offs) BATCH_HIP(hipFree(p.d_offs));
        p.d_offs = nullptr;
        p.cap_offs = 0;
        BATCH_HIP(scan_state_alloc(&p.d_offs, units * sizeof(unsigned long long)));
        p.cap_offs = units;
    }
    // stale status words must not carry the current epoch: start from zero and
    // restart the epoch whenever the table changes
    BATCH_HIP(hipMemsetAsync(p.d_status, 0, (kStatusGuard + p.cap_status) * sizeof(unsigned long long), st));
    BATCH_HIP(hipMemsetAsync(p.d_misc, 0, sizeof(unsigned long long), st));
    if (p.nseg) BATCH_HIP(launch_bump_epoch(p.d_misc, st));   // the next pass's; then the decompress kernel advances it
    p.epoch_used = false;
    if (!p.items.empty())
        BATCH_HIP(hipMemcpyAsync(p.d_items, p.items.data(), p.items.size() * sizeof(Item), hipMemcpyHostToDevice, st));
    BATCH_HIP(hipStreamSynchronize(st));   // the host table may be rebuilt right after
    p.built = true;
    return CUSZP_SUCCESS;
}

// A new epoch where the last one was used up by a call that failed halfway: the
// next pass would take that call's status words for its own.
int renew_epoch(cuszp_batch_plan_s& p, hipStream_t st) {
    if (!p.epoch_used) return CUSZP_SUCCESS;
    BATCH_HIP(launch_bump_epoch(p.d_misc, st));
    p.epoch_used = false;
    return CUSZP_SUCCESS;
}

int enqueue(cuszp_batch_plan_s& p, hipStream_t st) {
    if (p.items.empty()) return CUSZP_SUCCESS;
    // the kernels read the epoch word for the tag
    const ScanCtx sc = make_scan_ctx(p.d_status + kStatusGuard, (unsigned int*)(p.d_misc + kMiscErr),
                                     p.d_misc + kMiscDiag, 0, p.h_res);
    const uint32_t n = (uint32_t)p.items.size();
    if (p.dir == CUSZP_BATCH_COMPRESS) {
        BATCH_HIP(launch_bump_epoch(p.d_misc, st));
        BATCH_HIP(launch_compress_batch(p.waves, p.window, p.d_items, n, p.ntiles, sc, p.d_misc, st));
        return CUSZP_SUCCESS;
    }
    if (p.nseg) {
        const int rc = renew_epoch(p, st);
        if (rc) return rc;
        p.epoch_used = true;
        BATCH_HIP(launch_offsets_batch(p.waves, p.d_items, n, p.nseg, p.d_offs, sc, p.d_misc, st));
    }
    BATCH_HIP(launch_decompress_batch(p.waves, p.d_items, n, p.ntiles, p.nseg ? p.d_offs : nullptr,
                                      p.nseg ? p.d_misc : nullptr, st));
    p.epoch_used = false;
    return CUSZP_SUCCESS;
}

void drop_graph(cuszp_batch_plan_s& p) {
    if (p.exec) hipGraphExecDestroy(p.exec);
    if (p.graph) hipGraphDestroy(p.graph);
    p.exec = nullptr;
    p.graph = nullptr;
}

int capture(cuszp_batch_plan_s& p) {
    drop_graph(p);
    if (!p.cap_stream) BATCH_HIP(hipStreamCreateWithFlags(&p.cap_stream, hipStreamNonBlocking));
    BATCH_HIP(hipStreamBeginCapture(p.cap_stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue(p, p.cap_stream);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(p.cap_stream, &g);
    if (rc) {
        if (g) hipGraphDestroy(g);
        return rc;
    }
    BATCH_HIP(e);
    p.graph = g;
    BATCH_HIP(hipGraphInstantiate(&p.exec, p.graph, nullptr, nullptr, 0));
    return CUSZP_SUCCESS;
}

// Launch shapes chosen by the tuner, by direction and size class of the batch
// (log2 of its tile count and of its array count); later plans of the same
// class start from the recorded shape.
std::mutex g_tune_mu;
std::map<std::tuple<int, int, int>, std::tuple<int, int, int>> g_tuned;   // -> (waves per workgroup, chunks per wave, lookback window)

std::tuple<int, int, int> size_class(const cuszp_batch_plan_s& p) {
    uint64_t bytes = 0;
    for (const auto& s : p.src) bytes += s.nbEle * (s.type == CUSZP_TYPE_FLOAT ? 4 : 8);
    int lb = 0, lc = 0;
    while ((bytes >> lb) > 1) ++lb;
    while ((p.src.size() >> lc) > 1) ++lc;
    return std::make_tuple(p.dir, lb, lc);
}

}  // namespace

extern "C" {

int cuSZp_batch_plan_create(cuszp_batch_plan_t* out, const cuszp_batch_item_t* items, size_t count, int direction,
                            int flags, hipStream_t stream, size_t* bad_index) {
    if (!out) return CUSZP_ERROR_INVALID_ARGUMENT;
    *out = nullptr;
    if ((direction != CUSZP_BATCH_COMPRESS && direction != CUSZP_BATCH_DECOMPRESS) || (count && !items) ||
        count > 0xffffffffull)
        return CUSZP_ERROR_INVALID_ARGUMENT;
    bool pass = false;
    for (size_t i = 0; i < count; ++i) {
        Geom g;
        const int rc = check_item(items[i], direction, g);
        if (rc) {
            if (bad_index) *bad_index = i;
            return rc;
        }
        pass |= direction == CUSZP_BATCH_DECOMPRESS && g.H > kBatchDirectHeader;
    }
    cuszp_batch_plan_s* p = new cuszp_batch_plan_s();
    p->dir = direction;
    p->flags = flags;
    p->src.assign(items, items + count);
    int rc = CUSZP_SUCCESS;
    if (hipGetDevice(&p->dev) != hipSuccess) rc = CUSZP_ERROR_HIP;
    p->pass = pass;
    choose_shape(*p);
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        auto f = g_tuned.find(size_class(*p));
        if (f != g_tuned.end()) {
            std::tie(p->waves, p->kc, p->window) = f->second;
            if (p->pass) p->kc = std::max(p->kc, 4);
        }
    }
    if (!rc && hipMalloc((void**)&p->d_misc, kMiscWords * sizeof(unsigned long long)) != hipSuccess) rc = CUSZP_ERROR_HIP;
    const size_t n = count ? count : 1;
    if (!rc && hipMalloc((void**)&p->d_err, n * sizeof(unsigned int)) != hipSuccess) rc = CUSZP_ERROR_HIP;
    if (!rc && hipMalloc((void**)&p->d_sizes, n * sizeof(unsigned long long)) != hipSuccess) rc = CUSZP_ERROR_HIP;
    if (!rc && !(p->h_res = take_words(p->dev, 1 + n))) rc = CUSZP_ERROR_HIP;
    if (!rc && hipMemsetAsync(p->d_misc, 0, kMiscWords * sizeof(unsigned long long), stream) != hipSuccess)
        rc = CUSZP_ERROR_HIP;
    if (!rc && hipMemsetAsync(p->d_err, 0, n * sizeof(unsigned int), stream) != hipSuccess) rc = CUSZP_ERROR_HIP;
    if (!rc && hipMemsetAsync(p->d_sizes, 0, n * sizeof(unsigned long long), stream) != hipSuccess) rc = CUSZP_ERROR_HIP;
    if (!rc) rc = build_table(*p, stream);
    if (!rc && (flags & CUSZP_BATCH_TUNE)) rc = cuSZp_batch_plan_tune(p, stream, nullptr, nullptr);
    if (!rc && (flags & CUSZP_BATCH_GRAPH) && !p->exec) rc = capture(*p);
    if (rc) {
        cuSZp_batch_plan_destroy(p);
        return rc;
    }
    *out = p;
    return CUSZP_SUCCESS;
}

int cuSZp_batch_plan_execute(cuszp_batch_plan_t p, hipStream_t stream) {
    if (!p) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (!p->built) return CUSZP_ERROR_HIP;   // tuning ran out of memory, and so did going back
    if (p->exec) {
        const int rc = renew_epoch(*p, stream);
        if (rc) return rc;
        p->epoch_used = p->nseg != 0;   // until the launch has succeeded
        BATCH_HIP(hipGraphLaunch(p->exec, stream));
        p->epoch_used = false;
        return CUSZP_SUCCESS;
    }
    return enqueue(*p, stream);
}

int cuSZp_batch_plan_results(cuszp_batch_plan_t p, size_t* cmpSizes, int* statuses, hipStream_t stream) {
    if (!p) return CUSZP_ERROR_INVALID_ARGUMENT;
    const size_t n = p->src.size();
    // lengths are read where the kernels left them; the error words only if one
    // has a bit set (three copies of pageable memory and a second synchronisation
    // took 30-40 us per call of 256 arrays)
    BATCH_HIP(hipStreamSynchronize(stream));
    volatile unsigned long long* const h = p->h_res;
    if (!h[0]) {
        for (size_t i = 0; i < n; ++i) {
            if (statuses) statuses[i] = CUSZP_SUCCESS;
            if (cmpSizes) cmpSizes[i] = (size_t)h[1 + i];
        }
        return CUSZP_SUCCESS;
    }
    h[0] = 0;   // before the words are read: a bit set later marks again
    std::vector<unsigned long long> sizes(n ? n : 1);
    std::vector<unsigned int> errs(n ? n : 1);
    unsigned long long misc[kMiscWords];
    BATCH_HIP(hipMemcpyAsync(misc, p->d_misc, sizeof(misc), hipMemcpyDeviceToHost, stream));
    BATCH_HIP(hipMemcpyAsync(errs.data(), p->d_err, errs.size() * sizeof(unsigned int), hipMemcpyDeviceToHost, stream));
    BATCH_HIP(hipMemcpyAsync(sizes.data(), p->d_sizes, sizes.size() * sizeof(unsigned long long),
                             hipMemcpyDeviceToHost, stream));
    BATCH_HIP(hipStreamSynchronize(stream));
    const unsigned long long launch_bits = misc[kMiscErr] & 0xffffffffull;
    p->info |= (unsigned)(launch_bits & kInfoStolen);
    if (launch_bits & kErrStall)
        std::fprintf(stderr, "cuSZp: internal error: batched tile %llu stopped waiting for tile %llu\n", misc[4] - 1,
                     misc[5]);
    int first = CUSZP_SUCCESS;
    for (size_t i = 0; i < n; ++i) {
        const int st = status_from_bits(errs[i] | (launch_bits & kErrStall));
        if (statuses) statuses[i] = st;
        if (cmpSizes) cmpSizes[i] = (p->dir == CUSZP_BATCH_COMPRESS && status_delivers(st)) ? (size_t)sizes[i] : 0;
        if (st && !first) first = st;
    }
    if (launch_bits) {
        BATCH_HIP(hipMemsetAsync(p->d_misc + kMiscErr, 0, (kMiscCounters - kMiscErr) * sizeof(unsigned long long),
                                 stream));
    }
    if (first) BATCH_HIP(hipMemsetAsync(p->d_err, 0, (n ? n : 1) * sizeof(unsigned int), stream));
    BATCH_HIP(hipStreamSynchronize(stream));
    return first;
}

const unsigned long long* cuSZp_batch_plan_device_sizes(cuszp_batch_plan_t p) { return p ? p->d_sizes : nullptr; }

int cuSZp_batch_plan_scan_report(cuszp_batch_plan_t p, hipStream_t stream, cuszp_scan_report_t* report) {
    if (!p || !report) return CUSZP_ERROR_INVALID_ARGUMENT;
    std::memset(report, 0, sizeof(*report));
    unsigned long long misc[kMiscWords];
    BATCH_HIP(hipMemcpyAsync(misc, p->d_misc, sizeof(misc), hipMemcpyDeviceToHost, stream));
    BATCH_HIP(hipStreamSynchronize(stream));
    report->info = p->info | (unsigned)(misc[kMiscErr] & kInfoStolen);
    report->polls = misc[kMiscCounters + 0];
    report->waits = misc[kMiscCounters + 1];
    report->claims = misc[kMiscCounters + 2];
    report->wait_ticks = misc[kMiscCounters + 3];
    p->info = 0;
    BATCH_HIP(hipMemsetAsync(p->d_misc + kMiscCounters, 0, 4 * sizeof(unsigned long long), stream));
    BATCH_HIP(hipStreamSynchronize(stream));
    return CUSZP_SUCCESS;
}

}  // extern "C"

namespace {

// Times the plan in each shape and leaves it in the best one, on record for its size
// class. A failure leaves it in the shape that failed, perhaps without a table.
int try_shapes(cuszp_batch_plan_s* p, hipStream_t stream) {
    // (waves, chunks, window): the rule's shape, then full waves; decompress tiles do not look back
    std::vector<std::tuple<int, int, int>> shapes;
    choose_shape(*p);
    shapes.emplace_back(p->waves, p->kc, kLookbackWords);
    for (int window : {kLookbackWords, 2})
        for (int waves : {4, 8})
            if (window == kLookbackWords || p->dir == CUSZP_BATCH_COMPRESS) shapes.emplace_back(waves, kChunksOf<float>, window);
    hipEvent_t e0, e1;
    BATCH_HIP(hipEventCreate(&e0));
    BATCH_HIP(hipEventCreate(&e1));
    float best = 1e30f;
    std::tuple<int, int, int> best_shape = shapes[0];
    int rc = CUSZP_SUCCESS;
    for (const auto& shape : shapes) {
        std::tie(p->waves, p->kc, p->window) = shape;
        rc = build_table(*p, stream);
        if (rc) break;
        rc = enqueue(*p, stream);   // warm-up
        if (rc) break;
        hipEventRecord(e0, stream);
        for (int r = 0; r < 3 && !rc; ++r) rc = enqueue(*p, stream);
        hipEventRecord(e1, stream);
        if (rc || hipEventSynchronize(e1) != hipSuccess) {
            rc = rc ? rc : CUSZP_ERROR_HIP;
            break;
        }
        float ms = 0;
        hipEventElapsedTime(&ms, e0, e1);
        if (ms < best) {
            best = ms;
            best_shape = shape;
        }
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    if (rc) return rc;
    std::tie(p->waves, p->kc, p->window) = best_shape;
    rc = build_table(*p, stream);
    if (rc) return rc;
    {
        std::lock_guard<std::mutex> lk(g_tune_mu);
        g_tuned[size_class(*p)] = best_shape;
    }
    return CUSZP_SUCCESS;
}

}  // namespace

extern "C" {

int cuSZp_batch_plan_tune(cuszp_batch_plan_t p, hipStream_t stream, int* waves_out, unsigned* grid_out) {
    if (!p) return CUSZP_ERROR_INVALID_ARGUMENT;
    if (p->built && p->items.empty()) return CUSZP_SUCCESS;
    // a graph's kernels hold the present buffers, which a larger shape replaces
    BATCH_HIP(hipStreamSynchronize(stream));
    drop_graph(*p);
    const auto before = std::make_tuple(p->waves, p->kc, p->window);
    int rc = try_shapes(p, stream);
    if (rc) {   // back to the shape that worked, with whatever memory there is
        std::tie(p->waves, p->kc, p->window) = before;
        if (!build_table(*p, stream) && (p->flags & CUSZP_BATCH_GRAPH)) (void)capture(*p);
        return rc;
    }
    if (p->flags & CUSZP_BATCH_GRAPH) rc = capture(*p);
    // tuning runs leave per-array state from the candidate launches: clear it
    const size_t n = p->src.size() ? p->src.size() : 1;
    if (!rc && hipMemsetAsync(p->d_err, 0, n * sizeof(unsigned int), stream) != hipSuccess) rc = CUSZP_ERROR_HIP;
    if (!rc && hipMemsetAsync(p->d_misc + kMiscErr, 0, (kMiscWords - kMiscErr) * sizeof(unsigned long long),
                              stream) != hipSuccess)
        rc = CUSZP_ERROR_HIP;
    if (waves_out) *waves_out = p->waves;
    if (grid_out) *grid_out = (unsigned)(p->ntiles < kMaxGrid ? p->ntiles : kMaxGrid);
    return rc;
}

void cuSZp_batch_plan_destroy(cuszp_batch_plan_t p) {
    if (!p) return;
    drop_graph(*p);
    if (p->cap_stream) {
        hipStreamSynchronize(p->cap_stream);
        hipStreamDestroy(p->cap_stream);
    }
    int dev = p->dev;
    hipGetDevice(&dev);
    if (dev != p->dev) hipSetDevice(p->dev);
    const bool idle = hipDeviceSynchronize() == hipSuccess;   // no launch of this plan may still use its buffers
    if (p->d_items) hipFree(p->d_items);
    if (p->d_status) hipFree(p->d_status);
    if (p->d_offs) hipFree(p->d_offs);
    if (p->d_misc) hipFree(p->d_misc);
    if (p->d_err) hipFree(p->d_err);
    if (p->d_sizes) hipFree(p->d_sizes);
    return_words(p->dev, p->h_res, 1 + (p->src.empty() ? 1 : p->src.size()), idle);
    if (dev != p->dev) hipSetDevice(dev);
    delete p;
}

int cuSZp_compress_batch(const cuszp_batch_item_t* items, size_t count, size_t* cmpSizes, int* statuses,
                         hipStream_t stream) {
    cuszp_batch_plan_t p = nullptr;
    int rc = cuSZp_batch_plan_create(&p, items, count, CUSZP_BATCH_COMPRESS, 0, stream, nullptr);
    if (rc) return rc;
    rc = cuSZp_batch_plan_execute(p, stream);
    if (!rc) rc = cuSZp_batch_plan_results(p, cmpSizes, statuses, stream);
    cuSZp_batch_plan_destroy(p);
    return rc;
}

int cuSZp_decompress_batch(const cuszp_batch_item_t* items, size_t count, int* statuses, hipStream_t stream) {
    cuszp_batch_plan_t p = nullptr;
    int rc = cuSZp_batch_plan_create(&p, items, count, CUSZP_BATCH_DECOMPRESS, 0, stream, nullptr);
    if (rc) return rc;
    rc = cuSZp_batch_plan_execute(p, stream);
    if (!rc) rc = cuSZp_batch_plan_results(p, nullptr, statuses, stream);
    cuSZp_batch_plan_destroy(p);
    return rc;
}

}  // extern "C"
