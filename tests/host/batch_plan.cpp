// Host program for the batched plans: cuszp_batch.cpp over a HIP runtime and kernel
// launches that are replaced here by host memory and a log. It shows what the
// plan launches when a launch or an allocation fails, which needs no GPU.
//   batch_plan epoch   a decode launch that fails after its offset pass
//   batch_plan words   pinned result words that outlive their plan
//   batch_plan tune [graph], tune-lost [graph]
//                      an allocation that fails while shapes are tried, and again when the former one is restored
#include "../../cuszp_amd/csrc/cuszp_batch.cpp"

#include <cstdlib>
#include <string>

namespace {
std::vector<std::string> g_log;      // one entry per launch
std::vector<unsigned long long> g_pass_epochs;
int g_fail_decodes = 0;              // decode launches that fail
bool g_null = false;                 // a launch was given no buffer
int g_graphs = 0, g_captured = 0;
int g_pinned = 0, g_pinned_allocs = 0;   // pinned buffers alive, and ever allocated
int g_device = 0, g_synced = -1;     // the current device, and the last one that was synchronised
bool g_idle = true;                  // whether the device can be synchronised

#define CHECK(x)                                                    \
    do {                                                            \
        if (!(x)) {                                                 \
            std::printf("line %d: %s\n", __LINE__, #x);             \
            std::exit(1);                                           \
        }                                                           \
    } while (0)

void seen(const char* what, const void* items, const void* status, const void* offs) {
    g_log.push_back(what);
    g_null |= !items || status == (const unsigned long long*)nullptr + kStatusGuard || !offs;
}
}  // namespace

// ---- the runtime -----------------------------------------------------------
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return *p = std::calloc(n ? n : 1, 1), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return ++g_pinned, ++g_pinned_allocs, hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return --g_pinned, hipFree(p); }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = g_device, hipSuccess; }
hipError_t hipSetDevice(int d) { return g_device = d, hipSuccess; }
hipError_t hipDeviceSynchronize() { return g_synced = g_device, g_idle ? hipSuccess : hipErrorLaunchFailure; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return ++g_captured, *e = (hipGraphExec_t)1, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return ++g_graphs, hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 1.0f, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}

// ---- the launches ----------------------------------------------------------
namespace cuszp {
hipError_t launch_bump_epoch(unsigned long long* epoch, hipStream_t) { return ++*epoch, hipSuccess; }
hipError_t launch_compress_batch(int, int, const Item* items, uint32_t, uint64_t, const ScanCtx& sc, const unsigned long long*, hipStream_t) {
    return seen("compress", items, sc.status, items), hipSuccess;
}
hipError_t launch_offsets_batch(int, const Item* items, uint32_t, uint64_t, unsigned long long* offs, const ScanCtx& sc,
                                const unsigned long long* epoch, hipStream_t) {
    g_pass_epochs.push_back(*epoch);
    return seen("pass", items, sc.status, offs), hipSuccess;
}
hipError_t launch_decompress_batch(int, const Item* items, uint32_t, uint64_t, const unsigned long long* offs, unsigned long long* bump,
                                   hipStream_t) {
    if (g_fail_decodes && g_fail_decodes--) return hipErrorLaunchFailure;
    if (bump) ++*bump;
    return seen("decode", items, items, offs), hipSuccess;
}
}  // namespace cuszp

namespace {
char g_buf[8];   // arrays' addresses are not followed

// 4 Mi values: a header of 128 KiB, long enough for the offset pass. 16 Mi: 512
// tiles, of which the shapes of four waves make 1024
cuszp_batch_plan_t plan(int dir, size_t n = 4u << 20, int flags = 0) {
    cuszp_batch_item_t it{};
    it.d_in = g_buf;
    it.d_out = g_buf;
    it.nbEle = n;
    it.capacity = 1ull << 30;
    it.errorBound = 1e-3;
    it.dim = CUSZP_DIM_1D;
    it.type = CUSZP_TYPE_FLOAT;
    it.mode = CUSZP_MODE_PLAIN;
    cuszp_batch_plan_t p = nullptr;
    CHECK(cuSZp_batch_plan_create(&p, &it, 1, dir, flags, nullptr, nullptr) == CUSZP_SUCCESS);
    return p;
}

void epoch() {
    cuszp_batch_plan_t p = plan(CUSZP_BATCH_DECOMPRESS);
    CHECK(cuSZp_batch_plan_execute(p, nullptr) == CUSZP_SUCCESS);
    for (int k = 0; k < 2; ++k) {
        g_fail_decodes = 1;
        CHECK(cuSZp_batch_plan_execute(p, nullptr) == CUSZP_ERROR_HIP);
        CHECK(cuSZp_batch_plan_execute(p, nullptr) == CUSZP_SUCCESS);
    }
    CHECK(g_pass_epochs.size() == 5);
    for (size_t i = 0; i < 5; ++i)
        for (size_t j = 0; j < i; ++j) CHECK(g_pass_epochs[i] != g_pass_epochs[j]);   // no pass reads another's words as its own
    cuSZp_batch_plan_destroy(p);
}

// fails: status arrays that cannot be allocated while the shapes are tried
void tune(int flags, unsigned fails) {
    cuszp_batch_plan_t p = plan(CUSZP_BATCH_COMPRESS, 16u << 20, flags);
    CHECK(cuSZp_batch_plan_execute(p, nullptr) == CUSZP_SUCCESS);
    failing_allocs().store(fails);
    CHECK(cuSZp_batch_plan_tune(p, nullptr, nullptr, nullptr) == CUSZP_ERROR_HIP);
    failing_allocs().store(0);
    const size_t launches = g_log.size();
    const int graphs = g_graphs, rc = cuSZp_batch_plan_execute(p, nullptr);
    CHECK(!g_null);
    if (fails == 1) {   // the shape from before is there again, and so is its graph
        CHECK(rc == CUSZP_SUCCESS);
        CHECK(p->waves == 8 && p->ntiles == 512);
        CHECK(flags ? g_graphs == graphs + 1 && p->exec : g_log.size() == launches + 1);
        if (flags) CHECK(g_captured == 2);
    } else {            // no table: nothing is launched
        CHECK(rc == CUSZP_ERROR_HIP);
        CHECK(g_log.size() == launches && g_graphs == graphs);
    }
    CHECK(cuSZp_batch_plan_tune(p, nullptr, nullptr, nullptr) == CUSZP_SUCCESS);
    CHECK(cuSZp_batch_plan_execute(p, nullptr) == CUSZP_SUCCESS);
    CHECK(!g_null);
    cuSZp_batch_plan_destroy(p);
}

// n arrays of one value
cuszp_batch_plan_t plan_of(size_t n) {
    cuszp_batch_item_t it{};
    it.d_in = it.d_out = g_buf;
    it.nbEle = 1;
    it.capacity = 1 << 20;
    it.errorBound = 1e-3;
    it.dim = CUSZP_DIM_1D;
    it.type = CUSZP_TYPE_FLOAT;
    it.mode = CUSZP_MODE_PLAIN;
    std::vector<cuszp_batch_item_t> items(n, it);
    cuszp_batch_plan_t p = nullptr;
    CHECK(cuSZp_batch_plan_create(&p, items.data(), n, CUSZP_BATCH_COMPRESS, 0, nullptr, nullptr) == CUSZP_SUCCESS);
    for (size_t i = 0; i <= n; ++i) CHECK(p->h_res[i] == 0);   // nothing of a plan before
    std::memset(p->h_res, 0xff, (n + 1) * sizeof(*p->h_res));   // as its kernels would
    return p;
}

// Pinned words outlive their plan, a bounded number of them.
void words() {
    for (int k = 0; k < 20; ++k) cuSZp_batch_plan_destroy(plan_of(1 + 300 * k));
    CHECK(g_pinned_allocs == 1);
    std::vector<cuszp_batch_plan_t> many;
    for (int k = 0; k < 10; ++k) many.push_back(plan_of(3));
    for (size_t i = 0; i < many.size(); ++i)
        for (size_t j = 0; j < i; ++j) CHECK(many[i]->h_res != many[j]->h_res);
    for (auto p : many) cuSZp_batch_plan_destroy(p);
    CHECK(g_pinned == (int)kKeptBuffers);
    cuSZp_batch_plan_destroy(plan_of(kKeptWords - 1));   // the most that fits
    CHECK(g_pinned == (int)kKeptBuffers && g_pinned_allocs == 10);
    cuSZp_batch_plan_destroy(plan_of(kKeptWords));       // one more: its own buffer, freed with it
    CHECK(g_pinned == (int)kKeptBuffers && g_pinned_allocs == 11);
    cuSZp_batch_plan_destroy(plan_of(0));
    // a plan is finished on its own device, and its words stay there
    cuszp_batch_plan_t p = plan_of(3);
    unsigned long long* const w = p->h_res;
    g_device = 1;
    cuSZp_batch_plan_destroy(p);
    CHECK(g_synced == 0 && g_device == 1);
    p = plan_of(3);
    CHECK(p->h_res != w);
    // kernels may still write: not kept
    g_idle = false;
    const int alive = g_pinned;
    cuSZp_batch_plan_destroy(p);
    CHECK(g_pinned == alive - 1);
}
}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "epoch") epoch();
    else if (what == "tune") tune(argc > 2 ? CUSZP_BATCH_GRAPH : 0, 1);
    else if (what == "tune-lost") tune(argc > 2 ? CUSZP_BATCH_GRAPH : 0, 2);
    else if (what == "words") words();
    else return 2;
    std::puts("ok");
    return 0;
}
