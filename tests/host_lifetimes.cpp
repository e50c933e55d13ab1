// Host check of the lifetimes that csrc/serve.cpp and csrc/batch.cpp keep:
// both are compiled here against a stand-in for the HIP runtime and for the
// rest of the library, which runs nothing but knows its streams and events.
//   - an event is used and destroyed before the stream it was last recorded
//     on (the runtime reads that stream);
//   - a request that completes at once is not read by the call that
//     submitted it (the thread sanitizer sees it).
#include <cstdio>
#include <cstdlib>
#include <set>

#include "serve.cpp"
#include "batch.cpp"

static std::recursive_mutex g_hip;
#define HIP_LOCK std::lock_guard<std::recursive_mutex> hip_lock(g_hip)
struct Event {
    hipStream_t last = nullptr;
    bool captured = false;
};
static std::set<hipStream_t> g_live_streams;
static std::set<Event *> g_live_events;
static hipStream_t g_capturing = nullptr;
static int g_bad = 0;

static void expect(bool ok, const char *what)
{
    if (ok) return;
    std::fprintf(stderr, "%s\n", what);
    ++g_bad;
}
static void stream_ok(hipStream_t s) { expect(s == nullptr || g_live_streams.count(s), "use of a destroyed stream"); }
static Event *event(hipEvent_t e)
{
    expect(g_live_events.count((Event *) e), "use of a destroyed event");
    if (g_live_events.count((Event *) e)) {
        const hipStream_t last = ((Event *) e)->last;
        expect(last == nullptr || g_live_streams.count(last), "event outlives the stream it was recorded on");
    }
    return (Event *) e;
}

extern "C" {
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::calloc(n, 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    HIP_LOCK;
    stream_ok(st);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    HIP_LOCK;
    stream_ok(st);
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorName(hipError_t) { return ""; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    HIP_LOCK;
    *s = (hipStream_t) new char[1];   // never reused, so a stale handle is seen
    g_live_streams.insert(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    HIP_LOCK;
    stream_ok(s);
    g_live_streams.erase(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    HIP_LOCK;
    stream_ok(s);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    HIP_LOCK;
    Event *x = new Event();
    g_live_events.insert(x);
    *e = (hipEvent_t) x;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    HIP_LOCK;
    g_live_events.erase(event(e));
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    HIP_LOCK;
    event(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    HIP_LOCK;
    stream_ok(s);
    expect(g_live_events.count((Event *) e), "record of a destroyed event");
    ((Event *) e)->last = s;
    ((Event *) e)->captured = g_capturing != nullptr;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    HIP_LOCK;
    stream_ok(s);
    event(e);
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
    HIP_LOCK;
    g_capturing = s;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    HIP_LOCK;
    g_capturing = nullptr;
    for (Event *e : g_live_events)   // what a capture recorded is nothing afterwards
        if (e->captured) e->last = nullptr;
    *g = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

namespace imr {
std::atomic<bool> g_use_graphs{true};
thread_local ProfEvents g_prof;
int current_device(int *d) { *d = 0; return IMRESH_OK; }
bool line_supported(int n) { return n >= 1; }
int normalize(const imresh_params *p, Params &q)
{
    q.n_cycles = p->n_cycles;
    q.n_hio = p->n_hio_cycles;
    return IMRESH_OK;
}
int padded_weights(const Params &, std::vector<float> &rows, int *R) { rows.assign(64, 0.f); *R = 1; return IMRESH_OK; }
size_t pool_cap() { return (size_t) 1 << 30; }
size_t ws_bytes(int, int) { return 4096; }
int ws_alloc(int, int W, int H, Workspace **w)
{
    *w = new Workspace();
    (*w)->W = W;
    (*w)->H = H;
    (*w)->n = (size_t) W * H;
    return IMRESH_OK;
}
void ws_release(Workspace *w) { delete w; }
int ws_tune(Workspace *, hipStream_t) { return IMRESH_OK; }
int tune_size(int, int, int, hipStream_t) { return IMRESH_OK; }
int recon_begin(Workspace *, const float *, const Params &, hipStream_t) { return IMRESH_OK; }
int recon_cycle(Workspace *, const float *, const Params &, unsigned, hipStream_t) { return IMRESH_OK; }
int recon_end(Workspace *, float *, hipStream_t) { return IMRESH_OK; }
int recon_stage_results(Workspace *, hipStream_t) { return IMRESH_OK; }
void recon_read_staged(const Workspace *, imresh_result *, int *) {}
int get_plan2d(int, int W, int H, Plan2D *p) { *p = Plan2D{}; p->W = W; p->H = H; return IMRESH_OK; }
int blur_grid(int, int) { return 1; }
int row_grid(const Plan2D &p) { return p.H; }
int prepare_blur(int) { return IMRESH_OK; }
int launch_blur(const BlurArgs &, hipStream_t) { return IMRESH_OK; }
int launch_row(int, const Plan2D &, RowArgs, hipStream_t) { return IMRESH_OK; }
int launch_col(int, const Plan2D &, ColArgs, hipStream_t) { return IMRESH_OK; }
int launch_max_finalize_batch(const float *, int, float, float, float *, int *, int, hipStream_t) { return IMRESH_OK; }
int launch_err_finalize_batch(const float *, const unsigned *, int, float, float *, int *, int, hipStream_t) { return IMRESH_OK; }
int launch_gather_images(float *, const float *const *, size_t, int, hipStream_t) { return IMRESH_OK; }
int launch_scatter_real(float *const *, const float2 *, size_t, int, hipStream_t) { return IMRESH_OK; }
int launch_copy_from_real(float *, const float2 *, size_t, hipStream_t) { return IMRESH_OK; }
}  // namespace imr

static void batches()
{
    imresh_params p{};
    p.n_cycles = 2;
    p.n_hio_cycles = 1;
    for (int graphs = 0; graphs < 2; ++graphs) {
        imr::g_use_graphs = graphs != 0;
        for (int host = 0; host < 2; ++host) {
            std::vector<std::vector<float>> mem;
            std::vector<imresh_image> im;
            for (uint32_t n : {4u, 6u, 4u, 8u, 5u}) {
                mem.emplace_back((size_t) n * n, 1.f);
                im.push_back({mem.back().data(), n, n});
            }
            std::vector<imresh_result> res(im.size());
            for (int rep = 0; rep < 3; ++rep) {
                const int st = host ? imresh_shrinkwrap_batch(im.data(), (uint32_t) im.size(), &p, nullptr, res.data())
                                    : imresh_shrinkwrap_batch_device(im.data(), (uint32_t) im.size(), &p, nullptr,
                                                                     rep ? res.data() : nullptr);
                expect(st == IMRESH_OK, "batch status");
            }
        }
        imr::trim_idle_classes(0);
    }
    expect(imr::idle_class_bytes() == 0, "idle bytes after the release");
}

static void requests()
{
    imresh_params p{};
    p.n_cycles = 1;
    p.n_hio_cycles = 1;
    imresh_server *s = nullptr;
    expect(imresh_server_create(0, 0, 2, &s) == IMRESH_OK, "server");
    float x[16] = {};
    for (uint64_t i = 1; i <= 300; ++i) {
        uint64_t id = 0;
        expect(imresh_server_submit(s, x, 4, 4, &p, 1, nullptr, nullptr, &id) == IMRESH_OK && id == i, "submit");
        if (i % 10 == 0) imresh_server_drain(s);
    }
    imresh_server_destroy(s);
}

int main()
{
    batches();
    requests();
    std::printf("%d lifetime errors\n", g_bad);
    return g_bad != 0;
}
