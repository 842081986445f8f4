// The engine's host path over a HIP runtime of its own: this program defines the
// runtime's functions (the library's calls bind to them), keeps device memory on
// the heap, and runs, in place of the kernels, what they do to a scene's clock.
// What the host enqueues can then be followed without a GPU: which kernels, on
// which stream and device, under capture or not, over which memory.
//
// usage: host_runtime SCENARIO   (prints what went wrong; exit status 0 if nothing)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../acoustics_amd/csrc/engine.h"
#include "../../acoustics_amd/csrc/resident.h"
#include "fdtd_acoustics.h"

using namespace fdtd;

// ---------------------------------------------------------------------------
// the runtime
// ---------------------------------------------------------------------------
namespace {

struct Stream {
    int dev = 0;
    bool capturing = false;
    std::vector<std::function<void()>> graph;
};
struct Event {
    int dev = 0;
    Stream *on = nullptr;
};
struct Call {
    std::string what;           // kernel name, "record" or "wait"
    Stream *stream;
    bool captured;
    const void *scene;          // resident_kernel: one entry per scene of the launch
};

std::recursive_mutex g_mu;
int g_bad = 0;
std::vector<Call> g_log;
thread_local int t_dev = 0;
thread_local hipError_t t_error = hipSuccess;

void bad(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    std::printf("FAULT: ");
    std::vprintf(fmt, ap);
    std::printf("\n");
    va_end(ap);
    ++g_bad;
}
#define CHECK(c) do { if (!(c)) bad("%s:%d: %s (%s)", __FILE__, __LINE__, #c, fdtd_last_error()); } while (0)

std::map<const void *, std::string> &kernels()
{
    static std::map<const void *, std::string> k;
    return k;
}
struct Block { size_t n; int dev; };
std::map<char *, Block> g_mem;
long g_fail_malloc = -1;        // device allocations left before one fails (-1: none does)
bool g_fail_pinned = false;
int g_patience = 0;             // the last resident launch's wait limit

// what the resident kernel does
std::function<bool(const SceneDev &)> g_gives_up = [](const SceneDev &) { return false; };
std::function<double(const SceneDev &, long long)> g_signal = [](const SceneDev &, long long) { return 1.0; };

bool live(const void *p, size_t n = 1)
{
    auto it = g_mem.upper_bound((char *)p);
    if (it == g_mem.begin()) return false;
    --it;
    return (char *)p + n <= it->first + it->second.n;
}

// scenes whose clock has been seen
std::map<const void *, SceneDev> g_scenes;

void run_advance(const SceneDev *scenes, int count, int n)
{
    for (int i = 0; i < count; ++i) {
        const SceneDev &S = scenes[i];
        g_scenes[S.clock] = S;
        unsigned long long *c = S.clock;
        if ((long long)c[CLK_STEP] >= (long long)c[CLK_TARGET]) continue;
        c[CLK_STEP] = (unsigned long long)std::min((long long)c[CLK_STEP] + n, (long long)c[CLK_TARGET]);
        c[CLK_ARRIVED] = 0;
        c[CLK_GATE] = GATE_SHUT;
    }
}

void write_rows(const SceneDev &S, long long from, long long to)
{
    for (long long s = from; s < to; ++s)
        for (int q = 0; q < S.T; ++q) S.terms[(size_t)(s % S.cap) * S.T + q] = g_signal(S, s);
}

std::vector<const ResScene *> scenes_of(const ResItem *items, int n)
{
    std::vector<const ResScene *> out;
    if (!live(items, sizeof(ResItem) * (size_t)n)) { bad("a resident launch over memory that is not there"); return out; }
    for (int q = 0; q < n; ++q) {
        const ResScene *r = items[q].scene;
        if (!r || (!out.empty() && out.back() == r)) continue;
        if (!live(r, sizeof *r)) { bad("a resident launch lists a scene whose memory was freed"); continue; }
        out.push_back(r);
    }
    return out;
}

void run_resident(const ResItem *items, int n, int nsteps, int *trouble)
{
    for (const ResScene *r : scenes_of(items, n)) {
        const SceneDev &S = *r->S;
        unsigned long long *c = S.clock;
        const long long step = (long long)c[CLK_STEP], left = (long long)c[CLK_TARGET] - step;
        if (left <= 0) continue;
        if (c[CLK_GATE] != GATE_SHUT) bad("a scene's gate stands open before its launch (step %lld)", step);
        if (g_gives_up(S)) {
            c[CLK_GATE] = GATE_GIVEN_UP;
            c[CLK_HELD] = c[CLK_TARGET];
            c[CLK_TARGET] = (unsigned long long)step;
            *trouble = 1;
            continue;
        }
        c[CLK_GATE] = GATE_RUN;
        c[CLK_ARRIVED] = (unsigned long long)r->ntiles;
        write_rows(S, step, step + std::min<long long>(nsteps, left));
    }
}

void run_sums(const double *terms, int T, const int32_t *ptr, int L, long long rows, double *out)
{
    bool in_ring = false;
    for (const auto &e : g_scenes) {
        const SceneDev &S = e.second;
        in_ring = in_ring || (S.terms && terms >= S.terms && terms + (size_t)rows * T <= S.terms + (size_t)S.cap * S.T);
    }
    if (!in_ring) bad("listener sums over memory outside every ring");
    if (!live(terms, sizeof(double) * (size_t)rows * T)) return;
    for (long long r = 0; r < rows; ++r)
        for (int l = 0; l < L; ++l) {
            double v = 0;
            for (int q = ptr[l]; q < ptr[l + 1]; ++q) v += terms[r * T + q];
            out[r * L + l] = v;
        }
}

template <class T>
T arg(void **a, int i) { return *(T *)a[i]; }

Stream *stream_of(hipStream_t s) { return (Stream *)s; }

struct Dims { dim3 grid, block; size_t shared; hipStream_t stream; };
thread_local std::vector<Dims> t_config;

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) { static void *h = nullptr; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernels()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s)
{
    t_config.push_back({g, b, m, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s)
{
    const Dims d = t_config.back();
    t_config.pop_back();
    *g = d.grid; *b = d.block; *m = d.shared; *s = d.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **a, size_t, hipStream_t st)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    const std::string name = kernels()[f];
    Stream *s = stream_of(st);
    if (t_dev != s->dev) bad("%s launched on device %d's stream with device %d selected", name.c_str(), s->dev, t_dev);
    auto is = [&](const char *k) { return name.find(k) != std::string::npos; };
    std::function<void()> run = [] {};
    if (is("advance_kernel")) {
        const SceneDev *sc = arg<const SceneDev *>(a, 0);
        const int n = arg<int>(a, 1), count = (int)g.x;
        run = [=] { run_advance(sc, count, n); };
    } else if (is("resident_kernel")) {
        const ResItem *items = arg<const ResItem *>(a, 0);
        const int n = (int)g.x, steps = arg<int>(a, 1);
        int *trouble = arg<int *>(a, 4);
        for (const ResScene *r : scenes_of(items, n)) g_log.push_back({"resident scene", s, s->capturing, r->S->clock});
        g_patience = arg<int>(a, 3);
        if (s->capturing) bad("a resident launch is recorded in a graph");
        run = [=] { run_resident(items, n, steps, trouble); };
    } else if (is("sum_terms_kernel")) {
        run_sums(arg<const double *>(a, 0), arg<int>(a, 1), arg<const int32_t *>(a, 2), arg<int>(a, 3), (long long)(arg<long long>(a, 4) / arg<int>(a, 3)), arg<double *>(a, 5));
    }
    g_log.push_back({is("resident_kernel") ? "resident" : is("step_kernel") ? "step" : is("advance_kernel") ? "advance" : "other", s, s->capturing, nullptr});
    if (s->capturing) s->graph.push_back(run);
    else run();
    return hipSuccess;
}

hipError_t hipEventRecord(hipEvent_t e, hipStream_t s);
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t m, hipStream_t st, hipEvent_t, hipEvent_t stop, int)
{
    const hipError_t r = hipLaunchKernel(f, g, b, a, m, st);
    return r != hipSuccess || !stop ? r : hipEventRecord(stop, st);
}

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = t_dev; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_dev = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int, size_t)
{
    *n = kernels()[f].find("Li2E") != std::string::npos ? 2 : 3;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError(void) { const hipError_t e = t_error; t_error = hipSuccess; return e; }

hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    if (g_fail_malloc >= 0 && g_fail_malloc-- == 0) { *p = nullptr; return t_error = hipErrorOutOfMemory; }
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    std::memset(*p, 0, n);
    g_mem[(char *)*p] = {n, t_dev};
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    if (!p) return hipSuccess;
    auto it = g_mem.find((char *)p);
    if (it == g_mem.end()) { bad("hipFree of memory that is not there"); return hipErrorInvalidValue; }
    for (auto s = g_scenes.begin(); s != g_scenes.end();)
        s = (char *)s->first >= it->first && (char *)s->first < it->first + it->second.n ? g_scenes.erase(s) : std::next(s);
    g_mem.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (g_fail_pinned) { *p = nullptr; return t_error = hipErrorOutOfMemory; }
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind)
{
    for (size_t r = 0; r < h; ++r) std::memcpy((char *)d + r * dp, (const char *)s + r * sp, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **, const void *) { return hipErrorNotSupported; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    Stream *n = new Stream();
    n->dev = t_dev;
    *s = (hipStream_t)n;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { delete stream_of(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    return stream_of(s)->capturing ? (t_error = hipErrorStreamCaptureUnsupported) : hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c)
{
    *c = stream_of(s)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode)
{
    if (stream_of(s)->capturing) return t_error = hipErrorIllegalState;
    stream_of(s)->capturing = true;
    stream_of(s)->graph.clear();
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    stream_of(s)->capturing = false;
    *g = (hipGraph_t) new std::vector<std::function<void()>>(stream_of(s)->graph);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
    *x = (hipGraphExec_t) new std::vector<std::function<void()>>(*(std::vector<std::function<void()>> *)g);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    for (auto &f : *(std::vector<std::function<void()>> *)x) f();
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    Event *n = new Event();
    n->dev = t_dev;
    *e = (hipEvent_t)n;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    if (((Event *)e)->dev != stream_of(s)->dev) bad("an event recorded on another device's stream");
    ((Event *)e)->on = stream_of(s);
    g_log.push_back({"record", stream_of(s), stream_of(s)->capturing, nullptr});
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    const Stream *on = ((Event *)e)->on;
    if (on && on->capturing && !stream_of(s)->capturing) bad("a wait for an event of a stream under capture");
    g_log.push_back({"wait", stream_of(s), stream_of(s)->capturing, ((Event *)e)->on});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }

}  // extern "C"

// ---------------------------------------------------------------------------
// scenes and scenarios
// ---------------------------------------------------------------------------
namespace {

struct Scene {
    fdtd_scene sc{};
    fdtd_pressure_source src{};
    double ears[6];
    Scene(int nx, int ny, int nz, int pml, int scheme = FDTD_SCHEME_COLLOCATED)
    {
        fdtd_settings_default(&sc.settings);
        const int n[3] = {nx, ny, nz};
        for (int d = 0; d < 3; ++d) { sc.settings.divisions[d] = n[d]; sc.settings.min_bound[d] = -0.0025 * n[d]; }
        sc.settings.pml_width = pml;
        sc.settings.scheme = scheme;
        src.width_time = 1e-4;
        src.width_space = 0.0343;
        src.normalize_constant = 1.0;
        sc.n_pressure_sources = 1;
        sc.pressure_sources = &src;
        for (int d = 0; d < 3; ++d) { ears[d] = 0.01; ears[3 + d] = -0.012; }
        sc.n_listeners = 2;
        sc.listeners = ears;
    }
};

int count(const char *what, Stream *s = nullptr)
{
    std::lock_guard<std::recursive_mutex> lk(g_mu);
    int n = 0;
    for (const Call &c : g_log) n += c.what == what && (!s || c.stream == s);
    return n;
}
void forget() { std::lock_guard<std::recursive_mutex> lk(g_mu); g_log.clear(); }

hipStream_t new_stream()
{
    hipStream_t s;
    (void)hipStreamCreateWithFlags(&s, 0);
    return s;
}

std::vector<long long> clocks()
{
    std::vector<long long> c;
    for (const auto &e : g_scenes) c.push_back((long long)e.second.clock[CLK_STEP]);
    return c;
}

// Blocks of a batch on a captured stream are step kernels, and each replay runs them on.
void batch_capture()
{
    Scene a(48, 40, 44, 6), b(40, 40, 40, 6);
    const fdtd_scene sc[2] = {a.sc, b.sc};
    const int steps[2] = {300, 300};
    fdtd_batch_options o;
    fdtd_batch_options_default(&o);
    hipStream_t st = new_stream();
    o.stream = st;
    fdtd_batch *h = nullptr;
    CHECK(fdtd_batch_create(sc, steps, 2, &o, &h) == FDTD_OK);
    CHECK(fdtd_batch_step(h, 40) == FDTD_OK);
    CHECK(count("resident") > 0);
    forget();
    (void)hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed);
    CHECK(fdtd_batch_step(h, 20) == FDTD_OK);
    hipGraph_t g = nullptr;
    hipGraphExec_t x = nullptr;
    (void)hipStreamEndCapture(st, &g);
    (void)hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    CHECK(count("step") >= 20 && count("resident") == 0);
    for (long long c : clocks()) CHECK(c == 40);
    for (int r = 1; r <= 3; ++r) {
        (void)hipGraphLaunch(x, st);
        for (long long c : clocks()) CHECK(c == 40 + 20 * r);
    }
    CHECK(fdtd_batch_step(h, 50) == FDTD_OK);   // eager again
    for (long long c : clocks()) CHECK(c == 150);
    fdtd_batch_destroy(h);
}

// A load that finds no files leaves a staggered handle where it is.
void failed_load()
{
    Scene a(48, 40, 44, 6, FDTD_SCHEME_STAGGERED);
    fdtd_handle *h = nullptr;
    CHECK(fdtd_create(&a.sc, nullptr, &h) == FDTD_OK);
    CHECK(fdtd_step(h, 100) == FDTD_OK);
    CHECK(count("resident") == 1);
    const size_t held = g_mem.size();
    CHECK(fdtd_load_snapshot(h, "/nonexistent/%s", "0", 1) == FDTD_ERR_INVALID);
    CHECK(g_mem.size() == held);
    CHECK(fdtd_step(h, 40) == FDTD_OK);
    CHECK(count("resident") == 2);
    CHECK(clocks() == std::vector<long long>{140});
    double p[2];
    CHECK(fdtd_listen(h, p) == FDTD_OK);
    fdtd_destroy(h);
}

// A request whose first block is given up and falls on a finiteness check has no row to check yet.
void server_check()
{
    Scene a(40, 40, 40, 6), b(44, 40, 40, 6);
    fdtd_server_options o;
    fdtd_server_options_default(&o);
    o.steps_per_block = 8;
    fdtd_server *s = nullptr;
    CHECK(fdtd_server_create(&o, &s) == FDTD_OK);
    g_gives_up = [](const SceneDev &S) { return S.clock[CLK_TARGET] == 83 && S.clock[CLK_STEP] == 0; };
    int64_t id[2];
    const int steps[2] = {15 * 8, 83};   // the second one's first block is the sixteenth
    const Scene *sc[2] = {&a, &b};
    for (int q = 0; q < 2; ++q) {
        CHECK(fdtd_server_submit(s, &sc[q]->sc, steps[q], &id[q]) == FDTD_OK);
        CHECK(fdtd_server_wait(s, id[q], 60000) == FDTD_OK);
        std::vector<double> out(2 * (size_t)steps[q]);
        double ms;
        CHECK(fdtd_server_take_result(s, id[q], out.data(), &ms) == FDTD_OK);
    }
    fdtd_server_stats st;
    CHECK(fdtd_server_get_stats(s, &st) == FDTD_OK && st.completed == 2 && st.blocks_run >= 26);
    CHECK(count("resident") == 16);
    CHECK(count("step") >= 83);
    fdtd_server_destroy(s);
}

// A time chunk that is stopped early leaves the resident launches: its clock no
// longer moves, so no launch may find its gate as the one before left it.
void cut_chunk()
{
    Scene a(40, 40, 40, 6);
    fdtd_settings &s = a.sc.settings;
    s.time_parallel = 1;
    s.num_time_chunks = 4;
    const int64_t steps = 16000;            // chunks of 16000, 12000, 8000 and 4000 steps, sources in the first 4000
    s.overlap_time = 12000.5 * s.time_step;
    // the second one is quiet from step 4100 on, and stops 0.05 s (6000 steps) later
    g_signal = [](const SceneDev &S, long long step) { return S.cap == 12000 && step > 4100 ? 0.0 : 1.0; };
    std::vector<double> out((size_t)steps * 2);
    int64_t run[4];
    CHECK(fdtd_run_time_parallel(&a.sc, steps, nullptr, out.data(), run) == FDTD_OK);
    CHECK(run[0] == 16000 && run[1] > 10050 && run[1] < 10150 && run[2] == 8000 && run[3] == 4000);
    // one launch per block of 32 steps; the stopped chunk, and the finished ones,
    // are in none after the block it was stopped in
    std::map<const void *, int> launches;
    for (const Call &c : g_log)
        if (c.what == "resident scene") ++launches[c.scene];
    CHECK(launches.size() == 4);
    int all = 0;
    for (const auto &e : launches) {
        all += e.second == 500;
        CHECK(e.second == 500 || e.second <= (run[1] + 31) / 32);
    }
    CHECK(all == 1);
}

// Device memory that runs out while a batch lists its scenes anew: the call
// fails, nothing is launched over lists that are not there, and the batch goes
// on once there is memory.
void no_memory_for_lists()
{
    Scene a(40, 40, 40, 6), b(44, 40, 40, 6), c(112, 120, 128, 8);   // the third one of another tile shape
    for (int k = 0; k < 8; ++k) {
        const fdtd_scene sc[3] = {a.sc, b.sc, c.sc};
        const int steps[3] = {300, 301, 302};
        fdtd_batch *h = nullptr;
        CHECK(fdtd_batch_create(sc, steps, 3, nullptr, &h) == FDTD_OK);
        g_gives_up = [](const SceneDev &S) { return S.clock[CLK_TARGET] == 301 || S.clock[CLK_TARGET] == 302; };
        CHECK(fdtd_batch_step(h, 64) == FDTD_OK);
        double row[302 * 2];
        g_fail_malloc = k;
        const fdtd_status st = fdtd_batch_read_listener_series(h, 0, row);
        CHECK(st == FDTD_OK || st == FDTD_ERR_OOM);
        if (st == FDTD_OK) CHECK(fdtd_batch_step(h, 64) == FDTD_OK);
        else (void)fdtd_batch_step(h, 64);
        g_fail_malloc = -1;
        g_gives_up = [](const SceneDev &) { return false; };
        CHECK(fdtd_batch_run(h) == FDTD_OK);
        std::vector<long long> want{300, 301, 302}, got = clocks();
        std::sort(got.begin(), got.end());
        CHECK(got == want);
        fdtd_batch_destroy(h);
    }
}

// Without pinned memory for the newest row and the read-out, rows are copied.
void no_pinned_memory()
{
    for (int resident = 0; resident < 2; ++resident) {
        Scene a(40, 40, 40, 6);
        if (!resident) a.sc.settings.air_viscosity_alpha = 2e-6;
        fdtd_handle *h = nullptr;
        g_fail_pinned = true;
        CHECK(fdtd_create(&a.sc, nullptr, &h) == FDTD_OK);
        g_fail_pinned = false;
        if (!h) continue;
        CHECK(fdtd_step(h, 30) == FDTD_OK);
        double p[2];
        CHECK(fdtd_listen(h, p) == FDTD_OK);
        fdtd_destroy(h);
    }
}

// What reads a handle or batch of device 1 while device 0 is selected launches
// and allocates on device 1, and leaves device 0 selected.
void other_device()
{
    Scene a(40, 40, 40, 6), b(44, 40, 40, 6);
    g_gives_up = [](const SceneDev &S) { return S.clock[CLK_TARGET] == 301; };
    for (int gives_up = 0; gives_up < 2; ++gives_up) {
        if (gives_up) g_gives_up = [](const SceneDev &) { return true; };
        fdtd_options o;
        fdtd_options_default(&o);
        o.device = 1;
        std::vector<double> out(64000);
        for (int call = 0; call < 4; ++call) {
            fdtd_handle *h = nullptr;
            CHECK(fdtd_create(&a.sc, &o, &h) == FDTD_OK);
            CHECK(fdtd_step(h, 64) == FDTD_OK);
            t_dev = 0;
            CHECK((call == 0 ? fdtd_listen(h, out.data()) : call == 1 ? fdtd_read_listener_series(h, 0, 64, out.data()) :
                   call == 2 ? fdtd_read_pressure(h, out.data()) : fdtd_synchronize(h)) == FDTD_OK);
            CHECK(t_dev == 0);
            CHECK(fdtd_destroy(h) == FDTD_OK);
        }
        const fdtd_scene sc[2] = {a.sc, b.sc};
        const int steps[2] = {300, 301};
        fdtd_batch *h = nullptr;
        t_dev = 1;
        CHECK(fdtd_batch_create(sc, steps, 2, nullptr, &h) == FDTD_OK);
        CHECK(fdtd_batch_step(h, 64) == FDTD_OK);
        t_dev = 0;
        CHECK(fdtd_batch_read_listener_series(h, 0, out.data()) == FDTD_OK);
        CHECK(t_dev == 0);
        for (const auto &e : g_mem) CHECK(e.second.dev == 1);
        CHECK(fdtd_batch_destroy(h) == FDTD_OK);
    }
}

// Two handles whose blocks follow each other: the second one's waits for the
// first one's, and nothing is enqueued for it on the first one's stream, which
// its owner may be capturing.
void captured_neighbour()
{
    Scene a(128, 128, 128, 12);
    fdtd_options o;
    fdtd_options_default(&o);
    hipStream_t st = new_stream();
    o.stream = st;
    fdtd_handle *h[2] = {nullptr, nullptr};
    CHECK(fdtd_create(&a.sc, &o, &h[0]) == FDTD_OK);
    CHECK(fdtd_create(&a.sc, nullptr, &h[1]) == FDTD_OK);
    CHECK(fdtd_step(h[0], 64) == FDTD_OK);
    forget();
    (void)hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed);
    CHECK(fdtd_step(h[1], 64) == FDTD_OK);
    hipGraph_t g = nullptr;
    (void)hipStreamEndCapture(st, &g);
    bool waited = false;
    for (const Call &c : g_log) {
        if (c.stream == stream_of(st)) bad("%s on the other handle's stream", c.what.c_str());
        waited = waited || c.what == "wait";
    }
    CHECK(waited && count("resident") == 1);
    CHECK((clocks() == std::vector<long long>{64, 64}));
    for (fdtd_handle *x : h) CHECK(fdtd_destroy(x) == FDTD_OK);
}

// Blocks that fit the device together wait for nothing on other streams; one that does
// not fit beside them waits for them, and for none that have been waited for by the host.
void side_by_side()
{
    Scene a(64, 64, 64, 10), b(128, 128, 128, 12);
    fdtd_handle *h[5];
    for (int i = 0; i < 5; ++i) CHECK(fdtd_create(i < 4 ? &a.sc : &b.sc, nullptr, &h[i]) == FDTD_OK);
    auto waits = [&](int i) {
        forget();
        CHECK(fdtd_step(h[i], 64) == FDTD_OK && count("resident") == 1);
        return count("wait");
    };
    for (int i = 0; i < 3; ++i) CHECK(waits(i) == 0);
    CHECK(waits(0) == 0 && waits(2) == 0);
    CHECK(waits(3) == 3);                       // 4 x 208 workgroups of 768
    CHECK(waits(4) == 1);                       // of the other shape: behind the one that waited for all
    CHECK(waits(1) == 1);
    for (fdtd_handle *x : h) CHECK(fdtd_synchronize(x) == FDTD_OK);
    CHECK(waits(3) == 0 && waits(0) == 0 && waits(4) == 2);
    for (fdtd_handle *x : h) CHECK(fdtd_destroy(x) == FDTD_OK);
}

// Blocks too short to pay for a resident launch's load and store of the state are step kernels.
void short_blocks()
{
    Scene a(40, 40, 40, 6), b(44, 40, 40, 6), c(144, 146, 144, 8);   // the third one in the largest tiles
    auto resident = [&](auto step) {
        forget();
        CHECK(step() == FDTD_OK);
        return count("resident") > 0;
    };
    {
        const fdtd_scene sc[2] = {a.sc, b.sc};
        const int steps[2] = {600, 601};
        fdtd_batch *h = nullptr;
        CHECK(fdtd_batch_create(sc, steps, 2, nullptr, &h) == FDTD_OK);
        CHECK(!resident([&] { return fdtd_batch_step(h, 1); }) && count("step") >= 1);
        CHECK(!resident([&] { return fdtd_batch_step(h, 3); }) && count("step") >= 3);
        CHECK(resident([&] { return fdtd_batch_step(h, 4); }));
        CHECK(!resident([&] { return fdtd_batch_step(h, 2); }));
        CHECK((clocks() == std::vector<long long>{10, 10}));
        // a long call's remainder joins its last blocks
        CHECK(resident([&] { return fdtd_batch_step(h, 258); }) && count("step") == 0 && count("resident") == 2);
        CHECK(resident([&] { return fdtd_batch_run(h); }) && count("step") == 0);
        CHECK(fdtd_batch_destroy(h) == FDTD_OK);
    }
    {
        fdtd_handle *h = nullptr;
        CHECK(fdtd_create(&c.sc, nullptr, &h) == FDTD_OK);
        CHECK(!resident([&] { return fdtd_step(h, 7); }));
        CHECK(resident([&] { return fdtd_step(h, 8); }));
        CHECK(fdtd_destroy(h) == FDTD_OK);
    }
    for (int block : {2, 16}) {
        fdtd_server_options o;
        fdtd_server_options_default(&o);
        o.steps_per_block = block;
        fdtd_server *s = nullptr;
        int64_t id;
        CHECK(fdtd_server_create(&o, &s) == FDTD_OK);
        CHECK(resident([&] {
            const fdtd_status st = fdtd_server_submit(s, block == 2 ? &a.sc : &c.sc, 40, &id);
            return st == FDTD_OK ? fdtd_server_wait(s, id, 60000) : st;
        }) == false);
        CHECK(fdtd_server_destroy(s) == FDTD_OK);
    }
}

// A handle whose block was given up, because something else held the device, runs
// step kernels for a while and then tries again, after longer and longer whiles.
void tries_again()
{
    Scene a(40, 40, 40, 6);
    fdtd_handle *h = nullptr;
    CHECK(fdtd_create(&a.sc, nullptr, &h) == FDTD_OK);
    std::vector<double> out(2);
    g_gives_up = [](const SceneDev &) { return true; };
    long long last = 0, pause = 0;
    int tries = 0;
    for (long long s = 0; s < 200000; s += 250) {
        forget();
        CHECK(fdtd_step(h, 250) == FDTD_OK && fdtd_listen(h, out.data()) == FDTD_OK);
        CHECK(clocks() == std::vector<long long>{s + 250});
        if (!count("resident")) continue;
        if (tries) {
            CHECK(s - last >= 8000 && s - last >= 2 * pause - 500);
            pause = s - last;
        }
        last = s;
        ++tries;
    }
    CHECK(tries >= 3 && tries <= 6);
    g_gives_up = [](const SceneDev &) { return false; };
    CHECK(fdtd_step(h, 400000) == FDTD_OK);
    forget();
    CHECK(fdtd_step(h, 250) == FDTD_OK);
    CHECK(count("resident") == 1 && count("step") == 0);
    // not more than some hundredths of a second (a spin takes 0.2 us)
    CHECK(g_patience > 0 && g_patience <= 1 << 16);
    CHECK(fdtd_destroy(h) == FDTD_OK);
}

// The device memory that a handle reports holds its resident tables too.
void device_bytes()
{
    Scene a(64, 64, 64, 10);
    fdtd_handle *h = nullptr;
    CHECK(fdtd_create(&a.sc, nullptr, &h) == FDTD_OK);
    fdtd_info o;
    CHECK(fdtd_get_info(h, &o) == FDTD_OK);
    size_t held = 0;
    for (const auto &e : g_mem) held += e.second.n;
    CHECK((size_t)o.device_bytes <= held && o.device_bytes >= 0.95 * (double)held);   // (the launch lists are not counted)
    CHECK(fdtd_destroy(h) == FDTD_OK);
}

struct Scenario { const char *name; void (*run)(); };
const Scenario kScenarios[] = {
    {"batch_capture", batch_capture},
    {"failed_load", failed_load},
    {"server_check", server_check},
    {"cut_chunk", cut_chunk},
    {"no_memory_for_lists", no_memory_for_lists},
    {"no_pinned_memory", no_pinned_memory},
    {"other_device", other_device},
    {"captured_neighbour", captured_neighbour},
    {"side_by_side", side_by_side},
    {"short_blocks", short_blocks},
    {"tries_again", tries_again},
    {"device_bytes", device_bytes},
};

}  // namespace

int main(int argc, char **argv)
{
    for (const Scenario &s : kScenarios) {
        if (argc == 1) std::printf("%s\n", s.name);
        else if (s.name == std::string(argv[1])) {
            s.run();
            return g_bad ? 1 : 0;
        }
    }
    return argc == 1 ? 0 : 2;
}
