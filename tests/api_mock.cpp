// api_mock.cpp -- CPU tests of the C ABI's host side (q-pso_amd/csrc/qpso_api.cpp)
// against a mock HIP runtime: device memory is host memory, a stream's copies
// and launches run only when the stream is waited for (so staging that is
// reused or left too early shows), and failures are injected by call.  Built
// and run by tests/test_api_host.py with AddressSanitizer and
// UndefinedBehaviorSanitizer.  Prints one line per scenario; exits non-zero on
// the first violated check.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "qpso.h"
#include "qpso_internal.h"
#include "qpso_kernels.h"
#include "qpso_tables.h"

// ---- the mock runtime ---------------------------------------------------------
namespace {

struct Mock {
    using Op = std::function<void()>;
    std::map<hipStream_t, std::deque<Op>> queues;
    std::vector<Op>* capture = nullptr;
    bool no_pinned = false;    // hipHostMalloc fails
    int fail_copy_in = -1;     // the copy after this many fails to enqueue
    int host_mallocs = 0, host_frees = 0, frees = 0;
    size_t last_arena = 0;     // bytes of the last pool allocation
    std::map<void*, size_t> live;  // device allocations

    void put(hipStream_t st, Op op) {
        if (capture) capture->push_back(std::move(op));
        else queues[st].push_back(std::move(op));
    }
    void drain(hipStream_t st) {
        auto& q = queues[st];
        while (!q.empty()) {
            Op op = std::move(q.front());
            q.pop_front();
            op();
        }
    }
    void drain_all() {
        for (auto& kv : queues) drain(kv.first);
    }
    size_t pending() const {
        size_t n = 0;
        for (auto& kv : queues) n += kv.second.size();
        return n;
    }
} g;

struct Graph {
    std::vector<Mock::Op> ops;
};

hipError_t dev_alloc(void** p, size_t n) {
    *p = std::malloc(n ? n : 1);
    std::memset(*p, 0xa5, n);
    g.live[*p] = n;
    return hipSuccess;
}
hipError_t dev_free(void* p) {
    if (!p) return hipSuccess;
    if (!g.live.erase(p)) {
        std::printf("  free of an unknown pointer\n");
        std::exit(1);
    }
    std::free(p);
    return hipSuccess;
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(static_cast<void*>(p), 0, sizeof(*p));
    p->multiProcessorCount = 4;
    p->memoryPoolsSupported = 1;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "mock error"; }
hipError_t hipDeviceSynchronize(void) { g.drain_all(); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return dev_alloc(p, n); }
hipError_t hipFree(void* p) { ++g.frees; g.drain_all(); return dev_free(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (g.no_pinned) return hipErrorOutOfMemory;
    ++g.host_mallocs;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { ++g.host_frees; g.drain_all(); std::free(p); return hipSuccess; }
hipError_t hipMemPoolCreate(hipMemPool_t* p, const hipMemPoolProps*) { *p = reinterpret_cast<hipMemPool_t>(&g); return hipSuccess; }
hipError_t hipMemPoolDestroy(hipMemPool_t) { return hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void*) { return hipSuccess; }
hipError_t hipMallocFromPoolAsync(void** p, size_t n, hipMemPool_t, hipStream_t) {
    g.last_arena = n;
    return dev_alloc(p, n);
}
hipError_t hipFreeAsync(void* p, hipStream_t st) { g.put(st, [p] { dev_free(p); }); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(new int(0)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { g.drain(s); g.queues.erase(s); delete reinterpret_cast<int*>(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { g.drain(s); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(new int(0)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<int*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { g.drain_all(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { g.drain_all(); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    if (g.fail_copy_in >= 0 && g.fail_copy_in-- == 0) return hipErrorUnknown;
    g.put(st, [=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t st) {
    g.put(st, [=] {
        for (size_t y = 0; y < h; ++y) std::memcpy((char*)d + y * dp, (const char*)s + y * sp, w);
    });
    return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t st) {
    g.put(st, [=] { std::fill_n(static_cast<int*>(d), n, v); });
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { g.capture = new std::vector<Mock::Op>(); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* out) {
    auto* gr = new Graph{std::move(*g.capture)};
    delete g.capture;
    g.capture = nullptr;
    *out = reinterpret_cast<hipGraph_t>(gr);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* out, hipGraph_t gr, hipGraphNode_t*, char*, size_t) {
    *out = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph*>(gr)));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t gr) { delete reinterpret_cast<Graph*>(gr); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { delete reinterpret_cast<Graph*>(e); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t st) {
    for (auto& op : reinterpret_cast<Graph*>(e)->ops) g.put(st, op);
    return hipSuccess;
}
}  // extern "C"

// ---- the mock kernels: a solve's result is made from what was uploaded --------
namespace qpso_launch {
int rf_num_configs() { return 5; }
int rf_config_threads(int) { return 256; }
int rf_config_tile(int) { return 10112; }
bool rf_needs_windows(int, int) { return false; }
hipError_t scratch_address(int, void** p) {
    static std::vector<char> a(QPSO_NOALLOC_SCRATCH_BYTES);
    *p = a.data();
    return hipSuccess;
}
hipError_t init(const QpsoSolveDev* d, int n, hipStream_t st, hipEvent_t, hipEvent_t, bool) {
    g.put(st, [=] {
        for (int i = 0; i < n; ++i) {
            *d[i].flags = 0;
            d[i].counters[0] = d[i].counters[1] = d[i].counters[2] = 0;
        }
    });
    return hipSuccess;
}
// gbest: the sum of the crop and of its prefix table's last column
void finish(const QpsoSolveDev& S) {
    const int rw = S.rect[2] - S.rect[0], rh = S.rect[3] - S.rect[1];
    float sum = 0.0f, cnt = 0.0f;
    for (int i = 0; i < rw * rh; ++i) sum += S.obs[i];
    for (int y = 0; y < rh; ++y) cnt += S.obs_rows[y * (rw + 1) + rw];
    for (int d = 0; d < 7; ++d) S.gbest[d] = sum;
    S.gbest[7] = cnt;
    S.counters[0] = (unsigned long long)S.N;
}
hipError_t pso_step(const QpsoSolveDev* d, int n, hipStream_t st, hipEvent_t, hipEvent_t) {
    g.put(st, [=] {
        for (int i = 0; i < n; ++i) finish(d[i]);
    });
    return hipSuccess;
}
hipError_t pso_step_two(const QpsoSolveDev* d, int, int, hipStream_t st) {
    g.put(st, [=] { finish(*d); });
    return hipSuccess;
}
// a pose's fitness: the sum of its seven values
hipError_t render_fitness(int, int, const QpsoSolveDev* d, const QpsoItem* items, int n, hipStream_t st, hipEvent_t,
                          hipEvent_t, int it) {
    if (!items && it < 0)
        g.put(st, [=] {
            for (int p = 0; p < n; ++p) {
                float s = 0.0f;
                for (int k = 0; k < 7; ++k) s += d->pos[k * d->N + p];
                d->fit[p] = s;
                if (d->dbg_aabb)
                    for (int k = 0; k < 4; ++k) d->dbg_aabb[4 * p + k] = 10 * p + k;
            }
        });
    return hipSuccess;
}
hipError_t render_fitness_wrap(const QpsoSolveDev*, const QpsoItem*, int, hipStream_t, hipEvent_t, hipEvent_t) { return hipSuccess; }
hipError_t eval_begin(const QpsoSolveDev* d, const float* poses, int n, int, hipStream_t st) {
    g.put(st, [=] {
        for (int p = 0; p < n; ++p)
            for (int k = 0; k < 7; ++k) d->pos[k * d->N + p] = poses[k * n + p];
    });
    return hipSuccess;
}
hipError_t fill_frames(int32_t*, size_t, hipStream_t) { return hipSuccess; }
hipError_t obs_rows(const uint16_t*, uint16_t*, int, int, hipStream_t) { return hipSuccess; }
}  // namespace qpso_launch

// ---- scenarios ------------------------------------------------------------------
namespace {

#define CHECK(cond)                                                                 \
    do {                                                                            \
        if (!(cond)) {                                                              \
            std::printf("  check failed at line %d: %s\n", __LINE__, #cond);        \
            return false;                                                           \
        }                                                                           \
    } while (0)

struct World {
    qpso_ctx* ctx = nullptr;
    uint32_t mesh = 0;
    std::vector<uint16_t> depth = std::vector<uint16_t>(QPSO_ROWS * QPSO_COLS);
    qpso_params p{};
    World() {
        for (size_t i = 0; i < depth.size(); ++i) depth[i] = (uint16_t)(i % 7);
        qpso_params_default(&p);
        p.n_particles = 8;
        p.n_iters = 3;
        if (qpso_create(0, &ctx) != QPSO_OK) std::exit(1);
        const float soa[9] = {0, 1, 0, 0, 0, 1, 2, 2, 2};
        if (qpso_mesh_upload(ctx, soa, 1, &mesh) != QPSO_OK) std::exit(1);
    }
    ~World() { qpso_destroy(ctx); }
    qpso_cluster cluster(int w, int h) const {
        qpso_cluster c{};
        c.rect[0] = 0; c.rect[1] = 0; c.rect[2] = w; c.rect[3] = h;
        c.num_points = 1;
        c.depth = depth.data();
        return c;
    }
    bool right(const qpso_result& r, int w, int h) const {
        float sum = 0.0f, cnt = 0.0f;
        for (int y = 0; y < h; ++y)
            for (int x = 0; x < w; ++x) {
                sum += depth[y * QPSO_COLS + x];
                cnt += depth[y * QPSO_COLS + x] != 0 ? 1 : 0;
            }
        return r.pose[0] == sum && r.fit == cnt && r.raster_px == (uint64_t)p.n_particles && r.status == QPSO_OK;
    }
    bool scores_right(qpso_solve* s, int n) const {
        std::vector<float> poses(7 * n), fit(n);
        std::vector<int32_t> box(4 * n);
        for (int i = 0; i < 7 * n; ++i) poses[i] = (float)(i % 11);
        if (qpso_solve_eval_poses(s, n, poses.data(), fit.data(), box.data(), nullptr) != QPSO_OK) return false;
        for (int p = 0; p < n; ++p) {
            float sum = 0.0f;
            for (int k = 0; k < 7; ++k) sum += poses[k * n + p];
            if (fit[p] != sum || box[4 * p + 3] != 10 * p + 3) return false;
        }
        return true;
    }
};

// A copy of the results that cannot be enqueued: the call fails, and nothing it
// queued is left behind to write into memory that later calls use.
bool results_wait_on_failure() {
    World w;
    qpso_solve* s[3];
    for (int i = 0; i < 3; ++i) {
        const qpso_cluster c = w.cluster(10 + i, 6);
        CHECK(qpso_solve_create(w.ctx, w.mesh, &c, &w.p, 0, &s[i]) == QPSO_OK);
    }
    qpso_result r[3];
    CHECK(qpso_solve_run_batch(w.ctx, 3, s, r) == QPSO_OK);
    g.fail_copy_in = 1;  // the second solve's
    CHECK(qpso_solve_run_batch(w.ctx, 3, s, r) == QPSO_E_HIP);
    CHECK(g.pending() == 0);
    g.fail_copy_in = 0;
    CHECK(qpso_solve_run(s[0], r) == QPSO_E_HIP);
    CHECK(g.pending() == 0);
    g.fail_copy_in = -1;
    CHECK(qpso_solve_run_batch(w.ctx, 3, s, r) == QPSO_OK);
    for (int i = 0; i < 3; ++i) CHECK(w.right(r[i], 10 + i, 6));
    for (auto* x : s) qpso_solve_destroy(x);
    return true;
}

// Without pinned memory every call works as with it.
bool no_pinned_memory() {
    g.no_pinned = true;
    bool ok = false;
    {
        World w;
        ok = [&] {
            qpso_solve* s[2];
            for (int i = 0; i < 2; ++i) {
                const qpso_cluster c = w.cluster(200 + i, 300);
                CHECK(qpso_solve_create(w.ctx, w.mesh, &c, &w.p, 0, &s[i]) == QPSO_OK);
            }
            qpso_result r[2];
            CHECK(qpso_solve_run(s[0], r) == QPSO_OK && w.right(r[0], 200, 300));
            CHECK(qpso_solve_run_batch(w.ctx, 2, s, r) == QPSO_OK && w.right(r[1], 201, 300));
            CHECK(w.scores_right(s[1], 8));
            const qpso_cluster c = w.cluster(50, 40);
            CHECK(qpso_estimate_pose(w.ctx, w.mesh, &c, &w.p, r) == QPSO_OK && w.right(r[0], 50, 40));
            for (auto* x : s) qpso_solve_destroy(x);
            return true;
        }();
    }
    g.no_pinned = false;
    return ok;
}

// Pinned memory is taken once, with the context: no call waits for the device
// to grow it (the serving thread creates solves of any crop), and neither do
// larger scorings.
bool staging_keeps_its_size() {
    World w;
    w.p.n_iters = 1;
    int mallocs = 0, host_frees = 0, frees = 0;
    for (int k = 1; k <= 8; ++k) {
        const int cw = 80 * k, ch = 60 * k;
        const qpso_cluster c = w.cluster(cw, ch);
        qpso_solve* s = nullptr;
        w.p.n_particles = k == 8 ? 65535 : 1000 * k;
        CHECK(qpso_solve_create(w.ctx, w.mesh, &c, &w.p, 0, &s) == QPSO_OK);
        qpso_result r{};
        CHECK(qpso_solve_run(s, &r) == QPSO_OK && w.right(r, cw, ch));
        CHECK(w.scores_right(s, w.p.n_particles));
        CHECK(w.scores_right(s, 3));
        qpso_solve_destroy(s);
        if (k == 1) {
            mallocs = g.host_mallocs;
            host_frees = g.host_frees;
            frees = g.frees;
        }
        CHECK(g.host_mallocs == mallocs && g.host_frees == host_frees && g.frees == frees);
    }
    return true;
}

// More results than the staging holds.
bool many_results() {
    World w;
    constexpr int kN = 3500;
    const qpso_cluster c = w.cluster(9, 5);
    std::vector<qpso_solve*> s(kN);
    for (auto& x : s) CHECK(qpso_solve_create(w.ctx, w.mesh, &c, &w.p, 0, &x) == QPSO_OK);
    std::vector<qpso_result> r(kN);
    CHECK(qpso_solve_run_batch(w.ctx, kN, s.data(), r.data()) == QPSO_OK);
    for (auto& x : r) CHECK(w.right(x, 9, 5));
    for (auto* x : s) qpso_solve_destroy(x);
    return true;
}

// qpso_solve_bytes is a served solve's arena; one of up to 4,096 particles that
// may run on its own takes 32 bytes a particle and at most 1 KiB more.
bool arena_bytes() {
    World w;
    const qpso_cluster c = w.cluster(33, 21);
    for (const int n : {1, 8, 65, 257, 4096, 4097}) {
        w.p.n_particles = n;
        const uint64_t bytes = qpso_solve_bytes(&w.p, c.rect);
        qpso_solve* s = nullptr;
        CHECK(qpso_solve_create(w.ctx, w.mesh, &c, &w.p, 0, &s) == QPSO_OK);
        CHECK(g.last_arena >= bytes + (n <= 4096 ? 32 * n : 0) && g.last_arena <= bytes + (n <= 4096 ? 32 * n + 1024 : 0));
        qpso_solve_destroy(s);
        qpso_server* sv = nullptr;
        CHECK(qpso_server_create(w.ctx, uint64_t(1) << 32, &sv) == QPSO_OK);
        uint64_t t = 0;
        qpso_result r{};
        CHECK(qpso_server_submit(sv, w.mesh, &c, &w.p, &t) == QPSO_OK);
        CHECK(qpso_server_wait(sv, t, &r) == QPSO_OK && w.right(r, 33, 21));
        qpso_server_destroy(sv);
        CHECK(g.last_arena == bytes);
    }
    return true;
}

struct Scenario {
    const char* name;
    bool (*run)();
};
const Scenario kScenarios[] = {
    {"results_wait_on_failure", results_wait_on_failure},
    {"no_pinned_memory", no_pinned_memory},
    {"staging_keeps_its_size", staging_keeps_its_size},
    {"many_results", many_results},
    {"arena_bytes", arena_bytes},
};

}  // namespace

int main(int argc, char** argv) {
    for (const auto& s : kScenarios) {
        if (argc > 1 && std::strcmp(argv[1], s.name) != 0) continue;
        const bool ok = s.run();
        std::printf("%s %s\n", ok ? "PASS" : "FAIL", s.name);
        if (!ok) return 1;
        if (!g.live.empty()) {
            std::printf("FAIL %s: %zu device allocations left\n", s.name, g.live.size());
            return 1;
        }
    }
    return 0;
}
