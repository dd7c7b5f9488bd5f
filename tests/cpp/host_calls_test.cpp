// Host side of the host-buffer entry points without a GPU: the HIP calls of libqlinear.so
// bind to the definitions below (device memory is host memory, kernels do not run), so what
// is checked is the library's own bookkeeping.
//
//   host_calls_test exit        a workspace owned by an object with static storage, used by a
//                               host-buffer call, is freed after main returns
//   host_calls_test no_pinned   pinned memory runs out: the rows go through plain copies, and
//                               the failed calls' error is not taken for a launch's
//   host_calls_test capture     sets are allocated and freed in the relaxed capture mode, also
//                               the set of a call beyond those that stay idle
//   host_calls_test blocks      rows go through pinned blocks only where the weights, which every
//                               block streams again, cost less than the blocks save
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include <hip/hip_runtime_api.h>

#include "../../include/qlinear.h"

#ifdef hipGetDeviceProperties
#undef hipGetDeviceProperties
#endif

namespace {
thread_local hipError_t g_last = hipSuccess;  // as the runtime keeps it: until it is read
thread_local hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;
std::mutex g_mutex;
int g_pinned = 0, g_events = 0;  // live allocations, under g_mutex
bool g_exposed = false;          // one was made or freed outside the relaxed capture mode
int g_gate = 0;                  // event waits still to come before any returns
std::condition_variable g_gate_open;
void count(int& what, int d) {
    std::lock_guard<std::mutex> g(g_mutex);
    what += d;
    g_exposed |= g_mode != hipStreamCaptureModeRelaxed;
}
hipError_t err(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
hipError_t alloc(void** p, size_t n) {
    *p = std::calloc(1, n ? n : 1);
    return err(*p ? hipSuccess : hipErrorOutOfMemory);
}
enum Fail { kNone, kHostMalloc, kHostPointer, kEvent };
Fail g_fail = kNone;  // the call that fails
std::atomic<bool> g_coherent{false};  // the last pinned allocation asked for coherent memory
std::atomic<size_t> g_pinned_bytes{0};  // of the last one
std::atomic<int> g_launches{0};
int g_copied_in = 0;  // rows or words copied to device memory
}  // namespace

extern "C" {
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags) {
    g_coherent = flags & hipHostMallocCoherent;
    g_pinned_bytes = n;
    if (g_fail == kHostMalloc) return err(hipErrorOutOfMemory);
    count(g_pinned, 1);
    return alloc(p, n);
}
hipError_t hipHostFree(void* p) {
    count(g_pinned, -1);
    return std::free(p), hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    return *d = h, g_fail == kHostPointer ? err(hipErrorInvalidValue) : hipSuccess;
}
hipError_t hipMemset(void* p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    g_copied_in += k == hipMemcpyHostToDevice;
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind, hipStream_t) {
    for (size_t i = 0; i < h; ++i) std::memcpy(static_cast<char*>(d) + i * dp, static_cast<const char*>(s) + i * sp, w);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    void* p;
    const hipError_t e = alloc(&p, 1);
    *s = static_cast<hipStream_t>(p);
    return e;
}
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    void* p = nullptr;
    const hipError_t r = g_fail == kEvent ? err(hipErrorOutOfMemory) : alloc(&p, 1);
    if (p) count(g_events, 1);
    *e = static_cast<hipEvent_t>(p);
    return r;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    count(g_events, -1);
    return std::free(e), hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    std::unique_lock<std::mutex> g(g_mutex);
    if (g_gate > 0 && --g_gate == 0) g_gate_open.notify_all();
    g_gate_open.wait(g, [] { return g_gate == 0; });
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    const hipStreamCaptureMode was = g_mode;
    g_mode = *m;
    *m = was;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* st) {
    *g = *b = dim3(1);
    *lds = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return ++g_launches, hipSuccess; }
}

namespace {

// A linear and its workspace.
struct Pair {
    qlin_weights* w = nullptr;
    qlin_workspace* ws = nullptr;
    int K = 0, N = 0;
    int open(int bits, int k, int n, int rows) {
        K = k;
        N = n;
        const qlin_weight_config cfg = {bits, K, N};
        const std::vector<int8_t> packed((size_t)N * K * bits / 8);
        const std::vector<float> scales(N, 1.0f);
        if (int rc = qlin_weights_create_packed(&cfg, packed.data(), scales.data(), &w)) return rc;
        return qlin_workspace_create(rows, K, N, &ws);
    }
    int run(int rows) {
        const std::vector<float> a((size_t)rows * K, 0.5f);
        std::vector<float> c((size_t)rows * N);
        return qlin_run_f32(ws, w, rows, a.data(), c.data());
    }
    ~Pair() {
        qlin_workspace_free(ws);
        qlin_weights_free(w);
    }
};

Pair g_owner;  // freed after main, and after everything the library builds during main

int expect(bool ok, const char* what) {
    if (!ok) std::printf("FAIL %s\n", what);
    return ok ? 0 : 1;
}

int at_exit() {
    if (expect(g_owner.open(4, 256, 256, 4) == QLIN_OK, "create")) return 1;
    qlin_workspace_info info;
    if (expect(qlin_workspace_query(g_owner.ws, &info) == QLIN_OK && info.pinned_host_bytes == 0, "no set yet")) return 1;
    return expect(g_owner.run(4) == QLIN_OK, "run") | expect(g_pinned == 1, "one set") |
           expect(qlin_workspace_query(g_owner.ws, &info) == QLIN_OK && info.pinned_host_bytes == g_pinned_bytes,
                  "pinned bytes reported") |
           expect(g_coherent, "coherent memory");
}

int no_pinned() {
    int bad = 0;
    for (Fail f : {kHostMalloc, kHostPointer, kEvent}) {
        Pair p;
        if (expect(p.open(4, 256, 256, 4) == QLIN_OK, "create")) return 1;
        for (int call = 0; call < 2; ++call) {
            g_fail = f;
            g_copied_in = 0;
            bad |= expect(p.run(4) == QLIN_OK, "run through copies") | expect(g_copied_in == 1, "rows copied");
            g_fail = kNone;
            bad |= expect(hipGetLastError() == hipSuccess, "no error left behind");
        }
        g_copied_in = 0;  // and once it is there again, through the pinned blocks
        bad |= expect(p.run(4) == QLIN_OK, "run") | expect(g_copied_in == 0, "rows through pinned blocks");
    }
    return bad;
}

int capture() {
    constexpr int kCalls = 6, kIdle = 4;
    std::atomic<int> failed{0};
    int bad = 0;
    {
        Pair p[kCalls];
        for (Pair& x : p)
            if (expect(x.open(4, 256, 256, 4) == QLIN_OK, "create")) return 1;
        g_gate = kCalls;  // every call holds a set of its own before any gives it back
        std::vector<std::thread> threads;
        for (Pair& x : p) threads.emplace_back([&failed, &x] {
            if (x.run(4) != QLIN_OK) failed = 1;
        });
        for (std::thread& t : threads) t.join();
        bad |= expect(!failed, "runs") | expect(g_pinned == kIdle, "sets kept") | expect(!g_exposed, "sets given back");
    }
    return bad | expect(g_pinned == 0 && g_events == 0, "nothing kept without a workspace") |
           expect(!g_exposed, "sets freed with the last workspace");
}

int blocks() {
    const struct {
        int bits, K, N, rows, blocks;  // 0: one run through copies
    } cases[] = {
        {4, 2560, 6144, 128, 4},   {4, 4096, 2560, 128, 2},  {4, 2560, 19456, 128, 10}, {4, 9728, 2560, 128, 5},
        {8, 2560, 19456, 8, 1},    {4, 2560, 151936, 1, 1},  {4, 2560, 151936, 32, 0},  {8, 8192, 28672, 64, 0},
        {8, 32160, 192, 212, 0},
    };
    int bad = 0;
    for (const auto& c : cases) {
        Pair p;
        if (expect(p.open(c.bits, c.K, c.N, c.rows) == QLIN_OK, "create")) return 1;
        g_launches = g_copied_in = 0;
        bad |= expect(p.run(c.rows) == QLIN_OK, "run");
        const bool ok = c.blocks ? g_launches == 2 * c.blocks && g_copied_in == 0 : g_launches <= 2 && g_copied_in == 1;
        if (!ok) std::printf("W%d %d x %d, %d rows: %d launches, %d copies in\n", c.bits, c.K, c.N, c.rows, (int)g_launches, g_copied_in);
        bad |= expect(ok, "route");
    }
    return bad;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string mode = argc > 1 ? argv[1] : "";
    const int rc = mode == "exit" ? at_exit() : mode == "no_pinned" ? no_pinned() : mode == "capture" ? capture() : mode == "blocks" ? blocks() : expect(false, "mode");
    if (!rc) std::printf("PASS %s\n", mode.c_str());
    std::fflush(stdout);
    return rc;
}
