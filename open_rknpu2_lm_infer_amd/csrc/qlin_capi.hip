// C ABI of libqlinear: weights, workspaces, dispatch between the decode GEMV and the
// prefill GEMM, and the host-buffer entry points that mirror the reference's
// synchronous rk_npu_w4a8_run_f32 / rk_npu_f32i8f32_run_dynamic.
#include <hip/hip_runtime.h>

#include <atomic>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <tuple>
#include <vector>

#include "../../include/qlinear.h"
#include "qlin_internal.hpp"

using namespace qlin;

struct qlin_weights {
    int bits, K, N, Kp, Np, device;
    int64_t wrow;  // bytes per row
    uint8_t* W;
    float* scales;
};

// Environment overrides of the kernel-variant choices (tests, tuning experiments), read
// once when a workspace is created so the run path makes no getenv calls.  0 / -1: unset.
struct QlinOverrides {
    int gemv_item_width;  // QLIN_GEMV_ITEM_WIDTH, 1..16
    int gemv_waves;       // QLIN_GEMV_WAVES, 4 / 8 / 16
    int gemv_grid;        // QLIN_GEMV_GRID, >= 0 (0: one workgroup per item)
    int fused_max_rows;   // QLIN_FUSED_QUANT_MAX_ROWS (default 8)
    int gemm_splits;      // QLIN_GEMM_SPLITS
    int gemm_target_wgs;  // QLIN_GEMM_TARGET_WGS (default: the CU count)
    int gemm_group_m;     // QLIN_GEMM_GROUP_M (default 4)
    int gemm_deep;        // QLIN_GEMM_DEEP, 0 / 1
    int gemm_wn;          // QLIN_GEMM_WN, 2 / 4
    int gemm_kernel;      // QLIN_GEMM_KERNEL: 16 forces the 16x16x64 kernel
    int gemm_ks;          // QLIN_GEMM_KS: forces a wave-split-K configuration (0..19); -2: never that kernel
    int gemm_pp;          // QLIN_GEMM_PP: forces an alternating-waves configuration (0..7); -2: never
    int gemm_cfg;         // QLIN_GEMM_CFG: forces the 32x32x32 kernel with tile configuration 0..3 (3: W4 only)
};

struct qlin_workspace {
    int max_rows, max_k, max_n, max_kp, max_np, device, cu_count;
    QlinOverrides ov;
    int8_t* q;           // [max_rows, max_kp]
    float* s;            // [max_rows]
    uint32_t* counters;  // [n_counters], zero at rest
    int n_counters;
    int32_t* gemm_part;  // [part_ints]
    int64_t part_ints;   // capacity of gemm_part (ints)
    uint32_t* err;       // sticky error word
    float* dA;           // host-API staging [max_rows, max_k]
    float* dC;           // host-API staging [max_rows, max_n]
    hipStream_t stream;  // stream of the host-buffer entry points
    hipStream_t last;    // stream of the most recent run
    uint64_t device_bytes;
    bool counted;        // among the workspaces that keep staging sets alive
    bool err_used;       // a run that reports in err itself may have set it (also by a later graph replay)
};

namespace {

// ---- pinned staging of the host-buffer entry points ----------------------------------
//
// A set holds kSlots row blocks on their way in and out.  Sets are shared by the workspaces
// of a process: a call takes an idle one (or allocates), and puts it back; at most kIdleSets
// stay idle, and none once the last workspace is gone.  Each set serves one call at a time,
// so calls on several threads and streams use different sets.
constexpr int kSlots = 4;
constexpr size_t kSlotBytes = (size_t)1 << 20;  // of rows in and of rows out
constexpr size_t kSetBytes = 2 * kSlots * kSlotBytes + 256;
constexpr int kIdleSets = 4;

struct HostStage {
    int device;
    uint8_t* mem;     // kSlots x (in, out), then the error word
    uint8_t* dev;     // its device address
    hipEvent_t done[kSlots];
};

// Never destroyed (no destructor runs for any of these): the owner of a workspace may be an
// object with static storage, whose destructor comes after those of whatever this file built
// while the program ran.
std::mutex& stage_mutex() {
    static std::mutex& m = *new std::mutex;
    return m;
}
HostStage* g_idle[kIdleSets];  // idle sets, under stage_mutex as the counts
int g_n_idle = 0;
int g_workspaces = 0;          // live workspaces
std::atomic<int> g_sets{0};    // sets allocated, idle or in a call

// Keeps allocations and frees out of the checks of a graph that another thread records in global
// capture mode.  (The copies and waits of a host-buffer call end such a capture all the same.)
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

void free_stage(HostStage* h) {
    const RelaxedCapture relaxed;
    for (hipEvent_t e : h->done)
        if (e) (void)hipEventDestroy(e);
    if (h->mem) {
        (void)hipHostFree(h->mem);
        --g_sets;
    }
    delete h;
}

HostStage* take_stage(int device) {
    {
        std::lock_guard<std::mutex> g(stage_mutex());
        for (int i = 0; i < g_n_idle; ++i)
            if (g_idle[i]->device == device) {
                HostStage* h = g_idle[i];
                g_idle[i] = g_idle[--g_n_idle];
                return h;
            }
    }
    auto* h = new (std::nothrow) HostStage();
    if (!h) return nullptr;
    h->device = device;
    void *m = nullptr, *d = nullptr;
    const RelaxedCapture relaxed;
    // coherent by request, not by the runtime's default: the host reads rows and the error word after
    // an event, and the kernels read rows written between launches, without a flush
    bool ok = hipHostMalloc(&m, kSetBytes,
                            hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent) == hipSuccess;
    h->mem = static_cast<uint8_t*>(m);
    g_sets += m != nullptr;
    ok = ok && hipHostGetDevicePointer(&d, m, 0) == hipSuccess;
    h->dev = static_cast<uint8_t*>(d);
    for (int i = 0; ok && i < kSlots; ++i) ok = hipEventCreateWithFlags(&h->done[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        free_stage(h);
        (void)hipGetLastError();  // kept by the runtime until it is read: a launch would be taken to have failed
        return nullptr;
    }
    return h;
}

void give_back_stage(HostStage* h) {
    {
        std::lock_guard<std::mutex> g(stage_mutex());
        if (g_workspaces > 0 && g_n_idle < kIdleSets) {
            g_idle[g_n_idle++] = h;
            return;
        }
    }
    free_stage(h);
}

// Counts a workspace in (+1) or out (-1); the last one out frees the idle sets.
void count_workspace(int d) {
    HostStage* drop[kIdleSets];
    int n = 0;
    {
        std::lock_guard<std::mutex> g(stage_mutex());
        g_workspaces += d;
        while (g_workspaces == 0 && g_n_idle > 0) drop[n++] = g_idle[--g_n_idle];
    }
    while (n > 0) free_stage(drop[--n]);
}

}  // namespace

namespace {

constexpr int64_t kGemmPartInts = 16 << 20;  // split-K partial buffer: 64 MiB of int32
constexpr int kGemmTileM = 128, kGemmTileK = 128;

int64_t round_up(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

int env_int(const char* name, int dflt) {
    const char* v = std::getenv(name);
    return v && *v ? std::atoi(v) : dflt;
}

QlinOverrides read_overrides() {
    QlinOverrides o;
    o.gemv_item_width = env_int("QLIN_GEMV_ITEM_WIDTH", 0);
    o.gemv_waves = env_int("QLIN_GEMV_WAVES", 0);
    o.gemv_grid = env_int("QLIN_GEMV_GRID", -1);
    o.fused_max_rows = env_int("QLIN_FUSED_QUANT_MAX_ROWS", kFusedMaxRows);
    o.gemm_splits = env_int("QLIN_GEMM_SPLITS", 0);
    o.gemm_target_wgs = env_int("QLIN_GEMM_TARGET_WGS", 0);
    o.gemm_group_m = env_int("QLIN_GEMM_GROUP_M", 4);
    o.gemm_deep = env_int("QLIN_GEMM_DEEP", -1);
    o.gemm_wn = env_int("QLIN_GEMM_WN", 4);
    o.gemm_kernel = env_int("QLIN_GEMM_KERNEL", 0);
    o.gemm_ks = env_int("QLIN_GEMM_KS", -1);
    o.gemm_pp = env_int("QLIN_GEMM_PP", -1);
    o.gemm_cfg = env_int("QLIN_GEMM_CFG", -1);
    return o;
}

int current_device(int* dev) { return hipGetDevice(dev) == hipSuccess ? QLIN_OK : QLIN_ERR_NODEVICE; }

// ---- kernel-variant table (qlin_tune) ------------------------------------------------
// Key: bits, K, N, rows bucket, path (0 decode GEMV with fused quantization, 1 decode GEMV
// from quantized rows, 2 GEMM), SwiGLU.  Value: GEMV waves per group, or for a GEMM
// k splits + kTuneKernelStep * kernel, kernel 0 the planner's own pick, 1 the 16x16x64
// kernel, 2 + c the 32x32x32 kernel in tile configuration c (0..3; 3 for W4 only).  Plus
// kTunePlanner where the planner's own kernel beat every variant of the search: such
// an entry names the best of those but leaves the choice to the planner.
using TuneKey = std::tuple<int, int, int, int, int, int>;
constexpr int kTuneKernelStep = 100, kTuneMaxSplits = 64;
constexpr int kTuneKernel16 = 1, kTuneKernel32 = 2;
constexpr int kTunePlanner = 1 << 20;
std::map<TuneKey, int>& tune_table() {
    static std::map<TuneKey, int> t;
    return t;
}
std::mutex& tune_mutex() {
    static std::mutex m;
    return m;
}
thread_local int g_force_variant = 0;  // set by qlin_tune while it times one candidate (-1: the planner's own)
std::atomic<int> g_tune_entries{0};    // entries in the table: the run path skips the lock at 0

int rows_bucket(int rows) {
    if (rows <= kGemvMaxRows) return rows;
    int b = 32;
    while (b < rows && b < 4096) b *= 2;
    return rows <= 4096 ? b : (rows + 1023) / 1024 * 1024;
}

int tuned_variant(int bits, int K, int N, int rows, int path, bool sw) {
    if (g_force_variant) return std::max(g_force_variant, 0);
    if (g_tune_entries.load(std::memory_order_acquire) == 0) return 0;
    std::lock_guard<std::mutex> g(tune_mutex());
    auto it = tune_table().find(TuneKey{bits, K, N, rows_bucket(rows), path, sw ? 1 : 0});
    return it == tune_table().end() || it->second >= kTunePlanner ? 0 : it->second;
}



int cu_count(int dev) {
    static std::atomic<int> cached[64] = {};  // per device, 0 = not read yet
    if (dev >= 0 && dev < 64 && cached[dev].load(std::memory_order_relaxed) > 0) return cached[dev].load(std::memory_order_relaxed);
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    if (dev >= 0 && dev < 64) cached[dev].store(n, std::memory_order_relaxed);
    return n;
}

// W4 device order.  Each 32-bit word of a row holds the 8 codes of k = 8w .. 8w+7: byte b
// carries code 8w+b in its low nibble and code 8w+b+4 in its high nibble.  The kernels'
// unpack ((x << 4) & 0xF0 and x & 0xF0 per byte) then yields the codes in natural k order,
// so activations are used as they are.  The reference packing (byte j = codes 2j, 2j+1)
// differs only by a nibble permutation inside each word.
__host__ __device__ inline uint32_t w4_word_to_device(uint32_t x) {
    // x: nibble i holds code i (the reference packing of one word)
    auto spread = [](uint32_t v) {  // nibble i of a 16-bit value -> bits 8i .. 8i+3
        v = (v | (v << 8)) & 0x00FF00FFu;
        return (v | (v << 4)) & 0x0F0F0F0Fu;
    };
    return spread(x & 0xFFFFu) | (spread(x >> 16) << 4);
}

__global__ void w4_to_device_kernel(uint32_t* words, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        words[i] = w4_word_to_device(words[i]);
}

// compressed-tensors rows -> device rows.  W4 pack-quantized: the words' little-endian bytes
// hold codes 2j (low nibble) and 2j+1 as field = code + 8, whose two's-complement nibble is
// field ^ 8; W8 pack-quantized: byte ^ 0x80; W8 int-quantized: the byte itself.  Codes at
// k >= K and bytes past the row become zero.
__global__ void unpack_compressed_kernel(const uint8_t* src, int64_t src_row, int rows, int bits, int fmt, int K,
                                         uint8_t* dst, int64_t wrow) {
    const int64_t total = (int64_t)rows * wrow;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / wrow, j = i - r * wrow;
        uint8_t out = 0;
        if (bits == 4) {
            const int64_t klo = 8 * (j >> 2) + (j & 3), khi = klo + 4;  // device order
            auto code = [&](int64_t k) -> uint32_t {
                return k < K ? (((uint32_t)src[r * src_row + (k >> 1)] >> (4 * (k & 1))) & 0xFu) ^ 8u : 0u;
            };
            out = (uint8_t)(code(klo) | (code(khi) << 4));
        } else if (j < K) {
            const uint8_t b = src[r * src_row + j];
            out = fmt == 0 ? (uint8_t)(b ^ 0x80u) : b;
        }
        dst[i] = out;
    }
}

__global__ void pack_kn_kernel(const int8_t* codes, int K, int N, int Kp, int Np, int bits, uint8_t* out) {
    const int64_t row_bytes = bits == 4 ? Kp / 2 : Kp;
    const int64_t total = (int64_t)Np * row_bytes;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int n = (int)(i / row_bytes);
        const int j = (int)(i - (int64_t)n * row_bytes);
        if (bits == 8) {
            const int k = j;
            out[i] = (n < N && k < K) ? (uint8_t)codes[(int64_t)k * N + n] : 0;
        } else {
            const int k = 8 * (j >> 2) + (j & 3);  // device order: codes k and k + 4
            const int lo = (n < N && k < K) ? codes[(int64_t)k * N + n] : 0;
            const int hi = (n < N && k + 4 < K) ? codes[(int64_t)(k + 4) * N + n] : 0;
            out[i] = (uint8_t)((lo & 0xf) | ((hi & 0xf) << 4));
        }
    }
}

int check_config(const qlin_weight_config* c) {
    if (!c || (c->bits != 4 && c->bits != 8) || c->K <= 0 || c->N <= 0 || c->K > kMaxK ||
        c->N > (1 << 30))
        return QLIN_ERR_PARAM;
    return QLIN_OK;
}

int check_scales(const float* scales, int N) {
    if (!scales) return QLIN_ERR_PARAM;
    for (int n = 0; n < N; ++n)
        if (!(scales[n] > 0.0f) || !std::isfinite(scales[n])) return QLIN_ERR_PARAM;
    return QLIN_OK;
}

int alloc_weights(const qlin_weight_config* c, qlin_weights** w) {
    int dev;
    if (int rc = current_device(&dev)) return rc;
    auto* x = new (std::nothrow) qlin_weights();
    if (!x) return QLIN_ERR_NOMEM;
    x->bits = c->bits;
    x->K = c->K;
    x->N = c->N;
    x->Kp = (int)round_up(c->K, kKAlign);
    x->Np = (int)round_up(c->N, kNAlign);
    x->device = dev;
    x->wrow = c->bits == 4 ? x->Kp / 2 : x->Kp;
    if (hipMalloc(&x->W, (size_t)x->Np * x->wrow) != hipSuccess ||
        hipMalloc(&x->scales, (size_t)x->Np * sizeof(float)) != hipSuccess) {
        (void)hipFree(x->W);
        (void)hipFree(x->scales);
        delete x;
        return QLIN_ERR_NOMEM;
    }
    *w = x;
    return QLIN_OK;
}

int upload_scales(qlin_weights* x, const float* scales, hipMemcpyKind kind, hipStream_t st) {
    if (hipMemsetAsync(x->scales, 0, (size_t)x->Np * sizeof(float), st) != hipSuccess ||
        hipMemcpyAsync(x->scales, scales, (size_t)x->N * sizeof(float), kind, st) != hipSuccess)
        return QLIN_ERR_DEVICE;
    return QLIN_OK;
}

// Whether the rows go to the GEMV, or else to the tiled GEMM, where plan_rows leaves them to one of the
// two; it also names the path that qlin_run_plan reports and the variant table's key.  17..32 rows go
// through the GEMV's two row blocks where it measured faster than the tiled GEMM: every shape up to 20
// rows, and up to 32 for outputs of at most 4096 channels, whose GEMM grid is a few wide tiles split
// along K (W4 layer, us per linear with its quantize launch, tiled GEMM -> GEMV: o / down at 17 rows 14.3 /
// 18.9 -> 9.4 / 14.0, at 32 rows 14.4 / 19.1 -> 10.6 / 17.5; qkv / gate_up at 17 rows 14.7 / 16.4 -> 14.1 /
// 14.5, at 32 rows 14.8 / 16.5 -> 16.6 / 17.8).
bool gemv_ok(const qlin_workspace* ws, const qlin_weights* w, int rows) {
    (void)ws;
    if (rows <= kGemvMaxRows) return true;
    return rows <= kGemvMaxRowsWide && (rows <= 20 || w->N <= 4096);
}

}  // namespace

extern "C" {

const char* qlin_strerror(int rc) {
    switch (rc) {
        case QLIN_OK: return "success";
        case QLIN_ERR_PARAM: return "invalid parameter";
        case QLIN_ERR_NOMEM: return "out of device or host memory";
        case QLIN_ERR_DEVICE: return "HIP runtime error";
        case QLIN_ERR_NONFINITE: return "non-finite activation";
        case QLIN_ERR_UNSUPPORTED: return "shape not supported by this entry point";
        case QLIN_ERR_NODEVICE: return "no HIP device";
        default: return "unknown error";
    }
}

int qlin_device_query(int32_t device, qlin_device_info* out) {
    if (!out) return QLIN_ERR_PARAM;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return QLIN_ERR_NODEVICE;
    std::memset(out, 0, sizeof(*out));
    out->device = device;
    out->cu_count = prop.multiProcessorCount;
    out->sclk_khz = prop.clockRate;
    out->mclk_khz = prop.memoryClockRate;
    out->bus_width_bits = prop.memoryBusWidth;
    out->hbm_bytes = (int64_t)prop.totalGlobalMem;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) == 0) out->arch = 950;
    return QLIN_OK;
}

int qlin_weights_create(const qlin_weight_config* config, const int8_t* codes_kn, const float* scales,
                        qlin_weights** out) {
    if (!out) return QLIN_ERR_PARAM;
    *out = nullptr;
    if (int rc = check_config(config)) return rc;
    if (!codes_kn) return QLIN_ERR_PARAM;
    if (int rc = check_scales(scales, config->N)) return rc;
    const int64_t total = (int64_t)config->K * config->N;
    const int lo = config->bits == 4 ? -8 : -127, hi = config->bits == 4 ? 7 : 127;
    for (int64_t i = 0; i < total; ++i)
        if (codes_kn[i] < lo || codes_kn[i] > hi) return QLIN_ERR_PARAM;
    qlin_weights* w = nullptr;
    if (int rc = alloc_weights(config, &w)) return rc;
    int8_t* staging = nullptr;
    int rc = QLIN_OK;
    if (hipMalloc(&staging, (size_t)total) != hipSuccess) rc = QLIN_ERR_NOMEM;
    if (!rc && hipMemcpy(staging, codes_kn, (size_t)total, hipMemcpyHostToDevice) != hipSuccess) rc = QLIN_ERR_DEVICE;
    if (!rc) {
        hipLaunchKernelGGL(pack_kn_kernel, dim3(2048), dim3(256), 0, nullptr, staging, w->K, w->N, w->Kp, w->Np,
                           w->bits, w->W);
        if (hipGetLastError() != hipSuccess) rc = QLIN_ERR_DEVICE;
    }
    if (!rc) rc = upload_scales(w, scales, hipMemcpyHostToDevice, nullptr);
    if (!rc && hipDeviceSynchronize() != hipSuccess) rc = QLIN_ERR_DEVICE;
    (void)hipFree(staging);
    if (rc) {
        qlin_weights_free(w);
        return rc;
    }
    *out = w;
    return QLIN_OK;
}

static int create_packed(const qlin_weight_config* config, const void* packed, const float* scales,
                         hipMemcpyKind kind, hipStream_t st, qlin_weights** out) {
    if (!out) return QLIN_ERR_PARAM;
    *out = nullptr;
    if (int rc = check_config(config)) return rc;
    if (!packed || !scales) return QLIN_ERR_PARAM;
    if (config->bits == 4 && (config->K & 1)) return QLIN_ERR_PARAM;
    if (kind == hipMemcpyHostToDevice) {
        if (int rc = check_scales(scales, config->N)) return rc;
        if (config->bits == 8) {
            const int8_t* c = static_cast<const int8_t*>(packed);
            for (int64_t i = 0; i < (int64_t)config->K * config->N; ++i)
                if (c[i] == -128) return QLIN_ERR_PARAM;
        }
    }
    qlin_weights* w = nullptr;
    if (int rc = alloc_weights(config, &w)) return rc;
    const size_t src_row = config->bits == 4 ? (size_t)config->K / 2 : (size_t)config->K;
    int rc = QLIN_OK;
    if (hipMemsetAsync(w->W, 0, (size_t)w->Np * w->wrow, st) != hipSuccess ||
        hipMemcpy2DAsync(w->W, (size_t)w->wrow, packed, src_row, src_row, (size_t)config->N, kind, st) != hipSuccess)
        rc = QLIN_ERR_DEVICE;
    if (!rc && config->bits == 4) {
        // reference packing -> device order, in place (wrow is a multiple of 4 bytes)
        hipLaunchKernelGGL(w4_to_device_kernel, dim3(1024), dim3(256), 0, st, reinterpret_cast<uint32_t*>(w->W),
                           (int64_t)w->Np * w->wrow / 4);
        if (hipGetLastError() != hipSuccess) rc = QLIN_ERR_DEVICE;
    }
    if (!rc) rc = upload_scales(w, scales, kind, st);
    if (!rc && hipStreamSynchronize(st) != hipSuccess) rc = QLIN_ERR_DEVICE;
    if (rc) {
        qlin_weights_free(w);
        return rc;
    }
    *out = w;
    return QLIN_OK;
}

int qlin_weights_create_compressed(const qlin_weight_config* config, int32_t format, int32_t n_parts,
                                   const int32_t* part_n, const void* const* data, const float* const* scales,
                                   qlin_weights** out) {
    if (!out) return QLIN_ERR_PARAM;
    *out = nullptr;
    if (int rc = check_config(config)) return rc;
    if ((format != QLIN_PACK_QUANTIZED && format != QLIN_INT_QUANTIZED) || n_parts < 1 || !part_n || !data ||
        !scales || (format == QLIN_INT_QUANTIZED && config->bits != 8))
        return QLIN_ERR_PARAM;
    int64_t n_total = 0;
    for (int i = 0; i < n_parts; ++i) {
        if (part_n[i] <= 0 || !data[i]) return QLIN_ERR_PARAM;
        if (int rc = check_scales(scales[i], part_n[i])) return rc;
        n_total += part_n[i];
    }
    if (n_total != config->N) return QLIN_ERR_PARAM;
    const int64_t factor = 32 / config->bits;
    const int64_t src_row = format == QLIN_INT_QUANTIZED ? config->K : (config->K + factor - 1) / factor * 4;
    qlin_weights* w = nullptr;
    if (int rc = alloc_weights(config, &w)) return rc;
    int max_part = 0;
    for (int i = 0; i < n_parts; ++i) max_part = std::max(max_part, part_n[i]);
    uint8_t* staging = nullptr;
    int rc = QLIN_OK;
    if (hipMalloc(&staging, (size_t)max_part * src_row) != hipSuccess) rc = QLIN_ERR_NOMEM;
    if (!rc && (hipMemset(w->W, 0, (size_t)w->Np * w->wrow) != hipSuccess ||
                hipMemset(w->scales, 0, (size_t)w->Np * sizeof(float)) != hipSuccess))
        rc = QLIN_ERR_DEVICE;
    int64_t row0 = 0;
    for (int i = 0; i < n_parts && !rc; ++i) {
        if (hipMemcpy(staging, data[i], (size_t)part_n[i] * src_row, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(w->scales + row0, scales[i], (size_t)part_n[i] * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
            rc = QLIN_ERR_DEVICE;
            break;
        }
        hipLaunchKernelGGL(unpack_compressed_kernel, dim3(1024), dim3(256), 0, nullptr, staging, src_row, part_n[i],
                           config->bits, format, config->K, w->W + row0 * w->wrow, w->wrow);
        if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) rc = QLIN_ERR_DEVICE;
        row0 += part_n[i];
    }
    (void)hipFree(staging);
    if (rc) {
        qlin_weights_free(w);
        return rc;
    }
    *out = w;
    return QLIN_OK;
}

int qlin_weights_create_packed(const qlin_weight_config* config, const void* packed_nk, const float* scales,
                               qlin_weights** out) {
    return create_packed(config, packed_nk, scales, hipMemcpyHostToDevice, nullptr, out);
}

int qlin_weights_create_packed_device(const qlin_weight_config* config, const void* packed_nk,
                                      const float* scales, void* stream, qlin_weights** out) {
    return create_packed(config, packed_nk, scales, hipMemcpyDeviceToDevice, (hipStream_t)stream, out);
}

void qlin_weights_free(qlin_weights* w) {
    if (!w) return;
    (void)hipFree(w->W);
    (void)hipFree(w->scales);
    delete w;
}

int qlin_weights_query(const qlin_weights* w, qlin_weight_info* out) {
    if (!w || !out) return QLIN_ERR_PARAM;
    out->bits = w->bits;
    out->K = w->K;
    out->N = w->N;
    out->K_padded = w->Kp;
    out->N_padded = w->Np;
    out->device = w->device;
    out->device_bytes = (uint64_t)w->Np * w->wrow + (uint64_t)w->Np * sizeof(float);
    return QLIN_OK;
}

int qlin_workspace_create(int32_t max_rows, int32_t max_k, int32_t max_n, qlin_workspace** out) {
    if (!out) return QLIN_ERR_PARAM;
    *out = nullptr;
    if (max_rows <= 0 || max_k <= 0 || max_n <= 0 || max_k > kMaxK || max_n > (1 << 30)) return QLIN_ERR_PARAM;
    int dev;
    if (int rc = current_device(&dev)) return rc;
    auto* ws = new (std::nothrow) qlin_workspace();
    if (!ws) return QLIN_ERR_NOMEM;
    ws->max_rows = max_rows;
    ws->max_k = max_k;
    ws->max_n = max_n;
    ws->max_kp = (int)round_up(max_k, kKAlign);
    ws->max_np = (int)round_up(max_n, kNAlign);
    ws->device = dev;
    ws->cu_count = cu_count(dev);
    ws->ov = read_overrides();
    ws->part_ints = kGemmPartInts;
    ws->n_counters = std::max(ws->max_np / 16, 8192);
    const size_t bq = (size_t)max_rows * ws->max_kp, bs = (size_t)max_rows * sizeof(float);
    const size_t bc = (size_t)ws->n_counters * sizeof(uint32_t);
    const size_t bgm = (size_t)kGemmPartInts * sizeof(int32_t);
    const size_t bA = (size_t)max_rows * max_k * sizeof(float), bC = (size_t)max_rows * max_n * sizeof(float);
    bool ok = hipMalloc(&ws->q, bq) == hipSuccess && hipMalloc(&ws->s, bs) == hipSuccess &&
              hipMalloc(&ws->counters, bc) == hipSuccess &&
              hipMalloc(&ws->gemm_part, bgm) == hipSuccess && hipMalloc(&ws->err, 256) == hipSuccess &&
              hipMalloc(&ws->dA, bA) == hipSuccess && hipMalloc(&ws->dC, bC) == hipSuccess &&
              hipStreamCreateWithFlags(&ws->stream, hipStreamNonBlocking) == hipSuccess;
    if (ok)
        ok = hipMemset(ws->counters, 0, bc) == hipSuccess &&
             hipMemset(ws->err, 0, 256) == hipSuccess && hipMemset(ws->q, 0, bq) == hipSuccess &&
             hipDeviceSynchronize() == hipSuccess;
    ws->device_bytes = bq + bs + bc + bgm + 256 + bA + bC;
    ws->last = ws->stream;
    if (!ok) {
        qlin_workspace_free(ws);
        return QLIN_ERR_NOMEM;
    }
    count_workspace(1);
    ws->counted = true;
    *out = ws;
    return QLIN_OK;
}

void qlin_workspace_free(qlin_workspace* ws) {
    if (!ws) return;
    if (ws->stream) {
        (void)hipStreamSynchronize(ws->stream);
        (void)hipStreamDestroy(ws->stream);
    }
    (void)hipFree(ws->q);
    (void)hipFree(ws->s);
    (void)hipFree(ws->counters);
    (void)hipFree(ws->gemm_part);
    (void)hipFree(ws->err);
    (void)hipFree(ws->dA);
    (void)hipFree(ws->dC);
    if (ws->counted) count_workspace(-1);
    delete ws;
}

int qlin_workspace_query(const qlin_workspace* ws, qlin_workspace_info* out) {
    if (!ws || !out) return QLIN_ERR_PARAM;
    out->max_rows = ws->max_rows;
    out->reserved = 0;
    out->device_bytes = ws->device_bytes;
    out->pinned_host_bytes = (uint64_t)g_sets.load() * kSetBytes;
    return QLIN_OK;
}

int qlin_workspace_status(qlin_workspace* ws, int32_t clear) {
    if (!ws) return QLIN_ERR_PARAM;
    uint32_t e = 0;
    if (hipStreamSynchronize(ws->last) != hipSuccess) return QLIN_ERR_DEVICE;
    if (hipMemcpy(&e, ws->err, sizeof(e), hipMemcpyDeviceToHost) != hipSuccess) return QLIN_ERR_DEVICE;
    if (clear && e && hipMemset(ws->err, 0, sizeof(uint32_t)) != hipSuccess) return QLIN_ERR_DEVICE;
    return e ? QLIN_ERR_NONFINITE : QLIN_OK;
}

int qlin_quantize(int32_t rows, int32_t K, const void* A, int32_t a_dtype, int64_t lda, const float* gamma,
                  float eps, int8_t* q, int64_t ldq, float* s, uint32_t* err, uint32_t flags, void* stream) {
    if (rows <= 0 || K <= 0 || !A || !q || !s || lda < K || ldq < K || (a_dtype != QLIN_F32 && a_dtype != QLIN_F16))
        return QLIN_ERR_PARAM;
    if (gamma && !(eps > 0.0f && std::isfinite(eps))) return QLIN_ERR_PARAM;
    QuantParams p{};
    p.A = A;
    p.lda = lda;
    p.a_f16 = a_dtype == QLIN_F16;
    p.K = K;
    p.ldq = ldq;
    p.q = q;
    p.s = s;
    p.err = err;
    p.gamma = gamma;
    p.eps = eps;
    p.flags = flags & ~kFlagErrOnHost;
    return launch_quant(p, rows, (hipStream_t)stream) == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
}

}  // extern "C"

namespace {

// Residual update of the epilogue (qlin_run_residual, chain stages with QLIN_RESIDUAL).
struct ResidualArgs {
    const void* R;
    int64_t ldr;
    int r_f16;
    float mult;
};

// Waves per workgroup for a GEMV that quantizes (and normalizes) its rows itself: the
// usual count, or for up to 3 rows fewer when that many threads cannot hold the rows in
// registers (3 rows of K = 4096 at 16 waves); 0 when no count can.  Measured on o / down
// shapes (N = 2560, us per launch, fused at fewer waves vs separate quantize launch): W8
// K = 4096 3 rows 6.94 vs 7.38, 4 rows 7.79 vs 7.50 (every workgroup re-reads and
// quantizes all rows, so 4 rows keep the separate launch); K = 9728 2 rows 10.99 vs 10.96.
int gemv_fused_waves(int rows, int K, int groups, int steps, bool norm) {
    if (rows > kFusedRowsWide) return gemv_can_fuse(rows, K, 8, norm) ? 8 : 0;  // the 8-row instances
    for (int w = gemv_pick_waves(groups, steps); w >= 4; w /= 2) {
        if (gemv_can_fuse(rows, K, w, norm)) return w;
        if (rows >= 4) break;
    }
    return 0;
}

// Launch shape of a decode GEMV.
struct GemvPlan {
    int iw;     // output channels per item (QLIN_GEMV_ITEM_WIDTH, else the width in 8..16
                // that spreads the items most evenly over the CUs)
    int waves;  // waves per workgroup: 4, 8 or 16; 0 = the fused prologue cannot hold the rows
    int grid;   // workgroups; 0 = one per item
    int items;  // items of the launch
};

GemvPlan plan_gemv(const qlin_workspace* ws, const qlin_weights* w, int rows, bool fused, bool norm, uint32_t flags) {
    const QlinOverrides& ov = ws->ov;
    const bool sw = (flags & kFlagSwiglu) != 0;
    const int cols = sw ? w->N / 2 : w->N;
    GemvPlan g{};
    g.iw = ov.gemv_item_width >= 1 && ov.gemv_item_width <= 16 ? ov.gemv_item_width : gemv_item_width(cols, ws->cu_count);
    g.items = (cols + g.iw - 1) / g.iw;
    const int steps = w->Kp / (w->bits == 4 ? 256 : 128);
    int waves = ov.gemv_waves;
    if (waves != 4 && waves != 8 && waves != 16) {
        waves = tuned_variant(w->bits, w->K, w->N, rows, fused ? 0 : 1, sw);
        // a tuned count must still let the fused prologue hold the rows in registers
        if ((waves != 4 && waves != 8 && waves != 16) || (fused && !gemv_can_fuse(rows, w->K, waves, norm)))
            waves = fused ? gemv_fused_waves(rows, w->K, g.items, steps, norm) : gemv_pick_waves(g.items, steps);
    } else if (fused && !gemv_can_fuse(rows, w->K, waves, norm)) {
        waves = 0;
    }
    // 17..32 quantized rows: at most 8 waves (1024-thread workgroups would spill the two row
    // blocks' registers)
    if (!fused && rows > kGemvMaxRows && waves > 8) waves = 8;
    g.waves = waves;
    // More items than CUs with the quantization fused: one workgroup per CU (at most four
    // items each), so each CU quantizes the rows once.  On rows quantized beforehand, only
    // when one workgroup per item would take a second round of the CUs (1024-thread
    // workgroups one per CU, smaller ones 16 / waves per CU): 5..16 rows of gate_up 2560 x
    // 19456, 749 items of 8 waves, 15.5 -> 12.4 us at 8 rows, while qkv 2560 x 6144 (512
    // items, one round) ran 9.6 -> 10.2 us as 2 items per workgroup.
    const int per_cu = waves >= 16 || waves <= 0 ? 1 : 16 / waves;
    if (ov.gemv_grid >= 0)
        g.grid = ov.gemv_grid;
    else if (fused ? g.items > ws->cu_count : g.items > ws->cu_count * per_cu)
        g.grid = std::max(ws->cu_count, (g.items + 3) / 4);
    return g;
}

// Whether the decode GEMV may quantize (and normalize) the raw rows itself.
bool gemv_fusable(const qlin_workspace* ws, const qlin_weights* w, int rows, const void* A, int64_t lda,
                  const float* gamma, uint32_t flags) {
    if (rows > kGemvMaxRows || (flags & kFlagNoFusedQuant) || rows > ws->ov.fused_max_rows) return false;
    if ((reinterpret_cast<uintptr_t>(A) & 15) || (lda % 8) || (gamma && (reinterpret_cast<uintptr_t>(gamma) & 15)))
        return false;
    return plan_gemv(ws, w, rows, true, gamma != nullptr, flags).waves != 0;
}

int run_gemv(qlin_workspace* ws, const qlin_weights* w, int rows, const void* A, int a_f16, int64_t lda,
             const float* gamma, float eps, const int8_t* q, int64_t ldq, const float* s, void* C, int c_kind,
             int64_t ldc, uint32_t flags, hipStream_t st, const ResidualArgs* res = nullptr) {
    const GemvPlan g = plan_gemv(ws, w, rows, A != nullptr, gamma != nullptr, flags);
    if (g.waves == 0) return QLIN_ERR_UNSUPPORTED;  // callers check gemv_fusable first
    GemvParams p{};
    if (res) {
        p.R = res->R;
        p.ldr = res->ldr;
        p.r_f16 = res->r_f16;
        p.rmult = res->mult;
    }
    p.W = w->W;
    p.wscale = w->scales;
    p.wrow = w->wrow;
    p.K = w->K;
    p.Kp = w->Kp;
    p.N = w->N;
    p.Np = w->Np;
    p.M = rows;
    p.A = A;
    p.lda = lda;
    p.a_f16 = a_f16;
    p.gamma = gamma;
    p.eps = eps;
    p.q = q;
    p.ldq = ldq;
    p.s = s;
    p.C = C;
    p.ldc = ldc;
    p.c_kind = c_kind;
    p.flags = flags;
    p.err = ws->err;
    p.iw = g.iw;
    p.grid = g.grid;
    return launch_gemv(p, w->bits, g.waves, st) == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
}

// Launch shape of a prefill GEMM.
struct GemmPlan {
    int kernel;  // 32: the 32x32x32 kernel (tile configuration cfg), 16: the 16x16x64 kernel
    int cfg, bm, bn, threads;
    int m_tiles, n_tiles, splits, ktiles_per_split, group_m, deep, wn;
};

// Kernel and tile configuration for a shape.  Measured (MI355X, four Qwen3-4B linears, M = 512
// and 4096, fp16 out): the 32x32x32 kernel's 256 x 256 tile is ahead only where it leaves
// every CU several tiles (M = 4096 gate_up: 194-206 vs 212-227 us); with one round or less
// the 16x16x64 kernel is equal or ahead (M = 512: the 128 x 128 tiles of both run at the
// same copy rate, ~20 B per clock per CU), so it stays the default there.  (Where this picks the 32x32x32
// kernel without an override or a table entry, plan_rows takes the alternating-waves GEMM instead.)
// Returns -1 for the 16x16x64 kernel, else the 32x32x32 tile configuration.  `tuned` is the
// kernel field of a variant-table entry (0: none), below the environment overrides.
int gemm_pick(const qlin_workspace* ws, const qlin_weights* w, int rows, bool sw, int tuned) {
    if (ws->ov.gemm_kernel == 16) return -1;
    if (ws->ov.gemm_cfg >= 0 && ws->ov.gemm_cfg <= 3) return ws->ov.gemm_cfg == 3 && w->bits != 4 ? -1 : ws->ov.gemm_cfg;
    if (tuned == kTuneKernel16) return -1;
    if (tuned >= kTuneKernel32 && tuned <= kTuneKernel32 + 3)
        return tuned == kTuneKernel32 + 3 && w->bits != 4 ? -1 : tuned - kTuneKernel32;
    if (w->bits != 4) return -1;
    const GemmTileCfg big = gemm32_tile(w->bits, 1);
    const int cols = sw ? w->N / 2 : w->N, bcols = sw ? big.bn / 2 : big.bn;
    const int64_t big_tiles = (int64_t)((rows + big.bm - 1) / big.bm) * ((cols + bcols - 1) / bcols);
    if (big_tiles >= 4 * ws->cu_count) return 1;
    // A SiLU-gate GEMM whose 256 x 192 grid covers 3/4 to all of the CUs once (gate_up at
    // 512 tokens: 204 tiles) takes those tiles: twelve waves of 64 x 64 per CU do about 1.4x
    // the work per CU of two 128 x 128 tiles of the 16x16x64 kernel, whose 608 tiles would
    // leave a short second round (M = 512 gate_up 39.8 -> 35.2 us).
    if (sw) {
        const GemmTileCfg t3 = gemm32_tile(4, 3);
        const int64_t tiles3 = (int64_t)((rows + t3.bm - 1) / t3.bm) * ((cols + t3.bn / 2 - 1) / (t3.bn / 2));
        if (tiles3 <= ws->cu_count && 4 * tiles3 >= 3 * (int64_t)ws->cu_count) return 3;
    }
    return -1;
}

int plan_gemm(const qlin_workspace* ws, const qlin_weights* w, int rows, uint32_t flags, GemmPlan* out) {
    const QlinOverrides& ov = ws->ov;
    const bool sw = (flags & kFlagSwiglu) != 0;
    GemmPlan g{};
    const int tuned = tuned_variant(w->bits, w->K, w->N, rows, 2, sw);  // splits + step * kernel
    const int pick = gemm_pick(ws, w, rows, sw, tuned / kTuneKernelStep);
    g.kernel = pick < 0 ? 16 : 32;
    int64_t slice;  // ints of one partial tile
    if (g.kernel == 32) {
        g.cfg = pick;
        const GemmTileCfg t = gemm32_tile(w->bits, g.cfg);
        g.bm = t.bm;
        g.bn = t.bn;
        g.threads = t.threads;
        slice = (int64_t)t.regs * t.threads;
    } else {
        g.bm = kGemmTileM;
        g.bn = gemm_tile_n(w->bits, w->N);
        g.wn = ov.gemm_wn == 2 ? 2 : 4;  // 2 x 4 waves unless QLIN_GEMM_WN=2
        g.threads = 128 * g.wn;
        slice = (int64_t)gemm_regs_per_thread(g.bn) * 256;
    }
    const int cols = sw ? g.bn / 2 : g.bn;  // output channels per tile
    g.m_tiles = (rows + g.bm - 1) / g.bm;
    g.n_tiles = ((sw ? w->N / 2 : w->N) + cols - 1) / cols;
    const int ktiles = w->Kp / kGemmTileK;
    const int tiles = g.m_tiles * g.n_tiles;
    int S = ov.gemm_splits;
    if (S <= 0) S = tuned % kTuneKernelStep;
    if (S <= 0) {
        // Split K while the grid stays within one workgroup per CU (split-K's partial round
        // trip costs more than a second resident workgroup per CU gains), keeping >= 4 k
        // tiles per split, and take the count with the least estimated time: a split's
        // longest k range at ~0.45 us per k tile, plus for a split tile ~1.5 us of round
        // trips and its partials (written by every split, read by the last) at ~4.5 TB/s,
        // or ~9 TB/s when the tile count is a multiple of 8: then the XCD-contiguous order
        // puts all splits of a tile on one XCD.  Measured at M = 512 (80 tiles): o (K =
        // 4096) 15.2 us with 3 splits, 15.9 with 2; down (K = 9728) 23.8 / 26.1 us; 4
        // splits (more workgroups than CUs) 20.7 / 29.4.  With the splits of a tile on
        // different XCDs, o took 18.2 us with 2 splits, 18.9 with 3, and unsplit o / down
        // took 19.4 / 38.4 us.
        const int target = ov.gemm_target_wgs > 0 ? ov.gemm_target_wgs : ws->cu_count;
        const int smax = std::max(1, std::min((target + tiles / 2) / tiles, ktiles / 4));
        const double part_rate = tiles % 8 == 0 ? 9.0e6 : 4.5e6;  // partial bytes per us
        S = 1;
        double best = 1e30;
        for (int t = 1; t <= smax; ++t) {
            const int per = ((ktiles + t - 1) / t + 1) & ~1;  // even k tiles per split
            const double exch = t > 1 ? 1.5 + (2.0 * t - 1) * tiles * slice * 4.0 / part_rate : 0.0;
            const double est = 0.45 * per + exch;
            if (est < best - 1e-9) {
                best = est;
                S = t;
            }
        }
    }
    S = std::max(1, std::min(S, ktiles));
    while (S > 1 && ((int64_t)tiles * S * slice > ws->part_ints || tiles > ws->n_counters)) --S;
    // the 16x16x64 kernel's k loop takes two tiles per iteration: Kp is a multiple of 256,
    // so ktiles is even, and an even split size keeps every split's count even
    if (ktiles % 2) return QLIN_ERR_PARAM;
    g.ktiles_per_split = ((ktiles + S - 1) / S + 1) & ~1;
    g.splits = (ktiles + g.ktiles_per_split - 1) / g.ktiles_per_split;
    g.group_m = std::max(1, std::min(g.m_tiles, ov.gemm_group_m));
    // a grid with at most one workgroup per CU takes the deeper pipeline
    g.deep = ov.gemm_deep >= 0 ? (ov.gemm_deep != 0) : (int64_t)tiles * g.splits <= ws->cu_count;
    *out = g;
    return QLIN_OK;
}

int run_gemm(qlin_workspace* ws, const qlin_weights* w, int rows, const int8_t* q, int64_t ldq, const float* s,
             void* C, int c_kind, int64_t ldc, uint32_t flags, hipStream_t st, const ResidualArgs* res = nullptr) {
    GemmPlan g;
    if (int rc = plan_gemm(ws, w, rows, flags, &g)) return rc;
    GemmParams p{};
    if (res) {
        p.R = res->R;
        p.ldr = res->ldr;
        p.r_f16 = res->r_f16;
        p.rmult = res->mult;
    }
    p.W = w->W;
    p.wscale = w->scales;
    p.wrow = w->wrow;
    p.K = w->K;
    p.Kp = w->Kp;
    p.N = w->N;
    p.Np = w->Np;
    p.M = rows;
    p.q = q;
    p.ldq = ldq;
    p.s = s;
    p.C = C;
    p.ldc = ldc;
    p.c_kind = c_kind;
    p.flags = flags;
    p.m_tiles = g.m_tiles;
    p.n_tiles = g.n_tiles;
    p.ktiles_per_split = g.ktiles_per_split;
    p.splits = g.splits;
    p.group_m = g.group_m;
    p.part = ws->gemm_part;
    p.counters = ws->counters;
    p.deep = g.deep;
    p.wn = g.wn;
    const hipError_t e = g.kernel == 32 ? launch_gemm32(p, w->bits, g.cfg, st) : launch_gemm(p, w->bits, g.bn, st);
    return e == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
}

// Launch of a linear on quantized rows by the wave-split-K or the alternating-waves GEMM.
struct RowsPlan {
    enum Kind { kOther, kWaveSplitK, kAlternating } kind;  // kOther: the GEMV or the tiled GEMM
    int cfg, bm, tc, waves;  // tile rows, output channels
    int m_tiles, n_tiles;
};

RowsPlan rows_tiles(RowsPlan::Kind kind, int cfg, int bm, int bn, int waves, const qlin_weights* w, int rows, bool sw) {
    RowsPlan r{kind, cfg, bm, sw ? bn / 2 : bn, waves, 0, 0};
    r.m_tiles = (rows + r.bm - 1) / r.bm;
    r.n_tiles = ((sw ? w->N / 2 : w->N) + r.tc - 1) / r.tc;
    return r;
}

// Estimates of a launch on quantized rows, in us, behind the choice of its kernel.  Each is a sum of
// what the kernel does, with the factors of W4 and W8: least squares of the relative error to half of
// 21152 random shapes (K 64..32768, N 64..262144, 1..8192 rows, a third with SiLU-gate, fp16 out), each
// timed in graphs with every kernel and configuration that takes it, two thirds of them with eight copies
// of the weights in turn, the others with copies beyond the 256 MB cache, as the layers of a model have
// theirs.  rms error over the other half: wave-split-K 9%, alternating 5..7%, tiled 7..9%, GEMV 12..16%.
struct RowsCost {
    int rows, steps;          // 128-deep k steps
    double w, q, out, odd;    // MB: weights, quantized rows, fp16 outputs; outputs in rows not a multiple of 4
    int b;                    // 0: W4, 1: W8
    bool sw;
};

RowsCost rows_cost(const qlin_weights* w, int rows, bool sw) {
    const int ncols = sw ? w->N / 2 : w->N;
    RowsCost k{rows, w->Kp / 128, 1e-6 * w->N * w->wrow, 1e-6 * rows * w->Kp, 2e-6 * rows * ncols, 0.0, w->bits == 8, sw};
    if (ncols % 4) k.odd = k.out;
    return k;
}

// One round of workgroups: the KiB a workgroup copies (its rows and its weights), the partial sums'
// exchange, the MFMAs, the operands of all workgroups, the outputs, the weights and the rows once.
// Over more than 96 steps it comes out low (by a tenth at 128..255).
double ks_us(const RowsCost& k, const KsTile& t, int m_tiles, int n_tiles) {
    static constexpr double c[2][9] = {{3.08, 0.00383, 0.0127, 0.0154, 0.00245, 0.0115, 1.24, 0.0970, 0.119},
                                       {3.14, 0.00479, 0.0080, 0.0195, 0.00154, 0.0147, 0.928, 0.105, 0.103}};
    const double* f = c[k.b];
    const double own = (k.steps + t.wk - 1) / t.wk;  // k steps of the busiest wave
    const double us = f[0] + t.wk * own * (f[1] * 2 * t.mf + f[2] * t.nb * (1 + k.b)) +
                      t.wk * t.mf * t.nb * (f[3] + f[4] * own) + f[5] * (n_tiles * k.q + m_tiles * k.w) + f[6] * k.out +
                      f[7] * k.w + f[8] * k.q;
    return (k.steps > 96 ? 1.12 : 1.0) * t.rel[k.b] * us;
}

// Rounds of tiles at the configuration's cost per tile and k step, the weights once, the outputs (more
// where their rows take narrow stores), the operands of all tiles.  1.008: it comes out that much low.
double pp_us(const RowsCost& k, const PpTile& t, int tiles, int cus) {
    static constexpr double c[2][5] = {{3.16, 0.0182, 0.157, 0.581, 0.0133}, {2.97, 0.0654, 0.170, 0.598, 0.00819}};
    const double* f = c[k.b];
    const int rounds = tiles / cus + (tiles % cus != 0);
    const double operands = 128e-6 * tiles * k.steps * (t.bm + 0.5 * t.bn * (1 + k.b));
    return 1.008 * (f[0] + rounds * (t.tile_us[k.b] + k.steps * t.step_us[k.b]) + f[1] * k.w + f[2] * k.out +
                    f[3] * k.odd + f[4] * operands);
}

// The 16x16x64 tiled GEMM, unsplit or with K split over workgroups: rounds of k steps, workgroups per
// CU, operands, outputs, then the splits' exchange through memory, the weights and the rows once.
double tiled_us(const RowsCost& k, const GemmPlan& g, int cus) {
    static constexpr double c[2][2][10] = {{{4.48, 0.354, 0.238, 0.0099, 0.345, 0.547, 0.0, 0.0, 0.0355, 0.0306},
                                            {5.66, 0.355, 0.0, 0.00396, 0.744, 1.68, 0.658, 0.140, 0.0323, 0.0469}},
                                           {{3.96, 0.450, 1.45, 0.00963, 0.365, 0.540, 0.0, 0.0, 0.0382, 0.0},
                                            {4.89, 0.452, 0.0, 0.0, 1.15, 1.87, 0.704, 0.0967, 0.0661, 0.0320}}};
    const double* f = c[k.b][g.splits > 1];
    const double tiles = (double)g.m_tiles * g.n_tiles, wgs = tiles * g.splits;
    const double operands = 128e-6 * tiles * k.steps * (g.bm + 0.5 * g.bn * (1 + k.b));
    return f[0] + f[1] * std::ceil(wgs / cus) * g.ktiles_per_split + f[2] * wgs / cus + f[3] * operands + f[4] * k.out +
           f[5] * k.odd + f[6] * g.splits + f[7] * 4e-6 * wgs * g.bm * g.bn + f[8] * k.w + f[9] * k.q;
}

// The GEMV on up to 8, 16 and 32 rows: rounds of the longest wave's steps (16 waves a CU), the weights,
// the steps, the rows read for every 16 channels, the outputs, those channel groups, the second stream
// of a SiLU-gate.  Over 4..7 of its own steps (256 deep for W4) it comes out 7% high.
double gemv_us(const RowsCost& k, int N, int waves, int cus) {
    static constexpr double c[2][3][8] = {{{2.83, 0.111, 0.150, 0.0243, 7.47, 6.03, 0.0435, 0.0164},
                                           {2.97, 0.0843, 0.122, 0.0397, 12.8, 5.99, 0.0, 0.00792},
                                           {3.74, 0.301, 0.200, 0.0458, 0.0, 4.18, 0.0, 0.00271}},
                                          {{2.48, 0.270, 0.130, 0.0341, 0.0, 4.78, 0.0120, 0.0291},
                                           {2.49, 0.389, 0.0697, 0.0416, 22.7, 4.01, 0.0, 0.0203},
                                           {3.09, 0.582, 0.125, 0.0303, 0.0, 3.61, 0.0, 0.0228}}};
    const double* f = c[k.b][k.rows <= 8 ? 0 : k.rows <= 16 ? 1 : 2];
    const int groups = (N + 15) / 16, own = (k.steps + waves - 1) / waves;
    const int64_t rounds = ((int64_t)groups * waves + 16 * cus - 1) / (16 * cus);
    const double us = f[0] + f[1] * rounds * own + f[2] * k.w + f[3] * k.steps + f[4] * k.q * groups / cus +
                      f[5] * k.out + f[6] * groups / cus + (k.sw ? f[7] * k.steps : 0.0);
    const int deep = k.b ? k.steps : k.steps / 2;
    return deep >= 4 && deep < 8 ? 0.93 * us : us;
}

// Which kernel takes quantized rows: the one with the least estimate among
// - the wave-split-K GEMM in the configurations whose workgroups cover the output in one round, one per
//   CU (most rings leave room for one; a second round costs a whole launch again: gate_up at 128 rows
//   23.0 us in two rounds against 15.9 tiled),
// - the alternating-waves GEMM, above 16 rows,
// - what else takes the rows: the GEMV (gemv_ok) or the tiled GEMM.  Not its 32x32x32 kernel, whose
//   tiles are the alternating kernel's and slower on every grid.
//
// Over 3449 further shapes the choice takes 1.013 times the best of all measured (geometric mean) and 0.80
// times the GEMV or the tiled GEMM alone; 2.0% of them are over 4% slower than those, 0.4% over 10%, the
// worst 1.23x. W4 2560 x 6144 / 4096 x 2560 / 2560 x 19456 / 9728 x 2560, GEMV or tiled -> chosen, us: 16
// rows 8.0 / 5.7 / 11.2 / 9.0 -> 5.0 / 5.0 / 8.6 / 6.5; 128 rows 13.7 / 13.0 / 14.8 / 17.4 -> 8.7 / 7.3 /
// 14.1 / 11.3; 512 rows 16.1 / 15.3 / 31.6 / 22.3 -> 14.6 / 12.4 / 28.8 / 22.3; 4096 rows 71.1 / 51.3 /
// 198.6 / 107.4 -> 62.8 / 42.9 / 163.0 / 84.7.
//
// Overrides of the GEMV's or the tiled GEMM's launch shape, and table entries, select those.
RowsPlan plan_rows(const qlin_workspace* ws, const qlin_weights* w, int rows, int64_t ldq, uint32_t flags) {
    const RowsPlan other{RowsPlan::kOther, 0, 0, 0, 0, 0, 0};
    const QlinOverrides& ov = ws->ov;
    const bool sw = (flags & kFlagSwiglu) != 0, w4 = w->bits == 4;
    if (ldq > (1 << 22)) return other;  // row offsets of a tile are 32-bit
    auto ks_ok = [&](int c) { return gemm_ks_fits(w->bits, c) && !(sw && gemm_ks_tile(c).nb % 2); };
    auto pp_ok = [&](int c) {
        const PpTile t = gemm_pp_tile(c);
        return (w4 ? t.w4 : t.w8) && (sw ? t.swiglu : t.plain);
    };
    auto ks_plan = [&](int c) {
        const KsTile t = gemm_ks_tile(c);
        return rows_tiles(RowsPlan::kWaveSplitK, c, 16 * t.mf, 16 * t.nb, t.wk, w, rows, sw);
    };
    auto pp_plan = [&](int c) {
        const PpTile t = gemm_pp_tile(c);
        return rows_tiles(RowsPlan::kAlternating, c, t.bm, t.bn, 8, w, rows, sw);
    };
    if (ov.gemm_ks >= 0 && ov.gemm_ks < kKsConfigs) return ks_ok(ov.gemm_ks) ? ks_plan(ov.gemm_ks) : other;
    if (ov.gemm_pp >= 0 && ov.gemm_pp < kPpConfigs) return pp_ok(ov.gemm_pp) ? pp_plan(ov.gemm_pp) : other;
    if (ov.gemm_kernel || ov.gemm_cfg >= 0 || ov.gemm_splits > 0 || ov.gemv_waves > 0 || ov.gemv_grid >= 0 ||
        ov.gemv_item_width > 0)
        return other;
    if (tuned_variant(w->bits, w->K, w->N, rows, gemv_ok(ws, w, rows) ? 1 : 2, sw)) return other;
    const RowsCost k = rows_cost(w, rows, sw);
    const int cus = ws->cu_count;
    RowsPlan best = other;
    double best_us = 1e30;
    if (gemv_ok(ws, w, rows)) {
        best_us = gemv_us(k, w->N, plan_gemv(ws, w, rows, false, false, flags).waves, cus);
    } else {
        GemmPlan g;
        if (plan_gemm(ws, w, rows, flags, &g)) return other;
        if (g.kernel == 16) best_us = tiled_us(k, g, cus);
    }
    auto consider = [&](const RowsPlan& r, double us) {
        if (us < best_us) {
            best_us = us;
            best = r;
        }
    };
    for (int c = 0; c < kKsConfigs && ov.gemm_ks != -2; ++c) {
        if (!ks_ok(c)) continue;
        const RowsPlan r = ks_plan(c);
        if ((int64_t)r.m_tiles * r.n_tiles <= cus) consider(r, ks_us(k, gemm_ks_tile(c), r.m_tiles, r.n_tiles));
    }
    for (int c = 0; c < kPpConfigs && ov.gemm_pp != -2 && rows > 16; ++c) {
        if (!pp_ok(c)) continue;
        const RowsPlan r = pp_plan(c);
        const int64_t tiles = (int64_t)r.m_tiles * r.n_tiles;
        if (tiles <= INT32_MAX) consider(r, pp_us(k, gemm_pp_tile(c), (int)tiles, cus));
    }
    return best;
}

int run_planned(qlin_workspace* ws, const qlin_weights* w, const RowsPlan& r, int rows, const int8_t* q, int64_t ldq,
                const float* s, void* C, int c_kind, int64_t ldc, uint32_t flags, hipStream_t st,
                const ResidualArgs* res) {
    GemmParams p{};
    if (res) {
        p.R = res->R;
        p.ldr = res->ldr;
        p.r_f16 = res->r_f16;
        p.rmult = res->mult;
    }
    p.W = w->W;
    p.wscale = w->scales;
    p.wrow = w->wrow;
    p.K = w->K;
    p.Kp = w->Kp;
    p.N = w->N;
    p.Np = w->Np;
    p.M = rows;
    p.q = q;
    p.ldq = ldq;
    p.s = s;
    p.C = C;
    p.ldc = ldc;
    p.c_kind = c_kind;
    p.flags = flags;
    p.m_tiles = r.m_tiles;
    p.n_tiles = r.n_tiles;
    p.group_m = std::max(1, std::min(r.m_tiles, ws->ov.gemm_group_m));
    const hipError_t e = r.kind == RowsPlan::kWaveSplitK ? launch_gemm_ks(p, w->bits, r.cfg, st)
                                                         : launch_gemm_pp(p, w->bits, r.cfg, ws->cu_count, st);
    return e == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
}

// The linear on rows already quantized.
int run_rows(qlin_workspace* ws, const qlin_weights* w, int rows, const int8_t* q, int64_t ldq, const float* s, void* C,
             int c_kind, int64_t ldc, uint32_t flags, hipStream_t st, const ResidualArgs* res = nullptr) {
    const RowsPlan r = plan_rows(ws, w, rows, ldq, flags);
    if (r.kind != RowsPlan::kOther) return run_planned(ws, w, r, rows, q, ldq, s, C, c_kind, ldc, flags, st, res);
    if (gemv_ok(ws, w, rows))
        return run_gemv(ws, w, rows, nullptr, 0, 0, nullptr, 0.0f, q, ldq, s, C, c_kind, ldc, flags, st, res);
    return run_gemm(ws, w, rows, q, ldq, s, C, c_kind, ldc, flags, st, res);
}

int check_run(const qlin_workspace* ws, const qlin_weights* w, int rows, uint32_t flags) {
    if (!ws || !w || rows <= 0 || rows > ws->max_rows) return QLIN_ERR_PARAM;
    if (w->Kp > ws->max_kp || w->Np > ws->max_np) return QLIN_ERR_PARAM;
    if (w->device != ws->device) return QLIN_ERR_PARAM;
    // SiLU-gate pairs column j with j + N/2: any even N
    if ((flags & kFlagSwiglu) && (w->N & 1)) return QLIN_ERR_UNSUPPORTED;
    return QLIN_OK;
}

int run_impl(qlin_workspace* ws, const qlin_weights* w, int rows, const void* A, int a_dtype, int64_t lda,
             const float* gamma, float eps, void* C, int c_dtype, int64_t ldc, uint32_t flags, hipStream_t st,
             const ResidualArgs* res = nullptr) {
    if (int rc = check_run(ws, w, rows, flags)) return rc;
    if (!A || !C || lda < w->K || (a_dtype != QLIN_F32 && a_dtype != QLIN_F16) ||
        (c_dtype != QLIN_F32 && c_dtype != QLIN_F16))
        return QLIN_ERR_PARAM;
    const int ncols = (flags & kFlagSwiglu) ? w->N / 2 : w->N;
    if (ldc < ncols) return QLIN_ERR_PARAM;
    if (gamma && !(eps > 0.0f && std::isfinite(eps))) return QLIN_ERR_PARAM;
    ws->last = st;
    ws->err_used = true;
    if (gemv_fusable(ws, w, rows, A, lda, gamma, flags)) {
        return run_gemv(ws, w, rows, A, a_dtype == QLIN_F16, lda, gamma, eps, nullptr, 0, nullptr, C,
                        c_dtype == QLIN_F16, ldc, flags, st, res);
    }
    QuantParams qp{};
    qp.A = A;
    qp.lda = lda;
    qp.a_f16 = a_dtype == QLIN_F16;
    qp.K = w->K;
    qp.ldq = w->Kp;
    qp.q = ws->q;
    qp.s = ws->s;
    qp.err = ws->err;
    qp.gamma = gamma;
    qp.eps = eps;
    qp.flags = flags & ~kFlagErrOnHost;
    if (launch_quant(qp, rows, st) != hipSuccess) return QLIN_ERR_DEVICE;
    return run_rows(ws, w, rows, ws->q, w->Kp, ws->s, C, c_dtype == QLIN_F16, ldc, flags, st, res);
}

// Host-buffer run through device copies of the rows (pageable copies both ways).
int run_host_copies(qlin_workspace* ws, const qlin_weights* w, int rows, const float* A, float* C, int ncols,
                    uint32_t flags) {
    hipStream_t st = ws->stream;
    ws->err_used = true;
    if (hipMemsetAsync(ws->err, 0, sizeof(uint32_t), st) != hipSuccess) return QLIN_ERR_DEVICE;
    if (hipMemcpyAsync(ws->dA, A, (size_t)rows * w->K * sizeof(float), hipMemcpyHostToDevice, st) != hipSuccess)
        return QLIN_ERR_DEVICE;
    if (int rc = run_impl(ws, w, rows, ws->dA, QLIN_F32, w->K, nullptr, 0.0f, ws->dC, QLIN_F32, ncols, flags, st))
        return rc;
    if (hipMemcpyAsync(C, ws->dC, (size_t)rows * ncols * sizeof(float), hipMemcpyDeviceToHost, st) != hipSuccess)
        return QLIN_ERR_DEVICE;
    uint32_t e = 0;
    if (hipMemcpyAsync(&e, ws->err, sizeof(e), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
        return QLIN_ERR_DEVICE;
    return e ? QLIN_ERR_NONFINITE : QLIN_OK;
}

// Whether rows take longer in `blocks` pinned blocks than through device copies.  Every block
// streams all the weights and goes through a product of its own, K long; the copies do that once,
// but move the rows out at half the speed.  Two least-squares fits (7% and 13% rms) to 497 random
// shapes timed both ways (K 64..32768, N 64..262144, 2..1024 rows, weights to 500 MB): us, W and
// the rows in and out in MB.  With the 0.82, for the fits' error, one of those and of 366 shapes
// that the fits had not seen takes 5% longer than through copies and none more; without the rule 41
// of the 497 did, up to 2.1x.  W4 / W8 of 2560 x 151936 at 128 rows, a row a block: 5963 / 9549 us ->
// 4586 / 4642; W8 28672 x 8192, 15 blocks: 1064 -> 758; W8 32160 x 190 at 212 rows, a long K: 1250 ->
// 844; W4 2560 x 19456 at 128 rows, 10 blocks, stays at 358 (through copies 687).
bool blocks_lag(const qlin_weights* w, int rows, int blocks, size_t row_in, size_t row_out) {
    const double W = 1e-6 * w->N * w->wrow, in = 1e-6 * rows * row_in, out = 1e-6 * rows * row_out;
    const double block_us = 0.9 + 0.43e-3 * w->K + 0.36 * std::max(0.4 * W, 19.0 * out / blocks);
    return 21.0 + blocks * block_us + 25.5 * in + 30.0 * out > 0.82 * (58.0 + 0.256 * W + 32.6 * in + 55.0 * out);
}

// Host-buffer run in blocks of rows through pinned slots that the kernels read and write
// themselves: the quantize launch reads a block's rows over the bus (each row once), the GEMM
// stores its f32 rows straight into the slot, and while the GPU works on a block the host
// copies the next one in and the last one out.  What it replaces: pageable copies both ways
// (the runtime stages or pins the caller's pages on every call), a memset and a read of the
// error word, each a round trip of its own.  W4 Qwen3-4B linears, us per call on average: 1 row
// 50.7 -> 22.4, 128 rows 335 -> 207 (20.5 MB over the bus per four calls take 97 per call at 53
// GB/s; the reads, products and writes of one block are in a row on the stream).  Slots of 2 /
// 0.5 MiB took 229 / 229, a second stream for the odd blocks 203, copies by the DMA engine from
// device memory 310 (a small one alone costs 8-11 us).
int run_host(qlin_workspace* ws, const qlin_weights* w, int rows, const float* A, float* C, uint32_t flags) {
    if (int rc = check_run(ws, w, rows, flags)) return rc;
    if (!A || !C) return QLIN_ERR_PARAM;
    if (w->K > ws->max_k || w->N > ws->max_n) return QLIN_ERR_PARAM;
    const int ncols = (flags & kFlagSwiglu) ? w->N / 2 : w->N;
    const size_t row_in = (size_t)w->K * sizeof(float), row_out = (size_t)ncols * sizeof(float);
    const size_t per_slot = kSlotBytes / std::max(row_in, row_out);
    // rows whose quantization would read them by elements, or longer than a slot; buffers that
    // overlap, where a block's rows out could land on rows that are still to go in; weights that
    // cost more to stream for every block than the blocks save; a thread on another device, whose
    // events this stream could not record
    const uintptr_t a0 = reinterpret_cast<uintptr_t>(A), c0 = reinterpret_cast<uintptr_t>(C);
    const bool overlap = a0 < c0 + (size_t)rows * row_out && c0 < a0 + (size_t)rows * row_in;
    const int blocks = per_slot ? (int)((rows + per_slot - 1) / per_slot) : 0;
    int device = -1;
    if (w->K % 8 || blocks == 0 || overlap || blocks_lag(w, rows, blocks, row_in, row_out) ||
        hipGetDevice(&device) != hipSuccess || device != ws->device)
        return run_host_copies(ws, w, rows, A, C, ncols, flags);
    HostStage* h = take_stage(ws->device);
    if (!h) return run_host_copies(ws, w, rows, A, C, ncols, flags);
    hipStream_t st = ws->stream;
    ws->last = st;
    uint32_t* err_host = reinterpret_cast<uint32_t*>(h->mem + 2 * kSlots * kSlotBytes);
    *err_host = 0;
    const int step = (rows + blocks - 1) / blocks;
    int rc = QLIN_OK;
    // the workspace's word reports this call, as every host-buffer call's
    if (ws->err_used && hipMemsetAsync(ws->err, 0, sizeof(uint32_t), st) != hipSuccess) rc = QLIN_ERR_DEVICE;
    auto rows_of = [&](int b) { return std::min(step, rows - b * step); };
    auto finish = [&](int b) {  // waits for block b and copies its rows out
        if (!rc && hipEventSynchronize(h->done[b % kSlots]) != hipSuccess) rc = QLIN_ERR_DEVICE;
        if (!rc)
            std::memcpy(C + (size_t)b * step * ncols, h->mem + (2 * (b % kSlots) + 1) * kSlotBytes, rows_of(b) * row_out);
    };
    int issued = 0;
    for (int b = 0; b * step < rows && !rc; ++b) {
        if (b >= kSlots) finish(b - kSlots);
        if (rc) break;
        const int slot = b % kSlots, m = rows_of(b);
        const size_t in = 2 * slot * kSlotBytes, out = in + kSlotBytes;
        std::memcpy(h->mem + in, A + (size_t)b * step * w->K, m * row_in);
        QuantParams qp{};
        qp.A = h->dev + in;
        qp.lda = w->K;
        qp.K = w->K;
        qp.ldq = w->Kp;
        qp.q = ws->q;
        qp.s = ws->s;
        qp.err = reinterpret_cast<uint32_t*>(h->dev + 2 * kSlots * kSlotBytes);
        qp.flags = flags | kFlagErrOnHost;
        if (launch_quant(qp, m, st) != hipSuccess) rc = QLIN_ERR_DEVICE;
        if (!rc) rc = run_rows(ws, w, m, ws->q, w->Kp, ws->s, h->dev + out, 0, ncols, flags, st);
        if (!rc && hipEventRecord(h->done[slot], st) != hipSuccess) rc = QLIN_ERR_DEVICE;
        issued = b + 1;
    }
    for (int b = std::max(0, issued - kSlots); b < issued; ++b) finish(b);
    if (rc) {
        (void)hipStreamSynchronize(st);  // nothing still uses the set
    } else if (*const_cast<volatile uint32_t*>(err_host)) {
        rc = QLIN_ERR_NONFINITE;
        ws->err_used = true;  // so that the next call clears it
        if (hipMemcpyAsync(ws->err, err_host, sizeof(uint32_t), hipMemcpyHostToDevice, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess)
            rc = QLIN_ERR_DEVICE;
    }
    give_back_stage(h);
    return rc;
}

}  // namespace

extern "C" {

int qlin_run_f32(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const float* A, float* C) {
    return run_host(ws, w, rows, A, C, 0);
}

int qlin_run_swiglu_f32(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const float* A, float* C) {
    return run_host(ws, w, rows, A, C, kFlagSwiglu);
}

int qlin_run(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const void* A, int32_t a_dtype,
             int64_t lda, void* C, int32_t c_dtype, int64_t ldc, uint32_t flags, void* stream) {
    return run_impl(ws, w, rows, A, a_dtype, lda, nullptr, 0.0f, C, c_dtype, ldc, flags, (hipStream_t)stream);
}

int qlin_run_rmsnorm(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const void* A, int32_t a_dtype,
                     int64_t lda, const float* gamma, float eps, void* C, int32_t c_dtype, int64_t ldc,
                     uint32_t flags, void* stream) {
    if (!gamma) return QLIN_ERR_PARAM;
    return run_impl(ws, w, rows, A, a_dtype, lda, gamma, eps, C, c_dtype, ldc, flags, (hipStream_t)stream);
}

int qlin_run_residual(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const void* A, int32_t a_dtype,
                      int64_t lda, const void* R, int32_t r_dtype, int64_t ldr, float multiplier, void* C,
                      int32_t c_dtype, int64_t ldc, uint32_t flags, void* stream) {
    if (!w || (flags & kFlagSwiglu) || !R || (r_dtype != QLIN_F32 && r_dtype != QLIN_F16) || ldr < w->N ||
        !std::isfinite(multiplier))
        return QLIN_ERR_PARAM;
    // in place (the reference's hidden += projected) only element for element
    if (R == C && (ldr != ldc || r_dtype != c_dtype)) return QLIN_ERR_PARAM;
    const ResidualArgs res{R, ldr, r_dtype == QLIN_F16 ? 1 : 0, multiplier};
    return run_impl(ws, w, rows, A, a_dtype, lda, nullptr, 0.0f, C, c_dtype, ldc, flags, (hipStream_t)stream, &res);
}

int qlin_gemm_i32(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const int8_t* q, int64_t ldq,
                  int32_t* acc, int64_t ldacc, void* stream) {
    if (int rc = check_run(ws, w, rows, 0)) return rc;
    if (!q || !acc || ldq < w->Kp || ldq % 16 || (reinterpret_cast<uintptr_t>(q) & 15) || ldacc < w->N)
        return QLIN_ERR_PARAM;
    ws->last = (hipStream_t)stream;
    return run_rows(ws, w, rows, q, ldq, nullptr, acc, 2, ldacc, 0, (hipStream_t)stream);
}

int qlin_run_quantized(qlin_workspace* ws, const qlin_weights* w, int32_t rows, const int8_t* q, int64_t ldq,
                       const float* s, void* C, int32_t c_dtype, int64_t ldc, uint32_t flags, void* stream) {
    if (int rc = check_run(ws, w, rows, flags)) return rc;
    const int ncols = (flags & kFlagSwiglu) ? w->N / 2 : w->N;
    if (!q || !s || !C || ldq < w->Kp || ldq % 16 || (reinterpret_cast<uintptr_t>(q) & 15) || ldc < ncols ||
        (c_dtype != QLIN_F32 && c_dtype != QLIN_F16))
        return QLIN_ERR_PARAM;
    hipStream_t st = (hipStream_t)stream;
    ws->last = st;
    return run_rows(ws, w, rows, q, ldq, s, C, c_dtype == QLIN_F16, ldc, flags, st);
}

int qlin_run_plan(const qlin_workspace* ws, const qlin_weights* w, int32_t rows, const void* A, int64_t lda,
                  const float* gamma, uint32_t flags, qlin_plan* out) {
    if (!out || !A) return QLIN_ERR_PARAM;
    if (int rc = check_run(ws, w, rows, flags)) return rc;
    std::memset(out, 0, sizeof(*out));
    if (gemv_fusable(ws, w, rows, A, lda, gamma, flags)) {
        const GemvPlan g = plan_gemv(ws, w, rows, true, gamma != nullptr, flags);
        out->path = QLIN_PATH_GEMV_FUSED;
        out->launches = 1;
        out->waves = g.waves;
        out->item_width = g.iw;
        out->items = g.items;
        out->grid = g.grid > 0 && g.grid < g.items ? g.grid : g.items;
        return QLIN_OK;
    }
    out->launches = 2;
    const RowsPlan r = plan_rows(ws, w, rows, w->Kp, flags);
    if (r.kind != RowsPlan::kOther) {
        out->path = gemv_ok(ws, w, rows) ? QLIN_PATH_GEMV : QLIN_PATH_GEMM;
        out->waves = r.waves;
        out->tile_m = r.bm;
        out->tile_n = out->item_width = r.tc;
        out->items = out->grid = r.m_tiles * r.n_tiles;
        if (r.kind == RowsPlan::kAlternating) out->grid = std::min(out->items, ws->cu_count);
        out->splits = 1;
        return QLIN_OK;
    }
    if (gemv_ok(ws, w, rows)) {
        const GemvPlan g = plan_gemv(ws, w, rows, false, false, flags);
        out->path = QLIN_PATH_GEMV;
        out->waves = g.waves;
        out->item_width = g.iw;
        out->items = g.items;
        out->grid = g.items;
        return QLIN_OK;
    }
    GemmPlan g;
    if (int rc = plan_gemm(ws, w, rows, flags, &g)) return rc;
    out->path = QLIN_PATH_GEMM;
    out->waves = g.threads / 64;
    out->tile_m = g.bm;
    out->tile_n = (flags & kFlagSwiglu) ? g.bn / 2 : g.bn;
    out->items = g.m_tiles * g.n_tiles;
    out->splits = g.splits;
    out->grid = out->items * g.splits;
    return QLIN_OK;
}

int qlin_swiglu(int32_t rows, int32_t F, const void* X, int32_t x_dtype, int64_t ldx, void* Y, int32_t y_dtype,
                int64_t ldy, void* stream) {
    if (rows <= 0 || F <= 0 || !X || !Y || ldx < 2 * (int64_t)F || ldy < F ||
        (x_dtype != QLIN_F32 && x_dtype != QLIN_F16) || (y_dtype != QLIN_F32 && y_dtype != QLIN_F16))
        return QLIN_ERR_PARAM;
    return launch_swiglu(rows, F, X, x_dtype == QLIN_F16, ldx, Y, y_dtype == QLIN_F16, ldy, (hipStream_t)stream) ==
                   hipSuccess
               ? QLIN_OK
               : QLIN_ERR_DEVICE;
}

}  // extern "C"

// ---- runs without a workspace: scratch in a static device array --------------------
//
// qlin_run_noalloc serves callers that cannot allocate (code under HIP graph capture,
// tight serving loops).  Its scratch lives in `scratch`, a file-scope device array of
// kScratchBytes (32.05 MiB) that every GPU the library runs on holds until the process
// ends.  Layout: the error word, the split-K tile counters (zero at rest: the GEMM's
// last workgroup per tile re-zeroes its counter), the per-token scales, the quantized
// rows, the split-K partial sums.  In host code `scratch` names a host-side stand-in,
// not device memory: its device address is looked up once per device with
// hipGetSymbolAddress, and only that address is passed to kernels.

namespace {

constexpr size_t kNaErr = 0;                                   // uint32 error word (256 B)
constexpr int kNaCounters = 8192;                              // split-K tile counters
constexpr size_t kNaCountersOff = 256;
constexpr int kNaMaxRows = 4096;                               // rows per call
constexpr size_t kNaScalesOff = kNaCountersOff + kNaCounters * 4;          // 33,024
constexpr size_t kNaQOff = (kNaScalesOff + kNaMaxRows * 4 + 255) / 256 * 256;  // 49,408
constexpr size_t kNaQBytes = (size_t)16 << 20;                 // rows x K_padded <= 16 MiB
constexpr size_t kNaPartOff = kNaQOff + kNaQBytes;
constexpr int64_t kNaPartInts = (int64_t)4 << 20;              // 16 MiB of split-K partials
constexpr size_t kScratchBytes = kNaPartOff + (size_t)kNaPartInts * 4;
static_assert(kNaPartOff % 256 == 0 && kNaQOff % 256 == 0, "scratch regions stay 256-byte aligned");

}  // namespace

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace {

// Input of a variant search: fp16 values in [-2, 2) from a hash of the index.
__global__ void tune_fill_kernel(_Float16* a, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        uint32_t h = (uint32_t)i * 2654435761u;
        h ^= h >> 15;
        h *= 2246822519u;
        h ^= h >> 13;
        a[i] = (_Float16)((float)(h & 0xffffu) * (4.0f / 65536.0f) - 2.0f);
    }
}

__global__ void zero_words_kernel(uint32_t* p, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

constexpr int kNaMaxDevices = 64;
struct NoAllocDevice {
    std::atomic<uint8_t*> ptr{nullptr};  // device address of `scratch` on this device
    int cu_count = 0;
    QlinOverrides ov{};
};
NoAllocDevice g_noalloc[kNaMaxDevices];
std::mutex g_noalloc_mutex;

// Device address of this device's `scratch` (the current device must be `dev`).  The first
// call on a device looks it up and clears the error word and counters with a fill kernel on
// `st` (a kernel rather than a memset node, should the caller be capturing a graph).
int noalloc_scratch(int dev, hipStream_t st, uint8_t** out) {
    if (dev < 0 || dev >= kNaMaxDevices) return QLIN_ERR_NODEVICE;
    uint8_t* p = g_noalloc[dev].ptr.load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> g(g_noalloc_mutex);
        p = g_noalloc[dev].ptr.load(std::memory_order_relaxed);
        if (!p) {
            void* sym = nullptr;
            if (hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)) != hipSuccess || !sym) return QLIN_ERR_DEVICE;
            uint8_t* base = static_cast<uint8_t*>(sym);
            const int words = (int)(kNaScalesOff / 4);  // the error word's block and the counters
            hipLaunchKernelGGL(zero_words_kernel, dim3(32), dim3(256), 0, st, reinterpret_cast<uint32_t*>(base), words);
            if (hipGetLastError() != hipSuccess) return QLIN_ERR_DEVICE;
            g_noalloc[dev].cu_count = cu_count(dev);
            g_noalloc[dev].ov = read_overrides();
            g_noalloc[dev].ptr.store(base, std::memory_order_release);
            p = base;
        }
    }
    *out = p;
    return QLIN_OK;
}

}  // namespace

extern "C" int qlin_run_noalloc(const qlin_weights* w, int32_t rows, const void* A, int32_t a_dtype, int64_t lda,
                                const float* gamma, float eps, void* C, int32_t c_dtype, int64_t ldc, uint32_t flags,
                                uint32_t* err, void* stream) {
    if (!w || rows <= 0) return QLIN_ERR_PARAM;
    if (rows > kNaMaxRows || (int64_t)rows * w->Kp > (int64_t)kNaQBytes) return QLIN_ERR_UNSUPPORTED;
    int dev;
    if (int rc = current_device(&dev)) return rc;
    if (dev != w->device) return QLIN_ERR_PARAM;
    const hipStream_t st = (hipStream_t)stream;
    uint8_t* base = nullptr;
    if (int rc = noalloc_scratch(dev, st, &base)) return rc;
    // a workspace on the stack whose every buffer is a region of `scratch`
    qlin_workspace ws{};
    ws.max_rows = kNaMaxRows;
    ws.max_k = w->K;
    ws.max_n = w->N;
    ws.max_kp = w->Kp;
    ws.max_np = w->Np;
    ws.device = dev;
    ws.cu_count = g_noalloc[dev].cu_count;
    ws.ov = g_noalloc[dev].ov;
    ws.q = reinterpret_cast<int8_t*>(base + kNaQOff);
    ws.s = reinterpret_cast<float*>(base + kNaScalesOff);
    ws.counters = reinterpret_cast<uint32_t*>(base + kNaCountersOff);
    ws.n_counters = kNaCounters;
    ws.gemm_part = reinterpret_cast<int32_t*>(base + kNaPartOff);
    ws.part_ints = kNaPartInts;
    ws.err = err ? err : reinterpret_cast<uint32_t*>(base + kNaErr);
    ws.last = st;
    return run_impl(&ws, w, rows, A, a_dtype, lda, gamma, eps, C, c_dtype, ldc, flags, st);
}

// ---- decode chain --------------------------------------------------------------

#include "qlin_chain.hpp"

struct qlin_chain {
    int n, max_rows, device, grid;
    int x_cols;        // chain-input columns read by the stages
    int last_cols;     // output columns of the last stage
    int kp_max, k_max, kg_max, ipw_max;
    size_t lds;
    ChainParams layout;              // LDS carve-up
    std::vector<ChainStage> stages;  // host copy
    std::vector<int> cols;           // output columns per stage
    ChainStage* d_stages;
    std::vector<_Float16*> outs;     // per stage, null for the last
    std::vector<int64_t> ld;
    uint32_t* flags;   // [n][kChainFlagStride] completion epochs
    uint32_t* epochs;  // [grid] launches per workgroup
    uint32_t* err;
    int spin_limit;  // polls per stage wait before the kernel gives up (QLIN_CHAIN_SPIN_LIMIT)
    hipStream_t last;
};

void qlin_chain_free(qlin_chain* c) {
    if (!c) return;
    if (c->last) (void)hipStreamSynchronize(c->last);
    for (auto* o : c->outs) (void)hipFree(o);
    (void)hipFree(c->d_stages);
    (void)hipFree(c->flags);
    (void)hipFree(c->epochs);
    (void)hipFree(c->err);
    delete c;
}

// Items of a stage: each of the grid's workgroups owns ipw items of iw <= 16 output
// channels, the fewest channels per workgroup that cover the stage.
static void chain_items(int cols, int grid, int* iw, int* ipw) {
    const int per = (cols + grid - 1) / grid;
    *ipw = (per + 15) / 16;
    *iw = (per + *ipw - 1) / *ipw;
}

int qlin_chain_create(const qlin_chain_stage* st, int32_t n, int32_t max_rows, qlin_chain** out) {
    if (!out) return QLIN_ERR_PARAM;
    *out = nullptr;
    if (!st || n < 1 || max_rows < 1 || max_rows > 4) return QLIN_ERR_PARAM;
    int dev;
    if (int rc = current_device(&dev)) return rc;
    auto* c = new (std::nothrow) qlin_chain();
    if (!c) return QLIN_ERR_NOMEM;
    c->n = n;
    c->max_rows = max_rows;
    c->device = dev;
    c->grid = cu_count(dev);
    c->spin_limit = env_int("QLIN_CHAIN_SPIN_LIMIT", 1 << 18);  // ~0.3 s of polling per wait
    c->stages.resize(n);
    c->cols.resize(n);
    c->outs.assign(n, nullptr);
    c->ld.assign(n, 0);
    const uint32_t allowed = QLIN_SWIGLU | QLIN_ROUND_HALF_EVEN | QLIN_NORM_SEQUENTIAL | QLIN_RESIDUAL;
    int rc = c->grid > 0 && c->grid <= kChainFlagStride ? QLIN_OK : QLIN_ERR_UNSUPPORTED;
    for (int s = 0; s < n && rc == QLIN_OK; ++s) {
        const qlin_chain_stage& d = st[s];
        const qlin_weights* w = d.weights;
        if (!w || w->device != dev || (d.flags & ~allowed) || w->K % 8 || d.input < -1 || d.input >= s ||
            d.input_offset < 0 || d.input_offset % 8 || (s == 0 && d.input != -1)) {
            rc = QLIN_ERR_PARAM;
            break;
        }
        if ((d.flags & QLIN_SWIGLU) && w->N % 2) {
            rc = QLIN_ERR_PARAM;
            break;
        }
        if ((int64_t)w->Np * w->wrow >= ((int64_t)1 << 31)) {  // 32-bit buffer offsets
            rc = QLIN_ERR_UNSUPPORTED;
            break;
        }
        if (d.gamma && (!(d.eps > 0.0f && std::isfinite(d.eps)) || (reinterpret_cast<uintptr_t>(d.gamma) & 15))) {
            rc = QLIN_ERR_PARAM;
            break;
        }
        c->cols[s] = (d.flags & QLIN_SWIGLU) ? w->N / 2 : w->N;
        if (d.flags & QLIN_RESIDUAL) {
            if ((d.flags & QLIN_SWIGLU) || d.residual < -1 || d.residual >= s || d.residual_offset < 0 ||
                d.residual_offset % 8 || !std::isfinite(d.residual_multiplier) ||
                (d.residual >= 0 && d.residual_offset + c->cols[s] > c->cols[d.residual])) {
                rc = QLIN_ERR_PARAM;
                break;
            }
            if (d.residual == -1) c->x_cols = std::max(c->x_cols, d.residual_offset + c->cols[s]);
        }
        if (d.input == -1) {
            c->x_cols = std::max(c->x_cols, d.input_offset + w->K);
        } else if (d.input_offset + w->K > c->cols[d.input]) {
            rc = QLIN_ERR_PARAM;
            break;
        }
        ChainStage& cs = c->stages[s];
        cs.W = w->W;
        cs.wscale = w->scales;
        cs.wrow = w->wrow;
        cs.bits = w->bits;
        cs.K = w->K;
        cs.Kp = w->Kp;
        cs.N = w->N;
        cs.Np = w->Np;
        cs.flags = (int)(d.flags & (kFlagSwiglu | kFlagRne | kFlagNormSeq));
        cs.ncols = c->cols[s];
        chain_items(cs.ncols, c->grid, &cs.iw, &cs.ipw);
        cs.steps = w->Kp / (w->bits == 4 ? 256 : 128);
        cs.gamma = d.gamma;
        cs.eps = d.eps;
        cs.x_offset = d.input == -1 ? d.input_offset : 0;
        cs.res_kind = (d.flags & QLIN_RESIDUAL) ? (d.residual == -1 ? 1 : 2) : 0;
        cs.res_stage = cs.res_kind == 2 ? d.residual : -1;
        cs.res_x_offset = cs.res_kind == 1 ? d.residual_offset : 0;
        cs.rmult = d.residual_multiplier;
        c->kp_max = std::max(c->kp_max, w->Kp);
        c->k_max = std::max(c->k_max, w->K);
        if (d.gamma) c->kg_max = std::max(c->kg_max, w->K);
        c->ipw_max = std::max(c->ipw_max, cs.ipw);
    }
    if (rc == QLIN_OK) {
        c->last_cols = c->cols[n - 1];
        c->lds = chain_lds_layout(max_rows, c->kp_max, c->k_max, c->kg_max, c->ipw_max, &c->layout);
        if (c->lds > (size_t)kChainMaxLds) rc = QLIN_ERR_UNSUPPORTED;
    }
    // one workgroup per CU; every workgroup must be resident for the stage waits
    if (rc == QLIN_OK && chain_resident_per_cu(max_rows, c->lds) < 1) rc = QLIN_ERR_UNSUPPORTED;
    for (int s = 0; s < n - 1 && rc == QLIN_OK; ++s) {
        c->ld[s] = round_up(c->cols[s], 8);
        if (hipMalloc(&c->outs[s], (size_t)max_rows * c->ld[s] * sizeof(_Float16)) != hipSuccess) rc = QLIN_ERR_NOMEM;
    }
    for (int s = 0; s < n && rc == QLIN_OK; ++s) {
        ChainStage& cs = c->stages[s];
        const int in = st[s].input;
        cs.in = in >= 0 ? reinterpret_cast<const __half*>(c->outs[in]) + st[s].input_offset : nullptr;
        cs.ld_in = in >= 0 ? c->ld[in] : 0;
        cs.out = c->outs[s];
        cs.ld_out = c->ld[s];
        if (cs.res_kind == 2) {
            cs.res = reinterpret_cast<const __half*>(c->outs[st[s].residual]) + st[s].residual_offset;
            cs.ld_res = c->ld[st[s].residual];
        }
    }
    const size_t flag_bytes = sizeof(uint32_t) * (size_t)n * kChainFlagStride;
    if (rc == QLIN_OK &&
        (hipMalloc(&c->d_stages, sizeof(ChainStage) * n) != hipSuccess || hipMalloc(&c->flags, flag_bytes) != hipSuccess ||
         hipMalloc(&c->epochs, sizeof(uint32_t) * c->grid) != hipSuccess || hipMalloc(&c->err, sizeof(uint32_t)) != hipSuccess))
        rc = QLIN_ERR_NOMEM;
    if (rc == QLIN_OK &&
        (hipMemcpy(c->d_stages, c->stages.data(), sizeof(ChainStage) * n, hipMemcpyHostToDevice) != hipSuccess ||
         hipMemset(c->flags, 0, flag_bytes) != hipSuccess ||
         hipMemset(c->epochs, 0, sizeof(uint32_t) * c->grid) != hipSuccess ||
         hipMemset(c->err, 0, sizeof(uint32_t)) != hipSuccess || hipDeviceSynchronize() != hipSuccess))
        rc = QLIN_ERR_DEVICE;
    if (rc != QLIN_OK) {
        qlin_chain_free(c);
        return rc;
    }
    *out = c;
    return QLIN_OK;
}

int qlin_chain_run(qlin_chain* c, int32_t rows, const void* x, int64_t ldx, void* y, int64_t ldy, void* stream) {
    if (!c || rows < 1 || rows > c->max_rows || !x || !y || ldx < c->x_cols || ldx % 8 ||
        (reinterpret_cast<uintptr_t>(x) & 15) || ldy < c->last_cols || (reinterpret_cast<uintptr_t>(y) & 1))
        return QLIN_ERR_PARAM;
    int dev;
    if (int rc = current_device(&dev)) return rc;
    if (dev != c->device) return QLIN_ERR_PARAM;
    ChainParams p = c->layout;
    p.stages = c->d_stages;
    p.n_stages = c->n;
    p.M = rows;
    p.x = reinterpret_cast<const __half*>(x);
    p.ldx = ldx;
    p.y = reinterpret_cast<_Float16*>(y);
    p.ldy = ldy;
    p.flags = c->flags;
    p.epochs = c->epochs;
    p.err = c->err;
    p.spin_limit = c->spin_limit;
    p.kp_max = c->kp_max;
    const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    c->last = st;
    return launch_chain(p, c->grid, c->lds, st) == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
}

int qlin_chain_set_wait_limit(qlin_chain* c, int32_t polls) {
    if (!c || polls < 0) return QLIN_ERR_PARAM;
    c->spin_limit = polls;
    return QLIN_OK;
}

int qlin_chain_stage_output(const qlin_chain* c, int32_t stage, void** ptr, int64_t* ld) {
    if (!c || !ptr || !ld || stage < 0 || stage >= c->n - 1) return QLIN_ERR_PARAM;
    *ptr = c->outs[stage];
    *ld = c->ld[stage];
    return QLIN_OK;
}

int qlin_chain_status(qlin_chain* c, int32_t clear) {
    if (!c) return QLIN_ERR_PARAM;
    if (hipStreamSynchronize(c->last) != hipSuccess) return QLIN_ERR_DEVICE;
    uint32_t e = 0;
    if (hipMemcpy(&e, c->err, sizeof(e), hipMemcpyDeviceToHost) != hipSuccess) return QLIN_ERR_DEVICE;
    // a wait that gave up leaves nothing to repair: every workgroup still ran the launch
    // to its end and counted its epoch, so the next launch's flags are all fresh
    if (clear && e && hipMemset(c->err, 0, sizeof(uint32_t)) != hipSuccess) return QLIN_ERR_DEVICE;
    if (hipDeviceSynchronize() != hipSuccess) return QLIN_ERR_DEVICE;
    return (e & 2u) ? QLIN_ERR_DEVICE : (e ? QLIN_ERR_NONFINITE : QLIN_OK);
}

// ---- kernel-variant selection ---------------------------------------------------------

int qlin_tune(qlin_workspace* ws, const qlin_weights* w, int32_t rows, uint32_t flags, int32_t reps, void* stream) {
    if (!ws || !w || rows <= 0 || rows > ws->max_rows || reps < 1 || (flags & ~(uint32_t)QLIN_SWIGLU)) return QLIN_ERR_PARAM;
    if (int rc = check_run(ws, w, rows, flags)) return rc;
    const bool sw = (flags & kFlagSwiglu) != 0;
    const int ncols = sw ? w->N / 2 : w->N;
    const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    _Float16 *A = nullptr, *C = nullptr;
    const size_t a_bytes = (size_t)rows * w->K * sizeof(_Float16), c_bytes = (size_t)rows * ncols * sizeof(_Float16);
    if (hipMalloc(&A, a_bytes) != hipSuccess || hipMalloc(&C, c_bytes) != hipSuccess) {
        (void)hipFree(A);
        return QLIN_ERR_NOMEM;
    }
    // varied input values rather than a constant, so the timed kernels see data like real
    // activations
    const int64_t na = (int64_t)rows * w->K;
    tune_fill_kernel<<<(unsigned)((na + 255) / 256), 256, 0, st>>>(A, na);
    int rc = hipGetLastError() == hipSuccess ? QLIN_OK : QLIN_ERR_DEVICE;
    const bool fused = gemv_fusable(ws, w, rows, A, w->K, nullptr, flags);
    const int path = fused ? 0 : (gemv_ok(ws, w, rows) ? 1 : 2);
    std::vector<int> cand;
    g_force_variant = -1;
    if (!fused && plan_rows(ws, w, rows, w->Kp, flags).kind != RowsPlan::kOther) cand.push_back(-1);
    g_force_variant = 0;
    const size_t own = cand.size();  // the planner's own choice comes first where it is not one of the variants
    if (path < 2) {
        for (int v : {4, 8, 16})
            if (!fused || gemv_can_fuse(rows, w->K, v, false)) cand.push_back(v);
    } else {
        // every kernel and tile configuration with 1..8 k splits (the planner trims a split
        // count that its partial buffer or counters cannot hold)
        const int ktiles = w->Kp / kGemmTileK;
        for (int kern = kTuneKernel16; kern <= kTuneKernel32 + 3; ++kern) {
            if (kern == kTuneKernel32 + 3 && w->bits != 4) continue;  // 256 x 192 tiles: W4 only
            for (int v : {1, 2, 3, 4, 6, 8})
                if (2 * v <= ktiles) cand.push_back(v + kTuneKernelStep * kern);
        }
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (!rc && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)) rc = QLIN_ERR_DEVICE;
    std::vector<uint16_t> ref(c_bytes / 2), got(c_bytes / 2);
    // two passes over the candidates, each timed after a warm-up run, the faster pass
    // counting: a candidate's time does not depend on where in the sequence it ran
    std::vector<float> ms_min(cand.size(), 0.0f);
    for (int pass = 0; pass < 2 && !rc; ++pass) {
        for (size_t i = 0; i < cand.size() && !rc; ++i) {
            g_force_variant = cand[i];
            rc = run_impl(ws, w, rows, A, QLIN_F16, w->K, nullptr, 0.0f, C, QLIN_F16, ncols, flags, st);  // warm-up
            if (!rc && hipEventRecord(e0, st) != hipSuccess) rc = QLIN_ERR_DEVICE;
            for (int r = 0; r < reps && !rc; ++r)
                rc = run_impl(ws, w, rows, A, QLIN_F16, w->K, nullptr, 0.0f, C, QLIN_F16, ncols, flags, st);
            float ms = 0.0f;
            if (!rc && (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                        hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
                rc = QLIN_ERR_DEVICE;
            // every variant computes the same integers and epilogue: the outputs must agree
            if (!rc && pass == 0) {
                if (hipMemcpy((i == 0 ? ref : got).data(), C, c_bytes, hipMemcpyDeviceToHost) != hipSuccess)
                    rc = QLIN_ERR_DEVICE;
                else if (i > 0 && std::memcmp(ref.data(), got.data(), c_bytes) != 0)
                    rc = QLIN_ERR_DEVICE;
            }
            if (!rc && (pass == 0 || ms < ms_min[i])) ms_min[i] = ms;
        }
    }
    size_t bi = own;
    for (size_t i = own + 1; i < cand.size(); ++i)
        if (ms_min[i] < ms_min[bi]) bi = i;
    const int best = rc || cand.size() <= own ? 0 : cand[bi] + (own && ms_min[0] <= ms_min[bi] ? kTunePlanner : 0);
    g_force_variant = 0;
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(A);
    (void)hipFree(C);
    if (!rc && best) {
        std::lock_guard<std::mutex> g(tune_mutex());
        tune_table()[TuneKey{w->bits, w->K, w->N, rows_bucket(rows), path, sw ? 1 : 0}] = best;
        g_tune_entries.store((int)tune_table().size(), std::memory_order_release);
    }
    return rc;
}

int qlin_tune_count(void) {
    std::lock_guard<std::mutex> g(tune_mutex());
    return (int)tune_table().size();
}

void qlin_tune_clear(void) {
    std::lock_guard<std::mutex> g(tune_mutex());
    tune_table().clear();
    g_tune_entries.store(0, std::memory_order_release);
}

int qlin_tune_save(const char* path) {
    if (!path) return QLIN_ERR_PARAM;
    std::FILE* f = std::fopen(path, "w");
    if (!f) return QLIN_ERR_PARAM;
    std::lock_guard<std::mutex> g(tune_mutex());
    std::fprintf(f, "# qlinear variant table: bits K N rows_bucket path swiglu variant [planner]\n");
    for (auto& kv : tune_table())
        std::fprintf(f, "%d %d %d %d %d %d %d%s\n", std::get<0>(kv.first), std::get<1>(kv.first), std::get<2>(kv.first),
                     std::get<3>(kv.first), std::get<4>(kv.first), std::get<5>(kv.first), kv.second % kTunePlanner,
                     kv.second >= kTunePlanner ? " planner" : "");
    return std::fclose(f) == 0 ? QLIN_OK : QLIN_ERR_PARAM;
}

int qlin_tune_load(const char* path) {
    if (!path) return QLIN_ERR_PARAM;
    std::FILE* f = std::fopen(path, "r");
    if (!f) return QLIN_ERR_PARAM;
    char line[256];
    int n = 0, rc = QLIN_OK;
    std::lock_guard<std::mutex> g(tune_mutex());
    while (std::fgets(line, sizeof line, f)) {
        if (line[0] == '#' || line[0] == '\n') continue;
        int b = 0, K = 0, N = 0, r = 0, path_ = -1, swg = -1, v = 0;
        char word[9] = "";
        const bool parsed = std::sscanf(line, "%d %d %d %d %d %d %d %8s", &b, &K, &N, &r, &path_, &swg, &v, word) >= 7;
        // a GEMM entry: 1..64 splits and a kernel field of 0..5 (5, the 256 x 192 tiles, W4 only)
        const bool ok_gemm = v % kTuneKernelStep >= 1 && v % kTuneKernelStep <= kTuneMaxSplits &&
                             v / kTuneKernelStep <= kTuneKernel32 + (b == 4 ? 3 : 2);
        if (!parsed || (b != 4 && b != 8) || K <= 0 || N <= 0 || r <= 0 || path_ < 0 || path_ > 2 ||
            (swg != 0 && swg != 1) || v <= 0 || (path_ < 2 && v != 4 && v != 8 && v != 16) ||
            (path_ == 2 && !ok_gemm)) {
            rc = QLIN_ERR_PARAM;
            break;
        }
        // a trailing "planner": the planner's own kernel was faster than this variant
        tune_table()[TuneKey{b, K, N, r, path_, swg}] = v + (std::strcmp(word, "planner") == 0 ? kTunePlanner : 0);
        ++n;
    }
    g_tune_entries.store((int)tune_table().size(), std::memory_order_release);
    std::fclose(f);
    return rc ? rc : n;
}
