// Wave-split-K GEMM for a few to a few hundred quantized rows: int8 MFMA
// (v_mfma_i32_16x16x64_i8) with the dequant / SiLU-gate / residual epilogue.  Replaces the
// same native-library stage as gemm_kernel (QWEN3_W4A8_PIPELINE_REVIEW_20261020.md:28-31).
//
// Why.  At 5..256 rows a linear is a handful of 128 x 128 tiles: to fill the CUs the tiled
// GEMM has to split K over workgroups, whose partial sums then travel through memory (3-5
// us), and the 16-channel GEMV re-reads every activation for each group of 16 channels.
// Here a workgroup owns a small tile (16..96 rows x 16..96 channels, sized so that one round
// of workgroups covers the output) over the whole K, and its 4 or 8 waves split K among
// them: wave w multiplies the 128-deep k steps w, w + WK, ... of the whole tile, and the
// partial sums meet once, in LDS, at the end.
//
// A wave streams its own steps global -> LDS (buffer_load ... lds, 1 KiB per instruction)
// into a ring of R stages that no other wave touches, so the k loop has no barrier: a wave
// waits for its own copies (vmcnt), reads the fragments of the next step into registers,
// refills the stage and multiplies.  Loads straight into registers in fragment order (16
// rows x 16 bytes per quarter wave) ran at 38 GB/s per CU, one 16-byte lane per clock, where
// these copies (whole 64- or 128-byte row pieces) reach 116-150.  The stages hold the rows
// as gemm_kernel's do (same XOR swizzles, conflict-free fragment reads), and k is assigned
// to lanes the same way: 32 lc + 16 h for lane group lc and MFMA h.
//
// What bounds it: the launch and the first copies' round trip (~3.5 us in all), then the
// copies, (tile rows + channels * bits / 8) * K bytes at 64 bytes per clock and CU, and the
// weight stream (~4 TB/s); deeper rings, an L2 prefetch wave and contiguous k ranges per
// wave measured the same.  Per launch in a graph, quantized rows, eight copies of the weights in
// turn, W4 (us, before -> chosen; before is the GEMV up to 20 rows and for o / down up to 32, else
// the 128 x 128 GEMM; * another kernel than this one):
//     rows qkv 2560x6144      o 4096x2560        gate_up 2560x19456 down 9728x2560
//     16   8.0 ->  5.0        5.7 ->  5.0        11.2 ->  8.6       9.0 ->  6.5
//     24   12.0 ->  5.5       7.4 ->  5.3        12.9 ->  9.1       12.2 ->  7.4
//     64   12.7 ->  6.6       12.1 ->  6.2       13.8 -> 11.4       16.3 ->  9.1
//     128  13.7 ->  8.7       13.0 ->  7.3       14.8 -> 14.1*      17.4 -> 11.3
//     300  15.1 -> 13.4*      14.7 -> 10.6       30.2 -> 21.5*      19.7 -> 17.2
//     512  16.1 -> 14.6*      15.3 -> 12.4       31.6 -> 28.8*      22.3 -> 22.3*
#include <hip/hip_fp16.h>

#include "qlin_epilogue.hpp"

namespace qlin {

namespace ks {

constexpr int kBufferFlags = 0x00020000;  // raw buffer, 32-bit data format (gfx9 word 3)
constexpr int BK = 128;

typedef __attribute__((address_space(3))) void* lds_ptr;

template <int BITS, int MF, int NB, int WK, int R>
struct Geom {
    static constexpr int THREADS = 64 * WK;
    static constexpr int TM = 16 * MF, TN = 16 * NB;
    static constexpr int NBL = BITS == 4 ? 1 : 2;  // KiB of a channel block per k step
    static constexpr int NL = 2 * MF + NB * NBL;   // 1 KiB copies of a wave per k step
    static constexpr int STAGE = NL * 1024, RING = R * STAGE;
    // row fragments of a wave whose partial sums meet in LDS at once (1 KiB per fragment and wave)
    static constexpr int MFP = WK * MF * NB <= 128 ? MF : WK * (MF / 2) * NB <= 128 ? MF / 2 : MF / 4;
    static constexpr int PART = WK * MFP * NB * 1024;
    static constexpr int SCL = PART > WK * RING ? PART : WK * RING;  // scales after the ring and the partials
    static constexpr int LDS = SCL + (TM + TN) * 4;
    static_assert(MFP >= 1 && MF % MFP == 0, "phases");
    static_assert(TM + TN <= THREADS, "one scale per thread");
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, kBufferFlags);
}

// One 1 KiB copy, global memory -> LDS in lane order.
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint8_t* lds_block, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)lds_block, 16, voff, soff, 0, 0);
}

// s_waitcnt immediates (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Swizzles of the 16-byte chunks of 128-byte rows (activations, W8) and 64-byte rows (W4)
// that keep the fragment reads free of bank conflicts, as in gemm_kernel.
__device__ __forceinline__ int swz128(int r) { return ((r >> 1) & 1) | (((r >> 2) & 1) << 2); }
__device__ __forceinline__ int swz64(int r) { return (r >> 1) & 3; }

__device__ __forceinline__ v4i unpack2(int x, int y) {
    const unsigned ux = (unsigned)x, uy = (unsigned)y;
    return v4i{(int)((ux << 4) & 0xF0F0F0F0u), (int)(ux & 0xF0F0F0F0u), (int)((uy << 4) & 0xF0F0F0F0u),
               (int)(uy & 0xF0F0F0F0u)};
}

template <int BITS, bool SWIGLU, int MF, int NB, int WK, int R>
__global__ __launch_bounds__(64 * WK) void gemm_ks_kernel(GemmParams p) {
    using G = Geom<BITS, MF, NB, WK, R>;
    constexpr int NBL = G::NBL;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lc = lane >> 4;

    const int b = xcd_tile(blockIdx.x, p.m_tiles * p.n_tiles, p.m_tiles);
    const int nt = b / p.m_tiles, mt = b - nt * p.m_tiles;
    const int m0 = mt * G::TM;
    constexpr int TC = SWIGLU ? G::TN / 2 : G::TN;  // output channels of the tile
    const int n0 = nt * TC;
    const int nh = p.N >> 1;
    const int ncols = SWIGLU ? nh : p.N;

    // epilogue scales: one per thread, used after the k loop
    float pre = 0.0f;
    if (p.s) {
        if (tid < G::TM) {
            pre = p.s[min(m0 + tid, p.M - 1)];
        } else if (tid < G::TM + G::TN) {
            const int r = tid - G::TM;
            pre = p.wscale[SWIGLU && r >= TC ? nh + min(n0 + r - TC, ncols - 1) : min(n0 + r, ncols - 1)];
        }
    }

    const uint8_t* abase = reinterpret_cast<const uint8_t*>(p.q) + (int64_t)m0 * p.ldq;
    const int abytes = (min(p.M - m0, G::TM) - 1) * (int)p.ldq + p.Kp;
    const uint8_t* gbase = p.W + (int64_t)n0 * p.wrow;
    const int bbytes = min(ncols - n0, TC) * (int)p.wrow;
    const uint8_t* ubase = SWIGLU ? p.W + (int64_t)(nh + n0) * p.wrow : gbase;
    // copy offsets: activations (and W8) 8 rows of 128 bytes per KiB, W4 16 rows of 64
    int aoff[2 * MF], boff[NB * NBL];
#pragma unroll
    for (int i = 0; i < 2 * MF; ++i) {
        const int row = 8 * i + (lane >> 3);
        aoff[i] = row * (int)p.ldq + (((lane & 7) ^ swz128(row)) << 4);
    }
#pragma unroll
    for (int j = 0; j < NB * NBL; ++j) {
        const int jj = SWIGLU ? j % (NB * NBL / 2) : j;
        if constexpr (BITS == 4) {
            const int row = 16 * jj + (lane >> 2);
            boff[j] = row * (int)p.wrow + (((lane & 3) ^ swz64(row)) << 4);
        } else {
            const int row = 8 * jj + (lane >> 3);
            boff[j] = row * (int)p.wrow + (((lane & 7) ^ swz128(row)) << 4);
        }
    }

    v4i acc[MF][NB];
#pragma unroll
    for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = v4i{0, 0, 0, 0};

    const int steps = p.Kp / BK;
    const int n = (steps - wave + WK - 1) / WK;  // this wave's k steps: wave, wave + WK, ...
    uint8_t* ring = smem + wave * G::RING;
    // a step past the end copies through an empty descriptor: zeros, no memory access
    auto issue = [&](int s, int t) {
        const int k0 = (wave + t * WK) * BK;
        const bool in = t < n;
        const auto rg = rsrc(gbase, in ? bbytes : 0), ru = rsrc(ubase, in ? bbytes : 0);
        const auto ra = rsrc(abase, in ? abytes : 0);
        uint8_t* st = ring + s * G::STAGE;
#pragma unroll
        for (int j = 0; j < NB * NBL; ++j)
            dma16(SWIGLU && j >= NB * NBL / 2 ? ru : rg, st + 2 * MF * 1024 + j * 1024, boff[j], BITS == 4 ? k0 / 2 : k0);
#pragma unroll
        for (int i = 0; i < 2 * MF; ++i) dma16(ra, st + i * 1024, aoff[i], k0);
    };
    const int ard0 = lr * 128 + (((2 * lc) ^ swz128(lr)) << 4), ard1 = lr * 128 + (((2 * lc + 1) ^ swz128(lr)) << 4);
    const int brd = lr * 64 + ((lc ^ swz64(lr)) << 4);
    auto read = [&](v4i (&as)[MF][2], v4i (&ws)[NB][NBL], int s) {
        const uint8_t* st = ring + s * G::STAGE;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if constexpr (BITS == 4) {
                ws[j][0] = *reinterpret_cast<const v4i*>(st + 2 * MF * 1024 + j * 1024 + brd);
            } else {
                ws[j][0] = *reinterpret_cast<const v4i*>(st + 2 * MF * 1024 + j * 2048 + ard0);
                ws[j][1] = *reinterpret_cast<const v4i*>(st + 2 * MF * 1024 + j * 2048 + ard1);
            }
        }
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            as[i][0] = *reinterpret_cast<const v4i*>(st + i * 2048 + ard0);
            as[i][1] = *reinterpret_cast<const v4i*>(st + i * 2048 + ard1);
        }
    };
    auto mma = [&](const v4i (&as)[MF][2], const v4i (&ws)[NB][NBL]) {
#pragma unroll
        for (int j = 0; j < NB; ++j) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v4i x;
                if constexpr (BITS == 4) x = h == 0 ? unpack2(ws[j][0][0], ws[j][0][1]) : unpack2(ws[j][0][2], ws[j][0][3]);
                else x = ws[j][h];
#pragma unroll
                for (int i = 0; i < MF; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, as[i][h], acc[i][j], 0, 0, 0);
            }
        }
    };
    v4i a0[MF][2], a1[MF][2], w0[NB][NBL], w1[NB][NBL];
#pragma unroll
    for (int s = 0; s < R; ++s) issue(s, s);
    wait_vm<(R - 1) * G::NL>();
    asm volatile("" ::: "memory");
    read(a0, w0, 0);
    int cur = 0;  // ring slot of the step held in registers
    // one step: its slot is refilled once its reads have returned, the next step's fragments
    // are read, then it is multiplied
    auto step = [&](v4i (&ac)[MF][2], v4i (&wc)[NB][NBL], v4i (&an)[MF][2], v4i (&wn)[NB][NBL], int t) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(cur, t + R);
        cur = cur + 1 == R ? 0 : cur + 1;
        wait_vm<(R - 1) * G::NL>();
        asm volatile("" ::: "memory");
        read(an, wn, cur);
        __builtin_amdgcn_sched_barrier(0);
        mma(ac, wc);
    };
    for (int t = 0; t < n; t += 2) {
        step(a0, w0, a1, w1, t);
        if (t + 1 < n) step(a1, w1, a0, w0, t + 1);
    }
    wait_vm<0>();
    __syncthreads();

    // ---- the waves' partial sums meet in LDS; each wave finishes a share of the fragments ----
    constexpr int NBO = SWIGLU ? NB / 2 : NB, TASKS = G::MFP * NBO;
    float* scl = reinterpret_cast<float*>(smem + G::SCL);
    if (tid < G::TM + G::TN) scl[tid] = pre;
    const bool vec = c_rows_vec(p), rvec = r_rows_vec(p);
#pragma unroll
    for (int ph = 0; ph < MF / G::MFP; ++ph) {
        if (ph) lds_barrier();  // the previous fragments are read out
#pragma unroll
        for (int i = 0; i < G::MFP; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                *reinterpret_cast<v4i*>(smem + (((wave * G::MFP + i) * NB + j) << 10) + lane * 16) =
                    acc[ph * G::MFP + i][j];
        lds_barrier();
#pragma unroll
        for (int it = 0; it < (TASKS + WK - 1) / WK; ++it) {
            const int task = wave + it * WK;
            if (TASKS % WK != 0 && task >= TASKS) break;
            const int rf = task / NBO, j = task - rf * NBO;
            const int m_in = (ph * G::MFP + rf) * 16 + lr;
            const int c_in = 16 * j + 4 * lc;
            const int m = m0 + m_in, c = n0 + c_in;
            const bool live = m < p.M && c < ncols;
            float res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (!SWIGLU && p.R && live) residual4(p, m, c, ncols, rvec, res);
            v4i gate = {0, 0, 0, 0}, up = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < WK; ++k) {
                const uint8_t* at = smem + (((k * G::MFP + rf) * NB + j) << 10) + lane * 16;
                gate += *reinterpret_cast<const v4i*>(at);
                if constexpr (SWIGLU) up += *reinterpret_cast<const v4i*>(at + (NBO << 10));
            }
            if (live)
                finish4<BITS, SWIGLU>(p, p.c_kind, m, c, ncols, vec, gate, up, scl[m_in], scl + G::TM + c_in,
                                      scl + G::TM + TC + c_in, res);
        }
    }
}

template <int BITS, bool SWIGLU, int MF, int NB, int WK, int R>
static hipError_t launch_t(const GemmParams& p, hipStream_t stream) {
    using G = Geom<BITS, MF, NB, WK, R>;
    if constexpr (G::LDS > 160 * 1024) {  // W8 stages are larger: one stage less
        if constexpr (R > 2) return launch_t<BITS, SWIGLU, MF, NB, WK, R - 1>(p, stream);
        else return hipErrorInvalidValue;  // gemm_ks_fits
    } else {
        static const hipError_t attr = hipFuncSetAttribute(
            reinterpret_cast<const void*>(&gemm_ks_kernel<BITS, SWIGLU, MF, NB, WK, R>),
            hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
        if (attr != hipSuccess) return attr;
        gemm_ks_kernel<BITS, SWIGLU, MF, NB, WK, R><<<dim3(p.m_tiles * p.n_tiles), dim3(G::THREADS), G::LDS, stream>>>(p);
        return hipGetLastError();
    }
}

template <int MF, int NB, int WK, int R>
static hipError_t launch_c(const GemmParams& p, int bits, hipStream_t st) {
    const bool sw = (p.flags & kFlagSwiglu) != 0 && p.c_kind != 2;
    if constexpr (NB % 2 == 0) {
        if (sw) return bits == 4 ? launch_t<4, true, MF, NB, WK, R>(p, st) : launch_t<8, true, MF, NB, WK, R>(p, st);
    }
    if (sw) return hipErrorInvalidValue;
    return bits == 4 ? launch_t<4, false, MF, NB, WK, R>(p, st) : launch_t<8, false, MF, NB, WK, R>(p, st);
}

}  // namespace ks

// Tile configurations: row fragments MF and channel blocks NB of 16, waves WK along k, stages R of a
// wave's ring (as many as fit 160 KiB, at most what the shortest K uses), time against the planner's
// estimate (W4, W8).
#define QLIN_KS_CONFIGS(X)                                                                                              \
    X(0, 1, 1, 4, 6, 1.02, 1.01) X(1, 1, 1, 8, 4, 1, 1.03) X(2, 1, 2, 4, 4, 0.97, 0.99) X(3, 1, 3, 4, 4, 0.98, 1.01)    \
    X(4, 1, 6, 4, 4, 1.03, 0.98) X(5, 2, 1, 4, 4, 1.03, 0.99) X(6, 2, 2, 4, 4, 1.01, 1.01) X(7, 2, 3, 4, 3, 0.99, 0.98) \
    X(8, 2, 3, 8, 2, 0.93, 1) X(9, 2, 4, 4, 3, 0.98, 0.99) X(10, 2, 6, 4, 4, 0.99, 0.97) X(11, 3, 2, 4, 3, 1, 0.99)     \
    X(12, 3, 2, 8, 2, 0.94, 1) X(13, 3, 3, 4, 3, 1.01, 0.99) X(14, 4, 3, 4, 3, 1.02, 0.96) X(15, 4, 4, 4, 3, 1, 0.96)   \
    X(16, 4, 5, 4, 2, 0.97, 0.98) X(17, 4, 6, 4, 2, 0.96, 1) X(18, 6, 3, 4, 2, 1.02, 1.01) X(19, 6, 4, 4, 2, 0.99, 1)

KsTile gemm_ks_tile(int cfg) {
    switch (cfg) {
#define X(c, mf, nb, wk, r, rel4, rel8) \
    case c: return {mf, nb, wk, {rel4, rel8}};
        QLIN_KS_CONFIGS(X)
#undef X
        default: return {0, 0, 0, {0.0, 0.0}};
    }
}

bool gemm_ks_fits(int bits, int cfg) {
    const KsTile t = gemm_ks_tile(cfg);
    const int ring = t.wk * 2 * (2 * t.mf + t.nb * (bits == 4 ? 1 : 2)) * 1024;
    return t.mf && ring + (t.mf + t.nb) * 64 <= 160 * 1024;
}

hipError_t launch_gemm_ks(const GemmParams& p, int bits, int cfg, hipStream_t st) {
    switch (cfg) {
#define X(c, mf, nb, wk, r, rel4, rel8) \
    case c: return ks::launch_c<mf, nb, wk, r>(p, bits, st);
        QLIN_KS_CONFIGS(X)
#undef X
        default: return hipErrorInvalidValue;
    }
}

}  // namespace qlin
