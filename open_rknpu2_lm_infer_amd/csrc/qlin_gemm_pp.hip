// Prefill GEMM for grids that cover the CUs: int8 MFMA (v_mfma_i32_16x16x64_i8) with the
// dequant / SiLU-gate / residual epilogue.  Replaces the same native-library stage as
// gemm_kernel (QWEN3_W4A8_PIPELINE_REVIEW_20261020.md:28-31).
//
// Why.  gemm_kernel and gemm32_kernel run every wave through the same step at once: reads,
// copies and MFMAs of the eight waves meet at one barrier per step, the two waves of a SIMD
// want the matrix core at the same time and then leave it idle together (M = 4096 gate_up: 47%
// of its cycles busy).  Here the eight waves are two groups of four, one wave of each group per
// SIMD, half a step apart: while one group multiplies a 128-deep k step of its part of the
// tile, the other reads its fragments of the next from LDS and issues its share of the copies;
// a barrier swaps the roles.  The multiplying wave has its operands in registers and issues
// only MFMAs and the W4 unpack (spread over the MFMAs), at raised priority.
//
// NST stages of 128 k in LDS (three of 44-48 KiB for the large tiles, four below), filled by
// buffer_load ... lds copies of whole row pieces with the XOR swizzles of gemm_kernel.  The
// copies of step t + NST - 1 are issued in the memory phase of step t, into the stage both
// groups finished reading a phase ago, and are waited for a whole step later, before the
// barrier after which anyone reads them.  Issued between the MFMAs instead they stalled the
// multiplying wave (256 x 192 tile 0.84 -> 1.13 us per step).
//
// A workgroup takes tiles until its XCD's range is done: the next tile's first stages are
// copied under the epilogue.  fp16 rows leave through a padded buffer in the stage the next
// tile fills last, so a store covers 64-192 contiguous bytes of a row instead of 32 bytes of 16
// rows (M = 4096 qkv 64.5 -> 58.1 us).
//
// What bounds it: with the copies and LDS reads left out a 256 x 192 step takes 0.74 us (1536
// matrix-core cycles per SIMD), with them 0.84, the LDS reads' register writes most of the
// difference; per tile the epilogue (~3 us of VALU, more with SiLU-gate) and the first copies.
// M = 4096, quantized rows, W4 (us, before -> now): qkv 72.5 -> 58.1, o 49.2 -> 40.5, gate_up
// 195 -> 164 (2.1 -> 2.5 POPS), down 115 -> 82 (2.5 POPS); M = 512
// gate_up 33 -> 29, qkv 14.8 -> 12.8; W8 M = 4096 qkv 113 -> 72, gate_up 300 -> 218.
#include <algorithm>

#include <hip/hip_fp16.h>

#include "qlin_epilogue.hpp"

namespace qlin {

namespace pp {

constexpr int BK = 128;
constexpr int kBufferFlags = 0x00020000;  // raw buffer, 32-bit data format (gfx9 word 3)
constexpr int kPastEnd = 0x7fff0000;      // a buffer offset past every operand (reads return zeros)
typedef __attribute__((address_space(3))) void* lds_ptr;

template <int BITS, bool SWIGLU, int BM, int BN, int WM, int WN, int NST>
struct Geom {
    static constexpr int NW = WM * WN, THREADS = 64 * NW;
    static constexpr int TM = BM / WM, TN = BN / WN, MF = TM / 16, NB = TN / 16;
    static constexpr int B_ROW = BITS == 4 ? BK / 2 : BK;
    static constexpr int A_BYTES = BM * BK, B_BYTES = BN * B_ROW, STAGE = A_BYTES + B_BYTES;
    static constexpr int A_BLOCKS = A_BYTES / 1024, B_BLOCKS = B_BYTES / 1024;
    static constexpr int NA = A_BLOCKS / NW, NBC = (B_BLOCKS + NW - 1) / NW, NL = NA + NBC;
    static constexpr bool SPARE = NBC * NW > B_BLOCKS;
    static constexpr int SCRATCH = NST * STAGE;
    static constexpr int SCL = NST * STAGE + (SPARE ? 1024 : 0);  // epilogue scales
    static constexpr int LDS = SCL + (BM + BN) * 4;
    static constexpr int TNO = SWIGLU ? TN / 2 : TN;    // output channels of a wave
    static constexpr int PITCH = TNO * 2 + 16;          // bytes of a staged fp16 row
    static constexpr bool WIDE = 8 * 16 * PITCH <= STAGE;
    static_assert(NW == 8 && TM % 16 == 0 && TN % 16 == 0 && A_BLOCKS % NW == 0, "waves");
    static_assert(LDS <= 160 * 1024 && NST >= 3, "LDS stages");
    static_assert(BM + BN <= THREADS, "one scale per thread");
};

__device__ __forceinline__ int swz128(int r) { return ((r >> 1) & 1) | (((r >> 2) & 1) << 2); }
__device__ __forceinline__ int swz64(int r) { return (r >> 1) & 3; }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kBufferFlags);
}
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, uint8_t* lds_block, int voff, int soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)lds_block, 16, voff, soff, 0, 0);
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
__device__ __forceinline__ void phase_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ v4i unpack2(int x, int y) {
    const unsigned ux = (unsigned)x, uy = (unsigned)y;
    return v4i{(int)((ux << 4) & 0xF0F0F0F0u), (int)(ux & 0xF0F0F0F0u), (int)((uy << 4) & 0xF0F0F0F0u),
               (int)(uy & 0xF0F0F0F0u)};
}

// Instruction order of a compute phase: the next block's unpack spread over this block's MFMAs.
template <int N, int MF, int VALU>
__device__ __forceinline__ void order_mma() {
    if constexpr (N > 0) {
        __builtin_amdgcn_sched_group_barrier(0x008, MF / 2, 0);
        if constexpr (VALU > 0) __builtin_amdgcn_sched_group_barrier(0x002, VALU / 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, MF - MF / 2, 0);
        if constexpr (VALU > 0) __builtin_amdgcn_sched_group_barrier(0x002, VALU - VALU / 2, 0);
        order_mma<N - 1, MF, VALU>();
    }
}

template <int BITS, bool SWIGLU, int OUT, int BM, int BN, int WM, int WN, int NST>
__global__ __launch_bounds__(64 * WM * WN) void gemm_pp_kernel(GemmParams p) {
    using G = Geom<BITS, SWIGLU, BM, BN, WM, WN, NST>;
    constexpr int MF = G::MF, NB = G::NB, NL = G::NL;
    extern __shared__ __align__(16) uint8_t smem[];
    float* scl = reinterpret_cast<float*>(smem + G::SCL);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int lr = lane & 15, lc = lane >> 4;
    constexpr int TC = SWIGLU ? BN / 2 : BN;  // output channels of a tile
    const int nh = p.N >> 1, ncols = SWIGLU ? nh : p.N;

    // tiles of this workgroup: one, or every `stride`-th of a contiguous range per XCD
    const int NT = p.m_tiles * p.n_tiles, NG = gridDim.x;
    int tile = blockIdx.x, stride = NG, tile_end = NT;
    if (NT == NG) {
        tile = xcd_tile(tile, NT, p.m_tiles);
    } else if ((NG & 7) == 0) {
        const int per = (NT + 7) >> 3, x = tile & 7;
        stride = NG >> 3;
        tile_end = min(NT, (x + 1) * per);
        tile = x * per + (tile >> 3);
    }
    if (tile >= tile_end) return;

    // copy plan: blocks of 1 KiB dealt to the waves in turn, activations first
    int off[NL];
#pragma unroll
    for (int i = 0; i < G::NA; ++i) {
        const int row = (wave + 8 * i) * 8 + (lane >> 3);
        off[i] = row * (int)p.ldq + (((lane & 7) ^ swz128(row)) << 4);
    }
#pragma unroll
    for (int i = 0; i < G::NBC; ++i) {
        const int blk = wave + 8 * i;
        int row, chunk;
        if constexpr (BITS == 4) {
            row = blk * 16 + (lane >> 2);
            chunk = (lane & 3) ^ swz64(row);
        } else {
            row = blk * 8 + (lane >> 3);
            chunk = (lane & 7) ^ swz128(row);
        }
        if (SWIGLU && row >= TC) row -= TC;
        off[G::NA + i] = blk < G::B_BLOCKS ? row * (int)p.wrow + (chunk << 4) : kPastEnd;
    }
    int m0, n0;
    __amdgpu_buffer_rsrc_t ra, rg, ru;
    float pre = 0.0f;
    // tile t: its corner, buffer descriptors and this thread's epilogue scale
    auto open = [&](int t) {
        const int per_group = p.group_m * p.n_tiles;
        const int g = t / per_group, first_m = g * p.group_m;
        const int gm = min(p.m_tiles - first_m, p.group_m);
        const int r = t - g * per_group;
        const int nt = r / gm;
        m0 = (first_m + (r - nt * gm)) * BM;
        n0 = nt * TC;
        ra = rsrc(p.q + (int64_t)m0 * p.ldq, (int64_t)(min(p.M - m0, BM) - 1) * p.ldq + p.Kp);
        const int64_t wb = (int64_t)min(ncols - n0, TC) * p.wrow;
        rg = rsrc(p.W + (int64_t)n0 * p.wrow, wb);
        ru = SWIGLU ? rsrc(p.W + (int64_t)(nh + n0) * p.wrow, wb) : rg;
        if constexpr (OUT != 2) {
            if (tid < BM) {
                pre = p.s[min(m0 + tid, p.M - 1)];
            } else if (tid < BM + BN) {
                const int c = tid - BM;
                pre = p.wscale[SWIGLU && c >= TC ? nh + min(n0 + c - TC, ncols - 1) : min(n0 + c, ncols - 1)];
            }
        }
    };
    auto copy = [&](int i, int stage, int k0) {  // i: compile-time slot
        if (i < G::NA) {
            dma16(ra, smem + stage + (wave + 8 * i) * 1024, off[i], k0);
        } else {
            const int blk = wave + 8 * (i - G::NA);
            constexpr int ROWS = BITS == 4 ? 16 : 8;
            uint8_t* dst = G::SPARE && blk >= G::B_BLOCKS ? smem + G::SCRATCH : smem + stage + G::A_BYTES + blk * 1024;
            dma16(SWIGLU && blk * ROWS >= TC ? ru : rg, dst, off[i], BITS == 4 ? k0 / 2 : k0);
        }
    };
    const int T = p.Kp / BK, last = T - 1;
    auto fill_first = [&]() {  // the first NST - 1 stages
#pragma unroll
        for (int t = 0; t < NST - 1; ++t)
#pragma unroll
            for (int i = 0; i < NL; ++i) copy(i, t * G::STAGE, min(t, last) * BK);
    };

    const int ard[2] = {(wm * G::TM + lr) * 128 + (((2 * lc) ^ swz128(lr)) << 4),
                        (wm * G::TM + lr) * 128 + (((2 * lc + 1) ^ swz128(lr)) << 4)};
    // first weight row of the wave's block j
    auto brow = [&](int j) { return SWIGLU ? (j >= NB / 2 ? TC : 0) + wn * (G::TN / 2) + (j % (NB / 2)) * 16 : wn * G::TN + j * 16; };
    const int brd[2] = {BITS == 4 ? lr * 64 + ((lc ^ swz64(lr)) << 4) : lr * 128 + (((2 * lc) ^ swz128(lr)) << 4),
                        lr * 128 + (((2 * lc + 1) ^ swz128(lr)) << 4)};
    v4i acc[MF][NB];
    const bool vec = c_rows_vec(p), rvec = r_rows_vec(p);
    constexpr int NBO = SWIGLU ? NB / 2 : NB;
    const int cw = wn * (SWIGLU ? G::TN / 2 : G::TN) + 4 * lc;  // first channel of the lane in the tile
    const bool has_r = !SWIGLU && OUT != 2 && p.R;

    open(tile);
    fill_first();
    for (;;) {
        if constexpr (OUT != 2) {
            if (tid < BM + BN) scl[tid] = pre;
        }
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[i][j] = v4i{0, 0, 0, 0};
        wait_vm<(NST - 2) * NL>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        phase_barrier();
        if (wave >= 4) phase_barrier();
        int cur = 0, fill = (NST - 1) * G::STAGE;  // stage being read, stage being filled
        for (int t = 0; t < T; ++t) {
            // memory phase
            const uint8_t* st = smem + cur;
            const int k0 = min(t + NST - 1, last) * BK;
            v4i a[MF][2], w[NB][BITS == 4 ? 1 : 2];
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int h = 0; h < (BITS == 4 ? 1 : 2); ++h)
                    w[j][h] = *reinterpret_cast<const v4i*>(st + G::A_BYTES + brow(j) * G::B_ROW + brd[h]);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < MF; ++i) a[i][h] = *reinterpret_cast<const v4i*>(st + ard[h] + i * 2048);
#pragma unroll
            for (int i = 0; i < NL; ++i) copy(i, fill, k0);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            wait_vm<(NST - 2) * NL>();
            phase_barrier();
            // compute phase
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    v4i x;
                    if constexpr (BITS == 4) x = unpack2(w[j][0][2 * h], w[j][0][2 * h + 1]);
                    else x = w[j][h];
#pragma unroll
                    for (int i = 0; i < MF; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, a[i][h], acc[i][j], 0, 0, 0);
                }
            if constexpr (BITS == 4) __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            order_mma<2 * NB, MF, BITS == 4 ? 6 : 0>();
            __builtin_amdgcn_s_setprio(0);
            phase_barrier();
            cur = cur + G::STAGE == NST * G::STAGE ? 0 : cur + G::STAGE;
            fill = fill + G::STAGE == NST * G::STAGE ? 0 : fill + G::STAGE;
        }
        if (wave < 4) phase_barrier();
        wait_vm<0>();  // the surplus copies, before the stages are filled again
        __syncthreads();

        const int em0 = m0, en0 = n0;
        tile += stride;
        if (tile < tile_end) {
            open(tile);
            fill_first();
        }
        constexpr bool PRE = MF * NB <= 24;  // registers for two rows of residuals
        float res[PRE ? 2 : 1][NBO][4];
        const bool wide = OUT == 1 && G::WIDE && (p.ldc & 7) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && en0 + TC <= ncols;
        uint8_t* rowbuf = smem + (NST - 1) * G::STAGE + wave * 16 * G::PITCH;
        auto load_r = [&](int i, float (&r)[NBO][4]) {
            const int m = em0 + wm * G::TM + 16 * i + lr;
#pragma unroll
            for (int j = 0; j < NBO; ++j)
                if (m < p.M && en0 + cw + 16 * j < ncols) residual4(p, m, en0 + cw + 16 * j, ncols, rvec, r[j]);
        };
        if (PRE && has_r) load_r(0, res[0]);
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            if (!PRE && has_r) load_r(i, res[0]);
            if (PRE && has_r && i + 1 < MF) load_r(i + 1, res[(i + 1) & (PRE ? 1 : 0)]);  // ahead of this row's stores
            const int m_in = wm * G::TM + 16 * i + lr, m = em0 + m_in;
            if (wide) {
                // fp16 rows through the wave's part of the stage the next tile fills last, so that a
                // store covers whole row pieces instead of 32 bytes of 16 rows
                constexpr int RC = G::TNO / 8;  // 16-byte chunks of a row
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < NBO; ++j) {
                    const int c_in = cw + 16 * j;
                    float o[4];
                    values4<BITS, SWIGLU>(p, acc[i][j], acc[i][SWIGLU ? j + NBO : j], scl[m_in], scl + BM + c_in,
                                          scl + BM + TC + c_in, res[PRE ? i & 1 : 0][j], o);
                    h4 v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = f16_of_f32(o[e]);
                    *reinterpret_cast<h4*>(rowbuf + lr * G::PITCH + (16 * j + 4 * lc) * 2) = v;
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int k = 0; k < (16 * RC + 63) / 64; ++k) {
                    const int idx = k * 64 + lane, row = idx / RC, ch = idx - row * RC;
                    const int mr = em0 + wm * G::TM + 16 * i + row;
                    if ((16 * RC % 64 == 0 || idx < 16 * RC) && mr < p.M) {
                        const uint4 v = *reinterpret_cast<const uint4*>(rowbuf + row * G::PITCH + ch * 16);
                        *reinterpret_cast<uint4*>(reinterpret_cast<_Float16*>(p.C) + (int64_t)mr * p.ldc + en0 + wn * G::TNO +
                                                  ch * 8) = v;
                    }
                }
            } else if (m < p.M) {
#pragma unroll
                for (int j = 0; j < NBO; ++j) {
                    const int c_in = cw + 16 * j, c = en0 + c_in;
                    if (c < ncols)
                        finish4<BITS, SWIGLU>(p, OUT, m, c, ncols, vec, acc[i][j], acc[i][SWIGLU ? j + NBO : j], scl[m_in],
                                              scl + BM + c_in, scl + BM + TC + c_in, res[PRE ? i & 1 : 0][j]);
                }
            }
        }
        if (tile >= tile_end) break;
        wait_vm<0>();  // the stores, so that the copy waits count copies alone
        lds_barrier();  // the scales are read out
    }
}

template <int BITS, bool SWIGLU, int OUT, int BM, int BN, int WM, int WN, int NST>
static hipError_t launch_s(const GemmParams& p, int cus, hipStream_t stream) {
    using G = Geom<BITS, SWIGLU, BM, BN, WM, WN, NST>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&gemm_pp_kernel<BITS, SWIGLU, OUT, BM, BN, WM, WN, NST>),
        hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS);
    if (attr != hipSuccess) return attr;
    gemm_pp_kernel<BITS, SWIGLU, OUT, BM, BN, WM, WN, NST><<<dim3(std::min(p.m_tiles * p.n_tiles, cus)), dim3(G::THREADS), G::LDS, stream>>>(p);
    return hipGetLastError();
}

// NST: as many stages of 128 k as fit the LDS, at most four.
template <int BITS, int BM, int BN, int WM, int WN>
static hipError_t launch_c(const GemmParams& p, int cus, hipStream_t st) {
    constexpr int STAGE = BM * BK + BN * (BITS == 4 ? BK / 2 : BK);
    constexpr int NST = 4 * STAGE + 3072 <= 160 * 1024 ? 4 : 3;
    if (p.c_kind == 2) return launch_s<BITS, false, 2, BM, BN, WM, WN, NST>(p, cus, st);
    if (p.flags & kFlagSwiglu) {
        if constexpr (BN / WN / 16 % 2 == 0)
            return p.c_kind == 1 ? launch_s<BITS, true, 1, BM, BN, WM, WN, NST>(p, cus, st)
                                 : launch_s<BITS, true, 0, BM, BN, WM, WN, NST>(p, cus, st);
        else return hipErrorInvalidValue;
    }
    return p.c_kind == 1 ? launch_s<BITS, false, 1, BM, BN, WM, WN, NST>(p, cus, st)
                         : launch_s<BITS, false, 0, BM, BN, WM, WN, NST>(p, cus, st);
}

}  // namespace pp

// Tile configurations: tokens x weight rows, what each is built for, and the us per 128-deep k
// step and per tile (W4, W8) of the planner's estimate, from its fit.  Configuration 0 needs all
// 256 registers, and without SiLU-gate it would spill; 6 is 5 with the waves laid out for SiLU-gate
// (each wave then needs an even number of 16-row blocks).
constexpr PpTile kPpTiles[kPpConfigs] = {
    // bm, bn, W4, W8, plain, SiLU-gate, us per k step W4, W8, us per tile W4, W8
    {256, 256, true, false, false, true, {1.03, 0}, {5.63, 0}},
    {256, 192, true, false, true, true, {0.856, 0}, {4.54, 0}},
    {256, 128, true, true, true, true, {0.553, 0.574}, {3.24, 3.11}},
    {128, 96, true, true, true, false, {0.32, 0.348}, {1.95, 1.97}},
    {128, 128, true, true, true, true, {0.349, 0.383}, {1.84, 1.75}},
    {128, 192, true, true, true, false, {0.447, 0.527}, {3.2, 2.62}},
    {128, 192, true, true, false, true, {0.505, 0.534}, {3.15, 2.48}},
    {128, 256, true, true, true, true, {0.576, 0.632}, {3.53, 3.19}},
};

PpTile gemm_pp_tile(int cfg) { return kPpTiles[cfg]; }

hipError_t launch_gemm_pp(const GemmParams& p, int bits, int cfg, int cus, hipStream_t st) {
    const bool sw = (p.flags & kFlagSwiglu) != 0 && p.c_kind != 2;
    const PpTile t = kPpTiles[cfg];
    if (!(bits == 4 ? t.w4 : t.w8) || !(sw ? t.swiglu : t.plain)) return hipErrorInvalidValue;
    switch (cfg * 2 + (bits == 8)) {
        case 0:
            return p.c_kind == 1 ? pp::launch_s<4, true, 1, 256, 256, 2, 4, 3>(p, cus, st)
                                 : pp::launch_s<4, true, 0, 256, 256, 2, 4, 3>(p, cus, st);
        case 2: return pp::launch_c<4, 256, 192, 4, 2>(p, cus, st);
        case 4: return pp::launch_c<4, 256, 128, 4, 2>(p, cus, st);
        case 5: return pp::launch_c<8, 256, 128, 4, 2>(p, cus, st);
        case 6: return pp::launch_c<4, 128, 96, 4, 2>(p, cus, st);
        case 7: return pp::launch_c<8, 128, 96, 4, 2>(p, cus, st);
        case 8: return pp::launch_c<4, 128, 128, 2, 4>(p, cus, st);
        case 9: return pp::launch_c<8, 128, 128, 2, 4>(p, cus, st);
        case 10: return pp::launch_c<4, 128, 192, 2, 4>(p, cus, st);
        case 11: return pp::launch_c<8, 128, 192, 2, 4>(p, cus, st);
        case 12:
            return p.c_kind == 1 ? pp::launch_s<4, true, 1, 128, 192, 4, 2, 4>(p, cus, st)
                                 : pp::launch_s<4, true, 0, 128, 192, 4, 2, 4>(p, cus, st);
        case 13:
            return p.c_kind == 1 ? pp::launch_s<8, true, 1, 128, 192, 4, 2, 3>(p, cus, st)
                                 : pp::launch_s<8, true, 0, 128, 192, 4, 2, 3>(p, cus, st);
        case 14: return pp::launch_c<4, 128, 256, 2, 4>(p, cus, st);
        case 15: return pp::launch_c<8, 128, 256, 2, 4>(p, cus, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace qlin
