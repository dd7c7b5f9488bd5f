// Shared by the GEMM kernels whose lanes hold the int32 sums of four consecutive output channels of
// one row: the order of the tiles and the dequant / SiLU-gate / residual epilogue.
#pragma once

#include "qlin_internal.hpp"

namespace qlin {

typedef _Float16 h4 __attribute__((ext_vector_type(4)));

// Tile of workgroup b of n, in contiguous ranges per XCD (workgroups go round the eight XCDs), so that
// the tiles of a column find its weights in one L2; the first n % 8 ranges are one longer.  (With ranges
// only where 8 divides n, 189 tiles of the wave-split-K GEMM, 200 rows of W4 4096 x 2560, took 12.0 us;
// 9.7 so.  W8 9728 x 2560 at 100 rows, 189 tiles: 28.6 and 15.4.)  Columns of one tile have no weights
// to share, and keep the plain order where 8 does not divide n: W8 2560 x 19456 with SiLU-gate at 32 rows,
// 203 tiles, 14.0 us, in ranges 14.7.
__device__ __forceinline__ int xcd_tile(int b, int n, int m_tiles) {
    const int x = b & 7;
    if (m_tiles == 1 && (n & 7)) return b;
    return x * (n >> 3) + min(x, n & 7) + (b >> 3);
}

// Whether the rows of C / R take one vector access per four channels.
__device__ __forceinline__ bool c_rows_vec(const GemmParams& p) {
    return (p.ldc & 3) == 0 && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0;
}
__device__ __forceinline__ bool r_rows_vec(const GemmParams& p) {
    return (p.ldr & 3) == 0 && (reinterpret_cast<uintptr_t>(p.R) & 15) == 0;
}

// R[m, c .. c + 3] as floats; channels at or past ncols stay zero.
__device__ __forceinline__ void residual4(const GemmParams& p, int m, int c, int ncols, bool rvec, float r[4]) {
    const int64_t at = (int64_t)m * p.ldr + c;
    if (rvec && c + 3 < ncols) {
        if (p.r_f16) {
            const h4 v = *reinterpret_cast<const h4*>(reinterpret_cast<const _Float16*>(p.R) + at);
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = (float)v[e];
        } else {
            const float4 v = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.R) + at);
            r[0] = v.x;
            r[1] = v.y;
            r[2] = v.z;
            r[3] = v.w;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            r[e] = c + e >= ncols ? 0.0f
                   : p.r_f16      ? (float)reinterpret_cast<const _Float16*>(p.R)[at + e]
                                  : reinterpret_cast<const float*>(p.R)[at + e];
    }
}

// Output values of four channels from their sums (W4 sums carry a factor 16).  sm: the row's
// scale; sg / su: the channels' scales (gate and up); r: residual4's values, used when p.R is set.
template <int BITS, bool SWIGLU>
__device__ __forceinline__ void values4(const GemmParams& p, v4i gate, v4i up, float sm, const float* sg, const float* su,
                                        const float r[4], float o[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o[e] = ((float)(BITS == 4 ? gate[e] >> 4 : gate[e]) * sm) * sg[e];  // src/npu.rs:1117
        if constexpr (SWIGLU)
            o[e] = silu_gate(o[e], ((float)(BITS == 4 ? up[e] >> 4 : up[e]) * sm) * su[e]);  // src/npu.rs:1202-1208
    }
    if (!SWIGLU && p.R) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {  // src/model/dense.rs:486-489
            const float y = o[e] * p.rmult;
            o[e] = r[e] + y;
        }
    }
}

// Stores C[m, c .. c + 3].  kind: 0 f32, 1 fp16, 2 int32 (the sums themselves).
template <int BITS, bool SWIGLU>
__device__ __forceinline__ void finish4(const GemmParams& p, int kind, int m, int c, int ncols, bool vec, v4i gate, v4i up,
                                        float sm, const float* sg, const float* su, const float r[4]) {
    const int64_t at = (int64_t)m * p.ldc + c;
    if (kind == 2) {
        int32_t* C = reinterpret_cast<int32_t*>(p.C) + at;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (BITS == 4) gate[e] >>= 4;
        if (vec && c + 3 < ncols) {
            *reinterpret_cast<v4i*>(C) = gate;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < ncols) C[e] = gate[e];
        }
        return;
    }
    float o[4];
    values4<BITS, SWIGLU>(p, gate, up, sm, sg, su, r, o);
    if (kind == 1) {
        _Float16* C = reinterpret_cast<_Float16*>(p.C) + at;
        if (vec && c + 3 < ncols) {
            h4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = f16_of_f32(o[e]);
            *reinterpret_cast<h4*>(C) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < ncols) C[e] = f16_of_f32(o[e]);
        }
    } else {
        float* C = reinterpret_cast<float*>(p.C) + at;
        if (vec && c + 3 < ncols) {
            *reinterpret_cast<float4*>(C) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < ncols) C[e] = o[e];
        }
    }
}

}  // namespace qlin
