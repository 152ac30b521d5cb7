/* SPDX-License-Identifier: Unlicense */

/* Device helpers shared by the GEMM kernels: buffer windows, the tile
 * order over the XCDs, and the epilogue of a wave's accumulators. */

#ifndef ICOREG_GEMM_DEV_H
#define ICOREG_GEMM_DEV_H

#include "act.h"
#include "bilinear.h"
#include "gemm.h"

typedef float floatx16 __attribute__((ext_vector_type(16)));

/* Offset past the end of every window: the load reads 0. */
#define GEMM_OOB 0x80000000u
/* gfx9 s_waitcnt immediate: vmcnt(0), expcnt and lgkmcnt not waited on. */
#define GEMM_WAIT_VM0 0x0F70

/* Word 3 of a raw buffer resource on gfx9-family parts: 32-bit data. */
#define GEMM_RSRC_FLAGS 0x00020000

/* Buffer window of `bytes` bytes from p: loads at byte offsets at or past
 * its end return 0. */
static __device__ __forceinline__ __amdgpu_buffer_rsrc_t
gemm_rsrc(const float *p, long long bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0,
                                             (int)(unsigned)bytes,
                                             GEMM_RSRC_FLAGS);
}

/* Four consecutive floats at byte offset off of window r: one 16-byte
 * load (VEC: the four are either all inside the window or all past its
 * end), else four 4-byte loads. */
template <bool VEC>
__device__ __forceinline__ float4 gemm_load4(__amdgpu_buffer_rsrc_t r,
                                             unsigned off)
{
    if (VEC)
        return __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
    float4 v;

    v.x = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
    v.y = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off + 4, 0, 0));
    v.z = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off + 8, 0, 0));
    v.w = __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off + 12, 0, 0));
    return v;
}

/* Components i of v with lo + i >= hi set to 0. */
__device__ __forceinline__ float4 mask4(float4 v, int lo, int hi)
{
    v.x = lo < hi ? v.x : 0.0f;
    v.y = lo + 1 < hi ? v.y : 0.0f;
    v.z = lo + 2 < hi ? v.z : 0.0f;
    v.w = lo + 3 < hi ? v.w : 0.0f;
    return v;
}

/* Output tile of linear block id L among T tiles: blocks are dealt to
 * the 8 XCDs round-robin (L % 8), so give XCD x the x-th contiguous
 * band of tiles. A bijection of 0..T-1. */
__device__ __forceinline__ int xcd_tile(int L, int T)
{
    const int q = T >> 3, rem = T & 7, x = L & 7, idx = L >> 3;

    return (x < rem ? x * (q + 1) : rem * (q + 1) + (x - rem) * q) + idx;
}

/* C's and R's batch (b0, b1) of g. */
__device__ __forceinline__ float *gemm_c(const gemm_args &g, long long b0, long long b1)
{
    return g.C + b0 * g.sc0 + b1 * g.sc1;
}

__device__ __forceinline__ const float *gemm_r(const gemm_args &g, long long b0, long long b1)
{
    return g.R ? (g.rup ? g.R + b0 * g.rs0 : g.R + b0 * g.sc0 + b1 * g.sc1) : nullptr;
}

/* N values of C = act(alpha v + bias) + R in column col, rows row(r) for r
 * < N (those below g.M), all loads of bias and R issued before the first
 * store: C may be R, so the compiler keeps every load behind the stores
 * that come before it in the source, a round trip a value (the 4x resized
 * addend of ELoFTR's MLP: 64 of them in turn, 45 us of a 66 us launch). */
template <int N, class ROW>
__device__ __forceinline__ void gemm_out(const gemm_args &g, float *C, const float *R, int col,
                                         float (&v)[N], ROW row)
{
    float b[N], x[N];

    if (col >= g.N)
        return;
    if (g.bias) {
#pragma unroll
        for (int r = 0; r < N; r++)
            b[r] = g.bias[g.biasrow ? min(row(r), g.M - 1) : col];
    }
    if (R && g.rup) {
        const int ry = col / g.rwo, rx = col - ry * g.rwo;

#pragma unroll
        for (int r = 0; r < N; r++)
            x[r] = bl_up(R + (long long)min(row(r), g.M - 1) * g.rh * g.rw, g.rh, g.rw, g.rsc, ry,
                         rx);
    }
    else if (R) {
#pragma unroll
        for (int r = 0; r < N; r++)
            x[r] = R[(long long)min(row(r), g.M - 1) * g.ldc + col];
    }
#pragma unroll
    for (int r = 0; r < N; r++) {
        v[r] *= g.alpha;
        if (g.bias)
            v[r] += b[r];
        if (R && g.rpre)
            v[r] += x[r];
        v[r] = icoreg_act(v[r], g.act, g.slope);
        if (R && !g.rpre)
            v[r] += x[r];
    }
#pragma unroll
    for (int r = 0; r < N; r++)
        if (row(r) < g.M)
            C[(long long)row(r) * g.ldc + col] = v[r];
}

/* The epilogue of the TM x TN 32 x 32 tiles of a wave whose block of C
 * starts at (r0, c0), batch (b0, b1). Register r of a tile holds row (r /
 * 4) * 8 + (lane / 32) * 4 + r % 4, column lane % 32. */
template <int TM, int TN>
__device__ __forceinline__ void gemm_epilogue(const gemm_args &g, const floatx16 (&acc)[TM][TN],
                                              long long b0, long long b1, int r0, int c0,
                                              int lane)
{
    float *C = gemm_c(g, b0, b1);
    const float *R = gemm_r(g, b0, b1);

#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            /* Half a tile at a time: the loads in flight are registers. */
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int ri = r0 + i * 32 + h * 16 + (lane >> 5) * 4;
                float v[8];

#pragma unroll
                for (int r = 0; r < 8; r++)
                    v[r] = acc[i][j][8 * h + r];
                gemm_out(g, C, R, c0 + j * 32 + (lane & 31), v,
                         [=](int r) { return ri + (r >> 2) * 8 + (r & 3); });
            }
        }
}

#endif /* ICOREG_GEMM_DEV_H */
