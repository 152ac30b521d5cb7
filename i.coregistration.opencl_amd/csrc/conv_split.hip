/* SPDX-License-Identifier: Unlicense */

/* Direct 5 x 5 convolution, stride 1, one group (DISK's layers), on the bf16
 * matrix instructions: the contract of conv.hip, every value split exactly
 * into three bf16 parts and six products accumulated in float32 (split.h),
 * the five small ones apart from the large one.
 *
 * What bounds it: the matrix cores and their power (busy 64 % of the CUs'
 * busy cycles in the first layer below, vector instructions 9 %), then the
 * barriers of the one block that a CU's LDS holds. An implicit GEMM of output
 * channels x pixels, 16 input channels of one tap an instruction step:
 *  - a block computes 64 WM channels x 256 pixels, a wave 64 x 64 (two
 *    tiles each way: an operand read feeds two products of each kind);
 *  - the input patch of 16 channels is split once, by the thread that
 *    loads it, and sits in LDS as three planes of [pixel][16 channels]: a
 *    tap's operand is one ds_read_b128 at the tap's shift, and every value
 *    staged is used by all 25 taps, so the split costs little (a GEMM on
 *    the unfolded input would split each value 25 times);
 *  - the two 16-byte halves of a pixel change places every eight pixels, so
 *    that 16 neighbouring pixels' halves lie in 64 different banks;
 *  - the next 16 channels are loaded a task (8 channels of a pixel) at a
 *    time between the taps, split and put into the other LDS buffer;
 *  - the filters are split and laid out in operand order by
 *    conv_split_weights_kernel, one pass over them a call, and come to LDS
 *    G taps at a time, a group ahead, through registers (by LDS DMA the
 *    compiler puts a full wait before the next LDS read: 728 us for DISK's
 *    last layer; read by every wave straight into its operands: 807 us).
 * Tiles whose sums are not all finite are formed again by a second pass of
 * the block over the unsplit values (v_mfma_f32_32x32x2f32).
 *
 * Measured on an MI355X against conv_mfma (conv.hip): 80 -> 129 channels at
 * 512 x 512 with normalisation (its 129th channel on conv_fewk_kernel both
 * times) 1206 -> 702 us, 256 -> 256 at 400 x 400 4080 -> 2274 us (129 -> 231
 * TFLOP/s), 96 -> 64 at 256 x 256 179 -> 127 us; error against 64-bit sums
 * 8.2e-7 -> 3.0e-7 on the first. 3 x 3 layers stay with Winograd: direct they
 * took 1.3 - 2.4 times as long (256 channels at 80 x 80, 64 at 320 x 320). */

#include <algorithm>
#include <hip/hip_runtime.h>

#include "act.h"
#include "conv.h"
#include "split.h"

#define CS_KS 5
/* Offset past the end of a 32-bit window. */
#define CS_OOB 0x80000000u

static __device__ __forceinline__ __amdgpu_buffer_rsrc_t cs_rsrc(const float *p,
                                                                 unsigned long long bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, (int)(unsigned)bytes,
                                             0x00020000);
}

/* 16-byte operands of the filters, scaled as the input is (split.h):
 * [64-channel block][16 input channels][tap][part][32-channel half][lane].
 * Lane l holds output channel l % 32 of the half, input channels 8 (l / 32)
 * .. + 7; zeros past K and C. One thread per (block, slice, tap, half,
 * lane). */
__global__ void __launch_bounds__(256)
    conv_split_weights_kernel(const float *__restrict__ w, int K, int C, int nc,
                              split_u4 *__restrict__ wp, long long n)
{
    constexpr int kk = CS_KS * CS_KS;
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;

    if (e >= n)
        return;
    const int lane = (int)(e & 63), i = (int)(e >> 6) & 1;
    const long long q = e >> 7;
    const int t = (int)(q % kk), s = (int)(q / kk % nc), mb = (int)(q / kk / nc);
    const int m = mb * 64 + i * 32 + (lane & 31), c0 = s * 16 + (lane >> 5) * 8;
    float v[8];
    split_u4 p[3];

#pragma unroll
    for (int c = 0; c < 8; c++)
        v[c] = m < K && c0 + c < C ? w[((long long)m * C + c0 + c) * kk + t] : 0.0f;
    split8(v, SPLIT_UP, p[0], p[1], p[2]);
#pragma unroll
    for (int k = 0; k < 3; k++)
        wp[((q * 3 + k) * 2 + i) * 64 + lane] = p[k];
}

/* Tiles TW pixels wide, WM x 4 waves, filters of G taps at a time. */
template <int TW, int WM>
__global__ void __launch_bounds__(256 * WM, WM)
    conv_split_kernel(const conv_args a, const split_u4 *__restrict__ wp)
{
    constexpr int KS = CS_KS, G = 2, WN = 4;
    constexpr int NT = 64 * WM * WN, KK = KS * KS, RJ = 32 / TW, TH = 2 * RJ * WN;
    constexpr int PH = TH - 1 + KS, PW = TW - 1 + KS;
    constexpr int PLANE = PH * PW * 2;        /* 16-byte chunks of a part */
    /* Tasks of the two channel halves, each padded to whole waves. */
    constexpr int HT = (PH * PW + 63) / 64 * 64, TASKS = (2 * HT + NT - 1) / NT;
    constexpr int NG = (KK + G - 1) / G;      /* groups of taps */
    constexpr int FT = WM * 6;                /* KiB of filters a tap */
    static_assert(TASKS < KK && NG >= 2, "tasks end before the slice's last barrier");
    __shared__ split_u4 lds[2][3 * PLANE];
    __shared__ split_u4 fil[2][G * FT * 64];  /* [tap][64 channels][part, half][lane] */

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, r32 = lane & 31, kh = lane >> 5;
    const int tiles_w = (a.Wo + TW - 1) / TW;
    const int oy0 = blockIdx.x / tiles_w * TH, ox0 = blockIdx.x % tiles_w * TW;
    const int m0 = (blockIdx.y * WM + wm) * 64;
    const int iy0 = oy0 - a.pad, ix0 = ox0 - a.pad;
    const int C = a.C, H = a.H, W = a.W, nc = (C + 15) / 16;
    const long long HW = (long long)H * W;
    const int piece = blockIdx.z % a.split, img = blockIdx.z / a.split;
    const int per = (nc + a.split - 1) / a.split, s0 = piece * per, s1 = min(nc, s0 + per);
    const float *in = a.in + (long long)img * a.in_stride;
    /* Byte offset inside a channel plane of this thread's tasks' pixels,
     * and their LDS places; task q is tid + NT q: channel half first, so
     * that a wave loads runs of one row. */
    unsigned poff[TASKS];
    int at[TASKS];
    int boff[KS];
    split_f16x acc[2][2], low[2][2];

#pragma unroll
    for (int q = 0; q < TASKS; q++) {
        const int e = tid + NT * q, half = e >= HT, p = e - half * HT;
        const int py = p / PW, px = p - py * PW, y = iy0 + py, x = ix0 + px;

        poff[q] = p < PH * PW && (unsigned)y < (unsigned)H && (unsigned)x < (unsigned)W
                      ? (unsigned)((y * W + x) * 4)
                      : CS_OOB;
        at[q] = p < PH * PW ? (py * PW + px) * 2 + (half ^ (px >> 3 & 1)) : -1;
    }
    /* This lane's pixel of the wave's first tile, shifted by column tap x. */
    const int pr = wn * 2 * RJ + r32 / TW, pc = r32 % TW;

#pragma unroll
    for (int x = 0; x < KS; x++)
        boff[x] = (pr * PW + pc + x) * 2 + (kh ^ ((pc + x) >> 3 & 1));
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[i][j][r] = low[i][j][r] = 0.0f;

    /* Task q of slice s: 8 channels of a pixel. The channel half is the
     * same for a wave, so each channel's window is scalar: none for
     * channels past C, and pixels outside the image lie past its end. */
    auto channel = [&](int s, int q) {
        return s * 16 + (__builtin_amdgcn_readfirstlane(tid + NT * q) >= HT ? 8 : 0);
    };
    auto fetch = [&](int s, int q, float (&v)[8]) {
        const int c0 = channel(s, q);
        const float *p = in + min(c0, C - 1) * HW;

#pragma unroll
        for (int c = 0; c < 8; c++, p += c0 + c < C ? HW : 0)
            v[c] = __builtin_bit_cast(
                float, __builtin_amdgcn_raw_buffer_load_b32(
                           cs_rsrc(p, c0 + c < C ? HW * 4 : 0), (int)poff[q], 0, 0));
    };
    auto stash = [&](int s, int q, float (&v)[8], split_u4 *d) {
        split_u4 h, m, l;

        if (a.mean) {
            const int c0 = channel(s, q);

#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int cc = min(c0 + c, C - 1);
                float x = (v[c] - a.mean[cc]) * a.rstd[cc];

                if (a.gate)
                    x = x >= 0.0f ? x : a.gate[cc] * x;
                v[c] = poff[q] != CS_OOB && c0 + c < C ? x : 0.0f;
            }
        }
        split8(v, SPLIT_UP, h, m, l);
        if (at[q] >= 0) {
            d[at[q]] = h;
            d[PLANE + at[q]] = m;
            d[2 * PLANE + at[q]] = l;
        }
    };
    /* Group g of slice s: chunk tid + NT q of it into fr[q]. */
    constexpr int FL = (G * FT * 64 + NT - 1) / NT;
    split_u4 fr[FL];
    /* All threads have a chunk q of n. Blocks of 64 channels then go without
     * a branch, between which a load may wait for the one before it (DISK's
     * 64-channel layers at 256 x 256 134 - 157 us with them); blocks of 128
     * keep it, their schedule is better with it (80 -> 129 channels at 512 x
     * 512 692 us against 723). */
    auto all = [](int q, int n) { return WM == 1 && NT * (q + 1) <= n; };
    auto filters = [&](int s, int g) {
        const int n = min(G, KK - g * G) * FT * 64;

#pragma unroll
        for (int q = 0; q < FL; q++) {
            const int c = tid + NT * q, t = c / (FT * 64), r = c % (FT * 64);
            const int mb = r / 384;

            if (all(q, n) || c < n)
                fr[q] = wp[((((long long)blockIdx.y * WM + mb) * nc + s) * KK + g * G + t) * 384 +
                           r % 384];
        }
    };
    auto filters_stash = [&](int g, split_u4 *d) {
        const int n = min(G, KK - g * G) * FT * 64;

#pragma unroll
        for (int q = 0; q < FL; q++)
            if (all(q, n) || tid + NT * q < n)
                d[tid + NT * q] = fr[q];
    };

    filters(s0, 0);
    filters_stash(0, fil[0]);
#pragma unroll
    for (int q = 0; q < TASKS; q++) {
        float v[8];

        fetch(s0, q, v);
        stash(s0, q, v, lds[0]);
    }
    __syncthreads();
    int fb = 0;

    for (int s = s0; s < s1; s++) {
        const int cur = (s - s0) & 1;
        const bool more = s + 1 < s1;
        float v[8];

#pragma unroll
        for (int t = 0; t < KK; t++) {
            constexpr int EACH = (KK - 1) / TASKS; /* taps a task is in flight */
            const int g = t / G, q = t / EACH;
            const split_u4 *fs = fil[fb] + (t % G * FT + wm * 6) * 64 + lane;
            split_b8 f[3][2], b[3][2];

            if (t % G == 0) {
                if (g + 1 < NG)
                    filters(s, g + 1);
                else if (more)
                    filters(s + 1, 0);
            }
            if (q < TASKS && t % EACH == 0 && more)
                fetch(s + 1, q, v);
#pragma unroll
            for (int k = 0; k < 3; k++) {
#pragma unroll
                for (int i = 0; i < 2; i++)
                    f[k][i] = __builtin_bit_cast(split_b8, fs[(k * 2 + i) * 64]);
#pragma unroll
                for (int j = 0; j < 2; j++)
                    b[k][j] = __builtin_bit_cast(
                        split_b8,
                        lds[cur][k * PLANE + (j * RJ + t / KS) * PW * 2 + boff[t % KS]]);
            }
            constexpr int pa[6] = {0, 0, 1, 1, 2, 0}, pb[6] = {0, 1, 0, 1, 0, 2};
#pragma unroll
            for (int w = 0; w < 6; w++)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        split_f16x &d = w == 0 ? acc[i][j] : low[i][j];

                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f[pa[w]][i], b[pb[w]][j], d, 0,
                                                                    0, 0);
                    }
            if (q < TASKS && t % EACH == EACH - 1 && more)
                stash(s + 1, q, v, lds[cur ^ 1]);
            if (t % G == G - 1 || t == KK - 1) {
                if (g + 1 < NG || more)
                    filters_stash(g + 1 < NG ? g + 1 : 0, fil[fb ^ 1]);
                __syncthreads();
                fb ^= 1;
            }
        }
    }

    unsigned redo = 0; /* bit 2 i + j: a sum of the tile is not finite */

#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            float z = 0.0f;

#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[i][j][r] = (acc[i][j][r] + low[i][j][r]) * SPLIT_DOWN;
                z = fmaf(acc[i][j][r], 0.0f, z);
            }
            redo |= __any(z != 0.0f) ? 1u << (2 * i + j) : 0u;
        }
    if (__syncthreads_or((int)redo)) {
        /* Those tiles again, on the float32 instructions: the 16 channels of
         * a slice unsplit, planes half the banks apart, and a row of taps'
         * filters at a time, [tap][output][16 channels and one]. */
        constexpr int PP = (PH * PW + 31) / 64 * 64 + 32, FR = 64 * WM, FP = 17;
        static_assert(PP >= PH * PW && 16 * PP * 4 <= (int)sizeof(lds) &&
                          KS * FR * FP * 4 <= (int)sizeof(fil),
                      "slice and filters fit");
        float *const ps = (float *)lds, *const fs = (float *)fil;

#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    low[i][j][r] = 0.0f;
        for (int s = s0; s < s1; s++) {
            __syncthreads();
#pragma unroll 2
            for (int e = tid; e < 16 * PH * PW; e += NT) {
                const int c = e / (PH * PW), p = e % (PH * PW), k = min(s * 16 + c, C - 1);
                const int y = iy0 + p / PW, x = ix0 + p % PW;
                const bool in_ = s * 16 + c < C && (unsigned)y < (unsigned)H &&
                                 (unsigned)x < (unsigned)W;
                float v = in[k * HW + (in_ ? (long long)y * W + x : 0)];

                if (a.mean) {
                    v = (v - a.mean[k]) * a.rstd[k];
                    if (a.gate)
                        v = v >= 0.0f ? v : a.gate[k] * v;
                }
                ps[c * PP + p] = in_ ? v : 0.0f;
            }
#pragma unroll 1
            for (int ky = 0; ky < KS; ky++) {
                if (ky > 0)
                    __syncthreads();
#pragma unroll 4
                for (int e = tid; e < FR * 16 * KS; e += NT) {
                    const int m = e / (16 * KS), c = e % (16 * KS) / KS, x = e % KS;
                    const int k = blockIdx.y * FR + m;

                    fs[(x * FR + m) * FP + c] =
                        k < a.K && s * 16 + c < C
                            ? a.w[((long long)k * C + s * 16 + c) * KK + ky * KS + x]
                            : 0.0f;
                }
                __syncthreads();
#pragma unroll 1
                for (int x = 0; x < KS; x++) {
                    const float *f = fs + (x * FR + wm * 64 + r32) * FP + kh;
                    const float *b = ps + kh * PP + (pr + ky) * PW + pc + x;

#pragma unroll
                    for (int c = 0; c < 16; c += 2)
#pragma unroll
                        for (int i = 0; i < 2; i++)
#pragma unroll
                            for (int j = 0; j < 2; j++)
                                if (redo >> (2 * i + j) & 1u)
                                    low[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                        f[i * 32 * FP + c], b[c * PP + j * RJ * PW], low[i][j], 0,
                                        0, 0);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
                if (redo >> (2 * i + j) & 1u)
                    acc[i][j] = low[i][j];
    }

    const bool whole = a.split == 1;
    float *out = whole ? a.out + (long long)img * a.out_stride
                       : a.part + ((long long)piece * (gridDim.z / a.split) + img) * a.K * a.Ho *
                                      a.Wo;

#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int oy = oy0 + pr + j * RJ, ox = ox0 + pc;
        const bool inside = oy < a.Ho && ox < a.Wo;

#pragma unroll
        for (int i = 0; i < 2; i++) {
            float bias[16];
            const int mr = m0 + i * 32 + kh * 4;

#pragma unroll
            for (int r = 0; r < 16; r++)
                bias[r] = whole && a.bias ? a.bias[min(mr + (r >> 2) * 8 + (r & 3), a.K - 1)] : 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int m = mr + (r >> 2) * 8 + (r & 3);
                float v = acc[i][j][r];

                if (whole)
                    v = icoreg_act(v + bias[r], a.act, a.slope);
                if (inside && m < a.K)
                    out[((long long)m * a.Ho + oy) * a.Wo + ox] = v;
            }
        }
    }
}

/* ---- host --------------------------------------------------------------- */

size_t conv_split_weight_bytes(int K, int C)
{
    /* Whole blocks of 64 or 128 channels. */
    const int kb = K > 64 ? (K + 127) / 128 * 2 : 1;

    return (size_t)kb * ((C + 15) / 16) * CS_KS * CS_KS * 6 * 64 * 16;
}

template <int TW, int WM>
static void cs_launch(const conv_args &a, const void *wp, int nb, hipStream_t s)
{
    constexpr int TH = 256 / TW;
    const int tiles = ((a.Wo + TW - 1) / TW) * ((a.Ho + TH - 1) / TH);

    hipLaunchKernelGGL((conv_split_kernel<TW, WM>),
                       dim3(tiles, (a.K + 64 * WM - 1) / (64 * WM), nb * a.split), dim3(256 * WM),
                       0, s, a, (const split_u4 *)wp);
}

conv_split_plan conv_split_choose(const conv_args &a, int ks, int st, int nb, int cus)
{
    auto tiles = [&](int tw) {
        const int th = 256 / tw;

        return (long long)((a.Ho + th - 1) / th) * ((a.Wo + tw - 1) / tw);
    };
    conv_split_plan p;

    p.bm = a.K > 64 ? 128 : 64;
    p.tw = tiles(16) < tiles(32) ? 16 : 32;
    const long long blocks = tiles(p.tw) * ((a.K + p.bm - 1) / p.bm) * nb;
    const int nc = (a.C + 15) / 16;

    /* Pieces over the input channels where they shorten the slowest CU's
     * share. A CU holds one block (its LDS), and a round of blocks takes about 9
     * us and a slice of 16 channels 14.4 us (64 output channels) or 20.8 (128),
     * 2.5 and 1.4 more where it is normalised; pieces write and read their sums
     * at 2.3 or 3.6 TB/s (fitted to 22000 times of 7100 layers, within 5 % at the
     * median). Cut into about two blocks a CU instead, one layer in two ran 5 %
     * or more longer than it could, up to 1.6 times, and one in eight longer
     * than on conv_mfma, up to 1.9 times (19 -> 256 channels, normalised, at 38 x
     * 470: 83 us there, 97 in two pieces, 72 whole); so cut, one in 20: most have
     * 17 to 21 channels, whose second slice is nearly empty (up to 1.46 times), a
     * few a nearly empty second round of blocks (up to 1.6 times). */
    const double slice = p.bm == 64 ? 14.4 + (a.mean ? 2.5 : 0.0) : 20.8 + (a.mean ? 1.4 : 0.0);
    const double mb = 8e-6 * nb * a.K * a.Ho * a.Wo / (p.bm == 64 ? 2.3 : 3.6);
    double best = 1e30;

    p.split = 1;
    for (int s = 1; s <= std::min(nc, 16); s++) {
        const int per = (nc + s - 1) / s;
        const long long n = blocks * s;
        const double rounds = n <= 4LL * cus ? (double)((n + cus - 1) / cus) : (double)n / cus + 0.5;
        const double us = rounds * (8.6 + slice * per) + (s > 1 ? mb * s : 0.0);

        /* None empty, and the pieces' grid in range. */
        if ((nc + per - 1) / per == s && (s == 1 || nb * (long long)s <= 65535) && us < best) {
            best = us;
            p.split = s;
        }
    }
    /* Below 96 blocks of 64 channels on 256 CUs the smaller blocks of
     * conv_mfma win (128 -> 64 channels at 128 x 128, 64 blocks: 79 us against
     * 89; 64 -> 128 at 100 x 100, 98: 65 against 51). With one chunk of
     * input channels a block is mostly start and end: more than 32 outputs
     * need 256 (16 -> 64 at 62 x 370, 96: 31.5 us against 37; 16 -> 128 at 128 x
     * 128, 128: 31 against 41; 16 -> 64 at 256 x 256, 256: 43 -> 39). */
    p.ok = ks == CS_KS && st == 1 && a.C >= 16 && a.K >= 32 &&
           8 * blocks * (p.bm / 64) >= (a.C < 32 && a.K > 32 ? 8LL : 3LL) * cus;
    return p;
}

void conv_split_launch(const conv_args &a, const conv_split_plan &p, void *wp, int nb,
                       hipStream_t s)
{
    const long long n = (long long)(conv_split_weight_bytes(a.K, a.C) / 48);

    hipLaunchKernelGGL(conv_split_weights_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       s, a.w, a.K, a.C, (a.C + 15) / 16, (split_u4 *)wp, n);
    if (p.tw == 16 && p.bm == 128)
        cs_launch<16, 2>(a, wp, nb, s);
    else if (p.tw == 16)
        cs_launch<16, 1>(a, wp, nb, s);
    else if (p.bm == 128)
        cs_launch<32, 2>(a, wp, nb, s);
    else
        cs_launch<32, 1>(a, wp, nb, s);
}
