/* SPDX-License-Identifier: Unlicense */

/* The float32 GEMM of long sums: C = act(alpha A op(B) + bias) + R with every
 * operand value split exactly into three bf16 parts (split.h) and six
 * v_mfma_f32_32x32x16_bf16 products a 32 x 32 x 16 step, accumulated in
 * float32. The scale that keeps every operand's bits (split.h) is a multiply
 * a staged value: 159 -> 161 us on the first shape below.
 *
 * What bounds it: the matrix cores and the power they draw. Six bf16
 * products take 192 cycles where eight v_mfma_f32_32x32x2f32 take 512; on
 * random operands the bare instruction stream holds 1.75 - 1.82 PFLOP/s of
 * bf16 (2.48 on zeros: the clock falls), 291 - 302 TFLOP/s of float32 work,
 * and a large bf16 library product 1.34 PFLOP/s. What the kernel adds to the
 * stream: 6.5 vector instructions a staged value for the split and the LDS
 * traffic of three parts, both in proportion to the tile's sides, against
 * matrix work in proportion to its area; hence the largest tile that still
 * gives the CUs equal shares. Of the CUs' busy cycles the matrix pipes take
 * 0.57 and vector instructions 0.50 on the first shape below, 0.67 and 0.33
 * on the second.
 *
 *  - A block stages 32 k of both operands: buffer loads through windows
 *    over the tile's rows (past the edge they read 0) into registers a
 *    slice ahead, split there, three [row][k] planes in LDS (one buffer and
 *    two barriers a slice: the CU's other blocks fill the gap).
 *    A lane's MFMA operand is eight consecutive k: one ds_read_b128.
 *  - The 16-byte chunks of a row are stored XORed with bits of the row so
 *    that the 16 rows a quarter of a read touches lie in 64 different
 *    banks (conflicts take none of the LDS cycles with B N x K, 17 % with B
 *    K x N).
 *  - The five products below hh have accumulators of their own, added to
 *    hh's at the end: added to the large sums one by one they round away
 *    (mm of a sum of squares did, which moved such sums by -1.3e-7 of their
 *    value), and hh's sums take a sixth of the roundings.
 *  - 32 x 32 tiles whose sums are not all finite are formed again on
 *    v_mfma_f32_32x32x2f32 by a second pass of the block over its unsplit
 *    slices, so infinities, NaN and overflow come out as float32 products
 *    give them, at about the time of the fp32 kernel on top.
 *
 * Measured on an MI355X against the kernel on v_mfma_f32_32x32x2f32
 * (gemm.hip): 3202 x 4096 x 1024 with bias and GELU 241 -> 167 us (111 ->
 * 161 TFLOP/s of float32 work), 3202 x 1024 x 4096 248 -> 179 us, 1140 x
 * 11664 x 1140 (B given K x N) 291 -> 200 us; error against 64-bit sums at K
 * = 1024 6.4e-7 -> 2.1e-7. One block of a CU's two computes while the other
 * stages; 128 x 256 tiles of 4 x 64 x 128 waves ran 146 us on the first shape
 * with one accumulator set, but have no registers for two (199 us). */

#include <algorithm>
#include <hip/hip_runtime.h>

#include "gemm_dev.h"
#include "split.h"

/* Most pieces a tile is cut into over K. */
#define SPLIT_MAX 8

#define SPLIT_BK 32 /* k of a slice */

/* Tile shape: BM x BN outputs, WM x WN waves, at least OCC of them a SIMD. */
template <int BM_, int BN_, int WM_, int WN_, int OCC_> struct split_tile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, OCC = OCC_;
    static constexpr int NT = 64 * WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;
};
typedef split_tile<128, 128, 2, 4, 4> split_m;
typedef split_tile<64, 128, 2, 2, 3> split_s;
typedef split_tile<64, 64, 2, 2, 4> split_xs;

/* Row and column tile of tile number t: down the columns where there are
 * fewer rows of tiles, so that the tiles an XCD's L2 serves together share
 * the longer operand's panels. */
__device__ __forceinline__ void split_order(int t, int tiles_m, int tiles_n, int &tm, int &tn)
{
    if (tiles_m <= tiles_n) {
        tn = t / tiles_m;
        tm = t - tn * tiles_m;
    }
    else {
        tm = t / tiles_n;
        tn = t - tm * tiles_n;
    }
}

/* Eight floats at byte offset off of window r. */
template <bool VEC>
__device__ __forceinline__ void split_load8(__amdgpu_buffer_rsrc_t r, unsigned off, float (&v)[8])
{
    const float4 a = gemm_load4<VEC>(r, off), b = gemm_load4<VEC>(r, off + 16);

    v[0] = a.x;
    v[1] = a.y;
    v[2] = a.z;
    v[3] = a.w;
    v[4] = b.x;
    v[5] = b.y;
    v[6] = b.z;
    v[7] = b.w;
}

/* Element (k, column) of a convolution's unfolded input (0 in the
 * padding): window element k of the output pixel whose window starts at
 * (cy, cx), normalised and gated when g asks for it. */
__device__ __forceinline__ float split_gather(const gemm_args &g, const float *B, int k, int cy,
                                              int cx, bool in)
{
    const int khw = g.kh * g.kw, c = k / khw, rem = k - c * khw;
    const int ki = rem / g.kw, y = cy + ki * g.dy, x = cx + (rem - ki * g.kw) * g.dx;
    float v;

    in = in && (unsigned)y < (unsigned)g.ch && (unsigned)x < (unsigned)g.cw;
    v = B[in ? ((long long)c * g.ch + y) * g.cw + x : 0];
    if (g.mean) {
        v = (v - g.mean[c]) * g.rstd[c];
        if (g.gate)
            v = v >= 0.0f ? v : g.gate[c] * v;
    }
    return in ? v : 0.0f;
}

template <class T, int MODE, bool VEC>
__global__ void __launch_bounds__(T::NT, T::OCC) gemm_split_kernel(const gemm_args g)
{
    constexpr int BM = T::BM, BN = T::BN, BK = SPLIT_BK, WN = T::WN, NT = T::NT;
    constexpr int TM = T::TM, TN = T::TN, WR = BM / T::WM, WC = BN / WN;
    constexpr int CH = BK / 8;                /* 16-byte chunks of a row and plane */
    constexpr int PA = BM * CH, PB = BN * CH; /* chunks a plane */
    constexpr int AC = PA / NT, BC = PB / NT; /* chunks a thread */
    static_assert(PA % NT == 0 && PB % NT == 0 && BN % 64 == 0, "tile shape");
    __shared__ split_u4 lds[3 * (PA + PB)];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, r32 = lane & 31, kh = lane >> 5;
    const int M = g.M, N = g.N, K = g.K, nka = (K + BK - 1) / BK;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int L = blockIdx.x, piece = -1, kt0 = 0, kt1 = nka, tm, tn;

    if (g.split > 1 && L >= g.nfull) {
        const int p = L - g.nfull;

        piece = p % g.split;
        L = g.nfull + p / g.split;
        kt0 = piece * nka / g.split;
        kt1 = (piece + 1) * nka / g.split;
    }
    split_order(xcd_tile(L, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const long long bt = blockIdx.y, b0 = bt / g.nb1, b1 = bt % g.nb1;
    const float *A = g.A + b0 * g.sa0 + b1 * g.sa1;
    const float *B = g.B + b0 * g.sb0 + b1 * g.sb1;
    const long long lda = g.lda, ldb = g.ldb;
    const int rows_a = min(BM, M - m0), cols_b = min(BN, N - n0);
    const float *Ab = A + m0 * lda, *Bb = MODE == GEMM_B_NK ? B + n0 * ldb : B + n0;
    static_assert(NT % BN == 0, "a thread keeps its column of B");
    /* Chunk q of a plane: row q / CH, chunk q % CH; B given K x N: column
     * q % BN, chunk q / BN (the same for a whole wave). */
    unsigned aoff[AC], boff[BC];
    float ra[AC][8], rb[BC][8];
    floatx16 acc[TM][TN], low[TM][TN];

#pragma unroll
    for (int e = 0; e < AC; e++) {
        const int q = tid + NT * e;

        aoff[e] = (unsigned)(((q / CH) * lda + (q % CH) * 8) * 4);
    }
#pragma unroll
    for (int e = 0; e < BC; e++) {
        const int q = tid + NT * e;

        boff[e] = MODE == GEMM_B_NK ? (unsigned)(((q / CH) * ldb + (q % CH) * 8) * 4)
                                    : (unsigned)((q % BN) * 4);
    }
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                acc[i][j][r] = low[i][j][r] = 0.0f;

    /* Slice k0 into registers. Rows past the matrix lie past their
     * window's end and read 0; k past K read the next row of all but the
     * last one and are set to 0. */
    auto fetch = [&](int k0) {
        const __amdgpu_buffer_rsrc_t wa = gemm_rsrc(Ab + k0, ((rows_a - 1) * lda + K - k0) * 4);

#pragma unroll
        for (int e = 0; e < AC; e++)
            split_load8<VEC>(wa, aoff[e], ra[e]);
        if (MODE == GEMM_B_NK) {
            const __amdgpu_buffer_rsrc_t wb =
                gemm_rsrc(Bb + k0, ((cols_b - 1) * ldb + K - k0) * 4);

#pragma unroll
            for (int e = 0; e < BC; e++)
                split_load8<VEC>(wb, boff[e], rb[e]);
        }
        else if (MODE == GEMM_B_CONV) {
            /* A thread's column is the same in all its chunks (BN divides
             * the block's threads). */
            const int p = n0 + tid % BN;
            const int cy = p / g.wo * g.sy - g.py, cx = p % g.wo * g.sx - g.px;

#pragma unroll
            for (int e = 0; e < BC; e++) {
                const int kr = k0 + 8 * __builtin_amdgcn_readfirstlane((tid + NT * e) / BN);

#pragma unroll
                for (int i = 0; i < 8; i++)
                    rb[e][i] = split_gather(g, B, min(kr + i, K - 1), cy, cx,
                                            p < N && kr + i < K);
            }
        }
        else {
            /* A window a row of B: the base and its size are scalars. */
#pragma unroll
            for (int e = 0; e < BC; e++) {
                const int kr = k0 + 8 * __builtin_amdgcn_readfirstlane((tid + NT * e) / BN);
                const float *p = Bb + min(kr, K - 1) * ldb;

#pragma unroll
                for (int i = 0; i < 8; i++, p += kr + i < K ? ldb : 0) {
                    const __amdgpu_buffer_rsrc_t wb = gemm_rsrc(p, kr + i < K ? cols_b * 4 : 0);

                    rb[e][i] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(wb, (int)boff[e], 0, 0));
                }
            }
        }
        if (k0 + BK > K) {
#pragma unroll
            for (int e = 0; e < AC; e++)
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (k0 + ((tid + NT * e) % CH) * 8 + i >= K)
                        ra[e][i] = 0.0f;
            if (MODE == GEMM_B_NK) {
#pragma unroll
                for (int e = 0; e < BC; e++)
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (k0 + ((tid + NT * e) % CH) * 8 + i >= K)
                            rb[e][i] = 0.0f;
            }
        }
    };
    auto stash = [&]() {
        split_u4 *const as = lds, *const bs = as + 3 * PA, h, m, l;

#pragma unroll
        for (int e = 0; e < AC; e++) {
            const int q = tid + NT * e, row = q / CH;
            const int at = row * CH + ((q % CH) ^ ((row >> 2) & (CH - 1)));

            split8(ra[e], SPLIT_UP, h, m, l);
            as[at] = h;
            as[PA + at] = m;
            as[2 * PA + at] = l;
        }
#pragma unroll
        for (int e = 0; e < BC; e++) {
            const int q = tid + NT * e, row = MODE == GEMM_B_NK ? q / CH : q % BN;
            const int ch = MODE == GEMM_B_NK ? q % CH : q / BN;
            const int at = row * CH + (ch ^ ((row >> 2) & (CH - 1)));

            split8(rb[e], SPLIT_UP, h, m, l);
            bs[at] = h;
            bs[PB + at] = m;
            bs[2 * PB + at] = l;
        }
    };
    auto compute = [&]() {
        const split_u4 *const as = lds, *const bs = as + 3 * PA;

#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            split_b8 a[3][TM], b[3][TN];

#pragma unroll
            for (int p = 0; p < 3; p++) {
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const int row = wm * WR + i * 32 + r32;

                    a[p][i] = __builtin_bit_cast(
                        split_b8,
                        as[p * PA + row * CH + ((2 * ks + kh) ^ ((row >> 2) & (CH - 1)))]);
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const int row = wn * WC + j * 32 + r32;

                    b[p][j] = __builtin_bit_cast(
                        split_b8,
                        bs[p * PB + row * CH + ((2 * ks + kh) ^ ((row >> 2) & (CH - 1)))]);
                }
            }
            /* Parts (h, m, l) = (0, 1, 2); hh into acc, the other five
             * into low. */
            constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
            for (int t = 0; t < 6; t++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) {
                        floatx16 &d = t == 5 ? acc[i][j] : low[i][j];

                        d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[pa[t]][i], b[pb[t]][j], d,
                                                                    0, 0, 0);
                    }
        }
    };

    if (kt0 < kt1) {
        fetch(kt0 * BK);
        for (int kt = kt0; kt < kt1; kt++) {
            __syncthreads();
            stash();
            __syncthreads();
            if (kt + 1 < kt1)
                fetch((kt + 1) * BK);
            compute();
        }
    }
    unsigned redo = 0; /* bit i TN + j: a sum of the tile is not finite */

#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            float z = 0.0f; /* NaN if a sum is not finite */

#pragma unroll
            for (int r = 0; r < 16; r++) {
                acc[i][j][r] = (acc[i][j][r] + low[i][j][r]) * SPLIT_DOWN;
                z = fmaf(acc[i][j][r], 0.0f, z);
            }
            redo |= __any(z != 0.0f) ? 1u << (i * TN + j) : 0u;
        }
    if (__syncthreads_or((int)redo)) {
        /* Those tiles again, on the float32 instructions: the block stages
         * its slices unsplit, [row][k], rows one float apart in the banks. */
        constexpr int P = BK + 1;
        static_assert((BM + BN) * P <= 4 * 3 * (PA + PB), "the slices fit");
        float *const as = (float *)lds, *const bs = as + BM * P;

#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    low[i][j][r] = 0.0f;
        for (int kt = kt0; kt < kt1; kt++) {
            fetch(kt * BK);
            __syncthreads();
#pragma unroll
            for (int e = 0; e < AC; e++) {
                const int q = tid + NT * e;

#pragma unroll
                for (int x = 0; x < 8; x++)
                    as[q / CH * P + q % CH * 8 + x] = ra[e][x];
            }
#pragma unroll
            for (int e = 0; e < BC; e++) {
                const int q = tid + NT * e, row = MODE == GEMM_B_NK ? q / CH : q % BN;
                const int ch = MODE == GEMM_B_NK ? q % CH : q / BN;

#pragma unroll
                for (int x = 0; x < 8; x++)
                    bs[row * P + ch * 8 + x] = rb[e][x];
            }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    if (redo >> (i * TN + j) & 1u) {
                        const float *a = as + (wm * WR + i * 32 + r32) * P + kh;
                        const float *b = bs + (wn * WC + j * 32 + r32) * P + kh;

#pragma unroll
                        for (int k = 0; k < BK; k += 2)
                            low[i][j] =
                                __builtin_amdgcn_mfma_f32_32x32x2f32(a[k], b[k], low[i][j], 0, 0, 0);
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
                if (redo >> (i * TN + j) & 1u)
                    acc[i][j] = low[i][j];
    }
    if (piece >= 0) {
        /* The piece's sums: float4 e = 4 (i TN + j) + r / 4 of every
         * thread of the block, threads together. */
        float4 *pp = (float4 *)g.part +
                     ((long long)(L - g.nfull) * g.split + piece) * (TM * TN * 4 * NT) + tid;

#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    pp[((i * TN + j) * 4 + q) * NT] =
                        make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                                    acc[i][j][4 * q + 3]);
        return;
    }
    gemm_epilogue<TM, TN>(g, acc, b0, b1, m0 + wm * WR, n0 + wn * WC, lane);
}

/* The cut tiles (one batch): block e of a tile adds float4 e of every
 * thread of the tile's pieces, in piece order, then the epilogue. Bound by
 * the pieces' bytes (written once, read once: 2 x 27 MB in about 15 us for
 * a ViT's second MLP layer cut in two). */
template <class T>
__global__ void __launch_bounds__(T::NT) split_pieces_kernel(const gemm_args g)
{
    constexpr int TM = T::TM, TN = T::TN, NT = T::NT, E = TM * TN * 4;
    const int t = blockIdx.x / E, e = blockIdx.x % E;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tiles_m = (g.M + T::BM - 1) / T::BM, tiles_n = (g.N + T::BN - 1) / T::BN;
    const float4 *q = (const float4 *)g.part + ((long long)t * g.split * E + e) * NT + tid;
    int tm, tn;
    float4 p[SPLIT_MAX];

    split_order(xcd_tile(g.nfull + t, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const int row = tm * T::BM + wave / T::WN * (T::BM / T::WM) + e / (4 * TN) * 32 + (e & 3) * 8 +
                    (lane >> 5) * 4;
    const int col = tn * T::BN + wave % T::WN * (T::BN / T::WN) + (e / 4) % TN * 32 + (lane & 31);

    if (row >= g.M || col >= g.N)
        return;
#pragma unroll
    for (int s = 0; s < SPLIT_MAX; s++)
        if (s < g.split)
            p[s] = q[(long long)s * E * NT];
#pragma unroll
    for (int s = 1; s < SPLIT_MAX; s++)
        if (s < g.split) {
            p[0].x += p[s].x;
            p[0].y += p[s].y;
            p[0].z += p[s].z;
            p[0].w += p[s].w;
        }
    float v[4] = {p[0].x, p[0].y, p[0].z, p[0].w};

    gemm_out(g, g.C, g.R, col, v, [=](int r) { return row + r; });
}

/* ---- host --------------------------------------------------------------- */

namespace {

struct split_choice {
    int tile;         /* 0 .. 2: split_m, split_s, split_xs */
    int nfull, split; /* tiles run whole; pieces of the others */
};

constexpr int split_bm[3] = {split_m::BM, split_s::BM, split_xs::BM};
constexpr int split_bn[3] = {split_m::BN, split_s::BN, split_xs::BN};

long long split_tiles(int tile, int M, int N)
{
    return (long long)((M + split_bm[tile] - 1) / split_bm[tile]) *
           ((N + split_bn[tile] - 1) / split_bn[tile]);
}

/* Time model of a tile shape's grid, us: a CU's m tiles take m share a 1024 of
 * K, but no less than alone (one tile's waves do not fill the CU), and m fixed
 * for their ends; call for the launch and a tile's first loads, cut for the
 * second launch where tiles are cut over K. */
struct split_cost {
    double alone, share, fixed, call, cut;
};

/* split_m, split_s and split_xs by how the operands come (split_row), fitted
 * to 170000 times of 11600 products (M, N 16 .. 4096, K 513 .. 4096, every
 * tile and cut) on an MI355X: 16-byte rows within 2 - 3 % of them at the
 * median, 4-byte loads within 4 - 8 %. The gathered convolution, which is never
 * cut, has figures from the patch embedding. */
const split_cost split_costs[5][3] = {
    /* B N x K, 16-byte rows; else */
    {{41.6, 30.3, 1.6, 6.3, 0.0}, {35.1, 21.8, 0.1, 7.4, 0.0}, {22.5, 13.6, 0.0, 6.3, 0.8}},
    {{93.4, 76.0, 0.0, 0.0, 5.1}, {73.4, 55.1, 0.0, 6.7, 0.0}, {50.7, 38.3, 0.0, 3.9, 2.2}},
    /* B K x N, 16-byte rows of A; else */
    {{48.7, 34.4, 0.9, 7.1, 0.0}, {47.7, 26.2, 0.2, 7.5, 0.0}, {29.7, 14.3, 0.0, 6.4, 0.9}},
    {{74.8, 45.5, 4.7, 0.0, 1.6}, {62.9, 35.5, 0.0, 6.9, 0.1}, {44.9, 25.2, 0.0, 4.9, 1.6}},
    /* B gathered */
    {{42.0, 42.0, 4.0, 0.0, 0.0}, {35.0, 23.0, 2.5, 0.0, 0.0}, {22.0, 13.0, 1.0, 0.0, 0.0}},
};

int split_row(int bmode, bool va, bool vb)
{
    return bmode == GEMM_B_NK ? (va && vb ? 0 : 1) : bmode == GEMM_B_KN ? (va ? 2 : 3) : 4;
}

/* The tile shape and cut with the smallest estimated time on cus CUs. With
 * one batch and a plain epilogue, the tiles left over after an equal whole
 * number a CU, or all of them, may be cut over K into up to SPLIT_MAX pieces
 * of at least 128 k. */
split_choice split_plan(const gemm_args &g, int row, int nb, bool cut, int cus)
{
    split_choice best = {2, 0, 1};
    double tbest = 1e30;
    const double k = std::max(g.K, 32) / 1024.0;
    /* whole tiles, and pieces of 1 / s of K (their sums written and read at
     * about 4.5 TB/s): the CU with the most, past four of them leveled out. */
    auto consider = [&](int i, int full, long long whole, int pieces, int s) {
        const split_cost &c = split_costs[row][i];
        auto part = [&](long long n, int pieces_) {
            const double m =
                n <= 4LL * cus ? (double)((n + cus - 1) / cus) : (double)n / cus + 0.5;

            return n ? std::max(c.alone, m * c.share) * k / pieces_ + m * c.fixed : 0.0;
        };
        double t = c.call + part(whole, 1);

        if (pieces)
            t += part(pieces, s) + c.cut + 8.0 * pieces * split_bm[i] * split_bn[i] / 4.5e6;
        if (t < tbest) {
            tbest = t;
            best = {i, full, s};
        }
    };

    for (int i = 0; i < 3; i++) {
        const long long n = split_tiles(i, g.M, g.N);

        consider(i, 0, n * nb, 0, 1);
        if (!cut || nb != 1 || n >= 4LL * cus)
            continue;
        const int all = (int)n, rem = all % cus, smax = std::min(g.K / 128, SPLIT_MAX);

        for (int s = 2; s <= smax; s++) {
            consider(i, 0, 0, all * s, s);
            if (rem && rem < all)
                consider(i, all - rem, all - rem, rem * s, s);
        }
    }
    return best;
}

template <class T, int MODE>
void split_launch_mode(const gemm_args &g, int nb, bool vec, hipStream_t s)
{
    const int n = ((g.M + T::BM - 1) / T::BM) * ((g.N + T::BN - 1) / T::BN);
    const int tail = g.split > 1 ? n - g.nfull : 0;
    const dim3 grid(g.split > 1 ? g.nfull + tail * g.split : n, nb);

    if (vec)
        hipLaunchKernelGGL((gemm_split_kernel<T, MODE, true>), grid, dim3(T::NT), 0, s, g);
    else
        hipLaunchKernelGGL((gemm_split_kernel<T, MODE, false>), grid, dim3(T::NT), 0, s, g);
    if (tail)
        hipLaunchKernelGGL((split_pieces_kernel<T>), dim3(tail * T::TM * T::TN * 4), dim3(T::NT),
                           0, s, g);
}

template <class T>
void split_launch_tile(const gemm_args &g, int bmode, int nb, bool va, bool vb, hipStream_t s)
{
    if (bmode == GEMM_B_NK)
        split_launch_mode<T, GEMM_B_NK>(g, nb, va && vb, s);
    else if (bmode == GEMM_B_KN)
        split_launch_mode<T, GEMM_B_KN>(g, nb, va, s);
    else
        split_launch_mode<T, GEMM_B_CONV>(g, nb, va, s);
}

bool split_cut_ok(const gemm_args &g, int bmode, int nb)
{
    return bmode != GEMM_B_CONV && nb == 1 && g.nb1 == 1 && !g.rup;
}

} // namespace

size_t gemm_split_floats(const gemm_args &g, int bmode, int nb, bool va, bool vb, int cus)
{
    if (!split_cut_ok(g, bmode, nb))
        return 0;
    const split_choice c = split_plan(g, split_row(bmode, va, vb), nb, true, cus);

    return c.split > 1 ? (size_t)(split_tiles(c.tile, g.M, g.N) - c.nfull) * c.split *
                             split_bm[c.tile] * split_bn[c.tile]
                       : 0;
}

void gemm_split_launch(const gemm_args &g, int bmode, int nb, bool va, bool vb, int cus,
                       hipStream_t s)
{
    const split_choice c = split_plan(g, split_row(bmode, va, vb), nb,
                                      g.part && split_cut_ok(g, bmode, nb), cus);
    gemm_args a = g;

    a.nfull = c.nfull;
    a.split = c.split;
    switch (c.tile) {
    case 0:
        split_launch_tile<split_m>(a, bmode, nb, va, vb, s);
        break;
    case 1:
        split_launch_tile<split_s>(a, bmode, nb, va, vb, s);
        break;
    default:
        split_launch_tile<split_xs>(a, bmode, nb, va, vb, s);
        break;
    }
}
