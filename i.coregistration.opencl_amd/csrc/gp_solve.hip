/* SPDX-License-Identifier: Unlicense */

/* RoMa's Gaussian-process solve on the device, in double precision:
 * F = (K + noise I)^-1 F for the n x n cosine kernel K (float) and the
 * n x d position basis F (float). The reference factors and solves on
 * the host (roma.c:770-836 of i.coregistration.opencl: Cholesky, then
 * L Z = F and L^T X = Z, all in double), which costs a 10 MB read-back,
 * a host Cholesky of n = 1600 and a write per tile pair; here the same
 * arithmetic stays on the GPU.
 *
 * Blocked right-looking Cholesky with 64-column panels, the forward solve
 * carried along as extra columns of the right-hand side [F | I]: the
 * identity block makes the forward solve produce Minv = L^-1 beside
 * Y = L^-1 F, so that the backward solve X = Minv^T Y is a sum over the
 * panels of their block rows' products, added as each becomes final,
 * instead of a chain of one launch per panel after the factorisation.
 *  - chol_diag: the 64 x 64 diagonal block factored and its factor
 *    inverted by one work-group (one wave each, in registers), after
 *    applying the previous panel's update to the block itself
 *    (look-ahead); these run back to back on the main stream while
 *    everything else runs on a second stream, joined back at the end;
 *  - on the second stream, one launch per panel for both L21 = A21
 *    Linv^T and Y_b = Linv_b Z_b (Z_b over the right-hand-side columns
 *    that are not yet zero: F and the identity blocks of this panel and
 *    the ones before), one for the trailing update A22 -= L21 L21^T
 *    (lower tiles but the next diagonal block), Z_rest -= L21 Y_b and
 *    X[0 : k + nb] += Minv_b^T Y_F,b (fp64 GEMM tiles, up to three
 *    problems per launch).
 * Synchronisation, inside the kernels: the diagonal kernel of block b
 * sets a flag once its factor and inverse are stored, which panel b's
 * first products on the second stream poll before reading them; and it
 * waits itself for a flag that panel b - 1's first launch on the second
 * stream sets as it starts, after panel b - 2's trailing update. Neither stream then holds
 * a stream wait or an event record between its kernels (each costs 5-7
 * us of command-processor time, on the solve's critical path, and so did a
 * kernel of its own for the flag). Every
 * wait is bounded; one that gives up sets info = -1 and its kernel ends
 * (the caller then runs the solve again with event waits). Under stream
 * capture (a graph has no order between branches that an in-kernel wait
 * could rely on), the two streams wait through stream events instead.
 * Working matrices: A (n x n, the trailing updates), L (n x n, the
 * factor), Linv per panel, Z and Y (n x (d + n)), X (n x d), two flags
 * per panel. No launch reads what another running beside it writes. */

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <math.h>

#include <initializer_list>

#include "common.h"
#include "icoreg_kernels.h"

using namespace icoreg;

typedef double gp_d4 __attribute__((ext_vector_type(4)));

#define GP_NB 64 /* panel width */
#define GP_SB 16 /* columns factored between two updates of their block */
#define DG_T 64  /* GEMM output tile */
#define DG_K 32  /* GEMM reduction chunk */

/* C = alpha A B + beta C with A(i, q) = A[i a_ri + q a_rk], B(q, j) =
 * B[q b_rk + j b_rj], C(i, j) = C[i c_ri + j]; lower: skip output tiles
 * strictly above the diagonal; skip00: leave output tile (0, 0) alone.
 * The matrices have less than 2^31 values: 32-bit indices. */
struct dg_args {
    int M, N, K;
    const double *A;
    int a_ri, a_rk;
    const double *B;
    int b_rk, b_rj;
    double *C;
    int c_ri;
    double alpha;
    int beta, lower;
    int skip00;
};

/* Up to three independent problems per launch: blockIdx.z picks one.
 * wait (when given): a flag the launch's blocks poll (one thread each,
 * device-coherent loads, at most spin_max polls, then an acquire) before
 * they read their operands; a wait that gives up sets *info = -1 and
 * goes on, so that the launch still ends. mark (when given): a flag set
 * as the launch starts, which says that the launches before it on its
 * stream have finished (device-coherent store). */
#define DG_MAXP 3
struct dg_set {
    dg_args p[DG_MAXP];
    const int *wait;
    int spin_max;
    int *info;
    int *mark;
};

/* 64 x 64 outputs a block on v_mfma_f64_16x16x4f64, 32 x 32 a wave. The
 * products are short (64 terms): bound by the round trips of C and of the
 * two chunks, so registers for 3 blocks a CU and 32-bit indices count (64-bit
 * ones took as long as the products). The solve at n = 1600, d = 512 with 4 x
 * 4 outputs a thread on the vector unit 1073 us, so 967, with 3 blocks a CU
 * and no flag kernel 890, with 32-bit indices 883 -> 814. */
__global__ void __launch_bounds__(256, 3) dgemm_kernel(dg_set pr)
{
    __shared__ double As[DG_K][DG_T + 1], Bs[DG_K][DG_T + 1];
    const dg_args &a = pr.p[blockIdx.z];
    const int tid = threadIdx.x, wave = tid >> 6, kq = (tid & 63) >> 4, l16 = tid & 15;
    const int i0 = blockIdx.y * DG_T, j0 = blockIdx.x * DG_T;
    const int wi = 32 * (wave >> 1), wj = 32 * (wave & 1); /* the wave's 32 x 32 */
    gp_d4 acc[2][2], cprev[2][2];

    if (pr.mark && blockIdx.x + blockIdx.y + blockIdx.z == 0 && tid == 0)
        __hip_atomic_store(pr.mark, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (i0 >= a.M || j0 >= a.N || (a.lower && j0 > i0 + DG_T - 1) ||
        (a.skip00 && i0 == 0 && j0 == 0))
        return;
    if (pr.wait) {
        if (tid == 0) {
            int it = 0;

            while (__hip_atomic_load(pr.wait, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0 &&
                   ++it < pr.spin_max)
                __builtin_amdgcn_s_sleep(1);
            if (it >= pr.spin_max)
                __hip_atomic_store(pr.info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    /* The accumulated C is read at the start, so that its latency
     * overlaps the products. */
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = min(i0 + wi + 16 * p + kq + 4 * v, a.M - 1);
                const int j = min(j0 + wj + 16 * r + l16, a.N - 1);

                cprev[p][r][v] = a.beta ? a.C[i * a.c_ri + j] : 0.0;
                acc[p][r][v] = 0.0;
            }
    /* 32 x 64 of A and of B per chunk, 8 values per thread, the
     * unit-stride index fastest across threads. Every load reads a valid
     * address (indices clamped to the last row / column) and the value is
     * selected afterwards, so that the 16 loads are all in flight together;
     * the next chunk's loads are issued before the current chunk's
     * products. */
    double va[8], vb[8];
    bool oka[8], okb[8];

    auto fetch = [&](int k0) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int e = tid + 256 * t;
            const int i = a.a_rk == 1 ? e / DG_K : (e & (DG_T - 1));
            const int q = a.a_rk == 1 ? (e & (DG_K - 1)) : e / DG_T;
            const int j = a.b_rj == 1 ? (e & (DG_T - 1)) : e / DG_K;
            const int qb = a.b_rj == 1 ? e / DG_T : (e & (DG_K - 1));

            oka[t] = i0 + i < a.M && k0 + q < a.K;
            okb[t] = j0 + j < a.N && k0 + qb < a.K;
            va[t] = a.A[min(i0 + i, a.M - 1) * a.a_ri + min(k0 + q, a.K - 1) * a.a_rk];
            vb[t] = a.B[min(k0 + qb, a.K - 1) * a.b_rk + min(j0 + j, a.N - 1) * a.b_rj];
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < a.K; k0 += DG_K) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int e = tid + 256 * t;
            const int i = a.a_rk == 1 ? e / DG_K : (e & (DG_T - 1));
            const int q = a.a_rk == 1 ? (e & (DG_K - 1)) : e / DG_T;
            const int j = a.b_rj == 1 ? (e & (DG_T - 1)) : e / DG_K;
            const int qb = a.b_rj == 1 ? e / DG_T : (e & (DG_K - 1));

            As[q][i] = oka[t] ? va[t] : 0.0;
            Bs[qb][j] = okb[t] ? vb[t] : 0.0;
        }
        __syncthreads();
        if (k0 + DG_K < a.K)
            fetch(k0 + DG_K);
#pragma unroll
        for (int q = 0; q < DG_K; q += 4) {
            double av[2], bv[2];

#pragma unroll
            for (int p = 0; p < 2; p++) {
                av[p] = As[q + kq][wi + 16 * p + l16];
                bv[p] = Bs[q + kq][wj + 16 * p + l16];
            }
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    acc[p][r] =
                        __builtin_amdgcn_mfma_f64_16x16x4f64(av[p], bv[r], acc[p][r], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int i = i0 + wi + 16 * p + kq + 4 * v, j = j0 + wj + 16 * r + l16;

                if (i < a.M && j < a.N)
                    a.C[i * a.c_ri + j] = a.alpha * acc[p][r][v] + cprev[p][r][v];
            }
}

/* ---- the diagonal block ------------------------------------------------------------ */

/* 1 / sqrt(x) from the hardware estimate (within 2^29 ulp: about 2^-23
 * relative) and one Newton step, which squares that error (about 2^-46:
 * some 100 ulp of a double, far below what the float result can show).
 * -0.5 x does not depend on the estimate, so the step adds three
 * dependent operations to the pivot's chain. */
__device__ __forceinline__ double rsqrt_nr(double x)
{
    const double h = -0.5 * x;
    const double r = __builtin_amdgcn_rsq(x);

    return r * fma(h * r, r, 1.5);
}

/* Lane l's value of v, in every lane. */
__device__ __forceinline__ double readlane_d(double v, int l)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);

    return __builtin_bit_cast(
        double, ((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(b >> 32), l) << 32) |
                    (unsigned)__builtin_amdgcn_readlane((int)b, l));
}

/* Polls of a panel flag before the diagonal kernel gives up (with a
 * 64-clock sleep each: about 0.1 s, far beyond any trailing update): the wait
 * then ends with info = -1 instead of hanging. */
#define GP_SPIN_MAX (1 << 22)

/* Cholesky factor of the nb x nb diagonal block at (k, k) of A (n x n)
 * into L, and the inverse of that factor into Linv (nb x nb, row-major,
 * GP_NB apart). info gets 1 + the first column whose pivot is not
 * positive (the factor then holds NaN from there on), or -1 if the wait
 * for ready gave up. 256 threads.
 *  - ready (when given): set once the trailing update this block needs
 *    has finished on the other stream; polled with device-coherent loads,
 *    then an acquire, so the block's reads see that update.
 *  - done (when given): set to 1 after every store of the block, behind
 *    a release, for the panel's products on the other stream.
 *  - Look-ahead (lprev: the previous panel's Linv; its trailing update of
 *    this block is left to this kernel): P = A[k.., k - 64..] lprev^T,
 *    the block's row of that panel's L21, then s -= P P^T on the lower
 *    triangle, in 16 x 16 tiles on v_mfma_f64_16x16x4f64 (lane l gives
 *    A(l % 16, l / 16) and B(l / 16, l % 16) and holds D(l / 16 + 4 v,
 *    l % 16); the fp32 16 x 16 x 4 form holds rows 4 (l / 16) + v
 *    instead). Its operands (the block row of A, lprev) arrive in LDS in
 *    the same round trip as the block itself (all loads before the first
 *    LDS store: 16.5k -> 6.6k cycles); wave w holds the P tiles of rows
 *    16 w .. in registers until every wave has read lprev; P goes through
 *    f; the 10 lower P P^T tiles are dealt to the 4 waves, three chains a
 *    wave at once (14.6k -> 10k cycles for both products).
 *  - The block is then factored 16 columns at a time, without LDS round
 *    trips inside: in wave 0 lane r holds row r of the 16 columns. At
 *    step j every lane reads the 2 x 2 pivot block [p q; q s] of columns
 *    j, j + 1 from their lanes (cross-lane reads), forms 1 / sqrt(p), l21 =
 *    q / sqrt(p) and 1 / sqrt(s - l21^2), then
 *        L[r][j] = a[j] / sqrt(p),
 *        L[r][j + 1] = (a[j + 1] - L[r][j] l21) / sqrt(s - l21^2)
 *    and updates its other columns of the 16 with L[c][j], L[c][j + 1]
 *    read from lane c. The pivots stay in their lanes for one check at the
 *    end (a branch a step costs 300 cycles). Both columns go to LDS (lc,
 *    0 above the pivots). What is right of the 16 columns is updated by
 *    all waves on the matrix instructions.
 *  - Beside wave 0, 16 rows behind, waves 1 .. 3 run the forward
 *    substitution of L X = I in f, 16 columns a wave (wave 0 takes the last
 *    16 after its factor): within 16 rows in registers, below them on the
 *    matrix instructions.
 *  - All threads store factor and inverse in rows.
 * Bound by one wave's dependent chain, about 710 cycles a column pair. A
 * block at n = 1600: 41 us with a whole-row sweep of the 64 columns (an LDS
 * round trip and up to 62 updates a lane each step), 22 us so, of 54k
 * cycles 7k the loads, 10k the look-ahead, 23k the factor, 14k the last rows
 * of the inverse, the stores and the release (clock reads in a copy). */
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
    chol_diag_kernel(const double *__restrict__ A, double *__restrict__ L,
                      double *__restrict__ Linv, int n, int k, int nb,
                      const double *__restrict__ lprev, const int *ready, int spin_max,
                      int *__restrict__ info, int *done)
{
    __shared__ double s[GP_NB][GP_NB + 1], f[GP_NB][GP_NB + 1];
    /* lc[j][r] = L[r][j]: each column contiguous, read with wide LDS
     * loads (every lane the same address). Before the column sweep the
     * same memory holds ar, the look-ahead's block row of A. */
    __shared__ __align__(16) union {
        double lc[GP_NB][GP_NB];
        double ar[GP_NB][GP_NB + 1];
    } u;
    double (*const lc)[GP_NB] = u.lc;
    __shared__ double dinv[GP_NB];
    const int tid = threadIdx.x, lane = tid & 63, kq = lane >> 4, l16 = lane & 15;
    const int uw = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bad = 0;

    if (ready) {
        if (tid == 0) {
            int it = 0;

            while (__hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0 &&
                   ++it < spin_max)
                __builtin_amdgcn_s_sleep(1);
            if (it >= spin_max)
                bad = -1;
        }
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    /* The block's lower triangle; rows and columns past nb are zero with
     * a unit diagonal (their pivots stay 1 and they touch no real row).
     * With a look-ahead, its operands come in the same round trip: the
     * block row A[k.., k - 64..] (rows past nb zero) into ar and the
     * previous panel's inverse factor into f. */
    {
        double v[16], va[16], vl[16];

#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int e = tid + 256 * i, r = e >> 6, c = e & 63;

            v[i] = A[(long long)(k + min(r, nb - 1)) * n + k + min(c, nb - 1)];
        }
        if (lprev)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int e = tid + 256 * i, r = e >> 6, c = e & 63;

                va[i] = A[(long long)(k + min(r, nb - 1)) * n + k - GP_NB + c];
                vl[i] = lprev[e];
            }
        __builtin_amdgcn_sched_barrier(0); /* one round trip, not one a row */
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int e = tid + 256 * i, r = e >> 6, c = e & 63;

            s[r][c] = r < nb && c <= r ? v[i] : r == c ? 1.0 : 0.0;
        }
        if (lprev)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int e = tid + 256 * i, r = e >> 6, c = e & 63;

                u.ar[r][c] = r < nb ? va[i] : 0.0;
                f[r][c] = vl[i];
            }
    }
    __syncthreads();
    if (lprev) {
        gp_d4 pacc[4], acc[3];

        /* P rows 16 wave .., from LDS; lprev is lower triangular, so tile
         * column tc needs k < 16 (tc + 1). */
#pragma unroll
        for (int i = 0; i < 4; i++)
            pacc[i] = (gp_d4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
            const double av = u.ar[16 * uw + l16][4 * kk + kq];

#pragma unroll
            for (int tc = kk / 4; tc < 4; tc++)
                pacc[tc] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    av, f[16 * tc + l16][4 * kk + kq], pacc[tc], 0, 0, 0);
        }
        __syncthreads(); /* every wave is done reading f */
#pragma unroll
        for (int tc = 0; tc < 4; tc++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                f[16 * uw + kq + 4 * v][16 * tc + l16] = pacc[tc][v];
        __syncthreads();
        /* The 10 lower tiles of P P^T, three a wave at once (the last two
         * waves' third is the last tile again, not stored). */
        int tr[3], tc[3];

#pragma unroll
        for (int t = 0; t < 3; t++) {
            const int w = min(uw + 4 * t, 9);

            tr[t] = w >= 6 ? 3 : w >= 3 ? 2 : w >= 1 ? 1 : 0;
            tc[t] = w - tr[t] * (tr[t] + 1) / 2;
            acc[t] = (gp_d4){0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int kk = 0; kk < 16; kk++)
#pragma unroll
            for (int t = 0; t < 3; t++)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[16 * tr[t] + l16][4 * kk + kq],
                                                             f[16 * tc[t] + l16][4 * kk + kq],
                                                             acc[t], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 3; t++) {
            if (uw + 4 * t > 9)
                continue;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = 16 * tr[t] + kq + 4 * v, c = 16 * tc[t] + l16;

                if (r < nb && c <= r)
                    s[r][c] -= acc[t][v];
            }
        }
        __syncthreads();
    }
    /* The inverse begins as the identity, in f. */
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int e = tid + 256 * i;

        f[e >> 6][e & 63] = (e >> 6) == (e & 63) ? 1.0 : 0.0;
    }
    __syncthreads();
    const int nsub = (nb + GP_SB - 1) / GP_SB;

    for (int sp = 0; sp <= nsub; sp++) {
        if (uw == 0 && sp < nsub) {
            /* Columns base .. base + 15: lane r holds its row of them.
             * Pair j, j + 1: the 2 x 2 pivot block [p q; q s] from lanes
             * base + j and base + j + 1, p's root, then the second pivot s
             * - l21^2 and its root. Column j + 1 of a lane is its entry
             * less its column-j value times l21. Columns past nb are
             * padding (unit pivot, zero elsewhere) and change nothing. */
            const int base = GP_SB * sp;
            double a[GP_SB], piv = 1.0, root = 1.0;

#pragma unroll
            for (int c = 0; c < GP_SB; c++)
                a[c] = s[lane][base + c];
#pragma unroll
            for (int j = 0; j < GP_SB; j += 2) {
                const int row = lane - base - j; /* rows below the pivot */
                const double p = readlane_d(a[j], base + j), q = readlane_d(a[j], base + j + 1);
                const double sq = readlane_d(a[j + 1], base + j + 1);
                const double rp = rsqrt_nr(p);
                const double l21 = q * rp;
                const double s2 = fma(-l21, l21, sq);
                const double rs = rsqrt_nr(s2);
                /* The pivots' own lanes hold p and sq: the same products
                 * give their roots. Lanes above hold what nothing reads. */
                const double l0 = a[j] * rp;
                const double l1 = fma(-l0, l21, a[j + 1]) * rs;

                lc[base + j][lane] = row >= 0 ? l0 : 0.0;
                lc[base + j + 1][lane] = row >= 1 ? l1 : 0.0;
                piv = row == 0 ? p : row == 1 ? s2 : piv;
                root = row == 0 ? rp : row == 1 ? rs : root;
#pragma unroll
                for (int c = j + 2; c < GP_SB; c++)
                    a[c] = fma(-l1, readlane_d(l1, base + c),
                               fma(-l0, readlane_d(l0, base + c), a[c]));
            }
            /* Lane base + c has kept pivot c and its reciprocal root. */
            const bool mine = lane >= base && lane < base + GP_SB;
            const unsigned long long neg = __ballot(mine && !(piv > 0.0));

            if (mine)
                dinv[lane] = root;
            if (bad == 0 && neg)
                bad = k + __builtin_ctzll(neg) + 1;
        }
        else if (sp > 0) {
            /* Rows base .. base + 15 of the inverse, 16 columns a wave
             * (wave 0 takes the last ones, when its factor is done): T[j] /=
             * L[j][j], T[c] -= L[c][j] T[j] within the rows (every lane a
             * column, four times over), then the rows below on the matrix
             * instructions. */
            const int base = GP_SB * (sp - 1), ct = uw ? uw - 1 : 3;

            if (ct < sp) {
                const int col = GP_SB * ct + l16;
                double t[GP_SB];

#pragma unroll
                for (int c = 0; c < GP_SB; c++)
                    t[c] = f[base + c][col];
#pragma unroll
                for (int j = 0; j < GP_SB; j++) {
                    t[j] *= dinv[base + j];
#pragma unroll
                    for (int c = j + 1; c < GP_SB; c++)
                        t[c] = fma(-lc[base + j][base + c], t[j], t[c]);
                }
                if (lane < 16)
#pragma unroll
                    for (int c = 0; c < GP_SB; c++)
                        f[base + c][col] = t[c];
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                for (int rt = sp; rt < nsub; rt++) {
                    gp_d4 acc = {0.0, 0.0, 0.0, 0.0};

#pragma unroll
                    for (int kk = 0; kk < 4; kk++)
                        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            lc[base + 4 * kk + kq][GP_SB * rt + l16], f[base + 4 * kk + kq][col],
                            acc, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; v++)
                        f[GP_SB * rt + kq + 4 * v][col] -= acc[v];
                }
            }
        }
        __syncthreads();
        if (sp >= nsub - 1)
            continue;
        /* The block's rest: lower 16 x 16 tiles, dealt to the waves. */
        const int left = nsub - 1 - sp;

        for (int w = uw; w < left * (left + 1) / 2; w += 4) {
            const int tr = w >= 3 ? 2 : w >= 1 ? 1 : 0, tc = w - tr * (tr + 1) / 2;
            const int r0 = GP_SB * (sp + 1 + tr), c0 = GP_SB * (sp + 1 + tc);
            gp_d4 acc = {0.0, 0.0, 0.0, 0.0};

#pragma unroll
            for (int kk = 0; kk < 4; kk++) {
                const double *col = lc[GP_SB * sp + 4 * kk + kq];

                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(col[r0 + l16], col[c0 + l16], acc, 0,
                                                          0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; v++)
                s[r0 + kq + 4 * v][c0 + l16] -= acc[v];
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int e = tid + 256 * i, r = e >> 6, c = e & 63;

        if (r < nb && c < nb)
            Linv[e] = c <= r ? f[r][c] : 0.0;
    }
    __syncthreads();
    if (tid == 0 && bad && *info == 0)
        *info = bad;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int e = tid + 256 * i, r = e >> 6, c = e & 63;

        if (r < nb && c < nb)
            L[(long long)(k + r) * n + k + c] = lc[c][r];
    }
    if (done) {
        /* Every store of the block has reached L2 (the barrier waits for
         * them); the release writes them back for the other XCDs, then
         * the flag. */
        __syncthreads();
        if (tid == 0) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            __hip_atomic_store(done, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

/* A = K + noise I (double), Z = [F | I] (double, rows d + n wide), X = 0
 * (n x d), info and the nflags panel flags cleared. */
__global__ void __launch_bounds__(256)
    gp_init_kernel(const float *__restrict__ K, int n, double noise,
                   double *__restrict__ A, const float *__restrict__ F, int d,
                   double *__restrict__ Z, double *__restrict__ X, int *__restrict__ info,
                   int *__restrict__ flags, int nflags)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long nn = (long long)n * n, w = (long long)d + n, nz = n * w;

    if (idx == 0)
        *info = 0;
    if (idx < nflags)
        flags[idx] = 0;
    if (idx < nn) {
        const int r = (int)(idx / n), c = (int)(idx % n);

        A[idx] = (double)K[idx] + (r == c ? noise : 0.0);
    }
    if (idx < nz) {
        const long long r = idx / w, c = idx % w;

        Z[idx] = c < d ? (double)F[r * d + c] : c - d == r ? 1.0 : 0.0;
    }
    if (idx < (long long)n * d)
        X[idx] = 0.0;
}

__global__ void __launch_bounds__(256)
    gp_store_kernel(const double *__restrict__ X, long long nf, float *__restrict__ F)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;

    if (idx < nf)
        F[idx] = (float)X[idx];
}

static dg_args dg(int M, int N, int K, const double *A, int a_ri, int a_rk, const double *B,
                  int b_rk, int b_rj, double *C, int c_ri, double alpha, int beta, int lower)
{
    dg_args a = {M, N, K, A, a_ri, a_rk, B, b_rk, b_rj, C, c_ri, alpha, beta, lower, 0};

    return a;
}

/* One launch for the problems given (those with no output are skipped);
 * wait, spin_max, info, mark as in dg_set. */
static void dgemm(hipStream_t s, std::initializer_list<const dg_args *> ps,
                  const int *wait = nullptr, int spin_max = 0, int *info = nullptr,
                  int *mark = nullptr)
{
    dg_set pr;
    int np = 0, tx = 0, ty = 0;

    pr.wait = wait;
    pr.spin_max = spin_max;
    pr.info = info;
    pr.mark = mark;

    for (const dg_args *a : ps)
        if (a && a->M > 0 && a->N > 0) {
            if (np == DG_MAXP)
                icoreg_fatal("roma_gp_solve: more than %d products in one launch", DG_MAXP);
            pr.p[np++] = *a;
            tx = max(tx, (a->N + DG_T - 1) / DG_T);
            ty = max(ty, (a->M + DG_T - 1) / DG_T);
        }
    if (np == 0)
        return;
    hipLaunchKernelGGL(dgemm_kernel, dim3((unsigned)tx, (unsigned)ty, (unsigned)np),
                       dim3(256), 0, s, pr);
}

extern "C" size_t roma_gp_work_bytes(int n, int d)
{
    const size_t nblk = (size_t)(n + GP_NB - 1) / GP_NB, w = (size_t)d + n;

    return sizeof(double) * (2 * (size_t)n * n + nblk * GP_NB * GP_NB + 2 * (size_t)n * w +
                             (size_t)n * d) +
           sizeof(int) * 2 * nblk;
}

/* Test hooks (icoreg_gp_test_wait): the in-kernel waits' poll limit and
 * whether the panel flags are set at all (by the panels' first launches
 * and by the diagonal kernels). With the flags never set and a
 * short limit, every waiting kernel gives up at once (info = -1) and
 * still exits, so the give-up path and the caller's recovery can be
 * exercised without a stalled stream. */
static int g_spin_max = GP_SPIN_MAX;
static int g_set_flags = 1;

extern "C" void icoreg_gp_test_wait(int spin_max, int set_flags)
{
    g_spin_max = spin_max > 0 ? spin_max : GP_SPIN_MAX;
    g_set_flags = set_flags != 0;
}

/* events: the diagonal kernels wait through stream events (the form a
 * capture needs, and the fallback when the in-kernel wait gave up). */
static void gp_solve_run(struct ops *o, cl_mem K, int n, float noise, cl_mem F, int d,
                         cl_mem work, cl_mem info, bool events, const char *op)
{
    hipStream_t s;
    double *A, *L, *Li, *Z, *Y, *X;
    int *flags;
    const int nblk = (n + GP_NB - 1) / GP_NB;
    const long long nd = (long long)n * d;

    if (n < 1 || d < 1 || n > 46340)
        icoreg_fatal("%s: invalid sizes n=%d d=%d", op, n, d);
    count32((long long)n * n, op);
    count32((long long)n * ((long long)d + n), op);
    const int w = d + n;

    need_floats(K, 0, (long long)n * n, op, "K");
    need_floats(F, 0, nd, op, "F");
    need_bytes(work, 0, (long long)roma_gp_work_bytes(n, d), op, "work");
    need_bytes(info, 0, (long long)sizeof(int), op, "info");
    s = stream_of(o->ocl);
    A = (double *)work->ptr;
    L = A + (long long)n * n;
    Li = L + (long long)n * n;
    Z = Li + (long long)nblk * GP_NB * GP_NB;
    Y = Z + n * w;
    X = Y + n * w;
    flags = (int *)(X + nd);
    {
        prof_scope ps(o->ocl, op);
        const long long nn = (long long)n * n, nz = (long long)n * w;
        const long long tot = nn > nz ? nn : nz;
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;

        hip_check(hipStreamIsCapturing(s, &cs), "hipStreamIsCapturing");
        const bool capture = events || cs != hipStreamCaptureStatusNone;
        const int spin_max = g_spin_max;

        hipLaunchKernelGGL(gp_init_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s,
                           cfptr(K), n, (double)noise, A, cfptr(F), d, Z, X, (int *)info->ptr,
                           flags, 2 * nblk);
        /* The diagonal blocks on the main stream s, everything else of a
         * panel on the second stream s2: diagonal block b waits for the
         * trailing update of panel b - 2 (which has the whole of block
         * b - 1's factorisation to finish) and applies panel b - 1's
         * update to its own block itself; panel b's products wait for
         * block b. Y = L^-1 [F | I] alongside, over the columns that are
         * not yet zero (F and the identity blocks up to this panel's).
         * flags[b]: panel b's trailing update done (set on s2);
         * dflags[b]: block b factored (set by its diagonal kernel). */
        hipStream_t s2 = aux_stream_of(o->ocl);
        int *const dflags = flags + nblk;

        hip_check(hipEventRecord(aux_event(o->ocl, 2 * nblk), s), "hipEventRecord");
        hip_check(hipStreamWaitEvent(s2, aux_event(o->ocl, 2 * nblk), 0), "hipStreamWaitEvent");
        for (int b = 0; b < nblk; b++) {
            const int k = b * GP_NB, nb = n - k < GP_NB ? n - k : GP_NB;
            const int rest = n - k - nb, wb = d + k + nb;
            double *Lk = Li + (long long)b * GP_NB * GP_NB;
            double *L21 = L + (long long)(k + nb) * n + k;
            const double *lprev = b ? (const double *)(Lk - GP_NB * GP_NB) : nullptr;
            int *info_p = (int *)info->ptr;
            const hipEvent_t done_b = aux_event(o->ocl, 2 * b);

            if (capture) {
                if (b >= 2)
                    hip_check(hipStreamWaitEvent(s, aux_event(o->ocl, 2 * (b - 2) + 1), 0),
                              "hipStreamWaitEvent");
                hipLaunchKernelGGL(chol_diag_kernel, dim3(1), dim3(256), 0, s, A,
                                   L, Lk, n, k, nb, lprev, (const int *)nullptr, spin_max,
                                   info_p, (int *)nullptr);
                hip_check(hipEventRecord(done_b, s), "hipEventRecord");
                hip_check(hipStreamWaitEvent(s2, done_b, 0), "hipStreamWaitEvent");
            }
            else
                /* Panel b's first products wait for dflags[b] inside their
                 * kernel: no stream wait (5-6 us of command-processor
                 * time a panel on s2) and no completion event. */
                hipLaunchKernelGGL(chol_diag_kernel, dim3(1), dim3(256), 0, s, A, L, Lk, n, k,
                                   nb, lprev, b >= 2 ? (const int *)flags + b - 2 : nullptr,
                                   spin_max, info_p, g_set_flags ? dflags + b : nullptr);
            /* L21 = A21 Linv^T and Y_b = Linv_b Z_b. */
            const dg_args panel = dg(rest, nb, nb, A + (long long)(k + nb) * n + k, n, 1,
                                     Lk, 1, GP_NB, L21, n, 1.0, 0, 0);
            const dg_args yb = dg(nb, wb, nb, Lk, GP_NB, 1, Z + k * w, w, 1, Y + k * w, w,
                                  1.0, 0, 0);
            if (capture)
                dgemm(s2, {&yb, &panel});
            else
                dgemm(s2, {&yb, &panel}, dflags + b, spin_max, info_p,
                      b > 0 && g_set_flags ? flags + b - 1 : nullptr);
            /* X[0 : k + nb] += Minv_b^T Y_F,b: this panel's block row of
             * Minv = L^-1 (Y[k.., d..], zero right of its own identity
             * block) is final once Y_b is. */
            dg_args xacc = dg(k + nb, d, nb, Y + k * w + d, 1, w, Y + k * w, w, 1, X, d, 1.0, 1,
                              0);
            if (rest > 0) {
                /* A22 -= L21 L21^T (lower tiles but the next diagonal block,
                 * which its own kernel updates) and Z_rest -= L21 Y_b. */
                dg_args trail = dg(rest, rest, nb, L21, n, 1, L21, 1, n,
                                   A + (long long)(k + nb) * n + k + nb, n, -1.0, 1, 1);
                const dg_args zr = dg(rest, wb, nb, L21, n, 1, Y + k * w, w, 1,
                                      Z + (k + nb) * w, w, -1.0, 1, 0);

                trail.skip00 = 1;
                dgemm(s2, {&trail, &zr, &xacc});
            }
            else
                dgemm(s2, {&xacc});
            if (capture || b == nblk - 1)
                hip_check(hipEventRecord(aux_event(o->ocl, 2 * b + 1), s2), "hipEventRecord");
        }
        hip_check(hipStreamWaitEvent(s, aux_event(o->ocl, 2 * (nblk - 1) + 1), 0),
                  "hipStreamWaitEvent");
        hipLaunchKernelGGL(gp_store_kernel, dim3((unsigned)((nd + 255) / 256)), dim3(256), 0, s,
                           (const double *)X, nd, fptr(F));
    }
    launch_check(op);
}

extern "C" void roma_gp_solve(struct ops *o, cl_mem K, int n, float noise,
                              cl_mem F, int d, cl_mem work, cl_mem info)
{
    ICOREG_API_BEGIN
    gp_solve_run(o, K, n, noise, F, d, work, info, false, "roma_gp_solve");
    ICOREG_API_END
}

extern "C" void roma_gp_solve_events(struct ops *o, cl_mem K, int n, float noise,
                                     cl_mem F, int d, cl_mem work, cl_mem info)
{
    ICOREG_API_BEGIN
    gp_solve_run(o, K, n, noise, F, d, work, info, true, "roma_gp_solve_events");
    ICOREG_API_END
}
