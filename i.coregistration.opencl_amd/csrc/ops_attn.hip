/* SPDX-License-Identifier: Unlicense */

/* Blockwise scaled dot-product attention on the matrix cores:
 * O = softmax(scale Q K^T) V per head, never storing the scores. The
 * contract is the reference's attention kernel (ops.cl:604-687,
 * ops.c:444-474 of i.coregistration.opencl): token-major operands with
 * head h at columns h * d, d <= 128, optional key mask, a query with no
 * key left gets zeros.
 *
 * A block holds 4 waves of 32 queries each (128 queries of one head)
 * and streams its range of keys in tiles of 32 through double-buffered
 * LDS, shared by the 4 waves, one barrier per tile; with 16-byte
 * aligned rows the next tile is read into registers a tile ahead (the
 * fp32 block, att_block_f32; attention_split_kernel does the same on the
 * bf16 instructions, without loss, and is what 1 .. 64 and 97 .. 128
 * channels a head run on):
 *  - the scores are computed transposed, S^T = K Q^T, with
 *    v_mfma_f32_32x32x2f32 (A = K from LDS, B = the wave's queries,
 *    pre-scaled and held in registers for the whole kernel), so that
 *    each lane holds 16 keys of one query (its column);
 *  - the online softmax runs per lane on those registers, the two lane
 *    halves of a query combined with one cross-lane exchange; scores are
 *    kept in base 2 (log2 e folded into the query scale, one v_exp_f32
 *    per probability) and the running maximum is raised lazily, only
 *    when a tile exceeds it by 2^8, so the accumulator rescale is rare;
 *  - the output is accumulated transposed, O^T += V^T P^T, with the
 *    probabilities fed to the MFMA straight from the score registers:
 *    MFMA step r pairs, for lane half h, key (r / 4) * 8 + h * 4 + r % 4,
 *    which is where the score MFMA left it, and reads the matching V
 *    rows from LDS. No transpose of P through LDS.
 * When queries x heads give too few waves to fill the chip (ELoFTR's 400
 * tokens, the ViT's 1601 tokens per head), the keys are split into
 * ranges over grid z and a second kernel merges the partial results by
 * their running maxima and sums, as flash-decoding does. */

#include <hip/hip_runtime.h>

#include <mutex>

#include <math.h>

#include "common.h"
#include "ops.h"
#include "split.h"

using namespace icoreg;

typedef float floatx16 __attribute__((ext_vector_type(16)));

#define ATT_KT 32 /* keys per tile */
#define ATT_NW 4  /* waves per block, 32 queries each */
#define ATT_TAU 8.0f /* lazy rescaling threshold, base-2 units */
#define ATT_QUP 0x1p32f /* scale of the queries split into bf16 parts */
#define ATT_PF 2     /* LDS operand reads ahead of their MFMA */

/* Registers <- the key tile from key k0 (zeros past Nk and d), 16-byte
 * loads, consecutive threads along a key row. */
template <int NL, int DP>
__device__ __forceinline__ void att_fetch(float4 (&kr)[NL], float4 (&vr)[NL],
                                          const float *K, int ldk,
                                          const float *V, int ldv, int k0,
                                          int Nk, int d, int tid)
{
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int e = tid + 64 * ATT_NW * i, key = e / (DP / 4);
        const int dd = (e - key * (DP / 4)) * 4, kk = k0 + key;
        const bool ok = kk < Nk && dd < d;
        /* Always load from a valid address (the last key / last four
         * columns) and select per component: a select between whole
         * vectors or pointers is lowered through scratch memory. Nk >= 1
         * and d >= 4 here. */
        const long long kc = min(kk, Nk - 1), dc = min(dd, d - 4);
        const float4 a = *(const float4 *)(K + kc * ldk + dc);
        const float4 b = *(const float4 *)(V + kc * ldv + dc);

        kr[i].x = ok ? a.x : 0.0f;
        kr[i].y = ok ? a.y : 0.0f;
        kr[i].z = ok ? a.z : 0.0f;
        kr[i].w = ok ? a.w : 0.0f;
        vr[i].x = ok ? b.x : 0.0f;
        vr[i].y = ok ? b.y : 0.0f;
        vr[i].z = ok ? b.z : 0.0f;
        vr[i].w = ok ? b.w : 0.0f;
    }
}

/* Tile t of keys into LDS buffers ks / vs from the registers of a VEC
 * fetch (K stored with an odd row pitch, V with 16-byte rows). */
template <int NL, int DP, int KP, int VP>
__device__ __forceinline__ void att_stash(const float4 (&kr)[NL],
                                          const float4 (&vr)[NL], float *ks,
                                          float *vs, int tid)
{
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int e = tid + 64 * ATT_NW * i, key = e / (DP / 4);
        const int dd = (e - key * (DP / 4)) * 4;
        float *kd = ks + key * KP + dd;

        kd[0] = kr[i].x;
        kd[1] = kr[i].y;
        kd[2] = kr[i].z;
        kd[3] = kr[i].w;
        *(float4 *)(vs + key * VP + dd) = vr[i];
    }
}

/* The same straight from global memory, one float per thread and load
 * (rows not 16-byte aligned). */
template <int NL, int DP, int KP, int VP>
__device__ __forceinline__ void att_stash_direct(const float *K, int ldk,
                                                 const float *V, int ldv,
                                                 int k0, int Nk, int d,
                                                 float *ks, float *vs, int tid)
{
    for (int i = 0; i < NL; i++) {
        const int e = tid + 64 * ATT_NW * i, key = e / DP;
        const int dd = e - key * DP, kk = k0 + key;
        const bool ok = kk < Nk && dd < d;

        ks[key * KP + dd] = ok ? K[(long long)kk * ldk + dd] : 0.0f;
        vs[key * VP + dd] = ok ? V[(long long)kk * ldv + dd] : 0.0f;
    }
}

/* Arguments of the attention kernels (one image's operands; images bq .. bo
 * floats apart). */
struct att_args {
    const float *Q, *K, *V;
    float *O;
    const unsigned char *kmask;
    float *part_o;
    float2 *part_ml;
    int ldq, ldk, ldv, ldo, Nq, Nk, d, nh, tiles_per_split;
    float scale;
    long long bq, bk, bv, bo;
};

/* One block: 128 queries (4 waves x 32) of one head against the key
 * tiles [t0, t1) of 32 keys. K and V tiles are double-buffered in LDS
 * and shared by the 4 waves: the next tile (fetched into registers one
 * tile earlier) is written to the other buffer between the score and
 * the output MFMAs, so one barrier per tile suffices. With nsplit > 1
 * (blockIdx.z picks the key range) the unnormalised output and the
 * running (max, sum) go to part_o / part_ml for attn_merge_kernel; with
 * one split the normalised output goes to O directly. MASK: a key mask
 * is given. */
template <int ND, bool VEC, bool MASK>
__device__ __forceinline__ void att_block_f32(const att_args &a, float *lds, int bx, int by,
                                              int bz, int ny)
{
    const float *__restrict__ Q = a.Q, *__restrict__ K = a.K, *__restrict__ V = a.V;
    float *__restrict__ O = a.O, *__restrict__ part_o = a.part_o;
    float2 *__restrict__ part_ml = a.part_ml;
    const unsigned char *__restrict__ kmask = a.kmask;
    const int ldq = a.ldq, ldk = a.ldk, ldv = a.ldv, ldo = a.ldo;
    const int Nq = a.Nq, Nk = a.Nk, d = a.d, nh = a.nh, tiles_per_split = a.tiles_per_split;
    const float scale = a.scale;
    const long long bq = a.bq, bk = a.bk, bv = a.bv, bo = a.bo;
    constexpr int DP = 32 * ND;     /* padded head dimension */
    constexpr int KP = DP + 1;      /* K tile row pitch (odd: no conflicts) */
    constexpr int VP = DP + 4;      /* V tile row pitch */
    constexpr int NS = DP / 2;      /* score MFMA steps */
    constexpr int NL = VEC ? ATT_KT * DP / 4 / (64 * ATT_NW)
                           : ATT_KT * DP / (64 * ATT_NW); /* loads / thread */
    /* K tiles, then V tiles (16-byte rows). */
    float *const Vs_ = lds, *const Ks_ = lds + 2 * ATT_KT * VP;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = by % nh, bi = by / nh;
    const int half = lane >> 5, col = lane & 31;
    const int qi = (bx * ATT_NW + wave) * 32 + col;
    const int ntiles = (Nk + ATT_KT - 1) / ATT_KT;
    const int t0 = bz * tiles_per_split;
    const int t1 = min(ntiles, t0 + tiles_per_split);
    float q[NS];
    floatx16 o[ND];
    float m = -INFINITY, l = 0.0f;
    float4 kr4[VEC ? NL : 1], vr4[VEC ? NL : 1];

    /* Scores in the base-2 domain: softmax(x) = 2^(x log2 e - max) / sum,
     * so log2 e is folded into the query scale and every exponential is
     * one v_exp_f32. */
    const float qscale = scale * 1.4426950408889634f;

    Q += bi * bq + (long long)h * d;
    K += bi * bk + (long long)h * d;
    V += bi * bv + (long long)h * d;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int dd = 2 * s + half;

        q[s] = (qi < Nq && dd < d) ? Q[(long long)qi * ldq + dd] * qscale
                                   : 0.0f;
    }
#pragma unroll
    for (int t = 0; t < ND; t++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            o[t][r] = 0.0f;

    if (t0 < t1) {
        if constexpr (VEC) {
            att_fetch<NL, DP>(kr4, vr4, K, ldk, V, ldv, t0 * ATT_KT, Nk, d,
                              tid);
            att_stash<NL, DP, KP, VP>(kr4, vr4, Ks_, Vs_, tid);
            if (t0 + 1 < t1)
                att_fetch<NL, DP>(kr4, vr4, K, ldk, V, ldv,
                                  (t0 + 1) * ATT_KT, Nk, d, tid);
        }
        else {
            att_stash_direct<NL, DP, KP, VP>(K, ldk, V, ldv, t0 * ATT_KT, Nk,
                                             d, Ks_, Vs_, tid);
        }
    }
    __syncthreads();
    for (int t = t0; t < t1; t++) {
        const int k0 = t * ATT_KT, cur = (t - t0) & 1;
        const float *ks = Ks_ + cur * (ATT_KT * KP), *vs = Vs_ + cur * (ATT_KT * VP);
        floatx16 s;

#pragma unroll
        for (int r = 0; r < 16; r++)
            s[r] = 0.0f;
        {
            /* K operands read ATT_PF steps ahead of their MFMA; the
             * scheduling barriers keep the reads there. */
            const float *kb = ks + col * KP + half;
            float kv[ATT_PF + 1];

#pragma unroll
            for (int st = 0; st < ATT_PF; st++)
                kv[st] = kb[2 * st];
#pragma unroll
            for (int st = 0; st < NS; st++) {
                if (st + ATT_PF < NS)
                    kv[(st + ATT_PF) % (ATT_PF + 1)] = kb[2 * (st + ATT_PF)];
                __builtin_amdgcn_sched_barrier(0);
                s = __builtin_amdgcn_mfma_f32_32x32x2f32(
                    kv[st % (ATT_PF + 1)], q[st], s, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }

        /* Scores out of the accumulator into plain registers; keys past
         * Nk (last tile only) or masked out become -inf by a select on a
         * flag computed first (no conditional writes into the accumulator
         * vector). */
        float p[16];
        float mx = -INFINITY;

        if (MASK || k0 + ATT_KT > Nk) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int kk = k0 + (r >> 2) * 8 + half * 4 + (r & 3);
                bool keep = kk < Nk;

                if (MASK)
                    keep = keep && kmask[min(kk, Nk - 1)] != 0;
                p[r] = keep ? s[r] : -INFINITY;
                mx = fmaxf(mx, p[r]);
            }
        }
        else {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                p[r] = s[r];
                mx = fmaxf(mx, p[r]);
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        {
            /* Lazy rescaling: the reference maximum m moves only when a
             * tile's maximum exceeds it by more than ATT_TAU (so the
             * probabilities stay below 2^ATT_TAU), and the accumulated
             * output and sum are rescaled only then, by a wave-uniform
             * branch. Output and sum always share the same m, so the
             * normalised result is the same. */
            const bool need = mx > m + ATT_TAU;
            float sum = 0.0f;

            if (__any(need)) {
                const float mn = need ? mx : m;
                const float corr =
                    need ? (m == -INFINITY ? 0.0f
                                           : __builtin_amdgcn_exp2f(m - mn))
                         : 1.0f;

                m = mn;
                l *= corr;
#pragma unroll
                for (int tt = 0; tt < ND; tt++)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        o[tt][r] *= corr;
            }
            if (m == -INFINITY) {
#pragma unroll
                for (int r = 0; r < 16; r++)
                    p[r] = 0.0f;
            }
            else {
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    p[r] = __builtin_amdgcn_exp2f(p[r] - m);
                    sum += p[r];
                }
            }
            sum += __shfl_xor(sum, 32, 64);
            l += sum;
        }

        /* The next tile into the other buffer (last read one tile ago,
         * before the previous barrier), then its successor's loads. */
        if (t + 1 < t1) {
            if constexpr (VEC) {
                att_stash<NL, DP, KP, VP>(kr4, vr4, Ks_ + (cur ^ 1) * (ATT_KT * KP),
                                          Vs_ + (cur ^ 1) * (ATT_KT * VP), tid);
                if (t + 2 < t1)
                    att_fetch<NL, DP>(kr4, vr4, K, ldk, V, ldv,
                                      (t + 2) * ATT_KT, Nk, d, tid);
            }
            else {
                att_stash_direct<NL, DP, KP, VP>(K, ldk, V, ldv,
                                                 (t + 1) * ATT_KT, Nk, d,
                                                 Ks_ + (cur ^ 1) * (ATT_KT * KP),
                                                 Vs_ + (cur ^ 1) * (ATT_KT * VP), tid);
            }
        }

        {
            /* V operands of step r (key (r / 4) * 8 + half * 4 + r % 4)
             * read ATT_PF steps ahead, as for K. */
            const float *vb = vs + half * 4 * VP + col;
            float vv[ATT_PF + 1][ND];
            auto vread = [&](int r, float *v) {
#pragma unroll
                for (int tt = 0; tt < ND; tt++)
                    v[tt] = vb[((r >> 2) * 8 + (r & 3)) * VP + tt * 32];
            };

#pragma unroll
            for (int r = 0; r < ATT_PF; r++)
                vread(r, vv[r]);
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (r + ATT_PF < 16)
                    vread(r + ATT_PF, vv[(r + ATT_PF) % (ATT_PF + 1)]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int tt = 0; tt < ND; tt++)
                    o[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                        vv[r % (ATT_PF + 1)][tt], p[r], o[tt], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __syncthreads();
    }

    if (qi >= Nq)
        return;
    if (!part_o) {
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        float *out = O + bi * bo + (long long)qi * ldo + (long long)h * d;

#pragma unroll
        for (int tt = 0; tt < ND; tt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dd = tt * 32 + (r >> 2) * 8 + half * 4 + (r & 3);

                if (dd < d)
                    out[dd] = l > 0.0f ? o[tt][r] * inv : 0.0f;
            }
    }
    else {
        const long long row =
            ((long long)bz * ny + by) * Nq + qi;
        float *out = part_o + row * DP;

#pragma unroll
        for (int tt = 0; tt < ND; tt++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                out[tt * 32 + (r >> 2) * 8 + half * 4 + (r & 3)] = o[tt][r];
        if (half == 0)
            part_ml[row] = make_float2(m, l);
    }
}

/* Floats of LDS of att_block_f32: both operands' double-buffered tiles. */
template <int ND> constexpr int att_f32_lds = 2 * ATT_KT * (2 * 32 * ND + 5);

/* The block on the fp32 instructions (65 .. 96 channels a head). */
template <int ND, bool VEC, bool MASK>
__global__ void __launch_bounds__(64 * ATT_NW) attention_kernel(const att_args a)
{
    __shared__ __align__(16) float lds[att_f32_lds<ND>];

    att_block_f32<ND, VEC, MASK>(a, lds, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.y);
}

/* The same block on the bf16 instructions: queries, keys, values and
 * probabilities split exactly into three bf16 parts, six products each
 * (split.h). K tiles lie in LDS as [part][key][channels] and V tiles
 * transposed, [part][channel][keys], the keys of a row in the order in which
 * the score product leaves them in the lanes: slot j of lane half h of step u
 * is key 16 u + 8 (j / 4) + 4 h + j % 4, so the split probabilities are the
 * second product's operands as they stand. 16-byte chunks are stored XORed
 * with row bits, 16 rows to 64 banks. A score's 5 small products per 16
 * channels are summed before the large ones. The output's small products
 * have accumulators of their own: one by one onto a sum over all keys they
 * round away, all one way where the values have one sign (mean shift at 4000
 * keys -1.1e-8, so 3e-9; rms error at 128 keys, 32 channels 1.46e-7 against
 * the fp32 block's 1.05e-7, so 0.9e-7). With 64 channels these accumulators
 * would spill (160 us for 2 x 16 heads, 1601 tokens); there the small products
 * of 16 keys are summed apart and added once (155 us; of 32 keys 157; 147 with
 * no sums apart). With 128, adding so took 124 us for 8 heads, 1600 tokens,
 * accumulators 110 (101 with no sums apart).
 *
 * Per 32 keys, 32 queries and 64 channels 48 products (1536 cycles) run
 * beside 16 exponentials and 32 splits a lane (about 1200 cycles of vector
 * instructions): bound by those, by the loads' latency and by the two units
 * overlapping only between the 3 blocks that the registers hold. Measured on
 * one MI355X with the merge, against the fp32 block: 2 x 16 heads of 64, 1601
 * tokens 230 -> 169 us (on another 224 -> 155, 136 TFLOP/s); 16 heads of 64,
 * 785 tokens 59 -> 45; 2 x 8 heads of 32, 400 tokens 19.4 -> 17.2; 2 x 16 heads
 * of 32, 1601 tokens 147 -> 99; 8 heads of 128, 1600 tokens 167 -> 109; 2 x 16
 * heads of 128, 2304 tokens 937 -> 654; 4 heads of 64, 49 tokens 12.8 -> 12.4.
 * Tried, before the sums apart: the next tile's scores beside this one's
 * softmax in one wave, 2 blocks a CU (64 channels 147 -> 155, 128 channels 596
 * -> 604). Error against 64 bits two fifths of the fp32 block's on the first
 * shape (3.3e-7, 8.4e-7: its 64 terms round each time). The order of the
 * blocks and loads without a range check per value (rows past the keys read
 * the last key again) gave 188 -> 147 before the sums apart. 65 .. 96
 * channels stay on the fp32 block: rows of 12 chunks would not spread over the
 * banks this way.
 *
 * Values and probabilities are scaled as split.h says. Queries are scaled by
 * ATT_QUP and keys not: scores need absolute precision, and a query of 2^95
 * and above (after the softmax scale) is no longer finite, so what keys under
 * 2^-110 lose, at most 2^-134 each, moves a score by at most d 2^-38. The
 * scale leaves the scores in the exponential's multiply-add.
 *
 * If a sum is not finite (an infinity or NaN among the operands has no
 * split), the block runs again on the fp32 instructions. */
template <int ND, bool VEC, bool MASK>
__global__ void __launch_bounds__(64 * ATT_NW, ND == 4 ? 1 : 3)
    attention_split_kernel(const att_args a)
{
    constexpr int DP = 32 * ND, CH = DP / 8;  /* chunks of a K row */
    constexpr int RW = 16 / CH < 1 ? 1 : 16 / CH; /* K rows in 256 bytes */
    constexpr int PK = ATT_KT * CH;           /* chunks of a part: K and V alike */
    constexpr int NT = 64 * ATT_NW, NL = (PK + NT - 1) / NT;
    constexpr int LDSF = 2 * 6 * PK * 4;
    __shared__ split_u4 lds[(LDSF > att_f32_lds<ND> ? LDSF : att_f32_lds<ND>) / 4 + 1];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    /* Blocks are dealt to the 8 XCDs in turn: XCD x takes the x-th band of
     * the order (image and head, key range, queries), so that a head's K and
     * V stay in one L2. */
    const int nx = gridDim.x, ny = gridDim.y, T = nx * ny * gridDim.z;
    const int id = (blockIdx.z * ny + blockIdx.y) * nx + blockIdx.x;
    const int unit = (id & 7) * (T >> 3) + min(id & 7, T & 7) + (id >> 3);
    const int bx = unit % nx, bz = unit / nx % gridDim.z;
    const int by = unit / (nx * gridDim.z), h = by % a.nh, bi = by / a.nh;
    const int half = lane >> 5, col = lane & 31, d = a.d, Nk = a.Nk;
    const int qi = (bx * ATT_NW + wave) * 32 + col;
    const int ntiles = (Nk + ATT_KT - 1) / ATT_KT;
    const int t0 = bz * a.tiles_per_split, t1 = min(ntiles, t0 + a.tiles_per_split);
    const float *Q = a.Q + bi * a.bq + (long long)h * d;
    const float *K = a.K + bi * a.bk + (long long)h * d;
    const float *V = a.V + bi * a.bv + (long long)h * d;
    /* Threads past the chunks (32 channels a head): none in K, all in V. */
    constexpr bool APART = PK < NT;
    const bool has_k = !APART || tid < PK;
    const int vt = APART ? tid - PK : tid;
    float kr[NL][8], vr[NL][8];
    split_u4 q[2 * ND][3];
    /* The output's small products: of all keys (LOW), or of 16 at a time
     * where 16 registers a 32 channels more would spill. */
    constexpr bool LOW = ND != 2;
    floatx16 o[ND], low[LOW ? ND : 1];
    float m = -INFINITY, l = 0.0f;
    bool kept = !MASK && t0 < t1;

#pragma unroll
    for (int st = 0; st < 2 * ND; st++) {
        float x[8];

#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int dd = st * 16 + half * 8 + j;

            x[j] = qi < a.Nq && dd < d
                       ? Q[(long long)qi * a.ldq + dd] *
                             (a.scale * 1.4426950408889634f * ATT_QUP)
                       : 0.0f;
        }
        split8(x, 1.0f, q[st][0], q[st][1], q[st][2]);
    }
#pragma unroll
    for (int t = 0; t < ND; t++)
#pragma unroll
        for (int r = 0; r < 16; r++)
            o[t][r] = low[LOW ? t : 0][r] = 0.0f;

    /* Tile k0 into registers: K chunk e is key e / CH, channels 8 (e % CH)
     * ..; V chunk e channel e % DP, slots 8 (e / DP) .. + 7 (keys that a
     * wave's lanes share). Past Nk and d the last key and the last channels
     * are read again: the queries' channels there are 0, such keys get no
     * probability and such output channels are not stored. */
    auto fetch = [&](int k0) {
        const float *kt = K + (long long)k0 * a.ldk;
        const int last = Nk - 1 - k0;

        if (has_k) {
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const int e = tid + NT * i, dd = e % CH * 8;
                const float *p = kt + (long long)min(e / CH, last) * a.ldk;

                if (VEC) {
                    const float4 x = *(const float4 *)(p + min(dd, d - 4));
                    const float4 y = *(const float4 *)(p + min(dd + 4, d - 4));

                    kr[i][0] = x.x, kr[i][1] = x.y, kr[i][2] = x.z, kr[i][3] = x.w;
                    kr[i][4] = y.x, kr[i][5] = y.y, kr[i][6] = y.z, kr[i][7] = y.w;
                }
                else {
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        kr[i][j] = p[min(dd + j, d - 1)];
                }
            }
        }
        if (!APART || !has_k) {
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const int e = vt + NT * i;
                const unsigned dd = min(e % DP, d - 1);
                const int c = ND == 1 ? e / DP : __builtin_amdgcn_readfirstlane(e / DP);

#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int kk = (c >> 1) * 16 + (j >> 2) * 8 + (c & 1) * 4 + (j & 3);

                    vr[i][j] = (V + (long long)(k0 + min(kk, last)) * a.ldv)[dd];
                }
            }
        }
    };
    auto stash = [&](split_u4 *ks) {
        split_u4 *vs = ks + 3 * PK, x, y, z;

        if (has_k) {
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const int e = tid + NT * i, key = e / CH;
                const int at = key * CH + ((e % CH) ^ (key / RW % CH));

                split8(kr[i], 1.0f, x, y, z);
                ks[at] = x;
                ks[PK + at] = y;
                ks[2 * PK + at] = z;
            }
        }
        if (!APART || !has_k) {
#pragma unroll
            for (int i = 0; i < NL; i++) {
                const int e = vt + NT * i, dd = e % DP;
                const int at = dd * 4 + ((e / DP) ^ (dd >> 2 & 3));

                split8(vr[i], SPLIT_UP, x, y, z);
                vs[at] = x;
                vs[PK + at] = y;
                vs[2 * PK + at] = z;
            }
        }
    };
    constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};

    if (t0 < t1) {
        fetch(t0 * ATT_KT);
        stash(lds);
        if (t0 + 1 < t1)
            fetch((t0 + 1) * ATT_KT);
    }
    __syncthreads();
    for (int t = t0; t < t1; t++) {
        const int k0 = t * ATT_KT, cur = (t - t0) & 1;
        const split_u4 *ks = lds + cur * (6 * PK), *vs = ks + 3 * PK;
        auto key = [&](int p, int st) {
            return __builtin_bit_cast(
                split_b8, ks[p * PK + col * CH + ((2 * st + half) ^ (col / RW % CH))]);
        };
        floatx16 s;

#pragma unroll
        for (int r = 0; r < 16; r++)
            s[r] = 0.0f;
#pragma unroll
        for (int st = 0; st < 2 * ND; st++) {
            const split_b8 kf[3] = {key(0, st), key(1, st), key(2, st)};

#pragma unroll
            for (int w = 0; w < 5; w++)
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    kf[pa[w]], __builtin_bit_cast(split_b8, q[st][pb[w]]), s, 0, 0, 0);
        }
#pragma unroll
        for (int st = 0; st < 2 * ND; st++)
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                key(0, st), __builtin_bit_cast(split_b8, q[st][0]), s, 0, 0, 0);

        /* Online softmax as in att_block_f32. */
        float p[16], mx = -INFINITY, sum = 0.0f;

        if (MASK || k0 + ATT_KT > Nk) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int kk = k0 + (r >> 2) * 8 + half * 4 + (r & 3);
                bool keep = kk < Nk;

                if (MASK)
                    keep = keep && a.kmask[min(kk, Nk - 1)] != 0;
                kept = kept || keep;
                p[r] = keep ? s[r] : -INFINITY;
                mx = fmaxf(mx, p[r]);
            }
        }
        else {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                p[r] = s[r];
                mx = fmaxf(mx, p[r]);
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * (1.0f / ATT_QUP);
        const bool need = mx > m + ATT_TAU;

        if (__any(need)) {
            const float mn = need ? mx : m;
            const float corr =
                need ? (m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mn)) : 1.0f;

            m = mn;
            l *= corr;
#pragma unroll
            for (int tt = 0; tt < ND; tt++)
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    o[tt][r] *= corr;
                    if (LOW)
                        low[LOW ? tt : 0][r] *= corr;
                }
        }
        {
            /* No key kept yet: every score is -infinity, 2^-infinity = 0. */
            const float ref = m == -INFINITY ? 0.0f : m;

#pragma unroll
            for (int r = 0; r < 16; r++) {
                p[r] = __builtin_amdgcn_exp2f(fmaf(p[r], 1.0f / ATT_QUP, -ref));
                sum += p[r];
            }
        }
        l += sum + __shfl_xor(sum, 32, 64);

        /* The next tile into the other buffer (last read one tile ago,
         * before the previous barrier), then its successor's loads. */
        if (t + 1 < t1) {
            stash(lds + (cur ^ 1) * (6 * PK));
            if (t + 2 < t1)
                fetch((t + 2) * ATT_KT);
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            float x[8];
            split_u4 pp[3];

#pragma unroll
            for (int j = 0; j < 8; j++)
                x[j] = p[8 * u + j];
            split8(x, SPLIT_UP, pp[0], pp[1], pp[2]);
#pragma unroll
            for (int tt = 0; tt < ND; tt++) {
                const int dd = tt * 32 + col;
                split_b8 vf[3];
                floatx16 &part = low[LOW ? tt : 0];

                if (!LOW)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        part[r] = 0.0f;
#pragma unroll
                for (int k = 0; k < 3; k++)
                    vf[k] = __builtin_bit_cast(
                        split_b8, vs[k * PK + dd * 4 + ((2 * u + half) ^ (dd >> 2 & 3))]);
#pragma unroll
                for (int w = 0; w < 6; w++) {
                    floatx16 &c = w == 5 ? o[tt] : part;

                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        vf[pa[w]], __builtin_bit_cast(split_b8, pp[pb[w]]), c, 0, 0, 0);
                }
                if (!LOW)
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        o[tt][r] += part[r];
            }
        }
        __syncthreads();
    }

    {
        float z = l * 0.0f;

#pragma unroll
        for (int tt = 0; tt < ND; tt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                if (LOW)
                    o[tt][r] += low[LOW ? tt : 0][r];
                z = fmaf(o[tt][r], 0.0f, z);
            }
        /* No probability at all for keys that were kept: their scores lie
         * below the range. */
        if (__syncthreads_or(z != 0.0f || (l == 0.0f && __any(kept)))) {
            att_block_f32<ND, VEC, MASK>(a, (float *)lds, bx, by, bz, ny);
            return;
        }
    }
    if (qi >= a.Nq)
        return;
    if (!a.part_o) {
        const float inv = l > 0.0f ? 1.0f / l * SPLIT_DOWN : 0.0f;
        float *out = a.O + bi * a.bo + (long long)qi * a.ldo + (long long)h * d;

#pragma unroll
        for (int tt = 0; tt < ND; tt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int dd = tt * 32 + (r >> 2) * 8 + half * 4 + (r & 3);

                if (dd < d)
                    out[dd] = l > 0.0f ? o[tt][r] * inv : 0.0f;
            }
    }
    else {
        const long long row = ((long long)bz * ny + by) * a.Nq + qi;
        float *out = a.part_o + row * DP;

#pragma unroll
        for (int tt = 0; tt < ND; tt++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *(float4 *)(out + tt * 32 + g * 8 + half * 4) =
                    make_float4(o[tt][4 * g] * SPLIT_DOWN, o[tt][4 * g + 1] * SPLIT_DOWN,
                                o[tt][4 * g + 2] * SPLIT_DOWN, o[tt][4 * g + 3] * SPLIT_DOWN);
        if (half == 0)
            a.part_ml[row] = make_float2(m, l);
    }
}

/* Combine nsplit partial results per (image, query, head): weights
 * 2^(m_s - max m) (the maxima are in the base-2 domain), O = sum_s w_s O_s
 * / sum_s w_s l_s (zeros when no key was kept). One thread per output
 * value. */
__global__ void __launch_bounds__(256)
    attn_merge_kernel(const float *__restrict__ part_o,
                      const float2 *__restrict__ part_ml, int nsplit, int nb,
                      int nh, int Nq, int d, int DP, float *__restrict__ O,
                      int ldo, long long bo)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long total = (long long)nb * Nq * nh * d;

    if (idx >= total)
        return;
    const int dd = (int)(idx % d);
    const int h = (int)((idx / d) % nh);
    const long long bq = idx / ((long long)d * nh);
    const int qi = (int)(bq % Nq), bi = (int)(bq / Nq);
    const int y = bi * nh + h, ny = nb * nh;
    float mx = -INFINITY, L = 0.0f, acc = 0.0f;

    for (int s = 0; s < nsplit; s++)
        mx = fmaxf(mx, part_ml[((long long)s * ny + y) * Nq + qi].x);
    if (mx != -INFINITY)
        for (int s = 0; s < nsplit; s++) {
            const long long row = ((long long)s * ny + y) * Nq + qi;
            const float2 ml = part_ml[row];
            const float w =
                ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - mx);

            L += w * ml.y;
            acc += w * part_o[row * DP + dd];
        }
    O[bi * bo + (long long)qi * ldo + (long long)h * d + dd] =
        L > 0.0f ? acc / L : 0.0f;
}

/* attn_merge_kernel with four consecutive values of a row per thread
 * (d % 4 == 0, 16-byte aligned output rows): 16-byte loads and stores,
 * the (max, sum) pairs read once per four values. */
__global__ void __launch_bounds__(256)
    attn_merge4_kernel(const float4 *__restrict__ part_o,
                       const float2 *__restrict__ part_ml, int nsplit, int nb,
                       int nh, int Nq, int d, int DP, float *__restrict__ O,
                       int ldo, long long bo)
{
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const int d4 = d / 4;
    const long long total = (long long)nb * Nq * nh * d4;

    if (idx >= total)
        return;
    const int dq = (int)(idx % d4);
    const int h = (int)((idx / d4) % nh);
    const long long bq = idx / ((long long)d4 * nh);
    const int qi = (int)(bq % Nq), bi = (int)(bq / Nq);
    const int y = bi * nh + h, ny = nb * nh;
    float mx = -INFINITY, L = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);

    for (int s = 0; s < nsplit; s++)
        mx = fmaxf(mx, part_ml[((long long)s * ny + y) * Nq + qi].x);
    if (mx != -INFINITY)
        for (int s = 0; s < nsplit; s++) {
            const long long row = ((long long)s * ny + y) * Nq + qi;
            const float2 ml = part_ml[row];
            const float w =
                ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - mx);
            const float4 p = part_o[row * (DP / 4) + dq];

            L += w * ml.y;
            acc.x += w * p.x;
            acc.y += w * p.y;
            acc.z += w * p.z;
            acc.w += w * p.w;
        }
    *(float4 *)(O + bi * bo + (long long)qi * ldo + (long long)h * d + 4 * dq) =
        L > 0.0f ? make_float4(acc.x / L, acc.y / L, acc.z / L, acc.w / L)
                 : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

/* Key ranges of attention_split_kernel, at most `most`: the fewest
 * microseconds of the slowest CU (its share of the blocks, each a range's
 * tiles and about one for its start) and of the merge (3, and merge_us for
 * the partials of each range, written and read). A tile of one block takes
 * about 0.6 + 0.75 ND, a block beside it 0.55 more, as many as the
 * registers hold (4, 3, 1). Against the fp32 kernel's count (`most`, two
 * blocks per CU and evened out), which cuts finer than one block a CU
 * wherever few heads leave the chip short: 1600 tokens, 8 heads of 128, 2
 * ranges instead of 5 121 -> 95 us; 785 x 16 x 64, 2 instead of 5 43.5 -> 37;
 * 2 x 676 x 8 x 32, 2 instead of 7 27.9 -> 22.7; 2 x 1601 x 16 x 64 keeps
 * its 3 (147; 1: 152, 2: 164). */
template <int ND>
static int split_count(int most, long long blocks, int ntiles, int cus, double merge_us,
                       int &tps)
{
    constexpr int held = ND == 1 ? 4 : ND == 2 ? 3 : 1;
    double best = 0;
    int n = most;

    for (int s = 1; s <= most; s++) {
        const int len = (ntiles + s - 1) / s;
        const int ranges = len > 0 ? (ntiles + len - 1) / len : 1;
        const long long each = (blocks * ranges + cus - 1) / cus;
        const double rounds = (double)(each / held) * (0.45 + 0.55 * held) +
                              (each % held ? 0.45 + 0.55 * (each % held) : 0.0);
        const double us =
            (len + 1) * rounds * (0.6 + 0.75 * ND) + (ranges > 1 ? 3 + ranges * merge_us : 0.0);

        if (s == 1 || us < best) {
            best = us;
            n = ranges;
            tps = len;
        }
    }
    return n;
}

/* Partials of the key splits: the ops work buffer (grown on demand), or,
 * for ops_attention_noalloc, the fixed device array `fixed` of
 * fixed_bytes bytes (too small a one is a fatal error). */
template <int ND, bool VEC, bool MASK>
static void launch_nd(struct ops *ops, hipStream_t st, int nb, int nh,
                      const float *Q, int ldq, long long bq, const float *K,
                      int ldk, long long bk, const float *V, int ldv,
                      long long bv, float *O, int ldo, long long bo, int Nq,
                      int Nk, int d, float scale, const unsigned char *kmask,
                      float *fixed, size_t fixed_bytes)
{
    const int qb = (Nq + 32 * ATT_NW - 1) / (32 * ATT_NW);
    const int ntiles = (Nk + ATT_KT - 1) / ATT_KT;
    /* Key splits so that about 8 waves per CU are resident, each split at
     * least 2 key tiles (measured: more splits cost more in the merge
     * than they gain in occupancy). */
    const long long want = 8LL * (ops->ocl->cu_count > 0 ? ops->ocl->cu_count : 256);
    const long long base = (long long)qb * ATT_NW * nh * nb;
    int nsplit = (int)((want + base - 1) / base);
    int tps;

    nsplit = max(1, min(nsplit, min(ntiles / 2, 64)));
    /* With a block or more per CU, the CUs that get one block more than
     * the others set the time: raise the split (at most two steps) until
     * the blocks spread within 10 % of evenly (the ViT's 1601 tokens: 2
     * -> 3 splits, 4.875 blocks per CU instead of 3.25 on 4-block CUs). */
    {
        const long long cus = ops->ocl->cu_count > 0 ? ops->ocl->cu_count : 256;
        const long long qbh = (long long)qb * nh * nb;

        if (qbh * nsplit >= cus)
            for (int s = nsplit; s <= nsplit + 2 && s <= ntiles / 2; s++) {
                const long long blocks = qbh * s;

                if ((blocks + cus - 1) / cus * cus * 10 <= blocks * 11) {
                    nsplit = s;
                    break;
                }
            }
    }
    tps = ntiles > 0 ? (ntiles + nsplit - 1) / nsplit : 0;
    nsplit = tps > 0 ? (ntiles + tps - 1) / tps : 1;
    /* What the scratch must hold: the most splits that are considered. */
    const size_t rows = (size_t)nsplit * nb * nh * Nq;
    const size_t ob = nsplit > 1 ? rows * 32 * ND * sizeof(float) : 0;

    if (nsplit > 1 && fixed && ob + rows * sizeof(float2) > fixed_bytes)
        icoreg_fatal("ops_attention_noalloc: the key-split partials (%zu bytes) "
                     "exceed the %zu-byte scratch array",
                     ob + rows * sizeof(float2), fixed_bytes);
    if (ND != 3)
        nsplit = split_count<ND>(nsplit, (long long)qb * nh * nb, ntiles,
                                 ops->ocl->cu_count > 0 ? ops->ocl->cu_count : 256,
                                 5e-7 * 4 * nb * nh * Nq * 32 * ND, tps);

    auto launch = [&](dim3 grid, float *po, float2 *pml) {
        const att_args a = {Q,  K,  V, O,  kmask, po,    pml, ldq, ldk, ldv, ldo,
                            Nq, Nk, d, nh, tps,   scale, bq,  bk,  bv,  bo};

        if constexpr (ND == 3)
            hipLaunchKernelGGL((attention_kernel<ND, VEC, MASK>), grid, dim3(64 * ATT_NW), 0, st,
                               a);
        else
            hipLaunchKernelGGL((attention_split_kernel<ND, VEC, MASK>),
                               grid, dim3(64 * ATT_NW), 0, st, a);
    };

    if (nsplit == 1) {
        launch(dim3((unsigned)qb, (unsigned)(nh * nb), 1), nullptr, nullptr);
        return;
    }
    {
        float *po;

        if (fixed)
            po = fixed;
        else
            po = (float *)scratch_get(ops, ob + rows * sizeof(float2))->ptr;
        float2 *pml = (float2 *)((char *)po + ob);
        const long long total = (long long)nb * Nq * nh * d;

        launch(dim3((unsigned)qb, (unsigned)(nh * nb), (unsigned)nsplit), po, pml);
        if (d % 4 == 0 && ldo % 4 == 0 && bo % 4 == 0 && ((uintptr_t)O & 15) == 0)
            hipLaunchKernelGGL(attn_merge4_kernel,
                               dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0,
                               st, (const float4 *)po, pml, nsplit, nb, nh, Nq, d, 32 * ND,
                               O, ldo, bo);
        else
            hipLaunchKernelGGL(attn_merge_kernel,
                               dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                               st, po, pml, nsplit, nb, nh, Nq, d, 32 * ND, O, ldo,
                               bo);
    }
}

static void need_rows(const struct opnd &x, int nb, long long bs, int rows,
                      int cols, const char *op, const char *operand)
{
    if (x.off < 0 || x.ld < 0 || bs < 0)
        icoreg_fatal("%s: %s has a negative offset, ld or batch stride", op,
                     operand);
    need_floats(x.buf, x.off + (nb - 1) * bs,
                (long long)(rows - 1) * x.ld + cols, op, operand);
}

/* nb independent problems at batch strides bq .. bo floats (the key mask,
 * when given, is shared by all of them). */
static void attention_impl(struct ops *o, const char *op, int nb,
                           struct opnd Q, long long bq, struct opnd K,
                           long long bk, struct opnd V, long long bv,
                           struct opnd O, long long bo, int Nq, int Nk, int nh,
                           int d, float scale, cl_mem kmask, float *fixed = nullptr,
                           size_t fixed_bytes = 0)
{
    hipStream_t st = stream_of(o->ocl);

    if (d < 1 || d > OPS_MAX_HEAD_DIM)
        icoreg_fatal("HIP: attention head dimension %d not in 1..%d", d,
                     OPS_MAX_HEAD_DIM);
    if (Nq < 0 || Nk < 0 || nh < 1 || nb < 1 || (long long)nh * nb > 65535)
        icoreg_fatal("%s: invalid sizes Nq=%d Nk=%d nh=%d nb=%d", op, Nq, Nk,
                     nh, nb);
    if (Nq == 0)
        return;
    need_rows(Q, nb, bq, Nq, nh * d, op, "Q");
    need_rows(O, nb, bo, Nq, nh * d, op, "O");
    if (Nk > 0) {
        need_rows(K, nb, bk, Nk, nh * d, op, "K");
        need_rows(V, nb, bv, Nk, nh * d, op, "V");
    }
    if (kmask)
        need_bytes(kmask, 0, Nk, op, "kmask");
    prof_scope ps(o->ocl, "attention");
#define ARGS                                                                   \
    o, st, nb, nh, cfptr(Q.buf) + Q.off, Q.ld, bq, cfptr(K.buf) + K.off, K.ld, \
        bk, cfptr(V.buf) + V.off, V.ld, bv, fptr(O.buf) + O.off, O.ld, bo, Nq, \
        Nk, d, scale, kmask ? (const unsigned char *)kmask->ptr : nullptr, fixed,   \
        fixed_bytes
    {
        /* 16-byte K / V loads when every row and head start is aligned. */
        const bool vec = d % 4 == 0 && K.ld % 4 == 0 && V.ld % 4 == 0 &&
                         K.off % 4 == 0 && V.off % 4 == 0 && bk % 4 == 0 &&
                         bv % 4 == 0 && ((uintptr_t)K.buf->ptr & 15) == 0 &&
                         ((uintptr_t)V.buf->ptr & 15) == 0;

#define DISPATCH(ND)                                                           \
    if (kmask)                                                                 \
        vec ? launch_nd<ND, true, true>(ARGS)                                  \
            : launch_nd<ND, false, true>(ARGS);                                \
    else                                                                       \
        vec ? launch_nd<ND, true, false>(ARGS)                                 \
            : launch_nd<ND, false, false>(ARGS)
        if (d <= 32) {
            DISPATCH(1);
        }
        else if (d <= 64) {
            DISPATCH(2);
        }
        else if (d <= 96) {
            DISPATCH(3);
        }
        else {
            DISPATCH(4);
        }
#undef DISPATCH
    }
#undef ARGS
    launch_check("attention");
}

extern "C" void ops_attention(struct ops *o, struct opnd Q, struct opnd K,
                              struct opnd V, struct opnd O, int Nq, int Nk,
                              int nh, int d, float scale, cl_mem kmask)
{
    ICOREG_API_BEGIN
    attention_impl(o, "ops_attention", 1, Q, 0, K, 0, V, 0, O, 0, Nq, Nk, nh,
                   d, scale, kmask);
    ICOREG_API_END
}

/* ---- ops_attention without allocation ------------------------------------------ */

/* The key-split partials of ops_attention_noalloc: a fixed array per
 * GPU, held until the process ends, shared by every call on that GPU.
 * Its device memory is reserved wherever the library's code object is
 * loaded, whether or not the entry point is called, so it is sized to
 * the largest caller on the path: RoMa's ViT attention (1601 tokens, 16
 * heads of 64, 3 key splits) needs 20.3 MB. */
#define ATT_NOALLOC_BYTES ((size_t)24 << 20)
static __device__ __align__(256) float scratch[ATT_NOALLOC_BYTES / sizeof(float)];

/* scratch's device address on each GPU (hipGetSymbolAddress once per
 * device, with that device current); the host symbol is only a
 * stand-in and is never handed to a kernel or a copy. */
static float *scratch_dev[64];
static std::mutex scratch_mu;

static float *noalloc_scratch(void)
{
    int dev = -1;
    float *p;

    hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (dev < 0 || dev >= 64)
        icoreg_fatal("ops_attention_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_dev[dev]) {
        p = nullptr;
        hip_check(hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch)),
                  "hipGetSymbolAddress(scratch)");
        if (!p)
            icoreg_fatal("ops_attention_noalloc: no device address for the scratch array");
        scratch_dev[dev] = p;
    }
    return scratch_dev[dev];
}

extern "C" void ops_attention_noalloc(struct ops *o, struct opnd Q, struct opnd K,
                                      struct opnd V, struct opnd O, int Nq, int Nk,
                                      int nh, int d, float scale, cl_mem kmask)
{
    ICOREG_API_BEGIN
    float *p = noalloc_scratch();

    attention_impl(o, "ops_attention_noalloc", 1, Q, 0, K, 0, V, 0, O, 0, Nq, Nk, nh,
                   d, scale, kmask, p, ATT_NOALLOC_BYTES);
    ICOREG_API_END
}

extern "C" void ops_attention_batch(struct ops *o, int nb, struct opnd Q,
                                    long bq, struct opnd K, long bk,
                                    struct opnd V, long bv, struct opnd O,
                                    long bo, int Nq, int Nk, int nh, int d,
                                    float scale, cl_mem kmask)
{
    ICOREG_API_BEGIN
    attention_impl(o, "ops_attention_batch", nb, Q, bq, K, bk, V, bv, O, bo,
                   Nq, Nk, nh, d, scale, kmask);
    ICOREG_API_END
}
