/* SPDX-License-Identifier: Unlicense */

/* float32 products on the bf16 matrix instructions, without loss: a
 * float32 value, scaled by SPLIT_UP, is the sum of three bf16 values exactly
 * (8 + 8 + 8 significant bits, each part the round-to-nearest of what the
 * parts before it leave), x = h + m + l with |m| <= 2^-9 |h| and |l| <= 2^-18
 * |h|. Of the nine products of two such sums the six of order 2^-18 and
 * above, hh + (hm + mh) + (hl + mm + lh), are formed; each is exact (16
 * significant bits) and accumulates in float32 inside the matrix core, so
 * what is left out is at most 3 * 2^-27 of |x y|, three eighths of a float32
 * rounding. Six v_mfma_f32_32x32x16_bf16 (32 cycles each) do the work of eight
 * v_mfma_f32_32x32x2f32 (64 cycles each).
 *
 * The scale, 2^24: a float32 value is a multiple of 2^-149, bf16's last place
 * 2^-133. Unscaled, values under 2^-110 lose bits (sums of operands of 2^-116
 * were off by 2e-6, of 2^-126 by 2e-3); scaled, every part of every float32
 * value, subnormal ones included, is a multiple of 2^-125 and so no
 * subnormal bf16 value. SPLIT_DOWN scales a product of two back. Powers of
 * two: nothing is rounded.
 *
 * A value that is not finite makes m NaN and with it every sum it enters;
 * so does one of 2^104 and above, and sums from 2^80 on may overflow:
 * kernels look at their sums and form those that are not finite again from
 * the float32 values. */

#ifndef ICOREG_SPLIT_H
#define ICOREG_SPLIT_H

#include <hip/hip_runtime.h>

typedef float split_f16x __attribute__((ext_vector_type(16)));
typedef float split_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_b2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_b8 __attribute__((ext_vector_type(8)));
typedef unsigned split_u4 __attribute__((ext_vector_type(4)));

#define SPLIT_UP 0x1p24f     /* scale of a split operand */
#define SPLIT_DOWN 0x1p-48f  /* what takes it back from a product of two */

/* The bf16 values of a (low half) and b (high half). */
static __device__ __forceinline__ unsigned split_pk(float a, float b)
{
    const split_f2 v = {a, b};

    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, split_b2));
}

static __device__ __forceinline__ float split_lo(unsigned p)
{
    return __builtin_bit_cast(float, p << 16);
}

static __device__ __forceinline__ float split_hi(unsigned p)
{
    return __builtin_bit_cast(float, p & 0xffff0000u);
}

/* The three parts of a and b, packed in pairs. */
static __device__ __forceinline__ void split2(float a, float b, unsigned &h, unsigned &m,
                                              unsigned &l)
{
    h = split_pk(a, b);
    a -= split_lo(h);
    b -= split_hi(h);
    m = split_pk(a, b);
    a -= split_lo(m);
    b -= split_hi(m);
    l = split_pk(a, b);
}

/* The three parts of eight values times s, one 16-byte operand each. */
static __device__ __forceinline__ void split8(const float (&x)[8], float s, split_u4 &h,
                                              split_u4 &m, split_u4 &l)
{
#pragma unroll
    for (int i = 0; i < 4; i++) {
        unsigned a, b, c;

        split2(x[2 * i] * s, x[2 * i + 1] * s, a, b, c);
        h[i] = a;
        m[i] = b;
        l[i] = c;
    }
}

#endif /* ICOREG_SPLIT_H */
