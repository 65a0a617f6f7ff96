// An f32 value as two f16 values: x 2^e = hi + lo, e one exponent per row of an operand that takes the row's largest
// magnitude into [2^14, 2^15) (rows that stay below 2^-112 take ROW_EXP_MAX, which leaves them smaller).  hi carries 11 bits of x 2^e and lo
// the next 11 (12 with its sign), down to 2^-25 absolute: an element up to 2^18 times smaller than its row's largest keeps its 22 to
// 23 bits, smaller ones an error of 2^-40 of that largest.
#pragma once

#include "internal.h"
#include "wave_reduce.h"

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define ROW_EXP_MAX 126

// e of a row, from the largest of its magnitudes' bits (an infinity or a NaN has larger bits than any number).  Rows of zeros, and rows
// that hold an infinity or a NaN -- whose products are not finite either way --, take 0.
__device__ __forceinline__ int row_exponent(unsigned magnitude_bits) {
    const int ex = (int)(magnitude_bits >> 23);
    if (ex == 255 || magnitude_bits == 0u) return 0;
    const int e = 141 - ex;
    return e < ROW_EXP_MAX ? e : ROW_EXP_MAX;
}
__device__ __forceinline__ float exp2_int(int e) { return __uint_as_float((unsigned)(e + 127) << 23); }  // |e| <= ROW_EXP_MAX

__device__ __forceinline__ unsigned magnitude_bits(float x) { return __float_as_uint(x) & 0x7fffffffu; }
__device__ __forceinline__ unsigned magnitude_bits(const f32x4_t v) {
    const unsigned a = magnitude_bits(v.x), b = magnitude_bits(v.y), c = magnitude_bits(v.z), d = magnitude_bits(v.w);
    const unsigned ab = a > b ? a : b, cd = c > d ? c : d;
    return ab > cd ? ab : cd;
}

// Elements below this (bits), zeros aside, lose bits as pairs beside an element of magnitude `top_bits`.  (bf16 values, one f16 value each: RANGE 31.)
template <unsigned RANGE = 18>
__device__ __forceinline__ unsigned small_limit(unsigned top_bits) {
    const unsigned ex = top_bits >> 23;
    return ex > RANGE ? (ex - RANGE) << 23 : 1u;
}
__device__ __forceinline__ bool is_small(unsigned bits, unsigned limit) { return bits - 1u < limit - 1u; }

// What holds too many small elements for pairs is multiplied by f32 matrix instructions; its exponent is marked.  A row: more than one element in 32
// (normally distributed ones hold one in 10^5, products of two such one in 4000).  So what pairs leave of a row is within 2^-22 of all but a few of its
// elements, whatever lies beside them.
#define SPLIT_WIDE 1024
#define SPLIT_ROW_SMALL 32
__device__ __forceinline__ bool is_wide(int code) { return code > SPLIT_WIDE / 2; }
__device__ __forceinline__ int code_exponent(int code) { return is_wide(code) ? code - SPLIT_WIDE : code; }

// (a, b) s -> two dwords of f16 pairs.  Both roundings are to nearest; with s a power of two x s and x s - hi are exact in f32.
__device__ __forceinline__ void split_pair(float a, float b, float s, unsigned &hi, unsigned &lo) {
    const f16x2_t h = {(_Float16)fmaf(a, s, 0.f), (_Float16)fmaf(b, s, 0.f)};
    const f16x2_t l = {(_Float16)fmaf(a, s, -(float)h.x), (_Float16)fmaf(b, s, -(float)h.y)};
    hi = __builtin_bit_cast(unsigned, h);
    lo = __builtin_bit_cast(unsigned, l);
}

// Split rows lie in memory as [k / 16][hi, lo][16 f16] -- 64 bytes per 16 values, as many as the f32 values take.  Elements k .. k + 3 (k a
// multiple of 4) of the row that starts at `row`:
__device__ __forceinline__ void store_split4(uint16_t *row, int k, const f32x4_t v, float s) {
    unsigned h0, l0, h1, l1;
    split_pair(v.x, v.y, s, h0, l0);
    split_pair(v.z, v.w, s, h1, l1);
    uint16_t *o = row + 2 * (k & ~15) + (k & 15);
    *(u32x2_t *)o = u32x2_t{h0, h1};
    *(u32x2_t *)(o + 16) = u32x2_t{l0, l1};
}

// A row of dim elements (a multiple of 16) that a workgroup holds, elements 4 (thread + threads i) .. + 3 in v[i] and zeros past its end: to `row` as
// pairs, or as the f32 values it holds where pairs cannot, its exponent to *exp.  Every thread of the workgroup calls it, once per launch.
// The pairs are on their way before the small elements are counted: a row of the rare kind is written again.  (The count costs 0.2 us where 1024 threads
// have a row of 5632, 0.5 where 256 have one of 2048.)
template <int VPT>
__device__ __forceinline__ void leave_row(const f32x4_t (&v)[VPT], int dim, float *row, int *exp) {
    __shared__ unsigned row_top[16];
    __shared__ float row_small[16];
    const int tid = threadIdx.x, threads = blockDim.x, waves = threads >> 6;
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i) m = max(m, magnitude_bits(v[i]));
    m = wave_umax(m);
    if ((tid & 63) == 0) row_top[tid >> 6] = m;
    __syncthreads();
    m = 0;
    for (int w = 0; w < waves; ++w) m = max(m, row_top[w]);
    const int e = row_exponent(m);
    const float s = exp2_int(e);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int k = (tid + i * threads) * 4;
        if (k < dim) store_split4((uint16_t *)row, k, v[i], s);
    }
    const unsigned limit = small_limit(m);
    unsigned least = ~0u;  // (a zero is the largest here)
#pragma unroll
    for (int i = 0; i < VPT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) least = min(least, magnitude_bits(v[i][j]) - 1u);
    float sum = 0.f;
    if (__any(least < limit - 1u)) {  // uniform
        int n = 0;
#pragma unroll
        for (int i = 0; i < VPT; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) n += is_small(magnitude_bits(v[i][j]), limit);
        sum = wave_sum((float)n);
    }
    if ((tid & 63) == 0) row_small[tid >> 6] = sum;
    __syncthreads();
    float small = 0.f;
    for (int w = 0; w < waves; ++w) small += row_small[w];
    const bool wide = small * (float)SPLIT_ROW_SMALL > (float)dim;
    if (tid == 0) *exp = wide ? e + SPLIT_WIDE : e;
    if (!wide) return;
    __threadfence();  // (other threads' pairs lie where this thread's values go)
    __syncthreads();
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int k = (tid + i * threads) * 4;
        if (k < dim) *(f32x4_t *)(row + k) = v[i];
    }
}
