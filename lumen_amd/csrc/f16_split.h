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

// Elements below this (bits), zeros aside, lose bits as pairs beside an element of magnitude `top_bits`.
__device__ __forceinline__ unsigned small_limit(unsigned top_bits) {
    const unsigned ex = top_bits >> 23;
    return ex > 18 ? (ex - 18) << 23 : 1u;
}
__device__ __forceinline__ bool is_small(unsigned bits, unsigned limit) { return bits - 1u < limit - 1u; }

// What holds too many small elements for pairs is multiplied by f32 matrix instructions; its exponent is marked.
#define SPLIT_WIDE 1024
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
