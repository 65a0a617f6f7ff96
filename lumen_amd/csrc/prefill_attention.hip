// Causal GQA attention for a prompt (S > 1) on the matrix cores:
// self_attention.rs:308-419 with gqa_attention_no_repeat_bshd_view (:519-641)
// and softmax_inplace_view (:643-678) -- scores = Q K^T * scale, mask
// j > past_len + i, softmax with divisor (sum + 1e-9), ctx = P V, output BSHD.
//
// The reference materialises the S x L score matrix per head; here a
// workgroup keeps 128 (position, query head) rows of one KV group in
// registers and walks the cached keys in tiles of 32 with an online softmax,
// so scores never leave the compute unit and every K/V tile read from the
// cache serves all n_rep heads of the group and 128 / n_rep positions at once.
//
// The products run on the f16 matrix cores at f32 accuracy, as the prompt products of gemm_f16x2.hip do: every operand is the sum of two f16
// values (f16_split.h), a product the three part products down to 2^-22, accumulated in f32 by v_mfma_f32_32x32x16_f16.  A tile of
// keys has one exponent for its keys and one for its values (kv_tiles_kernel), every query its own, and a lane keeps the sum of its row in the units
// that its largest contribution so far -- weight times the tile's largest value -- asks for.  A tile in which some keys or channels are
// 2^18 times smaller than others, which pairs cannot hold beside each other, or a query row of that kind, sends the workgroups that meet
// it to f32 matrix instructions, from the f32 values: about three times slower, and met by no values of usual spread.
// So the error of a row does not depend on the magnitude of keys that it does not see, nor on that of other tiles.
// Bound by the matrix instructions and the softmax between them, which wait for each other within a wavefront; two per SIMD overlap.
// With three bf16 parts: 420 us for 3968 positions of 32 heads of 64 (4 KV heads), with f16 pairs 305 (288 with one exponent for all keys of a
// head, which is unsound); 509 of 32 heads of 128: 61 -> 47.
// Few positions behind a long cache leave most compute units without a block of queries: the keys are then cut into parts (128 positions
// behind 2900, 32 heads of 64: 111 us in one part, 33 in 16; 256 behind 2900, 16 heads of 128: 198 -> 56).
//
// Per wavefront (32 rows) and key tile, everything transposed so that a lane owns one query row:
//   S^T = K Q^T       K from LDS ([part][key][element], split on its way in) is the A operand, Q
//                     (split once, in registers) the B operand.  A lane then holds 16 of the
//                     tile's 32 scores of ITS row, lane ^ 32 the other 16
//   softmax           row max and sum in the lane (one exchange with lane ^ 32 for the max, one at
//                     the very end for the sum); scores in log2 units (Q pre-multiplied by
//                     scale * log2 e), P = exp2(S - m)
//   O^T += V^T P^T    V is staged transposed ([part][element][key position]) as the A operand; the
//                     lane's 16 weights are the B operand as they stand (split in the lane), no
//                     trip through LDS; the rescale by alpha is a per-lane scalar
#include "internal.h"
#include "attn_device.h"
#include "f16_split.h"

#include <algorithm>
#include <type_traits>

typedef float v16f __attribute__((ext_vector_type(16)));

#define FA_ROWS 128  // (position, head) rows per workgroup
#define FA_KEYS 32   // keys per tile
#define FA_THREADS 256

#define FA_P_EXP 14  // the largest weight of a tile that counts is split as 2^14

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));

// x[0..3] s -> two parts of 4 f16 (2 dwords each)
__device__ __forceinline__ void fa_split4(const v4f x, float s, v2u (&part)[2]) {
    unsigned h0, l0, h1, l1;
    split_pair(x.x, x.y, s, h0, l0);
    split_pair(x.z, x.w, s, h1, l1);
    part[0] = v2u{h0, h1};
    part[1] = v2u{l0, l1};
}

// Exponents (f16_split.h; marked where the tile takes f32 instructions) of the keys, and values, of each tile of KEYS of the L cached rows of a KV
// head: tiles [2][b hkv][ceil(L / KEYS)].  Small elements that a tile may hold as pairs: fewer than FA_SMALL, which is less than a key's
// or a channel's worth of them; 4096 normally distributed values hold 0.05.
#define FA_SMALL 16
template <int D, int KEYS>
__global__ __launch_bounds__(256) void kv_tiles_kernel(const float *k, const float *v, int max_seq, int L, int *tiles) {
    constexpr int PIECES = D * KEYS / 1024;
    __shared__ unsigned top[2][4];
    __shared__ float low[2][4];
    const int tid = threadIdx.x, head = blockIdx.y, j0 = (int)blockIdx.x * KEYS;
    const size_t base = ((size_t)head * max_seq + j0) * D;
    v4f x[2][PIECES];
    unsigned m[2] = {0u, 0u};
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
        const int at = (tid + p * 256) * 4;
        const bool in = j0 + at / D < L;
        x[0][p] = in ? *(const v4f *)(k + base + at) : v4f{0.f, 0.f, 0.f, 0.f};
        x[1][p] = in ? *(const v4f *)(v + base + at) : v4f{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int w = 0; w < 2; ++w) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned u = magnitude_bits(x[w][p][e]);
                m[w] = max(m[w], u < 0x7f800000u ? u : 0u);  // the largest finite one
            }
        m[w] = wave_umax(m[w]);
        if ((tid & 63) == 0) top[w][tid >> 6] = m[w];
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        m[w] = max(max(top[w][0], top[w][1]), max(top[w][2], top[w][3]));
        const unsigned limit = small_limit(m[w]);
        int n = 0;
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const unsigned u = magnitude_bits(x[w][p][e]);
                n += is_small(u, limit) ? 1 : u >= 0x7f800000u ? FA_SMALL : 0;
            }
        const float sum = wave_sum((float)n);
        if ((tid & 63) == 0) low[w][tid >> 6] = sum;
    }
    __syncthreads();
    if (tid < 2) {
        const unsigned t = m[tid];
        const int e = t ? row_exponent(t) : ROW_EXP_MAX;  // (zeros weigh nothing)
        const bool wide = (low[tid][0] + low[tid][1]) + (low[tid][2] + low[tid][3]) >= (float)FA_SMALL;
        tiles[((size_t)tid * gridDim.y + head) * gridDim.x + blockIdx.x] = wide ? e + SPLIT_WIDE : e;
    }
}

// KT: key tiles of 32 per trip of the loop (2 for head_dim 64: one barrier pair, one row maximum and one rescale of
// O per 64 keys; 1 for head_dim 128, whose K and V tiles fill LDS twice as fast).
// PART: blockIdx.z / b is a part of the keys (a.key_chunk each, whole trips); the unfinished rows go to a.part and a.part_ml for
// merge_parts_kernel.
template <int D, int NREP, int KT, bool PART>
__global__ __launch_bounds__(FA_THREADS, 2) void attn_prefill_f16x2_kernel(AttnPrefillArgs a) {
    constexpr int BQ = FA_ROWS / NREP;  // positions per workgroup
    constexpr int KEYS = FA_KEYS * KT;   // keys per trip
    constexpr int DT = D / 32;          // 32-wide tiles of the head dimension
    constexpr int PIECES = D * KEYS / 4 / FA_THREADS;  // 16-byte pieces of a K (or V) tile per thread
    // rows of 4 words more than a multiple of 32: the 16-byte reads of 8 neighbouring rows hit distinct banks
    constexpr int LDK = D + 8, LDV = KEYS + 8;
    __shared__ __align__(16) uint16_t Ks[2][KEYS][LDK];  // [part][key][element]
    __shared__ __align__(16) uint16_t Vt[2][D][LDV];        // [part][element][key position]

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 31, half = lane >> 5;
    // workgroups are dealt in index order: the blocks of late positions (most keys) go first
    const int q0 = (int)(gridDim.x - 1 - blockIdx.x) * BQ, hk = blockIdx.y, bb = PART ? (int)blockIdx.z % a.b : (int)blockIdx.z;
    const int key_part = PART ? (int)blockIdx.z / a.b : 0;
    const int L = a.past_len + a.s;
    const int n_tiles = (L + KEYS - 1) / KEYS;
    const int *ktab = a.kv_tiles + ((size_t)bb * a.hkv + hk / a.kv_div) * n_tiles, *vtab = ktab + (size_t)a.b * a.hkv * n_tiles;
    const size_t head_base = ((size_t)bb * a.hkv + hk / a.kv_div) * a.max_seq * D;  // kv_div > 1: grid row = query head
    const float *Kc = a.k_cache + head_base, *Vc = a.v_cache + head_base;

    // This lane's query row (the COLUMN it owns in S^T and O^T): (position, head) row wave * 32 + c of the workgroup
    const int my_row = wave * 32 + c;
    const int my_i = min(q0 + my_row / NREP, a.s - 1);  // clamped: rows past S are computed and dropped
    const int my_pos = a.past_len + q0 + my_row / NREP;  // absolute position: keys up to it are visible
    const int q_last = min(q0 + BQ, a.s) - 1;
    const int kbeg = PART ? key_part * a.key_chunk : 0;
    int kmax = a.causal ? min(L, a.past_len + q_last + 1) : L;
    if (PART) kmax = min(kmax, kbeg + a.key_chunk);
    const int wave_i_last = min(q0 + (wave * 32 + 31) / NREP, a.s - 1);
    const int wave_kmax = a.causal ? min(L, a.past_len + wave_i_last + 1) : L;
    // keys [0, wave_kfull) are visible to every row of this wavefront: no mask needed below it
    const int wave_kfull = a.causal ? min(L, a.past_len + q0 + (wave * 32) / NREP + 1) : L;

    // V^T is staged with bits 2 and 3 of the key index exchanged: the 8 keys a lane holds of S^T (4 + 4,
    // eight apart) then sit next to each other for the 16-byte operand read.  A thread takes 4 elements
    // (v_k4 ..) of the 4 keys that land on positions 4 v_g .. 4 v_g + 3 -- consecutive keys from v_key on --
    // so that one element of the four keys is one 8-byte LDS write.
    static_assert(PIECES == 4, "a thread stages four keys of V");
    constexpr int NG = KEYS / 4;  // groups of four key positions
    const int v_g = (tid >> 2) % NG, v_k4 = ((tid / (4 * NG)) * 4 + (tid & 3)) * 4;
    const int v_key = 4 * ((v_g & ~3) | ((v_g & 1) << 1) | ((v_g >> 1) & 1));
    v4f kreg[PIECES], vreg[PIECES];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int idx = tid + p * FA_THREADS;
            const int key = idx / (D / 4), k4 = (idx % (D / 4)) * 4;
            const int j = min(j0 + key, L - 1);  // keys past L are masked below
            kreg[p] = *(const v4f *)(Kc + (size_t)j * D + k4);
            vreg[p] = *(const v4f *)(Vc + (size_t)min(j0 + v_key + p, L - 1) * D + v_k4);
        }
    };

    // pairs or f32 instructions: one choice for all of this workgroup's tiles (a choice per tile keeps both forms' registers alive at once)
    int first_k = 0, first_v = 0, tile_wide = 0;
    if (kmax > kbeg) {
        fetch(kbeg);
        first_k = ktab[kbeg / KEYS];
        first_v = vtab[kbeg / KEYS];
    }
    for (int t = kbeg / KEYS + tid; t < (kmax + KEYS - 1) / KEYS; t += FA_THREADS) tile_wide |= is_wide(ktab[t]) || is_wide(vtab[t]);
    const float *qrow = a.q_rot + (((size_t)bb * a.s + my_i) * a.hq + (size_t)hk * NREP + my_row % NREP) * D;
    const float qf_scale = a.scale * LUMEN_LOG2E;
    // Q as the B operand of S^T = K Q^T: lane (column c, half g) holds elements ks * 16 + g * 8 .. + 7 of its row
    __shared__ int wide_any[FA_THREADS / 64];
    v4f x[D / 16][2];
    int eq;
    float q_scale;
    bool q_wide;
    {
        unsigned m = 0;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                x[ks][h] = *(const v4f *)(qrow + ks * 16 + half * 8 + h * 4);
                x[ks][h].x *= qf_scale; x[ks][h].y *= qf_scale; x[ks][h].z *= qf_scale; x[ks][h].w *= qf_scale;
                m = max(m, magnitude_bits(x[ks][h]));
            }
        m = max(m, (unsigned)__shfl_xor((int)m, 32, 64));
        eq = row_exponent(m);
        q_scale = exp2_int(eq);
        const unsigned limit = small_limit(m);
        int small = 0;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) small += is_small(magnitude_bits(x[ks][h][e]), limit);
        small += __shfl_xor(small, 32, 64);
        q_wide = small > D / 32 || m >= 0x7f800000u;
    }
    {
        const int any = __any(q_wide || tile_wide);
        if (lane == 0) wide_any[wave] = any;
    }
    __syncthreads();
    const bool wide = (wide_any[0] | wide_any[1] | wide_any[2] | wide_any[3]) != 0;

    auto rows = [&](auto form) {
        constexpr bool WIDE = decltype(form)::value;
        constexpr int PA_[3] = {1, 0, 0}, PB_[3] = {0, 1, 0};  // part products by ascending size: lo hi, hi lo, hi hi
        v4u qp[D / 16][2];
        if (!WIDE) {
#pragma unroll
            for (int ks = 0; ks < D / 16; ++ks) {
                v2u lo[2], hi[2];
                fa_split4(x[ks][0], q_scale, lo);
                fa_split4(x[ks][1], q_scale, hi);
#pragma unroll
                for (int p = 0; p < 2; ++p) qp[ks][p] = (v4u){lo[p].x, lo[p].y, hi[p].x, hi[p].y};
            }
        }
        // O^T: register r of tile t belongs to element 32 t + 8 (r / 4) + 4 half + r % 4 of this lane's row
        v16f O[DT];
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) O[t][r] = 0.f;
        float m_run = -INFINITY, l_run = 0.f;  // of this lane's row; l over this lane's half of the keys
        float o_run = -INFINITY;               // log2 of the largest contribution to O so far; O is in units of 2^(o_run - FA_P_EXP)
        // f32 instructions read [key][element] and [element][key], in the bytes of Ks and Vt
        float *Kf = (float *)&Ks[0][0][0], *Vf = (float *)&Vt[0][0][0];
        int k_code = first_k, v_code = first_v;
        for (int j0 = kbeg; j0 < kmax; j0 += KEYS) {
            const int ek = code_exponent(k_code), ev = code_exponent(v_code);
            const float k_scale = exp2_int(ek), v_scale = exp2_int(ev);
            if (!WIDE) {
#pragma unroll
                for (int p = 0; p < PIECES; ++p) {
                    const int idx = tid + p * FA_THREADS;
                    const int key = idx / (D / 4), k4 = (idx % (D / 4)) * 4;
                    v2u kp[2];
                    fa_split4(kreg[p], k_scale, kp);
#pragma unroll
                    for (int q = 0; q < 2; ++q) *(v2u *)&Ks[q][key][k4] = kp[q];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v2u vp[2];
                    fa_split4((v4f){vreg[0][e], vreg[1][e], vreg[2][e], vreg[3][e]}, v_scale, vp);
#pragma unroll
                    for (int q = 0; q < 2; ++q) *(v2u *)&Vt[q][v_k4 + e][4 * v_g] = vp[q];
                }
            } else {
#pragma unroll
                for (int p = 0; p < PIECES; ++p) {
                    const int idx = tid + p * FA_THREADS;
                    const int key = idx / (D / 4), k4 = (idx % (D / 4)) * 4;
                    *(v4f *)(Kf + key * LDK + k4) = (v4f){kreg[p].x * k_scale, kreg[p].y * k_scale, kreg[p].z * k_scale, kreg[p].w * k_scale};
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    *(v4f *)(Vf + (v_k4 + e) * LDV + v_key) =
                        (v4f){vreg[0][e] * v_scale, vreg[1][e] * v_scale, vreg[2][e] * v_scale, vreg[3][e] * v_scale};
            }
            __syncthreads();
            if (j0 + KEYS < kmax) {  // in flight during the matrix instructions below
                fetch(j0 + KEYS);
                k_code = ktab[j0 / KEYS + 1];
                v_code = vtab[j0 / KEYS + 1];
            }

            if (j0 < wave_kmax) {  // uniform per wavefront: tiles wholly above the causal diagonal are skipped
                // S^T = K Q^T: register r of tile kt holds key 32 kt + 8 (r / 4) + 4 half + r % 4 against this lane's row
                v16f S[KT];
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) S[kt][r] = 0.f;
                if (WIDE) {  // instruction w of eight elements: element 4 half + w of both operands
#pragma unroll 1
                    for (int e8 = 0; e8 < D; e8 += 8) {
                        v4f qx = *(const v4f *)(qrow + e8 + 4 * half), kx[KT];
                        qx.x *= qf_scale; qx.y *= qf_scale; qx.z *= qf_scale; qx.w *= qf_scale;
#pragma unroll
                        for (int kt = 0; kt < KT; ++kt) kx[kt] = *(const v4f *)(Kf + (32 * kt + c) * LDK + e8 + 4 * half);
#pragma unroll
                        for (int w = 0; w < 4; ++w)
#pragma unroll
                            for (int kt = 0; kt < KT; ++kt) S[kt] = __builtin_amdgcn_mfma_f32_32x32x2f32(kx[kt][w], qx[w] * q_scale, S[kt], 0, 0, 0);
                    }
                } else
#pragma unroll
                for (int ks = 0; ks < D / 16; ++ks) {
                    f16x8 kf[KT][2];
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                        for (int p = 0; p < 2; ++p)
                            kf[kt][p] = __builtin_bit_cast(f16x8, *(const v4u *)&Ks[p][32 * kt + c][ks * 16 + half * 8]);
#pragma unroll
                    for (int q = 0; q < 3; ++q)
#pragma unroll
                        for (int kt = 0; kt < KT; ++kt)
                            S[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kt][PA_[q]], __builtin_bit_cast(f16x8, qp[ks][PB_[q]]), S[kt], 0, 0, 0);
                }

                // what an accumulated score is to be multiplied by (the bounds: a score that f32 does not hold, or that is next to nothing)
                const float s_unit = exp2_int(min(max(-(ek + eq), -ROW_EXP_MAX), ROW_EXP_MAX));
                // softmax of this lane's row, in the lane: half of the trip's keys here, half in lane ^ 32
                float sc[16 * KT];
                float m_tile = -INFINITY;
                if (j0 + KEYS <= wave_kfull) {  // uniform per wavefront: every key of the trip is visible to every row
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            sc[16 * kt + r] = S[kt][r] * s_unit;
                            m_tile = fmaxf(m_tile, sc[16 * kt + r]);
                        }
                } else {
#pragma unroll
                    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int j = j0 + 32 * kt + 8 * (r >> 2) + 4 * half + (r & 3);
                            const bool valid = j < L && (!a.causal || j <= my_pos);
                            sc[16 * kt + r] = valid ? S[kt][r] * s_unit : -INFINITY;
                            m_tile = fmaxf(m_tile, sc[16 * kt + r]);
                        }
                }
                m_tile = fmaxf(m_tile, __shfl_xor(m_tile, 32, 64));
                const float m_new = fmaxf(m_run, m_tile);
                const float m_ref = m_new > -INFINITY ? m_new : 0.f;  // nothing visible yet: every weight below is exp2(-inf) = 0
                const float alpha = fast_exp2(m_run - m_ref);
                m_run = m_new;
                float psum = 0.f;
#pragma unroll
                for (int r = 0; r < 16 * KT; ++r) {
                    sc[r] = fast_exp2(sc[r] - m_ref);
                    psum += sc[r];
                }
                l_run = fmaf(l_run, alpha, psum);
                // the tile's largest contribution is 2^(m_tile - ev), times a value's 2^15; its weight goes in as 2^FA_P_EXP or less
                const float o_new = fmaxf(o_run, m_tile - (float)ev), o_ref = o_new > -INFINITY ? o_new : 0.f;
                const float o_alpha = fast_exp2(o_run - o_ref), p_scale = fast_exp2(fminf(m_ref - (o_ref + (float)(ev - FA_P_EXP)), 120.f));
                o_run = o_new;
#pragma unroll
                for (int t = 0; t < DT; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) O[t][r] *= o_alpha;

                // O^T += V^T P^T: P^T is this lane's weights, already where the B operand wants them
                // (registers 8 ks .. 8 ks + 7 are the keys at positions 16 ks + 8 half .. + 7 of V^T)
                if (WIDE) {
#pragma unroll
                    for (int g = 0; g < 4 * KT; ++g) {  // registers 4 g .. 4 g + 3: keys 8 g + 4 half .. + 3
                        v4f vx[DT];
#pragma unroll
                        for (int t = 0; t < DT; ++t) vx[t] = *(const v4f *)(Vf + (32 * t + c) * LDV + 8 * g + 4 * half);
#pragma unroll
                        for (int w = 0; w < 4; ++w)
#pragma unroll
                            for (int t = 0; t < DT; ++t) O[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx[t][w], sc[4 * g + w] * p_scale, O[t], 0, 0, 0);
                    }
                } else
#pragma unroll
                for (int ks = 0; ks < KEYS / 16; ++ks) {
                    f16x8 pf[2];
                    {
                        v2u lo[2], hi[2];
                        fa_split4((v4f){sc[8 * ks], sc[8 * ks + 1], sc[8 * ks + 2], sc[8 * ks + 3]}, p_scale, lo);
                        fa_split4((v4f){sc[8 * ks + 4], sc[8 * ks + 5], sc[8 * ks + 6], sc[8 * ks + 7]}, p_scale, hi);
#pragma unroll
                        for (int p = 0; p < 2; ++p) pf[p] = __builtin_bit_cast(f16x8, (v4u){lo[p].x, lo[p].y, hi[p].x, hi[p].y});
                    }
                    f16x8 vf[DT][2];
#pragma unroll
                    for (int t = 0; t < DT; ++t)
#pragma unroll
                        for (int p = 0; p < 2; ++p)
                            vf[t][p] = __builtin_bit_cast(f16x8, *(const v4u *)&Vt[p][32 * t + c][ks * 16 + half * 8]);
#pragma unroll
                    for (int q = 0; q < 3; ++q)
#pragma unroll
                        for (int t = 0; t < DT; ++t)
                            O[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t][PA_[q]], pf[PB_[q]], O[t], 0, 0, 0);
                }
            }
            __syncthreads();
        }

        const float l = l_run + __shfl_xor(l_run, 32, 64);
        // O in the units of the weights' sum; in two steps, neither of which leaves f32's range where the result does not
        const float o_unit = o_run > -INFINITY ? fast_exp2(o_run - m_run) : 0.f, p_unit = exp2_int(-FA_P_EXP);
        const int i = q0 + my_row / NREP;
        if (i >= a.s) return;
        if (PART) {
            const size_t n = (((size_t)bb * a.s + i) * a.hq + (size_t)hk * NREP + my_row % NREP) * (gridDim.z / a.b) + key_part;
            if (half == 0) {
                a.part_ml[2 * n] = m_run;
                a.part_ml[2 * n + 1] = l;
            }
#pragma unroll
            for (int t = 0; t < DT; ++t)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *(v4f *)(a.part + n * D + 32 * t + 8 * g + 4 * half) =
                        v4f{O[t][4 * g] * p_unit * o_unit, O[t][4 * g + 1] * p_unit * o_unit, O[t][4 * g + 2] * p_unit * o_unit, O[t][4 * g + 3] * p_unit * o_unit};
            return;
        }
        // out = ctx / (sum + 1e-9), self_attention.rs:670-676; [B,S,Hq,D]
        const float inv = p_unit / (l + 1e-9f);
        float *row = a.out + (((size_t)bb * a.s + i) * a.hq + (size_t)hk * NREP + my_row % NREP) * D;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *(v4f *)(row + 32 * t + 8 * g + 4 * half) =
                    v4f{O[t][4 * g] * inv * o_unit, O[t][4 * g + 1] * inv * o_unit, O[t][4 * g + 2] * inv * o_unit, O[t][4 * g + 3] * inv * o_unit};
    };
    if (wide) rows(std::true_type{});
    else rows(std::false_type{});
}

// The parts of a row's keys together, in part order; a thread takes four elements of a (position, head) row.  SPLIT: a workgroup has the whole
// row of a position and leaves it split, with an exponent of its own.
template <bool SPLIT>
__global__ __launch_bounds__(1024) void merge_parts_kernel(AttnPrefillArgs a, int parts) {
    const int per_pos = a.hq * a.d / 4, at = (int)(blockIdx.y * blockDim.x + threadIdx.x), tid = threadIdx.x;
    const size_t pos = (size_t)blockIdx.z * a.s + blockIdx.x;
    v4f o = {0.f, 0.f, 0.f, 0.f};
    if (at < per_pos) {
        const int head = at * 4 / a.d, e = at * 4 % a.d;
        const size_t n0 = (pos * a.hq + head) * parts;
        float m = -INFINITY;
        for (int p = 0; p < parts; ++p) m = fmaxf(m, a.part_ml[2 * (n0 + p)]);
        const float ref = m > -INFINITY ? m : 0.f;
        float l = 0.f;
#pragma unroll 4
        for (int p = 0; p < parts; ++p) {
            const float w = fast_exp2(a.part_ml[2 * (n0 + p)] - ref);
            const v4f x = *(const v4f *)(a.part + (n0 + p) * a.d + e);
            l = fmaf(w, a.part_ml[2 * (n0 + p) + 1], l);
            o.x = fmaf(w, x.x, o.x); o.y = fmaf(w, x.y, o.y); o.z = fmaf(w, x.z, o.z); o.w = fmaf(w, x.w, o.w);
        }
        const float inv = 1.0f / (l + 1e-9f);
        o = v4f{o.x * inv, o.y * inv, o.z * inv, o.w * inv};
    }
    float *row = a.out + pos * a.hq * a.d;
    if (!SPLIT) {
        if (at < per_pos) *(v4f *)(row + at * 4) = o;
        return;
    }
    const v4f all[1] = {o};
    leave_row<1>(all, per_pos * 4, row, a.out_exp + pos);
}

// Parts the keys are cut into where the blocks of queries leave compute units idle: at least 128 keys each (two trips of the loop; a part costs
// its start and its share of the pass that merges them), two workgroups per compute unit, 32 at most.
static int fa_key_parts(int num_cus, int blocks, int keys) {
    const int room = 2 * num_cus / (blocks > 0 ? blocks : 1), most = (keys + 127) / 128;
    const int n = room < most ? room : most;
    return n < 2 ? 1 : n < 32 ? n : 32;
}

// At most fa_key_parts' parts; a block of queries holds FA_ROWS rows, so parts times rows stay below two blocks per compute unit.
size_t attn_prefill_workspace(const lumen_ctx *ctx, int b, int s, int hq, int hkv, int d, int max_seq) {
    if (d != 64 && d != 128) return 0;
    const int trip = FA_KEYS * (d == 64 ? 2 : 1);
    const size_t most = std::min((max_seq + 127) / 128, 32);
    const size_t rows = most < 2 ? 0 : std::min(most * b * s * hq, (size_t)2 * ctx->num_cus * FA_ROWS);
    return 2 * (size_t)b * hkv * ((max_seq + trip - 1) / trip) + rows * (d + 2);
}

// Query heads of a KV group that share a workgroup, the grid of blocks of queries, and how the keys are cut.
struct FaPlan {
    int nrep, parts, key_chunk;
    dim3 grid;
};
static FaPlan fa_plan(int num_cus, const AttnPrefillArgs &a) {
    FaPlan p = {a.hq / a.hkv, 1, 0, dim3(1)};
    if (!(p.nrep == 1 || p.nrep == 2 || p.nrep == 4 || p.nrep == 8)) p.nrep = 1;  // any other group size: one query head per grid row
    const int L = a.past_len + a.s, trip = FA_KEYS * (a.d == 64 ? 2 : 1);
    p.grid = dim3((a.s + FA_ROWS / p.nrep - 1) / (FA_ROWS / p.nrep), a.hq / p.nrep, a.b);
    p.parts = fa_key_parts(num_cus, (int)(p.grid.x * p.grid.y * p.grid.z), L);
    if (p.parts > 1) {
        p.key_chunk = ((L + p.parts - 1) / p.parts + trip - 1) / trip * trip;
        p.parts = (L + p.key_chunk - 1) / p.key_chunk;
    }
    return p;
}
static bool merge_splits_rows(const AttnPrefillArgs &a, const FaPlan &p) { return p.parts > 1 && a.hq * a.d / 4 <= 1024; }

template <int D>
static int launch_fa_d(lumen_ctx *ctx, const AttnPrefillArgs &a_in) {
    AttnPrefillArgs a = a_in;
    const FaPlan plan = fa_plan(ctx->num_cus, a);
    const int nrep = plan.nrep, parts = plan.parts, L = a.past_len + a.s, trip = FA_KEYS * (D == 64 ? 2 : 1);
    if (nrep != a.hq / a.hkv) a.kv_div = a.hq / a.hkv;  // KV head of a grid row = head / n_rep
    dim3 grid = plan.grid;
    a.key_chunk = plan.key_chunk;
    const int tile = trip, tiles = (L + tile - 1) / tile;
    const size_t rows = parts > 1 ? (size_t)a.b * a.s * a.hq * parts : 0, codes = 2 * (size_t)a.b * a.hkv * tiles;
    const size_t need = codes + rows * (D + 2);
    if (!a.ws || need > a.ws_floats) LUMEN_FAIL(LUMEN_ERR_INVALID, "prompt attention: workspace of %zu floats, %zu wanted", a.ws_floats, need);
    a.part = a.ws;
    a.part_ml = a.part + rows * D;
    int *kv_tiles = (int *)(a.part_ml + 2 * rows);
    a.kv_tiles = kv_tiles;
    hipLaunchKernelGGL((kv_tiles_kernel<D, FA_KEYS * (D == 64 ? 2 : 1)>), dim3(tiles, a.b * a.hkv), dim3(256), 0, ctx->stream, a.k_cache, a.v_cache,
                       a.max_seq, L, kv_tiles);
    grid.z *= parts;
#define LAUNCH_FA(NR)                                                                                                                        \
    do {                                                                                                                                     \
        if (parts > 1) hipLaunchKernelGGL((attn_prefill_f16x2_kernel<D, NR, (D == 64 ? 2 : 1), true>), grid, dim3(FA_THREADS), 0, ctx->stream, a); \
        else hipLaunchKernelGGL((attn_prefill_f16x2_kernel<D, NR, (D == 64 ? 2 : 1), false>), grid, dim3(FA_THREADS), 0, ctx->stream, a);     \
    } while (0)
    switch (nrep) {
        case 1: LAUNCH_FA(1); break;
        case 2: LAUNCH_FA(2); break;
        case 4: LAUNCH_FA(4); break;
        default: LAUNCH_FA(8); break;
    }
#undef LAUNCH_FA
    const int pieces = a.hq * D / 4;  // of a position's row
    bool split_done = false;
    if (parts > 1) {
        if (a.out_exp && merge_splits_rows(a, plan)) {
            hipLaunchKernelGGL(merge_parts_kernel<true>, dim3(a.s, 1, a.b), dim3((pieces + 63) / 64 * 64), 0, ctx->stream, a, parts);
            split_done = true;
        } else {
            hipLaunchKernelGGL(merge_parts_kernel<false>, dim3(a.s, (pieces + 255) / 256, a.b), dim3(256), 0, ctx->stream, a, parts);
        }
    }
    LUMEN_CHECK_LAUNCH();
    if (a.out_exp && !split_done) return launch_split_rows(ctx, a.out, a.b * a.s, a.hq * D, a.out, a.out_exp);
    return LUMEN_OK;
}

// Against the row loop (one workgroup per position and head or two: its walk over the keys is a chain, and every position repeats it): where the
// cache is long, and where positions times keys are many.  Measured, row loop / this with its pass over the keys, us: 32 heads of 64, 4 KV heads,
// 96 first positions 10.3 / 16.4, 160 16.7 / 20.6, 192 20.9 / 21.2, 207 22.9 / 22.1, 64 behind 301 18.5 / 18.6, 32 behind 600 18.8 / 18.0, 2 behind 1000
// 18.4 / 17.0, 64 behind 2900 102 / 28; 16 heads of 64, 8 KV heads, 192 14.0 / 19.9, 256 21.1 / 20.1; 16 of 128, 8 KV heads, 207 25.7 / 27.7.  A KV
// head for every head (no rows shared): 32 of 64 160 21.2 / 22.8, 192 26.2 / 23.4, 71 of 64 96 21.7 / 19.8, 128 29.4 / 22.0; 32 of 128 96 19.6 / 22.4,
// 128 26.8 / 27.1, 64 behind 301 40 / 25, 2 behind 600 35 / 23, 2 behind 301 14 / 20.
bool attn_prefill_mfma_supported(const AttnPrefillArgs &a) {
    const long L = (long)a.past_len + a.s, work = (long)a.b * a.s * a.hq * (a.past_len + a.s / 2) * a.d;
    return (a.d == 64 || a.d == 128) && (L * a.d >= 64000 || work >= (a.hq == a.hkv ? 28000000 : 40000000));
}

bool attn_prefill_splits_rows(const lumen_ctx *ctx, const AttnPrefillArgs &a) {
    return attn_prefill_mfma_supported(a) && merge_splits_rows(a, fa_plan(ctx->num_cus, a));
}

int launch_attn_prefill_mfma(lumen_ctx *ctx, const AttnPrefillArgs &a) {
    if (a.d == 64) return launch_fa_d<64>(ctx, a);
    if (a.d == 128) return launch_fa_d<128>(ctx, a);
    LUMEN_FAIL(LUMEN_ERR_UNSUPPORTED, "matrix-core prefill attention: head_dim=%d (supported 64, 128)", a.d);
}

LUMEN_DEFINE_WARM(prefill_attention)
