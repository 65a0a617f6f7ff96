// C[M,N] = A[M,K] W[N,K]^T at f32 accuracy on the f16 matrix cores, for the prompt passes of the models.
//
// gemm.hip takes an f32 product as six bf16 products of three-part values.  f16 has three bits more per part, so two parts
// (f16_split.h) and three products -- hi hi, hi lo, lo hi -- carry 2^-22 of every product, and a bf16-stored weight is one
// f16 value: two products.  Half (two thirds) of the matrix instructions, a third less LDS and split arithmetic.  f16's
// range is what it costs: a row of either operand carries an exponent (A's is found by the kernel that makes A, W's once when a
// weight is set), so only callers that know them take this path; the others keep gemm.hip.
//
// A arrives as split rows (f16_split.h); W is split on its way into LDS.
//
// What bounds it: the matrix pipes, whose clock the chip lowers under them (a library bf16 product of 8192^3 runs at 1.16 PFLOP/s here; this
// kernel's 256 x 256 tiles issue 0.9 to 1.0), and with few rows the start of a launch and the partial products of K splits.
// Useful TFLOP/s, before (three bf16 parts) and after, with the error against a float64 product (relative, over all elements):
//   3968 x 11264 x 2048 f32   195 -> 297   6.8e-7 -> 4.9e-7      2048 x 8192 x 2048 bf16   318 -> 510   4.6e-7 -> 4.1e-7
//   3968 x  2048 x 5632 f32   183 -> 302   8.1e-7 -> 5.7e-7       509 x 4096 x 11008 bf16  251 -> 360   5.7e-7 -> 4.8e-7
//    512 x 11264 x 2048 f32   148 -> 204   5.0e-7 -> 3.4e-7       128 x 11264 x 2048 f32   125 -> 151   3.2e-7 -> 2.4e-7
//     64 x   512 x   64 f32   (1 piece)    1.3e-7 -> 1.1e-7       300 x 1024 x  256 f32    (4 pieces)   1.8e-7 -> 1.5e-7
// The error is smaller because half as many sums are rounded.
#include "f16_split.h"

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));



// In LDS a slice of 32 k is four planes of 8 k, [k / 8][row][8 f16] with two rows of padding: an operand read of 32 rows is 512
// contiguous bytes, and a staging write of two rows' pieces (the planes start 32 bytes apart, modulo the banks) covers all banks once.
// SCALED: the sums are in units of the rows' exponents.
template <int EPI, bool PARTIAL, bool SCALED, int FI, int FJ>
__device__ __forceinline__ void store_tiles(const GemmArgs &a, const v16f (&acc)[FI][FJ], const int *ae_tile, const int *we_tile, int bm, int bn, int wrow,
                                            int wcol, int lane) {
    const int M = a.M, N = a.N;
    float *part = PARTIAL ? a.part + (size_t)blockIdx.z * M * N : nullptr;
    int we[FJ];
#pragma unroll
    for (int j = 0; j < FJ; ++j) we[j] = we_tile[wcol + j * 32 + (lane & 31)];
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int trow = wrow + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3), row = bm + trow;
            const int ae = ae_tile[trow];
#pragma unroll
            for (int j = 0; j < FJ; ++j) {
                const int col = bn + wcol + j * 32 + (lane & 31);
                const float v = SCALED ? ldexpf(acc[i][j][r], -(ae + we[j])) : acc[i][j][r];
                if (PARTIAL) {
                    if (row < M && col < N) part[(size_t)row * N + col] = v;
                } else if (EPI == EPI_SWIGLU) {
                    const float up = __shfl_xor(v, 1, 64);
                    if (!(col & 1) && row < M && col < N) a.C[(size_t)row * (N >> 1) + (col >> 1)] = v / (1.0f + expf(-v)) * up;
                } else if (row < M && col < N) {
                    const size_t o = (size_t)row * N + col;
                    a.C[o] = (EPI == EPI_RESIDUAL) ? fmaf(a.alpha, v, a.residual[o]) : v;
                }
            }
        }
}

// A wavefront's share of a tile that meets a row of either operand pairs cannot hold: f32 matrix instructions on the f32 values, straight from memory;
// a row of A that is pairs all the same is put together (hi + lo is exact).  32 x 64 of C at a time, 16 of K in flight: the f32 instruction takes
// five times the pairs' three, so that is what bounds it.
template <bool WBF16, int EPI, bool PARTIAL, int FI, int FJ>
__device__ __forceinline__ void wide_tiles(const GemmArgs &a, const int *ae_tile, const int *we_tile, int bm, int bn, int wrow, int wcol, int lane, int k0, int k1) {
    const int c = lane & 31, half = lane >> 5, K = a.K;
    static_assert(FJ % 2 == 0, "two tiles side by side");
#pragma unroll 1
    for (int at = 0; at < FI * FJ / 2; ++at) {
        const int i = at / (FJ / 2), col0 = wcol + at % (FJ / 2) * 64;
        const char *wp[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) wp[j] = (const char *)a.W + (size_t)min(bn + col0 + j * 32 + c, a.N - 1) * K * (WBF16 ? 2 : 4);
        const int row = min(bm + wrow + i * 32 + c, a.M - 1), code = ae_tile[wrow + i * 32 + c];
        const bool plain = is_wide(code);
        const float unit = plain ? 1.f : exp2_int(-code);
        const char *ap = (const char *)a.a_split + (size_t)row * K * 4;
        v16f acc[1][2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][j][r] = 0.f;
        // elements 8 t + 4 half .. + 3 of 16 k (both operands of instruction w of eight elements: element 4 half + w)
        v2u x[2][2][2];
        v4u w[2][2][2];
        auto fetch = [&](int set, int k) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int e = 8 * t + 4 * half;
                x[set][t][0] = *(const v2u *)(ap + (size_t)k * 4 + (plain ? e * 4 : e * 2));
                x[set][t][1] = *(const v2u *)(ap + (size_t)k * 4 + (plain ? e * 4 + 8 : 32 + e * 2));
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (WBF16) {
                        const v2u b = *(const v2u *)(wp[j] + (size_t)(k + e) * 2);
                        w[set][t][j] = v4u{b.x << 16, b.x & 0xffff0000u, b.y << 16, b.y & 0xffff0000u};
                    } else {
                        w[set][t][j] = *(const v4u *)(wp[j] + (size_t)(k + e) * 4);
                    }
                }
            }
        };
        auto product = [&](int set) {
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const unsigned b[4] = {x[set][t][0].x, x[set][t][0].y, x[set][t][1].x, x[set][t][1].y};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f16x2_t hi = __builtin_bit_cast(f16x2_t, b[e >> 1]), lo = __builtin_bit_cast(f16x2_t, b[2 + (e >> 1)]);
                    const float v = plain ? __uint_as_float(b[e]) : ((float)hi[e & 1] + (float)lo[e & 1]) * unit;
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[0][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, __uint_as_float(w[set][t][j][e]), acc[0][j], 0, 0, 0);
                }
            }
        };
        if (k0 < k1) fetch(0, k0);
        for (int k = k0; k < k1; k += 32) {  // (whole slices of 64 of K: the launcher's condition)
            fetch(1, k + 16);
            product(0);
            fetch(0, min(k + 32, k1 - 16));
            product(1);
        }
        store_tiles<EPI, PARTIAL, false>(a, acc, ae_tile, we_tile, bm, bn, wrow + i * 32, col0, lane);
    }
}

// WM x WN wavefronts, FI x FJ tiles of 32 x 32 each; slices of HK of K in a ring of RING in LDS, D slices in flight from memory.  All operands of a
// slice are in registers before its first matrix instruction, so that the barrier and the LDS reads after it cost no time
// on the matrix pipe (operands read after the barrier: 260 instead of 297 TFLOP/s at 3968 x 11264 x 2048); every LDS access is
// conflict-free (the counter reads 0).  bf16 weights: slices of 32, because a 16-deep one would read 32 bytes of a row.
template <bool WBF16, int EPI, bool PARTIAL, int FI, int FJ, int WM, int WN, int DEPTH>
__global__ __launch_bounds__(64 * WM * WN, (FI * FJ > 8 ? 1 : 2)) void gemm_f16x2_kernel(GemmArgs a) {
    constexpr int T = 64 * WM * WN;
    constexpr int HK = WBF16 ? 32 : 16, KS = HK / 16, RING = WBF16 ? 3 : 4;
    constexpr int D = DEPTH;                          // slices in flight from memory
    constexpr int PW = WBF16 ? 1 : 2;                 // f16 parts of a weight
    constexpr int TM = 32 * FI * WM, TN = 32 * FJ * WN;
    constexpr int AST = TM * HK / 4 / T;              // 16-byte pieces of A (both parts) per thread and slice
    constexpr int WST = TN * HK / (WBF16 ? 8 : 4) / T;  // ... of W
    constexpr int NPROD = WBF16 ? 2 : 3;
    constexpr int APAD = WBF16 ? 1 : 2, WPAD = WBF16 ? 2 : 4;
    constexpr int GROUPS = KS * FJ;                   // groups of FI NPROD matrix instructions of a slice
    __shared__ __align__(16) uint16_t As[RING][KS][2][2][TM + APAD][8];   // [slot][k / 16][part][k half][row]
    __shared__ __align__(16) uint16_t Ws[RING][PW][KS][2][TN + WPAD][8];
    __shared__ int ae_tile[TM], we_tile[TN], wide_any[WM * WN];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wrow = wave / WN * (32 * FI), wcol = wave % WN * (32 * FJ);
    const int bm = blockIdx.y * TM, bn = blockIdx.x * TN;
    const int M = a.M, N = a.N, K = a.K;
    // this workgroup's slices: whole pieces of 64 of K (the launcher's condition on K)
    const int pieces = K / 64, per = (pieces + (int)gridDim.z - 1) / (int)gridDim.z;
    const int p0 = min((int)blockIdx.z * per, pieces), s0 = p0 * (64 / HK), n = min(per, pieces - p0) * (64 / HK);

    v16f acc[FI][FJ];
#pragma unroll
    for (int i = 0; i < FI; ++i)
#pragma unroll
        for (int j = 0; j < FJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // A piece i of this thread: row (tid + T i) / (HK / 4), piece (tid + T i) % (HK / 4) of the row's 4 HK bytes; f32 weights: row (tid + T i) / 4,
    // k 4 * (tid % 4); bf16 weights: row (tid + T i) / 4, k 8 * (tid % 4).  Rows past the end are clamped (their products are never stored).
    const char *abase = (const char *)a.a_split + ((size_t)bm * K + (size_t)s0 * HK) * 4;
    const char *wbase = (const char *)a.W + ((size_t)bn * K + (size_t)s0 * HK) * (WBF16 ? 2 : 4);
    unsigned aoff[AST], woff[WST];
    float ws[WST];
#pragma unroll
    for (int i = 0; i < AST; ++i) {
        const int idx = tid + i * T;
        aoff[i] = (unsigned)(min(bm + idx / (HK / 4), M - 1) - bm) * (unsigned)K * 4u + (unsigned)(idx % (HK / 4)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < WST; ++i) {
        const int row = min(bn + ((tid + i * T) >> 2), N - 1);
        woff[i] = (unsigned)(row - bn) * (unsigned)K * (WBF16 ? 2u : 4u) + (unsigned)(tid & 3) * 16u;
        ws[i] = exp2_int(a.w_exp[row]);
    }
    v4u va[D][AST], vw[D][WST];
    auto fetch_a = [&](int r, int i, int s) { va[r][i] = *(const v4u *)(abase + (size_t)s * (HK * 4) + aoff[i]); };
    auto fetch_w = [&](int r, int i, int s) { vw[r][i] = *(const v4u *)(wbase + (size_t)s * 64 + woff[i]); };
    auto stage_a = [&](int r, int slot, int i) {
        const int idx = tid + i * T, rem = idx % (HK / 4);
        *(v4u *)&As[slot][rem >> 2][(rem >> 1) & 1][rem & 1][idx / (HK / 4)][0] = va[r][i];
    };
    auto stage_w = [&](int r, int slot, int i) {
        const int row = (tid + i * T) >> 2;
        if (WBF16) {
            const unsigned src[4] = {vw[r][i].x, vw[r][i].y, vw[r][i].z, vw[r][i].w};
            unsigned dst[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const f16x2_t h = {(_Float16)fmaf(__uint_as_float(src[e] << 16), ws[i], 0.f), (_Float16)fmaf(__uint_as_float(src[e] & 0xffff0000u), ws[i], 0.f)};
                dst[e] = __builtin_bit_cast(unsigned, h);
            }
            *(v4u *)&Ws[slot][0][(tid & 3) >> 1][tid & 1][row][0] = v4u{dst[0], dst[1], dst[2], dst[3]};
        } else {
            unsigned h0, l0, h1, l1;
            split_pair(__uint_as_float(vw[r][i].x), __uint_as_float(vw[r][i].y), ws[i], h0, l0);
            split_pair(__uint_as_float(vw[r][i].z), __uint_as_float(vw[r][i].w), ws[i], h1, l1);
            *(v2u *)&Ws[slot][0][0][(tid & 3) >> 1][row][(tid & 1) * 4] = v2u{h0, h1};
            *(v2u *)&Ws[slot][PW - 1][0][(tid & 3) >> 1][row][(tid & 1) * 4] = v2u{l0, l1};
        }
    };
    const int c = lane & 31, gk = lane >> 5;
    f16x8 af[2][FI][2], wf[2][FJ][PW];  // operands of 16 k, two sets
    auto read_a = [&](int set, int slot, int ks, int i) {
#pragma unroll
        for (int p = 0; p < 2; ++p) af[set][i][p] = __builtin_bit_cast(f16x8, *(const v4u *)&As[slot][ks][p][gk][wrow + i * 32 + c][0]);
    };
    auto read_w = [&](int set, int slot, int ks, int j) {
#pragma unroll
        for (int p = 0; p < PW; ++p) wf[set][j][p] = __builtin_bit_cast(f16x8, *(const v4u *)&Ws[slot][p][ks][gk][wcol + j * 32 + c][0]);
    };
    // Slice s is multiplied from registers; meanwhile its later operands and the first ones of slice s + 1 are read from LDS, slice s + 2 is staged
    // (slot and values free since the barrier before the last) and slice s + 2 + D requested.  Nothing in it is conditional: past the end
    // the last slice is requested again, staged and not used.
    auto slice = [&](int set0, int r, int s, int slot, int slot1, int slot2) {
        const int next = min(s + 2 + D, n - 1);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int set = (set0 + ks) & 1;
            const bool over = ks + 1 == KS;
#pragma unroll
            for (int j = 0; j < FJ; ++j) {
                constexpr int PA_[3] = {1, 0, 0}, PW_[3] = {0, 1, 0};  // products by ascending size: lo hi, hi lo, hi hi (bf16 weights: lo w, hi w)
#pragma unroll
                for (int q = 0; q < NPROD; ++q)
#pragma unroll
                    for (int i = 0; i < FI; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[set][i][WBF16 ? 1 - q : PA_[q]], wf[set][j][WBF16 ? 0 : PW_[q]], acc[i][j], 0, 0, 0);
                if (j < FI) read_a(set ^ 1, over ? slot1 : slot, over ? 0 : ks + 1, j);
                read_w(set ^ 1, over ? slot1 : slot, over ? 0 : ks + 1, j);
                const int g = ks * FJ + j;
#pragma unroll
                for (int i = 0; i < AST; ++i)
                    if (i * GROUPS / AST == g) {
                        stage_a(r, slot2, i);
                        fetch_a(r, i, next);
                    }
#pragma unroll
                for (int i = 0; i < WST; ++i)
                    if (i * GROUPS / WST == g) {
                        stage_w(r, slot2, i);
                        fetch_w(r, i, next);
                    }
                if (FI == 4) {  // the group's order: everything else one by one in the shadows of its matrix instructions
                    constexpr int NM = FI * NPROD, VPM = 24 / NM, NR = 2 + PW;
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // a matrix instruction,
                        __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);  // vector ALU,
                        if (k < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           // an LDS read,
                        else if (k < NR + 3) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // an LDS write
                        else if (k < NR + 5) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // or a load
                    }
                }
            }
        }
        __syncthreads();
    };
    static_assert(D % 2 == 0 && (64 / HK) % D == 0, "a piece of K is a whole number of turns of the register sets");
    static_assert(FI <= FJ, "a group of matrix instructions per row tile whose operands are read under it");
    int wide = 0;
    for (int i = tid; i < TM; i += T) wide |= is_wide(ae_tile[i] = a.a_exp[min(bm + i, M - 1)]);
    for (int i = tid; i < TN; i += T) wide |= is_wide(we_tile[i] = a.w_exp[min(bn + i, N - 1)]);
    auto fetch = [&](int r, int s) {
#pragma unroll
        for (int i = 0; i < AST; ++i) fetch_a(r, i, min(s, n - 1));
#pragma unroll
        for (int i = 0; i < WST; ++i) fetch_w(r, i, min(s, n - 1));
    };
    auto stage = [&](int r, int slot) {
#pragma unroll
        for (int i = 0; i < AST; ++i) stage_a(r, slot, i);
#pragma unroll
        for (int i = 0; i < WST; ++i) stage_w(r, slot, i);
    };
    if (n > 0) {
        // slice 2 + r of the rest goes through register set r % D; the first two through sets 0 and 1
        fetch(0, 0);
        fetch(1, 1);
#pragma unroll
        for (int r = 2; r < D; ++r) fetch(r, 2 + r);
        stage(0, 0);
        fetch(0, 2);
        stage(1, 1);
        fetch(1, 3);
    }
    wide = __any(wide);
    if (lane == 0) wide_any[wave] = wide;
    __syncthreads();
    wide = 0;
#pragma unroll
    for (int w = 0; w < WM * WN; ++w) wide |= wide_any[w];
    if (wide) {
        wide_tiles<WBF16, EPI, PARTIAL, FI, FJ>(a, ae_tile, we_tile, bm, bn, wrow, wcol, lane, s0 * HK, (s0 + n) * HK);
        return;
    }
    if (n > 0) {
#pragma unroll
        for (int i = 0; i < FI; ++i) read_a(0, 0, 0, i);
#pragma unroll
        for (int j = 0; j < FJ; ++j) read_w(0, 0, 0, j);
        int slot = 0;
        auto after = [](int x) { return x + 1 == RING ? 0 : x + 1; };
        for (int s = 0; s < n; s += D) {
#pragma unroll
            for (int r = 0; r < D; ++r) {
                const int s1 = after(slot);
                slice(KS == 1 ? r & 1 : 0, r, s + r, slot, s1, after(s1));
                slot = s1;
            }
        }
    }
    store_tiles<EPI, PARTIAL, true, FI, FJ>(a, acc, ae_tile, we_tile, bm, bn, wrow, wcol, lane);
}

// Few rows of A (f32 rows).  The product is bound by the weights, which are streamed once and go straight into operand registers: a lane takes
// two 16-byte pieces (bf16 weights: one) of its row per 32 of K, whose four lanes complete 64 bytes of every row, splits them there and multiplies
// them by v_mfma_f32_16x16x32_f16 with the MT row tiles of A.  A workgroup's four wavefronts take 16 columns of C each and share A: chunks of 128 of K
// lie in LDS in operand order, split on their way in, every row of a wavefront's share (EB blocks of 32 k) with an exponent of its own, found as it
// passes; the sums of a share are scaled and added in f32.  A workgroup that met a share with more than SF_SMALL small values (f16_split.h) per 32, or a
// marked row of W, takes its range again by f32 instructions on the f32 values, straight from memory (a choice per chunk costs every launch 4 %:
// the branch stands between a chunk's barrier and its first operands).  What bounds it: the loads in flight (four blocks of W per wavefront; eight cost the
// occupancy what they gained: 4096 x 12288, bf16, 3 rows 24 -> 27 us, 23 rows of f32 spilled) and the barrier per chunk.  Before (the f32
// instruction, 32 cycles per four of K instead of 32 or 48 per 32, or three bf16 products on whole tiles) and now, N x K, us:
//     f32 weights, 23 rows:  11264 x 2048 38.6 -> 33    2048 x 5632 22.8 -> 20.2    2560 x 2048 12.1 -> 10.3    6144 x 1024 16.6 -> 14.7
//     bf16, 3-32 rows:       12288 x 4096 38 -> 24-34   4096 x 4096 19 -> 13-16     22016 x 4096 72 -> 47-66    4096 x 11008 42 -> 27-35
// Error against 64 bits before and now, relative to the root mean square of C (f32 weights; half as many or fewer sums are rounded):
//     16 rows 11264 x 2048 4.1e-7 -> 1.4e-7    23 rows 2048 x 5632 2.9e-7 -> 1.5e-7    3 rows 1000 x 192 1.3e-7 -> 0.9e-7
#define SF_SMALL 2
#define SF_BLOCKS 4  // blocks of 32 k in a chunk, and of W in flight per wavefront
template <bool WBF16, int MT, int EPI, bool PARTIAL>
__global__ __launch_bounds__(256, 3) void gemm_f16x2_stream_kernel(GemmArgs a) {
    constexpr int PW = WBF16 ? 1 : 2, NPROD = WBF16 ? 2 : 3, WP = WBF16 ? 1 : 2;
    constexpr int EB = MT;          // blocks of a wavefront's share of a chunk of A: MT tiles x 4 blocks over 4 wavefronts
    constexpr int PIECES = 2 * MT;  // 16-byte pieces of A per thread and chunk
    __shared__ __align__(16) uint16_t As[2][SF_BLOCKS][MT][2][64][8];  // [half][block][tile][part][operand lane]
    __shared__ int ae[2][SF_BLOCKS / EB][MT][16];
    __shared__ int wide_any[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int M = a.M, N = a.N, K = a.K;
    const int bn = blockIdx.x * 64 + wave * 16;
    const int blocks = K / 32, per = (blocks + (int)gridDim.z - 1) / (int)gridDim.z;
    const int b0 = min((int)blockIdx.z * per, blocks), n = min(per, blocks - b0);
    const int col = bn + c, wrow = min(col, N - 1);
    const int w_code = a.w_exp[wrow], we = code_exponent(w_code);
    const float ws = exp2_int(we);
    int wide = __any(is_wide(w_code));
    const char *wp = (const char *)a.W + ((size_t)wrow * K + (size_t)b0 * 32) * (WBF16 ? 2 : 4) + g * 16;
    // this wavefront's share of a chunk of A: tile share_t, blocks share_b .. share_b + EB - 1; piece p of lane (row c, g): k 4 (4 p + g) of it
    const int share_t = MT == 2 ? wave >> 1 : 0, share_b = MT == 2 ? (wave & 1) * 2 : wave;
    const float *ap = a.A + (size_t)min(share_t * 16 + c, M - 1) * K + (size_t)b0 * 32 + share_b * 32 + g * 4;

    v4f sum[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) sum[t] = v4f{0.f, 0.f, 0.f, 0.f};
    v4u vw[SF_BLOCKS][WP];
    v4f va[PIECES];
    auto fetch_w = [&](int slot, int d) {
#pragma unroll
        for (int i = 0; i < WP; ++i) vw[slot][i] = __builtin_nontemporal_load((const v4u *)(wp + (size_t)min(d, n - 1) * (WBF16 ? 64 : 128) + i * 64));
    };
    auto fetch_a = [&](int d) {  // (past the end: the last k of the range, multiplied by nothing)
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            const int k = min(d * 32 + share_b * 32 + p * 16 + g * 4, n * 32 - 4) - share_b * 32 - g * 4;
            va[p] = *(const v4f *)(ap + k);
        }
    };
    auto stage_a = [&](int half) {
        unsigned m = 0, least = ~0u;  // (of magnitudes - 1: a zero is the largest)
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const unsigned u = magnitude_bits(va[p][i]);
                m = max(m, u);
                least = min(least, u - 1u);
            }
        m = max(m, (unsigned)__shfl_xor((int)m, 16, 64));
        m = max(m, (unsigned)__shfl_xor((int)m, 32, 64));
        const int e = row_exponent(m);
        const float s = exp2_int(e);
        const unsigned limit = small_limit(m);
        if (__any(least < limit - 1u)) {  // uniform
            int small = 0;
#pragma unroll
            for (int p = 0; p < PIECES; ++p)
#pragma unroll
                for (int i = 0; i < 4; ++i) small += is_small(magnitude_bits(va[p][i]), limit);
            small += __shfl_xor(small, 16, 64);
            small += __shfl_xor(small, 32, 64);
            wide |= __any(small > SF_SMALL * EB);
        }
        if (g == 0) ae[half][share_b / EB][share_t][c] = e;
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            unsigned h0, l0, h1, l1;
            split_pair(va[p].x, va[p].y, s, h0, l0);
            split_pair(va[p].z, va[p].w, s, h1, l1);
            // k 16 (p & 1) + 4 g of block share_b + p / 2.  An operand lane (row, q) holds k 4 q .. + 3 and 16 + 4 q .. + 3 (bf16 weights: 8 q .. + 7)
            const int q = WBF16 ? (p & 1) * 2 + (g >> 1) : g, at = WBF16 ? (g & 1) * 4 : (p & 1) * 4;
            *(v2u *)&As[half][share_b + p / 2][share_t][0][q * 16 + c][at] = v2u{h0, h1};
            *(v2u *)&As[half][share_b + p / 2][share_t][1][q * 16 + c][at] = v2u{l0, l1};
        }
    };
    if (n > 0) {
#pragma unroll
        for (int j = 0; j < SF_BLOCKS; ++j) fetch_w(j, j);
        fetch_a(0);
        stage_a(0);
    }
    __syncthreads();
    int half = 0;
    for (int d = 0; d < n; d += SF_BLOCKS, half ^= 1) {
        fetch_a(d + SF_BLOCKS);
#pragma unroll
        for (int e0 = 0; e0 < SF_BLOCKS; e0 += EB) {
            v4f acc[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = e0; j < e0 + EB; ++j) {
                if (d + j >= n) break;  // (uniform)
                f16x8 wf[PW];
                if (WBF16) {
                    const unsigned src[4] = {vw[j][0].x, vw[j][0].y, vw[j][0].z, vw[j][0].w};
                    unsigned dst[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const f16x2_t h = {(_Float16)fmaf(__uint_as_float(src[e] << 16), ws, 0.f), (_Float16)fmaf(__uint_as_float(src[e] & 0xffff0000u), ws, 0.f)};
                        dst[e] = __builtin_bit_cast(unsigned, h);
                    }
                    wf[0] = __builtin_bit_cast(f16x8, v4u{dst[0], dst[1], dst[2], dst[3]});
                } else {
                    unsigned h[4], l[4];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const v4u w = vw[j][WP == 2 ? i : 0];
                        split_pair(__uint_as_float(w.x), __uint_as_float(w.y), ws, h[2 * i], l[2 * i]);
                        split_pair(__uint_as_float(w.z), __uint_as_float(w.w), ws, h[2 * i + 1], l[2 * i + 1]);
                    }
                    wf[0] = __builtin_bit_cast(f16x8, v4u{h[0], h[1], h[2], h[3]});
                    wf[PW - 1] = __builtin_bit_cast(f16x8, v4u{l[0], l[1], l[2], l[3]});
                }
                fetch_w(j, d + j + SF_BLOCKS);
                f16x8 af[MT][2];
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int p = 0; p < 2; ++p) af[t][p] = __builtin_bit_cast(f16x8, *(const v4u *)&As[half][j][t][p][lane][0]);
                constexpr int PA_[3] = {1, 0, 0}, PW_[3] = {0, 1, 0};  // lo hi, hi lo, hi hi (bf16 weights: lo w, hi w)
#pragma unroll
                for (int q = 0; q < NPROD; ++q)
#pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t][WBF16 ? 1 - q : PA_[q]], wf[WBF16 ? 0 : PW_[q]], acc[t], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[t][r] += ldexpf(acc[t][r], -(ae[half][e0 / EB][t][4 * g + r] + we));
        }
        if (d + SF_BLOCKS < n) stage_a(half ^ 1);
        __syncthreads();
    }
    if (lane == 0) wide_any[wave] = wide;
    __syncthreads();
    if (wide_any[0] | wide_any[1] | wide_any[2] | wide_any[3]) {
#pragma unroll
        for (int t = 0; t < MT; ++t) sum[t] = v4f{0.f, 0.f, 0.f, 0.f};
        const float *arow[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) arow[t] = a.A + (size_t)min(t * 16 + c, M - 1) * K + (size_t)b0 * 32;
#pragma unroll 1
        for (int d = 0; d < n; ++d) {
            // instruction (i, e): element e of this lane's piece i of the block, of both operands
            v4f ax[MT][2];
            float w[8];
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i) ax[t][i] = *(const v4f *)(arow[t] + d * 32 + (WBF16 ? 8 * g + 4 * i : 16 * i + 4 * g));
#pragma unroll
            for (int i = 0; i < WP; ++i) {
                const v4u b = *(const v4u *)(wp + (size_t)d * (WBF16 ? 64 : 128) + i * 64);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (WBF16) {
                        w[2 * e] = __uint_as_float(b[e] << 16);
                        w[2 * e + 1] = __uint_as_float(b[e] & 0xffff0000u);
                    } else {
                        w[4 * i + e] = __uint_as_float(b[e]);
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int t = 0; t < MT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ax[t][e >> 2][e & 3], w[e], sum[t], 0, 0, 0);
        }
    }
    float *part = PARTIAL ? a.part + (size_t)blockIdx.z * M * N : nullptr;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = t * 16 + 4 * g + r;
            const float v = sum[t][r];
            if (PARTIAL) {
                if (row < M && col < N) part[(size_t)row * N + col] = v;
            } else if (EPI == EPI_SWIGLU) {
                const float up = __shfl_xor(v, 1, 64);
                if (!(col & 1) && row < M && col < N) a.C[(size_t)row * (N >> 1) + (col >> 1)] = v / (1.0f + expf(-v)) * up;
            } else if (row < M && col < N) {
                const size_t o = (size_t)row * N + col;
                a.C[o] = (EPI == EPI_RESIDUAL) ? fmaf(a.alpha, v, a.residual[o]) : v;
            }
        }
}

// ------------------------------------------------------------------------------------------ exponents, split rows
// One wavefront per row of W.  (The second pass over a row counts its small elements; it is paid once, when the weight is set.)
template <bool BF16>
__global__ __launch_bounds__(256) void row_exponents_kernel(const void *W, int rows, int cols, int row0, int step, int *exps) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (r >= rows) return;
    const size_t row = (size_t)row0 + (size_t)r * step;
    auto bits = [&](int k) { return BF16 ? (unsigned)(((const uint16_t *)W)[row * cols + k] & 0x7fffu) << 16 : magnitude_bits(((const float *)W)[row * cols + k]); };
    unsigned m = 0;
    for (int k = lane; k < cols; k += 64) m = max(m, bits(k));
    m = wave_umax(m);
    const unsigned limit = small_limit<BF16 ? 31u : 18u>(m);
    int small = 0;
    for (int k = lane; k < cols; k += 64) small += is_small(bits(k), limit);
    const bool wide = wave_sum((float)small) * (float)SPLIT_ROW_SMALL > (float)cols;
    if (lane == 0) exps[row] = row_exponent(m) + (wide ? SPLIT_WIDE : 0);
}

// One workgroup per row, which is in registers before the first of it is stored (x and out may be the same).
template <int VPT>
__global__ __launch_bounds__(256) void split_rows_kernel(const float *x, int dim, float *out, int *exps) {
    const int tid = threadIdx.x;
    const size_t base = (size_t)blockIdx.x * dim;
    v4f v[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int k = (tid + i * 256) * 4;
        v[i] = v4f{0.f, 0.f, 0.f, 0.f};
        if (k < dim) v[i] = *(const v4f *)(x + base + k);
    }
    leave_row<VPT>(v, dim, out + base, exps + blockIdx.x);
}

// Adds the K splits of a gate|up product in split order, applies silu(gate) * up and leaves the row split: one workgroup of 1024 per row
// (a few hundred rows: what counts is that a thread has at most VPT trips to memory).
template <int VPT>
__global__ __launch_bounds__(1024) void reduce_swiglu_split_kernel(GemmArgs a, int splits) {
    const int tid = threadIdx.x, I = a.N >> 1;
    const size_t MN = (size_t)a.M * a.N, base = (size_t)blockIdx.x * a.N;
    v4f v[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
        const int k = (tid + i * 1024) * 4;  // of the I results; gate and up alternate in the product's columns
        v[i] = v4f{0.f, 0.f, 0.f, 0.f};
        if (k < I) {
            v4f p0 = {0.f, 0.f, 0.f, 0.f}, p1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
            for (int s = 0; s < splits; ++s) {
                const float *src = a.part + (size_t)s * MN + base + 2 * k;
                p0 += *(const v4f *)src;
                p1 += *(const v4f *)(src + 4);
            }
            v[i] = v4f{p0.x / (1.0f + expf(-p0.x)) * p0.y, p0.z / (1.0f + expf(-p0.z)) * p0.w, p1.x / (1.0f + expf(-p1.x)) * p1.y,
                       p1.z / (1.0f + expf(-p1.z)) * p1.w};
        }
    }
    leave_row<VPT>(v, I, a.C + (size_t)blockIdx.x * I, a.c_exp + blockIdx.x);
}

int launch_row_exponents(lumen_ctx *ctx, const void *W, int w_bf16, int rows, int cols, int row0, int step, int *exps) {
    if (rows <= 0) return LUMEN_OK;
    if (w_bf16) hipLaunchKernelGGL(row_exponents_kernel<true>, dim3((rows + 3) / 4), dim3(256), 0, ctx->stream, W, rows, cols, row0, step, exps);
    else hipLaunchKernelGGL(row_exponents_kernel<false>, dim3((rows + 3) / 4), dim3(256), 0, ctx->stream, W, rows, cols, row0, step, exps);
    LUMEN_CHECK_LAUNCH();
    return LUMEN_OK;
}

int launch_split_rows(lumen_ctx *ctx, const float *x, int rows, int dim, float *out, int *exps) {
    if (rows <= 0) return LUMEN_OK;
    if (dim % 16 || dim > 16384) LUMEN_FAIL(LUMEN_ERR_UNSUPPORTED, "split rows of %d", dim);
    if (dim <= 2048) hipLaunchKernelGGL(split_rows_kernel<2>, dim3(rows), dim3(256), 0, ctx->stream, x, dim, out, exps);
    else if (dim <= 6144) hipLaunchKernelGGL(split_rows_kernel<6>, dim3(rows), dim3(256), 0, ctx->stream, x, dim, out, exps);
    else hipLaunchKernelGGL(split_rows_kernel<16>, dim3(rows), dim3(256), 0, ctx->stream, x, dim, out, exps);
    LUMEN_CHECK_LAUNCH();
    return LUMEN_OK;
}

int launch_reduce_swiglu_split(lumen_ctx *ctx, const GemmArgs &a, int splits) {
    const int I = a.N / 2;
    if (I % 16 || I > 16384) LUMEN_FAIL(LUMEN_ERR_UNSUPPORTED, "split rows of %d", I);
    if (I <= 4096) hipLaunchKernelGGL(reduce_swiglu_split_kernel<1>, dim3(a.M), dim3(1024), 0, ctx->stream, a, splits);
    else if (I <= 8192) hipLaunchKernelGGL(reduce_swiglu_split_kernel<2>, dim3(a.M), dim3(1024), 0, ctx->stream, a, splits);
    else hipLaunchKernelGGL(reduce_swiglu_split_kernel<4>, dim3(a.M), dim3(1024), 0, ctx->stream, a, splits);
    LUMEN_CHECK_LAUNCH();
    return LUMEN_OK;
}

// Tile and K splits by what the busiest compute unit has to do, in microseconds measured on one MI355X (f32 / bf16 weights): a
// 128 x 128 tile takes 1.5 / 1.15 per piece of 64 of K alone on its compute unit and 1.45 / 0.9 each beside others, a 256 x 256 tile 5.2 /
// 3.1; a launch 7 / 8 besides; a K split 4 for the pass that adds the partial products and their bytes, written and read, at 9 TB/s (they stay
// in the memory-side cache).  At most 16 splits (the passes that add them), 256 MiB of partial products.
SplitPlan gemm_split_plan(int num_cus, int M, int N, int K, int w_bf16, bool sum_later) {
    SplitPlan best = {false, 1};
    double least = 0.0;
    const long pieces = K / 64, cus = num_cus;
    for (int big = 0; big < 2; ++big) {
        const long t = big ? 256 : 128, tiles = ((N + t - 1) / t) * ((M + t - 1) / t);
        for (long s = 1; s <= 16 && s <= pieces; ++s) {
            const double bytes = (double)s * M * N * 4.0;
            if (s > 1 && bytes > (double)((size_t)256 << 20)) break;
            const long per_cu = (tiles * s + cus - 1) / cus, each = (pieces + s - 1) / s;
            double us = (double)each * (double)per_cu * (big ? (w_bf16 ? 3.1 : 5.2) : per_cu == 1 ? (w_bf16 ? 1.15 : 1.5) : (w_bf16 ? 0.9 : 1.45));
            us += big ? 8.0 : 7.0;
            if (s > 1) us += (sum_later ? 0.0 : 4.0) + 2.0 * bytes / 9.0e6;
            if ((big == 0 && s == 1) || us < least) {
                least = us;
                best.big = big != 0;
                best.splits = (int)s;
            }
        }
    }
    return best;
}

template <bool BF16, int FI, int FJ, int DEPTH>
static void launch_f16x2(const GemmArgs &a, dim3 grid, hipStream_t s) {
    if (grid.z > 1) {
        hipLaunchKernelGGL((gemm_f16x2_kernel<BF16, EPI_STORE, true, FI, FJ, 2, 2, DEPTH>), grid, dim3(256), 0, s, a);
        return;
    }
    switch (a.epi) {
        case EPI_STORE: hipLaunchKernelGGL((gemm_f16x2_kernel<BF16, EPI_STORE, false, FI, FJ, 2, 2, DEPTH>), grid, dim3(256), 0, s, a); break;
        case EPI_RESIDUAL: hipLaunchKernelGGL((gemm_f16x2_kernel<BF16, EPI_RESIDUAL, false, FI, FJ, 2, 2, DEPTH>), grid, dim3(256), 0, s, a); break;
        default: hipLaunchKernelGGL((gemm_f16x2_kernel<BF16, EPI_SWIGLU, false, FI, FJ, 2, 2, DEPTH>), grid, dim3(256), 0, s, a); break;
    }
}

void launch_gemm_f16x2(const GemmArgs &a, const SplitPlan &p, hipStream_t s) {
    const int t = p.big ? 256 : 128;
    const dim3 grid((a.N + t - 1) / t, (a.M + t - 1) / t, p.splits);
    if (p.big) {
        if (a.w_bf16) launch_f16x2<true, 4, 4, 2>(a, grid, s);
        else launch_f16x2<false, 4, 4, 2>(a, grid, s);
    } else {
        if (a.w_bf16) launch_f16x2<true, 2, 2, 2>(a, grid, s);
        else launch_f16x2<false, 2, 2, 4>(a, grid, s);
    }
}

// K ranges of the few-row kernel over gridDim.z: the number that costs least, in units of what a workgroup takes for 32 of K (about 0.6 us).  A
// compute unit runs its workgroups side by side, bound by their loads, two more units go into a workgroup's start and end, and a unit with one
// workgroup alone does not keep enough loads in flight; partial products are written and read again at about 5.4 MB per block.  Best counts measured and this rule: 2048 x
// 11264 4, 4; 5632 x 2048 8, 8; 4096 x 12288 4, 4; 4096 x 4096 8, 8; 4096 x 22016 2, 2; 11008 x 4096 8, 8 (K x N).
int gemm_f16x2_stream_splits(int num_cus, int M, int N, int K) {
    const int tiles = (N + 63) / 64, blocks = K / 32;
    int best = 1;
    double least = 0;
    for (int s = 1; s <= 16 && s <= blocks; ++s) {
        const int per_cu = (int)(((long)tiles * s + num_cus - 1) / num_cus);
        double t = per_cu * ((blocks + s - 1) / s + 2.0) * (per_cu == 1 ? 1.25 : 1.0);
        if (s > 1) t += (double)s * M * N * 8 / 5.4e6;
        if (s == 1 || t < least) {
            best = s;
            least = t;
        }
    }
    return best;
}

template <bool BF16, int MT>
static void launch_f16x2_stream(const GemmArgs &a, dim3 grid, hipStream_t s) {
    if (grid.z > 1) {
        hipLaunchKernelGGL((gemm_f16x2_stream_kernel<BF16, MT, EPI_STORE, true>), grid, dim3(256), 0, s, a);
        return;
    }
    switch (a.epi) {
        case EPI_STORE: hipLaunchKernelGGL((gemm_f16x2_stream_kernel<BF16, MT, EPI_STORE, false>), grid, dim3(256), 0, s, a); break;
        case EPI_RESIDUAL: hipLaunchKernelGGL((gemm_f16x2_stream_kernel<BF16, MT, EPI_RESIDUAL, false>), grid, dim3(256), 0, s, a); break;
        default: hipLaunchKernelGGL((gemm_f16x2_stream_kernel<BF16, MT, EPI_SWIGLU, false>), grid, dim3(256), 0, s, a); break;
    }
}
void launch_gemm_f16x2_stream(const GemmArgs &a, int splits, hipStream_t s) {
    const dim3 grid((a.N + 63) / 64, 1, splits);
    if (!a.w_bf16) launch_f16x2_stream<false, 2>(a, grid, s);
    else if (a.M <= 16) launch_f16x2_stream<true, 1>(a, grid, s);
    else launch_f16x2_stream<true, 2>(a, grid, s);
}

LUMEN_DEFINE_WARM(gemm_f16x2)
