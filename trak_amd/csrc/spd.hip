// (A + lambda I)^-1 for a symmetric positive definite fp32 matrix on one GPU, plus the
// "divide by the mean absolute entry" step of the reference.
//
// Stands in for  xtx_inv = torch.linalg.inv(xtx + lambda_reg * eye);  xtx_inv /= xtx_inv.abs().mean()
// (trak/score_computers.py:160-166).  The reference inverts with LU; the matrix here is a Gram
// matrix plus a ridge, so this file uses a blocked Cholesky factorization instead:
//
//   1. W = A + lambda I, padded with an identity block up to a multiple of 128;
//   2. for every 128-block column j:  one workgroup factors the diagonal block in LDS
//      (L_jj) and inverts it; the panel below it is  W[j+1:, j] * L_jj^-T  and the trailing
//      matrix gets  W -= panel * panel^T   (MFMA products; the trailing update and the next
//      diagonal block share one launch, see spd_step_kernel);
//   3. L^-1 by rows of blocks beside the factorization (n <= 4096; see sum_tile), or afterwards by recursive halving:
//      inv([[A,0],[B,C]]) = [[A^-1,0],[-C^-1 B A^-1, C^-1]] (two products per node of the recursion tree);
//   4. inverse = L^-T L^-1 (one product), then the mean of |.| by a two-stage reduction in a
//      fixed order and a scaling pass (the products of 3 and 4: tri_product_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>
#include <vector>

#include "short_k_tile.h"
#include "trakhip_internal.h"

namespace {

constexpr int NB = 128;
constexpr uint64_t kStepTiles = 512;  // tiles of a trailing update that share a launch with the next diagonal block
constexpr uint64_t kStepBlocks = 32;  // n = 4096: blocks a side up to which every step's update has at most that many
constexpr int kSumBlocks = 1024;

// W = A + lambda I padded with an identity block, the 128-blocks on and below the diagonal only: nothing above them
// is read, and every block of L and Li that is read is written first.  A workgroup takes 1024 columns of one row
// (one scalar division per workgroup; with a 64-bit division per element the pass took 12 us at np = 2048 and 55 us
// at 4096, with Li cleared alongside).
constexpr int kInitCols = 1024;

__global__ __launch_bounds__(256) void spd_init_kernel(const float* __restrict__ A, uint64_t lda, float lambda,
                                                       uint32_t n, uint32_t np, uint32_t segments,
                                                       float* __restrict__ W, int32_t* __restrict__ status) {
    const uint32_t row = blockIdx.x / segments, seg = blockIdx.x % segments;
    if (blockIdx.x == 0 && threadIdx.x == 0 && status) *status = 0;
    const uint32_t end = (row / NB + 1) * NB;  // the row's blocks up to the diagonal one
    for (uint32_t c = 0; c < kInitCols; c += 256) {
        const uint32_t col = seg * kInitCols + c + threadIdx.x;
        if (col >= end) return;
        float v = row == col ? 1.0f : 0.0f;
        if (row < n && col < n) v = A[(uint64_t)row * lda + col] + (row == col ? lambda : 0.0f);
        W[(uint64_t)row * np + col] = v;
    }
}

// One workgroup of eight waves: Cholesky of the 128x128 diagonal block at W (lower triangle used),
// L block to Lout (upper part zero), its inverse to Linv_out.
//
// The block is handled as 4 x 4 sub-blocks of 32 in LDS.  ONE WAVE factors a 32 x 32 diagonal sub-block and inverts
// the factor, without barriers inside this strictly sequential part (see factor_sub_block).  Everything else is products of
// 16 x 32 strips on v_mfma_f32_16x16x4_f32, and what the next factorization does not wait for runs on waves of the other
// SIMDs beside it:
//
//   before    all waves: the panel's share of (0, 0) and (1, 1)
//   phase p   wave 0: factor and invert (p, p)         six waves: (t, p) for t > p and (p + 1, p + 1) less the panel's share
//                                                      and columns 0 .. p - 1 of the factor, and
//                                                      T_j = sum over m of L[p][m] X[m][j], j < p
//             L[t][p] = A[t][p] X_pp^T for t > p, X[p][j] = -X_pp T_j for j < p            (six strips)
//             A[p+1][p+1] -= L[p+1][p] L[p+1][p]^T                                        (two strips)
//
// so every sub-block is brought up to date in one pass just before it is needed, and the inverse of the factor grows row by
// row with the factorization and is complete one product after the last sub-block.  Bound: the four sub-blocks in
// sequence, 28 000 of 47 500 cycles; loads 4400, the first two sub-blocks' share of the panel 3300, strips 6800, their
// update 2700, stores 2300.  With the panel's share of the whole block taken off before the first sub-block (13 700
// cycles on all waves) and 7950 cycles per sub-block it took 64 700: a step of the factorization 28 us, now 22.
constexpr int kSub = 32;
constexpr int kPitch = NB + 4;            // 528-byte rows: 16-byte reads, conflict free over 16 rows
constexpr int kTPitch = 3 * kSub + 4;
constexpr int kDiagThreads = 512, kDiagWaves = kDiagThreads / 64;

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Row 8*(r/4) + 4*(lane/32) + r%4 of a 32x32 MFMA result is in register r; its column is lane % 32.
__device__ __forceinline__ int mfma_row(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Factor and invert the 32 x 32 sub-block at (base, base) of As with one wave: L over As, X = L^-1 to Dx (32 rows of
// kDxPitch floats).  A and X (initially the identity) sit in the result layout of a 32x32 MFMA: lane = column x, register
// r = row 8 (r / 4) + 4 (lane / 32) + r % 4, so that rows 4m .. 4m + 3 are four registers of one half-wave - and, A being
// symmetric, those four registers of lane x are also the four entries of row x in columns 4m .. 4m + 3.  Eight panels of
// four columns, then: the panel's columns are eliminated one by one inside these four registers (lanes of other columns
// through v_readlane), the same four eliminations go through rows 4m .. 4m + 3 of X, and everything behind the panel gets
// its four columns at once, A -= L4 L4^T and X -= L4 X4, two 32x32x2 MFMAs each whose operands are one
// v_permlane32_swap away.  Rows and columns that are finished go on being updated and are not looked at again.
//
// Bound: the chain of one wave from pivot to pivot (reciprocal root, Newton step, lane read, scale, lane read,
// multiply-add), 700 cycles per panel; the last of X's two products waits until the next panel's first pivot is
// through.  6200 cycles per sub-block; a column at a time with every multiply-add on the vector unit took 7950.  The 4 x 4
// block's factor worked out in all lanes without lane reads in the chain: 6400; X's rows a panel late between the
// pivots: 7300.
constexpr int kDxPitch = kSub + 4;

template <class F, int... S>
__device__ __forceinline__ void for_each_index(F& f, std::integer_sequence<int, S...>) {
    (f(std::integral_constant<int, S>{}), ...);
}

__device__ __forceinline__ void factor_sub_block(float* As, float* Dx, int base, int lane, int32_t first_index,
                                                 int32_t* status) {
    const int x = lane & 31, h = lane >> 5;
    floatx16 a, xi;  // both with their signs turned: the products below only add
    {
        // lower triangle only: row x left of the diagonal, column x below it
        floatx4 row[4];
        float col[16];
#pragma unroll
        for (int j = 0; j < 4; ++j) row[j] = *reinterpret_cast<const floatx4*>(As + (base + x) * kPitch + base + 8 * j + 4 * h);
#pragma unroll
        for (int r = 0; r < 16; ++r) col[r] = As[(base + mfma_row(r, h)) * kPitch + base + x];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a[r] = mfma_row(r, h) >= x ? -col[r] : -row[r >> 2][r & 3];
            xi[r] = mfma_row(r, h) == x ? -1.0f : 0.0f;
        }
    }
    // The pivots are kept, pivot k's in lane k of its half-wave, and looked at once at the end: one that is not positive
    // makes everything behind it NaN.
    float pivots = 1.0f;
    const bool first_of_four = (lane & 3) == 0, second_of_four = (lane & 3) == 1, third_of_four = (lane & 3) == 2;
    float l_late = 0.0f, y_late = 0.0f;  // operands of the product that a panel leaves to the next one
    auto panel = [&](auto m_const) __attribute__((always_inline)) {
        constexpr int m = decltype(m_const)::value, kHalf = m & 1, kReg = 4 * (m >> 1), kLane = 32 * kHalf + 4 * m;
        float l[4], y[4], d[4], s[4], b[4][4], l_pair[2];
#pragma unroll
        for (int t = 0; t < 4; ++t) l[t] = -a[kReg + t];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            // 1 / sqrt of the pivot (one Newton step on the 1 ulp hardware value): every lane works on its own value and
            // the pivot's lane is the one that counts
            d[t] = l[t];
            const float r = __builtin_amdgcn_rsqf(d[t]);
            s[t] = lane_value(r * __builtin_fmaf(-0.5f * d[t] * r, r, 1.5f), kLane + t);
            l[t] *= s[t];
#pragma unroll
            for (int u = t + 1; u < 4; ++u) {
                b[u][t] = lane_value(l[t], kLane + u);
                l[u] = __builtin_fmaf(-b[u][t], l[t], l[u]);
            }
            if constexpr (m > 0) {
                if (t == 1) xi = __builtin_amdgcn_mfma_f32_32x32x2f32(l_late, y_late, xi, 0, 0, 0);
            }
            if constexpr (m < 7) {
                if (t & 1) {  // lower half-wave: first column of a pair, upper half-wave: the second one
                    const auto pair =
                        __builtin_amdgcn_permlane32_swap(__float_as_uint(l[t - 1]), __float_as_uint(l[t]), false, false);
                    l_pair[t >> 1] = __uint_as_float(pair[kHalf]);
                    a = __builtin_amdgcn_mfma_f32_32x32x2f32(l_pair[t >> 1], l_pair[t >> 1], a, 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            y[t] = -xi[kReg + t];
#pragma unroll
            for (int u = 0; u < t; ++u) y[t] = __builtin_fmaf(-b[t][u], y[u], y[t]);
            y[t] *= s[t];
        }
        {
            int four = lane >> 2;
            asm volatile("" : "+v"(four));  // (compared here: held across the eight panels, the masks go to spilled registers)
            const float mine = first_of_four ? d[0] : second_of_four ? d[1] : third_of_four ? d[2] : d[3];
            pivots = four == kLane / 4 ? mine : pivots;
        }
        if (h == kHalf) {
            // (L is not read above its diagonal; X is zero there by construction)
#pragma unroll
            for (int t = 0; t < 4; ++t) Dx[(4 * m + t) * kDxPitch + x] = y[t];
            *reinterpret_cast<floatx4*>(As + (base + x) * kPitch + base + 4 * m) = floatx4{l[0], l[1], l[2], l[3]};
        }
        if constexpr (m < 7) {
            const auto q0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[0]), __float_as_uint(y[1]), false, false);
            const auto q1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[2]), __float_as_uint(y[3]), false, false);
            xi = __builtin_amdgcn_mfma_f32_32x32x2f32(l_pair[0], __uint_as_float(q0[kHalf]), xi, 0, 0, 0);
            l_late = l_pair[1], y_late = __uint_as_float(q1[kHalf]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for_each_index(panel, std::make_integer_sequence<int, 8>{});
    const uint64_t bad = __builtin_amdgcn_ballot_w64(!(pivots > 0.0f));
    const uint32_t which = (uint32_t)bad | (uint32_t)(bad >> 32);
    if (which != 0 && lane == 0 && status && *status == 0) *status = 1 + first_index + __builtin_ctz(which);
}

// acc[q] += A[16 x K] * op(B)[:, 16 q .. 16 q + 15], q = 0, 1: a strip of 16 rows and 32 columns (ONE: only its first
// 16 columns, acc[1] takes the odd steps).  A rows at `a` (pitch pa, k contiguous); B^T rows at `b` (B_T: pitch pb, k
// contiguous) or B rows at `b` (k down the rows).  Quarter g of the wave (lane / 16) takes k = 16 s + 4 g + t for the
// t-th MFMA of sub-step s, so that an operand whose k is contiguous is one 16-byte LDS read per four MFMAs.
template <bool B_T, bool ONE>
struct StripStep {
    static constexpr int kQ = ONE ? 1 : 2;
    floatx4 fa[2], fb[2][kQ];
    __device__ __forceinline__ void fetch(const float* a, int pa, const float* b, int pb, int k0, int lane) {
        const int x = lane & 15, g = lane >> 4;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int k = k0 + 16 * s + 4 * g;
            fa[s] = *reinterpret_cast<const floatx4*>(a + x * pa + k);
#pragma unroll
            for (int q = 0; q < kQ; ++q) {
                if (B_T) {
                    fb[s][q] = *reinterpret_cast<const floatx4*>(b + (16 * q + x) * pb + k);
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t) fb[s][q][t] = b[(k + t) * pb + 16 * q + x];
                }
            }
        }
    }
    __device__ __forceinline__ void multiply(floatx4 (&acc)[2]) const {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int q = 0; q < kQ; ++q) {
                    floatx4& c = acc[ONE ? t & 1 : q];
                    c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[s][t], fb[s][q][t], c, 0, 0, 0);
                }
        __builtin_amdgcn_sched_barrier(0);
    }
};

// K a multiple of 32
template <bool B_T, bool ONE = false>
__device__ __forceinline__ void strip_product(const float* a, int pa, const float* b, int pb, int K, floatx4 (&acc)[2],
                                              int lane) {
    for (int k0 = 0; k0 < K; k0 += 32) {
        StripStep<B_T, ONE> step;
        step.fetch(a, pa, b, pb, k0, lane);
        step.multiply(acc);
    }
}

// K = 32 STEPS, B^T rows: the reads of a step on their way under the MFMAs of the one before
template <int STEPS, bool ONE = false>
__device__ __forceinline__ void strip_product_fixed(const float* a, const float* b, floatx4 (&acc)[2], int lane) {
    StripStep<true, ONE> step[2];
    step[0].fetch(a, kPitch, b, kPitch, 0, lane);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        if (i + 1 < STEPS) step[(i + 1) & 1].fetch(a, kPitch, b, kPitch, 32 * (i + 1), lane);
        step[i & 1].multiply(acc);
    }
}

// Row 4 (lane / 16) + r of a 16 x 16 MFMA result is in register r; its column is lane % 16.
__device__ __forceinline__ void strip_load(const float* c, int pc, floatx4 (&acc)[2], int lane) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[q][r] = c[(4 * (lane >> 4) + r) * pc + 16 * q + (lane & 15)];
}

// (SIGN: -1 where the sum was kept with its sign turned)
template <int SIGN = 1>
__device__ __forceinline__ void strip_store(float* c, int pc, const floatx4 (&acc)[2], int lane) {
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            c[(4 * (lane >> 4) + r) * pc + 16 * q + (lane & 15)] = SIGN < 0 ? -acc[q][r] : acc[q][r];
}

__device__ __forceinline__ void strip_zero(floatx4 (&acc)[2]) {
    acc[0] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    acc[1] = acc[0];
}

// Rows 16 half .. 16 half + 15 of A[ti][tj] -= P[ti] P[tj]^T (P: the panel block, 128 columns, or null) and
// -= L[ti][c] L[tj][c]^T, columns c = c0 .. c0 + K - 1 of the factor (K may be 0).  Of a sub-block on the diagonal the upper
// rows need their first 16 columns only.
template <bool ONE>
__device__ __forceinline__ void update_strip_part(float* As, int ti, int tj, int row, const float* P, int c0, int K, int lane) {
    float* c = As + row * kPitch + kSub * tj + 4 * (lane >> 4) * kPitch + (lane & 15);
    floatx4 acc[2], old[2];  // (the sum with its sign turned, from zero: A is read under the products)
    strip_zero(acc);
#pragma unroll
    for (int q = 0; q < (ONE ? 1 : 2); ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) old[q][r] = c[r * kPitch + 16 * q];
    if (P) strip_product_fixed<NB / 32, ONE>(P + row * kPitch, P + kSub * tj * kPitch, acc, lane);
    strip_product<true, ONE>(As + row * kPitch + c0, kPitch, As + kSub * tj * kPitch + c0, kPitch, K, acc, lane);
    if constexpr (ONE) acc[0] += acc[1];
#pragma unroll
    for (int q = 0; q < (ONE ? 1 : 2); ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r * kPitch + 16 * q] = old[q][r] - acc[q][r];
}

__device__ __forceinline__ void update_strip(float* As, int ti, int tj, int half, const float* P, int c0, int K, int lane) {
    const int row = kSub * ti + 16 * half;
    if (ti == tj && half == 0)
        update_strip_part<true>(As, ti, tj, row, P, c0, K, lane);
    else
        update_strip_part<false>(As, ti, tj, row, P, c0, K, lane);
}

constexpr int kDiagLdsFloats = 2 * NB * kPitch + kSub * kTPitch + kSub * kDxPitch;  // 152 576 bytes

// `panel`, when not null, is the 128 x 128 block of the factor to the left of this diagonal block
// (row pitch ldp) whose contribution has not been taken off W yet: the block that is factored is
// W - panel panel^T (its lower triangle).
__device__ __forceinline__ void diag_block(const float* __restrict__ W, uint64_t ldw, float* __restrict__ Lout,
                                           float* __restrict__ Linv_out, uint64_t ldl, int32_t block_index,
                                           int32_t* __restrict__ status, const float* __restrict__ panel,
                                           uint64_t ldp, float* __restrict__ lds) {
    float* As = lds;                        // the block, overwritten by its factor
    float* Xs = As + NB * kPitch;           // the panel block; row by row of sub-blocks, the inverse of the factor
    float* Ts = Xs + NB * kPitch;           // T_j of the sub-block row at work
    float* Dx = Ts + kSub * kTPitch;        // the inverse of the sub-block at work
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;  // wave index in a scalar register
    constexpr int kBlocks = NB / kSub, kRows = NB * (NB / 4) / kDiagThreads;
    const int r0 = tid >> 5, c = 4 * (tid & 31);

    // thread -> (row tid / 32 + 16 i, four columns from 4 (tid % 32)); all loads in flight at once
    // (the block starts at a multiple of 128 floats of a 16-byte aligned matrix with ldw % 128 == 0)
    {
        floatx4 v[kRows], w[kRows];
#pragma unroll
        for (int i = 0; i < kRows; ++i) v[i] = *reinterpret_cast<const floatx4*>(W + (uint64_t)(r0 + 16 * i) * ldw + c);
        if (panel) {
#pragma unroll
            for (int i = 0; i < kRows; ++i) w[i] = *reinterpret_cast<const floatx4*>(panel + (uint64_t)(r0 + 16 * i) * ldp + c);
#pragma unroll
            for (int i = 0; i < kRows; ++i) *reinterpret_cast<floatx4*>(Xs + (r0 + 16 * i) * kPitch + c) = w[i];
        }
#pragma unroll
        for (int i = 0; i < kRows; ++i) *reinterpret_cast<floatx4*>(As + (r0 + 16 * i) * kPitch + c) = v[i];
    }
    __syncthreads();
    if (panel) {
        // the panel's share of (0, 0) and (1, 1): waves 0-3 a strip each, waves 4-7 the second half of its columns
        const int sub = (wave >> 1) & 1, half = wave & 1, row = kSub * sub + 16 * half, k0 = wave < 4 ? 0 : NB / 2;
        float* c_strip = As + row * kPitch + kSub * sub;
        float* other = Ts + (wave & 3) * 512 + 4 * lane;
        floatx4 acc[2];
        strip_zero(acc);
        strip_product_fixed<NB / 64>(Xs + row * kPitch + k0, Xs + kSub * sub * kPitch + k0, acc, lane);
        if (wave >= 4) {
#pragma unroll
            for (int q = 0; q < 2; ++q) *reinterpret_cast<floatx4*>(other + 256 * q) = acc[q];
        }
        __syncthreads();
        if (wave < 4) {
            floatx4 old[2];
            strip_load(c_strip, kPitch, old, lane);
#pragma unroll
            for (int q = 0; q < 2; ++q) acc[q] = old[q] - (acc[q] + *reinterpret_cast<const floatx4*>(other + 256 * q));
            strip_store(c_strip, kPitch, acc, lane);
        }
        __syncthreads();
    }

    for (int p = 0; p < kBlocks; ++p) {
        const int base = kSub * p, below = kBlocks - 1 - p;  // sub-blocks under the diagonal one
        if (wave == 0) {
            factor_sub_block(As, Dx, base, lane, block_index * NB + base, status);
        } else if (wave != 4) {  // (wave 4 shares wave 0's SIMD)
            // Everything that the sub-blocks below (p, p), and (p + 1, p + 1), lack up to column p - 1; then T_j.  Dealt so
            // that the three SIMDs get equal shares (waves 1 and 5, 2 and 6, 3 and 7): p = 1, eight units, the short ones
            // to wave 7; p = 2, eight units, to waves 6 and 7 the four T.
            const int strips = p == 0 ? (panel ? 2 * below : 0) : (below ? 2 * below + 2 : 0), units = strips + 2 * p;
            const int v = wave < 4 ? wave - 1 : wave - 2, several = p == 1 ? 5 : p == 2 ? 4 : 0;
            const int end = v < several ? v + 1 : units;
            for (int u = v; u < end; u += kDiagWaves - 2 - several) {
                const int i = u >> 1;
                if (u < strips) {  // of (p + 1, p + 1) the longer strip first
                    update_strip(As, i < below ? p + 1 + i : p + 1, i < below ? p : p + 1, i < below ? u & 1 : ~u & 1,
                                 panel ? Xs : nullptr, 0, base, lane);
                } else {
                    const int j = i - (strips >> 1), half = u & 1;
                    floatx4 acc[2];
                    strip_zero(acc);
                    strip_product<false>(As + (base + 16 * half) * kPitch + kSub * j, kPitch,
                                         Xs + kSub * j * kPitch + kSub * j, kPitch, base - kSub * j, acc, lane);
                    strip_store(Ts + 16 * half * kTPitch + kSub * j, kTPitch, acc, lane);
                }
            }
        }
        __syncthreads();
        {
            // six strips for waves 0-5, X_pp into its place by waves 6 and 7 (row p of the panel block is done with)
            const int half = wave & 1;
            floatx4 acc[2];
            strip_zero(acc);
            if (wave < 2 * below) {  // L[t][p], in place: a wave has read its rows before it writes them
                float* rows = As + (base + kSub * (1 + (wave >> 1)) + 16 * half) * kPitch + base;
                strip_product<true>(rows, kPitch, Dx, kDxPitch, kSub, acc, lane);
                strip_store(rows, kPitch, acc, lane);
            } else if (wave < 2 * (kBlocks - 1)) {  // X[p][j]
                const int j = (wave >> 1) - below;
                strip_product<false>(Dx + 16 * half * kDxPitch, kDxPitch, Ts + kSub * j, kTPitch, kSub, acc, lane);
                strip_store<-1>(Xs + (base + 16 * half) * kPitch + kSub * j, kPitch, acc, lane);
            } else {
                const int row = 16 * half + (lane >> 2), col = 8 * (lane & 3);
#pragma unroll
                for (int e = 0; e < 8; e += 4)
                    *reinterpret_cast<floatx4*>(Xs + (base + row) * kPitch + base + col + e) =
                        *reinterpret_cast<const floatx4*>(Dx + row * kDxPitch + col + e);
            }
        }
        __syncthreads();
        if (below == 0) break;
        if (wave < 2) update_strip(As, p + 1, p + 1, wave, nullptr, base, kSub, lane);
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const int r = r0 + 16 * i;
        floatx4 l = *reinterpret_cast<const floatx4*>(As + r * kPitch + c);
        floatx4 li = *reinterpret_cast<const floatx4*>(Xs + r * kPitch + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            l[e] = c + e <= r ? l[e] : 0.0f;
            li[e] = c + e <= r ? li[e] : 0.0f;
        }
        *reinterpret_cast<floatx4*>(Lout + (uint64_t)r * ldl + c) = l;
        *reinterpret_cast<floatx4*>(Linv_out + (uint64_t)r * ldl + c) = li;
    }
}

__global__ __launch_bounds__(kDiagThreads, 2) void spd_diag_kernel(const float* __restrict__ W, uint64_t ldw,
                                                       float* __restrict__ Lout, float* __restrict__ Linv_out,
                                                       uint64_t ldl, int32_t block_index,
                                                       int32_t* __restrict__ status) {
    __shared__ __attribute__((aligned(16))) float lds[kDiagLdsFloats];
    diag_block(W, ldw, Lout, Linv_out, ldl, block_index, status, nullptr, 0, lds);
}

// ---- the inverse of the factor, a row of blocks per step ------------------------------------------------------
//
// X = L^-1 grows with the factorization: row p is  X[p][c] = -X_pp T_c,  T_c = sum over m = c .. p - 1 of L[p][m] X[m][c].  The
// sums need rows of X and L that are there before block (p, p) is factored, so they run in the same launch as it, on CUs
// that the trailing update leaves idle (its tiles get fewer as the sums get longer); the product with X_pp runs beside the
// next panel.  Against L^-1 by recursive halving behind the factorization (two launches per depth, 27 us at n = 512, 104 at
// 2048, 346 at 4096) one launch of 6 us is left and the steps are as long as before up to n = 2048 (22 us).  Whole call: 256
// 122 -> 93 us, 512 220 -> 153, 2048 804 -> 534, 4096 1910 -> 1562, of which the panels of the diagonal block gave two fifths.

// T tile: 32 rows x 64 columns, tile number = 4 (column group) + row group; eight waves = two 32 x 32 parts x four
// quarters of every 128 values of k, whose sums are added up at the end.  Two chunks of 128 k in flight in registers.
constexpr int kSumRows = 32, kSumCols = 64;
constexpr int kSumPitchA = NB + 4, kSumPitchB = kSumCols + 8;  // conflict-free 16-byte reads; half-waves in other banks
constexpr int kSumFloats = kSumRows * kSumPitchA + NB * kSumPitchB;

__device__ __forceinline__ void sum_tile(const float* __restrict__ L, const float* __restrict__ Li, float* __restrict__ T,
                                         uint64_t np, uint32_t p, uint32_t tile, float* __restrict__ lds) {
    const uint32_t row0 = p * NB + kSumRows * (tile & 3), col0 = kSumCols * (tile >> 2), c = col0 / NB;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, x = lane & 31, h = lane >> 5;
    const int wk = wave >> 1, wn = wave & 1;
    constexpr int kA = kSumRows * (NB / 4) / kDiagThreads, kB = NB * (kSumCols / 4) / kDiagThreads;
    const float* a0 = L + (uint64_t)row0 * np + (uint64_t)c * NB;
    const float* b0 = Li + (uint64_t)c * NB * np + col0;
    const uint32_t count = p - c;
    floatx4 ra[2][kA], rb[2][kB];
    auto load = [&](uint32_t i, int u) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < kA; ++e) {
            const int id = tid + kDiagThreads * e;
            ra[u][e] = *reinterpret_cast<const floatx4*>(a0 + (uint64_t)(id >> 5) * np + i * NB + 4 * (id & 31));
        }
#pragma unroll
        for (int e = 0; e < kB; ++e) {
            const int id = tid + kDiagThreads * e;
            rb[u][e] = *reinterpret_cast<const floatx4*>(b0 + ((uint64_t)i * NB + (id >> 4)) * np + 4 * (id & 15));
        }
    };
    load(0, 0);
    if (count > 1) load(1, 1);
    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
    auto chunk = [&](uint32_t i, auto u_const) __attribute__((always_inline)) {
        constexpr int u = decltype(u_const)::value;
        // a buffer is written again two chunks later, behind the barrier that follows its reads
        float* as = lds + u * kSumFloats;
        float* bs = as + kSumRows * kSumPitchA;
#pragma unroll
        for (int e = 0; e < kA; ++e) {
            const int id = tid + kDiagThreads * e;
            *reinterpret_cast<floatx4*>(as + (id >> 5) * kSumPitchA + 4 * (id & 31)) = ra[u][e];
        }
#pragma unroll
        for (int e = 0; e < kB; ++e) {
            const int id = tid + kDiagThreads * e;
            *reinterpret_cast<floatx4*>(bs + (id >> 4) * kSumPitchB + 4 * (id & 15)) = rb[u][e];
        }
        if (i + 2 < count) load(i + 2, u);
        __syncthreads();
        floatx4 fa[4], fb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = 32 * wk + 8 * q + 4 * h;
            fa[q] = *reinterpret_cast<const floatx4*>(as + x * kSumPitchA + k);
#pragma unroll
            for (int t = 0; t < 4; ++t) fb[q][t] = bs[(k + t) * kSumPitchB + 32 * wn + x];
        }
        __builtin_amdgcn_sched_barrier(0);  // all reads of the chunk in flight before its first MFMA waits
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[q][t], fb[q][t], acc[q & 1], 0, 0, 0);
    };
    for (uint32_t i = 0; i < count; i += 2) {
        chunk(i, std::integral_constant<int, 0>{});
        if (i + 1 < count) chunk(i + 1, std::integral_constant<int, 1>{});
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) lds[(wave * 16 + r) * 64 + lane] = acc[0][r] + acc[1][r];
    __syncthreads();
    float* out = T + (uint64_t)row0 * np + col0 + 32 * wn + x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // registers 4 wk .. 4 wk + 3 of the four quarters' sums
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) v += lds[((2 * w + wn) * 16 + 4 * wk + r) * 64 + lane];
        out[(uint64_t)(8 * wk + 4 * h + r) * np] = v;
    }
}

// Launch between two steps: workgroups 0 .. panel_tiles - 1 the panel below diagonal block j, 32 rows each,
// L[j+1:, j] = W[j+1:, j] X_jj^T; the others row j of X, 32 columns each, X[j][c] = -X_jj T_c.
constexpr int kXPitchB = 32 + 8;
constexpr int kXFloats = NB * (NB + 4) + NB * kXPitchB;
constexpr int kPanelLdsFloats = kXFloats > short_k::lds_floats<32>() ? kXFloats : short_k::lds_floats<32>();

__global__ __launch_bounds__(256, 1) void spd_panel_kernel(const float* __restrict__ W, float* __restrict__ L,
                                                           float* __restrict__ Li, uint64_t np, uint32_t j,
                                                           uint32_t panel_tiles) {
    __shared__ __attribute__((aligned(16))) float lds[kPanelLdsFloats];
    const uint64_t diag = (uint64_t)j * NB * np + (uint64_t)j * NB;
    if (blockIdx.x < panel_tiles) {
        const uint64_t below = diag + NB * np;
        short_k::tile<32>(W + below, np, Li + diag, np, L + below, np, np - (j + 1) * NB, NB, NB, 1.0f, 0.0f, blockIdx.x, 0,
                          lds);
        return;
    }
    const uint32_t col0 = 32 * (blockIdx.x - panel_tiles);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, x = lane & 31, h = lane >> 5;
    const float* A = Li + diag;                              // X_jj, zero above its diagonal
    const float* B = W + (uint64_t)j * NB * np + col0;       // T
    floatx4 ra[16], rb[4];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int id = tid + 256 * i;
        ra[i] = *reinterpret_cast<const floatx4*>(A + (uint64_t)(id >> 5) * np + 4 * (id & 31));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int id = tid + 256 * i;
        rb[i] = *reinterpret_cast<const floatx4*>(B + (uint64_t)(id >> 3) * np + 4 * (id & 7));
    }
    float* as = lds;
    float* bs = lds + NB * (NB + 4);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int id = tid + 256 * i;
        *reinterpret_cast<floatx4*>(as + (id >> 5) * (NB + 4) + 4 * (id & 31)) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int id = tid + 256 * i;
        *reinterpret_cast<floatx4*>(bs + (id >> 3) * kXPitchB + 4 * (id & 7)) = rb[i];
    }
    __syncthreads();
    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
    for (int k0 = 0; k0 <= 32 * wave; k0 += 32) {  // rows 32 wave .. + 31 of a lower triangular operand
        floatx4 fa[4], fb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int k = k0 + 8 * q + 4 * h;
            fa[q] = *reinterpret_cast<const floatx4*>(as + (32 * wave + x) * (NB + 4) + k);
#pragma unroll
            for (int t = 0; t < 4; ++t) fb[q][t] = bs[(k + t) * kXPitchB + x];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[q][t], fb[q][t], acc[q & 1], 0, 0, 0);
    }
    float* out = Li + ((uint64_t)j * NB + 32 * wave) * np + col0 + x;
#pragma unroll
    for (int r = 0; r < 16; ++r) out[(uint64_t)mfma_row(r, h) * np] = -(acc[0][r] + acc[1][r]);
}

// One step of the factorization in one launch, after the panel below diagonal block j is known:
// workgroup 0 takes the next diagonal block (j+1, j+1) - its own trailing update, then factor and
// inverse - the next 8 (j+1) the sums T for row j+1 of X, and the others apply the trailing update W -= panel panel^T to
// the other lower-triangle tiles (tile numbers in the triangle's row-by-row order; number 0 is that diagonal
// block).  Nothing in the launch depends on anything else in it: the sequential diagonal work does not sit between two
// launches but beside the trailing update and the sums.  T takes the place of W[j+1][0 .. j], which the panels have read.
__global__ __launch_bounds__(kDiagThreads, 2) void spd_step_kernel(float* __restrict__ W, float* __restrict__ L,
                                                                   float* __restrict__ Li, uint64_t np, uint32_t j,
                                                                   uint32_t sum_tiles, int32_t* __restrict__ status) {
    constexpr int kLds = kDiagLdsFloats > short_k::lds_floats<NB>() ? kDiagLdsFloats : short_k::lds_floats<NB>();
    static_assert(2 * kSumFloats <= kLds && 8 * 16 * 64 <= kLds, "the sums' buffers");
    __shared__ __attribute__((aligned(16))) float lds[kLds];
    const uint64_t tr = (uint64_t)(j + 1) * NB * np + (uint64_t)(j + 1) * NB, rows = np - (uint64_t)(j + 1) * NB;
    const float* panel = L + tr - NB;  // L[j+1:, j]
    if (blockIdx.x == 0) {
        diag_block(W + tr, np, L + tr, Li + tr, np, (int32_t)(j + 1), status, panel, np, lds);
    } else if (blockIdx.x <= sum_tiles) {
        sum_tile(L, Li, W, np, j + 1, blockIdx.x - 1, lds);
    } else {
        uint32_t tile_m, tile_n;
        short_k::triangle_tile(blockIdx.x - sum_tiles, tile_m, tile_n);
        short_k::tile<NB, kDiagThreads>(panel, np, panel, np, W + tr, np, rows, rows, NB, -1.0f, 1.0f, tile_m, tile_n, lds);
    }
}

__device__ __forceinline__ float workgroup_sum(float s) {
    __shared__ float red[256];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    return red[0];
}

// Workgroup b adds up |M| over rows b, b + 1024, ... (partial[b] = 0 where there is none).
__global__ __launch_bounds__(256) void abs_sum_kernel(const float* __restrict__ M, uint64_t ld, uint32_t n,
                                                      float* __restrict__ partial) {
    float s = 0.0f;
    for (uint32_t row = blockIdx.x; row < n; row += kSumBlocks) {
        const float* m = M + (uint64_t)row * ld;
        for (uint32_t col = threadIdx.x; col < n; col += 256) s += fabsf(m[col]);
    }
    s = workgroup_sum(s);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// The mean from the partial sums - every workgroup works it out for itself (at most 8.3 KB from L2) instead of waiting for a
// launch that does only that - and M /= mean, rows b, b + gridDim.x, ... for workgroup b.
__global__ __launch_bounds__(256) void mean_scale_kernel(const float* __restrict__ partial, uint32_t count,
                                                         float* __restrict__ M, uint64_t ld, uint32_t n, int normalize,
                                                         float* __restrict__ mean_user) {
    float s = 0.0f;
#pragma unroll 4
    for (uint32_t e = threadIdx.x; e < count; e += 256) s += partial[e];
    const float mean = workgroup_sum(s) / ((float)n * (float)n);
    if (blockIdx.x == 0 && threadIdx.x == 0 && mean_user) *mean_user = mean;
    if (!normalize) return;
    const float inv = 1.0f / mean;
    for (uint32_t row = blockIdx.x; row < n; row += gridDim.x) {
        float* m = M + (uint64_t)row * ld;
        for (uint32_t col = threadIdx.x; col < n; col += 256) m[col] *= inv;
    }
}

// count: partial sums that are there already; 0: none are
int divide_by_mean(float* M, uint64_t ld, uint64_t n, int normalize, float* partial, uint32_t count, float* mean_user,
                   hipStream_t s) {
    if (!normalize && !mean_user) return TRAKHIP_OK;
    if (!count) {
        hipLaunchKernelGGL(abs_sum_kernel, dim3(kSumBlocks), dim3(256), 0, s, M, ld, (uint32_t)n, partial);
        count = kSumBlocks;
    }
    const uint32_t rows = normalize ? (uint32_t)(n < 2048 ? n : 2048) : 1;
    hipLaunchKernelGGL(mean_scale_kernel, dim3(rows), dim3(256), 0, s, partial, count, M, ld, (uint32_t)n, normalize, mean_user);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

// ---- products with a triangular operand ---------------------------------------------------------------------
//
// fp32 MFMA products of the triangular inverse by recursion (n > 4096) and the final L^-T L^-1 (n > 2048; below, see
// tri_gram_small_kernel).  Bound: the latency of the global loads in the recursion's small nodes (a [1024 x 1024] one has
// 2 GFLOP for the whole chip); L^-T L^-1 at n = 4096 runs at 86 TFLOP/s of the 124 that the general fp32 MFMA product reaches (64 x 64 tiles, the mirror image stored a row apart per lane).
// So: 64 x 64 tiles (256 workgroups where 128 x 128 tiles gave 64), four k steps of 32 in flight in registers while
// one is multiplied from LDS, and k ranges cut to the part where the triangular operand is not zero (rounded to
// 128, so a range is whole chunks of four steps), tiles with the longest range first.
enum class Tri { kLowerB, kLowerA, kGram };
//   kLowerB  C = alpha A B    A row-major along k, B lower triangular (k down the rows): k from the tile's columns on
//   kLowerA  C = alpha A B    A lower triangular: k up to the tile's rows
//   kGram    C = A^T A        A lower triangular, lower tiles + mirror image: k from the tile's rows on; n x n stored
// Operands have whole 128-blocks (row pitch np).  A wave owns one 32 x 32 tile, two accumulators (even and odd
// sub-steps) that are added at the end: error of the inverse against 64 bits 9.4e-7 at n = 2048, 1.26e-6 with one
// accumulator over the whole range in the earlier kernels.  Measured: a whole recursion of n = 4096
// 824 -> 350 us (128 x 128 tiles over the full k range), L^-T L^-1 516 -> 277 us (256 x 256 tiles of the
// six-term bf16 product, planes included).  The staging registers are vector types (arrays of HIP's float4 stayed in
// scratch) and all fragment reads of a step stand before its first MFMA: without these two the same products took
// twice as long.
constexpr int kTriTile = 64, kTriStep = 32, kTriDepth = NB / kTriStep;
constexpr int kRowPitch = kTriStep + 4;   // row-k tile, 64 rows: 144-byte rows, conflict-free 16-byte reads
constexpr int kColPitch = kTriTile + 8;   // k-row tile, 32 rows: the half-waves (4 rows apart) read other banks
constexpr int kTriFloats = kTriTile * kRowPitch;
static_assert(kTriStep * kColPitch == kTriFloats, "both operand layouts take the same room");

template <bool KROW>
__device__ __forceinline__ void tri_load(const float* __restrict__ p, uint64_t ld, uint32_t x0, uint32_t k0, int tid,
                                         floatx4 (&r)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int id = tid + 256 * i;
        const uint64_t at = KROW ? (uint64_t)(k0 + (id >> 4)) * ld + x0 + 4 * (id & 15)
                                 : (uint64_t)(x0 + (id >> 3)) * ld + k0 + 4 * (id & 7);
        r[i] = *reinterpret_cast<const floatx4*>(p + at);
    }
}

template <bool KROW>
__device__ __forceinline__ void tri_store(float* lds, int tid, const floatx4 (&r)[2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int id = tid + 256 * i;
        float* q = KROW ? lds + (id >> 4) * kColPitch + 4 * (id & 15) : lds + (id >> 3) * kRowPitch + 4 * (id & 7);
        *reinterpret_cast<floatx4*>(q) = r[i];
    }
}

// the values k = 8 s + 4 h + t, t = 0..3, of row or column x: lane half h's operands of four MFMAs
template <bool KROW>
__device__ __forceinline__ floatx4 tri_frag(const float* lds, int x, int h, int s) {
    if (!KROW) return *reinterpret_cast<const floatx4*>(lds + x * kRowPitch + 8 * s + 4 * h);
    const float* q = lds + (8 * s + 4 * h) * kColPitch + x;
    return floatx4{q[0], q[kColPitch], q[2 * kColPitch], q[3 * kColPitch]};
}

template <Tri KIND>
__global__ __launch_bounds__(256, 2) void tri_product_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                             float* __restrict__ C, uint64_t np, uint64_t ldc,
                                                             uint32_t M, uint32_t N, uint32_t K, float alpha,
                                                             trakhip::GemmBatch batch, float* __restrict__ abs_sums) {
    constexpr bool kKrowA = KIND == Tri::kGram;
    __shared__ __attribute__((aligned(16))) float lds[2][2][kTriFloats];
    const uint32_t tiles_m = M / kTriTile, tiles_n = N / kTriTile;
    uint32_t tm, tn, k_begin = 0, k_end = K;
    if (KIND == Tri::kGram) {
        short_k::triangle_tile(blockIdx.x, tm, tn);
        k_begin = tm * kTriTile / NB * NB;
    } else if (KIND == Tri::kLowerB) {
        tn = blockIdx.x / tiles_m, tm = blockIdx.x % tiles_m;
        k_begin = tn * kTriTile / NB * NB;
    } else {
        tm = tiles_m - 1 - blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
        k_end = (tm * kTriTile / NB + 1) * NB;
    }
    const uint32_t m0 = tm * kTriTile, n0 = tn * kTriTile;
    const uint32_t y = blockIdx.y;
    if (KIND != Tri::kGram) A += batch.a[y], B += batch.b[y], C += batch.c[y];

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int x = lane & 31, h = lane >> 5;
    const int wm = 32 * (wave >> 1), wn = 32 * (wave & 1);
    floatx4 ra[kTriDepth][2], rb[kTriDepth][2];
#pragma unroll
    for (int u = 0; u < kTriDepth; ++u) {
        tri_load<kKrowA>(A, np, m0, k_begin + kTriStep * u, tid, ra[u]);
        tri_load<true>(B, np, n0, k_begin + kTriStep * u, tid, rb[u]);
    }
    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
    for (uint32_t k0 = k_begin; k0 < k_end; k0 += NB) {
        const bool more = k0 + NB < k_end;
#pragma unroll
        for (int u = 0; u < kTriDepth; ++u) {
            // a buffer is written again two steps later, behind the barrier that follows its reads
            tri_store<kKrowA>(lds[u & 1][0], tid, ra[u]);
            tri_store<true>(lds[u & 1][1], tid, rb[u]);
            if (more) {
                tri_load<kKrowA>(A, np, m0, k0 + NB + kTriStep * u, tid, ra[u]);
                tri_load<true>(B, np, n0, k0 + NB + kTriStep * u, tid, rb[u]);
            }
            __syncthreads();
            floatx4 fa[kTriStep / 8], fb[kTriStep / 8];
#pragma unroll
            for (int s = 0; s < kTriStep / 8; ++s) {
                fa[s] = tri_frag<kKrowA>(lds[u & 1][0], wm + x, h, s);
                fb[s] = tri_frag<true>(lds[u & 1][1], wn + x, h, s);
            }
            __builtin_amdgcn_sched_barrier(0);  // all reads of the step in flight before its first MFMA waits
#pragma unroll
            for (int s = 0; s < kTriStep / 8; ++s)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[s & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[s][t], fb[s][t], acc[s & 1], 0, 0, 0);
        }
    }
    const uint32_t col = n0 + wn + x;
    float magnitude = 0.0f;  // kGram: sum of |entries| that this thread stores
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const uint32_t row = m0 + wm + mfma_row(r, h);
        const float v = acc[0][r] + acc[1][r];
        if (KIND != Tri::kGram) {
            C[(uint64_t)row * ldc + col] = alpha * v;
        } else if (row < M && col <= row) {
            C[(uint64_t)row * ldc + col] = v;
            C[(uint64_t)col * ldc + row] = v;
            magnitude += col < row ? 2.0f * fabsf(v) : fabsf(v);
        }
    }
    if (KIND == Tri::kGram && abs_sums) {
        magnitude = workgroup_sum(magnitude);
        if (tid == 0) abs_sums[blockIdx.x] = magnitude;
    }
}

// kGram on 32 x 32 tiles, for matrices whose 64 x 64 tiles leave CUs idle: the four waves share every 128 values of k (a quarter
// of the MFMAs in a row) and their sums are added up at the end, in order.  n = 512: 136 workgroups instead of 36, 15 -> 7 us;
// whole inverse at 1536 402 -> 385, at 2048 532 -> 519.
constexpr int kSmallGramPitch = 32 + 8;  // half-waves in other banks
constexpr uint64_t kSmallGram = 2048;    // up to this n; 64 x 64 tiles are level at 2560 and faster from 3072 on (903 us against 919)

__global__ __launch_bounds__(256, 2) void tri_gram_small_kernel(const float* __restrict__ Li, float* __restrict__ C, uint64_t np,
                                                                uint64_t ldc, uint32_t n, float* __restrict__ abs_sums) {
    __shared__ __attribute__((aligned(16))) float lds[2 * NB * kSmallGramPitch];
    static_assert(2 * NB * kSmallGramPitch >= 4 * 16 * 64, "the sums of four waves");
    uint32_t tm, tn;
    short_k::triangle_tile(blockIdx.x, tm, tn);
    const uint32_t m0 = 32 * tm, n0 = 32 * tn;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, x = lane & 31, h = lane >> 5;
    floatx4 ra[4], rb[4];
    auto load = [&](uint32_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int id = tid + 256 * i;
            const float* row = Li + (uint64_t)(k0 + (id >> 3)) * np + 4 * (id & 7);
            ra[i] = *reinterpret_cast<const floatx4*>(row + m0);
            rb[i] = *reinterpret_cast<const floatx4*>(row + n0);
        }
    };
    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
    uint32_t k0 = m0 / NB * NB;  // Li is zero above its diagonal
    load(k0);
    float* as = lds;
    float* bs = lds + NB * kSmallGramPitch;
    for (; k0 < np; k0 += NB) {
        __syncthreads();  // everyone is done reading the previous rows
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int id = tid + 256 * i;
            *reinterpret_cast<floatx4*>(as + (id >> 3) * kSmallGramPitch + 4 * (id & 7)) = ra[i];
            *reinterpret_cast<floatx4*>(bs + (id >> 3) * kSmallGramPitch + 4 * (id & 7)) = rb[i];
        }
        if (k0 + NB < np) load(k0 + NB);
        __syncthreads();
        float fa[4][4], fb[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int k = 32 * wave + 8 * q + 4 * h + t;
                fa[q][t] = as[k * kSmallGramPitch + x];
                fb[q][t] = bs[k * kSmallGramPitch + x];
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                acc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[q][t], fb[q][t], acc[q & 1], 0, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) lds[(wave * 16 + r) * 64 + lane] = acc[0][r] + acc[1][r];
    __syncthreads();
    float magnitude = 0.0f;
    const uint32_t col = n0 + x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // registers 4 wave .. 4 wave + 3 of the four sums: row 8 wave + 4 h + r
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) v += lds[(w * 16 + 4 * wave + r) * 64 + lane];
        const uint32_t row = m0 + 8 * wave + 4 * h + r;
        if (row < n && col <= row) {
            C[(uint64_t)row * ldc + col] = v;
            C[(uint64_t)col * ldc + row] = v;
            magnitude += col < row ? 2.0f * fabsf(v) : fabsf(v);
        }
    }
    magnitude = workgroup_sum(magnitude);
    if (tid == 0) abs_sums[blockIdx.x] = magnitude;
}

struct Ctx {
    float* W;
    float* L;
    float* Li;
    uint64_t np;
    hipStream_t s;
};

// Inverse of the block lower-triangular factor by recursive halving:
//   [A 0; B C]^-1 = [A^-1 0; -C^-1 B A^-1  C^-1],
// two products per node of the tree (T = B A^-1 into W, which is free once the factorization is
// done, then -C^-1 T into Li).  Diagonal blocks are already inverted.  Nodes of one depth are
// independent, so they are collected per depth and every group of equal shape goes out as one
// batched launch: a dozen launches instead of two per node.
struct Node {
    uint64_t lo, mid, hi;  // block units
};

void collect_nodes(uint64_t lo, uint64_t hi, size_t depth, std::vector<std::vector<Node>>& levels) {
    if (hi - lo <= 1) return;
    const uint64_t mid = lo + (hi - lo) / 2;
    if (levels.size() <= depth) levels.resize(depth + 1);
    levels[depth].push_back({lo, mid, hi});
    collect_nodes(lo, mid, depth + 1, levels);
    collect_nodes(mid, hi, depth + 1, levels);
}

int tri_inverse_impl(Ctx& c, uint64_t nblk) {
    std::vector<std::vector<Node>> levels;
    collect_nodes(0, nblk, 0, levels);
    const uint64_t np = c.np;
    for (size_t d = levels.size(); d-- > 0;) {  // children before parents
        std::vector<Node>& nodes = levels[d];
        std::vector<char> done(nodes.size(), 0);
        for (size_t first = 0; first < nodes.size(); ++first) {
            if (done[first]) continue;
            const uint64_t r = (nodes[first].hi - nodes[first].mid) * NB, q = (nodes[first].mid - nodes[first].lo) * NB;
            trakhip::GemmBatch t_of_b, out_of_t;  // T = B * Ainv;  out = -Cinv * T
            t_of_b.count = out_of_t.count = 0;
            for (size_t i = first; i < nodes.size() && t_of_b.count < trakhip::kGemmBatchMax; ++i) {
                const Node& n = nodes[i];
                if (done[i] || (n.hi - n.mid) * NB != r || (n.mid - n.lo) * NB != q) continue;
                done[i] = 1;
                const uint32_t y = t_of_b.count++;
                out_of_t.count = t_of_b.count;
                const uint64_t below = n.mid * NB * np + n.lo * NB;  // block (mid, lo)
                t_of_b.a[y] = below;                                // B      in L
                t_of_b.b[y] = n.lo * NB * np + n.lo * NB;           // A^-1   in Li
                t_of_b.c[y] = below;                                // T      in W
                out_of_t.a[y] = n.mid * NB * np + n.mid * NB;       // C^-1   in Li
                out_of_t.b[y] = below;                              // T      in W
                out_of_t.c[y] = below;                              // result in Li
            }
            const dim3 grid((uint32_t)(r / kTriTile * (q / kTriTile)), t_of_b.count);
            hipLaunchKernelGGL(tri_product_kernel<Tri::kLowerB>, grid, dim3(256), 0, c.s, c.L, c.Li, c.W, np, np,
                               (uint32_t)r, (uint32_t)q, (uint32_t)q, 1.0f, t_of_b, nullptr);
            hipLaunchKernelGGL(tri_product_kernel<Tri::kLowerA>, grid, dim3(256), 0, c.s, c.Li, c.W, c.Li, np, np,
                               (uint32_t)r, (uint32_t)q, (uint32_t)r, -1.0f, out_of_t, nullptr);
            if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        }
    }
    return TRAKHIP_OK;
}

// The node lists live in host containers; nothing they throw (std::bad_alloc) may cross the C ABI.
int tri_inverse(Ctx& c, uint64_t nblk) {
    try {
        return tri_inverse_impl(c, nblk);
    } catch (...) {
        return TRAKHIP_ERR_HOST_MEMORY;
    }
}

}  // namespace

namespace trakhip {

// Workspace: three np x np matrices (W, L, Li) and the reduction scratch.
size_t spd_inverse_workspace_bytes(uint64_t n) {
    if (n == 0) return 0;
    const uint64_t np = (n + NB - 1) / NB * NB;
    return (size_t)(3 * np * np + kSumBlocks) * sizeof(float);
}

int spd_inverse(const float* A, uint64_t lda, float lambda, float* inv, uint64_t ldi, uint64_t n, int normalize,
                float* mean_abs, int32_t* status, void* ws, size_t ws_bytes, hipStream_t s) {
    if (n == 0) return TRAKHIP_OK;
    if (!A || !inv || !ws) return TRAKHIP_ERR_NULL;
    if (lda < n || ldi < n || n > 0x40000) return TRAKHIP_ERR_SHAPE;
    if (ws_bytes < spd_inverse_workspace_bytes(n)) return TRAKHIP_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(ws) % 16) return TRAKHIP_ERR_ALIGN;
    const uint64_t np = (n + NB - 1) / NB * NB, nblk = np / NB;
    float* W = static_cast<float*>(ws);
    float* L = W + np * np;
    float* Li = L + np * np;
    float* partial = Li + np * np;

    const uint32_t segments = (uint32_t)((np + kInitCols - 1) / kInitCols);
    hipLaunchKernelGGL(spd_init_kernel, dim3((uint32_t)np * segments), dim3(256), 0, s, A, lda, lambda, (uint32_t)n,
                       (uint32_t)np, segments, W, status);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;

    // Diagonal block 0 alone; then per block column j: the panel below it with row j of L^-1, and one launch that holds
    // the trailing update, the next diagonal block and the sums for the next row of L^-1 (spd_step_kernel).  Where there are
    // more blocks (n > 4096): trailing updates of more than 512 tiles by the general product, with the diagonal block in a
    // launch of its own, and L^-1 by recursive halving afterwards (the sums would lengthen the steps).
    hipLaunchKernelGGL(spd_diag_kernel, dim3(1), dim3(kDiagThreads), 0, s, W, np, L, Li, np, 0, status);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
    if (nblk <= kStepBlocks) {
        for (uint32_t j = 0; j + 1 < nblk; ++j) {
            const uint32_t blocks = (uint32_t)nblk - j - 1, tiles = blocks * (blocks + 1) / 2, sums = 8 * (j + 1);
            hipLaunchKernelGGL(spd_panel_kernel, dim3(4 * blocks + 4 * j), dim3(256), 0, s, W, L, Li, np, j, 4 * blocks);
            hipLaunchKernelGGL(spd_step_kernel, dim3(tiles + sums), dim3(kDiagThreads), 0, s, W, L, Li, np, j, sums, status);
            if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        }
        if (nblk > 1) {
            const uint32_t j = (uint32_t)nblk - 1;
            hipLaunchKernelGGL(spd_panel_kernel, dim3(4 * j), dim3(256), 0, s, W, L, Li, np, j, 0u);
            if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        }
    } else {
        for (uint64_t j = 0; j + 1 < nblk; ++j) {
            const uint64_t off = j * NB * np + j * NB;
            const uint64_t rows = np - (j + 1) * NB;
            const uint64_t below = (j + 1) * NB * np + j * NB;
            const uint64_t tr = (j + 1) * NB * np + (j + 1) * NB;
            // panel = W[j+1:, j] * (L_jj^-1)^T
            int e = gemm_nt(W + below, np, Li + off, np, L + below, np, rows, NB, NB, 1.0f, 0.0f, nullptr, s);
            if (e) return e;
            const uint64_t blocks = rows / NB, tiles = blocks * (blocks + 1) / 2;
            if (tiles <= kStepTiles) {
                hipLaunchKernelGGL(spd_step_kernel, dim3((uint32_t)tiles), dim3(kDiagThreads), 0, s, W, L, Li, np, (uint32_t)j,
                                   0u, status);
                if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
                continue;
            }
            // trailing matrix -= panel * panel^T (only the lower triangle of W is ever read)
            e = gemm_nt(L + below, np, L + below, np, W + tr, np, rows, rows, NB, -1.0f, 1.0f, nullptr, s,
                        kGemmLowerTilesOnly);
            if (e) return e;
            hipLaunchKernelGGL(spd_diag_kernel, dim3(1), dim3(kDiagThreads), 0, s, W + tr, np, L + tr, Li + tr, np,
                               (int32_t)(j + 1), status);
            if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        }
        Ctx c = {W, L, Li, np, s};
        const int e = tri_inverse(c, nblk);
        if (e) return e;
    }

    // inverse = Li^T * Li: lower-triangle tiles and their mirror image, so the result is exactly symmetric.  Up to n = 4096 every
    // tile adds up its magnitudes as it stores them (into W, which is free now): one pass over the inverse less, 5 us at n = 512,
    // 7 at 2048, 21 at 4096.
    const uint64_t tiles = (n + kTriTile - 1) / kTriTile, lower = tiles * (tiles + 1) / 2;
    const bool summed = nblk <= kStepBlocks;
    if (np <= kSmallGram) {
        const uint32_t small = (uint32_t)((n + 31) / 32), count = small * (small + 1) / 2;
        hipLaunchKernelGGL(tri_gram_small_kernel, dim3(count), dim3(256), 0, s, Li, inv, np, ldi, (uint32_t)n, W);
        if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        return divide_by_mean(inv, ldi, n, normalize, W, count, mean_abs, s);
    }
    hipLaunchKernelGGL(tri_product_kernel<Tri::kGram>, dim3((uint32_t)lower), dim3(256), 0, s, Li, Li, inv, np, ldi, (uint32_t)n,
                       (uint32_t)n, (uint32_t)np, 1.0f, GemmBatch{}, summed ? W : nullptr);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
    return divide_by_mean(inv, ldi, n, normalize, summed ? W : partial, summed ? (uint32_t)lower : 0u, mean_abs, s);
}

}  // namespace trakhip

namespace {

// ---- inverse of a general matrix: elimination with partial pivoting -----------------------------------------
//
// For the matrices the Cholesky route above refuses: a Gram matrix rounded to fp16, or one of deficient
// rank with lambda = 0, is symmetric but need not be positive definite.  The reference inverts every
// matrix with LU and partial pivoting (torch.linalg.inv, trak/score_computers.py:163); this is the same
// pivoting on the device.  The augmented matrix [A + lambda I | I] (np x 2 np, np = n padded with an
// identity block to a multiple of 128) is reduced to [I | A^-1] block of columns by block of columns.
// For a block J of OB columns starting at j0 (the rows above j0 are finished pivot rows of earlier blocks):
//   1. the block's columns are factored as in a right-looking LU, SP columns at a time: gj_panel_kernel
//      (ONE workgroup holds rows j.. of the SP panel columns in registers) eliminates them column by column
//      with row pivoting (largest magnitude, lowest row on ties), leaves the multipliers (|l| <= 1) in the
//      rows below, the pivot rows' numbers, where the rows they displace go, and the packed factors of the
//      SP x SP pivot block; gj_rows_kernel moves the rows of the block's columns into place and turns the
//      pivot rows right of the panel into L11^-1 * (pivot rows); a product with SP values of k updates the
//      block's columns further right in the rows below.  Afterwards rows j0.. of J hold L \ U of the block.
//   2. the rest of the matrix (all columns right of the block, the identity half included) gets the block's
//      OB eliminations at once: gj_block_rows_kernel (one thread per column) applies the row moves, computes
//      Y = L_J^-1 * (pivot rows) (kept aside) and R = U_J^-1 * Y, which replaces the pivot rows;
//          rows below the block:  W[r, rest] -= L[r, J] * Y        (the LU update, multipliers at most 1)
//          rows above the block:  W[r, rest] -= W[r, J] * R        (the Gauss-Jordan part: back substitution
//                                                                   folded into the elimination)
//      two products with OB values of k.  No permutation is left to undo at the end: the row moves act on
//      whole rows of [A | I].
// OB = 64 from np = 3072 on (four or eight panels per block: the products over the rest move 12 np^2 bytes per
// block instead of per panel); below that OB = SP = 16 (fewer launches per column, which is what small
// matrices pay for).
//
// (Updating the rows below with the panel's original entries times D^-1 * (pivot rows), D the pivot block, would
// be one product for all rows; it is not done because its rounding errors grow with the condition of D, where
// the multipliers are at most 1.)

constexpr int kGjThreads = 1024;
constexpr int kGjMaxSp = 16;

struct GjStep {
    int32_t piv[kGjMaxSp];   // the row that becomes row j + c
    int32_t from[kGjMaxSp];  // rows of the pivot positions that were not chosen ...
    int32_t to[kGjMaxSp];    // ... and the vacated positions they move to
    int32_t moves;
    int32_t pad[3];
    float lu[kGjMaxSp * kGjMaxSp];  // the pivot block as packed factors: unit lower L below the diagonal, U on and above
};

__global__ __launch_bounds__(256) void gj_init_kernel(const float* __restrict__ A, uint64_t lda, float lambda,
                                                      uint64_t n, uint64_t np, float* __restrict__ W,
                                                      int32_t* __restrict__ status) {
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx == 0 && status) *status = 0;
    if (idx >= np * 2 * np) return;
    const uint64_t i = idx / (2 * np), j = idx % (2 * np);
    float v;
    if (j >= np)
        v = (j - np == i) ? 1.0f : 0.0f;
    else if (i < n && j < n)
        v = A[i * lda + j] + (i == j ? lambda : 0.0f);
    else
        v = (i == j) ? 1.0f : 0.0f;
    W[idx] = v;
}

// larger magnitude wins; on equal magnitudes the lower row (what a sequential search finds first)
__device__ __forceinline__ void gj_better(uint32_t& key, uint32_t& row, uint32_t okey, uint32_t orow) {
    if (okey > key || (okey == key && orow < row)) {
        key = okey;
        row = orow;
    }
}

template <class F, int... S>
__device__ __forceinline__ void gj_for_each(F& f, std::integer_sequence<int, S...>) {
    (f(std::integral_constant<int, S>{}), ...);
}

template <int SP, int RPT>
__global__ __launch_bounds__(kGjThreads) void gj_panel_kernel(float* __restrict__ W, uint64_t ld, uint32_t np,
                                                              uint32_t j, GjStep* __restrict__ step,
                                                              int32_t* __restrict__ status) {
    __shared__ uint32_t cand_key[kGjThreads / 64], cand_row[kGjThreads / 64];
    __shared__ float lu[SP][SP + 1];  // row c: the pivot row of column c as it was when chosen (packed L \ U)
    __shared__ int32_t piv[SP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float a[RPT][SP];
    uint32_t live = 0;  // bit i: row i of this thread exists and has not been a pivot
    // row slots of a thread that hold rows at all at this j (the panel shrinks as j grows)
    const int slots = (int)((np - j + kGjThreads - 1) / kGjThreads);
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        const uint32_t r = j + (uint32_t)tid + (uint32_t)kGjThreads * i;
        if (r < np) {
            live |= 1u << i;
            const float4* src = reinterpret_cast<const float4*>(W + (uint64_t)r * ld + j);
#pragma unroll
            for (int c4 = 0; c4 < SP / 4; ++c4) {
                const float4 v = src[c4];
                a[i][4 * c4] = v.x, a[i][4 * c4 + 1] = v.y, a[i][4 * c4 + 2] = v.z, a[i][4 * c4 + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int c = 0; c < SP; ++c) a[i][c] = 0.0f;
        }
    }
    // (the columns are written out through a compile-time sequence: `#pragma unroll` gives up on a body
    // of this size, and the register array would be indexed at run time, i.e. live in scratch memory)
    auto column = [&](auto c_const) __attribute__((always_inline)) {
        constexpr int c = decltype(c_const)::value;
        // the pivot of column c: largest |a| among the rows that have not been pivots
        uint32_t key = 0, row = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            if (i < slots) {  // the same for the whole workgroup: a scalar branch
                if (live & (1u << i))
                    gj_better(key, row, __float_as_uint(fabsf(a[i][c])), j + (uint32_t)tid + (uint32_t)kGjThreads * i);
            }
        }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1)
            gj_better(key, row, (uint32_t)__shfl_xor((int)key, d, 64), (uint32_t)__shfl_xor((int)row, d, 64));
        if (lane == 0) cand_key[wave] = key, cand_row[wave] = row;
        __syncthreads();
        // the sixteen waves' candidates, one per lane of every group of sixteen lanes, reduced inside the group
        static_assert(kGjThreads / 64 == 16, "one candidate per lane of a group of sixteen");
        key = cand_key[lane & 15], row = cand_row[lane & 15];
#pragma unroll
        for (int d = 1; d < 16; d <<= 1)
            gj_better(key, row, (uint32_t)__shfl_xor((int)key, d, 64), (uint32_t)__shfl_xor((int)row, d, 64));
        // its owner - one thread, known to all: row = j + thread + 1024 * slot - publishes the row (multipliers of
        // earlier columns in front, the eliminated row behind)
        const uint32_t rel = __builtin_amdgcn_readfirstlane(row) - j;
        const int owner = (int)(rel % kGjThreads), owner_slot = (int)(rel / kGjThreads);
        if (tid == owner) {
#pragma unroll
            for (int i = 0; i < RPT; ++i) {
                if (i == owner_slot) {
                    live &= ~(1u << i);
#pragma unroll
                    for (int c2 = 0; c2 < SP; ++c2) lu[c][c2] = a[i][c2];
                    if (a[i][c] == 0.0f && status) *status = (int32_t)(j + c + 1);  // exactly singular
                }
            }
            piv[c] = (int32_t)(rel + j);
        }
        __syncthreads();
        // multipliers by the reciprocal of the pivot, as LAPACK's unblocked LU scales a column
        const float rpivot = 1.0f / lu[c][c];
#pragma unroll
        for (int i = 0; i < RPT; ++i) {
            if (i < slots) {
                if (live & (1u << i)) {
                    const float l = a[i][c] * rpivot;
                    a[i][c] = l;
#pragma unroll
                    for (int c2 = c + 1; c2 < SP; ++c2) a[i][c2] = fmaf(-l, lu[c][c2], a[i][c2]);
                }
            }
        }
    };
    gj_for_each(column, std::make_integer_sequence<int, SP>{});
    // the rows that were never pivots now hold their SP multipliers: back to the matrix, where the row moves and
    // the update of the other columns find them
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
        if (i < slots && (live & (1u << i))) {
            float4* dst = reinterpret_cast<float4*>(W + (uint64_t)(j + (uint32_t)tid + (uint32_t)kGjThreads * i) * ld + j);
#pragma unroll
            for (int c4 = 0; c4 < SP / 4; ++c4)
                dst[c4] = make_float4(a[i][4 * c4], a[i][4 * c4 + 1], a[i][4 * c4 + 2], a[i][4 * c4 + 3]);
        }
    }
    // D = (rows piv[0..SP) of the panel as they were) = L U with the packed factors in lu
    if (tid < SP) {
#pragma unroll
        for (int q = 0; q < SP; ++q) step->lu[tid * SP + q] = lu[tid][q];
        step->piv[tid] = piv[tid];
    }
    if (tid == 0) {
        // rows at the pivot positions j .. j+SP-1 that were not chosen go to the positions that the chosen
        // rows from further down leave behind, both in ascending order
        int32_t moves = 0, to_n = 0;
        for (int q = 0; q < SP; ++q) {
            const int32_t pos = (int32_t)j + q;
            bool chosen = false;
            for (int c = 0; c < SP; ++c) chosen |= piv[c] == pos;
            if (!chosen) step->from[moves++] = pos;
        }
        // vacated positions below the pivot block, ascending (selection over at most SP values)
        int32_t last = (int32_t)j + SP - 1;
        for (int m = 0; m < moves; ++m) {
            int32_t best = 0x7FFFFFFF;
            for (int c = 0; c < SP; ++c)
                if (piv[c] > last && piv[c] < best) best = piv[c];
            step->to[to_n++] = best;
            last = best;
        }
        step->moves = moves;
    }
}

// One thread per column of [col_begin, col_end): the rows move into place (pivot rows to j.., the rows they
// displace to the vacated positions).  Left of the panel that is all (multipliers of earlier panels travel with
// their rows); in the panel's columns the pivot rows become the packed factors; right of it they become
// Y = L^-1 * (pivot rows).  With y_out (the one-panel blocks of small matrices, where "right of the panel" is the
// whole rest) Y goes to y_out[c * ld + col] and the pivot rows become R = U^-1 * Y.
template <int SP>
__global__ __launch_bounds__(256) void gj_rows_kernel(float* __restrict__ W, uint64_t ld, uint32_t j, uint32_t col_begin,
                                                      uint32_t col_end, const GjStep* __restrict__ step,
                                                      float* __restrict__ y_out) {
    __shared__ GjStep st;
    for (uint32_t i = threadIdx.x; i < sizeof(GjStep) / 4; i += 256)
        reinterpret_cast<uint32_t*>(&st)[i] = reinterpret_cast<const uint32_t*>(step)[i];
    __syncthreads();
    const uint64_t col = (uint64_t)col_begin + (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (col >= col_end) return;
    float v[SP], d[SP];
#pragma unroll
    for (int c = 0; c < SP; ++c) v[c] = W[(uint64_t)st.piv[c] * ld + col];
#pragma unroll
    for (int m = 0; m < SP; ++m) d[m] = m < st.moves ? W[(uint64_t)st.from[m] * ld + col] : 0.0f;
    if (col >= j && col < (uint64_t)j + SP) {
#pragma unroll
        for (int c = 0; c < SP; ++c) v[c] = st.lu[c * SP + (int)(col - j)];
    } else if (col >= (uint64_t)j + SP) {
        // forward substitution with the unit lower factor
#pragma unroll
        for (int r = 1; r < SP; ++r)
#pragma unroll
            for (int q = 0; q < r; ++q) v[r] = fmaf(-st.lu[r * SP + q], v[q], v[r]);
        if (y_out) {
#pragma unroll
            for (int c = 0; c < SP; ++c) y_out[(uint64_t)c * ld + col] = v[c];
            // back substitution with the upper one
#pragma unroll
            for (int r = SP - 1; r >= 0; --r) {
#pragma unroll
                for (int q = r + 1; q < SP; ++q) v[r] = fmaf(-st.lu[r * SP + q], v[q], v[r]);
                v[r] = v[r] / st.lu[r * SP + r];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < SP; ++c) W[(uint64_t)(j + c) * ld + col] = v[c];
#pragma unroll
    for (int m = 0; m < SP; ++m)
        if (m < st.moves) W[(uint64_t)st.to[m] * ld + col] = d[m];
}

__global__ __launch_bounds__(256) void gj_copy_out_kernel(const float* __restrict__ W, uint64_t ld, uint64_t np,
                                                          uint64_t n, float* __restrict__ inv, uint64_t ldi) {
    const uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= n * n) return;
    const uint64_t i = idx / n, c = idx % n;
    inv[i * ldi + c] = W[i * ld + np + c];
}

constexpr int kGjOb = 64;  // columns of a block of the large-matrix route

// One thread per column of the rest (col >= j0 + kGjOb).  The block's panels' row moves are applied one panel
// after the other (the pivot rows collect in LDS, one column of v per thread); then, with the factors L \ U that
// rows j0.. of the block's columns hold (F, read with wave-uniform addresses), Y = L^-1 v goes to
// y_out[c * ld + col] and R = U^-1 Y to rows j0.. of the column.  The 64 values are worked on eight at a time.
template <int SP>
__global__ __launch_bounds__(256) void gj_block_rows_kernel(float* __restrict__ W, uint64_t ld, uint32_t np, uint32_t j0,
                                                            const float* __restrict__ F,
                                                            const GjStep* __restrict__ steps, float* __restrict__ y_out) {
    constexpr int T = 8, NB8 = kGjOb / T, PANELS = kGjOb / SP;
    __shared__ float v[kGjOb][256];
    const int tid = threadIdx.x;
    const uint64_t col = (uint64_t)j0 + kGjOb + (uint64_t)blockIdx.x * 256 + tid;
    if (col >= 2ull * np) return;  // (no barrier below: a thread only reads the column of v that it wrote)
    for (int p = 0; p < PANELS; ++p) {
        const GjStep* st = steps + p;
        const int moves = st->moves;
        float x[SP], d[SP];
#pragma unroll
        for (int c = 0; c < SP; ++c) x[c] = W[(uint64_t)st->piv[c] * ld + col];
#pragma unroll
        for (int m = 0; m < SP; ++m) d[m] = m < moves ? W[(uint64_t)st->from[m] * ld + col] : 0.0f;
#pragma unroll
        for (int c = 0; c < SP; ++c) v[p * SP + c][tid] = x[c];
        // (a position j0 + p SP + c is never a source of a later panel: those take rows from further down)
#pragma unroll
        for (int m = 0; m < SP; ++m)
            if (m < moves) W[(uint64_t)st->to[m] * ld + col] = d[m];
    }
    // forward substitution with the unit lower factor, block row by block row
    for (int rb = 0; rb < NB8; ++rb) {
        float x[T];
#pragma unroll
        for (int i = 0; i < T; ++i) x[i] = v[rb * T + i][tid];
        for (int cb = 0; cb < rb; ++cb) {
            float y[T];
#pragma unroll
            for (int q = 0; q < T; ++q) y[q] = v[cb * T + q][tid];
            const float* l = F + (uint64_t)(rb * T) * ld + cb * T;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int q = 0; q < T; ++q) x[i] = fmaf(-l[(uint64_t)i * ld + q], y[q], x[i]);
        }
        const float* l = F + (uint64_t)(rb * T) * ld + rb * T;
#pragma unroll
        for (int i = 1; i < T; ++i)
#pragma unroll
            for (int q = 0; q < i; ++q) x[i] = fmaf(-l[(uint64_t)i * ld + q], x[q], x[i]);
#pragma unroll
        for (int i = 0; i < T; ++i) {
            v[rb * T + i][tid] = x[i];
            y_out[(uint64_t)(rb * T + i) * ld + col] = x[i];
        }
    }
    // back substitution with the upper factor
    for (int rb = NB8 - 1; rb >= 0; --rb) {
        float x[T];
#pragma unroll
        for (int i = 0; i < T; ++i) x[i] = v[rb * T + i][tid];
        for (int cb = rb + 1; cb < NB8; ++cb) {
            float y[T];
#pragma unroll
            for (int q = 0; q < T; ++q) y[q] = v[cb * T + q][tid];
            const float* u = F + (uint64_t)(rb * T) * ld + cb * T;
#pragma unroll
            for (int i = 0; i < T; ++i)
#pragma unroll
                for (int q = 0; q < T; ++q) x[i] = fmaf(-u[(uint64_t)i * ld + q], y[q], x[i]);
        }
        const float* u = F + (uint64_t)(rb * T) * ld + rb * T;
#pragma unroll
        for (int i = T - 1; i >= 0; --i) {
#pragma unroll
            for (int q = i + 1; q < T; ++q) x[i] = fmaf(-u[(uint64_t)i * ld + q], x[q], x[i]);
            x[i] = x[i] / u[(uint64_t)i * ld + i];
        }
#pragma unroll
        for (int i = 0; i < T; ++i) {
            v[rb * T + i][tid] = x[i];
            W[(uint64_t)(j0 + rb * T + i) * ld + col] = x[i];
        }
    }
}

// the two products that carry a block's eliminations to the columns right of it (OB values of k):
// rows above the block with their own entries of the block's columns times R (which now is rows j0.. of W),
// rows below with their multipliers times Y
int gj_update_rest(float* W, uint64_t ld, uint32_t np, uint32_t j0, uint32_t ob, const float* Y, hipStream_t s) {
    const uint32_t end = j0 + ob;
    const uint64_t rest = 2ull * np - end;
    if (ob < kGjOb && j0 > 0 && end < np) {
        // one-panel blocks (small matrices): both products in one launch, a launch being what they cost.
        // Y lies behind W in the same workspace, so one base pointer serves both B operands.
        trakhip::GemmBatch two;
        two.count = 2;
        two.a[0] = j0, two.b[0] = (uint64_t)j0 * ld + end, two.c[0] = end, two.m[0] = j0;
        two.a[1] = (uint64_t)end * ld + j0, two.b[1] = (uint64_t)(Y - W) + end, two.c[1] = (uint64_t)end * ld + end;
        two.m[1] = np - end;
        const uint64_t m = j0 > np - end ? j0 : np - end;
        return trakhip::gemm_nn_batched(W, ld, W, ld, W, ld, m, rest, ob, -1.0f, 1.0f, two, s);
    }
    if (j0 > 0) {
        const int e = trakhip::gemm_nn(W + j0, ld, W + (uint64_t)j0 * ld + end, ld, W + end, ld, j0, rest, ob, -1.0f, 1.0f,
                                       s, 0);
        if (e) return e;
    }
    if (end < np)
        return trakhip::gemm_nn(W + (uint64_t)end * ld + j0, ld, Y + end, ld, W + (uint64_t)end * ld + end, ld, np - end,
                                rest, ob, -1.0f, 1.0f, s, 0);
    return TRAKHIP_OK;
}

// blocks of one panel: the whole rest of the matrix after every SP columns
template <int SP, int RPT>
int gj_run_flat(float* W, float* Y, uint32_t np, GjStep* steps, int32_t* status, hipStream_t s) {
    const uint64_t ld = 2ull * np;
    for (uint32_t j = 0; j < np; j += SP) {
        GjStep* st = steps + (j / SP) % 2;  // two records in turn: the next panel never overwrites one still in use
        hipLaunchKernelGGL((gj_panel_kernel<SP, RPT>), dim3(1), dim3(kGjThreads), 0, s, W, ld, np, j, st, status);
        const uint32_t cols = 2 * np - j;
        hipLaunchKernelGGL((gj_rows_kernel<SP>), dim3((cols + 255) / 256), dim3(256), 0, s, W, ld, j, j, 2 * np, st, Y);
        if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        const int e = gj_update_rest(W, ld, np, j, SP, Y, s);
        if (e) return e;
    }
    return TRAKHIP_OK;
}

// blocks of kGjOb columns, kGjOb / SP panels each
template <int SP, int RPT>
int gj_run(float* W, float* Y, uint32_t np, GjStep* steps, int32_t* status, hipStream_t s) {
    const uint64_t ld = 2ull * np;
    for (uint32_t j0 = 0; j0 < np; j0 += kGjOb) {
        const uint32_t end = j0 + kGjOb;
        for (uint32_t j = j0; j < end; j += SP) {
            GjStep* st = steps + (j - j0) / SP;
            hipLaunchKernelGGL((gj_panel_kernel<SP, RPT>), dim3(1), dim3(kGjThreads), 0, s, W, ld, np, j, st, status);
            hipLaunchKernelGGL((gj_rows_kernel<SP>), dim3(1), dim3(256), 0, s, W, ld, j, j0, end, st, (float*)nullptr);
            if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
            if (j + SP < end && j + SP < np) {
                // the block's columns right of the panel, rows below it
                const int e = trakhip::gemm_nn(W + (uint64_t)(j + SP) * ld + j, ld, W + (uint64_t)j * ld + j + SP, ld,
                                               W + (uint64_t)(j + SP) * ld + j + SP, ld, np - j - SP, end - j - SP, SP,
                                               -1.0f, 1.0f, s, 0);
                if (e) return e;
            }
        }
        const uint32_t rest = 2 * np - end;
        hipLaunchKernelGGL((gj_block_rows_kernel<SP>), dim3((rest + 255) / 256), dim3(256), 0, s, W, ld, np, j0,
                           W + (uint64_t)j0 * ld + j0, steps, Y);
        if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
        const int e = gj_update_rest(W, ld, np, j0, kGjOb, Y, s);
        if (e) return e;
    }
    return TRAKHIP_OK;
}

}  // namespace

namespace trakhip {

constexpr uint64_t kGeneralInverseMaxN = 12288;

size_t general_inverse_workspace_bytes(uint64_t n) {
    if (n == 0 || n > kGeneralInverseMaxN) return 0;
    const uint64_t np = (n + NB - 1) / NB * NB;
    return (size_t)(2 * np * np + 2 * np * kGjOb + kSumBlocks) * sizeof(float) + (kGjOb / 8) * sizeof(GjStep);
}

int general_inverse(const float* A, uint64_t lda, float lambda, float* inv, uint64_t ldi, uint64_t n, int normalize,
                    float* mean_abs, int32_t* status, void* ws, size_t ws_bytes, hipStream_t s) {
    if (n == 0) return TRAKHIP_OK;
    if (!A || !inv || !ws) return TRAKHIP_ERR_NULL;
    if (lda < n || ldi < n || n > kGeneralInverseMaxN) return TRAKHIP_ERR_SHAPE;
    if (ws_bytes < general_inverse_workspace_bytes(n)) return TRAKHIP_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(ws) % 16) return TRAKHIP_ERR_ALIGN;
    const uint64_t np = (n + NB - 1) / NB * NB;
    float* W = static_cast<float*>(ws);
    float* Y = W + 2 * np * np;  // kGjOb x 2 np: L^-1 * (pivot rows) of the block at work
    float* partial = Y + 2 * np * kGjOb;
    GjStep* steps = reinterpret_cast<GjStep*>(partial + kSumBlocks);
    hipLaunchKernelGGL(gj_init_kernel, dim3((uint32_t)((2 * np * np + 255) / 256)), dim3(256), 0, s, A, lda, lambda, n,
                       np, W, status);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
    // the panel's rows live in the registers of one workgroup: 16 columns of up to 6144 rows, or 8 of up to 12288
    // the panel's rows live in the registers of one workgroup: 16 columns of up to 6144 rows, or 8 of up to 12288
    const int e = np < 3072      ? gj_run_flat<16, 6>(W, Y, (uint32_t)np, steps, status, s)
                  : np <= 6144   ? gj_run<16, 6>(W, Y, (uint32_t)np, steps, status, s)
                                 : gj_run<8, 12>(W, Y, (uint32_t)np, steps, status, s);
    if (e) return e;
    hipLaunchKernelGGL(gj_copy_out_kernel, dim3((uint32_t)((n * n + 255) / 256)), dim3(256), 0, s, W, 2 * np, np, n, inv,
                       ldi);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
    return divide_by_mean(inv, ldi, n, normalize, partial, 0u, mean_abs, s);
}

}  // namespace trakhip
