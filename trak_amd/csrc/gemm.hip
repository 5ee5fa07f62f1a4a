// fp32 GEMM on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32) for the scoring path.
//
// Stands in for the three torch matmuls of BasicScoreComputer: `block.T @ block`
// (trak/score_computers.py:153), `block @ xtx_inv` (:176) and `features @ target_grads.t()`
// (trak/utils.py:131), and is the building block of the blocked SPD inverse (spd.hip).
//
//   C[M, N] = alpha * op(A) * op(B) + beta * C      (then row i *= row_scale[i])
//
// Each operand is described by how it is stored relative to the contraction index k:
//   "row-k"  (KMAJOR = false): element (x, k) at ptr[x * ld + k]   (k contiguous)
//   "k-row"  (KMAJOR = true):  element (x, k) at ptr[k * ld + x]   (x contiguous)
// NT = (row-k, row-k), TN = (k-row, k-row), NN = (row-k, k-row).
//
// Workgroup = 256 threads = 4 waves in a 2x2 grid, 128 x BN tile of C (BN = 128 or 256), k step
// 16, two LDS buffers.  A wave owns 64 x BN/2 of C = 2 x (2 or 4) MFMA tiles (64 or 128
// accumulator VGPRs); the wide tile does twice the multiply-adds per LDS round trip and barrier
// and is used when C has at least 256 columns.  The MFMA sums over k in any order, so lane half
// h (= lane / 32) is given k = 8*s + 4*h + t for the t-th MFMA of sub-step s: a row-k operand
// then needs ONE 16-byte LDS read per four MFMAs.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "short_k_tile.h"
#include "trakhip_internal.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int BM = 128, BKT = 16;
constexpr int kThreads = 256;
constexpr int kRowKStride = BKT + 4;   // floats; 80 B rows keep 16-byte reads conflict free
// an operand tile has ROWS rows (128 or 256) and BKT k-values; k-row tiles use ROWS floats per k
template <int ROWS>
struct Tile {
    static constexpr int pieces = ROWS * BKT / 4 / kThreads;  // 16-byte pieces per thread
    static constexpr int floats = ROWS * kRowKStride;          // >= BKT * ROWS
};

// ---- global -> registers -------------------------------------------------------------------

template <bool KMAJOR, bool ALIGNED, int ROWS>
__device__ __forceinline__ void load_tile(const float* __restrict__ p, uint64_t ld, uint64_t x0, uint64_t X,
                                          uint64_t k0, uint64_t K, int tid, float4 (&r)[Tile<ROWS>::pieces]) {
#pragma unroll
    for (int i = 0; i < Tile<ROWS>::pieces; ++i) {
        const int id = tid + kThreads * i;
        float4 v = {0.f, 0.f, 0.f, 0.f};
        if (!KMAJOR) {
            const uint64_t x = x0 + (id >> 2), k = k0 + 4 * (id & 3);
            if (x < X && k < K) {
                const float* q = p + x * ld + k;
                if (ALIGNED && k + 4 <= K) {
                    v = *reinterpret_cast<const float4*>(q);
                } else {
                    v.x = q[0];
                    if (k + 1 < K) v.y = q[1];
                    if (k + 2 < K) v.z = q[2];
                    if (k + 3 < K) v.w = q[3];
                }
            }
        } else {
            const uint64_t k = k0 + id / (ROWS / 4), x = x0 + 4 * (id % (ROWS / 4));
            if (k < K && x < X) {
                const float* q = p + k * ld + x;
                if (ALIGNED && x + 4 <= X) {
                    v = *reinterpret_cast<const float4*>(q);
                } else {
                    v.x = q[0];
                    if (x + 1 < X) v.y = q[1];
                    if (x + 2 < X) v.z = q[2];
                    if (x + 3 < X) v.w = q[3];
                }
            }
        }
        r[i] = v;
    }
}

template <bool KMAJOR, int ROWS>
__device__ __forceinline__ void store_tile(float* lds, int tid, const float4 (&r)[Tile<ROWS>::pieces]) {
#pragma unroll
    for (int i = 0; i < Tile<ROWS>::pieces; ++i) {
        const int id = tid + kThreads * i;
        if (!KMAJOR)
            *reinterpret_cast<float4*>(lds + (id >> 2) * kRowKStride + 4 * (id & 3)) = r[i];
        else
            *reinterpret_cast<float4*>(lds + (id / (ROWS / 4)) * ROWS + 4 * (id % (ROWS / 4))) = r[i];
    }
}

// The 4 operand values (t = 0..3) of lane (x, h) for sub-step s.
template <bool KMAJOR, int ROWS>
__device__ __forceinline__ float4 read_frag(const float* lds, int x, int h, int s) {
    if (!KMAJOR) return *reinterpret_cast<const float4*>(lds + x * kRowKStride + 8 * s + 4 * h);
    const float* q = lds + (8 * s + 4 * h) * ROWS + x;
    float4 v;
    v.x = q[0];
    v.y = q[ROWS];
    v.z = q[2 * ROWS];
    v.w = q[3 * ROWS];
    return v;
}

// One 128 x BN tile of C, tile number `tile` of a row-major tile grid tiles_n wide.
template <bool AK, bool BK, bool ALIGNED, int WN>
__device__ __forceinline__ void gemm_tile(const float* __restrict__ A, uint64_t lda, const float* __restrict__ B,
                                          uint64_t ldb, float* __restrict__ C, uint64_t ldc, uint64_t M, uint64_t N,
                                          uint64_t K, float alpha, float beta, const float* __restrict__ row_scale,
                                          uint32_t tiles_n, uint32_t flags, uint32_t tile) {
    constexpr int BN = 64 * WN;  // two waves side by side, WN 32-column MFMA tiles each
    __shared__ __attribute__((aligned(16))) float lds[2][Tile<BM>::floats + Tile<BN>::floats];

    const uint32_t tile_m = tile / tiles_n, tile_n = tile % tiles_n;
    const uint64_t m0 = (uint64_t)tile_m * BM, n0 = (uint64_t)tile_n * BN;
    // tiles strictly above the diagonal are not needed by a caller that reads the lower triangle
    if ((flags & trakhip::kGemmLowerTilesOnly) && n0 > m0 + BM - 1) return;

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63;
    const int wm = wave >> 1, wn = wave & 1;
    const int x = lane & 31, h = lane >> 5;

    floatx16 acc[2][WN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const uint64_t nk = (K + BKT - 1) / BKT;
    float4 ra[Tile<BM>::pieces], rb[Tile<BN>::pieces];
    load_tile<AK, ALIGNED, BM>(A, lda, m0, M, 0, K, tid, ra);
    load_tile<BK, ALIGNED, BN>(B, ldb, n0, N, 0, K, tid, rb);
    store_tile<AK, BM>(lds[0], tid, ra);
    store_tile<BK, BN>(lds[0] + Tile<BM>::floats, tid, rb);
    __syncthreads();

    for (uint64_t kt = 0; kt < nk; ++kt) {
        const int cur = (int)(kt & 1);
        if (kt + 1 < nk) {
            load_tile<AK, ALIGNED, BM>(A, lda, m0, M, (kt + 1) * BKT, K, tid, ra);
            load_tile<BK, ALIGNED, BN>(B, ldb, n0, N, (kt + 1) * BKT, K, tid, rb);
        }
        const float* as = lds[cur];
        const float* bs = lds[cur] + Tile<BM>::floats;
#pragma unroll
        for (int s = 0; s < BKT / 8; ++s) {
            float4 fa[2], fb[WN];
#pragma unroll
            for (int i = 0; i < 2; ++i) fa[i] = read_frag<AK, BM>(as, wm * 64 + 32 * i + x, h, s);
#pragma unroll
            for (int j = 0; j < WN; ++j) fb[j] = read_frag<BK, BN>(bs, wn * (32 * WN) + 32 * j + x, h, s);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < WN; ++j) {
                        const float av = t == 0 ? fa[i].x : (t == 1 ? fa[i].y : (t == 2 ? fa[i].z : fa[i].w));
                        const float bv = t == 0 ? fb[j].x : (t == 1 ? fb[j].y : (t == 2 ? fb[j].z : fb[j].w));
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[i][j], 0, 0, 0);
                    }
        }
        if (kt + 1 < nk) {
            store_tile<AK, BM>(lds[cur ^ 1], tid, ra);
            store_tile<BK, BN>(lds[cur ^ 1] + Tile<BM>::floats, tid, rb);
        }
        __syncthreads();
    }

    // D[m][n] of a 32x32 MFMA: lane holds column n = lane % 32; register r holds row
    // 8*(r/4) + 4*(lane/32) + r%4.  When C is accumulated into, its old values are fetched for 32 rows
    // at a time before any of them is overwritten (loads and stores through one pointer would
    // otherwise alternate, one memory round trip per element).
    const uint64_t col0 = n0 + wn * (32 * WN) + x;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint64_t row0 = m0 + wm * 64 + 32 * i + 4 * h;
        floatx16 prev[WN];
        if (beta != 0.0f) {
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint64_t row = row0 + 8 * (r >> 2) + (r & 3), col = col0 + 32 * j;
                    prev[j][r] = (row < M && col < N) ? C[row * ldc + col] : 0.0f;
                }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint64_t row = row0 + 8 * (r >> 2) + (r & 3);
            if (row >= M) continue;
            const float rs = row_scale ? row_scale[row] : 1.0f;
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint64_t col = col0 + 32 * j;
                if (col >= N) continue;
                float v = alpha * acc[i][j][r];
                if (beta != 0.0f) v += beta * prev[j][r];
                C[row * ldc + col] = v * rs;
            }
        }
    }
}

template <bool AK, bool BK, bool ALIGNED, int WN>
__global__ __launch_bounds__(kThreads, 2) void gemm_kernel(const float* __restrict__ A, uint64_t lda,
                                                           const float* __restrict__ B, uint64_t ldb,
                                                           float* __restrict__ C, uint64_t ldc, uint64_t M,
                                                           uint64_t N, uint64_t K, float alpha, float beta,
                                                           const float* __restrict__ row_scale,
                                                           uint32_t tiles_n, uint32_t flags) {
    gemm_tile<AK, BK, ALIGNED, WN>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, tiles_n, flags,
                                   blockIdx.x);
}

// Several independent products of one shape in one launch: product y = blockIdx.y works on
// A + batch.a[y], B + batch.b[y], C + batch.c[y] (element offsets).  NN operands, 128 x 128 tiles.
__global__ __launch_bounds__(kThreads, 2) void gemm_nn_batched_kernel(const float* __restrict__ A, uint64_t lda,
                                                                      const float* __restrict__ B, uint64_t ldb,
                                                                      float* __restrict__ C, uint64_t ldc, uint64_t M,
                                                                      uint64_t N, uint64_t K, float alpha, float beta,
                                                                      uint32_t tiles_n, trakhip::GemmBatch batch) {
    const uint32_t y = blockIdx.y;
    const uint64_t my = batch.m[y] ? batch.m[y] : M;
    if ((uint64_t)(blockIdx.x / tiles_n) * BM >= my) return;  // (the whole workgroup: the grid is sized for the call's M)
    gemm_tile<false, true, true, 2>(A + batch.a[y], lda, B + batch.b[y], ldb, C + batch.c[y], ldc, my, N, K, alpha,
                                    beta, nullptr, tiles_n, 0u, blockIdx.x);
}

// NT product with a short contraction (K <= 128, the panel width of the blocked factorization):
// C[M, N] = alpha * A[M, K] * B[N, K]^T + beta * C, ROWS x 128 tiles.  The general kernel walks k in
// steps of 16 with one global-memory round trip per step, which is all latency when there are
// only eight steps; here both operand tiles are loaded whole (one round trip, one barrier) and the
// MFMAs run back to back.  Needs 16-byte aligned rows and K a multiple of 8.
// ROWS = 128: 2 x 2 waves of 64 x 64, 135 KB of LDS, one workgroup per CU.  ROWS = 32: 1 x 4 waves of
// 32 x 32 for products with few rows of tiles (the panel: N = 128), four times as many workgroups.
template <int ROWS>
__global__ __launch_bounds__(kThreads, 1) void gemm_nt_short_k_kernel(const float* __restrict__ A, uint64_t lda,
                                                                      const float* __restrict__ B, uint64_t ldb,
                                                                      float* __restrict__ C, uint64_t ldc, uint64_t M,
                                                                      uint64_t N, uint32_t K, float alpha, float beta,
                                                                      uint32_t tiles_n, uint32_t flags) {
    __shared__ __attribute__((aligned(16))) float lds[short_k::lds_floats<ROWS>()];
    // With kGemmLowerTilesOnly (square tiles only) the grid holds the lower-triangle tiles alone, numbered
    // row by row (a workgroup that only returns would still wait for a CU with this much LDS free).
    uint32_t tile_m, tile_n;
    if (ROWS == BM && (flags & trakhip::kGemmLowerTilesOnly)) {
        short_k::triangle_tile(blockIdx.x, tile_m, tile_n);
    } else {
        tile_m = blockIdx.x / tiles_n;
        tile_n = blockIdx.x % tiles_n;
    }
    short_k::tile<ROWS>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, tile_m, tile_n, lds);
}

// NT products of few tiles or few columns: C[M, N] = alpha * A[M, K] * B[N, K]^T + beta * C (row i *= row_scale[i]).
//
// WM x WN x WK = 4 waves; the tile has 32 WM x 32 WN entries, a stage 32 WK values of k, of which wave (.., wk) takes 32,
// and DEPTH stages are in flight in registers (the general kernel above goes to memory once per 16 values of k, and with a
// tile or less per CU nothing hides that).  WK > 1 shares one tile's k range out over the waves (their sums are
// added up in LDS at the end, in order), so a tile's chain of MFMAs is a quarter as long and a product of
// [2000 x 512] by [100 x 512] has 252 workgroups where 128 x 128 tiles give 16.  Every wave keeps two sums, of the
// even and the odd groups of eight k.  16-byte aligned rows, K a multiple of 32 WK DEPTH; rows past M or N are read from the last
// row and not stored.  Measured (general kernel; three-plane product, splits included; now; call to call):
// [2000 x 512][100 x 512]^T 55, 79, 14 us; [2000 x 512][512 x 512]^T 55, 72, 17 us; [8000 x 4096][40 x 4096]^T 348, 490, 54 us;
// [50 000 x 2048][100 x 2048]^T 305, 441, 253 us; [50 000 x 4096][20 x 4096]^T 574, 904, 184 us (4.5 TB/s of A).  Error against
// 64 bits 0.4 (32 x 32) and 0.8 (64 x 64) of the three-plane product's.
constexpr int kSmallPitchPad = 4;

template <int WM, int WN, int WK, int DEPTH>
__global__ __launch_bounds__(kThreads, 2) void gemm_nt_small_kernel(const float* __restrict__ A, uint64_t lda,
                                                                    const float* __restrict__ B, uint64_t ldb,
                                                                    float* __restrict__ C, uint64_t ldc, uint64_t M,
                                                                    uint64_t N, uint64_t K, float alpha, float beta,
                                                                    const float* __restrict__ row_scale, uint32_t tiles_n,
                                                                    uint32_t tiles) {
    static_assert(WM * WN * WK == 4 && DEPTH % 2 == 0, "four waves, two LDS buffers");
    constexpr int TM = 32 * WM, TN = 32 * WN, KS = 32 * WK;   // a stage: KS values of k
    constexpr int kPitch = KS + kSmallPitchPad;                // 16-byte reads of sixteen rows: conflict free
    constexpr int kPerRow = KS / 4;                            // 16-byte pieces of a row
    constexpr int kA = TM * kPerRow / kThreads, kB = TN * kPerRow / kThreads;
    constexpr int kFloats = (TM + TN) * kPitch;
    static_assert(2 * kFloats >= 4 * 16 * 64 || WK == 1, "the sums of four waves fit into the buffers");
    typedef float floatx4 __attribute__((ext_vector_type(4)));
    __shared__ __attribute__((aligned(16))) float lds[2][kFloats];

    // the column tiles of a row of tiles go to one XCD, one after another: its rows of A come from memory once
    const uint32_t xcd = blockIdx.x & 7u, lo = (uint32_t)((uint64_t)xcd * tiles / 8u), hi = (uint32_t)((xcd + 1ull) * tiles / 8u);
    const uint32_t tile = lo + (blockIdx.x >> 3);
    if (tile >= hi) return;
    const uint64_t m0 = (uint64_t)(tile / tiles_n) * TM, n0 = (uint64_t)(tile % tiles_n) * TN;

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wk = wave % WK, wn = wave / WK % WN, wm = wave / WK / WN;
    const int x = lane & 31, h = lane >> 5;

    // this thread's pieces: byte offsets from the tile's first row (pitches below 2^23 elements)
    const char* a_tile = reinterpret_cast<const char*>(A + m0 * lda);
    const char* b_tile = reinterpret_cast<const char*>(B + n0 * ldb);
    uint32_t at[kA], bt[kB];
#pragma unroll
    for (int i = 0; i < kA; ++i) {
        const uint32_t id = tid + kThreads * i, row = id / kPerRow;
        const uint64_t last = M - 1 - m0;
        at[i] = (uint32_t)((row < last ? row : last) * lda + 4 * (id % kPerRow)) * 4u;
    }
#pragma unroll
    for (int i = 0; i < kB; ++i) {
        const uint32_t id = tid + kThreads * i, row = id / kPerRow;
        const uint64_t last = N - 1 - n0;
        bt[i] = (uint32_t)((row < last ? row : last) * ldb + 4 * (id % kPerRow)) * 4u;
    }
    floatx4 ra[DEPTH][kA], rb[DEPTH][kB];
    auto load = [&](int u, uint64_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kA; ++i) ra[u][i] = *reinterpret_cast<const floatx4*>(a_tile + k0 * 4 + at[i]);
#pragma unroll
        for (int i = 0; i < kB; ++i) rb[u][i] = *reinterpret_cast<const floatx4*>(b_tile + k0 * 4 + bt[i]);
    };
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) load(u, KS * u);

    floatx16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.0f;
    for (uint64_t k0 = 0; k0 < K; k0 += KS * DEPTH) {
        const bool more = k0 + KS * DEPTH < K;
#pragma unroll
        for (int u = 0; u < DEPTH; ++u) {
            // a buffer is written again two stages later, behind the barrier that follows its reads
            float* buf = lds[u & 1];
#pragma unroll
            for (int i = 0; i < kA; ++i) {
                const int id = tid + kThreads * i;
                *reinterpret_cast<floatx4*>(buf + (id / kPerRow) * kPitch + 4 * (id % kPerRow)) = ra[u][i];
            }
#pragma unroll
            for (int i = 0; i < kB; ++i) {
                const int id = tid + kThreads * i;
                *reinterpret_cast<floatx4*>(buf + (TM + id / kPerRow) * kPitch + 4 * (id % kPerRow)) = rb[u][i];
            }
            if (more) load(u, k0 + KS * (DEPTH + u));
            __syncthreads();
            floatx4 fa[4], fb[4];
            const float* as = buf + (32 * wm + x) * kPitch + 32 * wk + 4 * h;
            const float* bs = buf + (TM + 32 * wn + x) * kPitch + 32 * wk + 4 * h;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                fa[q] = *reinterpret_cast<const floatx4*>(as + 8 * q);
                fb[q] = *reinterpret_cast<const floatx4*>(bs + 8 * q);
            }
            __builtin_amdgcn_sched_barrier(0);  // all reads of the stage in flight before its first MFMA waits
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[q & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[q][t], fb[q][t], acc[q & 1], 0, 0, 0);
        }
    }
    floatx16 sum = acc[0] + acc[1];
    // WK waves hold a share of the same entries: registers [first, first + kMine) of the sum are this wave's to store
    constexpr int kMine = 16 / WK;
    const int first = kMine * wk;
    float out[kMine];
    if constexpr (WK > 1) {
        float* shares = &lds[0][0];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) shares[(wave * 16 + r) * 64 + lane] = sum[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kMine; ++r) {
            out[r] = 0.0f;
#pragma unroll
            for (int w = 0; w < WK; ++w) out[r] += shares[((wave - wk + w) * 16 + first + r) * 64 + lane];
        }
    } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) out[r] = sum[r];
    }
    const uint64_t col = n0 + 32 * wn + x;
    if (col >= N) return;
    const uint64_t row0 = m0 + 32 * wm + 4 * h;
    float prev[kMine];
#pragma unroll
    for (int r = 0; r < kMine; ++r) {
        const uint64_t row = row0 + 8 * ((first + r) >> 2) + ((first + r) & 3);
        prev[r] = beta != 0.0f && row < M ? C[row * ldc + col] : 0.0f;
    }
#pragma unroll
    for (int r = 0; r < kMine; ++r) {
        const uint64_t row = row0 + 8 * ((first + r) >> 2) + ((first + r) & 3);
        if (row >= M) continue;
        float v = alpha * out[r];
        if (beta != 0.0f) v += beta * prev[r];
        C[row * ldc + col] = v * (row_scale ? row_scale[row] : 1.0f);
    }
}

// What an NT product takes, in microseconds: rounds of tiles over the 256 CUs times the time of one, which goes with K.  A tile
// of 32 x 32 entries shared by four waves takes 6.0 ns per value of k whether one or two of them share a CU (bound by what 256 CUs read from L2: 10.7 TB/s);
// a 64 x 64 tile 17.6 ns where two or more share a CU, 19.8 alone (120 TFLOP/s).  (The general kernel: 128 x 128 tiles 83 ns,
// 128 x 256 tiles, from 256 of them on, 134 ns.)
double tiles_of(uint64_t M, uint64_t N, uint64_t rows, uint64_t cols) {
    return (double)((M + rows - 1) / rows) * (double)((N + cols - 1) / cols);
}
double rounds_of(double tiles) { return tiles <= 256.0 ? 1.0 : tiles / 256.0; }
double one_tile_us(uint64_t M, uint64_t N, uint64_t K) {
    return 5.0 + 6.0e-3 * (double)K * rounds_of(tiles_of(M, N, 32, 32));
}
double four_tiles_us(uint64_t M, uint64_t N, uint64_t K) {
    const double tiles = tiles_of(M, N, 64, 64);
    const double rounds = tiles <= 256.0 ? 1.12 : tiles < 1e15 ? (double)(uint64_t)((tiles + 255.0) / 256.0) : tiles / 256.0;
    return 5.0 + 17.6e-3 * (double)K * rounds;
}
// Both operands split into planes (10 bytes of traffic per value) and their product (gemm_split.hip).
double split_us(uint64_t M, uint64_t N, uint64_t K) {
    return 18.0 + 2.0e-6 * ((double)M + (double)N) * (double)K + trakhip::split_product_us(M, N, K);
}
// Where the two are close these tell them apart: a round of tiles has its stores of C to make besides (0.3 and 0.8 us, which
// count where K is 256), and the planes of up to 15 million values are still in the 256 MB cache when the product reads them, 0.9
// us a million instead of 2.2.  They price the split with its product on 256 x 256 tiles only: its 128 x 128 ones are up to 20 %
// faster, but a product in place has the smaller error, and keeps what it does not do slower than that.  Call to call, 814
// products within a factor of 1.8 (M = 300 .. 50 000, N = 64 .. 3000, K = 256 .. 4096): none is more than 2.4 % above the split on 256 x 256
// tiles; by the estimates above alone 28 are, up to 30 % ([16 000 x 256] by 768 in place 68 us, split 52; [20 000 x 512] by 512 97, 84).
double close_in_place_us(uint64_t M, uint64_t N, uint64_t K) {
    const double k = (double)K, four = tiles_of(M, N, 64, 64);
    const double one_us = (0.3 + 6.0e-3 * k) * rounds_of(tiles_of(M, N, 32, 32));
    const double four_us = (0.8 + 17.0e-3 * k) * (four <= 256.0 ? 1.12 : __builtin_ceil(four / 256.0));
    return 5.0 + (one_us < four_us ? one_us : four_us);
}
double close_split_us(uint64_t M, uint64_t N, uint64_t K) {
    const double millions = 1e-6 * ((double)M + (double)N) * (double)K;
    const double passes = millions <= 15.0 ? 0.9 * millions : 0.9 * 15.0 + 2.2 * (millions - 15.0);
    return 15.0 + passes + trakhip::split_product_big_us(M, N, K);
}

template <int WM, int WN, int WK, int DEPTH>
int launch_small(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M, uint64_t N,
                 uint64_t K, float alpha, float beta, const float* row_scale, hipStream_t s) {
    const uint64_t tn = (N + 32 * WN - 1) / (32 * WN), tiles = (M + 32 * WM - 1) / (32 * WM) * tn;
    if (tiles > 0x7FFFFFF0ull) return TRAKHIP_ERR_SHAPE;
    hipLaunchKernelGGL((gemm_nt_small_kernel<WM, WN, WK, DEPTH>), dim3((uint32_t)((tiles + 7) / 8 * 8)), dim3(kThreads), 0, s,
                       A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, (uint32_t)tn, (uint32_t)tiles);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

template <bool AK, bool BK, int WN>
int launch_tiles(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
                 uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, bool aligned,
                 uint32_t flags, hipStream_t s) {
    constexpr int BN = 64 * WN;
    const uint64_t tm = (M + BM - 1) / BM, tn = (N + BN - 1) / BN;
    if (tm * tn > 0x7FFFFFFFull) return TRAKHIP_ERR_SHAPE;
    const dim3 grid((uint32_t)(tm * tn)), block(kThreads);
    if (aligned)
        hipLaunchKernelGGL((gemm_kernel<AK, BK, true, WN>), grid, block, 0, s, A, lda, B, ldb, C, ldc, M, N, K, alpha,
                           beta, row_scale, (uint32_t)tn, flags);
    else
        hipLaunchKernelGGL((gemm_kernel<AK, BK, false, WN>), grid, block, 0, s, A, lda, B, ldb, C, ldc, M, N, K,
                           alpha, beta, row_scale, (uint32_t)tn, flags);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

template <bool AK, bool BK>
int launch(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
           uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, uint32_t flags, hipStream_t s) {
    if (M == 0 || N == 0) return TRAKHIP_OK;
    if (!A || !B || !C) return TRAKHIP_ERR_NULL;
    const uint64_t min_lda = AK ? M : K, min_ldb = BK ? N : K;
    if (lda < min_lda || ldb < min_ldb || ldc < N) return TRAKHIP_ERR_SHAPE;
    const bool aligned = (reinterpret_cast<uintptr_t>(A) % 16 == 0) && (reinterpret_cast<uintptr_t>(B) % 16 == 0) &&
                         (lda % 4 == 0) && (ldb % 4 == 0);
    // the wide tile pays off once C has a few hundred 128 x 256 tiles; narrow C keeps 128 x 128
    const bool wide = N >= 256 && ((M + BM - 1) / BM) * ((N + 255) / 256) >= 256;
    if (wide)
        return launch_tiles<AK, BK, 4>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, aligned, flags, s);
    return launch_tiles<AK, BK, 2>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, aligned, flags, s);
}

}  // namespace

namespace trakhip {

int gemm_nt(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
            uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, hipStream_t s, uint32_t flags) {
    const bool aligned = A && B && (reinterpret_cast<uintptr_t>(A) % 16 == 0) &&
                         (reinterpret_cast<uintptr_t>(B) % 16 == 0) && (lda % 4 == 0) && (ldb % 4 == 0);
    if (M && N && C && aligned && !row_scale && K >= 8 && K <= short_k::kMaxK && K % 8 == 0 && lda >= K && ldb >= K &&
        ldc >= N) {
        const uint64_t tm = (M + BM - 1) / BM, tn = (N + BM - 1) / BM;
        // Lower tiles only: a square tile grid is launched as its triangle; otherwise the flag is dropped
        // (computing the upper tiles too is allowed, skipping them is an optimisation).
        const bool triangle = (flags & kGemmLowerTilesOnly) && tm == tn;
        const uint64_t working = triangle ? tm * (tm + 1) / 2 : tm * tn;
        const bool whole = triangle || !(flags & kGemmLowerTilesOnly);
        // too few 128-row tiles to occupy the CUs: 32-row tiles, four times as many workgroups
        if (whole && !triangle && working <= 64) {
            const uint64_t tm32 = (M + 31) / 32;
            hipLaunchKernelGGL(gemm_nt_short_k_kernel<32>, dim3((uint32_t)(tm32 * tn)), dim3(kThreads), 0, s, A, lda, B,
                               ldb, C, ldc, M, N, (uint32_t)K, alpha, beta, (uint32_t)tn, 0u);
            return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
        }
        // one workgroup per CU (its LDS) and no overlap inside it: worth it for up to two rounds
        if (whole && working <= 512) {
            hipLaunchKernelGGL(gemm_nt_short_k_kernel<BM>, dim3((uint32_t)working), dim3(kThreads), 0, s, A, lda, B, ldb,
                               C, ldc, M, N, (uint32_t)K, alpha, beta, (uint32_t)tn,
                               triangle ? kGemmLowerTilesOnly : 0u);
            return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
        }
    }
    return launch<false, false>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, flags, s);
}

bool gemm_nt_in_place_pays(uint64_t M, uint64_t N, uint64_t K) {
    if (M == 0 || N == 0 || K == 0 || K % 256) return false;
    const double one = one_tile_us(M, N, K), four = four_tiles_us(M, N, K);
    return (one < four ? one : four) < split_us(M, N, K) && close_in_place_us(M, N, K) < close_split_us(M, N, K);
}

int gemm_nt_in_place_tile(uint64_t M, uint64_t N, uint64_t K) {
    if (M == 0 || N == 0 || K == 0 || K % 256) return 0;
    return one_tile_us(M, N, K) < four_tiles_us(M, N, K) ? 32 : 64;
}

int gemm_nt_in_place(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
                     uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, hipStream_t s) {
    if (M == 0 || N == 0) return TRAKHIP_OK;
    // (a lane's byte offset inside the rows of a tile is kept in 32 bits)
    if (K == 0 || K % 256 || lda < K || ldb < K || ldc < N || lda >= (1ull << 23) || ldb >= (1ull << 23)) return TRAKHIP_ERR_SHAPE;
    if (!A || !B || !C) return TRAKHIP_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(A) % 16) || (reinterpret_cast<uintptr_t>(B) % 16) || (lda % 4) || (ldb % 4) ||
        (reinterpret_cast<uintptr_t>(C) % 4) || (reinterpret_cast<uintptr_t>(row_scale) % 4))
        return TRAKHIP_ERR_ALIGN;
    if (gemm_nt_in_place_tile(M, N, K) == 32)
        return launch_small<1, 1, 4, 2>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, s);
    return launch_small<2, 2, 1, 4>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, row_scale, s);
}

int gemm_tn(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
            uint64_t N, uint64_t K, float alpha, float beta, hipStream_t s, uint32_t flags) {
    return launch<true, true>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, nullptr, flags, s);
}

int gemm_nn(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
            uint64_t N, uint64_t K, float alpha, float beta, hipStream_t s, uint32_t flags) {
    return launch<false, true>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, nullptr, flags, s);
}

int gemm_nn_batched(const float* A, uint64_t lda, const float* B, uint64_t ldb, float* C, uint64_t ldc, uint64_t M,
                    uint64_t N, uint64_t K, float alpha, float beta, const GemmBatch& batch, hipStream_t s) {
    if (M == 0 || N == 0 || batch.count == 0) return TRAKHIP_OK;
    if (!A || !B || !C) return TRAKHIP_ERR_NULL;
    if (batch.count > kGemmBatchMax || lda < K || ldb < N || ldc < N) return TRAKHIP_ERR_SHAPE;
    // the batched kernel uses 16-byte loads: every operand start and pitch must allow them
    if ((reinterpret_cast<uintptr_t>(A) % 16) || (reinterpret_cast<uintptr_t>(B) % 16) || (lda % 4) || (ldb % 4))
        return TRAKHIP_ERR_ALIGN;
    for (uint32_t y = 0; y < batch.count; ++y) {
        if ((batch.a[y] % 4) || (batch.b[y] % 4)) return TRAKHIP_ERR_ALIGN;
        if (batch.m[y] > M) return TRAKHIP_ERR_SHAPE;
    }
    const uint64_t tm = (M + BM - 1) / BM, tn = (N + 127) / 128;
    if (tm * tn > 0x7FFFFFFFull) return TRAKHIP_ERR_SHAPE;
    hipLaunchKernelGGL(gemm_nn_batched_kernel, dim3((uint32_t)(tm * tn), batch.count), dim3(kThreads), 0, s, A, lda, B,
                       ldb, C, ldc, M, N, K, alpha, beta, (uint32_t)tn, batch);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

}  // namespace trakhip
