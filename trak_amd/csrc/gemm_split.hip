// fp32-accurate GEMM on the 16-bit matrix cores: C[M, N] = alpha * A * B^T + beta * C (row i *= row_scale[i]).
//
// The scoring GEMMs of BasicScoreComputer (trak/score_computers.py:153, :176, trak/utils.py:131)
// multiply fp32 matrices (or fp16 ones when TRAKer runs with use_half_precision, its default).
// v_mfma_f32_32x32x2_f32 runs at 157 TFLOP/s; v_mfma_f32_32x32x16_{bf16,f16} at 2.5 PFLOP/s,
// sixteen times the rate, with exact products and fp32 accumulation.
//
// fp32 operands: every fp32 value is the exact sum of three bf16 values (24 significand bits =
// 3 x 8), x = x1 + x2 + x3 with |x2| <= 2^-8 |x1|, |x3| <= 2^-16 |x1|, so
//     a * b = a1 b1 + (a1 b2 + a2 b1) + (a1 b3 + a2 b2 + a3 b1) + O(2^-24 |a b|)
// and six bf16 MFMAs give the product sum with the error of an fp32 dot product at 6/16 of the
// cost of the fp32 instruction.  The three terms left out are each below 2^-24 |a b|, the rounding
// a single fp32 multiplication makes.
// fp16 or bf16 operands (both of the same type): one plane, one MFMA, nothing left out.
// An opt-in cheaper variant for fp32 operands ("two fp16 planes"): every row is scaled by a power of two
// that brings its largest magnitude to [2^14, 2^15), then x = h1 + h2 with fp16 terms (22 significand
// bits for entries within 2^-18 of the row's largest, fewer below), and
//     a * b = a1 b1 + (a1 b2 + a2 b1) + O(2^-22 |a b|)
// with three fp16 MFMAs; the powers of two are taken out again in the epilogue.  Half the MFMAs of the
// three-plane product at four times its operand error bound.
//
// Operands are brought once, outside the GEMM, into "planes": plane p, k-octet o (8 consecutive k),
// row r is one 16-byte piece at ((p * K8 + o) * Rp + r) * 16 bytes, rows padded with zeros to a
// multiple of 256 and octets to a multiple of 8.  A 16-byte piece is exactly what one lane feeds to
// the MFMA (8 consecutive k of one row), consecutive rows are consecutive pieces, so global loads,
// LDS writes and LDS reads are all linear and conflict free, and the GEMM kernel moves 16-bit data
// only.
//
// Workgroup = 512 threads = 8 waves (4 x 2), 256 x 256 tile of C, a wave owns 64 x 128 of C (128
// accumulator VGPRs).  A step covers 16 S values of k (S = 1 for three planes, 4 for one plane):
// two LDS buffers of 48 or 64 KB filled by LDS-direct loads, one barrier per step, 48 or 32 MFMAs
// per wave and step.  Measured against this for three planes: 128 x 256 tiles with two workgroups
// per CU (9 % slower), 64 x 64 wave tiles at four waves per SIMD, three LDS buffers, register-staged
// loads, super-tile orders per XCD (all slower or equal).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "short_k_tile.h"
#include "store_cast.h"
#include "trakhip_internal.h"

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t piece __attribute__((ext_vector_type(4)));  // 16 bytes = 8 x 16 bit = one lane's MFMA operand

// Shapes of a workgroup's tile.  BigTile: 4 x 2 waves, each owns 64 x 128 of C.  SmallTile: 2 x 2 waves of 64 x 64, for products
// that leave CUs idle with the big one and for the rows of a product that are left behind whole rounds of tiles over the CUs;
// the same MFMAs in the same order, two (16-bit operands in place) or three (three planes) workgroups per CU.
struct BigTile {
    static constexpr int kWavesM = 4, kWavesN = 2, JT = 4, BM = 64 * kWavesM, BN = 32 * JT * kWavesN, kWaves = kWavesM * kWavesN;
    static constexpr int kPerSimd = 2;
};
struct SmallTile {
    static constexpr int kWavesM = 2, kWavesN = 2, JT = 2, BM = 64 * kWavesM, BN = 32 * JT * kWavesN, kWaves = kWavesM * kWavesN;
    static constexpr int kPerSimd = 3;
};
constexpr int kWavesM = BigTile::kWavesM, kWavesN = BigTile::kWavesN;
constexpr int BM = BigTile::BM, BN = BigTile::BN;
constexpr int kWaves = BigTile::kWaves;
constexpr uint32_t kGemmBandedGrid = 4u;            // kernel flag: the grid is numbered as banded_tile says
constexpr uint32_t kGemmTriangleGrid = 2u;          // kernel flag: the grid lists the lower-triangle tiles only
constexpr int kRowPad = 256;                       // rows of an operand are padded to this
constexpr int kOctetPad = 8;                       // octets (64 values of k) are padded to this

// ---- bringing operands into planes ---------------------------------------------------------

// binary32 -> nearest bf16 (ties to even) as a binary32 value; finite inputs
__device__ __forceinline__ float bf16_round(float x) {
    const uint32_t b = __float_as_uint(x);
    return __uint_as_float((b + 0x7FFFu + ((b >> 16) & 1u)) & 0xFFFF0000u);
}

// x = t[0] + t[1] + t[2] exactly (up to underflow of the last term), bf16 bit patterns
__device__ __forceinline__ void split3(float x, uint32_t (&t)[3]) {
    const float x1 = bf16_round(x);
    const float r1 = x - x1;
    const float x2 = bf16_round(r1);
    const float r2 = r1 - x2;
    t[0] = __float_as_uint(x1) >> 16;
    t[1] = __float_as_uint(x2) >> 16;
    t[2] = __float_as_uint(bf16_round(r2)) >> 16;
}

// One thread per (row r, octet o): reads 8 consecutive k of the row, writes its pieces.
// TRANS = false: src[r * ld + k];  TRANS = true: src[k * ld + r].  Rows >= rows and k >= K give
// zeros (the padding is rewritten on every call).  Threads of a workgroup cover 64 rows x 4 octets.
template <bool TRANS>
__global__ __launch_bounds__(256) void split_kernel(const float* __restrict__ src, uint64_t ld, uint64_t rows,
                                                    uint64_t K, uint64_t Rp, uint64_t K8, uint32_t row_blocks,
                                                    uint4* __restrict__ planes) {
    const uint64_t r = (uint64_t)(blockIdx.x % row_blocks) * 64 + (threadIdx.x & 63);
    const uint64_t o = (uint64_t)(blockIdx.x / row_blocks) * 4 + (threadIdx.x >> 6);
    if (r >= Rp || o >= K8) return;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint64_t k = 8 * o + i;
        v[i] = (r < rows && k < K) ? (TRANS ? src[k * ld + r] : src[r * ld + k]) : 0.0f;
    }
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t lo[3], hi[3];
        split3(v[2 * i], lo);
        split3(v[2 * i + 1], hi);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p][i] = lo[p] | (hi[p] << 16);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p) planes[((uint64_t)p * K8 + o) * Rp + r] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

// The same for a row-major source with 16-byte aligned rows: a workgroup takes 64 rows x 8 octets, reads whole 256-byte
// stretches of the rows and hands them to the (row, octet) threads through LDS.  (With every lane reading its own row, 32 bytes
// of a 128-byte line at a time, [50 000, 4096] took 527 us, now 459, 4.5 TB/s read and written; [49 999, 2560] 269 and 242, [4096, 4096] 30 and
// 27.  A copy reaches 5.3 TB/s at these sizes.)
constexpr int kSplitPitch = 64 + 4;  // floats; sixteen rows' 16-byte reads hit all banks
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ src, uint64_t ld, uint64_t rows,
                                                         uint64_t K, uint64_t Rp, uint64_t K8, uint32_t row_blocks,
                                                         uint4* __restrict__ planes) {
    __shared__ __attribute__((aligned(16))) float t[64 * kSplitPitch];
    const uint64_t r0 = (uint64_t)(blockIdx.x % row_blocks) * 64, o0 = (uint64_t)(blockIdx.x / row_blocks) * kOctetPad;
    const int tid = threadIdx.x, c = 4 * (tid & 15);
    const uint64_t k = 8 * o0 + c;
    float4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint64_t r = r0 + (tid >> 4) + 16 * i;
        v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (r < rows && k < K) {
            const float* q = src + r * ld + k;
            if (k + 4 <= K) {
                v[i] = *reinterpret_cast<const float4*>(q);
            } else {
                v[i].x = q[0];
                if (k + 1 < K) v[i].y = q[1];
                if (k + 2 < K) v[i].z = q[2];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<float4*>(t + ((tid >> 4) + 16 * i) * kSplitPitch + c) = v[i];
    __syncthreads();
    const int r = tid & 63;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int o = (tid >> 6) + 4 * j;
        const float4 lo = *reinterpret_cast<const float4*>(t + r * kSplitPitch + 8 * o);
        const float4 hi = *reinterpret_cast<const float4*>(t + r * kSplitPitch + 8 * o + 4);
        const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        uint32_t w[3][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t a[3], b[3];
            split3(x[2 * i], a);
            split3(x[2 * i + 1], b);
#pragma unroll
            for (int p = 0; p < 3; ++p) w[p][i] = a[p] | (b[p] << 16);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
            planes[((uint64_t)p * K8 + o0 + o) * Rp + r0 + r] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
    }
}

// The same for a 16-bit source (fp16 or bf16 bit patterns): one plane, the values themselves.
template <bool TRANS, bool ALIGNED>
__global__ __launch_bounds__(256) void relayout16_kernel(const uint16_t* __restrict__ src, uint64_t ld, uint64_t rows,
                                                         uint64_t K, uint64_t Rp, uint64_t K8, uint32_t row_blocks,
                                                         uint4* __restrict__ planes) {
    const uint64_t r = (uint64_t)(blockIdx.x % row_blocks) * 64 + (threadIdx.x & 63);
    const uint64_t o = (uint64_t)(blockIdx.x / row_blocks) * 4 + (threadIdx.x >> 6);
    if (r >= Rp || o >= K8) return;
    uint4 w;
    if (!TRANS && ALIGNED && r < rows && 8 * o + 8 <= K) {
        w = *reinterpret_cast<const uint4*>(src + r * ld + 8 * o);
    } else {
        uint32_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t k = 8 * o + i;
            v[i] = (r < rows && k < K) ? (uint32_t)(TRANS ? src[k * ld + r] : src[r * ld + k]) : 0u;
        }
        w = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
    }
    planes[o * Rp + r] = w;
}

// ---- two fp16 planes with a power-of-two scale per row ------------------------------------------

// Largest magnitude of every operand row as binary32 bits (non-negative floats order like unsigned
// integers).  Row-major operand: one wave per row.
__global__ __launch_bounds__(256) void absmax_rows_kernel(const float* __restrict__ src, uint64_t ld, uint64_t rows,
                                                          uint64_t K, uint32_t* __restrict__ maxbits) {
    const uint64_t r = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= rows) return;
    const int lane = threadIdx.x & 63;
    uint32_t m = 0;
    for (uint64_t k = lane; k < K; k += 64) {
        const uint32_t b = __float_as_uint(src[r * ld + k]) & 0x7FFFFFFFu;
        m = b > m ? b : m;
    }
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)m, w);
        m = o > m ? o : m;
    }
    if (lane == 0) maxbits[r] = m;
}

// Transposed operand (row r of the operand is column r of src[K, rows]): a thread walks one column over
// one chunk of k and merges with an atomic maximum (order independent); maxbits starts at zero.
constexpr int kColChunks = 64;
__global__ __launch_bounds__(256) void absmax_cols_kernel(const float* __restrict__ src, uint64_t ld, uint64_t rows,
                                                          uint64_t K, uint32_t* __restrict__ maxbits) {
    const uint64_t r = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (r >= rows) return;
    const uint64_t per = (K + kColChunks - 1) / kColChunks;
    const uint64_t k0 = (uint64_t)blockIdx.y * per, k1 = k0 + per < K ? k0 + per : K;
    uint32_t m = 0;
    for (uint64_t k = k0; k < k1; ++k) {
        const uint32_t b = __float_as_uint(src[k * ld + r]) & 0x7FFFFFFFu;
        m = b > m ? b : m;
    }
    if (m) atomicMax(maxbits + r, m);
}

__global__ __launch_bounds__(256) void zero_u32_kernel(uint32_t* __restrict__ p, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// Power of two that brings a row whose largest magnitude has these bits into [2^14, 2^15) (fp16 tops
// out at 65504), and its inverse.  A row of zeros, or one that holds an infinity or a NaN, is left alone.
__device__ __forceinline__ void row_factors(uint32_t maxbits, float& scale, float& unscale) {
    int sh = 0;
    if (maxbits != 0u && maxbits < 0x7F800000u) {
        sh = 14 - ((int)(maxbits >> 23) - 127);
        sh = sh > 126 ? 126 : sh;
    }
    scale = __uint_as_float((uint32_t)(127 + sh) << 23);
    unscale = __uint_as_float((uint32_t)(127 - sh) << 23);
}

// One thread per (row r, octet o), as split_kernel: x * scale = h1 + h2 with fp16 terms, planes 0 and 1.
template <bool TRANS, bool ALIGNED>
__global__ __launch_bounds__(256) void split2_kernel(const float* __restrict__ src, uint64_t ld, uint64_t rows,
                                                     uint64_t K, uint64_t Rp, uint64_t K8, uint32_t row_blocks,
                                                     const uint32_t* __restrict__ maxbits, uint4* __restrict__ planes,
                                                     float* __restrict__ unscale_out) {
    const uint64_t r = (uint64_t)(blockIdx.x % row_blocks) * 64 + (threadIdx.x & 63);
    const uint64_t o = (uint64_t)(blockIdx.x / row_blocks) * 4 + (threadIdx.x >> 6);
    if (r >= Rp || o >= K8) return;
    float scale = 1.0f, unscale = 1.0f;
    if (r < rows) row_factors(maxbits[r], scale, unscale);
    if (o == 0 && r < rows) unscale_out[r] = unscale;
    float v[8];
    if (!TRANS && ALIGNED && r < rows && 8 * o + 8 <= K) {
        const float4* q = reinterpret_cast<const float4*>(src + r * ld + 8 * o);
        const float4 lo = q[0], hi = q[1];
        v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w;
        v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t k = 8 * o + i;
            v[i] = (r < rows && k < K) ? (TRANS ? src[k * ld + r] : src[r * ld + k]) : 0.0f;
        }
    }
    uint32_t w[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t t[2][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float x = v[2 * i + e] * scale;  // exact: a power of two, no overflow by construction
            const _Float16 h1 = (_Float16)x;       // round to nearest even
            const _Float16 h2 = (_Float16)(x - (float)h1);
            t[0][e] = (uint32_t)__builtin_bit_cast(uint16_t, h1);
            t[1][e] = (uint32_t)__builtin_bit_cast(uint16_t, h2);
        }
        w[0][i] = t[0][0] | (t[0][1] << 16);
        w[1][i] = t[1][0] | (t[1][1] << 16);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) planes[((uint64_t)p * K8 + o) * Rp + r] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

// ---- GEMM ----------------------------------------------------------------------------------

template <bool F16>
__device__ __forceinline__ floatx16 mfma16(const piece& a, const piece& b, floatx16 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c,
                                                      0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                       c, 0, 0, 0);
}

typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// 4 x 4 transpose inside every quad of lanes: lane q of a quad holds M[a][q] in v[a] and ends up with
// M[q][c] in v[c].  Two exchanges, over lane distance 2 and 1: (register r, lane q) trades places with
// (register r ^ d, lane q ^ d) where bit d of r and q differ.
__device__ __forceinline__ void quad_transpose(float (&v)[4], int lane) {
    const bool b1 = lane & 2, b0 = lane & 1;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float send = b1 ? v[r] : v[r + 2];
        const float recv = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, send), 0x4E, 0xF, 0xF, true));  // quad_perm [2,3,0,1]
        if (b1) v[r] = recv; else v[r + 2] = recv;
    }
#pragma unroll
    for (int r = 0; r < 4; r += 2) {
        const float send = b0 ? v[r] : v[r + 1];
        const float recv = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, send), 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
        if (b0) v[r] = recv; else v[r + 1] = recv;
    }
}

// Epilogue of a wave's 64 x (32 JT) part of C.  D[m][n] of a 32x32 MFMA: lane holds column
// n = lane % 32; register r holds row 8*(r/4) + 4*(lane/32) + r%4.  When C is accumulated into (ACCUM),
// its old values are fetched for 32 rows at a time before any of them is overwritten (loads and stores
// through one pointer would otherwise alternate, one memory round trip per element).
// SCALED: the accumulators are products of operands whose rows were multiplied by powers of two;
// a_unscale[row] and b_unscale[col] are the inverse factors (applied one after the other, so that no
// intermediate leaves the binary32 range when the result does not).
//
// A wave whose part of C lies wholly inside the matrix (all but the last row and column of tiles) takes
// the path without bounds tests and with 16-byte stores: a store instruction costs the texture path about
// 32 cycles whatever it carries, and with one 4-byte store per accumulator register (1024 per tile and
// CU) the epilogue of a tile took 33 000 cycles, a seventh of a product with 4096 values of k.  Four
// registers of a lane are four rows of one column; a 4 x 4 transpose inside every quad of lanes (DPP
// quad_perm, 16 vector instructions) turns them into four columns of one row, i.e. one 16-byte store,
// and a store instruction then writes eight whole 128-byte lines.
template <bool ACCUM, int JT, bool SCALED = false>
__device__ __forceinline__ void store_c(const floatx16 (&acc)[2][JT], float* __restrict__ C, uint64_t ldc, uint64_t M,
                                        uint64_t N, uint64_t row_base, uint64_t col0, int h, float alpha, float beta,
                                        const float* __restrict__ row_scale,
                                        const float* __restrict__ a_unscale = nullptr,
                                        const float* __restrict__ b_unscale = nullptr) {
    // wave-uniform: col0 = first column of the wave's part + lane % 32
    const bool inside = row_base + 64 <= M && col0 - (threadIdx.x & 31) + 32 * JT <= N;
    if (!SCALED && inside) {
        const int lane = threadIdx.x & 63, q = lane & 3;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                // registers 4g .. 4g+3 are rows 8g + 4h + (0..3) of the lane's column; after the transpose inside
                // the quad the lane holds row 8g + 4h + q, columns 4 (x / 4) .. + 3 of every 32-column group
                const uint64_t row = row_base + 32 * i + 8 * g + 4 * h + q;
                const float rs = row_scale ? row_scale[row] : 1.0f;
                float* p = C + row * ldc + (col0 - q);
                float4u prev[ACCUM ? JT : 1];
                if constexpr (ACCUM) {
#pragma unroll
                    for (int j = 0; j < JT; ++j) prev[j] = *reinterpret_cast<const float4u*>(p + 32 * j);
                }
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                    quad_transpose(v, lane);
                    float4u o;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        if constexpr (ACCUM)
                            o[c] = (alpha * v[c] + beta * prev[j][c]) * rs;
                        else
                            o[c] = alpha * v[c] * rs;
                    }
                    // streaming store: C is written once and is far larger than L2, where the operand panels
                    // that other workgroups are about to read should stay
                    __builtin_nontemporal_store(o, reinterpret_cast<float4u*>(p + 32 * j));
                }
            }
        }
        return;
    }
    float ub[JT];
#pragma unroll
    for (int j = 0; j < JT; ++j) ub[j] = (SCALED && col0 + 32 * j < N) ? b_unscale[col0 + 32 * j] : 1.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint64_t row0 = row_base + 32 * i + 4 * h;
        float ua[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint64_t row = row0 + 8 * (r >> 2) + (r & 3);
            ua[r] = (SCALED && row < M) ? a_unscale[row] : 1.0f;
        }
        // old values of C: fetched for a group of columns before any of them is overwritten (all four
        // 32-column groups at once, two at a time when the unscale factors take registers as well)
        constexpr int JG = (ACCUM && SCALED) ? (JT + 1) / 2 : JT;
#pragma unroll
        for (int j0 = 0; j0 < JT; j0 += JG) {
            floatx16 prev[ACCUM ? JG : 1];
            if constexpr (ACCUM) {
#pragma unroll
                for (int j = 0; j < JG; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const uint64_t row = row0 + 8 * (r >> 2) + (r & 3), col = col0 + 32 * (j0 + j);
                        prev[j][r] = (j0 + j < JT && row < M && col < N) ? C[row * ldc + col] : 0.0f;
                    }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint64_t row = row0 + 8 * (r >> 2) + (r & 3);
                if (row >= M) continue;
                const float rs = row_scale ? row_scale[row] : 1.0f;
#pragma unroll
                for (int j = 0; j < JG; ++j) {
                    const uint64_t col = col0 + 32 * (j0 + j);
                    if (j0 + j >= JT || col >= N) continue;
                    float v = acc[i][j0 + j][r];
                    if constexpr (SCALED) v = (v * ua[r]) * ub[j0 + j];
                    if constexpr (ACCUM)
                        C[row * ldc + col] = (alpha * v + beta * prev[j][r]) * rs;
                    else
                        C[row * ldc + col] = alpha * v * rs;
                }
            }
        }
    }
}

// The same for a 16-bit C (OUT: its element type; beta = 0): rounded from the accumulators instead of by a pass over an
// fp32 result (94 us for [50 000, 2048]).  vec: C 8-byte aligned, ldc a multiple of 4.
template <int OUT, int JT>
__device__ __forceinline__ void store_c16(const floatx16 (&acc)[2][JT], uint16_t* __restrict__ C, uint64_t ldc, uint64_t M,
                                          uint64_t N, uint64_t row_base, uint64_t col0, int h, float alpha,
                                          const float* __restrict__ row_scale, bool vec) {
    const int lane = threadIdx.x & 63, q = lane & 3;
    if (vec && row_base + 64 <= M && col0 - (lane & 31) + 32 * JT <= N) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int g = 0; g < 4; ++g) {  // as in store_c: four columns of one row per lane
                const uint64_t row = row_base + 32 * i + 8 * g + 4 * h + q;
                const float rs = row_scale ? row_scale[row] : 1.0f;
                uint16_t* p = C + row * ldc + (col0 - q);
#pragma unroll
                for (int j = 0; j < JT; ++j) {
                    float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                    quad_transpose(v, lane);
                    trakhip::store4<OUT>(p + 32 * j, make_float4(alpha * v[0] * rs, alpha * v[1] * rs, alpha * v[2] * rs,
                                                                 alpha * v[3] * rs));
                }
            }
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint64_t row = row_base + 32 * i + 8 * (r >> 2) + 4 * h + (r & 3);
            if (row >= M) continue;
            const float rs = row_scale ? row_scale[row] : 1.0f;
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                const float v = alpha * acc[i][j][r] * rs;
                if (col0 + 32 * j < N)
                    C[row * ldc + col0 + 32 * j] = OUT == TRAKHIP_F16 ? trakhip::cast_f16_bits(v) : trakhip::cast_bf16_bits(v);
            }
        }
}

// A step of a tile is S sub-steps (two octets = one MFMA depth each); sub-step u holds
// [A: plane][half][256 rows] followed by [B: plane][half][256 rows].  The pieces are moved in chunks
// of 64 consecutive ones by the load unit straight into LDS (global_load_lds_dwordx4): the 64
// lanes of a wave fetch 64 consecutive rows of one (plane, octet), which land at 64 consecutive
// 16-byte slots starting at a wave-uniform LDS address; no staging registers, no LDS store
// instructions.  Wave w moves chunks w, w + 8, ...
//
// A chunk's 64 pieces are consecutive in memory as well (64 rows of one plane and octet), so its address
// is a wave-uniform base plus 16 bytes per lane, and the base moves by a fixed number of bytes from step
// to step: the bases live in scalar registers and a load costs two scalar additions.  (Computing the
// piece address per lane from plane, octet and row took about thirty instructions per load, in front of
// the MFMAs of every step.)
template <int P, int S, class Shape>
struct StepMover {
    static constexpr int BM = Shape::BM, BN = Shape::BN, kWaves = Shape::kWaves;
    static constexpr int kAChunks = P * 2 * BM / 64, kBChunks = P * 2 * BN / 64;
    static constexpr int kSubChunks = kAChunks + kBChunks, kChunks = S * kSubChunks;
    // the first kLoaders waves move the chunks: wave w chunks w, w + kLoaders, ...  (all eight: leaving the loads
    // to four waves, so that the other four start their MFMAs at once, measured 1 % faster on the three-plane
    // product and is not worth a second code path)
    static constexpr int kLoaders = kWaves;
    static_assert(kChunks % kLoaders == 0, "every loading wave moves the same number of chunks");
    static_assert(BM % 64 == 0 && BN % 64 == 0, "a chunk lies in one (plane, half)");
    static constexpr int kPerWave = kChunks / kLoaders;
    const char* base[kPerWave];  // of this wave's chunks at the next step to load (wave-uniform)
    uint64_t step_a, step_b;     // bytes from one step to the next

    __device__ __forceinline__ void init(const piece* A, uint64_t Rpa, const piece* B, uint64_t Rpb, uint64_t K8,
                                         uint64_t m0, uint64_t n0, uint64_t s, int wave) {
        step_a = 2 * S * Rpa * sizeof(piece);
        step_b = 2 * S * Rpb * sizeof(piece);
#pragma unroll
        for (int i = 0; i < kPerWave; ++i) {
            const int c = wave % kLoaders + kLoaders * i;  // wave-uniform
            const int u = c / kSubChunks, cc = c % kSubChunks;
            if (cc < kAChunks) {
                const int e = 64 * cc, row = e % BM, ph = e / BM;  // ph = plane * 2 + half
                base[i] = reinterpret_cast<const char*>(A + ((uint64_t)(ph >> 1) * K8 + 2 * (s * S + u) + (ph & 1)) * Rpa + m0 + row);
            } else {
                const int e = 64 * (cc - kAChunks), row = e % BN, ph = e / BN;
                base[i] = reinterpret_cast<const char*>(B + ((uint64_t)(ph >> 1) * K8 + 2 * (s * S + u) + (ph & 1)) * Rpb + n0 + row);
            }
        }
    }
    // chunk i of the wave for the step the bases point at; then the base moves on to the step after
    __device__ __forceinline__ void move(int i, int wave, uint32_t lane_bytes, piece* lds) {
        const int c = wave % kLoaders + kLoaders * i;
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(base[i] + lane_bytes),
                                         (void __attribute__((address_space(3)))*)(lds + 64 * c), 16, 0, 0);
        // kAChunks is a multiple of kLoaders: which operand chunk i belongs to does not depend on the wave
        base[i] += ((kLoaders * i) % kSubChunks) < kAChunks ? step_a : step_b;
    }
    static_assert(kAChunks % kLoaders == 0 && kSubChunks % kLoaders == 0, "operand of a chunk: the same for all waves");
    __device__ __forceinline__ void move_all(int wave, uint32_t lane_bytes, piece* lds) {
        if (wave >= kLoaders) return;
#pragma unroll
        for (int i = 0; i < kPerWave; ++i) move(i, wave, lane_bytes, lds);
    }
};

// Workgroup -> unit of a symmetric product (share of the k range, tile): the shares' lists of tiles one after another, of
// which each of the eight XCDs, which are handed the workgroups round-robin, takes a contiguous eighth.  The tiles of a
// share read the same rows of X at about the same time, so an XCD then fetches its share's rows once; with the tiles
// dealt out over all XCDs each of them fetched every row of X ([50 000, 2048] fp16: 1.6 GB; 285 us, 249 this way; the
// three-plane product of [4100, 2048] fp32 138 -> 126, of [50 000, 4096] 4.41 -> 4.33 ms).  The grid has a multiple of
// eight workgroups; false: one without a unit.
__device__ __forceinline__ bool xcd_unit(uint32_t units, uint32_t& unit) {
    const uint32_t xcd = blockIdx.x & 7u;
    unit = (uint32_t)((uint64_t)xcd * units / 8u) + (blockIdx.x >> 3);
    return unit < (uint32_t)((xcd + 1ull) * units / 8u);
}

// The same for the grid of tiles of a product: number `position` of an order in which neighbours share operands.  Up to eight
// columns are walked row by row, more of them in bands of at most eight, and each XCD takes a contiguous eighth of the walk,
// so that the 32 tiles of 256 x 256 that an XCD works on at a time are some four rows of eight columns.
// (Row by row over all XCDs, eight columns give each XCD one column of 32 rows: 33 operand panels where 12 would do.)
// [50 000, 2048] by 2048 columns fp16 441 -> 432 us, 1536 257 -> 245; fp32 2048 1.93 -> 1.89 ms, 2560 2.83 -> 2.71.  With
// 16 columns of 256 the same time, from 24 on 2-9 % slower: row by row, an XCD then has five or more columns of six or fewer rows.
constexpr uint32_t kBandedTiles = 12;
__device__ __forceinline__ void banded_tile(uint32_t position, uint32_t tiles_m, uint32_t tiles_n, uint32_t& tile_m,
                                            uint32_t& tile_n) {
    uint32_t first = 0, width = tiles_n;
    if (tiles_n > 8) {  // the first `wider` bands have a column more than the others
        const uint32_t bands = (tiles_n + 7) / 8, wider = tiles_n % bands;
        uint32_t band;
        width = tiles_n / bands;
        if (position < wider * (width + 1) * tiles_m) {
            ++width;
            band = position / (width * tiles_m);
            first = band * width;
        } else {
            band = (position - wider * tiles_m) / (width * tiles_m);
            first = band * width + wider;
        }
        position -= first * tiles_m;
    }
    tile_m = position / width;
    tile_n = first + position % width;
}
bool banded(uint64_t tiles_n) { return tiles_n > 1 && tiles_n <= kBandedTiles; }

// P planes per operand (3: split fp32, 1: a 16-bit type), F16 selects the fp16 MFMA, S sub-steps
// per barrier.
template <int P, bool F16, int S, bool ACCUM, class Shape = BigTile>
__global__ __launch_bounds__(64 * Shape::kWaves, Shape::kPerSimd) void gemm_split_kernel(
    const piece* __restrict__ A, uint64_t Rpa, const piece* __restrict__ B, uint64_t Rpb, uint64_t K8,
    float* __restrict__ C, uint64_t ldc, uint64_t M, uint64_t N, float alpha, float beta,
    const float* __restrict__ row_scale, uint32_t tiles_n, uint32_t flags, const float* __restrict__ a_unscale,
    const float* __restrict__ b_unscale, uint32_t parts, uint64_t part_stride) {
    constexpr int BM = Shape::BM, BN = Shape::BN, kWavesN = Shape::kWavesN;
    constexpr int JT = Shape::JT;                    // 32-column MFMA tiles per wave
    constexpr int kAPieces = P * 2 * BM;             // [plane][half][row]
    constexpr int kSubPieces = P * 2 * (BM + BN);    // three planes: 3072 pieces = 48 KB
    constexpr int kBufPieces = S * kSubPieces;
    __shared__ piece lds[2][kBufPieces];

    uint32_t tile_id = blockIdx.x, part = 0, tile_m, tile_n;
    if (flags & kGemmTriangleGrid) {
        // the tile list is the lower triangle, row by row; `parts` copies of it: copy p multiplies the p-th share of the k
        // steps and writes its sums to the p-th matrix at C (a later pass adds the shares in order)
        const uint32_t lower = tiles_n * (tiles_n + 1) / 2;
        uint32_t unit;
        if (!xcd_unit(lower * parts, unit)) return;
        part = unit / lower;
        tile_id = unit % lower;
        C += (uint64_t)part * part_stride;
        short_k::triangle_tile(tile_id, tile_m, tile_n);
    } else if (flags & kGemmBandedGrid) {
        const uint32_t tiles_m = (uint32_t)((M + BM - 1) / BM);
        if (!xcd_unit(tiles_m * tiles_n, tile_id)) return;
        banded_tile(tile_id, tiles_m, tiles_n, tile_m, tile_n);
    } else {
        tile_m = tile_id / tiles_n;
        tile_n = tile_id % tiles_n;
    }
    const uint64_t m0 = (uint64_t)tile_m * BM, n0 = (uint64_t)tile_n * BN;
    // a symmetric product needs only the tiles that touch the lower triangle
    if ((flags & trakhip::kGemmLowerTilesOnly) && n0 > m0 + BM - 1) return;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;  // the wave number as a scalar
    const int wm = wave / kWavesN, wn = wave % kWavesN;
    const int x = lane & 31, h = lane >> 5;

    floatx16 acc[2][JT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const uint64_t all_steps = K8 / (2 * S);
    const uint64_t first = all_steps * part / parts, steps = all_steps * (part + 1) / parts;  // [first, steps)
    StepMover<P, S, Shape> mover;
    mover.init(A, Rpa, B, Rpb, K8, m0, n0, first, wave);
    const uint32_t lane_bytes = (uint32_t)lane * (uint32_t)sizeof(piece);
    mover.move_all(wave, lane_bytes, lds[0]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // piece index of this lane's operand for plane p: A rows wm*64 + 32*i + x, B rows wn*128 + 32*j + x
    const int a_lane = h * BM + wm * 64 + x;
    const int b_lane = kAPieces + h * BN + wn * (32 * JT) + x;

    // Fetching its code is part of a step of the one-plane product: [5000 x 4096] by 20 rows takes 94 us where the loop begins
    // with a 64-byte line, 96 from word 9 of a line on and 102 from word 2, so one word of a line is left to what the compiler
    // puts in front of the loop.  (Three planes differ by 1 %, two by up to 6 %; both lie well, and no time of theirs depends on this.)
    if constexpr (P == 1) asm volatile(".p2align 6\n\t.fill 15, 4, 0xbf800000");  // s_nop 0
    for (uint64_t s = first; s < steps; ++s) {
        const int cur = (int)((s - first) & 1);
        // the other buffer was last read before the barrier that ended the previous step
        if (s + 1 < steps) mover.move_all(wave, lane_bytes, lds[cur ^ 1]);
#pragma unroll
        for (int u = 0; u < S; ++u) {
            const piece* l = lds[cur] + u * kSubPieces;
            piece fa[2][P];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int p = 0; p < P; ++p) fa[i][p] = l[a_lane + p * 2 * BM + 32 * i];
#pragma unroll
            for (int j = 0; j < JT; ++j) {
                piece fb[P];
#pragma unroll
                for (int p = 0; p < P; ++p) fb[p] = l[b_lane + p * 2 * BN + 32 * j];
                if constexpr (P == 3) {
                    // the six plane pairs (pa, pb) with pa + pb <= 2, smallest terms first
                    constexpr int kPa[6] = {0, 1, 2, 0, 1, 0};
                    constexpr int kPb[6] = {2, 1, 0, 1, 0, 0};
#pragma unroll
                    for (int t6 = 0; t6 < 6; ++t6)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            acc[i][j] = mfma16<F16>(fa[i][kPa[t6]], fb[kPb[t6]], acc[i][j]);
                } else if constexpr (P == 2) {
                    // the three plane pairs with pa + pb <= 1, smaller terms first
                    constexpr int kPa[3] = {0, 1, 0};
                    constexpr int kPb[3] = {1, 0, 0};
#pragma unroll
                    for (int t3 = 0; t3 < 3; ++t3)
#pragma unroll
                        for (int i = 0; i < 2; ++i)
                            acc[i][j] = mfma16<F16>(fa[i][kPa[t3]], fb[kPb[t3]], acc[i][j]);
                } else {
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[i][j] = mfma16<F16>(fa[i][0], fb[0], acc[i][j]);
                }
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's pieces of the next step are in LDS
        __syncthreads();
    }

    store_c<ACCUM, JT, P == 2>(acc, C, ldc, M, N, m0 + wm * 64, n0 + wn * (32 * JT) + x, h, alpha, beta, row_scale,
                               a_unscale, b_unscale);
}

// ---- 16-bit operands read in place -----------------------------------------------------------
//
// Row-major fp16 / bf16 operands A[M, K], B[N, K] with K a multiple of 64 and 16-byte aligned rows need
// no planes.  A step is 64 values of k = one 128-byte line of every row: chunk c of a step is the
// lines of rows 8c .. 8c+7 of [256 rows of A | 256 rows of B], lane l of the moving wave fetches
// the 16-byte piece of row r = 8c + l/8 that belongs in slot l % 8, i.e. LDS holds each row's eight
// octets permuted: octet o sits in slot o ^ ((r / 2) % 8).  A wave's load instruction reads eight full
// lines; LDS serves a ds_read_b128 sixteen lanes at a time from 64 banks (256 bytes), and the sixteen
// lanes of a group (sixteen consecutive rows, one octet) land on sixteen different 16-byte columns
// of those 256 bytes - rows of equal parity share a 128-byte half and differ in r / 2.  Linear global
// reads, conflict-free LDS reads (XOR with r % 8 instead leaves a two-way conflict), and the same MFMA loop as
// the one-plane kernel.  Rows past M or N are fetched from the last row (their results are not stored).
template <class Shape, bool F16, bool ACCUM, int OUT = TRAKHIP_F32>
__global__ __launch_bounds__(64 * Shape::kWaves, 2) void gemm_nt16_kernel(
    const piece* __restrict__ A, uint64_t lda8, const piece* __restrict__ B, uint64_t ldb8, uint64_t steps,
    void* __restrict__ C_any, uint64_t ldc, uint64_t M, uint64_t N, float alpha, float beta,
    const float* __restrict__ row_scale, uint32_t tiles_n, uint32_t tiles, uint32_t in_bands, bool vec16) {
    constexpr int BM = Shape::BM, BN = Shape::BN, JT = Shape::JT, kWaves = Shape::kWaves, kWavesN = Shape::kWavesN;
    constexpr int kBufPieces = 8 * (BM + BN);  // 64 KB, or 32
    constexpr int kMoves = (BM + BN) / 8 / kWaves, kMovesA = BM / 8 / kWaves;  // chunks per wave and step
    __shared__ piece lds[2][kBufPieces];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;  // the wave number as a scalar
    const int wm = wave / kWavesN, wn = wave % kWavesN;
    const int x = lane & 31, h = lane >> 5;
    const int a_row = (wm * 64 + x) * 8, b_row = (BM + wn * (32 * JT) + x) * 8;  // first piece of the lane's rows

    // The workgroups are persistent: those of an XCD go through its eighth of the tiles side by side.  A load's address is a
    // scalar base (first row of the tile, advanced by one 128-byte line per step) plus this lane's byte offset
    // inside the tile's rows.
    const char* a_tile;
    const char* b_tile;
    uint32_t voff[kMoves];
    const uint32_t tiles_m = tiles / tiles_n;
    auto place = [&](uint32_t t, uint32_t& tm, uint32_t& tn) {
        if (in_bands) {
            banded_tile(t, tiles_m, tiles_n, tm, tn);
        } else {
            tm = t / tiles_n;
            tn = t % tiles_n;
        }
    };
    auto set_tile = [&](uint32_t t) {
        uint32_t tm, tn;
        place(t, tm, tn);
        const uint64_t m0 = (uint64_t)tm * BM, n0 = (uint64_t)tn * BN;
        a_tile = reinterpret_cast<const char*>(A + m0 * lda8);
        b_tile = reinterpret_cast<const char*>(B + n0 * ldb8);
        // rows 8c + sub of chunk c = wave + 8 i': (row >> 1) % 8 = 4 (wave % 2) + sub / 2
        const int sub = lane >> 3, oct = (lane & 7) ^ ((4 * (wave & 1) + (sub >> 1)) & 7);
#pragma unroll
        for (int i = 0; i < kMoves; ++i) {
            const uint32_t row = 8 * (wave + kWaves * (i % kMovesA)) + sub;
            if (i < kMovesA) {
                const uint64_t last = M - 1 - m0;
                voff[i] = (uint32_t)(((row < last ? row : last) * lda8 + oct) * 16);
            } else {
                const uint64_t last = N - 1 - n0;
                voff[i] = (uint32_t)(((row < last ? row : last) * ldb8 + oct) * 16);
            }
        }
    };
    auto dma = [&](uint64_t s, piece* buf) {
#pragma unroll
        for (int i = 0; i < kMoves; ++i) {
            const int c = (i < kMovesA ? 0 : BM / 8) + wave + kWaves * (i % kMovesA);  // scalar
            const char* base = (i < kMovesA ? a_tile : b_tile) + s * 128;
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(base + voff[i]),
                                             (void __attribute__((address_space(3)))*)(buf + 64 * c), 16, 0, 0);
        }
    };

    // A step is four sub-steps of eight MFMAs (two A fragments x four B fragments).  The six fragments of
    // sub-step u + 1 are requested before the MFMAs of sub-step u are issued, so an LDS read has eight MFMAs
    // (256 cycles) to arrive instead of stalling the wave; the per-step barrier sits in front of the last
    // sub-step, whose MFMAs then cover the first reads from the other buffer.  Two register sets, alternating.
    piece fa[2][2], fb[2][JT];
    auto fetch = [&](int buf, int u, int set) {
        const piece* l = lds[buf] + ((2 * u + h) ^ ((x >> 1) & 7));
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[set][i] = l[a_row + 256 * i];
#pragma unroll
        for (int j = 0; j < JT; ++j) fb[set][j] = l[b_row + 256 * j];
    };

    uint32_t tile, end = tiles, stride = gridDim.x;
    if (in_bands) {
        const uint32_t xcd = blockIdx.x & 7u;
        tile = (uint32_t)((uint64_t)xcd * tiles / 8u) + (blockIdx.x >> 3);
        end = (uint32_t)((xcd + 1ull) * tiles / 8u);
        stride = gridDim.x >> 3;
    } else {
        tile = blockIdx.x;
    }
    if (tile >= end) return;
    set_tile(tile);
    int first = 0;  // buffer that holds step 0 of the current tile
    dma(0, lds[0]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    for (;;) {
        floatx16 acc[2][JT];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < JT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
        uint32_t tile_m, tile_n;
        place(tile, tile_m, tile_n);
        const uint64_t m0 = (uint64_t)tile_m * BM, n0 = (uint64_t)tile_n * BN;
        const uint32_t next = tile + stride;

        fetch(first, 0, 0);
        // As in gemm_split_kernel, the loop at the start of a 64-byte line: the instance that accumulates into C takes 4010 us for
        // [50 000 x 4096] by 10 000 rows there, 4120 where the compiler puts it (the others differ by less than 1 %).
        if constexpr (ACCUM && JT == 4) asm volatile(".p2align 6\n\t.fill 14, 4, 0xbf800000");  // s_nop 0
        for (uint64_t s = 0; s < steps; ++s) {
            const int cur = (int)((s + first) & 1);
            const bool last_step = s + 1 == steps;
            if (!last_step) {
                dma(s + 1, lds[cur ^ 1]);
            } else if (next < end) {
                // step 0 of the next tile arrives under the last MFMAs and the stores of this one
                set_tile(next);
                dma(0, lds[cur ^ 1]);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int set = u & 1;
                // Wait for this sub-step's fragments HERE, while they are the only LDS reads in flight: the
                // compiler waits for all outstanding LDS reads at once (it cannot order them against the
                // LDS-direct loads), so the next reads are issued after this point and stay in flight under
                // the MFMAs.
                asm volatile("" ::"v"(fa[set][0]), "v"(fa[set][1]), "v"(fb[set][0]), "v"(fb[set][1]));
                if constexpr (JT == 4) asm volatile("" ::"v"(fb[set][JT - 2]), "v"(fb[set][JT - 1]));
                __builtin_amdgcn_sched_barrier(0);
                if (u < 3) {
                    fetch(cur, u + 1, set ^ 1);
                } else {
                    // every read of this buffer has completed; wait for this wave's part of the next buffer,
                    // meet the other waves, then start on the next buffer
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    __syncthreads();
                    if (!last_step) fetch(cur ^ 1, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < JT; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[i][j] = mfma16<F16>(fa[set][i], fb[set][j], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (OUT == TRAKHIP_F32)
            store_c<ACCUM, JT>(acc, static_cast<float*>(C_any), ldc, M, N, m0 + wm * 64, n0 + wn * (32 * JT) + x, h, alpha, beta,
                               row_scale);
        else
            store_c16<OUT, JT>(acc, static_cast<uint16_t*>(C_any), ldc, M, N, m0 + wm * 64, n0 + wn * (32 * JT) + x, h, alpha,
                               row_scale, vec16);
        if (next >= end) break;
        first = (int)((steps + first) & 1);
        tile = next;
    }
}

// ---- Gram product of 16-bit rows read in place -------------------------------------------------
//
// C = alpha X^T X + beta C for a row-major fp16 / bf16 matrix X[K, N]: the contraction runs down the rows, an MFMA
// operand is eight values of one column.  A step is 64 rows of the tile's 256 columns (32 KB per operand); gfx950's
// transposing LDS read (ds_read_b64_tr_b16) hands sixteen lanes, which name four rows of sixteen columns, four rows of a
// column each, so that two of them make an operand and X needs no transposing pass (94 us and 410 MB of traffic for
// [50 000, 2048] fp16).  X^T X with the result rounded: [50 000, 2048] 349 -> 242 us (to 260 on other cards), [8200, 4096] 274 -> 196,
// [2000, 512] 39 -> 25; bound by the MFMAs' power and, per step, the 64 LDS-direct loads of a CU.
// LDS holds a row as 32 pieces of 16 bytes; the 64-byte units of row k are permuted, unit u in place u ^ (k % 4): the
// four rows that 32 lanes read at a time then lie in different quarters of the 64 banks.  A wave's LDS-direct load
// brings two rows' 512 bytes, whole lines.  Rows past K (in the last step) are written to LDS as zeros; columns past N
// are read from the last eight and not stored.  MFMAs, their order and with it every bit are those of the one-plane
// product; the fragment pipeline is gemm_nt16_kernel's.  The grid lists the lower-triangle tiles, `parts` copies of them as
// in gemm_split_kernel.
typedef short short4v __attribute__((ext_vector_type(4)));

// rows 4 r + i / 4 of the lane's operand, r = 0, 1 (i = lane % 16)
template <int kRowBytes>
__device__ __forceinline__ piece read_transposed(const char* at) {
    typedef __attribute__((address_space(3))) short4v* lds_ptr;
    typedef uint32_t pair __attribute__((ext_vector_type(2)));
    const pair a = __builtin_bit_cast(pair, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at)));
    const pair b = __builtin_bit_cast(pair, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at + 4 * kRowBytes)));
    return piece{a[0], a[1], b[0], b[1]};
}

template <class Shape, bool F16, bool ACCUM>
__global__ __launch_bounds__(64 * Shape::kWaves, 2) void gram16_kernel(const char* __restrict__ X, uint64_t ld, uint64_t K,
                                                                uint64_t N, float* __restrict__ C, uint64_t ldc, float alpha,
                                                                float beta, uint32_t parts, uint64_t part_stride) {
    constexpr int BM = Shape::BM, BN = Shape::BN, JT = Shape::JT, kWaves = Shape::kWaves, kWavesN = Shape::kWavesN;
    constexpr int kStep = 64, kRowBytes = 2 * BM, kOperandBytes = kStep * kRowBytes;  // 32 KB, or 16
    static_assert(BM == BN, "both operands are columns of X");
    constexpr int kMoves = kOperandBytes / 1024 / kWaves;    // loads per wave, step and operand
    constexpr int kLoadRows = 1024 / kRowBytes, kRowSlots = 64 / kLoadRows;  // rows of a load, 16-byte pieces of a row
    static_assert(kLoadRows * kWaves == 16 && kMoves == 4, "load i of a wave: 16 i rows further down");
    __shared__ __attribute__((aligned(16))) char lds[2][2 * kOperandBytes];

    const uint32_t tiles = (uint32_t)((N + BM - 1) / BM), lower = tiles * (tiles + 1) / 2;
    uint32_t unit, tile_m, tile_n;
    if (!xcd_unit(lower * parts, unit)) return;
    const uint32_t part = unit / lower;
    C += (uint64_t)part * part_stride;
    short_k::triangle_tile(unit % lower, tile_m, tile_n);
    const uint64_t m0 = (uint64_t)tile_m * BM, n0 = (uint64_t)tile_n * BN;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;  // the wave number as a scalar
    const int wm = wave / kWavesN, wn = wave % kWavesN;
    const int x = lane & 31, h = lane >> 5;

    floatx16 acc[2][JT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const uint64_t all_steps = (K + kStep - 1) / kStep;
    const uint64_t first = all_steps * part / parts, steps = all_steps * (part + 1) / parts;  // [first, steps)

    // load i of a wave: rows 16 i + kLoadRows wave .. of the step; the lane's slot holds piece `from` of its row
    const int row = kLoadRows * wave + lane / kRowSlots, slot = lane % kRowSlots;
    const uint32_t from = 8u * (uint32_t)(4 * ((slot >> 2) ^ (row & 3)) + (slot & 3));  // first column of the piece
    const uint64_t last_m = N - 8 - m0, last_n = N - 8 - n0;
    const uint32_t a_from = from < last_m ? from : (uint32_t)last_m, b_from = from < last_n ? from : (uint32_t)last_n;
    const uint32_t a_off = (uint32_t)(row * ld + a_from) * 2u, b_off = (uint32_t)(row * ld + b_from) * 2u;
    const char* a_tile = X + 2 * m0;
    const char* b_tile = X + 2 * n0;
    auto dma = [&](uint64_t s, char* buf, int lo, int hi) {  // loads [lo, hi) of the wave
        if ((s + 1) * kStep <= K) {
#pragma unroll
            for (int i = lo; i < hi; ++i) {
                const uint64_t at = (s * kStep + 16 * (i % kMoves)) * ld * 2;  // scalar
                const char* base = (i < kMoves ? a_tile : b_tile) + at;
                char* to = buf + (i < kMoves ? 0 : kOperandBytes) + 1024 * (wave + kWaves * (i % kMoves));
                __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(base + (i < kMoves ? a_off : b_off)),
                                                 (void __attribute__((address_space(3)))*)to, 16, 0, 0);
            }
        } else {
            for (int i = lo; i < hi; ++i) {
                const uint64_t k = s * kStep + 16 * (i % kMoves);
                piece v = {0u, 0u, 0u, 0u};
                if (k + row < K)
                    v = *reinterpret_cast<const piece*>((i < kMoves ? a_tile : b_tile) + k * ld * 2 + (i < kMoves ? a_off : b_off));
                *reinterpret_cast<piece*>(buf + (i < kMoves ? 0 : kOperandBytes) + 1024 * (wave + kWaves * (i % kMoves)) + 16 * lane) = v;
            }
        }
    };

    // this lane's part of an operand's address: row 8 h + i / 4 of a sub-step's sixteen, columns 16 (lane / 16 % 2) + 4 (i % 4)
    const int i16 = lane & 15, quarter = i16 >> 2;
    const int lane_at = (8 * h + quarter) * kRowBytes + 32 * ((lane >> 4) & 1) + 8 * (i16 & 3);
    int a_at[2], b_at[JT];
#pragma unroll
    for (int i = 0; i < 2; ++i) a_at[i] = lane_at + 64 * ((2 * wm + i) ^ quarter);
#pragma unroll
    for (int j = 0; j < JT; ++j) b_at[j] = kOperandBytes + lane_at + 64 * ((JT * wn + j) ^ quarter);

    piece fa[2][2], fb[2][JT];
    auto fetch = [&](int buf, int u, int set) {
        const char* l = lds[buf] + 16 * u * kRowBytes;
#pragma unroll
        for (int i = 0; i < 2; ++i) fa[set][i] = read_transposed<kRowBytes>(l + a_at[i]);
#pragma unroll
        for (int j = 0; j < JT; ++j) fb[set][j] = read_transposed<kRowBytes>(l + b_at[j]);
    };

    dma(first, lds[0], 0, 2 * kMoves);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    fetch(0, 0, 0);
    for (uint64_t s = first; s < steps; ++s) {
        const int cur = (int)((s - first) & 1);
        const bool last_step = s + 1 == steps;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int set = u & 1;
            // the fragments of this sub-step are waited for here, before the next ones are requested (see gemm_nt16_kernel)
            asm volatile("" ::"v"(fa[set][0]), "v"(fa[set][1]), "v"(fb[set][0]), "v"(fb[set][1]));
            if constexpr (JT == 4) asm volatile("" ::"v"(fb[set][JT - 2]), "v"(fb[set][JT - 1]));
            __builtin_amdgcn_sched_barrier(0);
            if (u < 3) {
                fetch(cur, u + 1, set ^ 1);
                // One operand's loads of the next step under each of the first two sub-steps: all eight of a wave at once
                // fill LDS's write side while every wave waits for its fragments (50 000 rows, 1024 / 2048 / 3072 columns:
                // 102 -> 95, 249 -> 242, 551 -> 521 us; no size slower).  gemm_nt16_kernel gains 0-2 % from it at 2048
                // columns and loses 2 % at 128, so it keeps its loads together.
                if (u < 2 && !last_step) dma(s + 1, lds[cur ^ 1], u * kMoves, (u + 1) * kMoves);
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (!last_step) fetch(cur ^ 1, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < JT; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) acc[i][j] = mfma16<F16>(fa[set][i], fb[set][j], acc[i][j]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    store_c<ACCUM, JT>(acc, C, ldc, N, N, m0 + wm * 64, n0 + wn * (32 * JT) + x, h, alpha, beta, nullptr);
}

// C[i][j] = C[j][i] for j > i: completes a symmetric matrix whose lower triangle was computed.
__global__ __launch_bounds__(256) void mirror_lower_kernel(float* __restrict__ C, uint64_t ldc, uint64_t n) {
    __shared__ float t[32][33];
    // 32 x 32 blocks strictly above or on the diagonal, read from their mirror image
    const uint32_t bi = blockIdx.y, bj = blockIdx.x;
    if (bj < bi) return;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int r = ty; r < 32; r += 8) {
        const uint64_t src_row = (uint64_t)bj * 32 + r, src_col = (uint64_t)bi * 32 + tx;  // block (bj, bi), lower
        t[r][tx] = (src_row < n && src_col < n) ? C[src_row * ldc + src_col] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int r = ty; r < 32; r += 8) {
        const uint64_t row = (uint64_t)bi * 32 + r, col = (uint64_t)bj * 32 + tx;
        if (row < n && col < n && col > row) C[row * ldc + col] = t[tx][r];
    }
}

// C = alpha * (P_0 + P_1 + ... in this order) + beta * C on the lower triangle, mirrored into the upper
// one: closes a symmetric product whose k range was shared out over `parts` matrices at P.  OUT: element type of C; 16-bit
// results are rounded here (beta = 0; C 8-byte aligned, ldc a multiple of 4) instead of in a pass of their own.
template <int OUT>
__device__ __forceinline__ void store_quad(char* C, uint64_t at, const float (&v)[4]) {
    if constexpr (OUT == TRAKHIP_F32)
        *reinterpret_cast<float4u*>(C + 4 * at) = float4u{v[0], v[1], v[2], v[3]};  // 4-byte aligned
    else
        trakhip::store4<OUT>(C + 2 * at, make_float4(v[0], v[1], v[2], v[3]));
}
template <int OUT>
__device__ __forceinline__ void store_one(char* C, uint64_t at, float v) {
    if constexpr (OUT == TRAKHIP_F32)
        reinterpret_cast<float*>(C)[at] = v;
    else
        reinterpret_cast<uint16_t*>(C)[at] = OUT == TRAKHIP_F16 ? trakhip::cast_f16_bits(v) : trakhip::cast_bf16_bits(v);
}

template <int OUT>
__global__ __launch_bounds__(256) void gram_combine_kernel(const float* __restrict__ P, uint64_t part_stride,
                                                           uint32_t parts, char* __restrict__ C, uint64_t ldc,
                                                           uint64_t n, float alpha, float beta) {
    __shared__ float t[32][33];
    const uint32_t bi = blockIdx.y, bj = blockIdx.x;  // 32 x 32 block (bi, bj) on or under the diagonal
    if (bj > bi) return;
    // A thread adds up four columns of one row, eight shares' loads in flight (a share that does not exist is read
    // from the last one and not added).  A block on the diagonal also adds what lies above it (the 256-row tiles hold
    // it) and does not store that.  Bound by the latency of its loads: seven shares of 2048 x 2048 take 24 us, fifteen
    // of 512 x 512 5 us (12 us with four rows per thread, one column wide, one after the other).
    const int r = threadIdx.x >> 3, c = 4 * (threadIdx.x & 7);
    const uint64_t row = (uint64_t)bi * 32 + r, col = (uint64_t)bj * 32 + c;
    const bool whole = row < n && col + 4 <= n;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (whole) {
        const float* q = P + row * n + col;
        for (uint32_t p = 0; p < parts; p += 8) {
            float4u s[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i)
                s[i] = *reinterpret_cast<const float4u*>(q + (uint64_t)(p + i < parts ? p + i : parts - 1) * part_stride);
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += p + i < parts ? s[i][e] : 0.0f;
        }
    } else if (row < n) {
        for (uint32_t p = 0; p < parts; ++p)
            for (int e = 0; e < 4; ++e)
                if (col + e < n) v[e] += P[(uint64_t)p * part_stride + row * n + col + e];
    }
    const uint64_t at = row * ldc + col;
    const float* old = reinterpret_cast<const float*>(C) + at;  // (32-bit results only)
    if (whole && bj < bi) {
        float4u prev = {0.0f, 0.0f, 0.0f, 0.0f};
        if (OUT == TRAKHIP_F32 && beta != 0.0f) prev = *reinterpret_cast<const float4u*>(old);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = alpha * v[e];
            if (OUT == TRAKHIP_F32 && beta != 0.0f) v[e] += beta * prev[e];
        }
        store_quad<OUT>(C, at, v);
    } else if (row < n) {
        for (int e = 0; e < 4; ++e) {
            if (col + e > row || col + e >= n) continue;
            v[e] = alpha * v[e];
            if (OUT == TRAKHIP_F32 && beta != 0.0f) v[e] += beta * old[e];
            store_one<OUT>(C, at + e, v[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) t[r][c + e] = v[e];
    __syncthreads();
    // the mirror image: four columns of row 32 bj + r, from column c .. c + 3 of the transpose
    const uint64_t mrow = (uint64_t)bj * 32 + r, mcol = (uint64_t)bi * 32 + c, mirror = mrow * ldc + mcol;
    if (bj < bi && mcol + 4 <= n) {  // (mrow < mcol then)
        const float o[4] = {t[c][r], t[c + 1][r], t[c + 2][r], t[c + 3][r]};
        store_quad<OUT>(C, mirror, o);
    } else {
        for (int e = 0; e < 4; ++e)
            if (mrow < n && mcol + e < n && mcol + e > mrow) store_one<OUT>(C, mirror + e, t[c + e][r]);
    }
}

uint64_t padded_rows(uint64_t rows) { return (rows + kRowPad - 1) / kRowPad * kRowPad; }
uint64_t octets(uint64_t K) { return (K + 8 * kOctetPad - 1) / (8 * kOctetPad) * kOctetPad; }
int planes_of(int dtype) { return dtype == TRAKHIP_F32 ? 3 : 1; }
bool known_dtype(int dtype) { return dtype == TRAKHIP_F16 || dtype == TRAKHIP_BF16 || dtype == TRAKHIP_F32; }

}  // namespace

namespace trakhip {

size_t split_bytes(uint64_t rows, uint64_t K, int dtype) {
    if (rows == 0 || K == 0 || !known_dtype(dtype)) return 0;
    return (size_t)(planes_of(dtype) * octets(K) * padded_rows(rows) * 16);
}

int split_rows(const void* src, int dtype, uint64_t ld, uint64_t rows, uint64_t K, int transposed, void* planes,
               size_t planes_bytes, hipStream_t s) {
    if (!known_dtype(dtype)) return TRAKHIP_ERR_DTYPE;
    if (rows == 0 || K == 0) return TRAKHIP_ERR_SHAPE;
    if (ld < (transposed ? rows : K)) return TRAKHIP_ERR_SHAPE;
    if (!src || !planes) return TRAKHIP_ERR_NULL;
    if (planes_bytes < split_bytes(rows, K, dtype)) return TRAKHIP_ERR_WORKSPACE;
    const size_t esz = dtype == TRAKHIP_F32 ? 4 : 2;
    if ((reinterpret_cast<uintptr_t>(src) % esz) || (reinterpret_cast<uintptr_t>(planes) % 16)) return TRAKHIP_ERR_ALIGN;
    const uint64_t Rp = padded_rows(rows), K8 = octets(K);
    const uint64_t gx = Rp / 64, gy = (K8 + 3) / 4;
    if (gx * gy > 0x7FFFFFFFull) return TRAKHIP_ERR_SHAPE;
    const dim3 grid((uint32_t)(gx * gy)), block(256);
    uint4* out = static_cast<uint4*>(planes);
    // 16-byte loads of 8 (fp32: 4) consecutive values need the row starts aligned
    const bool aligned = reinterpret_cast<uintptr_t>(src) % 16 == 0 && (ld * esz) % 16 == 0;
    if (dtype == TRAKHIP_F32) {
        const float* f = static_cast<const float*>(src);
        if (transposed)
            hipLaunchKernelGGL(split_kernel<true>, grid, block, 0, s, f, ld, rows, K, Rp, K8, (uint32_t)gx, out);
        else if (aligned)
            hipLaunchKernelGGL(split_rows_kernel, dim3((uint32_t)(gx * (K8 / kOctetPad))), block, 0, s, f, ld, rows, K, Rp, K8,
                               (uint32_t)gx, out);
        else
            hipLaunchKernelGGL(split_kernel<false>, grid, block, 0, s, f, ld, rows, K, Rp, K8, (uint32_t)gx, out);
    } else {
        const uint16_t* h = static_cast<const uint16_t*>(src);
        if (transposed)
            hipLaunchKernelGGL((relayout16_kernel<true, false>), grid, block, 0, s, h, ld, rows, K, Rp, K8, (uint32_t)gx, out);
        else if (aligned)
            hipLaunchKernelGGL((relayout16_kernel<false, true>), grid, block, 0, s, h, ld, rows, K, Rp, K8, (uint32_t)gx, out);
        else
            hipLaunchKernelGGL((relayout16_kernel<false, false>), grid, block, 0, s, h, ld, rows, K, Rp, K8, (uint32_t)gx, out);
    }
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

}  // namespace trakhip

namespace {

// completes a symmetric matrix whose lower-triangle tiles were computed
int mirror_lower(float* C, uint64_t ldc, uint64_t N, hipStream_t s) {
    const uint64_t blocks = (N + 31) / 32;
    if (blocks > 65535) return TRAKHIP_ERR_SHAPE;
    hipLaunchKernelGGL(mirror_lower_kernel, dim3((uint32_t)blocks, (uint32_t)blocks), dim3(256), 0, s, C, ldc, N);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

// sub-steps per barrier of each operand format
int sub_steps(int dtype, bool two_planes) { return two_planes ? 2 : (dtype == TRAKHIP_F32 ? 1 : 4); }

// parts > 1 (symmetric products only): the k steps are shared out over `parts` launches' worth of
// workgroups that write plain sums into `parts` N x N matrices at C; see gram_combine_kernel.
// Rpa: rows that A's planes are laid out with (M and more, where A is the rest of a taller operand).
template <class Shape>
int launch_split_tiles(const piece* a, uint64_t Rpa, uint64_t M, const piece* b, uint64_t N, uint64_t K, int dtype, float* C,
                       uint64_t ldc, float alpha, float beta, const float* row_scale, hipStream_t s, uint32_t flags,
                       const float* a_unscale, const float* b_unscale, uint32_t parts) {
    const uint64_t tiles_m = (M + Shape::BM - 1) / Shape::BM, tiles_n = (N + Shape::BN - 1) / Shape::BN;
    if (tiles_m * tiles_n > 0x7FFFFFF0ull) return TRAKHIP_ERR_SHAPE;
    uint64_t workgroups = tiles_m * tiles_n;
    if (parts > 1) {
        flags = kGemmTriangleGrid;
        workgroups = (tiles_m * (tiles_m + 1) / 2 * parts + 7) / 8 * 8;
    }
    constexpr bool kBig = Shape::BN == BN;
    if (parts == 1 && !flags && (kBig ? banded(tiles_n) : tiles_n > 1 && tiles_n <= 2 * kBandedTiles)) {
        flags = kGemmBandedGrid;
        workgroups = (workgroups + 7) / 8 * 8;
    }
    const dim3 grid((uint32_t)workgroups), block(64 * Shape::kWaves);
    const uint64_t Rpb = padded_rows(N), K8 = octets(K);
    // ACCUM (beta != 0) fetches the old C in the epilogue; kept out of the plain kernel
    void (*kernel)(const piece*, uint64_t, const piece*, uint64_t, uint64_t, float*, uint64_t, uint64_t, uint64_t, float,
                   float, const float*, uint32_t, uint32_t, const float*, const float*, uint32_t, uint64_t);
    const bool accum = beta != 0.0f;
    if constexpr (!kBig)  // three planes only
        kernel = accum ? gemm_split_kernel<3, false, 1, true, Shape> : gemm_split_kernel<3, false, 1, false, Shape>;
    else if (a_unscale)
        kernel = accum ? gemm_split_kernel<2, true, 2, true> : gemm_split_kernel<2, true, 2, false>;
    else if (dtype == TRAKHIP_F32)
        kernel = accum ? gemm_split_kernel<3, false, 1, true> : gemm_split_kernel<3, false, 1, false>;
    else if (dtype == TRAKHIP_F16)
        kernel = accum ? gemm_split_kernel<1, true, 4, true> : gemm_split_kernel<1, true, 4, false>;
    else
        kernel = accum ? gemm_split_kernel<1, false, 4, true> : gemm_split_kernel<1, false, 4, false>;
    hipLaunchKernelGGL(kernel, grid, block, 0, s, a, Rpa, b, Rpb, K8, C, ldc, M, N, alpha, beta, row_scale,
                       (uint32_t)tiles_n, flags, a_unscale, b_unscale, parts, (uint64_t)N * N);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

// Rows of a three-plane product that go to 256 x 256 tiles (the others to 128 x 128): as big_tile_rows, microseconds per 16 values
// of k: 256 x 256 2.12 a round (a last one that leaves CUs idle 1.64, up to 2.1 as it fills), 128 x 128 tiles 0.82 for one on
// a CU, 1.34 for two side by side, 1.8 for three.  196 products of M = 1000 .. 50 000, N = 100 .. 8000, K = 512 .. 4096: 0.2 %
// above the fastest of the three on average, 5 % at worst, 27 % below 256 x 256 tiles alone and nowhere more than 3 % above (6 %
// at 64 values of k): [4000 x 4096] by 1024 rows 427 -> 210 us, [16 000 x 1024] by 300 117 -> 81, [50 000 x 2048] by 1024 1036 ->
// 975, [25 000 x 2048] by 4096 1851 -> 1790.
constexpr uint64_t kPlanCus = 256;
double big_planes_us(uint64_t M, uint64_t N, uint64_t K) {
    if (M == 0) return 0.0;
    const uint64_t tiles = (M + 255) / 256 * ((N + 255) / 256), full = tiles / kPlanCus;
    const double rest = (double)(tiles % kPlanCus) / (double)kPlanCus, k = (double)K / 16.0;
    return (double)full * (5.0 + 2.12 * k) + (rest > 0.0 ? 8.0 + k * (1.64 + (rest > 0.5 ? 0.9 * (rest - 0.5) : 0.0)) : 0.0);
}
double small_planes_us(uint64_t M, uint64_t N, uint64_t K) {
    if (M == 0) return 0.0;
    const uint64_t tiles = (M + 127) / 128 * ((N + 127) / 128), per_cu = (tiles + kPlanCus - 1) / kPlanCus;
    const double last[3] = {0.0, 0.82, 1.34};
    return 5.0 + (double)K / 16.0 * (1.8 * (double)(per_cu / 3) + last[per_cu % 3]);
}
uint64_t big_plane_rows(uint64_t M, uint64_t N, uint64_t K, double& us) {
    const uint64_t tiles_n = (N + 255) / 256, tiles = (M + 255) / 256 * tiles_n;
    uint64_t whole = tiles / kPlanCus * kPlanCus / tiles_n * 256;
    if (whole > M) whole = M;
    const double big = big_planes_us(M, N, K), small = small_planes_us(M, N, K);
    const double both = big_planes_us(whole, N, K) + small_planes_us(M - whole, N, K) + 1.0;
    if (whole > 0 && whole < M && both < 0.99 * big && both < small) return us = both, whole;
    return small < big ? (us = small, 0) : (us = big, M);
}

// Whether a symmetric product in `parts` shares takes 128 x 128 tiles: with N <= 768 the lower tiles of 256 x 256 are three or six
// a share, and sixteen shares leave most CUs idle.  Three planes: the estimate of big_plane_rows per share; 16-bit rows in place
// 0.9 us a step for a small tile on a CU and 1.3 for two (they bring twice the rows per entry).  [50 000, 512] fp32 372 -> 206 us
// and fp16 89 -> 54, [2000, 512] 36 -> 30 and 25 -> 20; [50 000, 1024] fp16 stays at 103 (121 on 128 x 128).
bool gram_small_tiles(uint64_t N, uint64_t K, int dtype, uint32_t parts) {
    const uint64_t big = (N + 255) / 256, small = (N + 127) / 128;
    const uint64_t big_tiles = big * (big + 1) / 2 * parts, small_tiles = small * (small + 1) / 2 * parts;
    const uint64_t rounds = (big_tiles + kPlanCus - 1) / kPlanCus, per_cu = (small_tiles + kPlanCus - 1) / kPlanCus;
    const double three[3] = {0.0, 0.82, 1.34}, two[2] = {0.0, 0.9};
    const double steps = (double)K / (dtype == TRAKHIP_F32 ? 16.0 : 64.0) / (double)parts;
    const double per_step = dtype == TRAKHIP_F32 ? 1.8 * (double)(per_cu / 3) + three[per_cu % 3]
                                                 : 1.3 * (double)(per_cu / 2) + two[per_cu % 2];
    return 5.0 + steps * per_step < (double)rounds * (6.0 + 1.6 * steps);
}

int launch_split(const void* A_planes, uint64_t M, const void* B_planes, uint64_t N, uint64_t K, int dtype, float* C,
                 uint64_t ldc, float alpha, float beta, const float* row_scale, hipStream_t s, uint32_t flags,
                 const float* a_unscale, const float* b_unscale, uint32_t parts = 1) {
    if (M == 0 || N == 0) return TRAKHIP_OK;
    if (K == 0 || ldc < N) return TRAKHIP_ERR_SHAPE;
    if (!A_planes || !B_planes || !C) return TRAKHIP_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(A_planes) % 16) || (reinterpret_cast<uintptr_t>(B_planes) % 16) ||
        (reinterpret_cast<uintptr_t>(C) % 4))
        return TRAKHIP_ERR_ALIGN;
    const piece* a = static_cast<const piece*>(A_planes);
    const piece* b = static_cast<const piece*>(B_planes);
    const uint64_t Rpa = padded_rows(M);
    if (((M + 127) / 128) * ((N + 127) / 128) > 0x7FFFFFF0ull) return TRAKHIP_ERR_SHAPE;
    if (parts > 1 && dtype == TRAKHIP_F32 && !a_unscale && gram_small_tiles(N, K, dtype, parts))
        return launch_split_tiles<SmallTile>(a, Rpa, M, b, N, K, dtype, C, ldc, alpha, beta, row_scale, s, 0u, nullptr, nullptr, parts);
    const bool three = dtype == TRAKHIP_F32 && !a_unscale && parts == 1 && !flags;
    double us;
    const uint64_t big = three ? big_plane_rows(M, N, K, us) : M;
    if (big) {
        const int e = launch_split_tiles<BigTile>(a, Rpa, big, b, N, K, dtype, C, ldc, alpha, beta, row_scale, s, flags, a_unscale,
                                                  b_unscale, parts);
        if (e || big == M) return e;
    }
    return launch_split_tiles<SmallTile>(a + big, Rpa, M - big, b, N, K, dtype, C + big * ldc, ldc, alpha, beta,
                                         row_scale ? row_scale + big : nullptr, s, 0u, nullptr, nullptr, 1);
}

// C = alpha A B^T + beta C of 16-bit operands in place on one shape of tiles; `slots` workgroups at a time
template <class Shape>
int launch_nt16(const char* A, uint64_t lda, const void* B, uint64_t ldb, int dtype, int out_dtype, char* C, uint64_t ldc,
                uint64_t M, uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, int slots, hipStream_t s) {
    const uint64_t tiles_m = (M + Shape::BM - 1) / Shape::BM, tiles_n = (N + Shape::BN - 1) / Shape::BN;
    void (*kernel)(const piece*, uint64_t, const piece*, uint64_t, uint64_t, void*, uint64_t, uint64_t, uint64_t, float,
                   float, const float*, uint32_t, uint32_t, uint32_t, bool);
    const bool accum = beta != 0.0f, f16 = dtype == TRAKHIP_F16;
    if (out_dtype == TRAKHIP_F16)
        kernel = f16 ? gemm_nt16_kernel<Shape, true, false, TRAKHIP_F16> : gemm_nt16_kernel<Shape, false, false, TRAKHIP_F16>;
    else if (out_dtype == TRAKHIP_BF16)
        kernel = f16 ? gemm_nt16_kernel<Shape, true, false, TRAKHIP_BF16> : gemm_nt16_kernel<Shape, false, false, TRAKHIP_BF16>;
    else if (f16)
        kernel = accum ? gemm_nt16_kernel<Shape, true, true> : gemm_nt16_kernel<Shape, true, false>;
    else
        kernel = accum ? gemm_nt16_kernel<Shape, false, true> : gemm_nt16_kernel<Shape, false, false>;
    const bool vec16 = reinterpret_cast<uintptr_t>(C) % 8 == 0 && ldc % 4 == 0;  // 8-byte stores of a 16-bit result
    const uint32_t tiles = (uint32_t)(tiles_m * tiles_n);
    // (tiles of 128 x 128: twice as many columns, and 64 tiles of an XCD at a time)
    const bool in_bands = (Shape::BN < 256 ? tiles_n > 1 && tiles_n <= 2 * kBandedTiles : banded(tiles_n)) && slots >= 8;
    uint32_t workgroups = tiles < (uint32_t)slots ? tiles : (uint32_t)slots;
    if (in_bands) workgroups = tiles < (uint32_t)slots ? (tiles + 7) / 8 * 8 : (uint32_t)slots / 8 * 8;
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(64 * Shape::kWaves), 0, s, reinterpret_cast<const piece*>(A), lda / 8,
                       static_cast<const piece*>(B), ldb / 8, K / 64, C, ldc, M, N, alpha, beta, row_scale, (uint32_t)tiles_n,
                       tiles, in_bands ? 1u : 0u, vec16);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

// Rows of a 16-bit product in place that go to 256 x 256 tiles; the others go to 128 x 128: none, all, or those behind as many
// rows of tiles as make whole rounds over the CUs, whichever estimate is smallest.  Microseconds, per 64 values of k and
// round of tiles over the CUs: 256 x 256 1.75 and 8.5 for the stores of C (a last round that leaves CUs idle 1.33, up to
// 1.73 as it fills: the clock), 128 x 128, two per CU, 1.03 and 4.5 (a last round 0.5 to 1.1).  196 products of
// M = 1000 .. 50 000, N = 100 .. 8000, K = 512 .. 4096: on average 0.3 % above the fastest of the three, at worst 9 %, never
// more than 2 % slower than 256 x 256 tiles alone and three quarters of their time on average: [50 000 x 2048] by 100 rows
// 64 -> 43 us, by 2048 427 -> 410, [2000 x 512] by 512 21 -> 13, [4000 x 2048] by 1024 55 -> 28.
// Less than 512 values of k, 280 products: 4 % above the fastest, at worst 39 % ([12 000 x 256] by 1500 rows 54 us, all on 128 x 128 39);
// 16 % below 256 x 256 tiles alone, at worst 8 % above ([7000 x 128] by 3000 rows 46 us and 42).
double big_tiles_us(uint64_t M, uint64_t N, uint64_t K, int cus) {
    if (M == 0) return 0.0;
    const uint64_t tiles = (M + 255) / 256 * ((N + 255) / 256), full = tiles / cus;
    const double rest = (double)tiles / cus - (double)full, k = (double)K / 64.0;
    const double last = 8.0 + k * (1.33 + (rest > 0.5 ? 0.8 * (rest - 0.5) : 0.0));
    return (double)full * (8.5 + 1.75 * k) + (rest > 0.0 ? last : 0.0);
}
double small_tiles_us(uint64_t M, uint64_t N, uint64_t K, int cus) {
    if (M == 0) return 0.0;
    const uint64_t tiles = (M + 127) / 128 * ((N + 127) / 128), full = tiles / (2 * cus);
    const double rest = (double)tiles / (2 * cus) - (double)full, k = (double)K / 64.0;
    return (double)full * (4.5 + 1.03 * k) + (rest > 0.0 ? 5.0 + k * (0.5 + 0.6 * rest) : 0.0);
}
uint64_t big_tile_rows(uint64_t M, uint64_t N, uint64_t K, int cus) {
    const uint64_t tiles_n = (N + 255) / 256, tiles = (M + 255) / 256 * tiles_n;
    uint64_t whole = tiles / cus * cus / tiles_n * 256;
    if (whole > M) whole = M;
    const double big = big_tiles_us(M, N, K, cus), small = small_tiles_us(M, N, K, cus);
    const double both = big_tiles_us(whole, N, K, cus) + small_tiles_us(M - whole, N, K, cus) + 1.0;
    if (whole > 0 && whole < M && both < big && both < small) return whole;
    return small < big ? 0 : M;
}

// A symmetric product has (tiles + 1) tiles / 2 workgroups' worth of work; up to 170 of them leave a third of the
// CUs idle, and the k range is long enough to share out.  The number of shares, up to `most` and to what `room` bytes hold,
// is the one whose estimate is smallest: rounds of workgroups over the 256 CUs times the steps of a share (1.6 us each,
// 1.8 for two planes; 6 us for a workgroup's first loads and its stores), plus 0.2 us per MB that the pass behind the product
// goes over: the shares it adds up or, for one share, the matrix it mirrors.  Timed for all numbers of shares at
// N = 512 .. 4096, K = 2000 .. 50 000: on 256 x 256 tiles, which one and two planes always take, the choice is at most 3 % above the fastest
// number.  Of 16-bit rows in place and three planes, whose tiles gram_small_tiles chooses for the number that is fixed here, the pair is
// 3 and 6 % above the fastest pair on average and up to 31 % ([20 000, 1024] fp32: 166 us in sixteen shares of 256 x 256 tiles, 126 in fourteen of 128 x 128).
// N = 2048 takes seven (36 tiles: 252 workgroups; three gave 108), N = 512 at 2000 values of k sixteen, N = 4096 seven at
// 50 000 values of k (952 workgroups, 3.7 rounds; three leave the second of two rounds 60 % full) and one at 2000 of 16 bits
// (80 us; three 95).  A share has at least eight steps, and the shares together at most 512 MB.  Product and
// sum against three shares, X^T X of [50 000, 2048] fp16 from its planes: 445 -> 248 us, of [50 000, 512] 371 -> 87.
// (gram16_kernel takes the same numbers.)
constexpr uint32_t kGramPartsMax = 16, kGramPartsFew = 3, kGramTilesMax = 170;
uint32_t gram_parts(uint64_t N, uint64_t K, int dtype, bool two_planes, uint32_t most, size_t room = SIZE_MAX) {
    const uint64_t tiles = (N + BM - 1) / BM, lower = tiles * (tiles + 1) / 2;
    const uint64_t steps = octets(K) / (2 * sub_steps(dtype, two_planes));
    if (lower > kGramTilesMax || steps < 8 * kGramPartsFew) return 1;
    // (N is bounded from here on: N * N * 4 neither overflows nor is zero)
    const size_t fit = room / ((size_t)N * N * sizeof(float));
    constexpr uint64_t kCus = 256;
    const double share_mb = 4e-6 * (double)N * (double)N;
    const double step_us = two_planes ? 1.8 : 1.6;
    uint32_t best = 1;
    double best_us = 0;
    for (uint32_t p = 1; p <= most; ++p) {
        if (p > 1 && (p > fit || steps < 8 * p || p * share_mb > 512.0)) break;
        const uint64_t rounds = (lower * p + kCus - 1) / kCus;
        const double us = (double)rounds * (step_us * (double)((steps + p - 1) / p) + 6.0) + 0.2 * p * share_mb;
        if (p == 1 || us < best_us) best = p, best_us = us;
    }
    return best;
}

// adds up the shares at P and mirrors the sum
int combine_shares(const float* P, uint32_t parts, int out_dtype, void* C, uint64_t ldc, uint64_t N, float alpha, float beta,
                   hipStream_t s) {
    const uint64_t blocks = (N + 31) / 32;
    if (blocks > 65535) return TRAKHIP_ERR_SHAPE;
    const dim3 grid((uint32_t)blocks, (uint32_t)blocks);
    char* out = static_cast<char*>(C);
    auto kernel = out_dtype == TRAKHIP_F32   ? gram_combine_kernel<TRAKHIP_F32>
                  : out_dtype == TRAKHIP_F16 ? gram_combine_kernel<TRAKHIP_F16>
                                             : gram_combine_kernel<TRAKHIP_BF16>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, P, (uint64_t)N * N, parts, out, ldc, N, alpha, beta);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

int gram_impl(const void* A_planes, const float* a_scales, uint64_t N, uint64_t K, int dtype, float* C, uint64_t ldc,
              float alpha, float beta, void* ws, size_t ws_bytes, hipStream_t s) {
    if (N == 0) return TRAKHIP_OK;
    const bool two_planes = a_scales != nullptr;
    // a smaller scratch takes the number of shares that is fastest among those it holds
    const bool usable = ws && reinterpret_cast<uintptr_t>(ws) % 16 == 0;
    const uint32_t parts = usable ? gram_parts(N, K, dtype, two_planes, kGramPartsMax, ws_bytes) : 1;
    if (parts > 1) {
        if (!C) return TRAKHIP_ERR_NULL;
        if (ldc < N) return TRAKHIP_ERR_SHAPE;
        float* shares = static_cast<float*>(ws);
        const int e = launch_split(A_planes, N, A_planes, N, K, dtype, shares, N, 1.0f, 0.0f, nullptr, s, 0u, a_scales,
                                   a_scales, parts);
        if (e) return e;
        return combine_shares(shares, parts, TRAKHIP_F32, C, ldc, N, alpha, beta, s);
    }
    const int e = launch_split(A_planes, N, A_planes, N, K, dtype, C, ldc, alpha, beta, nullptr, s, trakhip::kGemmLowerTilesOnly,
                               a_scales, a_scales);
    if (e) return e;
    return mirror_lower(C, ldc, N, s);
}

}  // namespace

namespace trakhip {

double split_product_us(uint64_t M, uint64_t N, uint64_t K) {
    double us;
    big_plane_rows(M, N, K, us);
    return us;
}

double split_product_big_us(uint64_t M, uint64_t N, uint64_t K) { return big_planes_us(M, N, K); }

int gemm_nt_split(const void* A_planes, uint64_t M, const void* B_planes, uint64_t N, uint64_t K, int dtype, float* C,
                  uint64_t ldc, float alpha, float beta, const float* row_scale, hipStream_t s, uint32_t flags) {
    if (!known_dtype(dtype)) return TRAKHIP_ERR_DTYPE;
    return launch_split(A_planes, M, B_planes, N, K, dtype, C, ldc, alpha, beta, row_scale, s, flags, nullptr, nullptr);
}

size_t split2_bytes(uint64_t rows, uint64_t K) {
    if (rows == 0 || K == 0) return 0;
    return (size_t)(2 * octets(K) * padded_rows(rows) * 16);
}

int split2_rows(const float* src, uint64_t ld, uint64_t rows, uint64_t K, int transposed, void* planes,
                size_t planes_bytes, float* scales, hipStream_t s) {
    if (rows == 0 || K == 0) return TRAKHIP_ERR_SHAPE;
    if (ld < (transposed ? rows : K)) return TRAKHIP_ERR_SHAPE;
    if (!src || !planes || !scales) return TRAKHIP_ERR_NULL;
    if (planes_bytes < split2_bytes(rows, K)) return TRAKHIP_ERR_WORKSPACE;
    if ((reinterpret_cast<uintptr_t>(src) % 4) || (reinterpret_cast<uintptr_t>(planes) % 16) ||
        (reinterpret_cast<uintptr_t>(scales) % 4))
        return TRAKHIP_ERR_ALIGN;
    const uint64_t Rp = padded_rows(rows), K8 = octets(K);
    const uint64_t gx = Rp / 64, gy = (K8 + 3) / 4;
    if (gx * gy > 0x7FFFFFFFull || rows > 0x7FFFFFFFull) return TRAKHIP_ERR_SHAPE;
    // scales[0 .. rows) receives the inverse factors; scales[rows .. 2 rows) holds the row maxima meanwhile
    uint32_t* maxbits = reinterpret_cast<uint32_t*>(scales + rows);
    if (transposed) {
        hipLaunchKernelGGL(zero_u32_kernel, dim3((uint32_t)((rows + 255) / 256)), dim3(256), 0, s, maxbits, rows);
        hipLaunchKernelGGL(absmax_cols_kernel, dim3((uint32_t)((rows + 255) / 256), kColChunks), dim3(256), 0, s, src, ld,
                           rows, K, maxbits);
    } else {
        hipLaunchKernelGGL(absmax_rows_kernel, dim3((uint32_t)((rows + 3) / 4)), dim3(256), 0, s, src, ld, rows, K,
                           maxbits);
    }
    const dim3 grid((uint32_t)(gx * gy)), block(256);
    uint4* out = static_cast<uint4*>(planes);
    const bool aligned = reinterpret_cast<uintptr_t>(src) % 16 == 0 && (ld * 4) % 16 == 0;
    if (transposed)
        hipLaunchKernelGGL((split2_kernel<true, false>), grid, block, 0, s, src, ld, rows, K, Rp, K8, (uint32_t)gx, maxbits,
                           out, scales);
    else if (aligned)
        hipLaunchKernelGGL((split2_kernel<false, true>), grid, block, 0, s, src, ld, rows, K, Rp, K8, (uint32_t)gx, maxbits,
                           out, scales);
    else
        hipLaunchKernelGGL((split2_kernel<false, false>), grid, block, 0, s, src, ld, rows, K, Rp, K8, (uint32_t)gx,
                           maxbits, out, scales);
    return hipGetLastError() == hipSuccess ? TRAKHIP_OK : TRAKHIP_ERR_LAUNCH;
}

int gemm_nt_split2(const void* A_planes, const float* a_scales, uint64_t M, const void* B_planes, const float* b_scales,
                   uint64_t N, uint64_t K, float* C, uint64_t ldc, float alpha, float beta, const float* row_scale,
                   hipStream_t s, uint32_t flags) {
    if ((M && !a_scales) || (N && !b_scales)) return TRAKHIP_ERR_NULL;
    return launch_split(A_planes, M, B_planes, N, K, TRAKHIP_F32, C, ldc, alpha, beta, row_scale, s, flags, a_scales,
                        b_scales);
}

size_t gram_split_workspace_bytes(uint64_t N, uint64_t K, int dtype, int two_planes, bool most) {
    if (N == 0 || K == 0 || !known_dtype(dtype)) return 0;
    const uint32_t parts = gram_parts(N, K, dtype, two_planes != 0, most ? kGramPartsMax : kGramPartsFew);
    return parts > 1 ? (size_t)parts * N * N * sizeof(float) : 0;
}

int gram_split2(const void* A_planes, const float* a_scales, uint64_t N, uint64_t K, float* C, uint64_t ldc, float alpha,
                float beta, void* ws, size_t ws_bytes, hipStream_t s) {
    if (N && !a_scales) return TRAKHIP_ERR_NULL;
    return gram_impl(A_planes, a_scales, N, K, TRAKHIP_F32, C, ldc, alpha, beta, ws, ws_bytes, s);
}

int gemm_nt16(const void* A, uint64_t lda, const void* B, uint64_t ldb, int dtype, int out_dtype, void* C, uint64_t ldc,
              uint64_t M, uint64_t N, uint64_t K, float alpha, float beta, const float* row_scale, hipStream_t s) {
    if (dtype != TRAKHIP_F16 && dtype != TRAKHIP_BF16) return TRAKHIP_ERR_DTYPE;
    if (!known_dtype(out_dtype)) return TRAKHIP_ERR_DTYPE;
    if (M == 0 || N == 0) return TRAKHIP_OK;
    if (K == 0 || K % 64 || lda < K || ldb < K || ldc < N) return TRAKHIP_ERR_SHAPE;
    // a lane's byte offset inside the 256 rows of a tile is kept in 32 bits
    if (lda >= (1ull << 23) || ldb >= (1ull << 23)) return TRAKHIP_ERR_SHAPE;
    if (!A || !B || !C) return TRAKHIP_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(A) % 16) || (reinterpret_cast<uintptr_t>(B) % 16) || (lda % 8) || (ldb % 8) ||
        (reinterpret_cast<uintptr_t>(C) % (out_dtype == TRAKHIP_F32 ? 4 : 2)))
        return TRAKHIP_ERR_ALIGN;
    if (out_dtype != TRAKHIP_F32 && beta != 0.0f) return TRAKHIP_ERR_SHAPE;
    if (((M + 127) / 128) * ((N + 127) / 128) > 0x7FFFFFF0ull) return TRAKHIP_ERR_SHAPE;
    // persistent workgroups: one per CU with 256 x 256 tiles (128 KB of LDS each), two with 128 x 128
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    const char* a = static_cast<const char*>(A);
    char* c = static_cast<char*>(C);
    const uint64_t big = big_tile_rows(M, N, K, cus);
    if (big) {
        const int e = launch_nt16<BigTile>(a, lda, B, ldb, dtype, out_dtype, c, ldc, big, N, K, alpha, beta, row_scale, cus, s);
        if (e || big == M) return e;
    }
    return launch_nt16<SmallTile>(a + 2 * big * lda, lda, B, ldb, dtype, out_dtype, c + big * ldc * (out_dtype == TRAKHIP_F32 ? 4 : 2),
                                  ldc, M - big, N, K, alpha, beta, row_scale ? row_scale + big : nullptr, 2 * cus, s);
}

int gram16(const void* X, int dtype, uint64_t ld, uint64_t K, uint64_t N, int out_dtype, void* C, uint64_t ldc, float alpha,
           float beta, void* ws, size_t ws_bytes, hipStream_t s) {
    if (dtype != TRAKHIP_F16 && dtype != TRAKHIP_BF16) return TRAKHIP_ERR_DTYPE;
    if (!known_dtype(out_dtype)) return TRAKHIP_ERR_DTYPE;
    if (N == 0) return TRAKHIP_OK;
    // (a lane's byte offset inside sixteen rows is kept in 32 bits)
    if (K == 0 || N % 8 || ld % 8 || ld < N || ld >= (1ull << 23) || ldc < N) return TRAKHIP_ERR_SHAPE;
    if (!X || !C) return TRAKHIP_ERR_NULL;
    const bool wide = out_dtype == TRAKHIP_F32;
    if ((reinterpret_cast<uintptr_t>(X) % 16) || (reinterpret_cast<uintptr_t>(C) % (wide ? 4 : 8))) return TRAKHIP_ERR_ALIGN;
    if (!wide && (ldc % 4 || beta != 0.0f)) return TRAKHIP_ERR_SHAPE;
    const bool usable = ws && reinterpret_cast<uintptr_t>(ws) % 16 == 0;
    const uint32_t parts = usable ? gram_parts(N, K, dtype, false, kGramPartsMax, ws_bytes) : 1;
    // a 16-bit result is rounded by the pass behind the product, which needs the sums in scratch
    const bool scratch = parts > 1 || !wide;
    if (scratch && !(usable && ws_bytes / sizeof(float) / N >= N * parts)) return TRAKHIP_ERR_WORKSPACE;
    const bool small = gram_small_tiles(N, K, dtype, parts);
    const uint64_t tiles = small ? (N + SmallTile::BM - 1) / SmallTile::BM : (N + BM - 1) / BM, lower = tiles * (tiles + 1) / 2;
    if (lower * parts > 0x7FFFFFF0ull) return TRAKHIP_ERR_SHAPE;
    float* sums = scratch ? static_cast<float*>(ws) : static_cast<float*>(C);
    const bool accum = !scratch && beta != 0.0f, f16 = dtype == TRAKHIP_F16;
    void (*kernel)(const char*, uint64_t, uint64_t, uint64_t, float*, uint64_t, float, float, uint32_t, uint64_t);
    if (small)
        kernel = f16 ? (accum ? gram16_kernel<SmallTile, true, true> : gram16_kernel<SmallTile, true, false>)
                     : (accum ? gram16_kernel<SmallTile, false, true> : gram16_kernel<SmallTile, false, false>);
    else
        kernel = f16 ? (accum ? gram16_kernel<BigTile, true, true> : gram16_kernel<BigTile, true, false>)
                     : (accum ? gram16_kernel<BigTile, false, true> : gram16_kernel<BigTile, false, false>);
    hipLaunchKernelGGL(kernel, dim3((uint32_t)((lower * parts + 7) / 8 * 8)), dim3(64 * (small ? SmallTile::kWaves : kWaves)), 0, s,
                       static_cast<const char*>(X), ld, K, N, sums, scratch ? N : ldc, scratch ? 1.0f : alpha,
                       scratch ? 0.0f : beta, parts, (uint64_t)N * N);
    if (hipGetLastError() != hipSuccess) return TRAKHIP_ERR_LAUNCH;
    return scratch ? combine_shares(sums, parts, out_dtype, C, ldc, N, alpha, beta, s) : mirror_lower(sums, ldc, N, s);
}

int gram_split(const void* A_planes, uint64_t N, uint64_t K, int dtype, float* C, uint64_t ldc, float alpha, float beta,
               void* ws, size_t ws_bytes, hipStream_t s) {
    if (!known_dtype(dtype)) return TRAKHIP_ERR_DTYPE;
    return gram_impl(A_planes, nullptr, N, K, dtype, C, ldc, alpha, beta, ws, ws_bytes, s);
}

}  // namespace trakhip
