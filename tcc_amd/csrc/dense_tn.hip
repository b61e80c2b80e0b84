// Tall-skinny transposed products C = A^T B of the GCN layer backward, for
// gfx950 (reference: torch.mm(X_out.T, d_output),
// TAC_training_backend/train/tcgnn_conv_release.py:150).
//
// A [K x M] and B [K x N] are row-major with K = graph nodes (millions) and
// M, N = layer widths (hundreds or less).  K is split over workgroups; each
// accumulates the product of its rows for one block of C with MFMA (fp32
// ones, or for wide outputs bf16 ones of the operands' exact parts) and
// writes it to a partial buffer, and a second kernel sums the partials in a
// fixed order.
//
// MFMA operand layout (16x16x4, fp32): lane l supplies A(i = l%16, k = l/16)
// and B(k = l/16, j = l%16), and holds D(4*(l/16) + v, l%16) in accumulator
// register v.  For C = A^T B the A operand of a 16x16 tile at (m0, n0) and
// rows k..k+3 is A[k + l/16][m0 + l%16] and the B operand B[k + l/16][n0 + l%16]:
// both are 16 consecutive floats of one input row per lane quarter, so the
// operands are loaded straight from global memory without a transpose.
// Columns past M (N) are clamped to the last one: they only feed rows
// (columns) of C that are never stored.  Rows past K are zero.
#include <algorithm>
#include <mutex>

#include "../../include/tcc_gcn.h"
#include "../../include/tcc_swtcf.h"
#include "common.hpp"
#include "primitives.hpp"

namespace tcc {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct TnArgs {
    const float* A;
    const float* B;
    float* partial;  // [splits][M][N]
    std::uint32_t lda, ldb;
    std::uint32_t K, M, N;
    std::uint32_t rowsPerSplit;
    std::uint32_t blocksM;  // blocks of C along M
    // Wide outputs only (tn_split_kernel)
    std::uint32_t blocksN, splits;
    // Relu-gradient form only (see tn_split_kernel): G [K x C] with row
    // stride ldg, W2 [N x C], and the H^T G partials [splits][N][C].
    const float* G;
    const float* W2;
    float* partial2;
    std::uint32_t ldg, C;
};

__device__ __forceinline__ std::uint32_t tn_uniform(std::uint32_t v) {
    return static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

// Narrow outputs (M or N of 16 and less), bound by reading the rows.
// Workgroup = WM x WN waves; a wave owns TM x TN tiles of 16x16, so a
// workgroup covers a (16*TM*WM) x (16*TN*WN) block of C.  Each iteration
// takes U steps of 4 rows; the next iteration's operands are loaded while
// the current one is multiplied.
template <int TM, int TN, int WM, int WN, int U>
__global__ void __launch_bounds__(kWave * WM * WN) tn_partial_kernel(TnArgs a) {
    constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
    constexpr std::uint32_t kStep = 4 * U;
    const unsigned lane = __lane_id();
    const unsigned wave = tn_uniform(threadIdx.x / kWave);
    const unsigned wm = wave % WM, wn = wave / WM;
    const std::uint32_t cbm = blockIdx.y % a.blocksM, cbn = blockIdx.y / a.blocksM;
    const std::uint32_t m0 = cbm * BM + wm * 16 * TM, n0 = cbn * BN + wn * 16 * TN;
    const std::uint32_t k0 = blockIdx.x * a.rowsPerSplit;
    const std::uint32_t k1 = min(a.K, k0 + a.rowsPerSplit);
    const unsigned li = lane & 15u, lk = lane >> 4;

    // Per-lane element offsets inside a 4-row step (row lk, clamped column).
    std::uint32_t offA[TM], offB[TN];
#pragma unroll
    for (int t = 0; t < TM; ++t) offA[t] = lk * a.lda + min(m0 + 16 * t + li, a.M - 1);
#pragma unroll
    for (int t = 0; t < TN; ++t) offB[t] = lk * a.ldb + min(n0 + 16 * t + li, a.N - 1);

    f32x4 acc[TM][TN];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u) acc[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto load_full = [&](std::uint32_t k, float (&xa)[U][TM], float (&xb)[U][TN]) {
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const float* ra = a.A + static_cast<std::uint64_t>(k + 4 * s) * a.lda;
            const float* rb = a.B + static_cast<std::uint64_t>(k + 4 * s) * a.ldb;
#pragma unroll
            for (int t = 0; t < TM; ++t) xa[s][t] = ra[offA[t]];
#pragma unroll
            for (int t = 0; t < TN; ++t) xb[s][t] = rb[offB[t]];
        }
    };
    auto multiply = [&](const float (&xa)[U][TM], const float (&xb)[U][TN]) {
#pragma unroll
        for (int s = 0; s < U; ++s)
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int u = 0; u < TN; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[s][t], xb[s][u], acc[t][u], 0, 0, 0);
    };

    // Two operand buffers in turn; loads are unconditional (past the last
    // full iteration they repeat in-bounds rows and are not used), so the
    // loads of one buffer stay in flight while the other is multiplied.
    // (sched_barrier keeps the scheduler from sinking the loads to their
    // uses, which it does to lower register pressure.)
    const std::uint32_t rows = k1 > k0 ? k1 - k0 : 0u;
    const std::uint32_t nFull = rows / kStep;
    float ca[U][TM], cb[U][TN], na[U][TM], nb[U][TN];
    if (nFull > 0) load_full(k0, ca, cb);
    std::uint32_t i = 0;
    for (; i + 1 < nFull; i += 2) {
        const std::uint32_t k = k0 + i * kStep;
        load_full(k + kStep, na, nb);
        __builtin_amdgcn_sched_barrier(0);
        multiply(ca, cb);
        __builtin_amdgcn_sched_barrier(0);
        load_full(i + 2 < nFull ? k + 2 * kStep : k + kStep, ca, cb);
        __builtin_amdgcn_sched_barrier(0);
        multiply(na, nb);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (i < nFull) multiply(ca, cb);
    const std::uint32_t kt = k0 + nFull * kStep;
    if (kt < k1) {  // last rows of the split: zeros past k1
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const bool in = kt + 4 * s + lk < k1;
            const float* ra = a.A + static_cast<std::uint64_t>(kt + 4 * s) * a.lda;
            const float* rb = a.B + static_cast<std::uint64_t>(kt + 4 * s) * a.ldb;
#pragma unroll
            for (int t = 0; t < TM; ++t) ca[s][t] = in ? ra[offA[t]] : 0.0f;
#pragma unroll
            for (int t = 0; t < TN; ++t) cb[s][t] = in ? rb[offB[t]] : 0.0f;
        }
        multiply(ca, cb);
    }

    // Tile (t, u): accumulator v of lane l is C(16t + 4*(l/16) + v, 16u + l%16).
    float* out = a.partial + static_cast<std::uint64_t>(blockIdx.x) * a.M * a.N;
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int u = 0; u < TN; ++u) {
            const std::uint32_t n = n0 + 16 * u + li;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const std::uint32_t m = m0 + 16 * t + 4 * lk + v;
                if (m < a.M && n < a.N) out[static_cast<std::uint64_t>(m) * a.N + n] = acc[t][u][v];
            }
        }
}

// Two floats as three bf16 each: x = hi + mid + lo exactly (8 + 8 + 8 of the
// 24 significant bits, each part rounded to nearest), two to a register.
__device__ __forceinline__ void split3(float x0, float x1, std::uint32_t& hi, std::uint32_t& mid, std::uint32_t& lo) {
    const auto pack = [](float p, float q) {
        return __builtin_bit_cast(std::uint32_t, __builtin_convertvector(f32x2{p, q}, bf16x2));
    };
    hi = pack(x0, x1);
    const float r0 = x0 - __uint_as_float(hi << 16), r1 = x1 - __uint_as_float(hi & 0xFFFF0000u);
    mid = pack(r0, r1);
    lo = pack(r0 - __uint_as_float(mid << 16), r1 - __uint_as_float(mid & 0xFFFF0000u));
}

// A split is exact from 2^-110 on; parts of a smaller element go below bf16's
// smallest number, 2^-133 (the MFMA keeps subnormal operands and sums), and up
// to 2^-134 of it is lost.  Whether that counts depends on what the element
// meets: 2^-120 beside ones is nothing, against 2^119 it is most of the result.
// So a block is formed again with fp32 products where a loss in each of `rows`
// products, by the largest element of the other operand's column, comes to more
// than 2^-24 of an element of the result.
__device__ __forceinline__ float split_loss(std::uint32_t rows) { return 0x1p-109f * static_cast<float>(rows); }

// Smaller for smaller |x|, zero (which a split keeps) the largest.
__device__ __forceinline__ std::uint32_t smallness(float x) { return (__float_as_uint(x) << 1) - 1u; }
constexpr std::uint32_t kSplitExactBits = ((127u - 110u) << 24) - 1u;  // of 2^-110

// Sums of fewer products are left to the fp32 products.  The six part products
// give a single product to 1.6e-7 of it (the three left out and the MFMA's
// truncation), fp32 MFMA to 6e-8; sums of 1, 2, 3, 4 normal products are off by
// 3.5, 3.3, 3.3, 3.2e-8 of the result, in fp32 by 2.5, 3.1, 3.6, 4.0e-8, and the
// longer the sum, the further the part products are ahead (100 products: 5.6e-8
// against 1.8e-7): 32 rows are rounded together.  A long sum with one term that
// is not zero is a single product all the same.
constexpr std::uint32_t kSplitMinTerms = 4;

// Wide outputs.  fp32 MFMA runs at 1/16 of the bf16 rate, and the 100 x 256
// and 602 x 256 products over node rows were bound by it (110 TFLOP/s).  Here
// each operand is split into three bf16 parts (split3) and a product is the
// six largest of the nine part products, summed in fp32, smallest first: every
// bit of the inputs is used, and the three left out (middle by low and low by
// low) come to at most 2^-24 of a product, 2^-27.5 rms.  The bf16 products' own additions
// do not round to nearest: summed through all rows, 2.45M of them gave 4.5
// times the fp32 products' error; so 32 rows are summed by themselves and
// added to the running sum with an ordinary fma, the sign of A's rows changed
// from one 32 to the next, which cancels what is left of that bias (1.7e-6 to
// 3.3e-7 of the result).
//
// Workgroup = 2 x 4 waves, a (16*TM) x 256 block of C, one to a compute unit;
// 32 rows an iteration.  The rows' elements are split once per workgroup:
// waves w and w + 4 load rows 8w..8w+7 (a float of A and a float2 of B a row
// and thread), so that a thread holds 8 rows of its columns, the 16 bytes that
// a lane of the 16x16x32 product takes, and writes the parts to LDS as
// [part][8-row group][position][8 rows].  The position of B's column 2c + e is
// 128e + c, so that lanes write and read 16 consecutive bytes each, and a wave
// takes four of B's tiles that are pairs of columns of the result.  LDS holds
// two steps.  Waves w and w + 4 share a SIMD: the first stages the next step
// and then multiplies this one, the other multiplies first, so that the vector
// and the matrix pipe run side by side (509 us for 233k x 602 x 256 with two
// workgroups of 4 waves a compute unit and one step each in LDS).
//
// Infinities and NaN do not survive a split (and a sum near the largest float
// may overflow in parts only): a workgroup whose sums are not all finite, or
// with elements too small to split that count, forms its block again with fp32
// products.
//
// CT > 0 is the GCN relu-gradient form: B holds H (the relu output of the
// layer, [K x N]) and the B operand is formed while it is staged as
// (G W2^T) (.) [H > 0] from G [K x C] and W2 [N x C] (C <= CT), while H^T G
// is summed beside it into partial2 -- the layer-1 weight gradient and the
// layer-2 weight gradient of a two-layer GCN in one pass over its rows.
//
// 233k x 602 x 256: 0.43 ms (0.89 with fp32 products, in 3 turns of one
// workgroup a compute unit), 1.1 PFLOP/s of bf16 part products, the rate of a
// large bf16 matrix product here; 2.45M x 100 x 256: 0.87 ms (1.07), with the
// relu gradient of 2 classes 0.97 ms (1.28).  Error against 64 bits 2.4e-7,
// 3.3e-7 and 3.3e-7 of the result (8.6e-7, 1.3e-6 and 8.7e-7).
template <int TM, int CT, bool VB>
__global__ void __launch_bounds__(512) tn_split_kernel(TnArgs a) {
    constexpr std::uint32_t BM = 16 * TM, BN = 256;
    constexpr int TW = (TM + 1) / 2;  // tiles along M of the first four waves; TM / 2 of the others
    constexpr int GC = CT > 0 ? CT : 1;
    constexpr std::uint32_t kPartA = 4 * BM, kPartB = 4 * BN;  // 16-byte units of one part
    constexpr std::uint32_t kStage = 3 * (kPartA + kPartB);
    extern __shared__ uint4 parts[];  // [2 steps]: A's three parts, then B's
    const unsigned lane = __lane_id();
    const unsigned wave = tn_uniform(threadIdx.x / kWave);
    const unsigned wm = wave >> 2, wn = wave & 3u;  // wn: also the 8 rows that it stages
    const unsigned li = lane & 15u, lk = lane >> 4;
    // The blocks of one split read the same rows: splits go around in eights,
    // so that those blocks meet in one XCD's L2.
    const std::uint32_t blocks = a.blocksM * a.blocksN;
    const std::uint32_t g8 = blockIdx.x / (8 * blocks), in8 = blockIdx.x - g8 * 8 * blocks;
    const std::uint32_t n8 = min(8u, a.splits - 8 * g8);
    const std::uint32_t split = 8 * g8 + in8 % n8, block = in8 / n8;
    const std::uint32_t cbm = block % a.blocksM, cbn = block / a.blocksM;
    const std::uint32_t m0 = cbm * BM, n0 = cbn * BN;
    const std::uint32_t k0 = split * a.rowsPerSplit;
    const std::uint32_t k1 = min(a.K, k0 + a.rowsPerSplit);

    // This thread's columns (clamped: what they feed past M and N is not stored).
    const unsigned at = 64 * wm + lane;  // A's column, B's pair of columns
    const std::uint32_t colA = min(m0 + at, a.M - 1);
    std::uint32_t colB[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) colB[e] = VB ? min(n0 + 2 * at, a.N - 2) + e : min(n0 + 2 * at + e, a.N - 1);
    float w2[2][GC], dw2[2][GC];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int j = 0; j < GC; ++j) {
            dw2[e][j] = 0.0f;
            w2[e][j] = CT > 0 && static_cast<std::uint32_t>(j) < a.C
                           ? a.W2[static_cast<std::uint64_t>(colB[e]) * a.C + j] : 0.0f;
        }
    // largest and smallest nonzero magnitudes of the columns, and of G
    float maxA = 0.0f, maxB[2] = {0.0f, 0.0f}, maxG = 0.0f;
    std::uint32_t lowA = ~0u, lowB[2] = {~0u, ~0u};

    f32x4 acc[TW][4];
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // G's rows, of the relu-gradient form: lane CT r + j holds G(row r, j), read
    // back lane by lane.
    float xa[8], xb[8][2], xg = 0.0f;
    const std::uint32_t gr = CT > 0 ? lane / GC % 8 : 0u, gj = CT > 0 ? lane % GC : 0u;
    auto load = [&](std::uint32_t k) {  // rows k + 8 wn ..+7, the last row again past k1
#pragma unroll
        for (std::uint32_t r = 0; r < 8; ++r) {
            const std::uint64_t row = min(k + 8 * wn + r, k1 - 1);
            const float* rb = a.B + row * a.ldb;
            if constexpr (VB) {
                const float2 v = *reinterpret_cast<const float2*>(rb + colB[0]);
                xb[r][0] = v.x, xb[r][1] = v.y;
            } else {
#pragma unroll
                for (int e = 0; e < 2; ++e) xb[r][e] = rb[colB[e]];
            }
            xa[r] = a.A[row * a.lda + colA];
        }
        if constexpr (CT > 0) {
            const std::uint32_t row = k + 8 * wn + gr;
            xg = a.G[static_cast<std::uint64_t>(min(row, k1 - 1)) * a.ldg + min(gj, a.C - 1)];
        }
    };
    auto put = [&](uint4* to, std::uint32_t part, const float (&x)[8], std::uint32_t& low) {
        std::uint32_t h[4], m[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            split3(x[2 * q], x[2 * q + 1], h[q], m[q], l[q]);
            low = min(low, min(smallness(x[2 * q]), smallness(x[2 * q + 1])));
        }
        to[0] = make_uint4(h[0], h[1], h[2], h[3]);
        to[part] = make_uint4(m[0], m[1], m[2], m[3]);
        to[2 * part] = make_uint4(l[0], l[1], l[2], l[3]);
    };
    auto stage = [&](uint4* to, std::uint32_t k, float sign) {
        // Rows past the split's last (its row again) count zero times, by
        // their factor of A: what 0 makes of an infinity is summed again.
        float f[8];
#pragma unroll
        for (std::uint32_t r = 0; r < 8; ++r) f[r] = k + 8 * wn + r < k1 ? sign : 0.0f;
        const float gl = k + 8 * wn + gr < k1 && gj < a.C ? xg : 0.0f;
        if constexpr (CT > 0) maxG = fmaxf(maxG, fabsf(gl));
        if (BM == 128 || at < BM) {
            float x[8];
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                x[r] = f[r] * xa[r];
                if constexpr (CT > 0) maxA = fmaxf(maxA, fabsf(x[r]));
            }
            put(to + wn * BM + at, kPartA, x, lowA);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float x[8];
            float part[GC];  // of dW2, these 8 rows
#pragma unroll
            for (int j = 0; j < GC; ++j) part[j] = 0.0f;
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                x[r] = xb[r][e];
                if constexpr (CT > 0) {
                    if (k + 8 * wn + r >= k1) x[r] = 0.0f;
                    // dOut1 = (G W2^T) (.) [H > 0]; dW2 += H^T G
                    float d = 0.0f;
#pragma unroll
                    for (int j = 0; j < GC; ++j) {
                        const float g = __uint_as_float(static_cast<std::uint32_t>(
                            __builtin_amdgcn_readlane(static_cast<int>(__float_as_uint(gl)), GC * r + j)));
                        d = fmaf(g, w2[e][j], d);
                        part[j] = fmaf(x[r], g, part[j]);
                    }
                    x[r] = x[r] > 0.0f ? d : 0.0f;
                }
            }
            if constexpr (CT > 0) {
#pragma unroll
                for (int j = 0; j < GC; ++j) dw2[e][j] += part[j];
            }
            put(to + 3 * kPartA + wn * BN + 128 * e + at, kPartB, x, lowB[e]);
        }
    };
    // B's tile u of this wave: positions 128 (u / 2) + 32 wn + 16 (u % 2) + l%16.
    auto multiply = [&](const uint4* from, float sign) {
        bf16x8 b[4][3];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int s = 0; s < 3; ++s)
                b[u][s] = __builtin_bit_cast(
                    bf16x8, from[3 * kPartA + s * kPartB + lk * BN + 128 * (u / 2) + 32 * wn + 16 * (u % 2) + li]);
#pragma unroll
        for (int t = 0; t < TW; ++t) {
            if (TM % 2 != 0 && t == TW - 1 && wm != 0) break;
            bf16x8 x[3];
#pragma unroll
            for (int s = 0; s < 3; ++s)
                x[s] = __builtin_bit_cast(bf16x8, from[s * kPartA + lk * BM + 16 * (TW * wm + t) + li]);
            constexpr int kX[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};
            f32x4 sum[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) sum[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    sum[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[kX[s]], b[u][kB[s]], sum[u], 0, 0, 0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[t][u][v] = fmaf(sign, sum[u][v], acc[t][u][v]);
        }
    };

    load(k0);
    float sign = 1.0f;
    stage(parts, k0, sign);
    load(k0 + 32);
    __syncthreads();
    std::uint32_t cur = 0;
    for (std::uint32_t k = k0; k < k1; k += 32, sign = -sign, cur = kStage - cur) {
        if (wm != 0) multiply(parts + cur, sign);
        __builtin_amdgcn_sched_barrier(0);
        // past the last row too (zeros, and its row again): under a branch the
        // loaded registers would be copied, and waited for, where it ends
        stage(parts + (kStage - cur), k + 32, -sign);
        load(k + 64);
        __builtin_amdgcn_sched_barrier(0);
        if (wm == 0) multiply(parts + cur, sign);
        __syncthreads();
    }

    // Row r of tile t is column m of A, tile u's lane column n(u) of B.
    const auto mcol = [&](int t, unsigned r) { return m0 + 16 * (TW * wm + t) + r; };
    const auto ncol = [&](int u) { return n0 + 2 * (32 * wn + 16 * (u % 2) + li) + u / 2; };
    const int tiles = wm == 0 ? TW : TM / 2;

    bool redo = k1 - k0 < kSplitMinTerms;
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) redo |= !(fabsf(acc[t][u][v]) <= 0x1.fffffep127f);
    const bool tinyA = lowA < kSplitExactBits, tinyB[2] = {lowB[0] < kSplitExactBits, lowB[1] < kSplitExactBits};
    const bool tiny = tinyA || tinyB[0] || tinyB[1];
    const bool look = __syncthreads_or(redo || tiny) != 0;
    if (look && __syncthreads_or(tiny)) {
        // the columns' maxima and losses, of the four waves' rows: [4][BM] and
        // [4][BN] of each
        float* const topA = reinterpret_cast<float*>(parts);
        float* const lossA = topA + 4 * BM;
        float* const topB = lossA + 4 * BM;
        float* const lossB = topB + 4 * BN;
        const float loss = split_loss(k1 - k0);
        if constexpr (CT == 0) {  // the maxima, here alone: the products' loop is full without them
            for (std::uint32_t k = k0; k < k1; k += 32) {
                load(k);
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    maxA = fmaxf(maxA, fabsf(xa[r]));
                    maxB[0] = fmaxf(maxB[0], fabsf(xb[r][0]));
                    maxB[1] = fmaxf(maxB[1], fabsf(xb[r][1]));
                }
            }
        } else {  // small elements of G W2^T are common (confident predictions): bounded by G's
#pragma unroll
            for (int d = GC; d < 64; d *= 2) maxG = fmaxf(maxG, __shfl_xor(maxG, d));
#pragma unroll
            for (int j = 0; j < GC; ++j) {
                const float g = __shfl(maxG, j);
                maxB[0] = fmaf(g, fabsf(w2[0][j]), maxB[0]);
                maxB[1] = fmaf(g, fabsf(w2[1][j]), maxB[1]);
            }
        }
        if (at < BM) {
            topA[wn * BM + at] = maxA;
            lossA[wn * BM + at] = tinyA ? loss : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            topB[wn * BN + 2 * at + e] = maxB[e];
            lossB[wn * BN + 2 * at + e] = tinyB[e] ? loss : 0.0f;
        }
        __syncthreads();
        const auto most = [](const float* x, std::uint32_t i, std::uint32_t n) {
            return fmaxf(fmaxf(x[i], x[n + i]), fmaxf(x[2 * n + i], x[3 * n + i]));
        };
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if (t >= tiles) continue;
                const std::uint32_t m = mcol(t, 4 * lk + v) - m0;
                const float am = most(topA, m, BM), al = most(lossA, m, BM);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const std::uint32_t n = ncol(u) - n0;
                    redo |= !(fabsf(acc[t][u][v]) >= al * most(topB, n, BN) + am * most(lossB, n, BN));
                }
            }
    }
    if (look && __syncthreads_or(redo)) {
#pragma unroll
        for (int t = 0; t < TW; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[t][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // 16 rows at a time, all loads before the products.  Every block formed
        // again (all of G small), a 4-row step after the other : so, us: the relu
        // gradient of 9,041 x 43 x 256 with 8 classes 160 : 51, of 2.45M x 100 x
        // 256 with 2 10,630 : 2,700; A^T B there 5,120 : 3,000.
        constexpr int kSteps = 4;
        std::uint32_t cm[TW], cn[4];
        float wr[4][GC];
#pragma unroll
        for (int t = 0; t < TW; ++t) cm[t] = min(mcol(t, li), a.M - 1);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            cn[u] = min(ncol(u), a.N - 1);
#pragma unroll
            for (int j = 0; j < GC; ++j)
                wr[u][j] = CT > 0 && static_cast<std::uint32_t>(j) < a.C
                               ? a.W2[static_cast<std::uint64_t>(cn[u]) * a.C + j] : 0.0f;
        }
        for (std::uint32_t k = k0; k < k1; k += 4 * kSteps) {
            float x[kSteps][TW], y[kSteps][4], g[kSteps][GC];
#pragma unroll
            for (std::uint32_t s = 0; s < kSteps; ++s) {
                const std::uint64_t row = min(k + 4 * s + lk, k1 - 1);
#pragma unroll
                for (int u = 0; u < 4; ++u) y[s][u] = a.B[row * a.ldb + cn[u]];
#pragma unroll
                for (int t = 0; t < TW; ++t) x[s][t] = a.A[row * a.lda + cm[t]];
#pragma unroll
                for (int j = 0; j < GC; ++j)
                    g[s][j] = CT > 0 && static_cast<std::uint32_t>(j) < a.C ? a.G[row * a.ldg + j] : 0.0f;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (std::uint32_t s = 0; s < kSteps; ++s) {
                const bool in = k + 4 * s + lk < k1;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if constexpr (CT > 0) {
                        float d = 0.0f;
#pragma unroll
                        for (int j = 0; j < GC; ++j) d = fmaf(g[s][j], wr[u][j], d);
                        y[s][u] = y[s][u] > 0.0f ? d : 0.0f;
                    }
                    y[s][u] = in ? y[s][u] : 0.0f;
                }
#pragma unroll
                for (int t = 0; t < TW; ++t) {
                    const float xt = in ? x[s][t] : 0.0f;
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(xt, y[s][u], acc[t][u], 0, 0, 0);
                }
            }
        }
    }

    // Tile (t, u): accumulator v of lane l is C(mcol(t, 4*(l/16) + v), ncol(u)).
    float* out = a.partial + static_cast<std::uint64_t>(split) * a.M * a.N;
    const bool vec = a.N % 2 == 0 && (reinterpret_cast<std::uintptr_t>(a.partial) & 7u) == 0;
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const std::uint32_t m = mcol(t, 4 * lk + v);
            if (t >= tiles || m >= a.M) continue;
            float* o = out + static_cast<std::uint64_t>(m) * a.N;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const std::uint32_t n = ncol(u);
                if (vec) {
                    if (n < a.N) *reinterpret_cast<float2*>(o + n) = make_float2(acc[t][u][v], acc[t][u + 2][v]);
                } else {
                    if (n < a.N) o[n] = acc[t][u][v];
                    if (n + 1 < a.N) o[n + 1] = acc[t][u + 2][v];
                }
            }
        }
    if constexpr (CT > 0) {
        // H^T G of this split: a column's four groups of rows, added in order;
        // the first block row of C writes it.
        if (cbm != 0) return;
        float* part = reinterpret_cast<float*>(parts);  // [4][256][CT]
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int j = 0; j < GC; ++j) part[(wn * 256 + 2 * at + e) * GC + j] = dw2[e][j];
        __syncthreads();
        float* out2 = a.partial2 + static_cast<std::uint64_t>(split) * a.N * a.C;
        const std::uint32_t c = n0 + threadIdx.x;
        if (threadIdx.x >= 256 || c >= a.N) return;
        for (std::uint32_t j = 0; j < a.C; ++j) {
            float v = 0.0f;
#pragma unroll
            for (int w = 0; w < 4; ++w) v += part[(w * 256 + threadIdx.x) * GC + j];
            out2[static_cast<std::uint64_t>(c) * a.C + j] = v;
        }
    }
}

// ---------------------------------------------------------------- forward
// H = relu(AX W1) [K x Hd] and XW = H W2 [K x C] in one pass over the rows
// of AX (the first layer's transform, its activation and the second layer's
// transform of a two-layer GCN; tcgnn_conv_release.py:134 and :243-247).
//
// fp32 MFMA held this at 1.40 ms for 2.45M x 100 x 256; as tn_split_kernel, the
// operands are three bf16 parts each (split3) and a product is six part
// products: 1.03 ms, against 0.74 for AX and H at the rate of a large copy
// (200k rows 162 -> 102 us, 2000 rows 37 -> 13).  H's error against 64 bits
// 1.8e-7 -> 5.5e-8 of it.
//
// Workgroup = 8 waves, one to a compute unit, persistent over steps of 64 rows.
// Wave w holds the parts of W1's columns 32w .. 32w+31 in registers (first
// operand: lane l%16 is the hidden unit, 8 inputs from 8 (l/16) + 32 ks on),
// split once.  A step's rows are split once per workgroup: thread t takes
// inputs 8 (t%16) ..+7 of rows t/16 and t/16 + 32, and writes their parts to
// LDS as [part][8 inputs][row], 65 rows apart so that the 16 threads of a row
// meet different banks.  LDS holds two steps, and of the two waves of a SIMD one
// stages the next step first and the other multiplies first.  A lane ends with 4
// consecutive hidden units of a row: relu, a float4 store of H, and the sum over
// a wave's units, by lane and then over the waves through LDS, for H W2.
//
// A wave whose sums are not all finite forms its block with fp32 products, and
// so does one where elements too small to split count (a step or a part of W1
// that holds such an element is looked at closer).
struct ReluFwdArgs {
    const float* AX;
    const float* W1;  // [F x Hd]
    const float* W2;  // [Hd x C]
    float* H;
    float* XW;
    std::uint32_t ldax, ldh, ldxw;
    std::uint32_t K, F, Hd, C;
    std::uint32_t steps;  // ceil(K / 64)
    int vecH;             // H rows allow float4 stores
};

template <int KS, int CT, bool VEC>
__global__ void __launch_bounds__(512) gcn_relu_forward_kernel(ReluFwdArgs a) {
    constexpr std::uint32_t kPitch = 65;                      // rows of a group of inputs, in 16 bytes
    constexpr std::uint32_t kPart = 4 * KS * kPitch, kStage = 3 * kPart;
    extern __shared__ uint4 parts[];                          // [2 steps][3 parts][4 KS groups][65]
    __shared__ float red[2][8][64][CT];                       // a step's H W2, by wave
    __shared__ std::uint32_t small[2];                        // 1 + the last step with an element too small to split
    // largest magnitude of W1's columns and of a step's rows (where either
    // holds one), negative with elements too small to split
    __shared__ float rowTop[2][64], colTop[256];
    const unsigned lane = __lane_id();
    const unsigned li = lane & 15u, lk = lane >> 4;
    const unsigned wave = tn_uniform(threadIdx.x / kWave);
    const bool first = wave < 4;  // waves w and w + 4 share a SIMD

    // The wave's part of W1 and this lane's of W2.
    bf16x8 w[2][KS][3];
    bool smallW = false;  // an element of the wave's part
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const std::uint32_t n = 32 * wave + 16 * u + li;
        float top = 0.0f;
        std::uint32_t low = ~0u;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            std::uint32_t part[3][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float x[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const std::uint32_t k = 32 * ks + 8 * lk + 2 * q + e;
                    x[e] = n < a.Hd && k < a.F ? a.W1[static_cast<std::uint64_t>(k) * a.Hd + n] : 0.0f;
                    top = fmaxf(top, fabsf(x[e]));
                    low = min(low, smallness(x[e]));
                }
                split3(x[0], x[1], part[0][q], part[1][q], part[2][q]);
            }
#pragma unroll
            for (int s = 0; s < 3; ++s)
                w[u][ks][s] = __builtin_bit_cast(bf16x8, make_uint4(part[s][0], part[s][1], part[s][2], part[s][3]));
        }
        top = fmaxf(top, __shfl_xor(top, 16));
        top = fmaxf(top, __shfl_xor(top, 32));
        const std::uint64_t tiny = __ballot(low < kSplitExactBits);
        smallW |= tiny != 0;
        if (lk == 0) colTop[32 * wave + 16 * u + li] = ((tiny >> li) & 0x0001000100010001ull) != 0 ? -top : top;
    }
    float w2[2][4][CT];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const std::uint32_t n = 32 * wave + 16 * u + 4 * lk + v;
#pragma unroll
            for (int j = 0; j < CT; ++j)
                w2[u][v][j] = n < a.Hd && static_cast<std::uint32_t>(j) < a.C
                                  ? a.W2[static_cast<std::uint64_t>(n) * a.C + j] : 0.0f;
        }

    if (threadIdx.x < 2) small[threadIdx.x] = 0;
    const bool colsToo = __syncthreads_or(smallW) != 0;  // any wave's

    // This thread's inputs (clamped loads, zeros past F when staged).
    const std::uint32_t kg = threadIdx.x & 15u, row0 = threadIdx.x >> 4;
    const bool mine = kg < 4 * KS;
    float x[2][8];
    auto load = [&](std::uint32_t step) {
#pragma unroll
        for (std::uint32_t h = 0; h < 2; ++h) {
            const std::uint64_t at = static_cast<std::uint64_t>(step) * 64 + row0 + 32 * h;
            const float* r = a.AX + (at < a.K ? at : a.K - 1) * a.ldax;
            if constexpr (VEC) {
#pragma unroll
                for (std::uint32_t q = 0; q < 2; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(r + min(8 * kg + 4 * q, a.F - 4));
                    x[h][4 * q] = v.x, x[h][4 * q + 1] = v.y, x[h][4 * q + 2] = v.z, x[h][4 * q + 3] = v.w;
                }
            } else {
#pragma unroll
                for (std::uint32_t e = 0; e < 8; ++e) x[h][e] = r[min(8 * kg + e, a.F - 1)];
            }
        }
    };
    auto stage = [&](std::uint32_t step, unsigned buf) {
        uint4* const to = parts + buf * kStage;
#pragma unroll
        for (std::uint32_t h = 0; h < 2; ++h) {
            std::uint32_t hi[4], mid[4], lo[4], low = ~0u;
#pragma unroll
            for (std::uint32_t q = 0; q < 4; ++q) {
                const float p = 8 * kg + 2 * q < a.F ? x[h][2 * q] : 0.0f;
                const float r = 8 * kg + 2 * q + 1 < a.F ? x[h][2 * q + 1] : 0.0f;
                low = min(low, min(smallness(p), smallness(r)));
                split3(p, r, hi[q], mid[q], lo[q]);
            }
            if (mine) {
                uint4* const at = to + kg * kPitch + row0 + 32 * h;
                at[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
                at[kPart] = make_uint4(mid[0], mid[1], mid[2], mid[3]);
                at[2 * kPart] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
            }
            const std::uint64_t tiny = __ballot(low < kSplitExactBits);
            if (tiny) small[buf] = step + 1;
            float top = 0.0f;
            if (tiny || colsToo) {
#pragma unroll
                for (std::uint32_t e = 0; e < 8; ++e)
                    if (8 * kg + e < a.F) top = fmaxf(top, fabsf(x[h][e]));
#pragma unroll
                for (unsigned d = 1; d < 16; d *= 2) top = fmaxf(top, __shfl_xor(top, d));
            }
            if (kg == 0) rowTop[buf][row0 + 32 * h] = (tiny >> (lane & 48u) & 0xFFFFull) != 0 ? -top : top;
        }
    };
    auto multiply = [&](std::uint32_t step, unsigned buf) {
        const uint4* const from = parts + buf * kStage;
        const bool look = smallW || small[buf] == step + 1;
#pragma unroll
        for (std::uint32_t rt = 0; rt < 4; ++rt) {
            f32x4 acc[2] = {f32x4{0.0f, 0.0f, 0.0f, 0.0f}, f32x4{0.0f, 0.0f, 0.0f, 0.0f}};
            constexpr int kW[6] = {2, 0, 1, 1, 0, 0}, kX[6] = {0, 2, 1, 0, 1, 0};
            bf16x8 b[KS][3];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    b[ks][s] = __builtin_bit_cast(bf16x8, from[s * kPart + (4 * ks + lk) * kPitch + 16 * rt + li]);
            // the smallest part products of all inputs first
#pragma unroll
            for (int s = 0; s < 6; ++s)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][ks][kW[s]], b[ks][kX[s]], acc[u], 0, 0, 0);
            bool redo = a.F < kSplitMinTerms;
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int v = 0; v < 4; ++v) redo |= !(fabsf(acc[u][v]) <= 0x1.fffffep127f);
            if (look) {
                const float loss = split_loss(a.F), r = rowTop[buf][16 * rt + li];
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float c = colTop[32 * wave + 16 * u + 4 * lk + v];
                        redo |= !(fabsf(acc[u][v]) >= loss * ((r < 0.0f ? fabsf(c) : 0.0f) + (c < 0.0f ? fabsf(r) : 0.0f)));
                    }
            }
            const std::uint64_t row = static_cast<std::uint64_t>(step) * 64 + 16 * rt + li;
            if (__ballot(redo)) {
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                const float* r = a.AX + (row < a.K ? row : a.K - 1) * a.ldax;
                for (std::uint32_t k = 0; k < a.F; k += 4) {
                    const std::uint32_t kk = k + lk;
                    const float xv = kk < a.F ? r[kk] : 0.0f;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const std::uint32_t n = 32 * wave + 16 * u + li;
                        const float wv = kk < a.F && n < a.Hd ? a.W1[static_cast<std::uint64_t>(kk) * a.Hd + n] : 0.0f;
                        acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, xv, acc[u], 0, 0, 0);
                    }
                }
            }
            // Lane holds H(row, 32 wave + 16 u + 4 lk + v): relu (NaN kept, as clamp_min).
            float xw[CT];
#pragma unroll
            for (int j = 0; j < CT; ++j) xw[j] = 0.0f;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                float h[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    // units past Hd are 0 times the row: NaN for an infinity
                    h[v] = acc[u][v] < 0.0f || 32 * wave + 16 * u + 4 * lk + v >= a.Hd ? 0.0f : acc[u][v];
#pragma unroll
                    for (int j = 0; j < CT; ++j) xw[j] = fmaf(h[v], w2[u][v][j], xw[j]);
                }
                const std::uint32_t n = 32 * wave + 16 * u + 4 * lk;
                float* o = a.H + row * a.ldh + n;
                if (row < a.K && a.vecH) {
                    if (n < a.Hd) *reinterpret_cast<float4*>(o) = make_float4(h[0], h[1], h[2], h[3]);
                } else if (row < a.K) {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < a.Hd) o[v] = h[v];
                }
            }
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                xw[j] += __shfl_xor(xw[j], 16);
                xw[j] += __shfl_xor(xw[j], 32);
                if (lk == 0) red[buf][wave][16 * rt + li][j] = xw[j];
            }
        }
    };

    std::uint32_t step = blockIdx.x;
    load(step);
    stage(step, 0);
    load(step + gridDim.x);  // past the last: the last row again
    __syncthreads();
    for (unsigned buf = 0; step < a.steps; step += gridDim.x, buf ^= 1u) {
        if (!first) multiply(step, buf);
        __builtin_amdgcn_sched_barrier(0);
        stage(step + gridDim.x, buf ^ 1u);
        load(step + 2 * gridDim.x);
        __builtin_amdgcn_sched_barrier(0);
        if (first) multiply(step, buf);
        __syncthreads();
        // this step's H W2, its waves' sums in order; the next step's go to the
        // other half of `red`
        if (threadIdx.x < 64 * CT) {
            const std::uint32_t r = threadIdx.x / CT, j = threadIdx.x % CT;
            const std::uint64_t row = static_cast<std::uint64_t>(step) * 64 + r;
            float t = 0.0f;
#pragma unroll
            for (int v = 0; v < 8; ++v) t += red[buf][v][r][j];
            if (row < a.K && j < a.C) a.XW[row * a.ldxw + j] = t;
        }
    }
}

template <int KS, int CT>
void relu_forward_launch(const ReluFwdArgs& a, hipStream_t st) {
    constexpr std::uint32_t lds = 2 * 3 * 4 * KS * 65 * 16;
    const bool vec = a.F % 4 == 0 && a.ldax % 4 == 0 && reinterpret_cast<std::uintptr_t>(a.AX) % 16 == 0;
    const dim3 grid(std::max<std::uint32_t>(1, std::min<std::uint32_t>(device_cus(), a.steps)));
    if (vec) hipLaunchKernelGGL((gcn_relu_forward_kernel<KS, CT, true>), grid, dim3(512), lds, st, a);
    else hipLaunchKernelGGL((gcn_relu_forward_kernel<KS, CT, false>), grid, dim3(512), lds, st, a);
}

// C[m][n] (=|+=) sum over splits of partial[s][m][n], splits added in a fixed
// order: 16 elements per workgroup, 16 interleaved groups of splits summed
// per thread, then the 16 group sums in order.
// With `transposed` the partials hold C^T (an M x N block of C^T is C's
// N x M block): element (m, n) of the partials goes to C[n][m].
__global__ void __launch_bounds__(256) tn_reduce_kernel(const float* __restrict__ partial, std::uint32_t splits,
                                                        std::uint32_t M, std::uint32_t N, float* __restrict__ C,
                                                        std::uint32_t ldc, int accumulate, int transposed) {
    __shared__ float part[16][17];
    const std::uint64_t MN = static_cast<std::uint64_t>(M) * N;
    const unsigned col = threadIdx.x & 15u, grp = threadIdx.x >> 4;
    const std::uint64_t e = static_cast<std::uint64_t>(blockIdx.x) * 16 + col;
    float s = 0.0f;
    if (e < MN)
        for (std::uint32_t sp = grp; sp < splits; sp += 16) s += partial[sp * MN + e];
    part[grp][col] = s;
    __syncthreads();
    if (threadIdx.x < 16 && e < MN) {
        float t = 0.0f;
#pragma unroll
        for (int g = 0; g < 16; ++g) t += part[g][col];
        const std::uint32_t m = static_cast<std::uint32_t>(e / N), n = static_cast<std::uint32_t>(e % N);
        float* c = transposed ? C + static_cast<std::uint64_t>(n) * ldc + m : C + static_cast<std::uint64_t>(m) * ldc + n;
        *c = accumulate ? *c + t : t;
    }
}

// Shapes by output shape:
//  - anything wide: tn_split_kernel, TM = 4, 7 or 8 tiles along M, the fewest
//    that cover M, so that a 100-wide layer does not multiply 128 columns;
//  - N <= 16 (a class-width gradient): 4 waves along M with 4 x 1 tiles,
//    eight workgroups per CU for memory parallelism (~5 TB/s for 256x2);
//    M <= 16 the same along N.
enum class TnShape { Wide4, Wide7, Wide8, NarrowN, NarrowM };

struct TnPlan {
    TnShape shape;
    std::uint32_t step;  // rows per iteration (4*U)
    std::uint32_t BM, BN;
    std::uint32_t blocksM, blocksN;
    std::uint32_t splits, rowsPerSplit;
};

// Shape chosen from (M, N); block counts from (realM, realN) when given.
TnPlan tn_plan(std::uint32_t K, std::uint32_t M, std::uint32_t N, std::uint32_t realM = 0, std::uint32_t realN = 0,
               std::uint64_t splitCap = 0) {
    TnPlan p{};
    if (N <= 16) {
        p.shape = TnShape::NarrowN;  // TM=4, TN=1, WM=4, WN=1, U=8
        p.step = 32, p.BM = 256, p.BN = 16;
    } else if (M <= 16) {
        p.shape = TnShape::NarrowM;  // TM=1, TN=4, WM=1, WN=4, U=8
        p.step = 32, p.BM = 16, p.BN = 256;
    } else {
        p.shape = M <= 64 ? TnShape::Wide4 : M <= 112 ? TnShape::Wide7 : TnShape::Wide8;
        p.step = 32, p.BN = 256;
        p.BM = p.shape == TnShape::Wide4 ? 64 : p.shape == TnShape::Wide7 ? 112 : 128;
    }
    if (realM != 0) M = realM;
    if (realN != 0) N = realN;
    p.blocksM = (M + p.BM - 1) / p.BM;
    p.blocksN = (N + p.BN - 1) / p.BN;
    const std::uint64_t blocks = static_cast<std::uint64_t>(p.blocksM) * p.blocksN;
    // One (Wide*: what fits, so that none is left for a second turn) or about
    // eight workgroups per compute unit in all.
    const bool narrow = p.shape == TnShape::NarrowN || p.shape == TnShape::NarrowM;
    const std::uint64_t target = static_cast<std::uint64_t>(device_cus()) * (narrow ? 8 : 1);
    const std::uint64_t maxSplits = std::max<std::uint64_t>(1, (K + p.step - 1) / p.step);
    std::uint64_t splits = std::min<std::uint64_t>(maxSplits, std::max<std::uint64_t>(1, (target + (narrow ? blocks - 1 : 0)) / blocks));
    if (splitCap != 0) splits = std::min(splits, splitCap);
    std::uint64_t rps = (K + splits - 1) / splits;
    rps = std::max<std::uint64_t>(p.step, (rps + p.step - 1) / p.step * p.step);
    splits = std::max<std::uint64_t>(1, (K + rps - 1) / rps);
    p.splits = static_cast<std::uint32_t>(splits);
    p.rowsPerSplit = static_cast<std::uint32_t>(rps);
    return p;
}

// C = A^T B or, when N is the narrow side of a wide product (17..128 and
// below M), C^T = B^T A: the wide tiles lay 4 waves of 64 columns along N,
// so a narrow N would leave waves multiplying padding (602 x 64 ran at 10 ms
// as C, 2.5x torch.mm).
inline bool tn_swapped(std::uint32_t M, std::uint32_t N) { return M > 16 && N > 16 && N <= 128 && N < M; }

template <int TM, int TN, int WM, int WN, int U>
void tn_launch(const TnArgs& a, const TnPlan& p, hipStream_t st) {
    hipLaunchKernelGGL((tn_partial_kernel<TM, TN, WM, WN, U>), dim3(p.splits, p.blocksM * p.blocksN),
                       dim3(kWave * WM * WN), 0, st, a);
}

// Pairs of B's columns in one load a row where they allow it.
template <int TM, int CT>
void tn_split_launch(const TnArgs& a, const TnPlan& p, hipStream_t st) {
    const bool vb = a.N % 2 == 0 && a.ldb % 2 == 0 && reinterpret_cast<std::uintptr_t>(a.B) % 8 == 0;
    const dim3 grid(p.splits * p.blocksM * p.blocksN);
    constexpr std::uint32_t lds = 2 * 3 * 4 * 16 * (16 * TM + 256);
    if (vb) hipLaunchKernelGGL((tn_split_kernel<TM, CT, true>), grid, dim3(512), lds, st, a);
    else hipLaunchKernelGGL((tn_split_kernel<TM, CT, false>), grid, dim3(512), lds, st, a);
}

// The relu-gradient form always takes the wide shapes (N is the hidden width).
TnPlan relu_grad_plan(std::uint32_t K, std::uint32_t F, std::uint32_t Hd) {
    return tn_plan(K, std::max<std::uint32_t>(F, 17), std::max<std::uint32_t>(Hd, 17), F, Hd);
}

}  // namespace
}  // namespace tcc

using namespace tcc;

extern "C" {

size_t tcc_dense_tn_workspace_bytes(std::uint32_t K, std::uint32_t M, std::uint32_t N) {
    if (K == 0 || M == 0 || N == 0) return 0;
    const TnPlan p = tn_swapped(M, N) ? tn_plan(K, N, M) : tn_plan(K, M, N);
    return static_cast<size_t>(p.splits) * M * N * sizeof(float);
}

}  // extern "C"

namespace tcc {
namespace {

// C = A^T B (or +=) with the partial products in `workspace`; splitCap
// bounds the split of K (0 = none) so that the partials fit a fixed buffer.
int dense_tn_impl(const float* A, std::uint32_t lda, const float* B, std::uint32_t ldb, float* C, std::uint32_t ldc,
                  std::uint32_t K, std::uint32_t M, std::uint32_t N, int accumulate, void* workspace,
                  size_t workspaceBytes, std::uint64_t splitCapBytes, hipStream_t st) {
    TCC_REQUIRE(C && M >= 1 && N >= 1 && lda >= M && ldb >= N && ldc >= N, TCC_ERR_INVALID_ARGUMENT,
                "invalid dense A^T B arguments");
    TCC_REQUIRE(lda < (1u << 28) && ldb < (1u << 28) && ldc < (1u << 28), TCC_ERR_UNSUPPORTED,
                "dense A^T B row strides must be below 2^28");
    if (K == 0) {
        if (accumulate) return TCC_OK;
        for (std::uint32_t m = 0; m < M; ++m)  // C rows may be strided: clear row by row
            TCC_HIP_CHECK(fill<float>(C + static_cast<std::uint64_t>(m) * ldc, N, 0.0f, st));
        return TCC_OK;
    }
    TCC_REQUIRE(A && B && workspace, TCC_ERR_INVALID_ARGUMENT, "invalid dense A^T B arguments");
    const bool swapped = tn_swapped(M, N);
    if (swapped) {  // C^T = B^T A
        std::swap(A, B);
        std::swap(lda, ldb);
        std::swap(M, N);
    }
    const std::uint64_t splitBytes = static_cast<std::uint64_t>(M) * N * sizeof(float);
    const TnPlan p = tn_plan(K, M, N, 0, 0, splitCapBytes ? splitCapBytes / splitBytes : 0);
    TCC_REQUIRE(workspaceBytes >= static_cast<size_t>(p.splits) * M * N * sizeof(float), TCC_ERR_INVALID_ARGUMENT,
                "dense A^T B workspace too small (tcc_dense_tn_workspace_bytes)");
    TCC_REQUIRE(static_cast<std::uint64_t>(p.blocksM) * p.blocksN <= 65535, TCC_ERR_UNSUPPORTED,
                "dense A^T B output too large");
    TnArgs a{};
    a.A = A;
    a.B = B;
    a.partial = static_cast<float*>(workspace);
    a.lda = lda;
    a.ldb = ldb;
    a.K = K;
    a.M = M;
    a.N = N;
    a.rowsPerSplit = p.rowsPerSplit;
    a.blocksM = p.blocksM;
    a.blocksN = p.blocksN;
    a.splits = p.splits;
    switch (p.shape) {
        case TnShape::NarrowN: tn_launch<4, 1, 4, 1, 8>(a, p, st); break;
        case TnShape::NarrowM: tn_launch<1, 4, 1, 4, 8>(a, p, st); break;
        case TnShape::Wide4: tn_split_launch<4, 0>(a, p, st); break;
        case TnShape::Wide7: tn_split_launch<7, 0>(a, p, st); break;
        default: tn_split_launch<8, 0>(a, p, st); break;
    }
    TCC_LAUNCH_CHECK();
    const std::uint64_t MN = static_cast<std::uint64_t>(M) * N;
    hipLaunchKernelGGL(tn_reduce_kernel, dim3(grid_for(MN, 16)), dim3(256), 0, st,
                       static_cast<const float*>(workspace), p.splits, M, N, C, ldc, accumulate, swapped ? 1 : 0);
    TCC_LAUNCH_CHECK();
    return TCC_OK;
}

// Scratch of tcc_dense_tn_noalloc: the partial products, in device memory of
// the library's code object (one copy per GPU, held until the process ends).
constexpr std::size_t kTnScratchBytes = static_cast<std::size_t>(TCC_DENSE_TN_NOALLOC_SCRATCH_BYTES);
__device__ __align__(256) float tn_scratch[kTnScratchBytes / sizeof(float)];

// Device address of tn_scratch on the current device, looked up once per
// device (host code must not pass the symbol itself to a kernel: in host
// code it names a host-side stand-in).
int tn_scratch_address(float** out) {
    static std::mutex mu;
    static float* addr[64] = {};
    int dev = 0;
    TCC_HIP_CHECK(hipGetDevice(&dev));
    TCC_REQUIRE(dev >= 0 && dev < 64, TCC_ERR_UNSUPPORTED, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (addr[dev] == nullptr) {
        void* p = nullptr;
        TCC_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(tn_scratch)));
        TCC_REQUIRE(p != nullptr, TCC_ERR_HIP, "no device address for the dense A^T B scratch");
        addr[dev] = static_cast<float*>(p);
    }
    *out = addr[dev];
    return TCC_OK;
}

}  // namespace
}  // namespace tcc

extern "C" {

int tcc_dense_tn(const float* A, std::uint32_t lda, const float* B, std::uint32_t ldb, float* C, std::uint32_t ldc,
                 std::uint32_t K, std::uint32_t M, std::uint32_t N, int accumulate, void* workspace,
                 size_t workspaceBytes, void* stream) {
    clear_last_error();
    return dense_tn_impl(A, lda, B, ldb, C, ldc, K, M, N, accumulate, workspace, workspaceBytes, 0,
                         as_stream(stream));
}

int tcc_dense_tn_noalloc(const float* A, std::uint32_t lda, const float* B, std::uint32_t ldb, float* C,
                         std::uint32_t ldc, std::uint32_t K, std::uint32_t M, std::uint32_t N, int accumulate,
                         void* stream) {
    clear_last_error();
    TCC_REQUIRE(static_cast<std::uint64_t>(M) * N * sizeof(float) <= kTnScratchBytes, TCC_ERR_UNSUPPORTED,
                "dense A^T B without allocation: M x N above the 16 MiB scratch (4M floats)");
    float* scratch = nullptr;
    if (K > 0) {
        const int rc = tn_scratch_address(&scratch);
        if (rc) return rc;
    }
    return dense_tn_impl(A, lda, B, ldb, C, ldc, K, M, N, accumulate, scratch, kTnScratchBytes, kTnScratchBytes,
                         as_stream(stream));
}

int tcc_gcn_relu_forward(const float* AX, std::uint32_t ldax, const float* W1, const float* W2, float* H,
                         std::uint32_t ldh, float* XW, std::uint32_t ldxw, std::uint32_t K, std::uint32_t F,
                         std::uint32_t Hd, std::uint32_t C, void* stream) {
    clear_last_error();
    TCC_REQUIRE(W1 && W2 && H && XW && F >= 1 && Hd >= 1 && C >= 1 && ldax >= F && ldh >= Hd && ldxw >= C,
                TCC_ERR_INVALID_ARGUMENT, "invalid GCN relu-forward arguments");
    TCC_REQUIRE(F <= 128 && Hd <= 256 && C <= 4, TCC_ERR_UNSUPPORTED,
                "GCN relu-forward supports F <= 128, hidden <= 256 and at most 4 classes");
    if (K == 0) return TCC_OK;
    TCC_REQUIRE(AX != nullptr, TCC_ERR_INVALID_ARGUMENT, "invalid GCN relu-forward arguments");
    ReluFwdArgs a{};
    a.AX = AX;
    a.W1 = W1;
    a.W2 = W2;
    a.H = H;
    a.XW = XW;
    a.ldax = ldax;
    a.ldh = ldh;
    a.ldxw = ldxw;
    a.K = K;
    a.F = F;
    a.Hd = Hd;
    a.C = C;
    a.steps = static_cast<std::uint32_t>((static_cast<std::uint64_t>(K) + 63) / 64);
    a.vecH = Hd % 4 == 0 && ldh % 4 == 0 && reinterpret_cast<std::uintptr_t>(H) % 16 == 0;
    const hipStream_t st = as_stream(stream);
    const bool two = C <= 2;
    if (F <= 32) two ? relu_forward_launch<1, 2>(a, st) : relu_forward_launch<1, 4>(a, st);
    else if (F <= 64) two ? relu_forward_launch<2, 2>(a, st) : relu_forward_launch<2, 4>(a, st);
    else if (F <= 96) two ? relu_forward_launch<3, 2>(a, st) : relu_forward_launch<3, 4>(a, st);
    else two ? relu_forward_launch<4, 2>(a, st) : relu_forward_launch<4, 4>(a, st);
    TCC_LAUNCH_CHECK();
    return TCC_OK;
}

size_t tcc_gcn_relu_grad_workspace_bytes(std::uint32_t K, std::uint32_t F, std::uint32_t Hd, std::uint32_t C) {
    if (K == 0 || F == 0 || Hd == 0 || C == 0) return 0;
    const TnPlan p = relu_grad_plan(K, F, Hd);
    return static_cast<size_t>(p.splits) * (static_cast<size_t>(F) * Hd + static_cast<size_t>(Hd) * C) *
           sizeof(float);
}

int tcc_gcn_relu_grad(const float* AX, std::uint32_t ldax, const float* H, std::uint32_t ldh, const float* G,
                      std::uint32_t ldg, const float* W2, float* dW1, float* dW2, std::uint32_t K, std::uint32_t F,
                      std::uint32_t Hd, std::uint32_t C, void* workspace, size_t workspaceBytes, void* stream) {
    clear_last_error();
    TCC_REQUIRE(dW1 && dW2 && W2 && F >= 1 && Hd >= 1 && C >= 1 && ldax >= F && ldh >= Hd && ldg >= C,
                TCC_ERR_INVALID_ARGUMENT, "invalid GCN relu-gradient arguments");
    TCC_REQUIRE(C <= 8, TCC_ERR_UNSUPPORTED, "GCN relu-gradient supports at most 8 classes");
    TCC_REQUIRE(ldax < (1u << 28) && ldh < (1u << 28) && ldg < (1u << 28), TCC_ERR_UNSUPPORTED,
                "GCN relu-gradient row strides must be below 2^28");
    const hipStream_t st = as_stream(stream);
    if (K == 0) {
        TCC_HIP_CHECK(fill<float>(dW1, static_cast<std::uint64_t>(F) * Hd, 0.0f, st));
        TCC_HIP_CHECK(fill<float>(dW2, static_cast<std::uint64_t>(Hd) * C, 0.0f, st));
        return TCC_OK;
    }
    TCC_REQUIRE(AX && H && G && workspace, TCC_ERR_INVALID_ARGUMENT, "invalid GCN relu-gradient arguments");
    const TnPlan p = relu_grad_plan(K, F, Hd);
    const size_t need1 = static_cast<size_t>(p.splits) * F * Hd * sizeof(float);
    const size_t need2 = static_cast<size_t>(p.splits) * Hd * C * sizeof(float);
    TCC_REQUIRE(workspaceBytes >= need1 + need2, TCC_ERR_INVALID_ARGUMENT,
                "GCN relu-gradient workspace too small (tcc_gcn_relu_grad_workspace_bytes)");
    TCC_REQUIRE(static_cast<std::uint64_t>(p.blocksM) * p.blocksN <= 65535, TCC_ERR_UNSUPPORTED,
                "GCN relu-gradient output too large");
    TnArgs a{};
    a.A = AX;
    a.B = H;
    a.partial = static_cast<float*>(workspace);
    a.lda = ldax;
    a.ldb = ldh;
    a.K = K;
    a.M = F;
    a.N = Hd;
    a.rowsPerSplit = p.rowsPerSplit;
    a.blocksM = p.blocksM;
    a.G = G;
    a.W2 = W2;
    a.partial2 = reinterpret_cast<float*>(static_cast<char*>(workspace) + need1);
    a.ldg = ldg;
    a.C = C;
    a.blocksN = p.blocksN;
    a.splits = p.splits;
    const bool two = C <= 2;
    switch (p.shape) {
        case TnShape::Wide4: two ? tn_split_launch<4, 2>(a, p, st) : tn_split_launch<4, 8>(a, p, st); break;
        case TnShape::Wide7: two ? tn_split_launch<7, 2>(a, p, st) : tn_split_launch<7, 8>(a, p, st); break;
        default: two ? tn_split_launch<8, 2>(a, p, st) : tn_split_launch<8, 8>(a, p, st); break;
    }
    TCC_LAUNCH_CHECK();
    hipLaunchKernelGGL(tn_reduce_kernel, dim3(grid_for(static_cast<std::uint64_t>(F) * Hd, 16)), dim3(256), 0, st,
                       a.partial, p.splits, F, Hd, dW1, Hd, 0, 0);
    TCC_LAUNCH_CHECK();
    hipLaunchKernelGGL(tn_reduce_kernel, dim3(grid_for(static_cast<std::uint64_t>(Hd) * C, 16)), dim3(256), 0, st,
                       a.partial2, p.splits, Hd, C, dW2, C, 0, 0);
    TCC_LAUNCH_CHECK();
    return TCC_OK;
}

}  // extern "C"
