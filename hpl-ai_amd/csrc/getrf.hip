// getrf.hip — LU of a diagonal block (n <= 1024) and the inverses of its
// triangles, spread over the device.
//
// Products with inverses of 128-blocks take |A - L U| past the 2 (n + 80) u |L| |U|
// of elimination where the diagonal does not dominate (3.4 times for diagonals of
// 3 at 512, and refinement from such factors of 1024 with diagonals of 5 needed
// three times the steps or diverged).  So each sub-block's rows are looked at
// first: where the diagonal dominates, those products lose nothing; elsewhere
// strips of a sub-block whose triangles are not well conditioned are walked through
// with inverses of 32 x 32 blocks, and by substitution where one of those is not.
//
// Replaces getrf_nopiv (getrf_nopiv.hpp:124-160).  The block is walked in
// sub-blocks of 128 columns; per sub-block three kinds of work, all FP32 on
// v_mfma_f32_32x32x2_f32:
//   lu_update_kernel  workgroup 0 takes the 128 x 128 diagonal sub-block: its
//                     LU and the inverses of both triangles, all in LDS; the
//                     other workgroups update the rest of the trailing matrix;
//   lu_strip_kernel   L21 := A21 U11^-1 and U12 := L11^-1 A12 as products
//                     with those inverses, 32 rows or columns per workgroup,
//                     and in more workgroups, which form the strips that they
//                     need again, the update of the next diagonal sub-block.
// The inverses of the whole block grow by a sub-block q at a time,
//   Linv(q, J) = -Linv_qq T,   T  = sum_K L(q, K) Linv(K, J)
//   Uinv(J, q) = -T' Uinv_qq,  T' = sum_K Uinv(J, K) U(K, q)     (K < q),
// T by more workgroups of the launch that factors sub-block q, which leaves
// the device idle, and the products with Linv_qq and Uinv_qq by more
// workgroups of the next launch.  A block that is factored already joins the
// inverses of neighbouring sub-blocks (128 -> 256 -> 512 -> 1024) with the same
// two products, all pairs of a size at once.
//
// What bounds it: the chain of 32 x 32 LUs, inverses and strips (17k clocks a
// link, one or two waves working) and, between sub-blocks, two launches (9 us
// with the strips and the next sub-block's update).  One workgroup for the
// whole 512 block spent half its time on trailing updates through a single
// CU's path to the L2, and the inverses were two more kernels after it: 511 +
// 73 us, now 176 us with the inverses and 156 without (b = 512, alone); b = 60:
// 94 -> 14 us; n = 1000: 645 us with v_readlane steps, 327 us as here.  The
// next sub-block's update in the workgroup that factors it took 11 us of each
// sub-block (its operands, 192 KB, again through one CU): 198 us at b = 512.
// Joining the inverses by one workgroup per 32 columns took 39 us a size
// (product by product, each behind its loads) after the factorization.
#include <cfloat>
#include <cstddef>
#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"
#include "lu32.hpp"

namespace hplai {

typedef float floatx16g_t __attribute__((ext_vector_type(16)));

constexpr int kLuNB = 128;            // columns per sub-block
constexpr int kLuThreads = 512;
constexpr int kLuS = kLuNB + 1;       // LDS column stride: odd, so that walks along rows and columns both spread
using LuStride = std::integral_constant<int, kLuS>;
constexpr int kJoinMax = 512;         // largest half joined by tri_join_kernel
// Off-diagonal row sums up to this part of the diagonal entries bound the condition
// of a sub-block's triangles: with D its diagonal, |U^-1| |D|, |D^-1| |U| and so on
// have row sums of at most (1 + p) / (1 - p), |U^-1| |U| 4 at 0.6 and, rows scaled
// by D, |L^-1| |L| 16.  Those of HPL-AI matrices have about 128 / n (getrf of 512
// 156 us, 154 without the look).  Other sub-blocks look at their
// inverses (170 us), and strips go through those where no row sum of |X| |T| is past
// kCond128, else through 32-blocks (200 us).
constexpr float kCond128 = 16.0f;
constexpr float kDominance = 0.6f;

__device__ __forceinline__ floatx16g_t zero16()
{
    floatx16g_t z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.0f;
    return z;
}

struct LuLds {
    float S[kLuNB * kLuS];            // the sub-block, S[c * kLuS + r]
    float V[kLuNB * kLuS];            // its inverses: Linv below the diagonal (unit diagonal implied), Uinv on and above
    float Li[32 * 33], Ui[32 * 33];   // inverses of the current 32 x 32 triangles, row-major
    float w[2][32];                   // row sums of the current 32 x 32 triangles, L and U
    int poor[2];                      // they are not well conditioned
    float sums[2][4][kLuNB];          // row sums of the sub-block's magnitudes, later of its triangles', in parts
    int careful;                      // the sub-block's diagonal does not dominate
};

// entry (i, j) of a unit-lower / an upper triangle whose block also holds the other one
__device__ __forceinline__ float lower_entry(float v, int i, int j) { return i > j ? v : (i == j ? 1.0f : 0.0f); }
__device__ __forceinline__ float upper_entry(float v, int i, int j) { return i <= j ? v : 0.0f; }

// acc += A B of one 32 x 32 x 32 product from its operand registers.  The
// operands are loaded before: left to itself the compiler waits for each load
// right before its product.
__device__ __forceinline__ floatx16g_t mfma16(const float (&av)[16], const float (&bv)[16], floatx16g_t acc)
{
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[kk], bv[kk], acc, 0, 0, 0);
    return acc;
}

// Row q of Linv and column q of Uinv of the sub-block, 32 x 32 block by block:
//   Linv(q, b) = -Linv(q, q) T,   T  = sum_{b <= K < q} L(q, K) Linv(K, b)
//   Uinv(b, q) = -T' Uinv(q, q),  T' = sum_{b <= K < q} Uinv(b, K) U(K, q)
// T needs only what was final before step q, so it is formed while one wave
// factors the 32 x 32 block q; it stays in the wave's accumulators, whose rows
// set the order of the second product's K (acc_row).  The U side works on
// transposes so that T' is a right operand too.
template <bool UP>
__device__ __forceinline__ floatx16g_t inverse_row_product(const float *S, const float *V, int q, int b, int lane)
{
    const int l32 = lane & 31, lh = lane >> 5;
    floatx16g_t acc = zero16();
    for (int K = b; K < q; ++K) {
        float av[16], bv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            const int k = 2 * kk + lh;
            av[kk] = UP ? S[(32 * q + l32) * kLuS + 32 * K + k] : S[(32 * K + k) * kLuS + 32 * q + l32];
            bv[kk] = UP ? V[(32 * K + k) * kLuS + 32 * b + l32] : V[(32 * b + l32) * kLuS + 32 * K + k];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (K == b)   // the triangle's own block
#pragma unroll
            for (int kk = 0; kk < 16; ++kk) {
                const int k = 2 * kk + lh;
                bv[kk] = UP ? upper_entry(bv[kk], l32, k) : lower_entry(bv[kk], k, l32);
            }
        acc = mfma16(av, bv, acc);
    }
    return acc;
}

template <bool UP>
__device__ __forceinline__ void inverse_row_finish(float *V, int q, int b, int lane, const floatx16g_t &T)
{
    const int l32 = lane & 31, lh = lane >> 5;
    float av[16], bv[16];
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
        const int k = acc_row(kk, lh);
        av[kk] = UP ? V[(32 * q + l32) * kLuS + 32 * q + k] : V[(32 * q + k) * kLuS + 32 * q + l32];
        bv[kk] = T[kk];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
        const int k = acc_row(kk, lh);
        av[kk] = UP ? upper_entry(av[kk], k, l32) : lower_entry(av[kk], l32, k);
    }
    const floatx16g_t acc = mfma16(av, bv, zero16());
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        if (UP)
            V[(32 * q + acc_row(e, lh)) * kLuS + 32 * b + l32] = -acc[e];
        else
            V[(32 * b + l32) * kLuS + 32 * q + acc_row(e, lh)] = -acc[e];
    }
}

// One wave: block t of row q of Linv (t <= q) or column q of Uinv (t - q - 1)
// into the packed arrays, 16 floats per MFMA lane.  sides: 1
// Linv, 2 Uinv, 3 both.
__device__ __forceinline__ void write_inverse_row(const float *V, float *tri, int nb, int q0, int q, int t, int sides,
                                                  int lane)
{
    const int l32 = lane & 31, lh = lane >> 5;
    const bool up = t > q;
    if (tri == nullptr || t >= 2 * (q + 1) || !(sides & (up ? 2 : 1))) return;
    const int b = up ? t - q - 1 : t;
    float v[16];
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
        v[kk] = *(up ? &V[(32 * q + l32) * kLuS + 32 * b + 2 * kk + lh] : &V[(32 * b + 2 * kk + lh) * kLuS + 32 * q + l32]);
    __builtin_amdgcn_sched_barrier(0);
    if (b == q)
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            v[kk] = up ? upper_entry(v[kk], 2 * kk + lh, l32) : lower_entry(v[kk], l32, 2 * kk + lh);
    float4 *o = reinterpret_cast<float4 *>(up ? tri_block_u(tri, nb, q0 + b, q0 + q)
                                              : tri_block_l(tri, nb, q0 + q, q0 + b)) + lane;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e * 64] = float4{v[4 * e], v[4 * e + 1], v[4 * e + 2], v[4 * e + 3]};
}

// Position of entry (r, c) in a packed block, as a left or a right operand
__device__ __forceinline__ int left_pos(int r, int c) { return tri_pos(r + 32 * (c & 1), c >> 1); }
__device__ __forceinline__ int right_pos(int r, int c) { return tri_pos(c + 32 * (r & 1), r >> 1); }

// Copies of A21's and A12's blocks (I, J) beside a diagonal sub-block, [32 k +
// row or column], in the slots of the other triangle that the inverses leave
// free: the strips overwrite the blocks in A while others still need them.
__device__ __forceinline__ float *copy_l(float *tri, int nb, int I, int J) { return tri_block_u(tri, nb, I, J); }
__device__ __forceinline__ float *copy_u(float *tri, int nb, int I, int J) { return tri_block_l(tri, nb, I, J); }

__device__ __forceinline__ void packed16(const float *blk, int lane, float (&v)[16])
{
    const float4 *p = reinterpret_cast<const float4 *>(blk) + lane;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float4 q = p[e * 64];
        v[4 * e] = q.x;
        v[4 * e + 1] = q.y;
        v[4 * e + 2] = q.z;
        v[4 * e + 3] = q.w;
    }
}

// First product, 512 threads: for the four 32-blocks X = R .. R + 3 (< Rend)
//   L side:  T(X, J)  = sum_{J <= K < K1} L(X, K) Linv(K, J), as a right operand to Linv's slot (X, J)
//   U side:  T'(J, X) = sum_{J <= K < K1} Uinv(J, K) U(K, X), as a left operand to Uinv's slot (J, X)
// The inverse's strip comes out of its order through W (33 floats per k, the
// K1 - J blocks' 32 k each); two waves per X take every other K.
template <bool UP>
__device__ __forceinline__ void tri_mid(int n, int nb, const float *A, int64_t lda, float *tri, int J, int K1, int R,
                                        int Rend, float *W)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5, X = R + (wave & 3), half = wave >> 2;
#pragma unroll 4
    for (int e = tid; e < (K1 - J) * 1024; e += kLuThreads) {
        const int K = J + (e >> 10), ln = (e >> 2) & 63, kk = ((e >> 8) & 3) * 4 + (e & 3);   // as tri_pos
        const float *blk = UP ? tri_block_u(tri, nb, J, K) : tri_block_l(tri, nb, K, J);
        W[(32 * (K - J) + (ln & 31)) * 33 + 2 * kk + (ln >> 5)] = blk[e & 1023];
    }
    __syncthreads();
    floatx16g_t acc = zero16();
    const bool on = X < Rend;
    if (on) {
        const int x = 32 * X + l32;             // row of L, column of U
        const int64_t xo = min(x, n - 1);
        for (int K = J + half; K < K1; K += 8) {
            float av[4][16];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (K + 2 * u < K1)
#pragma unroll
                    for (int kk = 0; kk < 16; ++kk) {
                        const int64_t k = 32 * (K + 2 * u) + 2 * kk + lh;   // below n: the blocks before X are whole
                        av[u][kk] = UP ? A[xo * lda + k] : A[k * lda + xo];
                    }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (K + 2 * u < K1) {
                    float wv[16];
#pragma unroll
                    for (int kk = 0; kk < 16; ++kk) {
                        wv[kk] = W[(32 * (K + 2 * u - J) + 2 * kk + lh) * 33 + l32];
                        if (x >= n) av[u][kk] = 0.0f;
                    }
                    acc = UP ? mfma16(wv, av[u], acc) : mfma16(av[u], wv, acc);
                }
        }
    }
    __syncthreads();
    if (on && half == 1)
#pragma unroll
        for (int e = 0; e < 16; ++e) W[((wave & 3) * 16 + e) * 64 + lane] = acc[e];
    __syncthreads();
    if (on && half == 0) {
        float *o = UP ? tri_block_u(tri, nb, J, X) : tri_block_l(tri, nb, X, J);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int r = acc_row(e, lh);
            o[UP ? left_pos(r, l32) : right_pos(r, l32)] = acc[e] + W[(wave * 16 + e) * 64 + lane];
        }
    }
}

// Second product, in place, NW waves, at most PER * NW blocks X = R0 .. R1 - 1:
//   Linv(X, J) = -sum_{R0 <= K <= X} Linv(X, K) T(K, J),  Uinv(J, X) = -sum_{R0 <= K <= X} T'(J, K) Uinv(K, X)
template <bool UP, int NW, int PER>
__device__ __forceinline__ void tri_fin(int nb, float *tri, int J, int R0, int R1)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    floatx16g_t acc[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int X = R0 + wave + NW * i;
        acc[i] = zero16();
        if (X >= R1) continue;
        for (int K = R0; K <= X; K += 4) {
            float av[4][16], bv[4][16];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (K + u <= X) {
                    packed16(UP ? tri_block_u(tri, nb, J, K + u) : tri_block_l(tri, nb, X, K + u), lane, av[u]);
                    packed16(UP ? tri_block_u(tri, nb, K + u, X) : tri_block_l(tri, nb, K + u, J), lane, bv[u]);
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (K + u <= X) acc[i] = mfma16(av[u], bv[u], acc[i]);
        }
    }
    __syncthreads();   // every T of column (row) J is read
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int X = R0 + wave + NW * i;
        if (X >= R1) continue;
        float *o = UP ? tri_block_u(tri, nb, J, X) : tri_block_l(tri, nb, X, J);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int r = acc_row(e, lh);
            o[UP ? right_pos(r, l32) : left_pos(r, l32)] = -acc[i][e];
        }
    }
}

// Sub-block k0 of the n x n block A.  FACTOR: LU, inverses and whether the strips
// may go through these; the next workgroups update the rest of the trailing matrix
// with sub-block k0 - 128 (when there is one) and copy the blocks beside the
// diagonal one, and the last form the first products of the whole block's inverses.
// Without FACTOR: A is already factored and workgroup q inverts the triangles of
// sub-block q, or, without FULL, of its 32 x 32 blocks alone.
template <bool FACTOR, bool FULL>
__global__ __launch_bounds__(kLuThreads) void lu_update_kernel(int n, int k0, float *__restrict__ A, int64_t lda,
                                                               float *tri, int sides,
                                                               int *__restrict__ info)
{
    __shared__ LuLds sm;
    float *S = sm.S, *V = sm.V;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int nb = (n + 31) / 32;
    if (!FACTOR) k0 = static_cast<int>(blockIdx.x) * kLuNB;
    const int p0 = k0 - kLuNB;
    float *Ak = A + static_cast<int64_t>(k0) * lda + k0;

    if (FACTOR && blockIdx.x > 0) {
        // ---- a 128 x 64 tile of the trailing matrix, one 32 x 32 block per wave ----
        const int rest = n - k0, ct = (rest + 63) / 64, rt = (rest + 127) / 128;
        // tiles in row-major order without the two of the diagonal sub-block;
        // of the first sub-block only the four that are copied
        const int two = ct < 2 ? ct : 2, z = static_cast<int>(blockIdx.x) - 1;
        const int t = p0 >= 0 ? z + two : z < 2 ? ct + z : z;
        if (p0 >= 0 && t >= rt * ct) {
            static_assert(offsetof(LuLds, V) == sizeof(float) * kLuNB * kLuS && (1024 - kLuNB) * 33 <= 2 * kLuNB * kLuS,
                          "the strip of an inverse spans S and V");
            const int y = t - rt * ct, q0 = k0 / 32;
            if (y & 1)
                tri_mid<true>(n, nb, A, lda, tri, y >> 1, q0, q0, nb < q0 + 4 ? nb : q0 + 4, S);
            else
                tri_mid<false>(n, nb, A, lda, tri, y >> 1, q0, q0, nb < q0 + 4 ? nb : q0 + 4, S);
            return;
        }
        const int r0 = (t / ct) * 128 + (wave & 3) * 32, c0 = (t % ct) * 64, cw = c0 + (wave >> 2) * 32;
        // U12 (128 x 64) through LDS: its MFMA operand walks along columns
        if (p0 >= 0) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                const int c = (tid >> 7) + 4 * u, k = tid & 127;
                v[u] = A[static_cast<int64_t>(k0 + min(c0 + c, rest - 1)) * lda + p0 + k];
            }
#pragma unroll
            for (int u = 0; u < 16; ++u) S[((tid >> 7) + 4 * u) * kLuS + (tid & 127)] = v[u];
        }
        __syncthreads();
        if (r0 >= rest || cw >= rest) return;
        float cv[16];
#pragma unroll
        for (int e = 0; e < 16; ++e)
            cv[e] = Ak[static_cast<int64_t>(min(cw + l32, rest - 1)) * lda + min(r0 + acc_row(e, lh), rest - 1)];
        if (p0 >= 0) {
            const float *lp = A + static_cast<int64_t>(p0 + lh) * lda + k0 + min(r0 + l32, rest - 1);
            floatx16g_t acc = zero16();
            float av[64];
#pragma unroll
            for (int kk = 0; kk < 64; ++kk) av[kk] = lp[static_cast<int64_t>(2 * kk) * lda];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
                float bv[16];
#pragma unroll
                for (int kk = 0; kk < 16; ++kk) bv[kk] = S[(cw - c0 + l32) * kLuS + 32 * h + 2 * kk + lh];
#pragma unroll
                for (int kk = 0; kk < 16; ++kk)
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[16 * h + kk], bv[kk], acc, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) cv[e] -= acc[e];
            if (cw + l32 < rest) {
                float *cp = Ak + static_cast<int64_t>(cw + l32) * lda + r0;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int r = acc_row(e, lh);
                    if (r0 + r < rest) cp[r] = cv[e];
                }
            }
        }
        // the blocks right of and below the diagonal sub-block once more, k by k
        if (r0 >= kLuNB && r0 < 2 * kLuNB && cw < kLuNB) {
            float4 *o = reinterpret_cast<float4 *>(copy_l(tri, nb, (k0 + r0) / 32, (k0 + cw) / 32) + l32 * 32 + 4 * lh);
#pragma unroll
            for (int q = 0; q < 4; ++q) o[2 * q] = float4{cv[4 * q], cv[4 * q + 1], cv[4 * q + 2], cv[4 * q + 3]};
        } else if (r0 < kLuNB && cw >= kLuNB && cw < 2 * kLuNB) {
            float *o = copy_u(tri, nb, (k0 + r0) / 32, (k0 + cw) / 32);
#pragma unroll
            for (int e = 0; e < 16; ++e) o[acc_row(e, lh) * 32 + l32] = cv[e];
        }
        return;
    }

    // ---- the diagonal sub-block, padded to 128 with the identity ----
    const int w = n - k0 < kLuNB ? n - k0 : kLuNB;
    const int steps = (w + 31) / 32, q0 = k0 / 32;
    {
        const int r = tid & 127;
        float s = 0.0f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e)
                v[e] = Ak[static_cast<int64_t>(min((tid >> 7) + 4 * (16 * h + e), w - 1)) * lda + min(r, w - 1)];
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int c = (tid >> 7) + 4 * (16 * h + e);
                v[e] = (r < w && c < w) ? v[e] : (r == c ? 1.0f : 0.0f);
                S[c * kLuS + r] = v[e];
                if (FACTOR) s += fabsf(v[e]);
            }
        }
        if (FACTOR) sm.sums[0][tid >> 7][r] = s;
        if (FACTOR && tid == 0) sm.careful = 0;
    }
    __syncthreads();
    if (!FACTOR) {
        // waves 2 q, 2 q + 1 invert the triangles of 32-block q
        const int at = 32 * (wave >> 1) * (kLuS + 1);
        if (wave & 1)
            invert32<true>(S + at, LuStride{}, V + at, lane, nullptr);
        else
            invert32<false>(S + at, LuStride{}, V + at, lane, nullptr);
        wave_lds_sync();
        {
            float *w = sm.Li + 32 * wave;   // row sums of this wave's triangle
            if (wave & 1)
                row_sums32<true>(S + at, LuStride{}, w, lane);
            else
                row_sums32<false>(S + at, LuStride{}, w, lane);
            wave_lds_sync();
            const bool poor = poor32([&](int r, int c) {
                const float v = V[at + c * kLuS + r];
                return wave & 1 ? upper_entry(v, r, c) : lower_entry(v, r, c);
            }, w, lane);
            if (lane == 0 && (wave >> 1) < steps) tri_poor(tri, nb)[2 * q0 + wave] = poor ? 1.0f : 0.0f;
        }
        if (FULL) {
            for (int q = 0; q < steps; ++q) {
                if (wave < 2 * q) {
                    const int b = wave >> 1;
                    if (wave & 1)
                        inverse_row_finish<true>(V, q, b, lane, inverse_row_product<true>(S, V, q, b, lane));
                    else
                        inverse_row_finish<false>(V, q, b, lane, inverse_row_product<false>(S, V, q, b, lane));
                }
                __syncthreads();
                write_inverse_row(V, tri, nb, q0, q, wave, sides, lane);
            }
        } else {
            const int q = wave >> 1;
            if (q < steps) write_inverse_row(V, tri, nb, q0, q, wave & 1 ? 2 * q + 1 : q, sides, lane);
        }
        return;
    }

    // 32 x 32 block (r0, cc) of S takes the strips of the 32 columns at c0
    auto update = [&](int ln, int c0, int r0, int cc) {
        const int l32 = ln & 31, lh = ln >> 5;
        floatx16g_t acc = zero16();
        float av[16], bv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            const int k = 2 * kk + lh;
            av[kk] = S[(c0 + k) * kLuS + r0 + l32];
            bv[kk] = S[(cc + l32) * kLuS + c0 + k];
        }
        acc = mfma16(av, bv, acc);
#pragma unroll
        for (int e = 0; e < 16; ++e) S[(cc + l32) * kLuS + r0 + acc_row(e, lh)] -= acc[e];
    };
    int bad = 0;
    bool careful = false;   // strips by substitution where the inverses are not well conditioned
    for (int q = 0; q < steps; ++q) {
        const int c0 = 32 * q, t = 7 - wave;   // t: this wave's block of the inverses' row q
        // a lane number of the iteration's own: addresses and masks hoisted out
        // of this loop fill the register file
        int ln = lane;
        asm volatile("" : "+v"(ln));
        floatx16g_t T = zero16();
        // wave 0: the next diagonal block's update, then its LU; the other
        // waves meanwhile update the rest, write out the inverses' row q - 1
        // and form the products of row q
        if (wave == 0) {
            if (q > 0) {
                update(ln, c0 - 32, c0, c0);
                wave_lds_sync();
            }
            const int z = lu32(S + c0 * (kLuS + 1), LuStride{}, ln);
            if (bad == 0 && z != 0) bad = k0 + c0 + z;
        } else if (q > 0) {
            const int R = steps - q;
            for (int i = wave; i < R * R; i += kLuThreads / 64 - 1) update(ln, c0 - 32, c0 + 32 * (i % R), c0 + 32 * (i / R));
            write_inverse_row(V, tri, nb, q0, q - 1, wave - 1, sides, ln);
            if (tri != nullptr && t < 2 * q)
                T = t & 1 ? inverse_row_product<true>(S, V, q, t >> 1, ln) : inverse_row_product<false>(S, V, q, t >> 1, ln);
        } else if (wave >= 6) {
            const int r = 64 * (wave - 6) + ln;
            const float d = r < w ? fabsf(Ak[r * (lda + 1)]) : 1.0f;
            const float *p = &sm.sums[0][0][r], s = ((p[0] + p[kLuNB]) + p[2 * kLuNB]) + p[3 * kLuNB];
            if (!__all(s <= fminf((1.0f + kDominance) * d, FLT_MAX))) sm.careful = 1;
        }
        __syncthreads();
        if (q == 0) careful = __builtin_amdgcn_readfirstlane(sm.careful) != 0;
        if (wave == 0) {
            invert32<false>(S + c0 * (kLuS + 1), LuStride{}, V + c0 * (kLuS + 1), ln, sm.Li);
        } else if (wave == 1) {
            invert32<true>(S + c0 * (kLuS + 1), LuStride{}, V + c0 * (kLuS + 1), ln, sm.Ui);
        } else {
            if (careful && wave == 6) row_sums32<false>(S + c0 * (kLuS + 1), LuStride{}, sm.w[0], ln);
            if (careful && wave == 7) row_sums32<true>(S + c0 * (kLuS + 1), LuStride{}, sm.w[1], ln);
            if (q + 1 == steps)   // all of S is final: factors back to A
#pragma unroll 4
                for (int c = (wave - 2) >> 1; c < w; c += 3) {
                    const int r = 64 * (wave & 1) + ln;
                    if (r < w) Ak[static_cast<int64_t>(c) * lda + r] = S[c * kLuS + r];
                }
        }
        __syncthreads();
        // L21 := A21 U11^-1 and U12 := L11^-1 A12, one 32 x 32 block per wave
        const int R = steps - 1 - q;
        const bool mine = wave < 2 * R, up = wave >= R;
        const int o = c0 + 32 * (1 + (up ? wave - R : wave));
        floatx16g_t X = zero16();
        if (mine) {
            const int l32 = ln & 31, lh = ln >> 5;
            float av[16], bv[16];
            if (up) {
#pragma unroll
                for (int kk = 0; kk < 16; ++kk) {
                    av[kk] = sm.Li[l32 * 33 + 2 * kk + lh];
                    bv[kk] = S[(o + l32) * kLuS + c0 + 2 * kk + lh];
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < 16; ++kk) {
                    av[kk] = S[(c0 + 2 * kk + lh) * kLuS + o + l32];
                    bv[kk] = sm.Ui[(2 * kk + lh) * 33 + l32];
                }
            }
            X = mfma16(av, bv, X);
        } else if (careful && wave >= 6 && (R > 0 || tri != nullptr)) {
            const float *M = wave == 6 ? sm.Li : sm.Ui;
            const bool poor = poor32([&](int r, int c) { return M[r * 33 + c]; }, sm.w[wave - 6], ln);
            if (ln == 0) {
                sm.poor[wave - 6] = poor;
                if (tri != nullptr) tri_poor(tri, nb)[2 * (q0 + q) + wave - 6] = poor ? 1.0f : 0.0f;
            }
        }
        if (careful && R > 0) __syncthreads();
        if (careful && mine && sm.poor[up ? 0 : 1]) {
            // by substitution, a row or column per lane
            float *x = up ? S + (o + (ln & 31)) * kLuS + c0 : S + c0 * kLuS + o + (ln & 31);
            const int dx = up ? 1 : kLuS;
            if (ln < 32)
#pragma clang loop unroll(disable)
                for (int k = 0; k < 32; ++k) {
                    float v = x[k * dx];
                    if (!up) {
                        v *= 1.0f / S[(c0 + k) * kLuS + c0 + k];
                        x[k * dx] = v;
                    }
#pragma clang loop unroll_count(4)
                    for (int j = k + 1; j < 32; ++j)
                        x[j * dx] = fmaf(-v, up ? S[(c0 + k) * kLuS + c0 + j] : S[(c0 + j) * kLuS + c0 + k], x[j * dx]);
                }
        } else if (mine) {
            const int l32 = ln & 31, lh = ln >> 5;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int r = acc_row(e, lh);
                if (up)
                    S[(o + l32) * kLuS + c0 + r] = X[e];
                else
                    S[(c0 + l32) * kLuS + o + r] = X[e];
            }
        }
        if (tri != nullptr && t < 2 * q) {
            if (t & 1)
                inverse_row_finish<true>(V, q, t >> 1, ln, T);
            else
                inverse_row_finish<false>(V, q, t >> 1, ln, T);
        }
        __syncthreads();
    }
    write_inverse_row(V, tri, nb, q0, steps - 1, wave, sides, lane);
    if (k0 + kLuNB < n) {
        int poor = 0;
        if (careful) {
            // the largest row sum of |X| |T|: row sums of |T| first, a quarter of the
            // columns per two waves, side 0 L and side 1 U
            int i = tid;
            asm volatile("" : "+v"(i));   // as ln
            const int r = i & 127, g = wave >> 1;
            float sl = r >> 5 == g ? 1.0f : 0.0f, su = 0.0f;
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                const float v = fabsf(S[(32 * g + k) * kLuS + r]);
                sl += 32 * g + k < r ? v : 0.0f;
                su += 32 * g + k < r ? 0.0f : v;
            }
            sm.sums[0][g][r] = sl;
            sm.sums[1][g][r] = su;
            __syncthreads();
            const float *p = &sm.sums[0][0][32 * g + (i & 31)];
            const float wl = ((p[0] + p[kLuNB]) + p[2 * kLuNB]) + p[3 * kLuNB];
            p += 4 * kLuNB;
            const float wu = ((p[0] + p[kLuNB]) + p[2 * kLuNB]) + p[3 * kLuNB];
            __syncthreads();
            const float d = __shfl(wl, r & 31);
            sl = r >> 5 == g ? d : 0.0f;   // the unit diagonal's term
            su = 0.0f;
#pragma unroll
            for (int k = 0; k < 32; ++k) {
                const float v = fabsf(V[(32 * g + k) * kLuS + r]);
                const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), k));
                const float c = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wu), k));
                sl = fmaf(32 * g + k < r ? v : 0.0f, a, sl);
                su = fmaf(32 * g + k < r ? 0.0f : v, c, su);
            }
            sm.sums[0][g][r] = sl;
            sm.sums[1][g][r] = su;
            __syncthreads();
            p = &sm.sums[wave < 2 ? 0 : 1][0][r];
            poor = wave < 4 && !__all(((p[0] + p[kLuNB]) + p[2 * kLuNB]) + p[3 * kLuNB] <= kCond128);
            poor = __syncthreads_or(poor);
        }
        if (tid == 0) tri_careful(tri, nb)[q0 / 4] = poor ? 1.0f : 0.0f;
    }
    if (tid == 0 && info != nullptr && (k0 == 0 || (bad != 0 && *info == 0))) *info = bad;
}

// Block (r, c) of the next diagonal sub-block -= L21(r, :) U12(:, c), with its
// strips formed from the copies: wave J forms L21(r, J)^T and U12(J, c), whose
// accumulators are the operands of their product (k = acc_row either way).  With
// careful: nothing.
__device__ __forceinline__ bool next_diagonal(int n, int nb, int q0, int r, int c, float *A, int64_t lda, float *tri,
                                              float *XL, float *XU, int careful)
{
    const int tid = threadIdx.x, lane = tid & 63, J = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int R = q0 + 4 + r, C = q0 + 4 + c;
    float il[4][16], iu[4][16];   // the inverses' blocks, clamped to the last that is used
    float4 xl[4], xu[4];
#pragma unroll
    for (int K = 0; K < 4; ++K) {
        xl[K] = reinterpret_cast<const float4 *>(copy_l(tri, nb, R, q0 + K))[tid];
        xu[K] = reinterpret_cast<const float4 *>(copy_u(tri, nb, q0 + K, C))[tid];
    }
#pragma unroll
    for (int K = 0; K < 4; ++K) {
        packed16(tri_block_u(tri, nb, q0 + min(K, J), q0 + J), lane, il[K]);
        packed16(tri_block_l(tri, nb, q0 + J, q0 + min(K, J)), lane, iu[K]);
    }
    const int64_t col = min(32 * C + l32, n - 1);
    float d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = A[col * lda + min(32 * R + 8 * J + 4 * lh + i, n - 1)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int K = 0; K < 4; ++K) {
        float *x = XL + (32 * K + (tid >> 3)) * 33 + 4 * (tid & 7), *y = XU + (32 * K + (tid >> 3)) * 33 + 4 * (tid & 7);
        x[0] = xl[K].x;
        x[1] = xl[K].y;
        x[2] = xl[K].z;
        x[3] = xl[K].w;
        y[0] = xu[K].x;
        y[1] = xu[K].y;
        y[2] = xu[K].z;
        y[3] = xu[K].w;
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(careful) != 0) return false;
    floatx16g_t al = zero16(), au = zero16();
#pragma unroll
    for (int K = 0; K < 4; ++K) {
        if (K > J) break;
        float xv[16], yv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            xv[kk] = XL[(32 * K + 2 * kk + lh) * 33 + l32];
            yv[kk] = XU[(32 * K + 2 * kk + lh) * 33 + l32];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            al = __builtin_amdgcn_mfma_f32_32x32x2f32(il[K][kk], xv[kk], al, 0, 0, 0);
            au = __builtin_amdgcn_mfma_f32_32x32x2f32(iu[K][kk], yv[kk], au, 0, 0, 0);
        }
    }
    floatx16g_t acc = zero16();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(al[kk], au[kk], acc, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) XL[(J * 16 + e) * 64 + lane] = acc[e];
    __syncthreads();
    // wave J: rows 8 J + 4 lh + i, the waves' sums in order
    if (32 * C + l32 < n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float *p = XL + (4 * J + i) * 64 + lane;
            const int row = 32 * R + 8 * J + 4 * lh + i;
            if (row < n) A[col * lda + row] = d[i] - (((p[0] + p[1024]) + p[2048]) + p[3072]);
        }
    return true;
}

// The same 32-block by 32-block (trsm.hip has the walk for panels), where a
// sub-block is not well conditioned: y < 0: strip z, 32 rows of L21 or (up1)
// columns of U12; else both strips that block (r, c) = y of the next diagonal
// sub-block needs, from the copies, one after the other, and then that block.
// Wave J holds block J in its accumulators' order, transposed for L21.  xl: -X_K of
// both sides.
__device__ __forceinline__ void strip_walk(int n, int p0, float *A, int64_t lda, float *tri, int z, bool up1, int y,
                                           int nd, float (*xl)[4][1024])
{
    const int tid = threadIdx.x, lane = tid & 63, J = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int nb = (n + 31) / 32, q0 = p0 / 32, k1 = p0 + kLuNB;
    const float *T = A + static_cast<int64_t>(p0) * (lda + 1);
    const int r = y % nd, c = y / nd;
    const int o = k1 + 32 * z, cnt = n - o < 32 ? n - o : 32;   // a strip
    const int R = 32 * (q0 + 4 + r), C = 32 * (q0 + 4 + c) + l32;
    float next[4];   // rows 8 J + 4 lh + i of the next block
#pragma clang loop unroll(disable)
    for (int side = 0; side < (y >= 0 ? 2 : 1); ++side) {
        const bool up = y >= 0 ? side != 0 : up1;
        // entry k = 32 J + acc_row of row (L21) or column (U12) l32
        float own[16], left[3][16], iv[16], diag[16];
        const int64_t step = up ? 1 : lda;
        float *line = A + (up ? (o + min(l32, cnt - 1)) * lda + p0 + 32 * J + 4 * lh
                              : (p0 + 32 * J + 4 * lh) * lda + o + min(l32, cnt - 1));
        {
            const float *copy = up ? copy_u(tri, nb, q0 + J, q0 + 4 + c) : copy_l(tri, nb, q0 + 4 + r, q0 + J);
            const float *from = y >= 0 ? copy + 128 * lh + l32 : line;
            const int64_t d = y >= 0 ? 32 : step;
#pragma unroll
            for (int e = 0; e < 16; ++e) own[e] = from[acc_row(e, 0) * d];
            const float *blk = up ? tri_block_l(tri, nb, q0 + J, q0 + J) : tri_block_u(tri, nb, q0 + J, q0 + J);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int k = acc_row(e, lh);
                iv[e] = blk[tri_pos(l32 + 32 * (k & 1), k >> 1)];
                diag[e] = up ? 1.0f : blk[tri_pos(k + 32 * (k & 1), k >> 1)];
            }
            const int64_t dk = up ? lda : 1;
            const float *t = T + (up ? 32 * J + l32 + 4 * lh * lda : (32 * J + l32) * lda + 4 * lh);
#pragma unroll
            for (int K = 0; K < 3; ++K)
                if (K < J)
#pragma unroll
                    for (int e = 0; e < 16; ++e) left[K][e] = t[(32 * K + acc_row(e, 0)) * dk];
        }
        if (y >= 0 && side == 0)
#pragma unroll
            for (int i = 0; i < 4; ++i) next[i] = A[min(C, n - 1) * lda + min(R + 8 * J + 4 * lh + i, n - 1)];
        const bool poor = tri_poor(tri, nb)[2 * (q0 + J) + (up ? 0 : 1)] != 0.0f;
        floatx16g_t S = zero16(), x = zero16();
#pragma unroll
        for (int K = 0; K < 4; ++K) {
            float *xk = xl[up][K];
            if (J == K) {
                floatx16g_t D;
                bool fine = !poor;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    D[e] = own[e] + S[e];
                    fine = fine && isfinite(D[e]);
                }
                if (__all(fine)) {
#pragma unroll
                    for (int e = 0; e < 16; ++e)   // the diagonal's term last, in one rounding
                        x = __builtin_amdgcn_mfma_f32_32x32x2f32(acc_row(e, lh) == l32 ? 0.0f : iv[e], D[e], x, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 16; ++e) x[e] = fmaf(diag[e], own[e], fmaf(diag[e], S[e], x[e]));
                } else {
#pragma unroll
                    for (int e = 0; e < 16; ++e) xk[e * 64 + lane] = D[e];
                    const float *d = T + 32 * static_cast<int64_t>(K) * (lda + 1);
                    if (up)
                        subst32<true>(xk, d, lda, 32, lane);
                    else
                        subst32<false>(xk, d, lda, 32, lane);
#pragma unroll
                    for (int e = 0; e < 16; ++e) x[e] = xk[e * 64 + lane];
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) xk[e * 64 + lane] = -x[e];
            }
            if (K == 3 && y < 0) break;
            __syncthreads();
            if (J > K) {
                float xv[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) xv[e] = xk[e * 64 + lane];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    S = __builtin_amdgcn_mfma_f32_32x32x2f32(K == 0 ? left[0][e] : K == 1 ? left[1][e] : left[2][e], xv[e], S, 0, 0, 0);
            }
        }
        if (y < 0 && l32 < cnt)
#pragma unroll
            for (int e = 0; e < 16; ++e) line[acc_row(e, 0) * step] = x[e];
    }
    if (y < 0) return;
    // block (r, c) of the next diagonal sub-block: a product per wave, added in order
    float av[16], bv[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        av[e] = xl[0][J][e * 64 + lane];
        bv[e] = xl[1][J][e * 64 + lane];
    }
    __syncthreads();
    float *part = xl[0][0];
    const floatx16g_t acc = mfma16(av, bv, zero16());
#pragma unroll
    for (int e = 0; e < 16; ++e) part[(J * 16 + e) * 64 + lane] = acc[e];
    __syncthreads();
    if (C < n)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float *p = part + (4 * J + i) * 64 + lane;
            const int row = R + 8 * J + 4 * lh + i;
            if (row < n) A[C * lda + row] = next[i] - (((p[0] + p[1024]) + p[2048]) + p[3072]);
        }
}

// L21 := A21 Uinv and U12 := Linv A12 for the rows and columns past the
// sub-block at p0 (128 wide).  A workgroup owns 32 rows of L21 (blockIdx.x <
// strips) or 32 columns of U12; wave j computes its 32-wide block j.  The next
// workgroups update a block each of the next diagonal sub-block, the last ones
// finish the whole block's inverses of this one.  Where the sub-block is not well
// conditioned, the walk above takes their place; whether it does is looked up
// beside the operands' loads.
__global__ __launch_bounds__(256) void lu_strip_kernel(int n, int p0, float *A, int64_t lda, float *tri, int strips)
{
    __shared__ float X[2 * kLuNB * 33];
    static_assert(sizeof(X) >= sizeof(float[2][4][1024]), "the walk's blocks");
    auto walk = reinterpret_cast<float (*)[4][1024]>(X);
    const int tid = threadIdx.x, lane = tid & 63, J = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int nb = (n + 31) / 32, q0 = p0 / 32, k1 = p0 + kLuNB;
    const int careful = __float_as_int(tri_careful(tri, nb)[q0 / 4]);
    const int nd = strips < 4 ? strips : 4;
    if (static_cast<int>(blockIdx.x) >= 2 * strips) {
        const int y = static_cast<int>(blockIdx.x) - 2 * strips, z = y - nd * nd;
        if (z < 0) {
            if (!next_diagonal(n, nb, q0, y % nd, y / nd, A, lda, tri, X, X + kLuNB * 33, careful))
                strip_walk(n, p0, A, lda, tri, 0, false, y, nd, walk);
        } else if (z & 1)
            tri_fin<true, 4, 1>(nb, tri, z >> 1, q0, nb < q0 + 4 ? nb : q0 + 4);
        else
            tri_fin<false, 4, 1>(nb, tri, z >> 1, q0, nb < q0 + 4 ? nb : q0 + 4);
        return;
    }
    const bool up = static_cast<int>(blockIdx.x) >= strips;
    const int o = k1 + 32 * (static_cast<int>(blockIdx.x) - (up ? strips : 0));   // first row / column
    const int cnt = n - o < 32 ? n - o : 32;
    float iv[4][16];   // the inverse's blocks, clamped to the last that is used
    {
        float v[16];
        auto inverse = [&] {
#pragma unroll
            for (int K = 0; K < 4; ++K) {
                const int k = q0 + min(K, J);
                packed16(up ? tri_block_l(tri, nb, q0 + J, k) : tri_block_u(tri, nb, k, q0 + J), lane, iv[K]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (up) {
            // X[k * 33 + c]: row p0 + k, column o + c
#pragma unroll
            for (int u = 0; u < 16; ++u)
                v[u] = A[static_cast<int64_t>(o + min((tid >> 7) + 2 * u, cnt - 1)) * lda + p0 + (tid & 127)];
            inverse();
#pragma unroll
            for (int u = 0; u < 16; ++u) X[(tid & 127) * 33 + (tid >> 7) + 2 * u] = v[u];
        } else {
            // X[k * 33 + r]: column p0 + k, row o + r
#pragma unroll
            for (int u = 0; u < 16; ++u)
                v[u] = A[static_cast<int64_t>(p0 + (tid >> 5) + 8 * u) * lda + o + min(tid & 31, cnt - 1)];
            inverse();
#pragma unroll
            for (int u = 0; u < 16; ++u) X[((tid >> 5) + 8 * u) * 33 + (tid & 31)] = v[u];
        }
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(careful) != 0) {
        strip_walk(n, p0, A, lda, tri, static_cast<int>(blockIdx.x) - (up ? strips : 0), up, -1, nd, walk);
        return;
    }
    floatx16g_t acc = zero16();
#pragma unroll
    for (int K = 0; K < 4; ++K) {
        if (K > J) break;
        float xv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) xv[kk] = X[(32 * K + 2 * kk + lh) * 33 + l32];
        acc = up ? mfma16(iv[K], xv, acc) : mfma16(xv, iv[K], acc);
    }
    if (up) {
        if (l32 < cnt) {
            float *cp = A + static_cast<int64_t>(o + l32) * lda + p0 + 32 * J;
#pragma unroll
            for (int e = 0; e < 16; ++e) cp[acc_row(e, lh)] = acc[e];
        }
    } else {
        float *cp = A + static_cast<int64_t>(p0 + 32 * J + l32) * lda + o;
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (acc_row(e, lh) < cnt) cp[acc_row(e, lh)] = acc[e];
    }
}

// Joins the inverses of the halves [I0, I0 + H) and [I0 + H, I1) (32-blocks)
// of every pair: blockIdx.x the pair and J of its first half, blockIdx.z +
// side0 the L or the U side.  MID: the first product for four blocks of the
// second half (blockIdx.y); else the second product.
template <bool MID>
__global__ __launch_bounds__(kLuThreads) void tri_join_kernel(int n, int H, const float *__restrict__ A, int64_t lda,
                                                              float *tri, int side0)
{
    const int nb = (n + 31) / 32;
    const bool up = static_cast<int>(blockIdx.z) + side0 != 0;
    const int J = static_cast<int>(blockIdx.x) / H * 2 * H + static_cast<int>(blockIdx.x) % H;
    const int R0 = static_cast<int>(blockIdx.x) / H * 2 * H + H, R1 = R0 + H < nb ? R0 + H : nb;
    if constexpr (MID) {
        __shared__ float W[kJoinMax * 33];
        const int R = R0 + 4 * static_cast<int>(blockIdx.y), Rend = R + 4 < R1 ? R + 4 : R1;
        if (R >= Rend) return;
        if (up)
            tri_mid<true>(n, nb, A, lda, tri, J, R0, R, Rend, W);
        else
            tri_mid<false>(n, nb, A, lda, tri, J, R0, R, Rend, W);
    } else {
        if (R0 >= R1) return;
        if (up)
            tri_fin<true, 8, kJoinMax / 32 / 8>(nb, tri, J, R0, R1);
        else
            tri_fin<false, 8, kJoinMax / 32 / 8>(nb, tri, J, R0, R1);
    }
}

int64_t tri_floats(int b)
{
    const int64_t nb = ceil_div(b, 32);
    return 2 * nb * nb * 1024 + 128;
}

int64_t getrf_scratch_floats(int n) { return n > kLuNB ? tri_floats(n) : 0; }

int launch_getrf(int n, float *A, int64_t lda, int *info, float *tri, bool full, hipStream_t s)
{
    if (n <= 0) return HPLAI_OK;
    for (int k = 0; k < n; k += kLuNB) {
        const int rest = n - k;
        const int rt = (rest + 127) / 128, ct = (rest + 63) / 64;
        const int tiles = k == 0 ? (rest > kLuNB ? 4 : 0) : rt * ct - (ct < 2 ? ct : 2);
        // the whole block's inverses, and the last sub-block's, serve only a caller who asked for them
        const unsigned join = full ? 2 * (k / 32) : 0;
        hipLaunchKernelGGL((lu_update_kernel<true, true>), dim3(static_cast<unsigned>(1 + tiles) + join), dim3(kLuThreads),
                           0, s, n, k, A, lda, !full && rest <= kLuNB ? nullptr : tri, 3, info);
        HPLAI_HIP(hipGetLastError());
        const int strips = rest > kLuNB ? (rest - kLuNB + 31) / 32 : 0;
        const int nd = strips < 4 ? strips : 4;
        if (strips + join > 0) {
            hipLaunchKernelGGL(lu_strip_kernel, dim3(static_cast<unsigned>(2 * strips + nd * nd) + join), dim3(256), 0, s,
                               n, k, A, lda, tri, strips);
            HPLAI_HIP(hipGetLastError());
        }
    }
    return HPLAI_OK;
}

int launch_tri_inverse(int b, const float *LU, int64_t lda, float *tri, int sides, bool join, hipStream_t s)
{
    if (b <= 0) return HPLAI_OK;
    const dim3 g(static_cast<unsigned>(ceil_div(b, kLuNB)));
    if (join)
        hipLaunchKernelGGL((lu_update_kernel<false, true>), g, dim3(kLuThreads), 0, s, b, 0, const_cast<float *>(LU), lda,
                           tri, sides, nullptr);
    else
        hipLaunchKernelGGL((lu_update_kernel<false, false>), g, dim3(kLuThreads), 0, s, b, 0, const_cast<float *>(LU), lda,
                           tri, sides, nullptr);
    HPLAI_HIP(hipGetLastError());
    const int nb = static_cast<int>(ceil_div(b, 32));
    for (int H = kLuNB / 32; join && H < nb; H *= 2) {
        const unsigned cols = static_cast<unsigned>(ceil_div(nb, 2 * H)) * H, z = sides == 3 ? 2 : 1;
        hipLaunchKernelGGL((tri_join_kernel<true>), dim3(cols, H / 4, z), dim3(kLuThreads), 0, s, b, H, LU, lda, tri,
                           sides == 2 ? 1 : 0);
        hipLaunchKernelGGL((tri_join_kernel<false>), dim3(cols, 1, z), dim3(kLuThreads), 0, s, b, H, LU, lda, tri,
                           sides == 2 ? 1 : 0);
        HPLAI_HIP(hipGetLastError());
    }
    return HPLAI_OK;
}

}  // namespace hplai
