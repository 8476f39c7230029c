// trisolve.hip — triangular solves with FP32 factors and FP64 right-hand
// sides: x := L^-1 x, U^-1 x, U^-T x, L^-T x for any number of columns.
//
// Replaces panel_trsvL / panel_trsvU (panel_trsv.hpp:310-758, with tttrsvL/U,
// 115-153, and ttgemv, 10-45): FP32 factor entries widened to FP64, all
// arithmetic in FP64, here on v_mfma_f64_16x16x4_f64.
//
// The rows are walked in blocks of 512.  The diagonal blocks' inverses are
// formed first, all at once and in FP64 (16 -> 256 by block substitution, one
// wave per 16 columns; 256 -> 512 by two products), so that the chain from
// block to block is two launches:
//   tri64_solve_kernel    x_k := T_kk^-1 x_k, a product over many workgroups
//   tri64_update_kernel   x_rest -= T(rest, k) x_k
// What bounds it: that chain, 6 + 13 us a block with 64 columns and 5 + 5 us
// with one (the inverses of both triangles together: 40 + 28 + 23 us at 8192).
// Substitution in one workgroup per block and reading the factors once per
// column took, both triangles, 2707 us at 8192 x 64 (6320 us transposed), now
// 751 (729); 2060 us at 8192 x 1, now 529; 285 us at 1200 x 3, now 120; 9.5 ms
// at 30000 x 1, now 2.8.
// A product with an inverse has the error of substitution times the condition
// of the 512 x 512 block.  So each block's condition, a bound of the largest row
// sum of |T_kk^-1| |T_kk|, is formed with its inverse, by workgroups and registers
// that have the operands anyway (2 us at 1200, 9 at 8192; a kernel of its own took
// 8 and 22), and a block past kTsCond is solved by substitution instead
// (tri64_substitute): all blocks so, 2.5 ms at 8192 x 64 (3.4 transposed), 2.3 at
// 8192 x 1, 0.37 at 1200 x 3, bound by the triangle's way into one CU.
//
// An upper triangle is a lower one with rows and columns taken from the end;
// TriView numbers entries that way, so the kernels only know lower ones.
#include "device_common.hpp"
#include "internal.hpp"

namespace hplai {

typedef double doublex4s_t __attribute__((ext_vector_type(4)));

constexpr int kTsBlock = 512, kTsHalf = 256;
constexpr int kTsInv = 32 * 32 * 256;     // doubles of one block's inverse, 16 x 16 tiles (I, K) of 256
constexpr int kTsMid = 16 * 16 * 256;     // doubles of one block's intermediate product
constexpr int kTsGroup = 32;              // blocks inverted at a time (96 MiB a triangle)
constexpr int kTsCols = 1024;             // right-hand sides at a time
// doubles of one block's condition: row sums of |A|, of |B|, its mark, and from
// kTsPart the parts of |C A^-1| |A| and of |C| for row r of the second half at J 256 + r, J < 16 and 16
constexpr int kTsPart = kTsBlock + 16, kTsRow = kTsPart + 17 * kTsHalf;
// Largest condition that is solved through the inverse.  Errors of inverse /
// substitution (FP64, order 512, b = T x): condition 3.6 (factors of HPL-AI
// matrices) 1.2e-16 / 1.2e-16 of the solution, 18 1.5e-16 / 1.3e-16, 54 3.5e-16
// / 1.4e-16, 3e2 2.7e-15 / 4.8e-16, 6e5 2.6e-8 / 1.1e-12.
constexpr double kTsCond = 16.0;

// MFMA layout: left operand lane -> (row lane % 16, k lane / 16), right operand
// lane -> (k lane / 16, column lane % 16), result q -> (row lane / 16 + 4 q,
// column lane % 16).  A tile of an inverse is stored in left-operand order,
// [lane 4 + t] = (row lane % 16, column 4 t + lane / 16).
__device__ __forceinline__ int tile_pos(int row, int col) { return ((col & 3) * 16 + row) * 4 + (col >> 2); }

template <bool UPPER, bool TRANS>
struct TriView {
    const float *LU;
    int64_t lda, n;
    static constexpr bool kUnit = UPPER == TRANS;   // L has the unit diagonal
    __device__ __forceinline__ int64_t index(int64_t i) const { return UPPER ? n - 1 - i : i; }
    __device__ __forceinline__ const float *ptr(int64_t i, int64_t j) const
    {
        return TRANS ? LU + index(i) * lda + index(j) : LU + index(j) * lda + index(i);
    }
    // entry (i, j), i and j clamped to the matrix: rows and columns past the
    // end are multiplied by zeros or dropped
    __device__ __forceinline__ double at(int64_t i, int64_t j) const
    {
        return static_cast<double>(*ptr(min(i, n - 1), min(j, n - 1)));
    }
};

// Inverses of the 256 x 256 diagonal blocks.  blockIdx.x: block; a wave owns
// the 16 columns of tile column J = 4 wave + blockIdx.y and walks down:
//   V_I = -Dinv_I sum_{K < I} E(I, K) V_K   (V_J = Dinv_J, V_K = 0 above)
// with V_K in its registers, whose layout is that of a right operand.  Row I
// of E is staged in LDS for the four waves while row I - 1 is used.
// bop: V of the blocks' first halves once more, in right-operand order.
struct TsInvLds {
    double D[16][16][17];     // diagonal tiles
    double rd[16][16];        // reciprocals of their diagonals
    double P[16][256];        // their inverses, packed
    float R[2][240 * 17];     // E(I, :) of two rows of tiles, R[col * 17 + row]
    double sum[16][257];      // each thread's part of the row sums of |E(I, :)|
};

template <bool UPPER, bool TRANS>
__device__ __forceinline__ void tri64_inv(const TriView<UPPER, TRANS> &E, int64_t first, double *__restrict__ inv,
                                          double *__restrict__ bop, double *__restrict__ rows, TsInvLds &sm)
{
    auto &D = sm.D;
    auto &P = sm.P;
    auto &R = sm.R;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lk = lane >> 4;
    const int64_t e0 = first + static_cast<int64_t>(blockIdx.x) * kTsHalf;
    if (e0 >= E.n) return;
    // consecutive threads along the contiguous direction of the factor
    float rv[15];
    auto fetch = [&](int I) {
#pragma unroll
        for (int u = 0; u < 15; ++u)
            if (u < I) {
                const int r = TRANS ? tid >> 4 : tid & 15, c = 16 * u + (TRANS ? tid & 15 : tid >> 4);
                rv[u] = *E.ptr(min(e0 + 16 * I + r, E.n - 1), min(e0 + c, E.n - 1));
            }
    };
    auto stage = [&](int I) {
        double part = 0.0;
#pragma unroll
        for (int u = 0; u < 15; ++u)
            if (u < I) {
                const int r = TRANS ? tid >> 4 : tid & 15, c = 16 * u + (TRANS ? tid & 15 : tid >> 4);
                R[I & 1][c * 17 + r] = rv[u];
                part += fabs(static_cast<double>(rv[u]));
            }
        sm.sum[I][tid] = part;
    };
    fetch(1);
    {
        const int r = TRANS ? tid >> 4 : tid & 15, c = TRANS ? tid & 15 : tid >> 4;
        float dv[16];
#pragma unroll
        for (int T = 0; T < 16; ++T)
            dv[T] = *E.ptr(min(e0 + 16 * T + r, E.n - 1), min(e0 + 16 * T + c, E.n - 1));
#pragma unroll
        for (int T = 0; T < 16; ++T) {
            const int64_t i = e0 + 16 * T + r, j = e0 + 16 * T + c;
            double v = r >= c ? static_cast<double>(dv[T]) : 0.0;
            if (i >= E.n || j >= E.n || (r == c && TriView<UPPER, TRANS>::kUnit)) v = r == c ? 1.0 : 0.0;
            D[T][r][c] = v;
        }
    }
    stage(1);
    __syncthreads();
    sm.rd[tid >> 4][tid & 15] = 1.0 / D[tid >> 4][tid & 15][tid & 15];
    __syncthreads();
    {   // lane: column l16 of the inverse of tile 4 wave + lk
        const int T = 4 * wave + lk;
        double x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            double s = i == l16 ? 1.0 : 0.0;
#pragma unroll
            for (int k = 0; k < i; ++k) s = fma(-D[T][i][k], x[k], s);
            x[i] = s * sm.rd[T][i];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) P[T][tile_pos(i, l16)] = x[i];
    }
    const int J = 4 * wave + static_cast<int>(blockIdx.y);
    // tile (I, J) of this 256-block inside its 512-block's array
    const int64_t h = e0 / kTsHalf - first / kTsHalf;
    double *out = inv + (h >> 1) * kTsInv + ((h & 1) * 16 * 32 + (h & 1) * 16) * 256;
    double *bo = bop + (h >> 1) * kTsMid;
    doublex4s_t V[16];
#pragma unroll
    for (int I = 0; I < 16; ++I) {
        __syncthreads();   // row I is staged, row I - 1 no longer read
        if (I > 0 && I < 15) fetch(I + 1);
        // operands first, two sums: neither the LDS nor a product's latency between products
        float a[15][4];
#pragma unroll
        for (int K = 0; K < I; ++K)
#pragma unroll
            for (int t = 0; t < 4; ++t) a[K][t] = R[I & 1][(16 * K + 4 * t + lk) * 17 + l16];
        double pv[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) pv[t] = P[I][lane * 4 + t];
        __builtin_amdgcn_sched_barrier(0);
        doublex4s_t T = {0.0, 0.0, 0.0, 0.0}, T1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int K = 0; K < I; ++K)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t & 1)
                    T1 = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a[K][t]), V[K][t], T1, 0, 0, 0);
                else
                    T = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a[K][t]), V[K][t], T, 0, 0, 0);
            }
#pragma unroll
        for (int t = 0; t < 4; ++t) T[t] += T1[t];
        doublex4s_t Q = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int t = 0; t < 4; ++t)
            Q = __builtin_amdgcn_mfma_f64_16x16x4f64(pv[t], T[t], Q, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double d = P[I][tile_pos(lk + 4 * q, l16)];
            V[I][q] = I < J ? 0.0 : I == J ? d : -Q[q];
        }
        if (I >= J)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                out[(I * 32 + J) * 256 + tile_pos(lk + 4 * q, l16)] = V[I][q];
                if ((h & 1) == 0) bo[(I * 16 + J) * 256 + q * 64 + lane] = V[I][q];
            }
        if (I > 0 && I < 15) stage(I + 1);
    }
    if (blockIdx.y != 0) return;
    // row sums of |E|, a row per thread, zeros past the end
    __syncthreads();
    const int I = tid >> 4, r = tid & 15;
    double s = 0.0;
#pragma unroll
    for (int c = 0; c < 16; ++c) s += fabs(D[I][r][c]);
    if (I > 0)
#pragma unroll
        for (int c = 0; c < 16; ++c) s += sm.sum[I][TRANS ? 16 * r + c : 16 * c + r];
    double *row = rows + (h >> 1) * kTsRow;
    row[(h & 1) * kTsHalf + tid] = e0 + tid < E.n ? s : 0.0;
    if ((h & 1) == 0 && tid == 0) row[kTsBlock] = 0.0;
}

// blockIdx.z (+ upper0): the lower or the upper triangle of the pair that one
// lu_solve needs; z2: doubles from the first's scratch to the second's
template <bool TRANS>
__global__ __launch_bounds__(256) void tri64_inv_kernel(const float *__restrict__ LU, int64_t lda, int64_t n,
                                                        int64_t first, int upper0, double *__restrict__ inv,
                                                        double *__restrict__ bop, double *__restrict__ rows, int64_t z2)
{
    __shared__ TsInvLds sm;
    inv += blockIdx.z * z2;
    bop += blockIdx.z * z2;
    rows += blockIdx.z * z2;
    if ((upper0 + static_cast<int>(blockIdx.z)) & 1)
        tri64_inv(TriView<true, TRANS>{LU, lda, n}, first, inv, bop, rows, sm);
    else
        tri64_inv(TriView<false, TRANS>{LU, lda, n}, first, inv, bop, rows, sm);
}

// 256 -> 512: the lower left quarter -B^-1 C A^-1.  MID: tile (I, J) of
// M = C A^-1 to mid in right-operand order [q 64 + lane], and the tile's parts of
// the row sums of |M| |A| and |C|; else of -B^-1 mid.
template <bool UPPER, bool TRANS, bool MID>
__device__ __forceinline__ void tri64_merge(const TriView<UPPER, TRANS> &E, int64_t first, double *__restrict__ inv,
                                            const double *__restrict__ bop, double *__restrict__ mid,
                                            double *__restrict__ rows)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lk = lane >> 4;
    const int64_t e0 = first + static_cast<int64_t>(blockIdx.x) * kTsBlock;
    if (e0 + kTsHalf >= E.n) return;
    const int tile = static_cast<int>(blockIdx.y) * 4 + wave, I = tile >> 4, J = tile & 15;
    double *bi = inv + static_cast<int64_t>(blockIdx.x) * kTsInv, *m = mid + static_cast<int64_t>(blockIdx.x) * kTsMid;
    const double *bo = bop + static_cast<int64_t>(blockIdx.x) * kTsMid;
    double *row = rows + static_cast<int64_t>(blockIdx.x) * kTsRow;
    double w = 0.0, cs = 0.0;
    if (MID) w = row[16 * J + l16];
    // four tiles' operands in flight; steps past the end take zeros
    const int K0 = MID ? J : 0, K1 = MID ? 16 : I + 1;
    const int64_t i = min(e0 + kTsHalf + 16 * I + l16, E.n - 1);
    doublex4s_t T = {0.0, 0.0, 0.0, 0.0};
    for (int K = K0; K < K1; K += 4) {
        double a[4][4], b[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = K + u < K1 ? K + u : K1 - 1;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if constexpr (MID) {
                    // K of a step: 4 t + lk, or 4 lk + t where that is contiguous for a lane
                    a[u][t] = static_cast<double>(*E.ptr(i, e0 + 16 * k + (TRANS ? 4 * lk + t : 4 * t + lk)));
                    b[u][t] = bo[(k * 16 + J) * 256 + (TRANS ? lk * 64 + t * 16 + l16 : t * 64 + lane)];
                } else {
                    a[u][t] = bi[((16 + I) * 32 + 16 + k) * 256 + lane * 4 + t];
                    b[u][t] = m[(k * 16 + J) * 256 + t * 64 + lane];
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (K + u < K1)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    T = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][t], b[u][t], T, 0, 0, 0);
                    if (MID && J == 0) cs += fabs(a[u][t]);
                }
    }
    // rows past the end hold copies of the last: dropped with the rows of the inverse below them
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if constexpr (MID)
            m[(I * 16 + J) * 256 + q * 64 + lane] = T[q];
        else
            bi[((16 + I) * 32 + J) * 256 + tile_pos(lk + 4 * q, l16)] = -T[q];
    }
    if constexpr (MID) {
        double v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = fabs(T[q]) * w;
#pragma unroll
        for (int off = 1; off < 16; off *= 2)
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += __shfl_xor(v[q], off);
        if (l16 == 0)
#pragma unroll
            for (int q = 0; q < 4; ++q) row[kTsPart + J * kTsHalf + 16 * I + lk + 4 * q] = v[q];
        if (J == 0) {
            cs += __shfl_xor(cs, 16);
            cs += __shfl_xor(cs, 32);
            if (lane < 16) row[kTsPart + 16 * kTsHalf + 16 * I + lane] = cs;
        }
    }
}

// Marks the 512-block where a row sum of |A^-1| |A|, or of |B^-1| (|C A^-1| |A| +
// |B| + |C|), which bounds the second half's of |T^-1| |T|, is past kTsCond or no
// number.  Row tile blockIdx.y - 64; the four waves split K.  left: rows of the
// matrix from the group's first.
__device__ __forceinline__ void tri64_mark(int64_t left, const double *__restrict__ inv, double *rows, double *u,
                                           double (&red)[4][16])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lk = lane >> 4;
    const double *bi = inv + static_cast<int64_t>(blockIdx.x) * kTsInv;
    double *row = rows + static_cast<int64_t>(blockIdx.x) * kTsRow;
    const int tile = static_cast<int>(blockIdx.y) - 64, h = tile >> 4, I = tile & 15;
    const int64_t over = left - static_cast<int64_t>(blockIdx.x) * kTsBlock;
    const int w = over < kTsBlock ? static_cast<int>(over) : kTsBlock;
    if (16 * tile >= w) return;
    if (tid < 16 * (I + 1)) {
        double s = row[kTsHalf * h + tid];
        if (h != 0) {
            double p[17];
#pragma unroll
            for (int J = 0; J < 17; ++J) p[J] = row[kTsPart + J * kTsHalf + tid];
#pragma unroll
            for (int J = 0; J < 17; ++J) s += p[J];
        }
        u[tid] = s;
    }
    double a[4][4];   // K = wave + 4 q
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int t = 0; t < 4; ++t) a[q][t] = bi[(tile * 32 + 16 * h + min(wave + 4 * q, I)) * 256 + lane * 4 + t];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (wave + 4 * q <= I)
#pragma unroll
            for (int t = 0; t < 4; ++t) s = fma(fabs(a[q][t]), u[16 * (wave + 4 * q) + 4 * t + lk], s);
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if (lane < 16) red[wave][lane] = s;
    __syncthreads();
    if (wave == 0) {
        s = ((red[0][l16] + red[1][l16]) + red[2][l16]) + red[3][l16];
        if (__any(16 * tile + l16 < w && !(s <= kTsCond)) && lane == 0) row[kTsBlock] = 1.0;
    }
}

// without MID also the marks (blockIdx.y from 64 on)
template <bool TRANS, bool MID>
__global__ __launch_bounds__(256) void tri64_merge_kernel(const float *__restrict__ LU, int64_t lda, int64_t n,
                                                          int64_t first, int upper0, double *__restrict__ inv,
                                                          const double *__restrict__ bop, double *__restrict__ mid,
                                                          double *__restrict__ rows, int64_t z2)
{
    __shared__ double u[kTsHalf], red[4][16];
    inv += blockIdx.z * z2;
    bop += blockIdx.z * z2;
    mid += blockIdx.z * z2;
    rows += blockIdx.z * z2;
    if (!MID && blockIdx.y >= 64)
        tri64_mark(n - first, inv, rows, u, red);
    else if ((upper0 + static_cast<int>(blockIdx.z)) & 1)
        tri64_merge<true, TRANS, MID>(TriView<true, TRANS>{LU, lda, n}, first, inv, bop, mid, rows);
    else
        tri64_merge<false, TRANS, MID>(TriView<false, TRANS>{LU, lda, n}, first, inv, bop, mid, rows);
}

// Position of entry (k, column c) in the solved block's array: 16 x 16 tiles
// of a column block in right-operand order, [lane 4 + t].  The K of one MFMA
// step is 4 t + lane / 16, or, where a lane reads its four K's from
// consecutive addresses of the transposed factor, 4 (lane / 16) + t.
template <bool TRANS>
__device__ __forceinline__ int64_t solved_pos(int k, int c)
{
    const int g = k & 15;
    const int lane = (TRANS ? g >> 2 : g & 3) * 16 + (c & 15), t = TRANS ? g & 3 : g >> 2;
    return (static_cast<int64_t>(c >> 4) * 32 + (k >> 4)) * 256 + lane * 4 + t;
}

__device__ __forceinline__ double readlane64(double v, int lane)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// One column of T_kk^-1 x_k by substitution, 256 threads, rows tid and tid + 256
// in registers.  The 16 rows of a tile are solved in the wave that owns them
// (x_c by v_readlane, diagonals as reciprocals), the rows further on subtract
// the tile's 16 columns, loaded a tile ahead.  A barrier a tile: the parts of xs take turns.
template <bool UPPER, bool TRANS>
__device__ __forceinline__ void tri64_substitute(const TriView<UPPER, TRANS> &E, int64_t kb, const double *x, double *xt,
                                                 int col, double (&xs)[2][16])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int w = E.n - kb < kTsBlock ? static_cast<int>(E.n - kb) : kTsBlock;
    double xr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) xr[q] = x[E.index(min(kb + tid + 256 * q, E.n - 1))];
    __syncthreads();   // xs: the column before
    float t[2][16], next[2][16];
    auto load = [&](float (&v)[2][16], int c0) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (256 * q + 64 * wave + 63 >= c0)   // rows that the tile reaches
#pragma unroll
                for (int c = 0; c < 16; ++c)
                    v[q][c] = *E.ptr(min(kb + tid + 256 * q, E.n - 1), min(kb + c0 + c, E.n - 1));
    };
    load(t, 0);
    for (int s0 = 0; s0 < w; s0 += 16) {
        double *part = xs[(s0 >> 4) & 1];
        if (s0 + 16 < w) load(next, s0 + 16);
        auto diagonal = [&](const float (&a)[16], double &x) {
            const int i = lane - (s0 & 63);   // row s0 + i for 0 <= i < 16
            double v = x, rinv = 1.0;
            if (!TriView<UPPER, TRANS>::kUnit) {
                float d = 1.0f;
#pragma unroll
                for (int c = 0; c < 16; ++c) d = c == i ? a[c] : d;
                rinv = 1.0 / static_cast<double>(d);
            }
#pragma unroll
            for (int c = 0; c < 16; ++c) {
                if (s0 + c >= w) break;
                if (!TriView<UPPER, TRANS>::kUnit && i == c) v *= rinv;
                const double xc = readlane64(v, (s0 & 63) + c);
                if (i > c && i < 16) v = fma(-static_cast<double>(a[c]), xc, v);
            }
            if (i >= 0 && i < 16) {
                part[i] = v;
                x = v;
            }
        };
        if (wave == (s0 & 255) >> 6) {
            if (s0 < 256)
                diagonal(t[0], xr[0]);
            else
                diagonal(t[1], xr[1]);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (tid + 256 * q >= s0 + 16) {
                double acc = 0.0;
#pragma unroll
                for (int c = 0; c < 16; ++c) acc = fma(static_cast<double>(t[q][c]), part[c], acc);
                xr[q] -= acc;
            }
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int c = 0; c < 16; ++c) t[q][c] = next[q][c];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (tid + 256 * q < w) xt[solved_pos<TRANS>(tid + 256 * q, col)] = xr[q];
}

// Rows 16 I .. + 15 (blockIdx.x) of T_kk^-1 x_k for 16 columns (blockIdx.y) to
// xt.  The four waves split K and are added in order.  A marked block: the
// workgroups take a column each instead.
template <bool UPPER, bool TRANS>
__global__ __launch_bounds__(256) void tri64_solve_kernel(TriView<UPPER, TRANS> E, int64_t kb,
                                                          const double *__restrict__ inv, const double *__restrict__ mark,
                                                          const double *__restrict__ X, int64_t ldx, int nrhs,
                                                          double *__restrict__ xt)
{
    __shared__ double red[3][4][64];
    __shared__ double xs[2][16];
    const double marked = *mark;   // asked for after the product's loads
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, lk = lane >> 4;
    const int I = static_cast<int>(blockIdx.x), c0 = static_cast<int>(blockIdx.y) * 16;
    const double *xc = X + static_cast<int64_t>(min(c0 + l16, nrhs - 1)) * ldx;
    doublex4s_t acc = {0.0, 0.0, 0.0, 0.0};
    // at most eight tiles per wave, four tiles' operands in flight
    for (int K = wave; K <= I; K += 16) {
        double a[4][4], b[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = K + 4 * u <= I ? K + 4 * u : I;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int64_t r = kb + 16 * k + 4 * t + lk;
                a[u][t] = inv[(I * 32 + k) * 256 + lane * 4 + t];
                b[u][t] = xc[E.index(min(r, E.n - 1))];
                if (r >= E.n) b[u][t] = 0.0;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (K + 4 * u <= I) {
                if (K + 4 * u == I &&
                    __any(!(isfinite(b[u][0]) && isfinite(b[u][1]) && isfinite(b[u][2]) && isfinite(b[u][3])))) {
                    // the zeros above the diagonal would carry it to the rows before
                    for (int g = 0; g < 16; ++g) {
                        const double bt = (g >> 2) == 0   ? b[u][0]
                                          : (g >> 2) == 1 ? b[u][1]
                                          : (g >> 2) == 2 ? b[u][2]
                                                          : b[u][3];
                        const double x = __shfl(bt, (g & 3) * 16 + l16);
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            if (g <= lk + 4 * q)
                                acc[q] = fma(inv[(I * 32 + I) * 256 + tile_pos(lk + 4 * q, g)], x, acc[q]);
                    }
                    continue;
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u][t], b[u][t], acc, 0, 0, 0);
            }
    }
    if (marked != 0.0) {
        for (int c = static_cast<int>(blockIdx.x); c < 16 && c0 + c < nrhs; c += static_cast<int>(gridDim.x))
            tri64_substitute(E, kb, X + static_cast<int64_t>(c0 + c) * ldx, xt, c0 + c, xs);
        return;
    }
    if (wave > 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave - 1][q][lane] = acc[q];
    __syncthreads();
    if (wave == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xt[solved_pos<TRANS>(16 * I + lk + 4 * q, c0 + l16)] =
                ((acc[q] + red[0][q][lane]) + red[1][q][lane]) + red[2][q][lane];
}

// x_rest -= T(rest, k) x_k, a workgroup per 16 RB rows and 16 CB columns; the
// first 16 CB workgroups move x_k from xt into X instead.  Four waves for each
// 16 rows split K (added in order), each with 8 / CB groups of 16 in flight
// and as many being used.  One block of columns is bound by reading the factor,
// 32 rows (whole cache lines of its columns) a workgroup; with four the
// right-hand sides' operands outweigh it and 16 rows leave more workgroups.
template <bool UPPER, bool TRANS, int CB, int RB>
__global__ __launch_bounds__(256 * RB) void tri64_update_kernel(TriView<UPPER, TRANS> E, int64_t kb, int w,
                                                           const double *__restrict__ xt, double *__restrict__ X,
                                                           int64_t ldx, int nrhs)
{
    constexpr int GW = kTsBlock / 16 / 4, PB = 8 / CB;   // groups per wave, per batch
    __shared__ double red[RB][4][CB * 4][64];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = wv >> 2, wave = wv & 3;
    const int l16 = lane & 15, lk = lane >> 4;
    const int c0 = static_cast<int>(blockIdx.y) * 16 * CB;
    if (static_cast<int>(blockIdx.x) < 16 * CB) {   // a column of the solved block
        const int c = c0 + static_cast<int>(blockIdx.x);
        if (c < nrhs)
#pragma unroll
            for (int k = tid; k < kTsBlock; k += 256 * RB)
                if (k < w) X[static_cast<int64_t>(c) * ldx + E.index(kb + k)] = xt[solved_pos<TRANS>(k, c)];
        return;
    }
    const int64_t i0 = kb + kTsBlock + (static_cast<int64_t>(blockIdx.x - 16 * CB) * RB + rb) * 16;
    const int64_t row = min(i0 + l16, E.n - 1);
    // wave w finishes column block w
    const int cw = c0 + 16 * wave + l16;
    double xv[4];
    if (wave < CB)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            xv[q] = X[static_cast<int64_t>(min(cw, nrhs - 1)) * ldx + E.index(min(i0 + lk + 4 * q, E.n - 1))];
    const double *bp = xt + static_cast<int64_t>(c0 >> 4) * 32 * 256 + lane * 4;
    doublex4s_t acc[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) acc[c] = doublex4s_t{0.0, 0.0, 0.0, 0.0};
    float a[2][PB][4];
    double b[2][PB][CB][4];
    auto load = [&](int h, int g0) {
#pragma unroll
        for (int u = 0; u < PB; ++u) {
            const int kg = GW * wave + g0 + u;
#pragma unroll
            for (int t = 0; t < 4; ++t) a[h][u][t] = *E.ptr(row, kb + 16 * kg + (TRANS ? 4 * lk + t : 4 * t + lk));
#pragma unroll
            for (int c = 0; c < CB; ++c)
#pragma unroll
                for (int t = 0; t < 4; ++t) b[h][u][c][t] = bp[(c * 32 + kg) * 256 + t];
        }
    };
    load(0, 0);
#pragma unroll
    for (int g = 0; g < GW; g += PB) {
        const int h = (g / PB) & 1;
        if (g + PB < GW) load(h ^ 1, g + PB);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < PB; ++u)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a[h][u][t]), b[h][u][c][t],
                                                                  acc[c], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[rb][wave][c * 4 + q][lane] = acc[c][q];
    __syncthreads();
    if (wave >= CB || cw >= nrhs) return;
    double *xc = X + static_cast<int64_t>(cw) * ldx;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int64_t i = i0 + lk + 4 * q;
        const int e = wave * 4 + q;
        const double sum = ((red[rb][0][e][lane] + red[rb][1][e][lane]) + red[rb][2][e][lane]) + red[rb][3][e][lane];
        if (i < E.n) xc[E.index(i)] = xv[q] - sum;
    }
}

static int64_t tri_group(int64_t n)
{
    const int64_t blocks = ceil_div(n, kTsBlock);
    return blocks < kTsGroup ? blocks : kTsGroup;
}
static int64_t tri_inv_doubles(int64_t n) { return tri_group(n) * (kTsInv + 2 * kTsMid + kTsRow); }
static double *tri_rows(int64_t n, double *inv) { return inv + tri_group(n) * (kTsInv + 2 * kTsMid); }

// both triangles' inverses fit beside each other where one group holds all
int64_t tri_solve_work_doubles(int64_t n, int nrhs)
{
    const int64_t cols = nrhs < kTsCols ? ceil_div(nrhs, 64) * 64 : kTsCols;
    return (ceil_div(n, kTsBlock) <= kTsGroup ? 2 : 1) * tri_inv_doubles(n) + cols * kTsBlock;
}

// Inverses of a group's diagonal blocks, of one triangle or of both.
template <bool TRANS>
static int tri_invert(bool upper, bool both, int64_t n, int64_t first, const float *LU, int64_t lda, double *inv,
                      hipStream_t s)
{
    const int64_t g = tri_group(n), left = ceil_div(n - first, kTsBlock);
    const unsigned gc = static_cast<unsigned>(left < g ? left : g), z = both ? 2 : 1;
    double *mid = inv + g * kTsInv, *bop = mid + g * kTsMid, *rows = tri_rows(n, inv);
    const int64_t z2 = tri_inv_doubles(n);
    hipLaunchKernelGGL((tri64_inv_kernel<TRANS>), dim3(2 * gc, 4, z), dim3(256), 0, s, LU, lda, n, first,
                       upper ? 1 : 0, inv, bop, rows, z2);
    if (n - first > kTsHalf)
        hipLaunchKernelGGL((tri64_merge_kernel<TRANS, true>), dim3(gc, 64, z), dim3(256), 0, s, LU, lda, n, first,
                           upper ? 1 : 0, inv, bop, mid, rows, z2);
    hipLaunchKernelGGL((tri64_merge_kernel<TRANS, false>), dim3(gc, 96, z), dim3(256), 0, s, LU, lda, n, first,
                       upper ? 1 : 0, inv, bop, mid, rows, z2);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

// inv: the inverses of all blocks are there already (ready), or room for a group's
template <bool UPPER, bool TRANS>
static int tri_solve(int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs, double *inv, bool ready,
                     double *xt, hipStream_t s)
{
    const TriView<UPPER, TRANS> E{LU, lda, n};
    const int64_t blocks = ceil_div(n, kTsBlock), group = tri_group(n);
    for (int64_t q = 0; q < blocks; ++q) {
        if (!ready && q % group == 0) {
            const int rc = tri_invert<TRANS>(UPPER, false, n, q * kTsBlock, LU, lda, inv, s);
            if (rc) return rc;
        }
        const int64_t kb = q * kTsBlock, rest = n - kb - kTsBlock;
        const int w = n - kb < kTsBlock ? static_cast<int>(n - kb) : kTsBlock;
        const unsigned rows = static_cast<unsigned>(rest > 0 ? ceil_div(rest, 32) : 0);
        for (int c = 0; c < nrhs; c += kTsCols) {
            const int nc = nrhs - c < kTsCols ? nrhs - c : kTsCols;
            double *Xc = X + static_cast<int64_t>(c) * ldx;
            hipLaunchKernelGGL((tri64_solve_kernel<UPPER, TRANS>),
                               dim3(static_cast<unsigned>((w + 15) / 16), static_cast<unsigned>((nc + 15) / 16)),
                               dim3(256), 0, s, E, kb, inv + (q % group) * kTsInv,
                               tri_rows(n, inv) + (q % group) * kTsRow + kTsBlock, Xc, ldx, nc, xt);
            if (nc <= 16)
                hipLaunchKernelGGL((tri64_update_kernel<UPPER, TRANS, 1, 2>), dim3(16 + rows, 1), dim3(512), 0, s, E, kb,
                                   w, xt, Xc, ldx, nc);
            else if (nc <= 32)
                hipLaunchKernelGGL((tri64_update_kernel<UPPER, TRANS, 2, 2>), dim3(32 + rows, 1), dim3(512), 0, s, E, kb,
                                   w, xt, Xc, ldx, nc);
            else
                hipLaunchKernelGGL((tri64_update_kernel<UPPER, TRANS, 4, 1>),
                                   dim3(64 + 2 * rows, static_cast<unsigned>((nc + 63) / 64)), dim3(256), 0, s, E, kb,
                                   w, xt, Xc, ldx, nc);
            HPLAI_HIP(hipGetLastError());
        }
    }
    return HPLAI_OK;
}

template <bool TRANS>
static int tri_solve_side(bool upper, int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs,
                          double *inv, bool ready, double *xt, hipStream_t s)
{
    // the rows of op(T) run upwards for U and for L^T
    return upper != TRANS ? tri_solve<true, TRANS>(n, LU, lda, X, ldx, nrhs, inv, ready, xt, s)
                          : tri_solve<false, TRANS>(n, LU, lda, X, ldx, nrhs, inv, ready, xt, s);
}

int launch_tri_solve(bool upper, int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs,
                     double *work, hipStream_t s)
{
    if (n <= 0 || nrhs <= 0) return HPLAI_OK;
    return tri_solve_side<false>(upper, n, LU, lda, X, ldx, nrhs, work, false, work + tri_inv_doubles(n), s);
}

template <bool TRANS>
static int lu_solve(int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs, double *work,
                    hipStream_t s)
{
    // the first triangle's walk is lower in TriView's numbering either way:
    // L, or U^T
    const bool both = ceil_div(n, kTsBlock) <= kTsGroup;
    double *inv2 = both ? work + tri_inv_doubles(n) : work, *xt = inv2 + tri_inv_doubles(n);
    int rc = both ? tri_invert<TRANS>(false, true, n, 0, LU, lda, work, s) : HPLAI_OK;
    if (rc == HPLAI_OK) rc = tri_solve_side<TRANS>(TRANS, n, LU, lda, X, ldx, nrhs, work, both, xt, s);
    if (rc == HPLAI_OK) rc = tri_solve_side<TRANS>(!TRANS, n, LU, lda, X, ldx, nrhs, inv2, both, xt, s);
    return rc;
}

// A = L U: L then U; A^T = U^T L^T: U^T then L^T
int launch_lu_solve(bool trans, int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs,
                    double *work, hipStream_t s)
{
    if (n <= 0 || nrhs <= 0) return HPLAI_OK;
    return trans ? lu_solve<true>(n, LU, lda, X, ldx, nrhs, work, s)
                 : lu_solve<false>(n, LU, lda, X, ldx, nrhs, work, s);
}

}  // namespace hplai
