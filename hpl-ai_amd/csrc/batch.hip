// batch.hip — many independent HPL-AI systems of uneven sizes (n <= 1024,
// 1-4 right-hand sides) solved by one persistent launch.
//
// No reference counterpart: the reference solves one system per run.  Each
// system applies the reference's arithmetic to its own matrix: the LCG matrix
// of hpl_rand.hpp (element (i,j) = state 1+i+n*j from the system's seed,
// diagonal = FP64 row sum of |a_ij|, rhs r = column n+r of the stream), an
// unpivoted LU with FP32 panels and an FP16 Schur update with FP32 accumulation
// (the reference's plain method), and FP64 iterative refinement to HPL-AI
// harness < 16 (iterative_refinement.hpp:18-57) against the FP64 matrix, for
// every right-hand side.
//
// Scheduling: the grid is a fixed number of workgroups (one per CU); each
// workgroup takes the next system from a device counter (one vector atomic by
// one thread) until the list is exhausted, largest systems first.  One
// workgroup owns one system: generation, LU and refinement run without any
// grid-wide synchronisation, and every workgroup leaves the loop once the
// counter passes the end.  1024 threads: a row of the matrix each.
//
// LU of one system: left-looking, a block of 32 columns at a time in LDS (n x
// 32 FP32), so that the matrix is read and written once and the FP16 L about
// n / 64 times.  Right-looking, with the trailing matrix in memory after each of
// the 64 panels of 16 columns that LDS then held, 256 systems of 1024 moved 45
// GB.  What bounds it now: the chain of 32 x 32 blocks and the reads of L.
// 256 systems, us each, before / now: order 1024 15188 / 3570 (update 7855 /
// 1431, panels 1646 / 328, U 1545 / in the update, generation 978 / 148,
// residuals 1493 / 358, triangular solves 1153 / 460), 512 3045 / 1060, 200 672 /
// 370, 64 258 / 180; 1024 systems of 32 .. 1024: 20.7 -> 5.9 ms.
// Joining a step's norms and leaving out waves without rows (batch_norms) took
// that to 5.7 ms, and 256 systems with 1 to 4 right-hand sides of order 64 from
// 181 to 141 us, 200 513 to 445, 512 1415 to 1312 (1024: 4060, the same).
#include <algorithm>
#include <cfloat>
#include <chrono>
#include <type_traits>
#include <vector>

#include "device_common.hpp"
#include "internal.hpp"
#include "lu32.hpp"

namespace hplai {

typedef _Float16 half8b_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4b_t __attribute__((ext_vector_type(4)));
typedef float floatx16b_t __attribute__((ext_vector_type(16)));

constexpr int kBT = 1024;                 // threads per workgroup: a row each
constexpr int kBatchMaxN = 1024;
constexpr int kNB = 32;                   // panel width; nb = 64 takes two as one, nb = 16 runs as 32
constexpr int kBuckets = 4;               // [32,128) [128,256) [256,512) [512,1024]

struct BatchSys {
    int32_t n, nrhs, nb, lda;             // lda = n rounded up to 4 (16-byte row groups)
    uint64_t x1;                          // lcg_init(seed)
    int64_t a32, d, b, x, r, lh;          // offsets into the float / double / FP16 pools
    LcgCoeff col;                         // n steps of the generator: the next entry of a row
};

struct BatchOut {
    double harness[4];
    int32_t steps[4];
    int32_t info;                         // 0, or k+1 for the first zero / non-finite pivot
    int32_t pad;
    uint64_t t0, t1;                      // wall clock at start / end of the system
};

// The thread's number, as a value of the place that asks for it: what is
// computed from it in one phase is then not kept in registers, or spilled,
// through all others of the workgroup's loop over systems.
__device__ __forceinline__ int own_tid()
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

__device__ __forceinline__ double block_max(double v, double *red)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off));
    if (lane == 0) red[wave] = v;
    __syncthreads();
    double r = red[0];
#pragma unroll
    for (int q = 1; q < kBT / 64; ++q) r = fmax(r, red[q]);
    __syncthreads();
    return r;
}

// ---- generation: A32 = (float)a_ij with (float)d on the diagonal, d, and the
// right-hand sides (stream columns n .. n + nrhs - 1).  A thread walks a row;
// d is its sum of |a_ij|, j ascending, j != i (calc_diag,
// hpl_rand.hpp:108-123).  The FP64 matrix is not kept: 8 MB a pass and
// workgroup from memory take longer than generating them again. ----
__device__ __forceinline__ void batch_generate(const BatchSys &S, float *A32, double *d, double *B)
{
    const int n = S.n, lda = S.lda, tid = own_tid();
    if (const int i = tid; i < n) {
        uint64_t s = lcg_jump(S.x1, static_cast<uint64_t>(i));
        float *row = A32 + i;
        double sum = 0.0;
#pragma unroll 4
        for (int j = 0; j < n; ++j) {
            const double v = lcg_value(s);
            row[static_cast<int64_t>(j) * lda] = static_cast<float>(v);
            sum += j != i ? fabs(v) : 0.0;
            s = S.col.a * s + S.col.c;
        }
        for (int r = 0; r < S.nrhs; ++r) {
            B[static_cast<int64_t>(r) * n + i] = lcg_value(s);
            s = S.col.a * s + S.col.c;
        }
        d[i] = sum;
        row[static_cast<int64_t>(i) * lda] = static_cast<float>(sum);
    }
    __syncthreads();
}

// ---- unpivoted LU of the n x n FP32 matrix A (leading dimension lda, a
// multiple of 4), padded with the identity to whole panels ----
// LDS: the column block P (column c at c * ldp), two blocks of U in FP16 (K
// rows of 32 halves per column, 16-byte chunks XOR-swizzled).  FP16 L: panel p,
// row r at lh + (p n32 + r) 32; behind it the inverses of the panels' L11.
constexpr int kCuLds = 160 * 1024;
constexpr int kBatchStaticLds = 3 * 1024;   // the kernel's own arrays, rounded up
__host__ __device__ constexpr int batch_n32(int n) { return (n + kNB - 1) / kNB * kNB; }
__host__ __device__ constexpr int batch_ldp(int n) { return batch_n32(n) + 4; }   // float4 walks along columns spread over the banks
constexpr int kUBytes = kNB * kNB * 2;
__host__ __device__ constexpr int batch_lds(int n)
{
    return batch_ldp(n) * kNB * 4 + 2 * kUBytes + kNB * 33 * 4 + kNB * 4 + 16;
}
constexpr int64_t batch_lh_halves(int n) { return static_cast<int64_t>(batch_n32(n)) * (batch_n32(n) + 2 * kNB); }
static_assert(batch_lds(kBatchMaxN) + kBatchStaticLds <= kCuLds, "the largest system fits a CU");
static_assert(batch_lds(kBatchMaxN) >= 4 * kBatchMaxN * 8, "the refinement's four x fit too");

__device__ __forceinline__ int u_chunk(int c, int ch) { return c * 64 + ((ch ^ ((c >> 2) & 3)) * 16); }

// wide: panels 2 i and 2 i + 1 are one FP32 panel of 64, so the second takes
// the first's update in FP32
__device__ __forceinline__ int batch_lu(int n, int lda, float *A, _Float16 *Lh, bool wide, uint8_t *lds)
{
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n32 = batch_n32(n), nt = n32 / kNB, ldp = batch_ldp(n);
    float *P = reinterpret_cast<float *>(lds);
    uint8_t *Ub = lds + ldp * kNB * 4;
    float *M = reinterpret_cast<float *>(Ub + 2 * kUBytes);   // inverse of L11, row-major, stride 33
    float *rinv = M + kNB * 33;
    float4 *Li = reinterpret_cast<float4 *>(Lh + static_cast<int64_t>(n32) * n32);
    int *bad = reinterpret_cast<int *>(rinv + kNB);
    int info = 0;
    constexpr int kOthers = kBT / 64 - 1, kMax = 2;
    static_assert(kMax * kOthers >= kBatchMaxN / kNB - 2, "tiles below the first two");

    // rows 32 ti .. of the column block -= L21(ti, p) U(p)
    auto operands = [&](int ln, int p, int ti, half8b_t (&a)[2]) {
        const int l32 = ln & 31, lg = ln >> 5;
        const _Float16 *r = Lh + (static_cast<int64_t>(p) * n32 + 32 * min(ti, nt - 1) + l32) * kNB;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) a[kk] = *reinterpret_cast<const half8b_t *>(r + 16 * kk + 8 * lg);
    };
    // element e of a lane: row acc_row(e, lg) of the tile, column l32
    auto tile = [&](int ln, int ti) {
        return reinterpret_cast<float4 *>(P + (ln & 31) * ldp + 32 * ti + 4 * (ln >> 5));
    };
    auto updated = [&](int ln, int ti, const half8b_t (&a)[2], const uint8_t *U, floatx16b_t &x) {
        const int l32 = ln & 31, lg = ln >> 5;
        const float4 *c = tile(ln, ti);
        floatx16b_t acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
        half8b_t b[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) b[kk] = *reinterpret_cast<const half8b_t *>(U + u_chunk(l32, 2 * kk + lg));
        float4 v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = c[2 * q];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[kk], b[kk], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            x[4 * q] = v[q].x - acc[4 * q];
            x[4 * q + 1] = v[q].y - acc[4 * q + 1];
            x[4 * q + 2] = v[q].z - acc[4 * q + 2];
            x[4 * q + 3] = v[q].w - acc[4 * q + 3];
        }
    };
    auto updated32 = [&](int ln, int p, int ti, floatx16b_t &x) {
        const int l32 = ln & 31, lg = ln >> 5;
        const float4 *c = tile(ln, ti);
        floatx16b_t acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
        const int row = 32 * ti + l32;
        const float *lp = A + static_cast<int64_t>(kNB * p + lg) * lda + min(row, n - 1);
        float av[16], bv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            av[kk] = lp[static_cast<int64_t>(2 * kk) * lda];
            bv[kk] = P[l32 * ldp + kNB * p + 2 * kk + lg];
        }
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(row < n ? av[kk] : 0.0f, bv[kk], acc, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = c[2 * q];
            x[4 * q] = v.x - acc[4 * q];
            x[4 * q + 1] = v.y - acc[4 * q + 1];
            x[4 * q + 2] = v.z - acc[4 * q + 2];
            x[4 * q + 3] = v.w - acc[4 * q + 3];
        }
    };
    auto put = [&](int ln, int ti, const floatx16b_t &x) {
        float4 *c = tile(ln, ti);
#pragma unroll
        for (int q = 0; q < 4; ++q) c[2 * q] = float4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
    };
    // U block p := L11^-1 x; x, a product's result, is the right operand of the
    // next with the K order of acc_row, in which the inverse is stored
    auto inverse = [&](int ln, int p, half8b_t (&v)[3][2]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[1 + (q >> 1)][q & 1] = __builtin_bit_cast(half8b_t, Li[(4 * p + q) * 64 + ln]);
    };
    auto solve_u = [&](int ln, int p, const half8b_t (&iv)[3][2], const floatx16b_t &x) {
        const int l32 = ln & 31, lg = ln >> 5;
        floatx16b_t u;
#pragma unroll
        for (int e = 0; e < 16; ++e) u[e] = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 v = __builtin_bit_cast(float4, iv[1 + (q >> 1)][q & 1]);
            u = __builtin_amdgcn_mfma_f32_32x32x2f32(v.x, x[4 * q], u, 0, 0, 0);
            u = __builtin_amdgcn_mfma_f32_32x32x2f32(v.y, x[4 * q + 1], u, 0, 0, 0);
            u = __builtin_amdgcn_mfma_f32_32x32x2f32(v.z, x[4 * q + 2], u, 0, 0, 0);
            u = __builtin_amdgcn_mfma_f32_32x32x2f32(v.w, x[4 * q + 3], u, 0, 0, 0);
        }
        put(ln, p, u);
        uint8_t *U = Ub + (p & 1) * kUBytes;
#pragma unroll
        for (int q = 0; q < 4; ++q) {   // rows 8 q + 4 lg ..: half of 16-byte chunk q
            half4b_t h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = static_cast<_Float16>(u[4 * q + e]);
            *reinterpret_cast<half4b_t *>(U + u_chunk(l32, q) + 8 * lg) = h;
        }
    };

    for (int k = 0; k < nt; ++k) {
        const int tid = own_tid(), lane = tid & 63, l32 = lane & 31, lg = lane >> 5;
        const int c0 = kNB * k, w = n - c0 < kNB ? n - c0 : kNB;
        // the column block, zero past the matrix and one on the padding's diagonal
        const int chunks = n32 / 4;
        for (int base = tid; base < chunks * kNB; base += 8 * kBT) {
            float4 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = min(base + u * kBT, chunks * kNB - 1), c = e / chunks, r = 4 * (e - c * chunks);
                v[u] = *reinterpret_cast<const float4 *>(A + static_cast<int64_t>(c0 + min(c, w - 1)) * lda +
                                                         min(r, lda - 4));
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = base + u * kBT;
                if (e >= chunks * kNB) continue;
                const int c = e / chunks, r = 4 * (e - c * chunks);
                const float x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
                float y[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) y[q] = c < w ? (r + q < n ? x[q] : 0.0f) : (r + q == c0 + c ? 1.0f : 0.0f);
                *reinterpret_cast<float4 *>(P + c * ldp + r) = float4{y[0], y[1], y[2], y[3]};
            }
        }
        __syncthreads();
        // panels 0 .. k - 1 in turn.  Wave 0 carries the chain: the tile that
        // the next U block is made of, then that block; the others take the
        // rows below.
        if (k > 0) {
            // a wave's operands of the panel after: its tiles' L21, or wave 0's
            // one tile and behind it the next inverse
            using Ahead = half8b_t[3][2];
            Ahead even, odd;
            auto ahead = [&](int ln, int p, Ahead &o) {
                if (wave == 0) {
                    operands(ln, p, p + 1, o[0]);
                    inverse(ln, min(p + 1, k - 1), o);
                } else {
#pragma unroll
                    for (int j = 0; j < kMax; ++j) operands(ln, p, p + 1 + wave + kOthers * j, o[j]);
                }
            };
            if (wave == 0) {
                inverse(lane, 0, odd);
                floatx16b_t x;
                const float4 *c = tile(lane, 0);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = c[2 * q];
                    x[4 * q] = v.x;
                    x[4 * q + 1] = v.y;
                    x[4 * q + 2] = v.z;
                    x[4 * q + 3] = v.w;
                }
                solve_u(lane, 0, odd, x);
            }
            ahead(lane, 0, even);
            __syncthreads();
            auto panel = [&](int p, const Ahead &now, Ahead &next) {
                const int ln = own_tid() & 63;
                const uint8_t *U = Ub + (p & 1) * kUBytes;
                ahead(ln, p + 1, next);
                __builtin_amdgcn_sched_barrier(0);
                floatx16b_t x;
                if (wave == 0) {
                    updated(ln, p + 1, now[0], U, x);
                    solve_u(ln, p + 1, now, x);
                } else {
#pragma unroll
                    for (int j = 0; j < kMax; ++j) {
                        const int ti = p + 1 + wave + kOthers * j;
                        if (ti >= nt) break;
                        updated(ln, ti, now[j], U, x);
                        put(ln, ti, x);
                    }
                }
                __syncthreads();
            };
            int p = 0;
            for (; p + 2 < k; p += 2) {
                panel(p, even, odd);
                panel(p + 1, odd, even);
            }
            if (p + 1 < k) {
                panel(p, even, odd);
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int kk = 0; kk < 2; ++kk) even[j][kk] = odd[j][kk];
                ++p;
            }
            // the last one before this block's own panel
            const int ln = own_tid() & 63;
            floatx16b_t x;
#pragma unroll
            for (int j = 0; j < kMax; ++j) {
                const int ti = p + 1 + wave + kOthers * j;
                if (ti >= nt || (wave == 0 && j > 0)) break;
                if (wide && (k & 1))
                    updated32(ln, p, ti, x);
                else
                    updated(ln, ti, even[j], Ub + (p & 1) * kUBytes, x);
                put(ln, ti, x);
            }
            __syncthreads();
        }
        // the panel: its diagonal block by one wave, then a row of L21 per thread
        if (wave == 0) {
            const int z = lu32(P + c0, ldp, lane);
            wave_lds_sync();
            if (lane < 32) rinv[lane] = 1.0f / P[lane * ldp + c0 + lane];
            if (lane == 0) *bad = z;
        }
        __syncthreads();
        if (info == 0 && *bad != 0) info = c0 + *bad;
        if (wave == kBT / 64 - 1 && k + 1 < nt) {
            // L11's inverse as the left operand of solve_u
            invert32<false>(P + c0, ldp, nullptr, lane, M);
            wave_lds_sync();
            float v[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = M[l32 * 33 + acc_row(e, lg)];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                Li[(4 * k + q) * 64 + lane] = float4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
        }
        if (const int r = c0 + kNB + own_tid(); r < n32) {
            float x[kNB];
#pragma unroll
            for (int c = 0; c < kNB; ++c) x[c] = P[c * ldp + r];
#pragma unroll
            for (int c = 0; c < kNB; ++c) {
#pragma unroll
                for (int q = 0; q < (c + 3) / 4; ++q) {
                    const float4 u = *reinterpret_cast<const float4 *>(P + c * ldp + c0 + 4 * q);
                    const float uv[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * q + e < c) x[c] = fmaf(-x[4 * q + e], uv[e], x[c]);
                }
                x[c] *= rinv[c];
            }
#pragma unroll
            for (int c = 0; c < kNB; ++c) P[c * ldp + r] = x[c];
            half8b_t *o = reinterpret_cast<half8b_t *>(Lh + (static_cast<int64_t>(k) * n32 + r) * kNB);
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                half8b_t h;
#pragma unroll
                for (int e = 0; e < 8; ++e) h[e] = static_cast<_Float16>(x[8 * ch + e]);
                o[ch] = h;
            }
        }
        __syncthreads();
        // factors back to A; rows go in aligned groups of 4 (lda % 4 == 0, so a
        // group never leaves the allocation)
        const int rows4 = (n + 3) / 4;
        for (int e = own_tid(); e < rows4 * w; e += kBT) {
            const int c = e / rows4, r = 4 * (e - c * rows4);
            *reinterpret_cast<float4 *>(A + static_cast<int64_t>(c0 + c) * lda + r) =
                *reinterpret_cast<const float4 *>(P + c * ldp + r);
        }
        __syncthreads();
    }
    return info;
}

__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// strip loader: dst[c] = element (row tid, column col0 + c), columns clamped;
// rows that the strip's triangle does not reach are left out
template <bool UPPER>
__device__ __forceinline__ void trsv_load_strip(const float *__restrict__ M, int64_t lda, int bs,
                                                int col0, int tid, float (&dst)[32])
{
    if (tid < bs && (UPPER ? tid < col0 + 32 : tid >= col0)) {
#pragma unroll
        for (int c = 0; c < 32; ++c) dst[c] = M[static_cast<int64_t>(min(col0 + c, bs - 1)) * lda + tid];
    }
}

// Solves T x = x in place for the bs x bs triangle T (lower or upper, unit or
// not; bs <= kBT) and the NR right-hand sides of a system at once (columns x +
// rr bs), the diagonal-block step of panel_trsvL / panel_trsvU
// (panel_trsv.hpp:310-758).  Thread t owns row t and keeps its x in registers.
// The triangle is walked in 32-column strips, each loaded once for all
// right-hand sides, a strip ahead.  The 32 x 32 diagonal sub-block is solved by
// the half-wave that owns its rows: x_c is broadcast with v_readlane and the
// other lanes subtract l_ic x_c; the strip's final x goes through LDS to the
// threads owning the rows further on.  Non-unit diagonals are applied as a
// multiply by 1 / t_cc computed before the dependent chain (one rounding
// different from a division).  xs: 2 x 4 x 32 doubles of LDS, by turns.
template <bool UPPER, bool UNIT, int NR>
__device__ __forceinline__ void batch_trsv(int bs, int lda, const float *__restrict__ T, double *__restrict__ x,
                                           double *xs)
{
    const int tid = own_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    double xr[NR];
#pragma unroll
    for (int rr = 0; rr < NR; ++rr) xr[rr] = tid < bs ? x[static_cast<int64_t>(rr) * bs + tid] : 0.0;
    const int nsb = (bs + 31) / 32;
    float cur[32], nxt[32];
    trsv_load_strip<UPPER>(T, lda, bs, (UPPER ? nsb - 1 : 0) * 32, tid, cur);
    for (int step = 0; step < nsb; ++step) {
        const int q = UPPER ? nsb - 1 - step : step;
        const int sb = q * 32;
        const int w = bs - sb < 32 ? bs - sb : 32;
        double *xq = xs + (step & 1) * 4 * 32;
        if (step + 1 < nsb) trsv_load_strip<UPPER>(T, lda, bs, (UPPER ? q - 1 : q + 1) * 32, tid, nxt);
        const int half = q & 1;
        if (wave == q / 2) {
            const int i = lane - 32 * half;
            const bool mine = i >= 0 && i < w;
            double rinv = 1.0;
            if (!UNIT) {
                float dg = 1.0f;
#pragma unroll
                for (int c = 0; c < 32; ++c)
                    if (c == i) dg = cur[c];
                rinv = 1.0 / static_cast<double>(dg);
            }
#pragma unroll
            for (int cc = 0; cc < 32; ++cc) {
                const int c = UPPER ? 31 - cc : cc;
                if (c < w) {
                    const bool on = mine && (UPPER ? i < c : i > c);
#pragma unroll
                    for (int rr = 0; rr < NR; ++rr) {
                        if (!UNIT && i == c) xr[rr] *= rinv;
                        const double xc = readlane_f64(xr[rr], 32 * half + c);
                        if (on) xr[rr] = fma(-static_cast<double>(cur[c]), xc, xr[rr]);
                    }
                }
            }
            if (mine)
#pragma unroll
                for (int rr = 0; rr < NR; ++rr) xq[rr * 32 + i] = xr[rr];
        }
        __syncthreads();
        if (UPPER ? tid < sb : (tid >= sb + w && tid < bs)) {
#pragma unroll
            for (int rr = 0; rr < NR; ++rr) {
                double acc = 0.0;
#pragma unroll
                for (int c = 0; c < 32; ++c)
                    if (c < w) acc = fma(static_cast<double>(cur[c]), xq[rr * 32 + c], acc);
                xr[rr] -= acc;
            }
        }
#pragma unroll
        for (int c = 0; c < 32; ++c) cur[c] = nxt[c];
    }
#pragma unroll
    for (int rr = 0; rr < NR; ++rr)
        if (tid < bs) x[static_cast<int64_t>(rr) * bs + tid] = xr[rr];
    __syncthreads();
}

// L^-1 and then U^-1 for NR right-hand sides
template <int NR>
__device__ __forceinline__ void batch_solve(int n, int lda, const float *A, double *x, double *xs)
{
    batch_trsv<false, true, NR>(n, lda, A, x, xs);
    batch_trsv<true, false, NR>(n, lda, A, x, xs);
}

// acc[r] = b - A x for row tid (those past n repeat the last) and NR right-hand sides, A's entries from the generator, j ascending; x at xl
template <int NR>
__device__ __forceinline__ void batch_residual(const BatchSys &S, const double *__restrict__ d,
                                               const double *__restrict__ B, const double *xl, double (&acc)[4])
{
    const int n = S.n, i = min(own_tid(), n - 1);
    uint64_t s = lcg_jump(S.x1, static_cast<uint64_t>(i));
    const double di = d[i];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = B[static_cast<int64_t>(r) * n + i];
    constexpr int UN = 4;
    for (int j0 = 0; j0 < n; j0 += UN) {
        double x[NR][UN];
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
            for (int u = 0; u < UN; ++u) x[r][u] = xl[r * n + min(j0 + u, n - 1)];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            double a = lcg_value(s);
            s = S.col.a * s + S.col.c;
            a = j0 + u == i ? di : a;
            if (j0 + u < n)
#pragma unroll
                for (int r = 0; r < NR; ++r) acc[r] = fma(-a, x[r][u], acc[r]);
        }
    }
}

// |b - A x| and |x| of NR right-hand sides, their maxima over the rows at once:
// one barrier, and only the waves that own rows: latency-bound at small orders,
// where a reduction for each of the eight maxima over all 16 waves took longer
// than the residual (150 systems of order 4 to 16: 97 -> 71 us, of order 100:
// 369 -> 305 us).  red is free again after the caller's next barrier.
template <int NR>
__device__ __forceinline__ void batch_norms(int n, const double (&acc)[4], const double *xl, double *R, double *red,
                                            double (&rm)[4], double (&xm)[4])
{
    constexpr int NV = 2 * NR;
    const int tid = own_tid(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = (n + 63) / 64;
    if (wave < nw) {
        double v[NV];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            v[2 * r] = v[2 * r + 1] = 0.0;
            if (tid < n) {
                R[static_cast<int64_t>(r) * n + tid] = acc[r];
                v[2 * r] = fabs(acc[r]);
                v[2 * r + 1] = fabs(xl[r * n + tid]);
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
#pragma unroll
            for (int q = 0; q < NV; ++q) v[q] = fmax(v[q], __shfl_xor(v[q], off));
        if (lane == 0)
#pragma unroll
            for (int q = 0; q < NV; ++q) red[wave * NV + q] = v[q];
    }
    __syncthreads();
    double m[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) m[q] = red[q];
    for (int w = 1; w < nw; ++w)
#pragma unroll
        for (int q = 0; q < NV; ++q) m[q] = fmax(m[q], red[w * NV + q]);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        // rows past the end count as zeros, also beside NaNs
        rm[r] = nw < kBT / 64 ? fmax(m[2 * r], 0.0) : m[2 * r];
        xm[r] = nw < kBT / 64 ? fmax(m[2 * r + 1], 0.0) : m[2 * r + 1];
    }
}

// ---- FP64 refinement of every right-hand side (iterative_refinement.hpp:18-57) ----
__device__ __forceinline__ void batch_refine(const BatchSys &S, const float *LU, const double *d,
                             const double *B, double *X, double *R, double *xl, double *xs, double *red,
                             BatchOut &o, int maxit)
{
    // every right-hand side refines on its own (its own harness, steps and
    // stop), but the residuals of all that still refine come from one pass
    // over A per step: each element is generated once and feeds up to 4 FMAs
    // in the same order as a pass per right-hand side would
    const int n = S.n, lda = S.lda, tid = own_tid(), nr = S.nrhs;
    double dm = 0.0;
    for (int i = tid; i < n; i += kBT) dm = fmax(dm, fabs(d[i]));
    const double norma = 2.0 * block_max(dm, red);          // hpl_infnorm, panel_norm.hpp:78-84
    double normb[4] = {0.0, 0.0, 0.0, 0.0}, h[4] = {-1.0, -1.0, -1.0, -1.0};
    int steps[4] = {0, 0, 0, 0};
    bool done[4] = {false, false, false, false};
    for (int rr = 0; rr < nr; ++rr) {
        const double *b = B + static_cast<int64_t>(rr) * n;
        double *x = X + static_cast<int64_t>(rr) * n;
        double bm = 0.0;
        for (int i = tid; i < n; i += kBT) {
            x[i] = b[i] / d[i];                              // x0 = b ./ diag(A)
            bm = fmax(bm, fabs(b[i]));
        }
        normb[rr] = block_max(bm, red);
    }
    for (int it = 0; it < maxit; ++it) {
        // r = b - A x in FP64 for the right-hand sides still refining (x staged in LDS)
        for (int rr = 0; rr < nr; ++rr)
            if (!done[rr])
                for (int i = tid; i < n; i += kBT) xl[rr * n + i] = X[static_cast<int64_t>(rr) * n + i];
        __syncthreads();
        double xm[4] = {0.0, 0.0, 0.0, 0.0}, rm[4] = {0.0, 0.0, 0.0, 0.0};
        auto residual = [&](auto nrhs) {
            constexpr int NR = decltype(nrhs)::value;
            double acc[4];
            if ((tid & ~63) < n) batch_residual<NR>(S, d, B, xl, acc);   // waves that own rows
            batch_norms<NR>(n, acc, xl, R, red, rm, xm);
        };
        switch (nr) {
        case 1: residual(std::integral_constant<int, 1>{}); break;
        case 2: residual(std::integral_constant<int, 2>{}); break;
        case 3: residual(std::integral_constant<int, 3>{}); break;
        default: residual(std::integral_constant<int, 4>{}); break;
        }
        bool all = true;
        for (int rr = 0; rr < nr; ++rr) {
            if (done[rr]) continue;
            h[rr] = rm[rr] / (norma * xm[rr] + normb[rr]) * 1. / (static_cast<double>(n) * DBL_EPSILON / 2);
            steps[rr] = it + 1;
            done[rr] = h[rr] < 16.0;
            all = all && done[rr];
        }
        if (all) break;
        // corrections of all right-hand sides in one pass over each triangle
        // (the ones already done are solved too and not used)
        switch (nr) {
        case 1: batch_solve<1>(n, lda, LU, R, xs); break;
        case 2: batch_solve<2>(n, lda, LU, R, xs); break;
        case 3: batch_solve<3>(n, lda, LU, R, xs); break;
        default: batch_solve<4>(n, lda, LU, R, xs); break;
        }
        for (int rr = 0; rr < nr; ++rr) {
            if (done[rr]) continue;
            const double *r = R + static_cast<int64_t>(rr) * n;
            double *x = X + static_cast<int64_t>(rr) * n;
            for (int i = tid; i < n; i += kBT) x[i] += r[i];
        }
        __syncthreads();
    }
    if (tid == 0)
        for (int rr = 0; rr < nr; ++rr) {
            o.harness[rr] = h[rr];
            o.steps[rr] = steps[rr];
        }
    __syncthreads();
}

__global__ __launch_bounds__(kBT) void batch_kernel(const BatchSys *__restrict__ sys,
                                                    const int32_t *__restrict__ order, int count,
                                                    float *__restrict__ fpool, double *__restrict__ dpool,
                                                    _Float16 *__restrict__ hpool, BatchOut *__restrict__ out, int32_t *counter, int maxit)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ double xs[2 * 4 * 32];
    __shared__ double red[kBT / 64 * 8];
    __shared__ int32_t next;
    for (;;) {
        if (threadIdx.x == 0) next = atomicAdd(counter, 1);
        __syncthreads();
        const int q = next;
        __syncthreads();
        if (q >= count) break;
        const int sid = order[q];
        const BatchSys S = sys[sid];
        const uint64_t t0 = wall_clock64();
        float *A32 = fpool + S.a32;
        double *d = dpool + S.d, *B = dpool + S.b, *X = dpool + S.x,
               *R = dpool + S.r;
        batch_generate(S, A32, d, B);
        const int info = batch_lu(S.n, S.lda, A32, hpool + S.lh, S.nb == 64, lds);
        BatchOut o;
        o.info = info;
        if (info == 0)
            batch_refine(S, A32, d, B, X, R, reinterpret_cast<double *>(lds), xs, red, o, maxit);
        __syncthreads();
        if (threadIdx.x == 0) {
            BatchOut &g = out[sid];
            for (int r = 0; r < 4; ++r) {
                g.harness[r] = (info == 0 && r < S.nrhs) ? o.harness[r] : -1.0;
                g.steps[r] = (info == 0 && r < S.nrhs) ? o.steps[r] : 0;
            }
            g.info = info;
            g.t0 = t0;
            g.t1 = wall_clock64();
        }
    }
}

__global__ void batch_reset_kernel(int32_t *counter) { *counter = 0; }

}  // namespace hplai

// ===========================================================================
// host side
// ===========================================================================
using namespace hplai;

struct hplai_batch_s {
    hplai_ctx ctx = nullptr;
    int count = 0;
    std::vector<int32_t> n, nrhs;
    std::vector<uint64_t> seed;
    std::vector<BatchSys> sys;
    std::vector<int32_t> order;           // largest first
    int32_t nb_table[kBuckets] = {32, 32, 32, 32};
    BatchSys *d_sys = nullptr;
    int32_t *d_order = nullptr, *d_counter = nullptr;   // d_counter[0]: one launch; [1 + s]: system s alone
    int32_t *d_ident = nullptr;                          // systems in input order
    hipStream_t streams[4] = {};                          // baseline: per-system launches on 4 streams
    float *fpool = nullptr;
    double *dpool = nullptr;
    _Float16 *hpool = nullptr;
    BatchOut *d_out = nullptr;
    std::vector<BatchOut> out;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int graph_maxit = -1;
    double clock_khz = 100000.0;
};

namespace {

int bucket_of(int n) { return n < 128 ? 0 : n < 256 ? 1 : n < 512 ? 2 : 3; }

int upload_sys(hplai_batch b)
{
    for (int s = 0; s < b->count; ++s) b->sys[s].nb = b->nb_table[bucket_of(b->n[s])];
    HPLAI_HIP(hipMemcpy(b->d_sys, b->sys.data(), sizeof(BatchSys) * b->count, hipMemcpyHostToDevice));
    return HPLAI_OK;
}

int launch_batch(hplai_batch b, const int32_t *d_order, int count, int grid, int maxit, hipStream_t s,
                 int32_t *counter = nullptr)
{
    if (counter == nullptr) counter = b->d_counter;
    hipLaunchKernelGGL(batch_reset_kernel, dim3(1), dim3(1), 0, s, counter);
    hipLaunchKernelGGL(batch_kernel, dim3(grid), dim3(kBT), batch_lds(kBatchMaxN), s, b->d_sys, d_order, count, b->fpool,
                       b->dpool, b->hpool, b->d_out, counter, maxit);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

}  // namespace

extern "C" {

int hplai_batch_create(hplai_ctx ctx, int count, const int32_t *n, const int32_t *nrhs, const uint64_t *seed,
                       hplai_batch *out)
{
    HPLAI_CHECK(ctx != nullptr && out != nullptr && n != nullptr && nrhs != nullptr && seed != nullptr,
                "hplai_batch_create: NULL argument");
    HPLAI_CHECK(count > 0, "hplai_batch_create: count %d", count);
    for (int s = 0; s < count; ++s) {
        HPLAI_CHECK(n[s] >= 1 && n[s] <= kBatchMaxN, "hplai_batch_create: system %d has n=%d (1..%d)", s, n[s],
                    kBatchMaxN);
        HPLAI_CHECK(nrhs[s] >= 1 && nrhs[s] <= 4, "hplai_batch_create: system %d has %d rhs (1..4)", s,
                    nrhs[s]);
    }
    HPLAI_HIP(hipSetDevice(ctx->device));
    hplai_batch b = new hplai_batch_s;
    b->ctx = ctx;
    b->count = count;
    b->n.assign(n, n + count);
    b->nrhs.assign(nrhs, nrhs + count);
    b->seed.assign(seed, seed + count);
    b->sys.resize(count);
    int64_t fo = 0, dof = 0, ho = 0;
    auto up = [](int64_t v) { return (v + 63) / 64 * 64; };
    for (int s = 0; s < count; ++s) {
        BatchSys &S = b->sys[s];
        S.n = n[s];
        S.nrhs = nrhs[s];
        S.nb = 32;
        S.lda = (n[s] + 3) / 4 * 4;
        const int64_t nn = static_cast<int64_t>(S.lda) * n[s];
        S.x1 = lcg_init(seed[s]);
        S.a32 = fo;
        fo += up(nn);
        S.col = lcg_pow_host(static_cast<uint64_t>(n[s]));
        S.lh = ho;
        ho += batch_lh_halves(n[s]);
        S.d = dof;
        dof += up(n[s]);
        S.b = dof;
        dof += up(static_cast<int64_t>(n[s]) * nrhs[s]);
        S.x = dof;
        dof += up(static_cast<int64_t>(n[s]) * nrhs[s]);
        S.r = dof;
        dof += up(static_cast<int64_t>(n[s]) * nrhs[s]);
    }
    b->order.resize(count);
    for (int s = 0; s < count; ++s) b->order[s] = s;
    std::stable_sort(b->order.begin(), b->order.end(), [&](int a, int c) { return b->n[a] > b->n[c]; });
    b->out.resize(count);
    int rc = HPLAI_OK;
    auto alloc = [&](void **p, size_t bytes) {
        if (rc != HPLAI_OK) return;
        const hipError_t e = device_malloc(ctx->device, p, bytes);
        if (e != hipSuccess) rc = hip_fail(e, "hplai_batch_create: hipMalloc");
    };
    alloc(reinterpret_cast<void **>(&b->d_sys), sizeof(BatchSys) * count);
    alloc(reinterpret_cast<void **>(&b->d_order), sizeof(int32_t) * count);
    alloc(reinterpret_cast<void **>(&b->d_counter), sizeof(int32_t) * (count + 1));
    alloc(reinterpret_cast<void **>(&b->d_ident), sizeof(int32_t) * count);
    alloc(reinterpret_cast<void **>(&b->fpool), sizeof(float) * fo);
    alloc(reinterpret_cast<void **>(&b->dpool), sizeof(double) * dof);
    alloc(reinterpret_cast<void **>(&b->hpool), sizeof(_Float16) * ho);
    alloc(reinterpret_cast<void **>(&b->d_out), sizeof(BatchOut) * count);
    if (rc == HPLAI_OK &&
        hipMemcpy(b->d_order, b->order.data(), sizeof(int32_t) * count, hipMemcpyHostToDevice) != hipSuccess)
        rc = hip_fail(hipGetLastError(), "hplai_batch_create: copy");
    if (rc == HPLAI_OK) {
        std::vector<int32_t> ident(count);
        for (int q = 0; q < count; ++q) ident[q] = q;
        if (hipMemcpy(b->d_ident, ident.data(), sizeof(int32_t) * count, hipMemcpyHostToDevice) != hipSuccess)
            rc = hip_fail(hipGetLastError(), "hplai_batch_create: copy");
    }
    for (int q = 0; q < 4 && rc == HPLAI_OK; ++q)
        if (hipStreamCreateWithFlags(&b->streams[q], hipStreamNonBlocking) != hipSuccess)
            rc = hip_fail(hipGetLastError(), "hplai_batch_create: streams");
    if (rc == HPLAI_OK) rc = upload_sys(b);
    if (rc == HPLAI_OK &&
        hipFuncSetAttribute(reinterpret_cast<const void *>(batch_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, batch_lds(kBatchMaxN)) != hipSuccess)
        rc = hip_fail(hipGetLastError(), "hplai_batch_create: LDS size");
    int khz = 0;
    if (rc == HPLAI_OK && hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ctx->device) == hipSuccess &&
        khz > 0)
        b->clock_khz = khz;
    if (rc != HPLAI_OK) {
        hplai_batch_destroy(b);
        return rc;
    }
    *out = b;
    return HPLAI_OK;
}

int hplai_batch_destroy(hplai_batch b)
{
    if (b == nullptr) return HPLAI_OK;
    (void)hipSetDevice(b->ctx->device);
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    (void)hipFree(b->d_sys);
    (void)hipFree(b->d_order);
    (void)hipFree(b->d_counter);
    (void)hipFree(b->d_ident);
    for (int q = 0; q < 4; ++q)
        if (b->streams[q]) (void)hipStreamDestroy(b->streams[q]);
    (void)hipFree(b->fpool);
    (void)hipFree(b->dpool);
    (void)hipFree(b->hpool);
    (void)hipFree(b->d_out);
    delete b;
    return HPLAI_OK;
}

int hplai_batch_set_nb(hplai_batch b, const int32_t nb[4])
{
    HPLAI_CHECK(b != nullptr && nb != nullptr, "hplai_batch_set_nb: NULL argument");
    for (int k = 0; k < kBuckets; ++k)
        HPLAI_CHECK(nb[k] == 16 || nb[k] == 32 || nb[k] == 64, "hplai_batch_set_nb: nb %d not in {16,32,64}",
                    nb[k]);
    for (int k = 0; k < kBuckets; ++k) b->nb_table[k] = nb[k];
    // a captured graph stays valid: it reads the descriptors through the same pointer
    return upload_sys(b);
}

int hplai_batch_get_nb(hplai_batch b, int32_t nb[4])
{
    HPLAI_CHECK(b != nullptr && nb != nullptr, "hplai_batch_get_nb: NULL argument");
    for (int k = 0; k < kBuckets; ++k) nb[k] = b->nb_table[k];
    return HPLAI_OK;
}

int hplai_batch_run(hplai_batch b, int mode, int maxit, hplai_batch_stats *st)
{
    HPLAI_CHECK(b != nullptr && st != nullptr, "hplai_batch_run: NULL argument");
    HPLAI_CHECK(mode >= 0 && mode <= 4, "hplai_batch_run: mode %d", mode);
    if (maxit <= 0) maxit = 50;
    HPLAI_HIP(hipSetDevice(b->ctx->device));
    hipStream_t s = b->ctx->side;
    const int grid = b->ctx->num_cu > 0 ? b->ctx->num_cu : 256;
    HPLAI_HIP(hipStreamSynchronize(s));
    const auto t0 = std::chrono::steady_clock::now();
    int rc = HPLAI_OK;
    if (mode == 0) {
        rc = launch_batch(b, b->d_order, b->count, grid, maxit, s);
    } else if (mode == 1) {
        if (b->exec == nullptr || b->graph_maxit != maxit) {
            if (b->exec) (void)hipGraphExecDestroy(b->exec);
            if (b->graph) (void)hipGraphDestroy(b->graph);
            b->exec = nullptr;
            b->graph = nullptr;
            HPLAI_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
            rc = launch_batch(b, b->d_order, b->count, grid, maxit, s);
            hipGraph_t g = nullptr;
            const hipError_t e = hipStreamEndCapture(s, &g);
            if (rc == HPLAI_OK && e != hipSuccess) rc = hip_fail(e, "hplai_batch_run: capture");
            if (rc == HPLAI_OK) {
                b->graph = g;
                const hipError_t e2 = hipGraphInstantiate(&b->exec, g, nullptr, nullptr, 0);
                if (e2 != hipSuccess) rc = hip_fail(e2, "hplai_batch_run: instantiate");
                b->graph_maxit = maxit;
            } else if (g) {
                (void)hipGraphDestroy(g);
            }
        }
        if (rc == HPLAI_OK) HPLAI_HIP(hipGraphLaunch(b->exec, s));
    } else if (mode == 2) {
        // baseline: one launch (one workgroup) per system, in the same order
        for (int q = 0; q < b->count && rc == HPLAI_OK; ++q)
            rc = launch_batch(b, b->d_order + q, 1, 1, maxit, s);
    } else if (mode == 3) {
        // baseline: one launch per system, round-robin over four streams (the
        // process has four hardware queues), each launch with its own counter
        for (int q = 0; q < b->count && rc == HPLAI_OK; ++q)
            rc = launch_batch(b, b->d_order + q, 1, 1, maxit, b->streams[q & 3], b->d_counter + 1 + q);
        for (int q = 0; q < 4; ++q) HPLAI_HIP(hipStreamSynchronize(b->streams[q]));
    } else {
        // baseline: one launch of one workgroup per system in input order (a
        // plain batched grid: no largest-first order, no persistent workgroups)
        rc = launch_batch(b, b->d_ident, b->count, b->count, maxit, s);
    }
    HPLAI_HIP(hipStreamSynchronize(s));
    const auto t1 = std::chrono::steady_clock::now();
    if (rc) return rc;
    HPLAI_HIP(hipMemcpy(b->out.data(), b->d_out, sizeof(BatchOut) * b->count, hipMemcpyDeviceToHost));
    std::vector<double> us(b->count);
    int failed = 0, max_steps = 0;
    double max_h = 0.0;
    for (int s2 = 0; s2 < b->count; ++s2) {
        const BatchOut &o = b->out[s2];
        us[s2] = static_cast<double>(o.t1 - o.t0) / b->clock_khz * 1e3;
        bool ok = o.info == 0;
        for (int r = 0; r < b->nrhs[s2]; ++r) {
            if (!(o.harness[r] >= 0.0 && o.harness[r] < 16.0)) ok = false;
            max_h = std::max(max_h, o.harness[r]);
            max_steps = std::max(max_steps, o.steps[r]);
        }
        if (!ok) ++failed;
    }
    std::vector<double> sorted = us;
    std::sort(sorted.begin(), sorted.end());
    auto pct = [&](double p) { return sorted[std::min<size_t>(sorted.size() - 1, static_cast<size_t>(p * sorted.size()))]; };
    st->seconds = std::chrono::duration<double>(t1 - t0).count();
    st->systems_per_s = b->count / st->seconds;
    st->p50_us = pct(0.50);
    st->p99_us = pct(0.99);
    st->max_us = sorted.back();
    st->failed = failed;
    st->max_harness = max_h;
    st->max_steps = max_steps;
    return HPLAI_OK;
}

int hplai_batch_results(hplai_batch b, double *harness, int32_t *steps, int32_t *info, double *time_us)
{
    HPLAI_CHECK(b != nullptr, "hplai_batch_results: NULL batch");
    for (int s = 0; s < b->count; ++s) {
        const BatchOut &o = b->out[s];
        for (int r = 0; r < 4; ++r) {
            if (harness) harness[4 * s + r] = o.harness[r];
            if (steps) steps[4 * s + r] = o.steps[r];
        }
        if (info) info[s] = o.info;
        if (time_us) time_us[s] = static_cast<double>(o.t1 - o.t0) / b->clock_khz * 1e3;
    }
    return HPLAI_OK;
}

int hplai_batch_solution(hplai_batch b, int s, double *x_host)
{
    HPLAI_CHECK(b != nullptr && x_host != nullptr && s >= 0 && s < b->count, "hplai_batch_solution: bad argument");
    HPLAI_HIP(hipSetDevice(b->ctx->device));
    const BatchSys &S = b->sys[s];
    HPLAI_HIP(hipMemcpy(x_host, b->dpool + S.x, sizeof(double) * S.n * S.nrhs, hipMemcpyDeviceToHost));
    return HPLAI_OK;
}

int hplai_batch_autotune(hplai_batch b, int maxit, int32_t nb_out[4])
{
    HPLAI_CHECK(b != nullptr, "hplai_batch_autotune: NULL batch");
    if (maxit <= 0) maxit = 50;
    HPLAI_HIP(hipSetDevice(b->ctx->device));
    hipStream_t s = b->ctx->side;
    const int grid = b->ctx->num_cu > 0 ? b->ctx->num_cu : 256;
    const int cands[2] = {32, 64};
    int32_t best[kBuckets];
    for (int k = 0; k < kBuckets; ++k) best[k] = b->nb_table[k];
    int32_t *d_sub = nullptr;
    HPLAI_HIP(device_malloc(b->ctx->device, reinterpret_cast<void **>(&d_sub), sizeof(int32_t) * b->count));
    int rc = HPLAI_OK;
    for (int k = 0; k < kBuckets && rc == HPLAI_OK; ++k) {
        // up to 2 systems per CU of this bucket, largest first
        std::vector<int32_t> sub;
        for (int q = 0; q < b->count && static_cast<int>(sub.size()) < 2 * grid; ++q)
            if (bucket_of(b->n[b->order[q]]) == k) sub.push_back(b->order[q]);
        if (sub.empty()) continue;
        if (hipMemcpy(d_sub, sub.data(), sizeof(int32_t) * sub.size(), hipMemcpyHostToDevice) != hipSuccess) {
            rc = hip_fail(hipGetLastError(), "hplai_batch_autotune: copy");
            break;
        }
        double best_t = 1e300;
        for (int c = 0; c < 2 && rc == HPLAI_OK; ++c) {
            const int nb = cands[c];
            for (int32_t sid : sub) b->sys[sid].nb = nb;
            if (hipMemcpy(b->d_sys, b->sys.data(), sizeof(BatchSys) * b->count, hipMemcpyHostToDevice) != hipSuccess) {
                rc = hip_fail(hipGetLastError(), "hplai_batch_autotune: copy");
                break;
            }
            // one untimed pass, then the timed one
            double t = 0.0;
            for (int pass = 0; pass < 2 && rc == HPLAI_OK; ++pass) {
                const auto t0 = std::chrono::steady_clock::now();
                rc = launch_batch(b, d_sub, static_cast<int>(sub.size()), grid, maxit, s);
                if (rc == HPLAI_OK && hipStreamSynchronize(s) != hipSuccess)
                    rc = hip_fail(hipGetLastError(), "hplai_batch_autotune: run");
                t = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            }
            // 5 % faster, or the choice would be the clock's and differ from run to run
            if (rc == HPLAI_OK && t < 0.95 * best_t) {
                best_t = t;
                best[k] = nb;
            }
        }
    }
    (void)hipFree(d_sub);
    if (rc) return rc;
    for (int k = 0; k < kBuckets; ++k) b->nb_table[k] = best[k];
    if (nb_out)
        for (int k = 0; k < kBuckets; ++k) nb_out[k] = best[k];
    return upload_sys(b);
}

}  // extern "C"
