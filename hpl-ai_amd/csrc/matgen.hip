// matgen.hip — the HPL-AI matrix generator on gfx950, bit-exact with
// hpl_rand.hpp (RIKEN-RCCS/hpl-ai).
//
// Element (i,j) of the n x n matrix is the LCG state reached after 1+i+n*j
// steps from the seed, mapped to [-0.5, 0.5).  Rows are consecutive states,
// columns jump by (a,c)^n.  The diagonal entry is sum_{j != i} |a_ij|,
// accumulated in FP64 with j ascending, exactly as calc_diag does.
#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace hplai {

constexpr int kGenRows = 256;   // rows per block (one per thread)
constexpr int kGenCols = 64;    // columns per thread: amortises the jump-ahead

// fill_one_panel_with_rand (hpl_rand.hpp:59-106) for a block at (i0, j0) without
// partial sums, the plain generation: a thread's columns in groups of kGenPlain
// from as many states, all their stores in flight, and the diagonal looked for
// only where the workgroup's block meets it.  Bound by the stores; one column per
// iteration, behind the conditions of the general form, took 106 us for 10007 x
// 10007, now 97 (8.1 -> 7.1 ms at 98304).
constexpr int kGenPlain = 8;

__global__ __launch_bounds__(kGenRows) void gen_plain_kernel(uint64_t n, uint64_t x1, int64_t i0, int64_t j0, int64_t m,
                                                             int64_t k, int64_t row_blocks, LcgCoeff jn, LcgCoeff jgroup,
                                                             const double *__restrict__ d, float *__restrict__ A,
                                                             int64_t lda)
{
    const int64_t rb = blockIdx.x % row_blocks, cg = blockIdx.x / row_blocks;
    const int64_t ib = rb * kGenRows, jb = cg * kGenCols;
    const int64_t il = ib + threadIdx.x;
    if (il >= m) return;
    const int nc = static_cast<int>(k - jb < kGenCols ? k - jb : kGenCols);
    uint64_t s[kGenPlain];
    s[0] = lcg_jump_lanes<8>(x1, static_cast<uint64_t>(i0 + ib) + n * static_cast<uint64_t>(j0 + jb), threadIdx.x);
#pragma unroll
    for (int u = 1; u < kGenPlain; ++u) s[u] = jn.a * s[u - 1] + jn.c;
    float *col = A + jb * lda + ib;   // uniform
    for (int c0 = 0; c0 < nc; c0 += kGenPlain) {
        float v[kGenPlain];
#pragma unroll
        for (int u = 0; u < kGenPlain; ++u) {
            v[u] = static_cast<float>(lcg_value(s[u]));
            s[u] = jgroup.a * s[u] + jgroup.c;
        }
#pragma unroll
        for (int u = 0; u < kGenPlain; ++u)
            if (c0 + u < nc) (col + (c0 + u) * lda)[threadIdx.x] = v[u];
    }
    // rows [i0 + ib, + 256) and columns [j0 + jb, + nc)
    if (d != nullptr && i0 + ib < j0 + jb + nc && j0 + jb < i0 + ib + kGenRows) {
        const int64_t jl = i0 + il - j0;
        if (jl >= jb && jl < jb + nc) A[jl * lda + il] = static_cast<float>(d[i0 + il]);
    }
}

// The general form: added to what is there, with the FP16 partial sums.
__global__ __launch_bounds__(kGenRows) void gen_matrix_kernel(
    int64_t n, uint64_t x1, int64_t i0, int64_t j0, int64_t m, int64_t k, int64_t row_blocks,
    LcgCoeff jn, const double *__restrict__ d, float *__restrict__ A, int64_t lda, int accumulate,
    const uint16_t *__restrict__ P, const uint16_t *__restrict__ Q, int64_t ldp, float pscale)
{
    const int64_t rb = blockIdx.x % row_blocks;
    const int64_t cg = blockIdx.x / row_blocks;
    const int64_t il = rb * kGenRows + threadIdx.x;
    if (il >= m) return;
    const int64_t jl0 = cg * kGenCols;
    const int64_t jl1 = jl0 + kGenCols < k ? jl0 + kGenCols : k;
    const int64_t gi = i0 + il;
    uint64_t s = lcg_jump(x1, static_cast<uint64_t>(gi) +
                                  static_cast<uint64_t>(n) * static_cast<uint64_t>(j0 + jl0));
    float *col = A + jl0 * lda + il;
    const uint16_t *pcol = P != nullptr ? P + jl0 * ldp + il : nullptr;
    const uint16_t *qcol = Q != nullptr ? Q + jl0 * ldp + il : nullptr;
    for (int64_t jl = jl0; jl < jl1; ++jl, col += lda) {
        float v = static_cast<float>(lcg_value(s));
        if (d != nullptr && gi == j0 + jl) v = static_cast<float>(d[gi]);
        // lazy initialisation merges the partial sum: to = scale * from + a_ij
        // (LazyInitializer::update, lazy_init.hpp:147-227); the FP16 trailing
        // storage holds the partial sums of earlier outer steps times 1 / scale
        if (pcol != nullptr) {
            // with the back buffer Q (lazy_init.hpp:229-329): x = P + 32 Q
            float x = f16_bits_to_f32(*pcol);
            if (qcol != nullptr) {
                x = fmaf(32.0f, f16_bits_to_f32(*qcol), x);
                qcol += ldp;
            }
            v = fmaf(pscale, x, v);
            pcol += ldp;
        }
        *col = accumulate ? *col + v : v;
        s = jn.a * s + jn.c;
    }
}

// calc_diag (hpl_rand.hpp:108-123): the FP64 sum of a row runs j = 0..n-1 in
// order, so the additions of a row are one chain.  A workgroup takes 64 rows:
// wave 0 adds, one row per lane, while the other seven waves generate the next
// kDiagCols columns into LDS (generating costs about eight times the add).
// With a thread per row doing both, a matrix of 10^4 rows gave the device 157
// waves: 382 us at n = 10007, now 99 us; 2.48 -> 1.80 ms at n = 61440 (VALU
// bound there, 75 clocks an element).
constexpr int kDiagPer = 8;                  // columns per generating wave and chunk
constexpr int kDiagCols = 7 * kDiagPer;

__global__ __launch_bounds__(512) void gen_diag_kernel(int64_t n, uint64_t x1, int64_t i0, int64_t cnt, LcgCoeff jn,
                                                       LcgCoeff jn2, LcgCoeff jchunk, double *__restrict__ d)
{
    __shared__ double buf[2][kDiagCols][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t t = static_cast<int64_t>(blockIdx.x) * 64 + lane;
    const int64_t i = i0 + (t < cnt ? t : cnt - 1);
    const int64_t chunks = (n + kDiagCols - 1) / kDiagCols;
    if (wave == 0) {
        double sum = 0.0;
        for (int64_t p = 0; p < chunks; ++p) {
            __syncthreads();
            const double *col = &buf[p & 1][0][lane];
#pragma unroll
            for (int c0 = 0; c0 < kDiagCols; c0 += 14) {
                double v[14];
#pragma unroll
                for (int c = 0; c < 14; ++c) v[c] = col[64 * (c0 + c)];
#pragma unroll
                for (int c = 0; c < 14; ++c) sum = __dadd_rn(sum, fabs(v[c]));
            }
        }
        if (t < cnt) d[t] = sum;
    } else {
        int64_t j = (wave - 1) * kDiagPer;
        const int64_t b0 = i0 + static_cast<int64_t>(blockIdx.x) * 64;   // the workgroup's first row
        // states of columns j and j + 1
        uint64_t s0 = lcg_jump_lanes<6>(x1, static_cast<uint64_t>(b0) + static_cast<uint64_t>(n) * static_cast<uint64_t>(j),
                                        static_cast<uint32_t>(i - b0));
        uint64_t s1 = jn.a * s0 + jn.c;
        for (int64_t p = 0; p < chunks; ++p) {
            double *col = &buf[p & 1][(wave - 1) * kDiagPer][lane];
            // adding +0.0 leaves a non-negative sum unchanged: the diagonal
            // and the columns past the last are stored as zeros
            auto columns = [&](auto mask) {
#pragma unroll
                for (int c = 0; c < kDiagPer; c += 2) {
                    double v0 = lcg_value(s0), v1 = lcg_value(s1);
                    if (decltype(mask)::value && (j + c == i || j + c >= n)) v0 = 0.0;
                    if (decltype(mask)::value && (j + c + 1 == i || j + c + 1 >= n)) v1 = 0.0;
                    col[64 * c] = v0;
                    col[64 * (c + 1)] = v1;
                    s0 = jn2.a * s0 + jn2.c;
                    s1 = jn2.a * s1 + jn2.c;
                }
            };
            if (j + kDiagPer <= n && (j + kDiagPer <= b0 || j >= b0 + 64))
                columns(std::false_type{});
            else
                columns(std::true_type{});
            s0 = jchunk.a * s0 + jchunk.c;   // past the other waves' columns
            s1 = jchunk.a * s1 + jchunk.c;
            j += kDiagCols;
            __syncthreads();
        }
    }
}

// pcolvgen (matgen.hpp:193-207): b_i = value of state 1 + i + n*n.
__global__ void gen_rhs_kernel(int64_t n, uint64_t x1, int64_t i0, int64_t cnt,
                               double *__restrict__ b)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= cnt) return;
    uint64_t idx = static_cast<uint64_t>(i0 + t) + static_cast<uint64_t>(n) * static_cast<uint64_t>(n);
    b[t] = lcg_value(lcg_jump(x1, idx));
}

int launch_gen_matrix(int64_t n, uint64_t seed, int64_t i0, int64_t j0, int64_t m, int64_t k,
                      const double *d, float *A, int64_t lda, int accumulate, hipStream_t s,
                      const uint16_t *P, int64_t ldp, float pscale, const uint16_t *Q)
{
    if (m <= 0 || k <= 0) return HPLAI_OK;
    const int64_t row_blocks = ceil_div(m, kGenRows);
    const int64_t col_groups = ceil_div(k, kGenCols);
    const LcgCoeff jn = lcg_pow_host(static_cast<uint64_t>(n));
    // split launches so the grid stays below 2^32 threads
    const int64_t max_groups = row_blocks < kGridX ? kGridX / row_blocks : 1;
    for (int64_t g0 = 0; g0 < col_groups; g0 += max_groups) {
        int64_t g = col_groups - g0 < max_groups ? col_groups - g0 : max_groups;
        int64_t jj = g0 * kGenCols;
        int64_t kk = (k - jj) < g * kGenCols ? (k - jj) : g * kGenCols;
        if (P == nullptr && !accumulate) {
            hipLaunchKernelGGL(gen_plain_kernel, dim3(static_cast<unsigned>(row_blocks * g)), dim3(kGenRows), 0, s,
                               static_cast<uint64_t>(n), lcg_init(seed), i0, j0 + jj, m, kk, row_blocks, jn,
                               lcg_pow_host(static_cast<uint64_t>(n) * kGenPlain), d, A + jj * lda, lda);
            HPLAI_HIP(hipGetLastError());
            continue;
        }
        hipLaunchKernelGGL(gen_matrix_kernel, dim3(static_cast<unsigned>(row_blocks * g)),
                           dim3(kGenRows), 0, s, n, lcg_init(seed), i0, j0 + jj, m, kk, row_blocks,
                           jn, d, A + jj * lda, lda, accumulate, P != nullptr ? P + jj * ldp : nullptr,
                           Q != nullptr ? Q + jj * ldp : nullptr, ldp, pscale);
        HPLAI_HIP(hipGetLastError());
    }
    return HPLAI_OK;
}

// Back-buffer write-back (bb_writeback_b_impl_fp16, back_buffer.cpp:32-55 in
// its non-SVE form): the front P (the trailing updates' target) folds into
// the back Q with a compensated sum in FP16 arithmetic, Q := fl(Q + P/32),
// P := 32 (P/32 - (Q_new - Q)), so P keeps the rounding error.
__global__ __launch_bounds__(256) void backbuffer_kernel(int64_t m, int64_t k, uint16_t *__restrict__ P,
                                                         uint16_t *__restrict__ Q, int64_t ldp)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= m) return;
    const int64_t j = blockIdx.y;
    uint16_t *pp = P + j * ldp + i, *qq = Q + j * ldp + i;
    const _Float16 t0 = __builtin_bit_cast(_Float16, *qq);
    const _Float16 t1 = __builtin_bit_cast(_Float16, *pp) * static_cast<_Float16>(1.0f / 32.0f);
    const _Float16 t2 = t0 + t1;
    const _Float16 t3 = t2 - t0;
    const _Float16 t4 = t1 - t3;
    *qq = __builtin_bit_cast(uint16_t, t2);
    *pp = __builtin_bit_cast(uint16_t, static_cast<_Float16>(t4 * static_cast<_Float16>(32.0f)));
    (void)k;
}

int launch_backbuffer(int64_t m, int64_t k, uint16_t *P, uint16_t *Q, int64_t ldp, hipStream_t s)
{
    if (m <= 0 || k <= 0) return HPLAI_OK;
    for (int64_t j0 = 0; j0 < k; j0 += 65535) {
        const int64_t kk = k - j0 < 65535 ? k - j0 : 65535;
        hipLaunchKernelGGL(backbuffer_kernel, dim3(static_cast<unsigned>(ceil_div(m, 256)), static_cast<unsigned>(kk)),
                           dim3(256), 0, s, m, kk, P + j0 * ldp, Q + j0 * ldp, ldp);
        HPLAI_HIP(hipGetLastError());
    }
    return HPLAI_OK;
}

int launch_gen_diag(int64_t n, uint64_t seed, int64_t i0, int64_t cnt, double *d, hipStream_t s)
{
    if (cnt <= 0) return HPLAI_OK;
    const LcgCoeff jn = lcg_pow_host(static_cast<uint64_t>(n));
    const LcgCoeff jn2 = lcg_mul(jn, jn);
    LcgCoeff jchunk{1, 0};
    for (int c = 0; c < kDiagCols - kDiagPer; c += 2) jchunk = lcg_mul(jn2, jchunk);
    hipLaunchKernelGGL(gen_diag_kernel, dim3(static_cast<unsigned>(ceil_div(cnt, 64))), dim3(512), 0, s, n,
                       lcg_init(seed), i0, cnt, jn, jn2, jchunk, d);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

int launch_gen_rhs(int64_t n, uint64_t seed, int64_t i0, int64_t cnt, double *b, hipStream_t s)
{
    if (cnt <= 0) return HPLAI_OK;
    hipLaunchKernelGGL(gen_rhs_kernel, dim3(static_cast<unsigned>(ceil_div(cnt, 256))), dim3(256), 0,
                       s, n, lcg_init(seed), i0, cnt, b);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

}  // namespace hplai
