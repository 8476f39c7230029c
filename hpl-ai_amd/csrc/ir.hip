// ir.hip — FP64 iterative-refinement kernels on gfx950: the matrix-free
// residual GEMV (A regenerated from the LCG), the blocked triangular solves
// with FP32 factors and FP64 vectors, norms, vector updates and the factor
// checksum.
#include <type_traits>

#include "device_common.hpp"
#include "internal.hpp"

namespace hplai {

// ---------------------------------------------------------------------------
// otf_gemv (panel_gemv.hpp:57-83, otf_gemv.cpp:5-131).
// Pass 1: partial[c][i] = sum_{j in chunk c, j != i} (double)(int64)state_ij * x_j
// (raw integers, like otf_gemv_kernel; the 2^-64-style scale is applied once;
// one 64-bit integer's halves are summed apart).
// Pass 2: y_i += alpha * (scale * sum_c partial[c][i] + d_i x_i), chunks in order.
// ---------------------------------------------------------------------------
constexpr int kGemvRows = 256;
constexpr int kGemvChunk = 2048;

// Columns per workgroup: as many as leave the device about eight workgroups
// per CU, since a workgroup pays for its jump into the stream, 64 at least.
// (2048 for every n left n = 1134 five workgroups: 22 us.)  The partial sums
// stay under 32 MiB up to n = 92160 either way.
static int otf_gemv_chunk(int64_t n)
{
    int chunk = kGemvChunk;
    while (chunk > 64 && ceil_div(n, kGemvRows) * ceil_div(n, chunk) < 2048) chunk /= 2;
    return chunk;
}

// What bounds it: VALU issue.  An element is one 64-bit LCG step (a 32 x 32 ->
// 64 multiply-add and two 32-bit multiplies), the conversion of its two halves
// and an FMA for each half into a sum of its own (one more rounding step per
// element than converting the 64-bit integer first, without its shift and add,
// and no less exact: the high sum is scaled and joined once).  x is uniform
// over the wave and read through the scalar cache.
__global__ __launch_bounds__(kGemvRows) void otf_gemv_partial_kernel(
    int64_t n, uint64_t x1, int chunk, int row_blocks, LcgCoeff jn, LcgCoeff jn2, const double *__restrict__ x,
    double *__restrict__ partial)
{
    const int block = static_cast<int>(block_number(blockIdx.y));
    const int rb = block % row_blocks, cb = block / row_blocks;
    const int64_t r0 = static_cast<int64_t>(rb) * kGemvRows, j0 = static_cast<int64_t>(cb) * chunk;
    if (j0 >= n) return;
    const int len = static_cast<int>(j0 + chunk < n ? chunk : n - j0);
    const int64_t i = r0 + threadIdx.x;
    uint64_t s0 = lcg_jump_lanes<8>(x1, static_cast<uint64_t>(r0) + static_cast<uint64_t>(n) * static_cast<uint64_t>(j0),
                                    threadIdx.x);
    uint64_t s1 = jn.a * s0 + jn.c;
    const double *xc = x + j0;
    double h0 = 0.0, l0 = 0.0, h1 = 0.0, l1 = 0.0;
    auto add = [](uint64_t s, double xv, double &h, double &l) {
        h = fma(static_cast<double>(static_cast<int32_t>(s >> 32)), xv, h);
        l = fma(static_cast<double>(static_cast<uint32_t>(s)), xv, l);
    };
    int t = 0;
    const int idiag = static_cast<int>(i - j0);   // in [0, len) when the diagonal is in this chunk
    // columns t .. te - 1 (te - t a multiple of 8 but for the last range); with
    // MASK the diagonal element counts as zero
    auto range = [&](auto mask, int te) {
        constexpr bool MASK = decltype(mask)::value;
        for (; t + 8 <= te; t += 8) {
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                add(MASK && t + u == idiag ? 0 : s0, xc[t + u], h0, l0);
                add(MASK && t + u + 1 == idiag ? 0 : s1, xc[t + u + 1], h1, l1);
                s0 = jn2.a * s0 + jn2.c;
                s1 = jn2.a * s1 + jn2.c;
            }
        }
        for (; t < te; ++t) {
            add(MASK && t == idiag ? 0 : s0, xc[t], h0, l0);
            const uint64_t next = jn2.a * s0 + jn2.c;
            s0 = s1;
            s1 = next;
        }
    };
    // the row block's own columns, where the diagonal is
    const int64_t d0 = r0 - j0, d1 = d0 + kGemvRows;
    if (d1 > 0 && d0 < len) {
        if (d0 > 0) range(std::false_type{}, static_cast<int>(d0));
        range(std::true_type{}, static_cast<int>(d1 < len ? d1 : len));
    }
    range(std::false_type{}, len);
    if (i < n) partial[static_cast<int64_t>(cb) * n + i] = fma(h0 + h1, 0x1p32, l0 + l1);
}

__global__ void otf_gemv_reduce_kernel(int64_t n, int64_t nchunks, double alpha,
                                       const double *__restrict__ d, const double *__restrict__ x,
                                       const double *__restrict__ partial, double *__restrict__ y)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int64_t c = 0; c < nchunks; ++c) s += partial[c * n + i];
    const double ax = fma(s, 0x1.fffffffffffffP-65, d[i] * x[i]);
    y[i] = fma(alpha, ax, y[i]);
}

int64_t otf_gemv_work_doubles(int64_t n) { return ceil_div(n, otf_gemv_chunk(n)) * n; }

int launch_otf_gemv(int64_t n, uint64_t seed, const double *d, double alpha, const double *x,
                    double *y, double *work, hipStream_t s)
{
    if (n <= 0) return HPLAI_OK;
    const int chunk = otf_gemv_chunk(n);
    const int64_t row_blocks = ceil_div(n, kGemvRows);
    const int64_t nchunks = ceil_div(n, chunk);
    const LcgCoeff jn = lcg_pow_host(static_cast<uint64_t>(n));
    const LcgCoeff jn2 = lcg_mul(jn, jn);
    hipLaunchKernelGGL(otf_gemv_partial_kernel, dim3(grid_x(row_blocks * nchunks), grid_rest(row_blocks * nchunks)),
                       dim3(kGemvRows), 0, s, n, lcg_init(seed), chunk, static_cast<int>(row_blocks), jn, jn2, x, work);
    HPLAI_HIP(hipGetLastError());
    hipLaunchKernelGGL(otf_gemv_reduce_kernel, dim3(static_cast<unsigned>(ceil_div(n, 256))),
                       dim3(256), 0, s, n, nchunks, alpha, d, x, work, y);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

// ---------------------------------------------------------------------------
// The solve's own triangular solves (panel_trsvL / panel_trsvU,
// panel_trsv.hpp:310-758; trisolve.hip has the general ones): one right-hand
// side, diagonal blocks through the inverses the LU stored.
// ---------------------------------------------------------------------------
constexpr int kTrsvMax = 512;

// y(0:m) -= P(m x w) * xb(0:w), P column-major (ttgemv, panel_trsv.hpp:10-45).
// Workgroup = 64 rows x 16 column groups; the partial sums of a row are added
// in a fixed order through LDS.  A thread's 32 loads are all in flight: with 4
// groups of 128 columns, 8 loads at a time, the latencies one after the other
// were 12 us of a 7680 x 512 update, now 7.  Workgroup 0 also stores xb into
// xcopy(0:w): the solved segment goes from its scratch copy to x while the
// update runs.
constexpr int kGemvRowsT = 64, kGemvGroups = 16, kGemvCols = kTrsvMax / kGemvGroups;

__global__ __launch_bounds__(kGemvRowsT * kGemvGroups) void trsv_gemv_kernel(
    int64_t m, int w, const float *__restrict__ P, int64_t lda, const double *__restrict__ xb, double *__restrict__ y,
    double *__restrict__ xcopy)
{
    __shared__ double xs[kTrsvMax];
    __shared__ double part[kGemvGroups][kGemvRowsT];
    const int lr = threadIdx.x % kGemvRowsT, g = __builtin_amdgcn_readfirstlane(threadIdx.x / kGemvRowsT);
    const int64_t r = static_cast<int64_t>(blockIdx.x) * kGemvRowsT + lr;
    const int cw = (w + kGemvGroups - 1) / kGemvGroups, c0 = g * cw;
    const float *pr = P + (r < m ? r : m - 1);
    float v[kGemvCols];
#pragma unroll
    for (int q = 0; q < kGemvCols; ++q) v[q] = pr[static_cast<int64_t>(min(c0 + q, w - 1)) * lda];
    const int c = threadIdx.x;
    if (c < w) {
        xs[c] = xb[c];
        if (blockIdx.x == 0) xcopy[c] = xs[c];
    }
    __syncthreads();
    double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
    for (int q = 0; q < kGemvCols; q += 2) {
        if (q < cw && c0 + q < w) acc0 = fma(static_cast<double>(v[q]), xs[c0 + q], acc0);
        if (q + 1 < cw && c0 + q + 1 < w) acc1 = fma(static_cast<double>(v[q + 1]), xs[c0 + q + 1], acc1);
    }
    part[g][lr] = acc0 + acc1;
    __syncthreads();
    if (g == 0 && r < m) {
        double sum = part[0][lr];
#pragma unroll
        for (int q = 1; q < kGemvGroups; ++q) sum += part[q][lr];
        y[r] -= sum;
    }
}

static void launch_gemv(int64_t m, int w, const float *P, int64_t lda, const double *xb, double *y, double *xcopy,
                        hipStream_t s)
{
    hipLaunchKernelGGL(trsv_gemv_kernel, dim3(static_cast<unsigned>(ceil_div(m, kGemvRowsT))),
                       dim3(kGemvRowsT * kGemvGroups), 0, s, m, w, P, lda, xb, y, xcopy);
}

// The block solves with the diagonal blocks applied through the inverses the
// LU stored (packed, one set per block at inv + q inv_stride): x_q := Tinv_q r_q into the scratch
// segment xsc (bs doubles), then the update of the other rows from xsc, whose
// workgroup 0 also moves x_q into x.  One right-hand side; n % bs == 0 and
// tri_inverse_ok(bs).
int launch_trsv_lower_inv(int64_t n, int bs, const float *LU, int64_t lda, double *x, const float *inv,
                          int64_t inv_stride, double *xsc, hipStream_t s)
{
    HPLAI_CHECK(tri_inverse_ok(bs) && n % bs == 0, "trsv: no stored inverses for bs=%d", bs);
    for (int64_t kb = 0; kb < n; kb += bs) {
        int rc = launch_tri_trsv(false, bs, inv + (kb / bs) * inv_stride, x + kb, xsc, s);
        if (rc) return rc;
        const int64_t m = n - kb - bs;
        if (m > 0) {
            launch_gemv(m, bs, LU + kb * lda + kb + bs, lda, xsc, x + kb + bs, x + kb, s);
            HPLAI_HIP(hipGetLastError());
        } else {
            HPLAI_HIP(hipMemcpyAsync(x + kb, xsc, sizeof(double) * bs, hipMemcpyDeviceToDevice, s));
        }
    }
    return HPLAI_OK;
}

int launch_trsv_upper_inv(int64_t n, int bs, const float *LU, int64_t lda, double *x, const float *inv,
                          int64_t inv_stride, double *xsc, hipStream_t s)
{
    HPLAI_CHECK(tri_inverse_ok(bs) && n % bs == 0, "trsv: no stored inverses for bs=%d", bs);
    for (int64_t kb = n - bs; kb >= 0; kb -= bs) {
        int rc = launch_tri_trsv(true, bs, inv + (kb / bs) * inv_stride, x + kb, xsc, s);
        if (rc) return rc;
        if (kb > 0) {
            launch_gemv(kb, bs, LU + kb * lda, lda, xsc, x, x + kb, s);
            HPLAI_HIP(hipGetLastError());
        } else {
            HPLAI_HIP(hipMemcpyAsync(x + kb, xsc, sizeof(double) * bs, hipMemcpyDeviceToDevice, s));
        }
    }
    return HPLAI_OK;
}

// ---------------------------------------------------------------------------
// norms and vector ops (panel_norm.hpp:8-41, panel.hpp:277-330)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void norm_inf_kernel(int64_t n, const double *__restrict__ x,
                                                        double *__restrict__ out)
{
    __shared__ double red[1024];
    double m = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) m = fmax(m, fabs(x[i]));
    red[threadIdx.x] = m;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + off]);
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

__global__ void vec_div_kernel(int64_t n, const double *num, const double *den, double *out)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) out[i] = num[i] / den[i];
}

__global__ void vec_add_kernel(int64_t n, const double *x, double *y)
{
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) y[i] += x[i];
}

int launch_norm_inf(int64_t n, const double *x, double *out, hipStream_t s)
{
    hipLaunchKernelGGL(norm_inf_kernel, dim3(1), dim3(1024), 0, s, n, x, out);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

int launch_vec_div(int64_t n, const double *num, const double *den, double *out, hipStream_t s)
{
    if (n <= 0) return HPLAI_OK;
    hipLaunchKernelGGL(vec_div_kernel, dim3(static_cast<unsigned>(ceil_div(n, 256))), dim3(256), 0, s,
                       n, num, den, out);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

int launch_vec_add(int64_t n, const double *x, double *y, hipStream_t s)
{
    if (n <= 0) return HPLAI_OK;
    hipLaunchKernelGGL(vec_add_kernel, dim3(static_cast<unsigned>(ceil_div(n, 256))), dim3(256), 0, s,
                       n, x, y);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

// ---------------------------------------------------------------------------
// panel_check fingerprint (panel_check.hpp:9-65): sum |diag|, |strict U|,
// |strict L| in FP64.  Column sums then a fixed-order final pass, so the
// result is deterministic.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void checksum_col_kernel(int64_t n, const float *__restrict__ LU,
                                                           int64_t lda, double *__restrict__ cols)
{
    __shared__ double red[3][256];
    const int64_t j = blockIdx.x;
    const float *c = LU + j * lda;
    double su = 0.0, sl = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        const double v = fabs(static_cast<double>(c[i]));
        if (i < j) su += v;
        else if (i > j) sl += v;
    }
    red[0][threadIdx.x] = su;
    red[1][threadIdx.x] = sl;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            red[0][threadIdx.x] += red[0][threadIdx.x + off];
            red[1][threadIdx.x] += red[1][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        cols[j] = fabs(static_cast<double>(c[j]));
        cols[n + j] = red[0][0];
        cols[2 * n + j] = red[1][0];
    }
}

__global__ __launch_bounds__(1024) void checksum_final_kernel(int64_t n, const double *__restrict__ cols,
                                                              double *__restrict__ out)
{
    __shared__ double red[1024];
    for (int q = 0; q < 3; ++q) {
        double s = 0.0;
        for (int64_t j = threadIdx.x; j < n; j += 1024) s += cols[q * n + j];
        red[threadIdx.x] = s;
        __syncthreads();
        for (int off = 512; off > 0; off >>= 1) {
            if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
            __syncthreads();
        }
        if (threadIdx.x == 0) out[q] = red[0];
        __syncthreads();
    }
}

int launch_checksum(int64_t n, const float *LU, int64_t lda, double *cols, double *out3, hipStream_t s)
{
    hipLaunchKernelGGL(checksum_col_kernel, dim3(static_cast<unsigned>(n)), dim3(256), 0, s, n, LU, lda,
                       cols);
    hipLaunchKernelGGL(checksum_final_kernel, dim3(1), dim3(1024), 0, s, n, cols, out3);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

}  // namespace hplai
