// dense64.hip — the passes over a dense FP64 matrix that the differentiable
// solve needs besides its products (no reference counterpart: the reference
// generates its matrix in FP32): the transposed FP32 copy that is factored and
// the infinity norm of A or A^T.  One read of A each; as elementwise library
// calls (transpose, cast, abs, sums, maximum) an 8192 x 64 solve with its
// gradient moved 4 GB more: 9.9 -> 9.3 ms.
#include "device_common.hpp"
#include "internal.hpp"

namespace hplai {

constexpr int kTile64 = 64;

// F(i, j) = (float)A(i, j), A row-major, F column-major: a 64 x 64 tile through
// LDS, whole lines on both sides.  HBM-bound: 12 n^2 bytes, 8192: 178 us (4.5 TB/s).
__global__ __launch_bounds__(256) void narrow_transpose_kernel(int64_t n, const double *__restrict__ A, int64_t lda,
                                                               float *__restrict__ F, int64_t ldf)
{
    __shared__ float T[kTile64][kTile64 + 1];
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kTile64, j0 = static_cast<int64_t>(blockIdx.y) * kTile64;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    double v[16];
    const int64_t j = j0 + tx < n ? j0 + tx : n - 1;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int64_t i = i0 + ty + 4 * u;
        v[u] = A[(i < n ? i : n - 1) * lda + j];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) T[ty + 4 * u][tx] = static_cast<float>(v[u]);
    __syncthreads();
    if (i0 + tx >= n) return;
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int64_t c = j0 + ty + 4 * u;
        if (c < n) F[c * ldf + i0 + tx] = T[tx][ty + 4 * u];
    }
}

// part[row] = sum_j |A(row, j)|: a wave per row
__global__ __launch_bounds__(256) void row_abs_sum_kernel(int64_t n, const double *__restrict__ A, int64_t lda,
                                                          double *__restrict__ part)
{
    const int lane = threadIdx.x & 63;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const double *a = A + row * lda;
    double s = 0.0;
    for (int64_t j0 = 0; j0 < n; j0 += 512) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t j = j0 + 64 * u + lane;
            v[u] = a[j < n ? j : n - 1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) s += j0 + 64 * u + lane < n ? fabs(v[u]) : 0.0;
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) part[row] = s;
}

// part[chunk n + col] = sum of |A(i, col)| over the chunk's rows
__global__ __launch_bounds__(256) void col_abs_sum_kernel(int64_t n, int64_t rows, const double *__restrict__ A,
                                                          int64_t lda, double *__restrict__ part)
{
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const int64_t r0 = blockIdx.y * rows, r1 = r0 + rows < n ? r0 + rows : n;
    const double *a = A + (j < n ? j : n - 1);
    double s = 0.0;
    for (int64_t i0 = r0; i0 < r1; i0 += 16) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = a[(i0 + u < r1 ? i0 + u : r1 - 1) * lda];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += i0 + u < r1 ? fabs(v[u]) : 0.0;
    }
    if (j < n) part[blockIdx.y * n + j] = s;
}

// *out = max over k < n of the sum of the C chunks' part[chunk n + k] (chunks
// past the last hold nothing); a NaN wins
template <int C>
__global__ __launch_bounds__(1024) void max_of_sums_kernel(int64_t n, int chunks, const double *__restrict__ part,
                                                           double *__restrict__ out)
{
    __shared__ double red[1024];
    constexpr int UN = 16 / C;   // 16 loads in flight
    double m = 0.0;
    for (int64_t k0 = threadIdx.x; k0 < n; k0 += 1024 * UN) {
        double v[UN][C];
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (int c = 0; c < C; ++c)
                v[u][c] = part[min(c, chunks - 1) * n + (k0 + 1024 * u < n ? k0 + 1024 * u : k0)];
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < C; ++c) s += c < chunks ? v[u][c] : 0.0;
            m = m > s || m != m ? m : s;
        }
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (threadIdx.x < off) {
            const double o = red[threadIdx.x + off], t = red[threadIdx.x];
            red[threadIdx.x] = t > o || t != t ? t : o;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

// rows of a column chunk: at most 16 chunks, of at least 128 rows
constexpr int kChunks = 16;
static int64_t chunk_rows(int64_t n) { return n <= 128 * kChunks ? 128 : ceil_div(n, kChunks); }

}  // namespace hplai

using namespace hplai;

extern "C" int hplai_narrow_transpose_f32(hplai_ctx ctx, int64_t n, const double *A, int64_t lda, float *F,
                                          int64_t ldf, void *stream)
{
    HPLAI_CHECK(ctx != nullptr, "null hplai_ctx");
    HPLAI_HIP(hipSetDevice(ctx->device));
    HPLAI_CHECK(n >= 0 && n <= (int64_t(1) << 21), "narrow_transpose: n %lld", (long long)n);
    if (n == 0) return HPLAI_OK;
    HPLAI_CHECK(A != nullptr && F != nullptr && lda >= n && ldf >= n, "narrow_transpose: NULL or a short leading dimension");
    const unsigned t = static_cast<unsigned>(ceil_div(n, kTile64));
    hipLaunchKernelGGL(narrow_transpose_kernel, dim3(t, t), dim3(256), 0, static_cast<hipStream_t>(stream), n, A, lda,
                       F, ldf);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

extern "C" int hplai_norm_abs_f64(hplai_ctx ctx, int trans, int64_t n, const double *A, int64_t lda, double *out_dev,
                                  void *stream)
{
    HPLAI_CHECK(ctx != nullptr, "null hplai_ctx");
    HPLAI_HIP(hipSetDevice(ctx->device));
    HPLAI_CHECK(n > 0 && n <= (int64_t(1) << 21) && A != nullptr && out_dev != nullptr && lda >= n,
                "norm_abs: n %lld, NULL or a short leading dimension", (long long)n);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int chunks = trans ? static_cast<int>(ceil_div(n, chunk_rows(n))) : 1;
    ScratchLease work(ctx, s, sizeof(double) * n * chunks);
    if (work.rc) return work.rc;
    if (trans)
        hipLaunchKernelGGL(col_abs_sum_kernel, dim3(static_cast<unsigned>(ceil_div(n, 256)), chunks), dim3(256), 0, s,
                           n, chunk_rows(n), A, lda, work.as<double>());
    else
        hipLaunchKernelGGL(row_abs_sum_kernel, dim3(static_cast<unsigned>(ceil_div(n, 4))), dim3(256), 0, s, n, A, lda,
                           work.as<double>());
    HPLAI_HIP(hipGetLastError());
    if (trans)
        hipLaunchKernelGGL(max_of_sums_kernel<kChunks>, dim3(1), dim3(1024), 0, s, n, chunks, work.as<double>(), out_dev);
    else
        hipLaunchKernelGGL(max_of_sums_kernel<1>, dim3(1), dim3(1024), 0, s, n, 1, work.as<double>(), out_dev);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}
