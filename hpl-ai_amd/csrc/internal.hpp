// internal.hpp — host-side plumbing shared by the library's translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <string>

#include "../../include/hplai.h"

namespace hplai {
// temporaries of the asynchronous entry points, one buffer per stream (memory.hip)
struct StreamScratch {
    struct Entry {
        hipStream_t stream;
        void *p;
        hipEvent_t done;   // end of the last use
        size_t bytes;
        bool owned;        // its stream's buffer, not an outgrown one
    };
    static constexpr int kMax = 32;
    static constexpr size_t kTotal = size_t(1) << 30;   // kept in all
    std::mutex mu;
    Entry entries[kMax];
    int count = 0;
    size_t total = 0;
    Entry *find(hipStream_t stream);
    Entry *replace(int device, Entry *old, hipStream_t stream, size_t bytes, hipError_t *err);
    void clear(int device);
};
}  // namespace hplai

struct hplai_ctx_s {
    int device = 0;
    int num_cu = 0;
    hipStream_t side = nullptr;    // second stream for look-ahead panel work
    hipStream_t bulk = nullptr;    // third stream: the panel's rows below the outer block
    hipEvent_t ev[8] = {};
    // buffers kept by hplai_solve(keep_factors)
    float *A = nullptr;
    int64_t n = 0, lda = 0;
    double *x = nullptr;
    size_t A_bytes = 0, x_bytes = 0;   // block_free's sizes of the two
    bool cache_open = false;
    hplai::StreamScratch pool;
    // device address of this device's scratch array (hplai_otf_gemv_f64_noalloc)
    void *scratch = nullptr;
};

namespace hplai {

void set_error(const char *fmt, ...);
int hip_fail(hipError_t e, const char *what);

#define HPLAI_HIP(call)                                              \
    do {                                                             \
        hipError_t _e = (call);                                      \
        if (_e != hipSuccess) return ::hplai::hip_fail(_e, #call);   \
    } while (0)

#define HPLAI_CHECK(cond, ...)                                       \
    do {                                                             \
        if (!(cond)) {                                               \
            ::hplai::set_error(__VA_ARGS__);                         \
            return HPLAI_EINVAL;                                     \
        }                                                            \
    } while (0)

// ---- device memory (memory.hip) ----
int block_cache_open(int device, size_t device_bytes);
void block_cache_close(int device);
bool block_cache_empty(int device);
hipError_t device_malloc(int device, void **p, size_t bytes);
hipError_t block_alloc(int device, void **p, size_t *bytes);
void block_free(int device, void *p, size_t bytes);
bool block_put(int device, void *p, size_t bytes);

// `bytes` of scratch for one call's kernels on `stream`, from construction to
// the end of the scope that enqueues them.
constexpr size_t kScratchMax = size_t(512) << 20;   // larger leases are allocated and freed in stream order
class ScratchLease {
public:
    ScratchLease(hplai_ctx ctx, hipStream_t stream, size_t bytes);
    ~ScratchLease();
    ScratchLease(const ScratchLease &) = delete;
    ScratchLease &operator=(const ScratchLease &) = delete;
    template <typename T>
    T *as() const
    {
        return static_cast<T *>(ptr);
    }
    void *ptr = nullptr;
    int rc = HPLAI_OK;

private:
    hipStream_t stream_;
    std::unique_lock<std::mutex> lock_;
    hipEvent_t done_ = nullptr;
    bool async_ = false;
};

inline hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }
__host__ __device__ inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
// x and y (or z) of a grid of `blocks` workgroups and up to x - 1 more: a launch
// has at most 2^32 threads along a dimension (block_number)
constexpr int64_t kGridX = int64_t(1) << 22;
inline unsigned grid_x(int64_t blocks) { return static_cast<unsigned>(blocks < kGridX ? blocks : kGridX); }
inline unsigned grid_rest(int64_t blocks) { return static_cast<unsigned>(ceil_div(blocks, kGridX)); }

// ---- kernel launchers (no argument validation; callers validate) ----
// accumulate != 0: A += generated block (lazy initialisation); P (FP16,
// leading dimension ldp, may be NULL): A += pscale * P as well (the FP16
// trailing storage's partial sums of the block)
int launch_gen_matrix(int64_t n, uint64_t seed, int64_t i0, int64_t j0, int64_t m, int64_t k,
                      const double *d, float *A, int64_t lda, int accumulate, hipStream_t s,
                      const uint16_t *P = nullptr, int64_t ldp = 0, float pscale = 0.0f,
                      const uint16_t *Q = nullptr);
// back-buffer write-back of an m x k block of the FP16 trailing storage:
// Q := fl16(Q + P / 32), P := the rounding error times 32
int launch_backbuffer(int64_t m, int64_t k, uint16_t *P, uint16_t *Q, int64_t ldp, hipStream_t s);
int launch_gen_diag(int64_t n, uint64_t seed, int64_t i0, int64_t cnt, double *d, hipStream_t s);
// Higham's HPL-AI matrix (higham.hip)
int higham_coeffs(int64_t n, double cond, double rho, double *alpha, double *beta);
int launch_gen_higham(double alpha, double beta, int64_t i0, int64_t j0, int64_t m, int64_t k, float *A,
                      int64_t lda, int accumulate, hipStream_t s);
int launch_higham_diag(double alpha, double beta, int64_t i0, int64_t cnt, double *d, hipStream_t s);
int64_t higham_gemv_work_doubles(int64_t n);
int launch_higham_gemv(int64_t n, double alpha, double beta, double scale, const double *x, double *y,
                       double *work, hipStream_t s);
int launch_higham_norm(int64_t n, double alpha, double beta, double *ones, double *rows, double *work,
                       double *out, hipStream_t s);
int launch_gen_rhs(int64_t n, uint64_t seed, int64_t i0, int64_t cnt, double *b, hipStream_t s);

// LU of an n x n block (n <= 1024) in place.  tri: tri_floats(n), packed
// (device_common.hpp): the full inverses of the triangles (full), or scratch
// (may be NULL up to getrf_scratch_floats(n) == 0).
int launch_getrf(int n, float *A, int64_t lda, int *info, float *tri, bool full, hipStream_t s);
int64_t getrf_scratch_floats(int n);
int64_t tri_floats(int b);
// the same inverses of a block that is already factored, without join those of
// its 32-blocks only; sides: 1 L, 2 U, 3 both
int launch_tri_inverse(int b, const float *LU, int64_t lda, float *tri, int sides, bool join, hipStream_t s);
// tri: the packed inverses of the factored diagonal block
// half: where the results also go as FP16 (dst NULL: nowhere), operand rows ld
// bytes apart, each slice padded to whole 32-blocks; packed as for launch_quantize
struct TrsmHalf {
    void *dst = nullptr;
    int64_t ld = 0;
    int packed = 0;
};
int launch_trsm_l(int64_t m, int b, const float *tri, float *L, int64_t ldl, float *amax, int tb, hipStream_t s,
                  TrsmHalf half = {});
int launch_trsm_u(int b, int64_t n, const float *tri, float *U, int64_t ldu, float *amax, int tb, hipStream_t s,
                  TrsmHalf half = {});
// A panel of m columns (up: P := L^-1 P) or rows (P := P U^-1) with the caller's
// triangle in T; tri: tri_floats(b) of scratch
int launch_trsm_panel(bool up, int64_t m, int b, const float *T, int64_t ldt, float *tri, float *P, int64_t ldp,
                      hipStream_t s);
// amax: per-tile maxima of |src|; NULL: the exponents are in exps (FMT_F16: 0).
// packed: dst in the panel-packed layout (packed_off), rows a multiple of 256 from its base.
int launch_quantize(int fmt, int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds,
                    void *dst, int64_t ldd, const float *amax, int32_t *exps, hipStream_t s,
                    bool packed = false, int slots = 1);
// Exponents of a panel's tiles for launch_quantize without amax: written to
// exps when one workgroup serves a tile (tile_amax_splits 1, amax NULL), else
// the maxima to amax: tile_amax_slots a tile, one slot a part, or one where all
// parts meet (zeroed by the caller).
constexpr int kAmaxSlots = 4;
int tile_amax_splits(int64_t m, int64_t k, int tb, int num_cu);
int tile_amax_slots(int64_t m, int64_t k, int tb, int num_cu);
int launch_tile_amax(int fmt, int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds, float *amax,
                     int32_t *exps, int num_cu, hipStream_t s);
int launch_fill_f32(float *p, int64_t cnt, float v, hipStream_t s);
// packed: Lq and Uq in the panel-packed layout (packed_off) from their bases.
int launch_schur(int fmt, int64_t m, int64_t n, int nslices, int kslice, const void *Lq,
                 int64_t ldl, const int32_t *eL, int64_t ldel, const void *Uq, int64_t ldu,
                 const int32_t *eU, int64_t ldeu, int tb, float *C, int64_t ldc, int num_cu,
                 hipStream_t s, bool packed = false, hplai_ctx ctx = nullptr);
// The same update of the FP16 trailing storage: C := fp16(C - cscale * L U),
// C holding cscale times the partial sums (m, n multiples of 128).
int launch_schur_c16(int fmt, int64_t m, int64_t n, int nslices, int kslice, const void *Lq,
                     int64_t ldl, const int32_t *eL, int64_t ldel, const void *Uq, int64_t ldu,
                     const int32_t *eU, int64_t ldeu, int tb, uint16_t *C, int64_t ldc, float cscale,
                     int num_cu, hipStream_t s, bool packed = false);
// true when launch_schur runs the streamed 256 x 256 kernel for this shape
bool schur_large_tiles(int fmt, int64_t m, int64_t n, int64_t K, int tb, int num_cu);

// the reference's column-major gemmschur seam (gemmschur.hip): both operands
// staged K-contiguous with K padded to 64 in `scratch`
// (gemmschur_scratch_bytes), then C(n x m) -= A B with FP32 accumulation
int64_t gemmschur_scratch_bytes(int64_t n, int64_t m, int64_t k);
int launch_gemmschur_f16(int64_t n, int64_t m, int64_t k, const uint16_t *a, int64_t lda, const uint16_t *b,
                         int64_t ldb, float *c, int64_t ldc, uint16_t *scratch, int num_cu, hipStream_t s);

int launch_otf_gemv(int64_t n, uint64_t seed, const double *d, double alpha, const double *x,
                    double *y, double *work, hipStream_t s);
int64_t otf_gemv_work_doubles(int64_t n);
// address of the no-allocation scratch array on `device` (current), looked up once per device
int noalloc_setup(int device, void **out);
// X := L^-1 X or U^-1 X, and X := (L U)^-1 X or (L U)^-T X, with the triangles
// of LU; X FP64, nrhs columns with stride ldx (trisolve.hip)
int64_t tri_solve_work_doubles(int64_t n, int nrhs);
int launch_tri_solve(bool upper, int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs,
                     double *work, hipStream_t s);
int launch_lu_solve(bool trans, int64_t n, const float *LU, int64_t lda, double *X, int64_t ldx, int nrhs,
                    double *work, hipStream_t s);
// one column, diagonal blocks through stored inverses (FP32 entries)
bool tri_inverse_ok(int b);
int launch_tri_trsv(bool upper, int b, const float *tri, const double *xin, double *xout, hipStream_t s);
int launch_trsv_lower_inv(int64_t n, int bs, const float *LU, int64_t lda, double *x, const float *inv,
                          int64_t inv_stride, double *xsc, hipStream_t s);
int launch_trsv_upper_inv(int64_t n, int bs, const float *LU, int64_t lda, double *x, const float *inv,
                          int64_t inv_stride, double *xsc, hipStream_t s);
int launch_norm_inf(int64_t n, const double *x, double *out, hipStream_t s);
int launch_vec_div(int64_t n, const double *num, const double *den, double *out, hipStream_t s);
int launch_vec_add(int64_t n, const double *x, double *y, hipStream_t s);
// cols: 3 n doubles of scratch
int launch_checksum(int64_t n, const float *LU, int64_t lda, double *cols, double *out3, hipStream_t s);

}  // namespace hplai
