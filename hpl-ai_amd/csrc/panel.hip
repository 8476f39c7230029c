// panel.hip — the conversion of FP32 panels for the Schur update: per-tile
// |max| and the FP32 -> FP16 / FP8-e4m3 quantizer that feeds the MFMA kernels.
#include "device_common.hpp"
#include "internal.hpp"

namespace hplai {

template <int FMT>
__device__ __forceinline__ int amax_exponent(float a)
{
    return FMT == HPLAI_FMT_E4M3 ? e4m3_exponent(a) : tile_exponent(a, kF16MrFrac, kF16Er);
}

// ---------------------------------------------------------------------------
// per-tile max|x| of a panel (side 0: m x k L panel, tiles by row / tb;
// side 1: k x m U panel, tiles by column / tb).  blockIdx.x is the tile: `in`
// contiguous entries of `out` columns.  One workgroup per tile writes the
// tile's exponent itself; with blockIdx.y splitting the columns its maximum
// goes to the tile's slot of that part (slots 4), or they meet in amax
// (slots 1).  HBM-bound: 512 x 32768 in 18 us (26 with a workgroup per tile,
// which keeps 64 of the 256 CUs busy; 151 with a thread per row or column,
// whose loads of a U panel were 2 KB apart).
// ---------------------------------------------------------------------------
constexpr int kAmaxThreads = 1024;

template <int FMT>
__global__ __launch_bounds__(kAmaxThreads) void tile_amax_kernel(int side, int64_t m, int64_t k, int tb,
                                                                 const float *__restrict__ src, int64_t lds,
                                                                 float *__restrict__ amax, int slots,
                                                                 int32_t *__restrict__ exps)
{
    __shared__ float red[kAmaxThreads / 64];
    const int64_t t0 = static_cast<int64_t>(blockIdx.x) * tb;
    const int64_t h = m - t0 < tb ? m - t0 : tb;
    const int64_t in = side == 0 ? h : k, out = side == 0 ? k : h;
    const float *base = src + (side == 0 ? t0 : t0 * lds);
    const int64_t cols = (out + gridDim.y - 1) / gridDim.y, c0 = blockIdx.y * cols;
    const int64_t c1 = c0 + cols < out ? c0 + cols : out;
    // `lanes` threads along a column, the others on further columns
    const int tid = threadIdx.x;
    auto scan = [&](auto vec, int64_t n) {
        using V = decltype(vec);
        int lanes = 1;
        while (lanes < kAmaxThreads && lanes * 2 <= n) lanes *= 2;
        const int step = kAmaxThreads / lanes;
        float v = 0.0f;
        for (int64_t r = tid % lanes; r < n; r += lanes) {
            constexpr int UN = 8;   // loads in flight per thread
            for (int64_t c = c0 + tid / lanes; c < c1; c += static_cast<int64_t>(UN) * step) {
                V x[UN];
#pragma unroll
                for (int u = 0; u < UN; ++u) {
                    const int64_t cc = c + static_cast<int64_t>(u) * step;
                    x[u] = reinterpret_cast<const V *>(base + (cc < c1 ? cc : c) * lds)[r];
                }
#pragma unroll
                for (int u = 0; u < UN; ++u) {
                    if constexpr (sizeof(V) == 16)
                        v = fmaxf(fmaxf(v, fmaxf(fabsf(x[u].x), fabsf(x[u].y))), fmaxf(fabsf(x[u].z), fabsf(x[u].w)));
                    else
                        v = fmaxf(v, fabsf(x[u]));
                }
            }
        }
        return v;
    };
    const bool vec = in % 4 == 0 && lds % 4 == 0 && reinterpret_cast<uintptr_t>(base) % 16 == 0;
    float v = vec ? scan(float4{}, in / 4) : scan(0.0f, in);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int q = 1; q < kAmaxThreads / 64; ++q) v = fmaxf(v, red[q]);
        if (amax != nullptr && slots > 1)
            amax[static_cast<int64_t>(blockIdx.x) * kAmaxSlots + blockIdx.y] = v;
        else if (amax != nullptr)
            atomic_max_pos(amax + blockIdx.x, v);
        else
            exps[blockIdx.x] = amax_exponent<FMT>(v);
    }
}

// The same for tiles of fewer than kAmaxShort lines: a workgroup takes the whole
// tiles of up to 64 lines, rows along the lanes (side 0) or a column per wave
// (side 1), and the lines' maxima meet in LDS.
template <int FMT>
__global__ __launch_bounds__(kAmaxThreads) void tile_amax_short_kernel(int side, int64_t m, int64_t k, int tb, int group,
                                                                       const float *__restrict__ src, int64_t lds,
                                                                       int32_t *__restrict__ exps)
{
    constexpr int W = kAmaxThreads / 64, UN = 8;
    __shared__ float part[W][64], line[64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t l0 = static_cast<int64_t>(blockIdx.x) * group;
    const int cnt = m - l0 < group ? static_cast<int>(m - l0) : group;
    if (side == 0) {
        const float *row = src + l0 + min(lane, cnt - 1);
        float v = 0.0f;
        for (int64_t c = wave; c < k; c += W * UN) {
            float x[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) x[u] = row[(c + W * u < k ? c + W * u : c) * lds];
#pragma unroll
            for (int u = 0; u < UN; ++u) v = fmaxf(v, fabsf(x[u]));
        }
        part[wave][lane] = v;
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int q = 1; q < W; ++q) v = fmaxf(v, part[q][lane]);
            line[lane] = v;
        }
    } else {
        for (int j = wave; j < cnt; j += W) {
            const float *col = src + (l0 + j) * lds;
            float v = 0.0f;
            for (int64_t r = lane; r < k; r += 64 * UN) {
                float x[UN];
#pragma unroll
                for (int u = 0; u < UN; ++u) x[u] = col[r + 64 * u < k ? r + 64 * u : r];
#pragma unroll
                for (int u = 0; u < UN; ++u) v = fmaxf(v, fabsf(x[u]));
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
            if (lane == 0) line[j] = v;
        }
    }
    __syncthreads();
    if (tid * tb < cnt) {
        float v = line[tid * tb];
        for (int q = tid * tb + 1; q < min(tid * tb + tb, cnt); ++q) v = fmaxf(v, line[q]);
        exps[l0 / tb + tid] = amax_exponent<FMT>(v);
    }
}

__global__ void fill_f32_kernel(float *p, int64_t cnt, float v)
{
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t < cnt) p[t] = v;
}

// ---------------------------------------------------------------------------
// Quantizer (convert_left_panels / convert_right_panels, panel_trf.hpp:173-233)
// q = round(x * 2^e) with e from the tile's max (0 for plain FP16), the largest
// of its kAmaxSlots where slots > 1; without amax the exponents are in exps
// already.
// side 0: L panel m x k col-major -> dst[i*ldd + kk] (transposed through LDS)
// side 1: U panel k x m col-major -> dst[j*ldd + kk]
// ---------------------------------------------------------------------------
template <int FMT>
__device__ __forceinline__ int fmt_exponent(const float *amax, int slots, const int32_t *exps, int64_t tile)
{
    if (FMT == HPLAI_FMT_F16) return 0;
    if (amax != nullptr && slots > 1) {
        static_assert(kAmaxSlots == 4, "one float4 a tile");
        const float4 a = reinterpret_cast<const float4 *>(amax)[tile];
        return amax_exponent<FMT>(fmaxf(fmaxf(a.x, a.y), fmaxf(a.z, a.w)));
    }
    return amax != nullptr ? amax_exponent<FMT>(amax[tile]) : exps[tile];
}

template <int FMT, bool PACKED>
__global__ __launch_bounds__(256) void quant_l_kernel(int64_t m, int64_t k, int tb,
                                                      const float *__restrict__ src, int64_t lds,
                                                      void *__restrict__ dst, int64_t ldd,
                                                      const float *__restrict__ amax, int slots,
                                                      int32_t *__restrict__ exps)
{
    __shared__ float T[64][65];
    const int64_t r0 = block_number(blockIdx.z) * 64;
    const int64_t c0 = static_cast<int64_t>(blockIdx.y) * 64;
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    {
        const int64_t gr = r0 + tx;
        const float *col = src + (gr < m ? gr : m - 1);
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int64_t gc = c0 + ty + 4 * u;
            v[u] = col[(gc < k ? gc : k - 1) * lds];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) T[ty + 4 * u][tx] = (gr < m && c0 + ty + 4 * u < k) ? v[u] : 0.0f;
    }
    __syncthreads();
    // each thread writes 4 consecutive k values of one row (16 rows x 16 chunks per pass)
    for (int p = threadIdx.x; p < 64 * 16; p += 256) {
        const int r = p / 16, kc = (p % 16) * 4;
        const int64_t gr = r0 + r;
        if (gr >= m || c0 + kc >= k) continue;
        const int e = fmt_exponent<FMT>(amax, slots, exps, gr / tb);
        if (amax != nullptr && (gr % tb) == 0 && c0 == 0 && kc == 0) exps[gr / tb] = e;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = ldexp_fast(T[kc + q][r], e);
        const int nk = k - (c0 + kc) < 4 ? static_cast<int>(k - (c0 + kc)) : 4;
        if (FMT == HPLAI_FMT_E4M3) {
            uint8_t *d8 = static_cast<uint8_t *>(dst) + (PACKED ? packed_off(gr, c0 + kc, ldd) : gr * ldd + c0 + kc);
            uint32_t w = f32x4_to_e4m3x4(v[0], v[1], v[2], v[3]);
            if (nk == 4 && (reinterpret_cast<uintptr_t>(d8) & 3) == 0)
                *reinterpret_cast<uint32_t *>(d8) = w;   // one 4-byte store
            else
                for (int q = 0; q < nk; ++q) d8[q] = static_cast<uint8_t>(w >> (8 * q));
        } else {
            uint16_t *d16 = PACKED ? reinterpret_cast<uint16_t *>(static_cast<uint8_t *>(dst) +
                                                                packed_off(gr, 2 * (c0 + kc), 2 * ldd))
                                   : static_cast<uint16_t *>(dst) + gr * ldd + c0 + kc;
            if (nk == 4 && (reinterpret_cast<uintptr_t>(d16) & 7) == 0) {
                uint2 w;
                w.x = f32_to_f16_bits(v[0]) | (static_cast<uint32_t>(f32_to_f16_bits(v[1])) << 16);
                w.y = f32_to_f16_bits(v[2]) | (static_cast<uint32_t>(f32_to_f16_bits(v[3])) << 16);
                *reinterpret_cast<uint2 *>(d16) = w;     // one 8-byte store
            } else {
                for (int q = 0; q < nk; ++q) d16[q] = f32_to_f16_bits(v[q]);
            }
        }
    }
}

template <int FMT, bool PACKED>
__global__ __launch_bounds__(256) void quant_u_kernel(int64_t m, int64_t k, int tb,
                                                      const float *__restrict__ src, int64_t lds,
                                                      void *__restrict__ dst, int64_t ldd,
                                                      const float *__restrict__ amax, int slots,
                                                      int32_t *__restrict__ exps)
{
    // thread handles 4 consecutive rows (k index) of one column j
    const int64_t kq = ceil_div(k, 4);
    const int64_t t = block_number(blockIdx.y) * 256 + threadIdx.x;
    const int64_t j = t / kq, r = (t % kq) * 4;
    if (j >= m) return;
    const int e = fmt_exponent<FMT>(amax, slots, exps, j / tb);
    if (amax != nullptr && r == 0 && (j % tb) == 0) exps[j / tb] = e;
    const int nk = k - r < 4 ? static_cast<int>(k - r) : 4;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = q < nk ? ldexp_fast(src[j * lds + r + q], e) : 0.0f;
    if (FMT == HPLAI_FMT_E4M3) {
        uint8_t *d8 = static_cast<uint8_t *>(dst) + (PACKED ? packed_off(j, r, ldd) : j * ldd + r);
        uint32_t w = f32x4_to_e4m3x4(v[0], v[1], v[2], v[3]);
        if (nk == 4 && (reinterpret_cast<uintptr_t>(d8) & 3) == 0)
            *reinterpret_cast<uint32_t *>(d8) = w;
        else
            for (int q = 0; q < nk; ++q) d8[q] = static_cast<uint8_t>(w >> (8 * q));
    } else {
        uint16_t *d16 = PACKED ? reinterpret_cast<uint16_t *>(static_cast<uint8_t *>(dst) + packed_off(j, 2 * r, 2 * ldd))
                               : static_cast<uint16_t *>(dst) + j * ldd + r;
        if (nk == 4 && (reinterpret_cast<uintptr_t>(d16) & 7) == 0) {
            uint2 w;
            w.x = f32_to_f16_bits(v[0]) | (static_cast<uint32_t>(f32_to_f16_bits(v[1])) << 16);
            w.y = f32_to_f16_bits(v[2]) | (static_cast<uint32_t>(f32_to_f16_bits(v[3])) << 16);
            *reinterpret_cast<uint2 *>(d16) = w;
        } else {
            for (int q = 0; q < nk; ++q) d16[q] = f32_to_f16_bits(v[q]);
        }
    }
}

// 16 consecutive K values of one row scaled by 2^e and stored at d (16 bytes
// of e4m3 or 32 bytes of FP16; d 16-byte aligned).
template <int FMT>
__device__ __forceinline__ void store_q16(uint8_t *d, const float (&v)[16], int e)
{
    float x[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) x[q] = ldexp_fast(v[q], e);
    if constexpr (FMT == HPLAI_FMT_E4M3) {
        uint4 w;
        w.x = f32x4_to_e4m3x4(x[0], x[1], x[2], x[3]);
        w.y = f32x4_to_e4m3x4(x[4], x[5], x[6], x[7]);
        w.z = f32x4_to_e4m3x4(x[8], x[9], x[10], x[11]);
        w.w = f32x4_to_e4m3x4(x[12], x[13], x[14], x[15]);
        *reinterpret_cast<uint4 *>(d) = w;
    } else {
        uint32_t h[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
            h[q] = f32_to_f16_bits(x[2 * q]) | (static_cast<uint32_t>(f32_to_f16_bits(x[2 * q + 1])) << 16);
        *reinterpret_cast<uint4 *>(d) = uint4{h[0], h[1], h[2], h[3]};
        *reinterpret_cast<uint4 *>(d + 16) = uint4{h[4], h[5], h[6], h[7]};
    }
}

// The same quantizers with 16 values per thread for aligned shapes (k % 16 == 0,
// 16-byte aligned source columns and destination rows): 64-byte loads and one
// 16-byte (e4m3) or 32-byte (FP16) store per thread.
// L panel: a 64 x 64 block through LDS; thread p takes row p % 64 of the block
// and K values 16 (p / 64) .. + 15, so a half-wave reads 32 distinct banks.
template <int FMT, bool PACKED>
__global__ __launch_bounds__(256) void quant_l16_kernel(int64_t m, int64_t k, int tb,
                                                        const float *__restrict__ src, int64_t lds,
                                                        void *__restrict__ dst, int64_t ldd,
                                                        const float *__restrict__ amax, int slots,
                                                        int32_t *__restrict__ exps)
{
    __shared__ float T[64][65];
    constexpr int es = FMT == HPLAI_FMT_E4M3 ? 1 : 2;
    const int64_t r0 = block_number(blockIdx.z) * 64;
    const int64_t c0 = static_cast<int64_t>(blockIdx.y) * 64;
    const int tid = threadIdx.x;
    // loads: 64 columns x 16 float4; thread tid takes float4 i = tid % 16 of
    // columns tid / 16 + 16 u
    {
        const int i = tid & 15;
        const int64_t gr = r0 + 4 * i;
        float4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = (tid >> 4) + 16 * u;
            const int64_t gc = c0 + c < k ? c0 + c : k - 1;
            const float *col = src + gc * lds;
            if (gr + 3 < m) {
                v[u] = *reinterpret_cast<const float4 *>(col + gr);
            } else {
                v[u].x = gr < m ? col[gr] : 0.0f;
                v[u].y = gr + 1 < m ? col[gr + 1] : 0.0f;
                v[u].z = gr + 2 < m ? col[gr + 2] : 0.0f;
                v[u].w = 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = (tid >> 4) + 16 * u;
            T[c][4 * i] = v[u].x;
            T[c][4 * i + 1] = v[u].y;
            T[c][4 * i + 2] = v[u].z;
            T[c][4 * i + 3] = v[u].w;
        }
    }
    __syncthreads();
    const int r = tid & 63, kc = (tid >> 6) * 16;
    const int64_t gr = r0 + r;
    if (gr >= m || c0 + kc >= k) return;
    const int e = fmt_exponent<FMT>(amax, slots, exps, gr / tb);
    if (amax != nullptr && (gr % tb) == 0 && c0 == 0 && kc == 0) exps[gr / tb] = e;
    float v[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = T[kc + q][r];
    uint8_t *d = static_cast<uint8_t *>(dst) +
                 (PACKED ? packed_off(gr, es * (c0 + kc), es * ldd) : (gr * ldd + c0 + kc) * es);
    store_q16<FMT>(d, v, e);
}

// U panel: thread t takes K values 16 (t % (k / 16)) .. + 15 of column t / (k / 16).
template <int FMT, bool PACKED>
__global__ __launch_bounds__(256) void quant_u16_kernel(int64_t m, int64_t k, int tb,
                                                        const float *__restrict__ src, int64_t lds,
                                                        void *__restrict__ dst, int64_t ldd,
                                                        const float *__restrict__ amax, int slots,
                                                        int32_t *__restrict__ exps)
{
    constexpr int es = FMT == HPLAI_FMT_E4M3 ? 1 : 2;
    const int64_t kq = k / 16;
    const int64_t t = block_number(blockIdx.y) * 256 + threadIdx.x;
    const int64_t j = t / kq, r = (t % kq) * 16;
    if (j >= m) return;
    const int e = fmt_exponent<FMT>(amax, slots, exps, j / tb);
    if (amax != nullptr && r == 0 && (j % tb) == 0) exps[j / tb] = e;
    const float4 *s4 = reinterpret_cast<const float4 *>(src + j * lds + r);
    float v[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 x = s4[q];
        v[4 * q] = x.x;
        v[4 * q + 1] = x.y;
        v[4 * q + 2] = x.z;
        v[4 * q + 3] = x.w;
    }
    uint8_t *d = static_cast<uint8_t *>(dst) + (PACKED ? packed_off(j, es * r, es * ldd) : (j * ldd + r) * es);
    store_q16<FMT>(d, v, e);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// Tiles with more entries than kAmaxTile are split over up to 64 workgroups.
// Up to kAmaxSlots parts have a slot each; more meet in amax (zeroed).  Smaller
// tiles of at least kAmaxPart entries are split in kAmaxSlots as well where
// there are no more parts than CUs: 64 tiles of 512 x 512 take 18 us instead of
// 26 from HBM (with the conversion, panels that are in the cache: 16 tiles of
// 512 x 1024 21 for 32, 8 of 512 x 512 12 for 14, 64 of them 31 for 30; 120 of
// them were 49 for 43, hence the line).
// Tiles of fewer than kAmaxShort lines share a workgroup.
constexpr int64_t kAmaxTile = int64_t(1) << 19, kAmaxPart = int64_t(1) << 18;
constexpr int kAmaxShort = 16;

int tile_amax_splits(int64_t m, int64_t k, int tb, int num_cu)
{
    if (tb < kAmaxShort) return 1;
    const int64_t entries = (m < tb ? m : tb) * k, s = ceil_div(entries, kAmaxTile);
    if (s > kAmaxSlots) return static_cast<int>(s < 64 ? s : 64);
    return s > 1 || (entries >= kAmaxPart && ceil_div(m, tb) * kAmaxSlots <= num_cu) ? kAmaxSlots : 1;
}

int tile_amax_slots(int64_t m, int64_t k, int tb, int num_cu)
{
    return tile_amax_splits(m, k, tb, num_cu) == kAmaxSlots ? kAmaxSlots : 1;
}

int launch_tile_amax(int fmt, int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds, float *amax,
                     int32_t *exps, int num_cu, hipStream_t s)
{
    if (m <= 0 || k <= 0) return HPLAI_OK;
    const unsigned parts = amax != nullptr ? static_cast<unsigned>(tile_amax_splits(m, k, tb, num_cu)) : 1u;
    const int slots = tile_amax_slots(m, k, tb, num_cu);
    const bool e4m3 = fmt == HPLAI_FMT_E4M3, together = tb < kAmaxShort && amax == nullptr;
    const int group = together ? 64 / tb * tb : tb;
    // a launch has at most 2^32 threads
    const int64_t most = (int64_t(1) << 21) * group;
    for (int64_t l0 = 0; l0 < m; l0 += most) {
        const int64_t lines = m - l0 < most ? m - l0 : most;
        const float *from = src + (side == 0 ? l0 : l0 * lds);
        int32_t *ex = exps + l0 / tb;
        float *am = amax != nullptr ? amax + l0 / tb * slots : nullptr;
        const dim3 g(static_cast<unsigned>(ceil_div(lines, group)), parts), th(kAmaxThreads);
        if (together && e4m3)
            hipLaunchKernelGGL(tile_amax_short_kernel<HPLAI_FMT_E4M3>, g, th, 0, s, side, lines, k, tb, group, from, lds, ex);
        else if (together)
            hipLaunchKernelGGL(tile_amax_short_kernel<HPLAI_FMT_F16_TILE>, g, th, 0, s, side, lines, k, tb, group, from, lds,
                               ex);
        else if (e4m3)
            hipLaunchKernelGGL(tile_amax_kernel<HPLAI_FMT_E4M3>, g, th, 0, s, side, lines, k, tb, from, lds, am, slots, ex);
        else
            hipLaunchKernelGGL(tile_amax_kernel<HPLAI_FMT_F16_TILE>, g, th, 0, s, side, lines, k, tb, from, lds, am, slots,
                               ex);
        HPLAI_HIP(hipGetLastError());
    }
    return HPLAI_OK;
}

int launch_fill_f32(float *p, int64_t cnt, float v, hipStream_t s)
{
    if (cnt <= 0) return HPLAI_OK;
    hipLaunchKernelGGL(fill_f32_kernel, dim3(static_cast<unsigned>(ceil_div(cnt, 256))), dim3(256), 0,
                       s, p, cnt, v);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

template <int FMT, bool PACKED>
static int quant_dispatch(int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds,
                          void *dst, int64_t ldd, const float *amax, int slots, int32_t *exps, hipStream_t s)
{
    constexpr int es = FMT == HPLAI_FMT_E4M3 ? 1 : 2;
    const bool v16 = k % 16 == 0 && lds % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(dst) % 16 == 0 && (ldd * es) % 16 == 0;
    if (side == 0 && v16) {
        dim3 grid(grid_x(ceil_div(m, 64)), static_cast<unsigned>(ceil_div(k, 64)), grid_rest(ceil_div(m, 64)));
        hipLaunchKernelGGL((quant_l16_kernel<FMT, PACKED>), grid, dim3(256), 0, s, m, k, tb, src, lds, dst, ldd,
                           amax, slots, exps);
    } else if (side == 0) {
        dim3 grid(grid_x(ceil_div(m, 64)), static_cast<unsigned>(ceil_div(k, 64)), grid_rest(ceil_div(m, 64)));
        hipLaunchKernelGGL((quant_l_kernel<FMT, PACKED>), grid, dim3(256), 0, s, m, k, tb, src, lds, dst, ldd,
                           amax, slots, exps);
    } else if (v16) {
        const int64_t thr = m * (k / 16);
        hipLaunchKernelGGL((quant_u16_kernel<FMT, PACKED>), dim3(grid_x(ceil_div(thr, 256)), grid_rest(ceil_div(thr, 256))),
                           dim3(256), 0, s, m, k, tb, src, lds, dst, ldd, amax, slots, exps);
    } else {
        const int64_t thr = m * ceil_div(k, 4);
        hipLaunchKernelGGL((quant_u_kernel<FMT, PACKED>), dim3(grid_x(ceil_div(thr, 256)), grid_rest(ceil_div(thr, 256))),
                           dim3(256), 0, s, m, k, tb, src, lds, dst, ldd, amax, slots, exps);
    }
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

template <int FMT>
static int quant_dispatch(bool packed, int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds,
                          void *dst, int64_t ldd, const float *amax, int slots, int32_t *exps, hipStream_t s)
{
    return packed ? quant_dispatch<FMT, true>(side, m, k, tb, src, lds, dst, ldd, amax, slots, exps, s)
                  : quant_dispatch<FMT, false>(side, m, k, tb, src, lds, dst, ldd, amax, slots, exps, s);
}

int launch_quantize(int fmt, int side, int64_t m, int64_t k, int tb, const float *src, int64_t lds,
                    void *dst, int64_t ldd, const float *amax, int32_t *exps, hipStream_t s, bool packed, int slots)
{
    if (m <= 0 || k <= 0) return HPLAI_OK;
    switch (fmt) {
    case HPLAI_FMT_F16:
        return quant_dispatch<HPLAI_FMT_F16>(packed, side, m, k, tb, src, lds, dst, ldd, amax, slots, exps, s);
    case HPLAI_FMT_F16_TILE:
        return quant_dispatch<HPLAI_FMT_F16_TILE>(packed, side, m, k, tb, src, lds, dst, ldd, amax, slots, exps, s);
    case HPLAI_FMT_E4M3:
        return quant_dispatch<HPLAI_FMT_E4M3>(packed, side, m, k, tb, src, lds, dst, ldd, amax, slots, exps, s);
    default:
        set_error("quantize: unknown format %d", fmt);
        return HPLAI_EINVAL;
    }
}

}  // namespace hplai
