// trsm.hip — panel TRSMs of the blocked LU as products with the inverse of
// the diagonal block's triangle (getrf.hip), b <= 1024:
//   L := A Uinv,  U := Linv A,
// and for a caller's own triangle block by block (trsm_walk_kernel, at the end).
// One workgroup owns a strip of 32 rows (L panel) or 32 columns (U panel)
// with all b entries of its other dimension in LDS.  The strip's 32 x 32
// output blocks are independent, so the eight waves run without barriers
// between them instead of walking a substitution chain.  Products run on
// v_mfma_f32_32x32x2_f32 (FP32 inputs and accumulation); the inverse is read
// from global memory (L2-resident) in MFMA operand order (tri_pos).  b need not
// be a multiple of 32: the strip is padded with zeros and the packed inverse
// with the identity.  What bounds it: the FP32 matrix cores, 14.5 us of the 20
// a strip takes at b = 512 with two workgroups per CU.  (One workgroup per CU
// that walks over its strips and loads ahead, in the same or in two more waves,
// was slower: 512 x 98304 L 253 -> 274 us, U 237 -> 262.)
// MFMA layout: A operand lane -> (row lane % 32, k 2 kk + lane / 32), B
// operand lane -> (k 2 kk + lane / 32, column lane % 32); output acc[4 q + r]
// is row 8 q + 4 (lane / 32) + r, column lane % 32.
#include "device_common.hpp"
#include "internal.hpp"
#include "lu32.hpp"

namespace hplai {

typedef float floatx16t_t __attribute__((ext_vector_type(16)));

constexpr int kStrip = 32;          // strip width: two workgroups per CU at b <= 512
constexpr int kXS = kStrip + 1;     // LDS stride (bank spread)
constexpr int kTrsvMaxB = 512;      // largest diagonal block of tri_trsv_kernel
constexpr int kTriThreads = 512;

// Snake assignment of output blocks to the eight waves, largest first: block
// nb - 1 - p goes to wave snake(p), so every wave gets about the same number
// of 32 x 32 x 32 products (block q costs q + 1 of them; with nb = 16 every
// wave gets 17).
__device__ __forceinline__ int tri_snake(int p) { return ((p >> 3) & 1) ? 7 - (p & 7) : (p & 7); }

// Strip loads into LDS: all of a thread's 16-byte loads are issued at once
// (one memory latency per strip), and the 32 lanes of a half-wave write 32
// distinct banks: each half-wave covers 8 row chunks i (4 rows each) of 4
// columns j, which land on bank (4 i + j + const) mod 32 (kXS = 1 mod 32).
// L strip (32 rows x b columns, column-major, 16-byte aligned, b a multiple
// of 64 up to 512): X[c * kXS + r].
__device__ __forceinline__ void load_strip_l(const float *__restrict__ L, int64_t ldl, int64_t i0, int b, float *X,
                                             int wave, int lane)
{
    const int i = lane & 7, j = lane >> 3;       // row chunk, column of an instruction's 8
    const int per_wave = b / 64;
    float4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (u < per_wave)
            v[u] = *reinterpret_cast<const float4 *>(L + static_cast<int64_t>(8 * (wave * per_wave + u) + j) * ldl + i0 +
                                                     4 * i);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        if (u < per_wave) {
            float *d = X + (8 * (wave * per_wave + u) + j) * kXS + 4 * i;
            d[0] = v[u].x;
            d[1] = v[u].y;
            d[2] = v[u].z;
            d[3] = v[u].w;
        }
    }
}

// any strip (nr <= 32 rows) of any b: rows past nr and columns past b read as zero
__device__ __forceinline__ void load_strip_l_any(const float *__restrict__ L, int64_t ldl, int64_t i0, int nr, int b,
                                                 int nb, float *X, int wave, int lane)
{
    const int r = lane & 31, h = lane >> 5;
    const float *src = L + i0 + min(r, nr - 1);
    for (int base = 0; base < nb * 32; base += 256) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u)
            v[u] = src[static_cast<int64_t>(min(base + 16 * u + 2 * wave + h, b - 1)) * ldl];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = base + 16 * u + 2 * wave + h;
            if (c < nb * 32) X[c * kXS + r] = (r < nr && c < b) ? v[u] : 0.0f;
        }
    }
}

// U strip (b rows x 32 columns, column-major, 16-byte aligned, b a multiple
// of 64 up to 512): X[r * kXS + c]; columns past nc read as zero.  Wave w
// loads columns 4 w .. + 3, 16 row chunks per instruction.
__device__ __forceinline__ void load_strip_u(const float *__restrict__ U, int64_t ldu, int64_t j0, int nc, int b,
                                             float *X, int wave, int lane)
{
    const int i = (lane & 7) + 8 * (lane >> 5), j = (lane >> 3) & 3;
    const int c = 4 * wave + j;
    const float *col = U + (j0 + min(c, nc - 1)) * ldu;
    const int groups = b / 64;
    float4 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u)
        if (u < groups) v[u] = *reinterpret_cast<const float4 *>(col + 64 * u + 4 * i);
    const bool in = c < nc;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        if (u < groups) {
            float *d = X + (64 * u + 4 * i) * kXS + c;
            d[0] = in ? v[u].x : 0.0f;
            d[kXS] = in ? v[u].y : 0.0f;
            d[2 * kXS] = in ? v[u].z : 0.0f;
            d[3 * kXS] = in ? v[u].w : 0.0f;
        }
    }
}

__device__ __forceinline__ void load_strip_u_any(const float *__restrict__ U, int64_t ldu, int64_t j0, int nc, int b,
                                                 int nb, float *X, int wave, int lane)
{
    for (int base = 0; base < nb * 32; base += 256) {
        float v[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[q][u] = U[(j0 + min(4 * wave + q, nc - 1)) * ldu + min(base + 64 * u + lane, b - 1)];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int c = 4 * wave + q, r = base + 64 * u + lane;
                if (r < nb * 32) X[r * kXS + c] = (c < nc && r < b) ? v[q][u] : 0.0f;
            }
    }
}

// One 32 x 32 output block: the sum over k-blocks 0 .. last of the strip's
// rows X and the inverse's blocks at inv + 1024 k (INV_LEFT: the inverse is
// the left operand).
template <bool INV_LEFT>
__device__ __forceinline__ floatx16t_t tri_product(const float *X, const float *__restrict__ inv, int last, int lane)
{
    const int l32 = lane & 31, lh = lane >> 5;
    const float4 *ip = reinterpret_cast<const float4 *>(inv) + lane;
    floatx16t_t acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[e] = 0.0f;
    // the inverse two blocks ahead (L2 latency under a full GPU)
    float4 cur[4], nxt[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) cur[e] = ip[e * 64];
#pragma unroll
    for (int e = 0; e < 4; ++e) nxt[e] = ip[min(1, last) * 256 + e * 64];
    for (int kb = 0; kb <= last; ++kb) {
        float4 nx2[4];
        const float4 *in = ip + min(kb + 2, last) * 256;
#pragma unroll
        for (int e = 0; e < 4; ++e) nx2[e] = in[e * 64];
        float xv[16];
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) xv[kk] = X[(32 * kb + 2 * kk + lh) * kXS + l32];
        // keeps the operand loads where they are: without it the compiler
        // re-issues each global load right before its MFMA and waits on it
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const float iv[16] = {cur[0].x, cur[0].y, cur[0].z, cur[0].w, cur[1].x, cur[1].y, cur[1].z, cur[1].w,
                              cur[2].x, cur[2].y, cur[2].z, cur[2].w, cur[3].x, cur[3].y, cur[3].z, cur[3].w};
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
            acc = INV_LEFT ? __builtin_amdgcn_mfma_f32_32x32x2f32(iv[kk], xv[kk], acc, 0, 0, 0)
                           : __builtin_amdgcn_mfma_f32_32x32x2f32(xv[kk], iv[kk], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            cur[e] = nxt[e];
            nxt[e] = nx2[e];
        }
    }
    return acc;
}

// The same for a strip of 16 rows or columns, on v_mfma_f32_16x16x4_f32: a
// lane's K of step t is 2 (8 (lane / 32) + t) + (lane / 16) % 2, which makes its
// part of a packed block whole quarters.  acc[h]: the
// block's columns (INV_LEFT: rows) 16 h .. + 15; acc[h][r] is row 4 (lane / 16)
// + r, column lane % 16.
typedef float floatx4t_t __attribute__((ext_vector_type(4)));
constexpr int kStrip16 = 16, kXS16 = kStrip16 + 1;

template <bool INV_LEFT>
__device__ __forceinline__ void tri_product16(const float *X, const float *__restrict__ inv, int last, int lane,
                                              floatx4t_t (&acc)[2])
{
    const int l16 = lane & 15, odd = (lane >> 4) & 1, hi = lane >> 5;
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[h] = floatx4t_t{0.0f, 0.0f, 0.0f, 0.0f};
    // packed lane 32 odd + 16 h + l16, quarters 2 hi and 2 hi + 1
    const float4 *ip = reinterpret_cast<const float4 *>(inv) + 128 * hi + 32 * odd + l16;
    float4 cur[4], nxt[4];
    auto fetch = [&](float4 (&v)[4], int kb) {
        const float4 *p = ip + min(kb, last) * 256;
        v[0] = p[0];
        v[1] = p[64];
        v[2] = p[16];
        v[3] = p[80];
    };
    fetch(cur, 0);
    fetch(nxt, 1);
    for (int kb = 0; kb <= last; ++kb) {
        float4 nx2[4];
        fetch(nx2, kb + 2);
        float xv[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) xv[t] = X[(32 * kb + 2 * (8 * hi + t) + odd) * kXS16 + l16];
        asm volatile("" ::: "memory");   // as in tri_product
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](int h, int t, bool on) {
            const float4 &q = cur[2 * h + (t >> 2)];
            const float e = (t & 3) == 0 ? q.x : (t & 3) == 1 ? q.y : (t & 3) == 2 ? q.z : q.w;
            const float iv = on ? e : 0.0f;
            acc[h] = INV_LEFT ? __builtin_amdgcn_mfma_f32_16x16x4f32(iv, xv[t], acc[h], 0, 0, 0)
                              : __builtin_amdgcn_mfma_f32_16x16x4f32(xv[t], iv, acc[h], 0, 0, 0);
        };
        if (kb < last) {
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h) step(h, t, true);
        } else {
            // the triangle's own block: K in ascending order, so that the
            // diagonal's term, the largest, is the last one added (in the order
            // above the result has twice the error: 4.8e-8 against 2.3e-8)
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                step(0, t, true);
                step(1, t, hi == 0);
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) step(1, t, hi == 1);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            cur[e] = nxt[e];
            nxt[e] = nx2[e];
        }
    }
}

// The FP16 copies of a panel's results for the Schur update (the quantizer's
// plain FP16 form, the same bits), straight from the accumulators instead of a
// pass over the panel (7 + 3 of the 47 us of a panel of 1140 x 60): operand
// row i (a row of L, a column of U), K along the bytes.  Columns past b are the
// padding's zeros.
__device__ __forceinline__ uint8_t *half_at(const TrsmHalf &o, int64_t i, int kbyte)
{
    return static_cast<uint8_t *>(o.dst) + (o.packed ? packed_off(i, kbyte, o.ld) : i * o.ld + kbyte);
}
// Four consecutive rows (v) of one column per lane, columns along the lanes:
// neighbouring lanes swap, the even one then holds both columns of rows 0 and 1,
// the odd one of rows 2 and 3.
__device__ __forceinline__ void store_half_rows(const TrsmHalf &o, int64_t i0, int left, int k, int lane, const float (&v)[4])
{
    const bool odd = lane & 1;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const float give = odd ? v[r] : v[r + 2], keep = odd ? v[r + 2] : v[r];
        const float got = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(give), 0xB1, 0xF, 0xF, true));
        const uint32_t w = f32_to_f16_bits(odd ? got : keep) |
                           (static_cast<uint32_t>(f32_to_f16_bits(odd ? keep : got)) << 16);
        const int row = odd ? r + 2 : r;
        if (row < left) *reinterpret_cast<uint32_t *>(half_at(o, i0 + row, 2 * (k & ~1))) = w;
    }
}
// Four consecutive K of one column of U
__device__ __forceinline__ void store_half_ks(const TrsmHalf &o, int64_t j, int k, const float (&v)[4])
{
    uint2 w;
    w.x = f32_to_f16_bits(v[0]) | (static_cast<uint32_t>(f32_to_f16_bits(v[1])) << 16);
    w.y = f32_to_f16_bits(v[2]) | (static_cast<uint32_t>(f32_to_f16_bits(v[3])) << 16);
    *reinterpret_cast<uint2 *>(half_at(o, j, 2 * k)) = w;
}

// L(m x b) := L Ukk^-1 (update_left_panels, panel_trf.hpp:143-157) as
// L := L Uinv: output block jb = sum_{kb <= jb} X(:, kb) Uinv(kb, jb).
// PMAX: the LDS strip's height; VEC: aligned16, b a multiple of 64, b <= 512.
template <int PMAX, bool VEC>
__global__ __launch_bounds__(kTriThreads) void trsm_l_tri_kernel(int64_t m, int b, const float *__restrict__ tri,
                                                                 float *__restrict__ L, int64_t ldl,
                                                                 float *__restrict__ amax, int tb, TrsmHalf half)
{
    __shared__ float X[PMAX * kXS];   // X[c * kXS + r]: column c, row i0 + r
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, lh = lane >> 5;
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kStrip;
    const int nr = m - i0 < kStrip ? static_cast<int>(m - i0) : kStrip;
    const int nb = (b + kStrip - 1) / kStrip;
    if (VEC && nr == kStrip)
        load_strip_l(L, ldl, i0, b, X, wave, lane);
    else
        load_strip_l_any(L, ldl, i0, nr, b, nb, X, wave, lane);
    __syncthreads();
    float vmax = 0.0f;
    for (int p = 0; p < nb; ++p) {
        if (tri_snake(p) != wave) continue;
        const int jb = nb - 1 - p;
        const floatx16t_t acc = tri_product<false>(X, tri_block_u(tri, nb, 0, jb), jb, lane);
        const int c = 32 * jb + l32;
        if (half.dst != nullptr)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float o[4] = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
                store_half_rows(half, i0 + 8 * q + 4 * lh, nr - (8 * q + 4 * lh), c, lane, o);
            }
        float *dst = L + static_cast<int64_t>(c) * ldl + i0 + 4 * lh;
        if (VEC && nr == kStrip) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 o = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
                *reinterpret_cast<float4 *>(dst + 8 * q) = o;
                vmax = fmaxf(vmax, fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fmaxf(fabsf(o.z), fabsf(o.w))));
            }
        } else if (c < b) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (8 * q + 4 * lh + r < nr) {
                        dst[8 * q + r] = acc[4 * q + r];
                        vmax = fmaxf(vmax, fabsf(acc[4 * q + r]));
                    }
        }
    }
    tile_max_reduce(amax, i0 / tb, vmax, true);
}

// U(b x n) := Lkk^-1 U (update_right_panels, panel_trf.hpp:158-171) as
// U := Linv U: output block rb = sum_{kb <= rb} Linv(rb, kb) X(kb, :).
template <int PMAX, bool VEC>
__global__ __launch_bounds__(kTriThreads) void trsm_u_tri_kernel(int b, int64_t n, const float *__restrict__ tri,
                                                                 float *__restrict__ U, int64_t ldu,
                                                                 float *__restrict__ amax, int tb, TrsmHalf half)
{
    __shared__ float X[PMAX * kXS];   // X[r * kXS + c]: row r of column j0 + c
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l32 = lane & 31, lh = lane >> 5;
    const int64_t j0 = static_cast<int64_t>(blockIdx.x) * kStrip;
    const int nc = n - j0 < kStrip ? static_cast<int>(n - j0) : kStrip;
    const int nb = (b + kStrip - 1) / kStrip;
    if (VEC)
        load_strip_u(U, ldu, j0, nc, b, X, wave, lane);
    else
        load_strip_u_any(U, ldu, j0, nc, b, nb, X, wave, lane);
    __syncthreads();
    float vmax = 0.0f;
    for (int p = 0; p < nb; ++p) {
        if (tri_snake(p) != wave) continue;
        const int rb = nb - 1 - p;
        const floatx16t_t acc = tri_product<true>(X, tri_block_l(tri, nb, rb, 0), rb, lane);
        if (l32 >= nc) continue;
        if (half.dst != nullptr)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float o[4] = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
                store_half_ks(half, j0 + l32, 32 * rb + 8 * q + 4 * lh, o);
            }
        float *dst = U + (j0 + l32) * ldu + 32 * rb + 4 * lh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (VEC) {
                const float4 o = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
                *reinterpret_cast<float4 *>(dst + 8 * q) = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (32 * rb + 8 * q + 4 * lh + r < b) dst[8 * q + r] = acc[4 * q + r];
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) vmax = fmaxf(vmax, fabsf(acc[4 * q + r]));
        }
    }
    tile_max_reduce(amax, j0 / tb, vmax, true);
}

// Panels that 32-wide strips leave CUs idle with: 16-wide ones, b <= 512, any
// alignment.  A strip's time is its products on one CU, the same for one strip
// as for a device full, so half the strip is half the time: 512 x 2048, L 27 ->
// 22 us, U 25 -> 19 us (the inverse's 0.5 MB through one CU are the other part).
__global__ __launch_bounds__(kTriThreads) void trsm_l_tri16_kernel(int64_t m, int b, const float *__restrict__ tri,
                                                                   float *__restrict__ L, int64_t ldl,
                                                                   float *__restrict__ amax, int tb, TrsmHalf half)
{
    __shared__ float X[512 * kXS16];   // X[c * kXS16 + r]: column c, row i0 + r
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kStrip16;
    const int nr = m - i0 < kStrip16 ? static_cast<int>(m - i0) : kStrip16;
    const int nb = (b + 31) / 32;
    {
        const int r = tid & 15;
        const float *src = L + i0 + min(r, nr - 1);
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = src[static_cast<int64_t>(min((tid >> 4) + 32 * u, b - 1)) * ldl];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int c = (tid >> 4) + 32 * u;
            if (u < nb) X[c * kXS16 + r] = (r < nr && c < b) ? v[u] : 0.0f;
        }
    }
    __syncthreads();
    float vmax = 0.0f;
    for (int p = 0; p < nb; ++p) {
        if (tri_snake(p) != wave) continue;
        const int jb = nb - 1 - p;
        floatx4t_t acc[2];
        tri_product16<false>(X, tri_block_u(tri, nb, 0, jb), jb, lane, acc);
        const int r0 = 4 * (lane >> 4);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int c = 32 * jb + 16 * h + (lane & 15);
            if (half.dst != nullptr) {
                const float o[4] = {acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
                store_half_rows(half, i0 + r0, nr - r0, c, lane, o);
            }
            if (c >= b) continue;
            float *dst = L + static_cast<int64_t>(c) * ldl + i0 + r0;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r0 + r < nr) {
                    dst[r] = acc[h][r];
                    vmax = fmaxf(vmax, fabsf(acc[h][r]));
                }
        }
    }
    tile_max_reduce(amax, i0 / tb, vmax, true);
}

__global__ __launch_bounds__(kTriThreads) void trsm_u_tri16_kernel(int b, int64_t n, const float *__restrict__ tri,
                                                                   float *__restrict__ U, int64_t ldu,
                                                                   float *__restrict__ amax, int tb, TrsmHalf half)
{
    __shared__ float X[512 * kXS16];   // X[r * kXS16 + c]: row r of column j0 + c
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t j0 = static_cast<int64_t>(blockIdx.x) * kStrip16;
    const int nc = n - j0 < kStrip16 ? static_cast<int>(n - j0) : kStrip16;
    const int nb = (b + 31) / 32;
    {   // wave w: columns 2 w, 2 w + 1, 64 rows an access
        float v[2][8];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int u = 0; u < 8; ++u)
                v[q][u] = U[(j0 + min(2 * wave + q, nc - 1)) * ldu + min(64 * u + lane, b - 1)];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int c = 2 * wave + q, r = 64 * u + lane;
                if (r < nb * 32) X[r * kXS16 + c] = (c < nc && r < b) ? v[q][u] : 0.0f;
            }
    }
    __syncthreads();
    float vmax = 0.0f;
    for (int p = 0; p < nb; ++p) {
        if (tri_snake(p) != wave) continue;
        const int rb = nb - 1 - p;
        floatx4t_t acc[2];
        tri_product16<true>(X, tri_block_l(tri, nb, rb, 0), rb, lane, acc);
        const int c = lane & 15;
        if (c >= nc) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r0 = 32 * rb + 16 * h + 4 * (lane >> 4);
            if (half.dst != nullptr) {
                const float o[4] = {acc[h][0], acc[h][1], acc[h][2], acc[h][3]};
                store_half_ks(half, j0 + c, r0, o);
            }
            float *dst = U + (j0 + c) * ldu + r0;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (r0 + r < b) {
                    dst[r] = acc[h][r];
                    vmax = fmaxf(vmax, fabsf(acc[h][r]));
                }
        }
    }
    tile_max_reduce(amax, j0 / tb, vmax, true);
}

// The caller's own triangle (hplai_trsm_*) where b > 512 or b % 32 != 0: the
// strip is solved 32 rows (U panel) or columns (L panel) at a time through the
// inverses of the 32 x 32 diagonal blocks only, or by substitution where such a
// block is not well conditioned (poor32).  A product with the whole
// inverse has the error of that walk times the triangle's condition: 31 u
// against 2.7 u of |T| |X| for order 777 and condition 1e4, 6e5 u against 3.2 u
// for 4e8.  (b <= 512 in whole 32-blocks takes the whole inverse, and so does
// the LU, whose triangles are its own factors.)
// The strip lives in accumulators, transposed for the L panel, so that a block
// of the result is the right operand of the next products as it is (k =
// acc_row); wave w of W holds blocks w, w + W, ..  An accumulator sums the
// products of a block; its entries (in LDS, [kk 64 + lane]) with the diagonal's
// term, the largest, are added last, in one rounding.  Step K: X_K is in LDS; the wave of
// block K + 1 updates that block, solves it and stores it before its other
// blocks, so a step is two products of the chain or the updates, whichever is
// longer.  A wave's operands of the next step are loaded as soon as the
// registers are free.  What bounds it: those two products a step up to a strip
// per CU, then the FP32 matrix cores at one workgroup per CU (256 registers at b
// > 512).  b = 777, L / U, with the inverses: 4000 wide 127 / 127 us, 40000 wide
// 593 / 587 (with the whole inverse 167 / 143 and 419 / 387, by substitution on
// one row or column per thread 2784 / 11500 and 4267 / 15062); b = 60, 40000 wide
// 23 / 24 (28.6 / 27.9; 50 / 63 with the walk in LDS).  Error for factors of
// HPL-AI matrices, b = 60 .. 1000: 2.4e-8 U, 4.1e-8 L, as with the whole inverse
// (2.8e-8 / 4.4e-8 for 60, 4.5e-7 for 777 by substitution).
template <bool UP, int W, int PER, bool VEC>
__global__ __launch_bounds__(64 * W) void trsm_walk_kernel(int64_t m, int b, const float *__restrict__ tri,
                                                                const float *__restrict__ T, int64_t ldt,
                                                                float *__restrict__ P, int64_t ldp)
{
    __shared__ float xl[2][1024];   // -X_K, [kk 64 + lane]
    __shared__ float own[W * PER][1024], diag[32 * W * PER], poor[W * PER];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5, nb = (b + 31) / 32;
    const int64_t p0 = static_cast<int64_t>(blockIdx.x) * kStrip;
    const int cnt = m - p0 < kStrip ? static_cast<int>(m - p0) : kStrip;
    // row (U panel) or column (L panel) `index` of the strip's lane
    const int64_t step = UP ? 1 : ldp;
    float *strip = P + (UP ? (p0 + min(l32, cnt - 1)) * ldp : p0 + min(l32, cnt - 1));
    // left operand of block J's product with X_K: T(J, K), for the L panel U(K, J)^T
    auto load_left = [&](float (&v)[16], int J, int K) {
        const int64_t j = min(32 * J + l32, b - 1);
        if constexpr (UP) {
            const float *row = T + j + static_cast<int64_t>(32 * K + 4 * lh) * ldt;
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = row[acc_row(e, 0) * ldt];
        } else {
            const float *col = T + j * ldt + 32 * K + 4 * lh;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (VEC) {
                    const float4 x = *reinterpret_cast<const float4 *>(col + 8 * q);
                    v[4 * q] = x.x;
                    v[4 * q + 1] = x.y;
                    v[4 * q + 2] = x.z;
                    v[4 * q + 3] = x.w;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[4 * q + r] = col[8 * q + r];
                }
            }
        }
    };
    // the inverse of diagonal block J: entry (l32, acc_row), for the L panel (acc_row, l32)
    auto inverse = [&](int J) { return UP ? tri_block_l(tri, nb, J, J) : tri_block_u(tri, nb, J, J); };
    // without its diagonal
    float iv[16];
    auto load_inverse = [&](int J) {
        const float *o = inverse(J) + l32 * 4 + 2 * lh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float2 even = *reinterpret_cast<const float2 *>(o + 256 * q);
            const float2 odd = *reinterpret_cast<const float2 *>(o + 256 * q + 128);
            iv[4 * q] = even.x;
            iv[4 * q + 1] = odd.x;
            iv[4 * q + 2] = even.y;
            iv[4 * q + 3] = odd.y;
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) iv[e] = acc_row(e, lh) == l32 ? 0.0f : iv[e];
    };
    floatx16t_t acc[PER];
    float left[PER][16];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int J = wave + W * i;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
        if (J > 0 && J < nb) load_left(left[i], J, 0);
    }
    if (wave < nb) load_inverse(wave);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int J = wave + W * i;
        if (J >= nb) continue;
        float v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = strip[min(32 * J + acc_row(e, lh), b - 1) * step];
#pragma unroll
        for (int e = 0; e < 16; ++e) own[J][e * 64 + lane] = 32 * J + acc_row(e, lh) < b ? v[e] : 0.0f;
    }
    if (tid < nb) poor[tid] = tri_poor(tri, nb)[2 * tid + (UP ? 0 : 1)];
    for (int j = tid; j < 32 * nb; j += 64 * W) {
        const int r = j & 31;
        diag[j] = UP ? 1.0f : inverse(j >> 5)[tri_pos(r + 32 * (r & 1), r >> 1)];
    }
    // X_J := inverse of block J times D, the block less its products (-S)
    auto solve = [&](int J, const floatx16t_t &S) {
        int ln = lane;   // addresses that are not kept through the walk
        asm volatile("" : "+v"(ln));
        const int h = ln >> 5;
        float *out = &xl[J & 1][ln];
        const float *a = &own[J][ln];
        floatx16t_t D, x;
        bool fine = true;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            D[e] = a[64 * e] + S[e];
            x[e] = 0.0f;
            fine = fine && isfinite(D[e]);
        }
        fine = __all(fine && poor[J] == 0.0f);
        if (fine) {
#pragma unroll
            for (int e = 0; e < 16; ++e) x = __builtin_amdgcn_mfma_f32_32x32x2f32(iv[e], D[e], x, 0, 0, 0);
        } else {
            // the zeros of the inverse would carry it to the entries before
#pragma unroll
            for (int e = 0; e < 16; ++e) out[64 * e] = D[e];
            subst32<UP>(xl[J & 1], T + 32 * static_cast<int64_t>(J) * (ldt + 1), ldt, min(32, b - 32 * J), ln);
        }
        float *dst = strip + (32 * J + 4 * h) * step;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float d = diag[32 * J + acc_row(e, h)];
            x[e] = fine ? fmaf(d, a[64 * e], fmaf(d, S[e], x[e])) : out[64 * e];
            out[64 * e] = -x[e];
            if ((ln & 31) < cnt && 32 * J + acc_row(e, h) < b) dst[acc_row(e, 0) * step] = x[e];
        }
        if (J + W < nb) load_inverse(J + W);
    };
    auto update = [&](int i, int J, int K, const float (&xv)[16]) {
        if (32 * J + 32 > b)
#pragma unroll
            for (int e = 0; e < 16; ++e) left[i][e] = 32 * J + l32 < b ? left[i][e] : 0.0f;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(left[i][e], xv[e], acc[i], 0, 0, 0);
        if (J > K + 1) load_left(left[i], J, K + 1);
    };
    for (int K = -1; K + 1 < nb; ++K) {
        __syncthreads();   // X_K is there, X_(K-1) no longer read
        float xv[16];
        if (K >= 0)
#pragma unroll
            for (int e = 0; e < 16; ++e) xv[e] = xl[K & 1][e * 64 + lane];
        __builtin_amdgcn_sched_barrier(0);
        floatx16t_t S;
        bool mine = false;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (wave + W * i == K + 1) {
                if (K >= 0) update(i, K + 1, K, xv);
                S = acc[i];
                mine = true;
            }
        if (mine) solve(K + 1, S);
        if (K < 0) continue;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int J = wave + W * i;
            if (J > K + 1 && J < nb) update(i, J, K, xv);
        }
    }
}

// x_out := Tinv x_in for one factored diagonal block (the IR's diagonal-block
// solve as a product with the stored inverse): Linv (UPPER = false, the unit
// lower solve) or Uinv (UPPER = true).  Workgroup I computes rows
// 32 I .. 32 I + 31; its 256 threads are 32 rows x 8 column-block groups,
// FP32 inverse entries times the FP64 vector summed in FP64, the 8 partial
// sums of a row added in a fixed order.  Out of place: every workgroup reads
// the whole input segment.
template <bool UPPER>
__global__ __launch_bounds__(256) void tri_trsv_kernel(int b, const float *__restrict__ tri,
                                                       const double *__restrict__ xin, double *__restrict__ xout)
{
    __shared__ double xs[kTrsvMaxB];
    __shared__ double part[8][kStrip];
    const int tid = threadIdx.x, rho = tid & 31, p = tid >> 5;
    const int nb = b / kStrip, I = blockIdx.x;
    for (int c = tid; c < b; c += 256) xs[c] = xin[c];
    __syncthreads();
    double acc = 0.0;
    if (!UPPER) {
        for (int J = p; J <= I; J += 8) {
            const float *blk = tri_block_l(tri, nb, I, J);
            const float4 *ev = reinterpret_cast<const float4 *>(blk) + rho;   // gamma = 2 kk
            const float4 *od = ev + 32;                                       // gamma = 2 kk + 1
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float4 a = ev[e * 64], c = od[e * 64];
                const double *xj = xs + 32 * J + 8 * e;
                acc = fma(static_cast<double>(a.x), xj[0], acc);
                acc = fma(static_cast<double>(c.x), xj[1], acc);
                acc = fma(static_cast<double>(a.y), xj[2], acc);
                acc = fma(static_cast<double>(c.y), xj[3], acc);
                acc = fma(static_cast<double>(a.z), xj[4], acc);
                acc = fma(static_cast<double>(c.z), xj[5], acc);
                acc = fma(static_cast<double>(a.w), xj[6], acc);
                acc = fma(static_cast<double>(c.w), xj[7], acc);
            }
        }
    } else {
        for (int J = I + p; J < nb; J += 8) {
            const float *blk = tri_block_u(tri, nb, I, J) + tri_pos(32 * (rho & 1), rho >> 1);
            const double *xj = xs + 32 * J;
#pragma unroll
            for (int g = 0; g < 32; ++g) acc = fma(static_cast<double>(blk[g * 4]), xj[g], acc);
        }
    }
    part[p][rho] = acc;
    __syncthreads();
    if (p == 0) {
        double y = part[0][rho];
#pragma unroll
        for (int q = 1; q < 8; ++q) y += part[q][rho];
        xout[32 * I + rho] = y;
    }
}

bool tri_inverse_ok(int b) { return b % kStrip == 0 && b <= kTrsvMaxB; }

int launch_tri_trsv(bool upper, int b, const float *tri, const double *xin, double *xout, hipStream_t s)
{
    const dim3 grid(static_cast<unsigned>(b / kStrip));
    if (upper)
        hipLaunchKernelGGL(tri_trsv_kernel<true>, grid, dim3(256), 0, s, b, tri, xin, xout);
    else
        hipLaunchKernelGGL(tri_trsv_kernel<false>, grid, dim3(256), 0, s, b, tri, xin, xout);
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

static bool aligned16(const float *p, int64_t ld)
{
    return (ld % 4) == 0 && (reinterpret_cast<uintptr_t>(p) % 16) == 0;
}

// 16-byte strip loads need whole 64-row groups and, for the register batch of
// one memory latency, b <= 512; the 1024-row strip leaves one workgroup per CU.
static int tri_variant(int b, const float *P, int64_t ld)
{
    return b > 512 ? 2 : (b % 64 == 0 && aligned16(P, ld)) ? 0 : 1;
}

// Largest number of 32-wide strips that is split into 16-wide ones instead:
// half the CUs.  Both measured at b = 512, L / U: 4001 wide 36 / 25 against 29 /
// 20 us, 6000 wide 31 / 26 against 37 / 31.
constexpr int64_t kStrips16 = 128;

int launch_trsm_l(int64_t m, int b, const float *tri, float *L, int64_t ldl, float *amax, int tb, hipStream_t s,
                  TrsmHalf half)
{
    if (m <= 0 || b <= 0) return HPLAI_OK;
    HPLAI_CHECK(amax == nullptr || tb % kStrip == 0, "trsm: tile %d not a multiple of %d", tb, kStrip);
    const dim3 g(static_cast<unsigned>(ceil_div(m, kStrip))), th(kTriThreads);
    if (b <= 512 && g.x <= kStrips16) {
        hipLaunchKernelGGL(trsm_l_tri16_kernel, dim3(static_cast<unsigned>(ceil_div(m, kStrip16))), th, 0, s, m, b, tri, L, ldl, amax, tb, half);
        HPLAI_HIP(hipGetLastError());
        return HPLAI_OK;
    }
    switch (tri_variant(b, L, ldl)) {
    case 0: hipLaunchKernelGGL((trsm_l_tri_kernel<512, true>), g, th, 0, s, m, b, tri, L, ldl, amax, tb, half); break;
    case 1: hipLaunchKernelGGL((trsm_l_tri_kernel<512, false>), g, th, 0, s, m, b, tri, L, ldl, amax, tb, half); break;
    default: hipLaunchKernelGGL((trsm_l_tri_kernel<1024, false>), g, th, 0, s, m, b, tri, L, ldl, amax, tb, half); break;
    }
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

int launch_trsm_u(int b, int64_t n, const float *tri, float *U, int64_t ldu, float *amax, int tb, hipStream_t s,
                  TrsmHalf half)
{
    if (n <= 0 || b <= 0) return HPLAI_OK;
    HPLAI_CHECK(amax == nullptr || tb % kStrip == 0, "trsm: tile %d not a multiple of %d", tb, kStrip);
    const dim3 g(static_cast<unsigned>(ceil_div(n, kStrip))), th(kTriThreads);
    if (b <= 512 && g.x <= kStrips16) {
        hipLaunchKernelGGL(trsm_u_tri16_kernel, dim3(static_cast<unsigned>(ceil_div(n, kStrip16))), th, 0, s, b, n, tri, U, ldu, amax, tb, half);
        HPLAI_HIP(hipGetLastError());
        return HPLAI_OK;
    }
    switch (tri_variant(b, U, ldu)) {
    case 0: hipLaunchKernelGGL((trsm_u_tri_kernel<512, true>), g, th, 0, s, b, n, tri, U, ldu, amax, tb, half); break;
    case 1: hipLaunchKernelGGL((trsm_u_tri_kernel<512, false>), g, th, 0, s, b, n, tri, U, ldu, amax, tb, half); break;
    default: hipLaunchKernelGGL((trsm_u_tri_kernel<1024, false>), g, th, 0, s, b, n, tri, U, ldu, amax, tb, half); break;
    }
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

template <bool UP>
static int trsm_walk(int64_t m, int b, const float *tri, const float *T, int64_t ldt, float *P, int64_t ldp,
                     hipStream_t s)
{
    const dim3 g(static_cast<unsigned>(ceil_div(m, kStrip)));
    const int nb = (b + 31) / 32;
    auto launch = [&](auto waves, auto per) {
        constexpr int W = decltype(waves)::value, PER = decltype(per)::value;
        if (!UP && aligned16(T, ldt))   // L's columns are read along the lanes
            hipLaunchKernelGGL((trsm_walk_kernel<UP, W, PER, !UP>), g, dim3(64 * W), 0, s, m, b, tri, T, ldt, P, ldp);
        else
            hipLaunchKernelGGL((trsm_walk_kernel<UP, W, PER, false>), g, dim3(64 * W), 0, s, m, b, tri, T, ldt, P, ldp);
    };
    using std::integral_constant;
    if (nb <= 2)   // more workgroups on a CU
        launch(integral_constant<int, 2>{}, integral_constant<int, 1>{});
    else if (nb <= 4)
        launch(integral_constant<int, 4>{}, integral_constant<int, 1>{});
    else if (nb <= 8)
        launch(integral_constant<int, 8>{}, integral_constant<int, 1>{});
    else if (nb <= 16)
        launch(integral_constant<int, 8>{}, integral_constant<int, 2>{});
    else
        launch(integral_constant<int, 8>{}, integral_constant<int, 4>{});
    HPLAI_HIP(hipGetLastError());
    return HPLAI_OK;
}

constexpr int64_t kTrsmLines = int64_t(1) << 27;

int launch_trsm_panel(bool up, int64_t m, int b, const float *T, int64_t ldt, float *tri, float *P, int64_t ldp,
                      hipStream_t s)
{
    if (m <= 0 || b <= 0) return HPLAI_OK;
    const bool whole = b <= 512 && b % 32 == 0;
    const int rc = launch_tri_inverse(b, T, ldt, tri, up ? 1 : 2, whole, s);
    if (rc) return rc;
    // a launch has at most 2^32 threads: 2^28 lines
    for (int64_t l0 = 0; l0 < m; l0 += kTrsmLines) {
        const int64_t c = m - l0 < kTrsmLines ? m - l0 : kTrsmLines;
        float *Q = P + (up ? l0 * ldp : l0);
        const int r = up ? (whole ? launch_trsm_u(b, c, tri, Q, ldp, nullptr, 1, s) : trsm_walk<true>(c, b, tri, T, ldt, Q, ldp, s))
                         : (whole ? launch_trsm_l(c, b, tri, Q, ldp, nullptr, 1, s) : trsm_walk<false>(c, b, tri, T, ldt, Q, ldp, s));
        if (r) return r;
    }
    return HPLAI_OK;
}

}  // namespace hplai
