// lu32.hpp — LU of a 32 x 32 FP32 block in LDS and the inverses of its
// triangles, by one wave each.
#pragma once
#include <type_traits>
#include <utility>

#include "device_common.hpp"

namespace hplai {

// acc[4 q + r] of a 32 x 32 MFMA result is row 8 q + 4 (lane / 32) + r, column lane % 32
__device__ __forceinline__ int acc_row(int e, int lh) { return 8 * (e >> 2) + 4 * lh + (e & 3); }

// LDS stores of the wave's lanes before, seen by its other lanes after
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The 32 x 32 steps run in one wave, lane = 16 g + r: r is a row of 16 and g
// splits the columns four ways.  A pivot row then reaches the other rows of
// its 16 lanes as a DPP row broadcast inside the multiply-add; with one row
// per lane and v_readlane the same steps took 2.2 (LU) and 4 times (inverse)
// as long, one scalar broadcast per element.
// (written out: the compiler does not fold the broadcast into v_fmac_f32.  A
// DPP operand must not be one of the last two instructions' results, so each
// sequence waits two slots first and reads nothing that it has written.)
template <int K>
__device__ __forceinline__ float bcast16(float v)   // lane K of every 16
{
    float o;
    asm("s_nop 1\n\tv_mov_b32_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf" : "=v"(o) : "v"(v), "n"(K));
    return o;
}
#define HPLAI_FMAC16(D, B, M) "\n\tv_fmac_f32_dpp " D ", " B ", " M " row_newbcast:%[k] row_mask:0xf bank_mask:0xf"
// p += mp * q and then q += mq * q, with q's lane K of every 16 for the last q
template <int K>
__device__ __forceinline__ void fmac16_2(float &p, float mp, float &q, float mq)
{
    asm("s_nop 1" HPLAI_FMAC16("%0", "%1", "%2") HPLAI_FMAC16("%1", "%1", "%3")
        : "+&v"(p), "+&v"(q)
        : "v"(mp), "v"(mq), [k] "n"(K));
}
template <int K>
__device__ __forceinline__ void fmac16_2x4(float &p0, float &p1, float &p2, float &p3, float mp, float &q0, float &q1,
                                           float &q2, float &q3, float mq)
{
    asm("s_nop 1" HPLAI_FMAC16("%0", "%4", "%8") HPLAI_FMAC16("%1", "%5", "%8") HPLAI_FMAC16("%2", "%6", "%8")
            HPLAI_FMAC16("%3", "%7", "%8") HPLAI_FMAC16("%4", "%4", "%9") HPLAI_FMAC16("%5", "%5", "%9")
                HPLAI_FMAC16("%6", "%6", "%9") HPLAI_FMAC16("%7", "%7", "%9")
        : "+&v"(p0), "+&v"(p1), "+&v"(p2), "+&v"(p3), "+&v"(q0), "+&v"(q1), "+&v"(q2), "+&v"(q3)
        : "v"(mp), "v"(mq), [k] "n"(K));
}
// q += m * q's lane K of every 16
template <int K>
__device__ __forceinline__ void fmac16_1(float &q, float m)
{
    asm("s_nop 1" HPLAI_FMAC16("%0", "%0", "%1") : "+&v"(q) : "v"(m), [k] "n"(K));
}
template <int K>
__device__ __forceinline__ void fmac16_1x4(float &q0, float &q1, float &q2, float &q3, float m)
{
    asm("s_nop 1" HPLAI_FMAC16("%0", "%0", "%4") HPLAI_FMAC16("%1", "%1", "%4") HPLAI_FMAC16("%2", "%2", "%4")
            HPLAI_FMAC16("%3", "%3", "%4")
        : "+&v"(q0), "+&v"(q1), "+&v"(q2), "+&v"(q3)
        : "v"(m), [k] "n"(K));
}
// columns J .. N - 1 of p and q (fmac16_2) or of q alone
template <int K, int J, int N>
__device__ __forceinline__ void fmac16_cols(float *p, float mp, float *q, float mq)
{
    if constexpr (J + 4 <= N) {
        fmac16_2x4<K>(p[J], p[J + 1], p[J + 2], p[J + 3], mp, q[J], q[J + 1], q[J + 2], q[J + 3], mq);
        fmac16_cols<K, J + 4, N>(p, mp, q, mq);
    } else if constexpr (J < N) {
        fmac16_2<K>(p[J], mp, q[J], mq);
        fmac16_cols<K, J + 1, N>(p, mp, q, mq);
    }
}
template <int K, int J, int N>
__device__ __forceinline__ void fmac16_cols(float *q, float m)
{
    if constexpr (J + 4 <= N) {
        fmac16_1x4<K>(q[J], q[J + 1], q[J + 2], q[J + 3], m);
        fmac16_cols<K, J + 4, N>(q, m);
    } else if constexpr (J < N) {
        fmac16_1<K>(q[J], m);
        fmac16_cols<K, J + 1, N>(q, m);
    }
}

template <int... I, typename F>
__device__ __forceinline__ void unrolled(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled(F &&f)
{
    unrolled(std::make_integer_sequence<int, N>{}, f);
}

// Reciprocal of a pivot: v_rcp_f32 and one Newton step (half the instructions
// of the IEEE division) for magnitudes where that cannot over- or underflow;
// EXACT divides.
template <bool EXACT>
__device__ __forceinline__ float pivot_rcp(float p)
{
    if (EXACT) return 1.0f / p;
    const float r = __builtin_amdgcn_rcpf(p);
    return fmaf(fmaf(-p, r, 1.0f), r, r);
}

// LU of the 32 x 32 block at B (columns ld apart) in place.  Every group of 16 lanes
// holds all 16 columns of the current panel (Pt: rows 0..15, Pb: rows 16..31)
// and a quarter of the columns right of it.  Returns the pivot of lane
// (row) lane % 32; without EXACT the block is not written when a pivot's
// magnitude is outside [2^-100, 2^100].
// ld: an int or a std::integral_constant.
template <bool EXACT, typename Ld>
__device__ __forceinline__ float lu32_run(float *B, Ld ld, int lane)
{
    const int r = lane & 15, g = lane >> 4;
    float Pt[16], Pb[16], Rt[4], Rb[4];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        Pt[c] = B[c * ld + r];
        Pb[c] = B[c * ld + 16 + r];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        Rt[u] = B[(16 + 4 * u + g) * ld + r];
        Rb[u] = B[(16 + 4 * u + g) * ld + 16 + r];
    }
    unrolled<16>([&](auto kc) {
        constexpr int k = kc;
        const float inv = pivot_rcp<EXACT>(bcast16<k>(Pt[k]));
        const float lt = r > k ? Pt[k] * inv : 0.0f, lb = Pb[k] * inv;
        Pt[k] = r > k ? lt : Pt[k];
        Pb[k] = lb;
        fmac16_cols<k, k + 1, 16>(Pb, -lb, Pt, -lt);
        fmac16_cols<k, 0, 4>(Rb, -lb, Rt, -lt);
    });
    // the second panel, rows 16..31 of columns 16..31, to every group
    float Q[16];
#pragma unroll
    for (int c = 0; c < 16; ++c)
        Q[c] = __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (16 * (c & 3) + r), __float_as_int(Rb[c >> 2])));
    unrolled<16>([&](auto kc) {
        constexpr int k = kc;
        const float inv = pivot_rcp<EXACT>(bcast16<k>(Q[k]));
        const float l = r > k ? Q[k] * inv : 0.0f;
        Q[k] = r > k ? l : Q[k];
        fmac16_cols<k, k + 1, 16>(Q, -l);
    });
    // pivot of row lane % 32 (groups 0, 2: the first panel's, 1, 3: the second's)
    float piv = 1.0f;
#pragma unroll
    for (int c = 0; c < 16; ++c) piv = r == c ? ((g & 1) ? Q[c] : Pt[c]) : piv;
    if (!EXACT) {
        const float m = fabsf(piv);
        if (__any(!(m >= 0x1p-100f && m <= 0x1p100f))) return piv;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) B[(16 + 4 * u + g) * ld + r] = Rt[u];
#pragma unroll
    for (int c = 0; c < 16; ++c)
        if (g == c >> 2) {
            B[c * ld + r] = Pt[c];
            B[c * ld + 16 + r] = Pb[c];
            B[(16 + c) * ld + 16 + r] = Q[c];
        }
    return piv;
}

// returns 1 + the first zero or non-finite pivot, or 0
template <typename Ld>
__device__ __forceinline__ int lu32(float *B, Ld ld, int lane)
{
    float piv = lu32_run<false>(B, ld, lane);
    const float m = fabsf(piv);
    if (__any(!(m >= 0x1p-100f && m <= 0x1p100f))) piv = lu32_run<true>(B, ld, lane);
    const uint32_t z = static_cast<uint32_t>(__ballot(!(piv != 0.0f && isfinite(piv))));
    return __ffs(z);
}

// Inverse of the unit-lower (UP = false) or upper triangle of the 32 x 32
// block at (c0, c0) of S by Gauss-Jordan, one wave: the triangle's rows are in
// every group, the inverse's columns 4 u + g in group g.  U = D V with V unit
// upper, so Uinv = Vinv D^-1.  To M (row-major, stride 33, when given) and V.
template <bool UP, typename Ld>
__device__ __forceinline__ void invert32(const float *B, Ld ld, float *V, int lane, float *M)
{
    const int r = lane & 15, g = lane >> 4;
    float Tt[32], Tb[32];   // rows r and 16 + r of the triangle, negated
#pragma unroll
    for (int c = 0; c < 32; ++c) {
        if (UP || c < 16) Tt[c] = -B[c * ld + r];
        if (!UP || c >= 16) Tb[c] = -B[c * ld + 16 + r];
    }
    float Xt[8], Xb[8];     // columns 4 u + g
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        Xt[u] = 4 * u + g == r ? 1.0f : 0.0f;
        Xb[u] = 4 * u + g == 16 + r ? 1.0f : 0.0f;
    }
    if constexpr (!UP) {
        unrolled<16>([&](auto cc) {
            constexpr int c = cc;
            fmac16_cols<c, 0, c / 4 + 1>(Xb, Tb[c], Xt, r > c ? Tt[c] : 0.0f);
        });
        unrolled<16>([&](auto cc) {
            constexpr int c = cc;
            fmac16_cols<c, 0, 4 + c / 4 + 1>(Xb, r > c ? Tb[16 + c] : 0.0f);
        });
    } else {
        float dt = -1.0f, db = -1.0f;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            dt = r == c ? Tt[c] : dt;
            db = r == c ? Tb[16 + c] : db;
        }
        dt = -1.0f / dt;
        db = -1.0f / db;
        unrolled<16>([&](auto cc) {
            constexpr int c = 15 - cc;
            fmac16_cols<c, 4 + c / 4, 8>(Xt, Tt[16 + c] * dt, Xb, r < c ? Tb[16 + c] * db : 0.0f);
        });
        unrolled<16>([&](auto cc) {
            constexpr int c = 15 - cc;
            fmac16_cols<c, c / 4, 8>(Xt, r < c ? Tt[c] * dt : 0.0f);
        });
        // column j times 1 / d_j
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int src = 4 * ((4 * u + g) & 15);
            const float d = __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(u < 4 ? dt : db)));
            Xt[u] *= d;
            Xb[u] *= d;
        }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int j = 4 * u + g;
        if (M != nullptr) {
            M[r * 33 + j] = Xt[u];
            M[(16 + r) * 33 + j] = Xb[u];
        }
        if (V != nullptr && (UP ? r <= j : r > j)) V[j * ld + r] = Xt[u];
        if (V != nullptr && (UP ? 16 + r <= j : 16 + r > j)) V[j * ld + 16 + r] = Xb[u];
    }
}

// Whether a triangle is not well conditioned: a row sum of |X| |T| past kCond32,
// or no number, X its inverse.  A product with X then costs accuracy that
// substitution (subst32) does not.  In two parts, one wave each: the row sums of
// |T| (block at B, columns ld apart) to w, and the rest with X(r, c) from entry.
constexpr float kCond32 = 16.0f;

template <bool UP, typename Ld>
__device__ __forceinline__ void row_sums32(const float *B, Ld ld, float *w, int lane)
{
    const int r = lane & 31;
    float s = UP ? 0.0f : 1.0f;
#pragma unroll
    for (int c = 0; c < 32; ++c) {
        const float v = fabsf(B[c * ld + r]);
        s += (UP ? c >= r : c < r) ? v : 0.0f;
    }
    if (lane < 32) w[r] = s;
}
template <typename F>
__device__ __forceinline__ bool poor32(F &&entry, const float *w, int lane)
{
    const int r = lane & 31, h = 16 * (lane >> 5);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) s = fmaf(fabsf(entry(r, h + j)), w[h + j], s);
    s += __shfl_xor(s, 32);
    return __any(!(s <= kCond32));
}

// x := L^-1 x (UP) or U^-T x for the w x w triangle at T (columns ldt apart) by
// substitution, one wave, one column per lane below 32: x in LDS, entry k of
// column c at (index of k's accumulator) 64 + 32 (k / 4 % 2) + c (acc_row).
template <bool UP>
__device__ __forceinline__ void subst32(float *xb, const float *T, int64_t ldt, int w, int lane)
{
    wave_lds_sync();
    if (lane < 32) {
        auto at = [&](int k) -> float & { return xb[((k >> 3) * 4 + (k & 3)) * 64 + ((k >> 2) & 1) * 32 + lane]; };
#pragma clang loop unroll(disable)
        for (int k = 0; k < w; ++k) {
            float x = at(k);
            if (!UP) {
                x *= 1.0f / T[k * ldt + k];
                at(k) = x;
            }
#pragma clang loop unroll_count(4)
            for (int j = k + 1; j < w; ++j) at(j) = fmaf(-x, UP ? T[k * ldt + j] : T[j * ldt + k], at(j));
        }
    }
    wave_lds_sync();
}

}  // namespace hplai
