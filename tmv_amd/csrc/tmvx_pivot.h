// Pivot search helpers shared by the blocked and the batched LU kernels:
// TMV's underflow threshold and a DPP wave search with TMV's tie rule
// (largest |a|, lowest index on ties: FindMaxAbsElement's strict '>',
// src/TMV_Vector.cpp:473-504).
#pragma once
#include "tmvx_common.h"
#include <cfloat>

namespace tmvx {

template <typename T> __device__ __forceinline__ T tiny();
template <> __device__ __forceinline__ double tiny<double>() { return DBL_MIN; }
template <> __device__ __forceinline__ float tiny<float>() { return FLT_MIN; }

// One DPP step of a maximum (NaN ignored, as fmax does).
template <int CTRL, int RM, typename T>
__device__ __forceinline__ T dpp_max_step(T v)
{
    if constexpr (sizeof(T) == 8) {
        const long long b = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, CTRL, RM, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, RM, 0xf, false);
        return fmax(v, __longlong_as_double(((long long)hi << 32) | (unsigned)lo));
    } else {
        return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v),
                                                                   CTRL, RM, 0xf, false)));
    }
}

// Pivot search on integer keys.  |a| >= 0 orders as its bits do, so the
// search runs on the high 32 bits alone (one v_max_u32 with DPP a stage,
// where a double's maximum takes two moves and two v_max_f64); only lanes
// that tie there compare the low words, then positions (TMV's tie rule).
// Rows out of the search and NaN carry key 0, and a winner below
// mag_tiny() is TMV's underflow (|a| < DBL_MIN / FLT_MIN), for which the
// caller does not use the winner.
__device__ __forceinline__ unsigned mag_hi(double a)
{
    const unsigned h = (unsigned)((unsigned long long)__double_as_longlong(a) >> 32) & 0x7fffffffu;
    return a == a ? h : 0u;
}
__device__ __forceinline__ unsigned mag_hi(float a)
{
    const unsigned h = __float_as_uint(a) & 0x7fffffffu;
    return a == a ? h : 0u;
}
__device__ __forceinline__ unsigned mag_lo(double a) { return (unsigned)__double_as_longlong(a); }
__device__ __forceinline__ unsigned mag_lo(float) { return 0u; }
template <typename T> __device__ __forceinline__ constexpr unsigned mag_tiny()
{ return sizeof(T) == 8 ? 0x00100000u : 0x00800000u; }

template <int CTRL, int RM>
__device__ __forceinline__ unsigned dpp_umax_step(unsigned v)
{
    const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, RM, 0xf, false);
    return v > o ? v : o;
}

template <int NL>
__device__ __forceinline__ unsigned lanes_umax(unsigned v)
{
    static_assert(NL == 64 || NL == 16 || NL == 8 || NL == 4, "lanes 0..NL-1");
    v = dpp_umax_step<0xB1, 0xf>(v);                             // quad_perm [1,0,3,2]
    v = dpp_umax_step<0x4E, 0xf>(v);                             // quad_perm [2,3,0,1]
    if constexpr (NL >= 8) v = dpp_umax_step<0x141, 0xf>(v);     // row_half_mirror
    if constexpr (NL >= 16) v = dpp_umax_step<0x140, 0xf>(v);    // row_mirror
    if constexpr (NL == 64) {
        v = dpp_umax_step<0x142, 0xa>(v);                        // row_bcast:15
        v = dpp_umax_step<0x143, 0xc>(v);                        // row_bcast:31
    }
    return (unsigned)__builtin_amdgcn_readlane((int)v, NL == 64 ? 63 : 0);
}

// The lane (of 0..NL-1) with the largest magnitude, lowest position on
// ties; m receives its high key.  Positions of distinct candidates differ.
template <int NL, typename T>
__device__ __forceinline__ int lanes_best(unsigned hi, unsigned lo, int pos, unsigned& m)
{
    m = lanes_umax<NL>(hi);
    constexpr unsigned long long in = NL == 64 ? ~0ull : (1ull << NL) - 1;
    unsigned long long hit = __builtin_amdgcn_ballot_w64(hi == m) & in;
    if (__builtin_popcountll(hit) > 1 && m >= mag_tiny<T>()) {
        const int lane = threadIdx.x & 63;
        if constexpr (sizeof(T) == 8) {
            const unsigned l = lanes_umax<NL>(((hit >> lane) & 1) ? lo : 0u);
            hit &= __builtin_amdgcn_ballot_w64(lo == l);
        }
        if (__builtin_popcountll(hit) > 1) {
            // lowest position = largest complement
            const unsigned q = lanes_umax<NL>(((hit >> lane) & 1) ? ~(unsigned)pos : 0u);
            hit &= __builtin_amdgcn_ballot_w64(~(unsigned)pos == q);
        }
    }
    return (int)__builtin_ctzll(hit);
}

// Lane C of each row of 16 lanes, in all 16 (DPP row_newbcast): one move
// where a v_readlane of the same value makes the next vector instruction
// wait for its scalar register (~37 cycles each in a chain of them).  Call
// with every lane active.
template <int C>
__device__ __forceinline__ double row_bcast(double v)
{
    static_assert(C >= 0 && C < 16, "lane of a row");
    return __longlong_as_double(__builtin_amdgcn_update_dpp(
        0l, (long)__double_as_longlong(v), 0x150 + C, 0xf, 0xf, true));
}
template <int C>
__device__ __forceinline__ float row_bcast(float v)
{
    static_assert(C >= 0 && C < 16, "lane of a row");
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + C, 0xf, 0xf,
                                                      true));
}

// r[c] += (lane 8 H + c of each row of 16 lanes of u) * l, c < 8: broadcast
// and multiply-add in one instruction (v_fmac with DPP row_newbcast, which the
// compiler does not form by itself; as moves and multiply-adds apart, they
// also get apart, and the moves' results spill).  Call with every lane active.
// The leading s_nop: a DPP operand is not read within two wait states of the
// vector instruction that wrote it.  Early-clobber results: the first is
// written while u and l are still to be read.
#define TMVX_FMAC8(SUF, A, B, C, D, E, F, G, I)                                                 \
    __asm__ volatile("s_nop 1\n\t"                                                              \
                     "v_fmac_" SUF "_dpp %0, %8, %9 row_newbcast:" A " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %1, %8, %9 row_newbcast:" B " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %2, %8, %9 row_newbcast:" C " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %3, %8, %9 row_newbcast:" D " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %4, %8, %9 row_newbcast:" E " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %5, %8, %9 row_newbcast:" F " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %6, %8, %9 row_newbcast:" G " row_mask:0xf bank_mask:0xf\n\t" \
                     "v_fmac_" SUF "_dpp %7, %8, %9 row_newbcast:" I " row_mask:0xf bank_mask:0xf"   \
                     : "+&v"(r[C0]), "+&v"(r[C0 + 1]), "+&v"(r[C0 + 2]), "+&v"(r[C0 + 3]),              \
                       "+&v"(r[C0 + 4]), "+&v"(r[C0 + 5]), "+&v"(r[C0 + 6]), "+&v"(r[C0 + 7])          \
                     : "v"(u), "v"(l))
template <int H, int C0, int N, typename T>
__device__ __forceinline__ void bcast_fma8(T (&r)[N], T u, T l)
{
    static_assert((H == 0 || H == 1) && C0 >= 0 && C0 + 8 <= N, "eight entries");
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(T) == 8) {
        if constexpr (H == 0) TMVX_FMAC8("f64", "0", "1", "2", "3", "4", "5", "6", "7");
        else TMVX_FMAC8("f64", "8", "9", "10", "11", "12", "13", "14", "15");
    } else {
        if constexpr (H == 0) TMVX_FMAC8("f32", "0", "1", "2", "3", "4", "5", "6", "7");
        else TMVX_FMAC8("f32", "8", "9", "10", "11", "12", "13", "14", "15");
    }
#endif
}
#undef TMVX_FMAC8

} // namespace tmvx
