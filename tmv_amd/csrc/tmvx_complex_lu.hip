// Complex LU with partial pivoting and the solves with its factors
// (interleaved std::complex storage).
//
// TMV's LU_Decompose and LU_LDivEq / LU_RDivEq for complex T
// (src/TMV_LUDecompose.cpp:217-407, src/TMV_LUDiv.cpp:185-226, 369-410): the
// pivot is the candidate of largest modulus (TMV_ABS), first index on ties
// (FindMaxAbsElement, src/TMV_Vector.cpp:473-504); a column whose largest
// candidate underflows is zeroed from the diagonal down and interchanged with
// itself (src/TMV_LUDecompose.cpp:162-169); the column below the pivot is
// scaled by the pivot's reciprocal.
//
// While more than ZN_MMAX rows are left: 64-column panels, each by ONE
// workgroup column by column in global memory, U12 by one thread per column,
// A22 -= L21 U12 on the complex GEMM.
// From there on (the whole of a system up to that order): panels of 16 (8)
// columns, two launches each:
//   znpanel_kernel: one workgroup, its rows in registers (one to four a
//     thread).  Rows never move: each carries its position.  Per column one
//     barrier: every wave's best row (largest modulus, found on integer keys)
//     goes to LDS with the reciprocal of its pivot, every wave picks the
//     winner and updates its rows, the pivot row's entries handed on by DPP
//     broadcasts;
//   znupdate_kernel: 8 columns per workgroup: U12 with a row per lane, then the
//     rank-16 update with a row of L21 per lane; the interchanges are the rows
//     that the update reads from.
// The interchanges of the columns to the left are applied once, at the end.
// Solves up to ZS_NMAX: one workgroup per right-hand side, the vector in LDS,
// 16 rows at a time (substitution on 16 lanes, then the rows to come with the
// next 16 columns already loaded); above: column sweeps by one workgroup.
// Bound: the panel's chain (1.4-1.9 us a column, most of it hypot, the pivot's
// reciprocal and one barrier) and two launches per 16 columns.  Measured at
// n = 1000, 4 right-hand sides, FP64: 22.1 -> 3.3 ms (panels 12.0 -> 1.7, U12
// and update 5.8 -> 0.8, solves 2.9 -> 0.6, left interchanges 0.1).
#include "tmvx_lu.h"
#include "tmvx_pivot.h"

#include <algorithm>
#include <cfloat>

namespace tmvx {

template <typename R> struct CplxT;
template <> struct CplxT<double> { typedef double2 type; static constexpr double rmin = DBL_MIN; };
template <> struct CplxT<float> { typedef float2 type; static constexpr float rmin = FLT_MIN; };

__global__ void set_i64_kernel(i64* p, i64 v) { *p = v; }
__global__ void set_int_kernel(int* p, int v) { *p = v; }

template <typename Z> __device__ __forceinline__ Z cmul(Z a, Z b)
{
    Z r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
template <typename Z> __device__ __forceinline__ Z csub(Z a, Z b)
{
    Z r;
    r.x = a.x - b.x;
    r.y = a.y - b.y;
    return r;
}
// a / b by Smith's method (scaled: no overflow for large |b|).
template <typename Z> __device__ __forceinline__ Z cdiv(Z a, Z b)
{
    Z r;
    if (fabs(b.x) >= fabs(b.y)) {
        const auto t = b.y / b.x, d = b.x + b.y * t;
        r.x = (a.x + a.y * t) / d;
        r.y = (a.y - a.x * t) / d;
    } else {
        const auto t = b.x / b.y, d = b.x * t + b.y;
        r.x = (a.x * t + a.y) / d;
        r.y = (a.y * t - a.x) / d;
    }
    return r;
}

constexpr int ZP_NB = 64;        // panel width
constexpr int ZP_NTH = 1024;     // panel workgroup

// Factor panel columns [j0, j1) of the n x n matrix; rows swapped over all n
// columns.  One workgroup.
template <typename R>
__global__ void __launch_bounds__(ZP_NTH)
zpanel_kernel(i64 n, typename CplxT<R>::type* __restrict__ A, i64 lda, i64 j0, i64 j1,
              i64* __restrict__ piv, i64* __restrict__ first_zero)
{
    typedef typename CplxT<R>::type Z;
    constexpr int NW = ZP_NTH / 64;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    __shared__ R s_v[NW];
    __shared__ i64 s_i[NW];
    __shared__ i64 s_p;
    __shared__ int s_zero;
    __shared__ Z s_prow[ZP_NB];
    __shared__ Z s_inv;
    for (i64 j = j0; j < j1; ++j) {
        // pivot search: largest modulus, lowest row on ties
        R bv = R(-1);
        i64 bi = n;
        for (i64 i = j + t; i < n; i += ZP_NTH) {
            const Z a = A[i + j * lda];
            const R v = hypot(a.x, a.y);
            if (v > bv) { bv = v; bi = i; }
        }
        for (int off = 32; off > 0; off >>= 1) {
            const R v2 = __shfl_xor(bv, off);
            const i64 i2 = __shfl_xor(bi, off);
            if (v2 > bv || (v2 == bv && i2 < bi)) { bv = v2; bi = i2; }
        }
        if (lane == 0) { s_v[wave] = bv; s_i[wave] = bi; }
        __syncthreads();
        if (t == 0) {
            R v = s_v[0];
            i64 ii = s_i[0];
            for (int q = 1; q < NW; ++q)
                if (s_v[q] > v || (s_v[q] == v && s_i[q] < ii)) { v = s_v[q]; ii = s_i[q]; }
            const bool zero = !(v >= CplxT<R>::rmin);
            s_zero = zero ? 1 : 0;
            s_p = zero ? j : ii;
            piv[j] = zero ? j : ii;
            if (zero)
                atomicMin(reinterpret_cast<unsigned long long*>(first_zero),
                          (unsigned long long)(j + 1));
        }
        __syncthreads();
        const i64 p = s_p;
        if (s_zero) {
            Z z0;
            z0.x = R(0);
            z0.y = R(0);
            for (i64 i = j + t; i < n; i += ZP_NTH) A[i + j * lda] = z0;
            __syncthreads();
            continue;
        }
        if (p != j)
            for (i64 c = t; c < n; c += ZP_NTH) {
                const Z x = A[j + c * lda];
                A[j + c * lda] = A[p + c * lda];
                A[p + c * lda] = x;
            }
        __syncthreads();
        if (t < ZP_NB && j + 1 + t < j1) s_prow[t] = A[j + (j + 1 + t) * lda];
        if (t == 0) {
            Z one;
            one.x = R(1);
            one.y = R(0);
            s_inv = cdiv(one, A[j + j * lda]);
        }
        __syncthreads();
        const Z inv = s_inv;
        const int nc = (int)(j1 - j - 1);
        for (i64 i = j + 1 + t; i < n; i += ZP_NTH) {
            const Z l = cmul(A[i + j * lda], inv);
            A[i + j * lda] = l;
            for (int c = 0; c < nc; ++c)
                A[i + (j + 1 + c) * lda] = csub(A[i + (j + 1 + c) * lda], cmul(l, s_prow[c]));
        }
        __syncthreads();
    }
}

// U12 := L11^-1 A12 for the panel rows [j0, j0 + jb) and columns [c0, n).
template <typename R>
__global__ void ztrsm_u12_kernel(i64 n, typename CplxT<R>::type* __restrict__ A, i64 lda, i64 j0,
                                 int jb, i64 c0)
{
    typedef typename CplxT<R>::type Z;
    const i64 c = c0 + (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    Z* col = A + c * lda + j0;
    const Z* L = A + j0 + j0 * lda;
    for (int r = 1; r < jb; ++r) {
        Z acc = col[r];
        for (int q = 0; q < r; ++q) acc = csub(acc, cmul(L[r + (i64)q * lda], col[q]));
        col[r] = acc;
    }
}

// ---- panels in registers -------------------------------------------------

constexpr int ZN_NTH = 512;              // panel workgroup
constexpr int ZN_NW = ZN_NTH / 64;
constexpr i64 ZN_MMAX = 4 * ZN_NTH;      // rows a panel can hold (four a thread)

// s += l u
template <typename Z> __device__ __forceinline__ void caddmul(Z& s, Z l, Z u)
{
    s.x = fma(l.x, u.x, fma(-l.y, u.y, s.x));
    s.y = fma(l.x, u.y, fma(l.y, u.x, s.y));
}
// x -= l u: the product first, or x would take two roundings at its size
template <typename Z> __device__ __forceinline__ void csubmul(Z& x, Z l, Z u)
{ x = csub(x, cmul(l, u)); }
template <int C, typename Z> __device__ __forceinline__ Z row_bcast_z(Z v)
{
    Z r;
    r.x = row_bcast<C>(v.x);
    r.y = row_bcast<C>(v.y);
    return r;
}

// (xr, xi) -= sum over k in [K0, K0 + 4) of l[k] (lane k of each row of 16 lanes of u),
// given -u.x, -u.y and u.y: broadcast and multiply-add in one instruction
// (cf. bcast_fma8).  Call with every lane active.
#define ZN_STEP(SUF, K, LX, LY)                                                              \
    "v_fmac_" SUF "_dpp %0, %2, " LX " row_newbcast:" K " row_mask:0xf bank_mask:0xf\n\t"      \
    "v_fmac_" SUF "_dpp %1, %3, " LX " row_newbcast:" K " row_mask:0xf bank_mask:0xf\n\t"      \
    "v_fmac_" SUF "_dpp %0, %4, " LY " row_newbcast:" K " row_mask:0xf bank_mask:0xf\n\t"      \
    "v_fmac_" SUF "_dpp %1, %2, " LY " row_newbcast:" K " row_mask:0xf bank_mask:0xf\n\t"
#define ZN_FMAC4(SUF, A, B, C, D)                                                            \
    __asm__ volatile("s_nop 1\n\t" ZN_STEP(SUF, A, "%5", "%9") ZN_STEP(SUF, B, "%6", "%10")   \
                         ZN_STEP(SUF, C, "%7", "%11") ZN_STEP(SUF, D, "%8", "%12")           \
                     : "+&v"(xr), "+&v"(xi)                                                    \
                     : "v"(nux), "v"(nuy), "v"(uy), "v"(l[K0].x), "v"(l[K0 + 1].x),          \
                       "v"(l[K0 + 2].x), "v"(l[K0 + 3].x), "v"(l[K0].y), "v"(l[K0 + 1].y),   \
                       "v"(l[K0 + 2].y), "v"(l[K0 + 3].y))
template <int K0, typename R, typename Z, int N>
__device__ __forceinline__ void zbcast_fma4(R& xr, R& xi, R nux, R nuy, R uy, const Z (&l)[N])
{
    static_assert(K0 % 4 == 0 && K0 < 16 && K0 + 4 <= N, "four of sixteen lanes");
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (sizeof(R) == 8) {
        if constexpr (K0 == 0) ZN_FMAC4("f64", "0", "1", "2", "3");
        else if constexpr (K0 == 4) ZN_FMAC4("f64", "4", "5", "6", "7");
        else if constexpr (K0 == 8) ZN_FMAC4("f64", "8", "9", "10", "11");
        else ZN_FMAC4("f64", "12", "13", "14", "15");
    } else {
        if constexpr (K0 == 0) ZN_FMAC4("f32", "0", "1", "2", "3");
        else if constexpr (K0 == 4) ZN_FMAC4("f32", "4", "5", "6", "7");
        else if constexpr (K0 == 8) ZN_FMAC4("f32", "8", "9", "10", "11");
        else ZN_FMAC4("f32", "12", "13", "14", "15");
    }
#endif
}
#undef ZN_FMAC4
#undef ZN_STEP

// Columns [j0, j0 + jb) of the m = n - j0 rows from j0 on, m <= RPT ZN_NTH:
// row t + q ZN_NTH of the panel in thread t's slot q.  from[r]: the panel-
// relative row that ends at position r.
template <typename R, int RPT, int NB>
__global__ void __launch_bounds__(ZN_NTH)
znpanel_kernel(i64 n, typename CplxT<R>::type* __restrict__ Ag, i64 lda, i64 j0, int jb,
               i64* __restrict__ piv, i64* __restrict__ first_zero, int* __restrict__ from)
{
    typedef typename CplxT<R>::type Z;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int m = (int)(n - j0);
    Z* __restrict__ A = Ag + j0 + j0 * lda;
    __shared__ __attribute__((aligned(16))) Z s_row[2][ZN_NW][16];
    __shared__ unsigned s_hi[2][ZN_NW], s_lo[2][ZN_NW];
    __shared__ int s_pos[2][ZN_NW];
    Z row[RPT][NB];
    int pos[RPT];
    bool used[RPT];
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * ZN_NTH;
        pos[q] = r;
        used[q] = r >= m;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            Z z;
            z.x = z.y = R(0);
            if (r < m && c < jb) z = A[r + c * lda];
            row[q][c] = z;
        }
    });
    // (columns past jb run as zero columns, with nothing recorded)
    static_for<0, NB>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, par = k & 1;
        // the thread's best row: largest modulus, lowest position
        unsigned hi = 0u, lo = 0u;
        int bp = INT_MAX, bq = 0;
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            const R v = R(hypot(row[q][k].x, row[q][k].y));
            const unsigned h = mag_hi(v), l = mag_lo(v);
            if (!used[q] && (bp == INT_MAX || h > hi || (h == hi && (l > lo || (l == lo && pos[q] < bp))))) {
                hi = h; lo = l; bp = pos[q]; bq = q;
            }
        });
        unsigned gm;
        const int wl = lanes_best<64, R>(hi, lo, bp, gm);
        if (lane == wl) {
            s_hi[par][wave] = hi;
            s_lo[par][wave] = lo;
            s_pos[par][wave] = bp;
        }
        const int bu = __builtin_amdgcn_readlane(bq, wl);
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            if (bu == q) {                             // uniform
                Z one;
                one.x = R(1);
                one.y = R(0);
                const Z inv = cdiv(one, row[q][k]);    // in place of the pivot
                if (lane == wl) {
                    s_row[par][wave][k] = inv;
                    static_for<k + 1, NB>([&](auto cc) __attribute__((always_inline)) {
                        constexpr int c = decltype(cc)::value;
                        s_row[par][wave][c] = row[q][c];
                    });
                }
                __asm__ volatile("" ::: "memory");     // (keeps the slots' code apart: merged,
                                                       // it would index the rows in memory)
            }
        });
        __syncthreads();
        const int cp = s_pos[par][lane & (ZN_NW - 1)];
        const int ww = lanes_best<8, R>(s_hi[par][lane & (ZN_NW - 1)], s_lo[par][lane & (ZN_NW - 1)],
                                        cp, gm);
        const bool zero = gm < mag_tiny<R>();                         // TMV_Underflow
        const int p = zero ? k : __builtin_amdgcn_readlane(cp, ww);
        const Z uv = s_row[par][ww][lane & 15];        // lane li: entry li of the pivot row
        if (t == 0 && k < jb) {
            piv[j0 + k] = j0 + p;
            if (zero)
                atomicMin(reinterpret_cast<unsigned long long*>(first_zero),
                          (unsigned long long)(j0 + k + 1));
        }
        Z u[NB];
        static_for<k, NB>([&](auto cc) __attribute__((always_inline)) {
            u[decltype(cc)::value] = row_bcast_z<decltype(cc)::value>(uv);
        });
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            if (zero && !used[q]) row[q][k].x = row[q][k].y = R(0);
            const bool isp = !used[q] && pos[q] == p;
            if (!used[q] && pos[q] == k) pos[q] = p;
            if (isp) pos[q] = k;
            used[q] = used[q] || isp;
            if (!used[q] && !zero) {
                const Z l = cmul(row[q][k], u[k]);
                row[q][k] = l;
                static_for<k + 1, NB>([&](auto cc) __attribute__((always_inline)) {
                    constexpr int c = decltype(cc)::value;
                    csubmul(row[q][c], l, u[c]);
                });
            }
        });
    });
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * ZN_NTH;
        if (r >= m) return;
        from[pos[q]] = r;
#pragma unroll
        for (int c = 0; c < NB; ++c)
            if (c < jb) A[pos[q] + c * lda] = row[q][c];
    });
}

constexpr int ZU_CW = 8;                 // columns per workgroup of the update

// The columns right of a panel of NB columns at j0: interchanges, U12 =
// L11^-1 A12 and A22 -= L21 U12.
template <typename R, int NB>
__global__ void __launch_bounds__(256)
znupdate_kernel(i64 n, typename CplxT<R>::type* __restrict__ Ag, i64 lda, i64 j0,
                const int* __restrict__ from)
{
    typedef typename CplxT<R>::type Z;
    __shared__ __attribute__((aligned(16))) Z s_u[ZU_CW][16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, li = lane & 15, g = lane >> 4;
    const int m = (int)(n - j0);
    const i64 c0 = j0 + NB + (i64)blockIdx.x * ZU_CW;
    const int nc = n - c0 < ZU_CW ? (int)(n - c0) : ZU_CW;
    Z* __restrict__ A = Ag + j0;
    const Z* __restrict__ L = A + j0 * lda;
    if (wave < 2) {
        // column 4 wave + g, row li
        const int c = 4 * wave + g;
        const bool in = c < nc && li < NB;
        Z x, sum, l[NB];                     // (products summed apart from x)
        x.x = x.y = sum.x = sum.y = R(0);
        if (in) x = A[from[li] + (c0 + c) * lda];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            l[k].x = l[k].y = R(0);
            if (li > k && li < NB) l[k] = L[li + k * lda];
        }
        static_for<0, NB>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const Z xk = row_bcast_z<k>(csub(x, sum));
            if (li > k) caddmul(sum, l[k], xk);
        });
        s_u[c][li] = csub(x, sum);
    }
    __syncthreads();
    for (int r0 = NB + 64 * wave; r0 < m; r0 += 256) {
        const int r = r0 + lane, rc = r < m ? r : m - 1, fr = from[rc];
        Z l[NB], x[ZU_CW];
#pragma unroll
        for (int k = 0; k < NB; ++k) l[k] = L[rc + k * lda];
#pragma unroll
        for (int c = 0; c < ZU_CW; ++c) x[c] = A[fr + (c0 + (c < nc ? c : nc - 1)) * lda];
#pragma unroll
        for (int c = 0; c < ZU_CW; ++c) {
            const Z uv = s_u[c][li];
            const R nux = -uv.x, nuy = -uv.y;
            R sr = R(0), si = R(0);          // minus the products, summed apart from x
            static_for<0, NB / 4>([&](auto kc) __attribute__((always_inline)) {
                zbcast_fma4<4 * decltype(kc)::value>(sr, si, nux, nuy, uv.y, l);
            });
            x[c].x += sr;
            x[c].y += si;
        }
        if (r < m) {
#pragma unroll
            for (int c = 0; c < ZU_CW; ++c)
                if (c < nc) A[r + (c0 + c) * lda] = x[c];
        }
    }
    __syncthreads();
    // U12 over the old top rows, which the update has taken by now
    if (t < 16 * ZU_CW) {
        const int c = t >> 4, k = t & 15;
        if (c < nc && k < NB) A[k + (c0 + c) * lda] = s_u[c][k];
    }
}

// The interchanges of the rows [jn, n) (at most ZN_MMAX of them) that columns
// [cbeg, cend) still lack: those from the end of the column's panel (of ncol
// columns) or from jn on.  Row i takes the row that the interchanges, taken
// backwards, trace it to.  A workgroup per panel.
template <typename R>
__global__ void __launch_bounds__(ZN_NTH)
znleft_kernel(i64 n, typename CplxT<R>::type* __restrict__ A, i64 lda, i64 jn, i64 cbeg, i64 cend,
              int ncol, const i64* __restrict__ piv)
{
    typedef typename CplxT<R>::type Z;
    constexpr int RPT = (int)(ZN_MMAX / ZN_NTH);
    __shared__ short s_piv[ZN_MMAX];
    const int t = threadIdx.x, m = (int)(n - jn);
    const i64 c0 = cbeg + (i64)blockIdx.x * ncol, c1 = c0 + ncol < cend ? c0 + ncol : cend;
    const int k0 = c1 > jn ? (int)(c1 - jn) : 0;
    for (int i = t; i < m; i += ZN_NTH) s_piv[i] = (short)(piv[jn + i] - jn);
    __syncthreads();
    int src[RPT];
#pragma unroll
    for (int q = 0; q < RPT; ++q) src[q] = t + q * ZN_NTH;
    for (int k = m - 1; k >= k0; --k) {
        const int p = s_piv[k];
#pragma unroll
        for (int q = 0; q < RPT; ++q) src[q] = src[q] == k ? p : src[q] == p ? k : src[q];
    }
    for (i64 c = c0; c < c1; ++c) {
        Z* a = A + jn + c * lda;
        Z x[RPT];
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            x[q].x = x[q].y = R(0);
            if (t + q * ZN_NTH < m) x[q] = a[src[q]];
        }
        __syncthreads();                             // every load before any store
#pragma unroll
        for (int q = 0; q < RPT; ++q)
            if (t + q * ZN_NTH < m && src[q] != t + q * ZN_NTH) a[t + q * ZN_NTH] = x[q];
    }
}

// Factor rows and columns [jn, n), n - jn <= ZN_MMAX, and give the columns
// left of jn their interchanges.  from: n ints.
template <typename R>
int zgetrf_tail(i64 n, typename CplxT<R>::type* A, i64 lda, i64 jn, i64* piv, i64* d_fz, int* from,
                hipStream_t s)
{
    // the panel width follows the rows a thread holds (registers)
    i64 jw = n;                              // the first wide panel
    for (i64 j0 = jn; j0 < n;) {
        const i64 m = n - j0;
        const int nb = m > 2 * ZN_NTH ? 8 : 16;
        if (nb == 16 && jw == n) jw = j0;
        const int jb = (int)(m < nb ? m : nb);
#define ZN_PANEL(RPT, NB)                                                                      \
    hipLaunchKernelGGL((znpanel_kernel<R, RPT, NB>), dim3(1), dim3(ZN_NTH), 0, s, n, A, lda,   \
                       j0, jb, piv, d_fz, from)
        if (m > 2 * ZN_NTH) ZN_PANEL(4, 8);
        else if (m > ZN_NTH) ZN_PANEL(2, 16);
        else ZN_PANEL(1, 16);
#undef ZN_PANEL
        const i64 right = n - j0 - nb;
        if (right > 0) {
            const dim3 grid((unsigned)((right + ZU_CW - 1) / ZU_CW));
            if (nb == 8)
                hipLaunchKernelGGL((znupdate_kernel<R, 8>), grid, dim3(256), 0, s, n, A, lda, j0,
                                   from);
            else
                hipLaunchKernelGGL((znupdate_kernel<R, 16>), grid, dim3(256), 0, s, n, A, lda, j0,
                                   from);
        }
        TMVX_CHECK_LAUNCH();
        j0 += jb;
    }
    auto left = [&](i64 cbeg, i64 cend, int ncol) {
        if (cend > cbeg)
            hipLaunchKernelGGL(znleft_kernel<R>, dim3((unsigned)((cend - cbeg + ncol - 1) / ncol)),
                               dim3(ZN_NTH), 0, s, n, A, lda, jn, cbeg, cend, ncol, piv);
    };
    left(0, jn, 16);
    left(jn, jw, 8);
    left(jw, n, 16);
    return hip_status(hipGetLastError());
}

template <typename R>
int zgetrf_impl(i64 n, R* Ar, i64 lda, i64* piv, i64* info, hipStream_t s)
{
    typedef typename CplxT<R>::type Z;
    if (n < 0 || lda < (n > 0 ? n : 1) || !info) return TMVX_ERR_ARG;
    *info = 0;
    if (n == 0) return TMVX_OK;
    if (!Ar || !piv) return TMVX_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(Ar) % sizeof(Z)) return TMVX_ERR_ARG;
    Z* A = reinterpret_cast<Z*>(Ar);
    i64* d_fz = nullptr;                     // the first zero pivot, then zgetrf_tail's row map
    if (hipMallocAsync((void**)&d_fz, sizeof(i64) + sizeof(int) * ZN_MMAX, s) != hipSuccess)
        return TMVX_ERR_ALLOC;
    const i64 big = n + 1;
    hipLaunchKernelGGL(set_i64_kernel, dim3(1), dim3(1), 0, s, d_fz, big);
    int rc = hip_status(hipGetLastError());
    for (i64 j0 = 0; j0 < n && rc == TMVX_OK; j0 += ZP_NB) {
        if (n - j0 <= ZN_MMAX) {
            rc = zgetrf_tail<R>(n, A, lda, j0, piv, d_fz, reinterpret_cast<int*>(d_fz + 1), s);
            break;
        }
        const int jb = ZP_NB;
        const i64 j1 = j0 + jb;
        hipLaunchKernelGGL(zpanel_kernel<R>, dim3(1), dim3(ZP_NTH), 0, s, n, A, lda, j0, j1, piv,
                           d_fz);
        if ((rc = hip_status(hipGetLastError())) != TMVX_OK) break;
        const i64 nr = n - j1;
        hipLaunchKernelGGL(ztrsm_u12_kernel<R>, dim3((unsigned)((nr + 255) / 256)), dim3(256), 0, s,
                           n, A, lda, j0, jb, j1);
        if ((rc = hip_status(hipGetLastError())) != TMVX_OK) break;
        rc = gemm_complex<R>(TMVX_COLMAJOR, TMVX_COLMAJOR, 0, 0, nr, nr, jb, R(-1), R(0),
                             reinterpret_cast<const R*>(A + j1 + j0 * lda), lda,
                             reinterpret_cast<const R*>(A + j0 + j1 * lda), lda, R(1), R(0),
                             reinterpret_cast<R*>(A + j1 + j1 * lda), lda, s);
    }
    i64 fz = big;
    if (hipMemcpyAsync(&fz, d_fz, sizeof(i64), hipMemcpyDeviceToHost, s) != hipSuccess &&
        rc == TMVX_OK)
        rc = TMVX_ERR_HIP;
    hipFreeAsync(d_fz, s);
    if (hipStreamSynchronize(s) != hipSuccess && rc == TMVX_OK) rc = TMVX_ERR_HIP;
    *info = fz <= n ? fz : 0;
    return rc;
}

// Interchanges on B's rows, one thread per right-hand side: in order
// (forward) or in reverse order (undo).
template <typename R>
__global__ void zpermute_kernel(i64 n, i64 nrhs, typename CplxT<R>::type* __restrict__ B, i64 ldb,
                                const i64* __restrict__ piv, int reverse)
{
    typedef typename CplxT<R>::type Z;
    const i64 r = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrhs) return;
    Z* b = B + r * ldb;
    for (i64 q = 0; q < n; ++q) {
        const i64 j = reverse ? n - 1 - q : q;
        const i64 p = piv[j];
        if (p != j && p >= 0 && p < n) {
            const Z x = b[j];
            b[j] = b[p];
            b[p] = x;
        }
    }
}

// Triangular column sweep on one right-hand side b (memory or LDS) by a
// workgroup.
//   mode 0: L x = b (unit lower), forward      mode 1: U x = b (upper), backward
//   mode 2: U^T x = b (lower), forward         mode 3: L^T x = b (unit upper), backward
// A zero U diagonal met by a non-zero entry sets *singular.
template <typename R>
__device__ __forceinline__ void zsweep(i64 n, const typename CplxT<R>::type* __restrict__ LU,
                                       i64 lda, typename CplxT<R>::type* b, int mode,
                                       typename CplxT<R>::type& s_x, int* __restrict__ singular)
{
    typedef typename CplxT<R>::type Z;
    const int t = threadIdx.x;
    const bool fwd = mode == 0 || mode == 2;
    const bool diag = mode == 1 || mode == 2;
    for (i64 q = 0; q < n; ++q) {
        const i64 j = fwd ? q : n - 1 - q;
        if (t == 0) {
            Z x = b[j];
            if (diag) {
                const Z d = LU[j + j * lda];
                if (d.x == R(0) && d.y == R(0)) {
                    if (x.x != R(0) || x.y != R(0)) *singular = 1;
                    x.x = R(0);
                    x.y = R(0);
                } else {
                    x = cdiv(x, d);
                }
                b[j] = x;
            }
            s_x = x;
        }
        __syncthreads();
        const Z x = s_x;
        if (x.x != R(0) || x.y != R(0)) {
            if (fwd) {
                for (i64 i = j + 1 + t; i < n; i += blockDim.x) {
                    // mode 0: L(i, j); mode 2: U^T(i, j) = U(j, i)
                    const Z a = mode == 0 ? LU[i + j * lda] : LU[j + i * lda];
                    b[i] = csub(b[i], cmul(a, x));
                }
            } else {
                for (i64 i = t; i < j; i += blockDim.x) {
                    // mode 1: U(i, j); mode 3: L^T(i, j) = L(j, i)
                    const Z a = mode == 1 ? LU[i + j * lda] : LU[j + i * lda];
                    b[i] = csub(b[i], cmul(a, x));
                }
            }
        }
        __syncthreads();
    }
}

template <typename R>
__global__ void __launch_bounds__(256)
zsweep_kernel(i64 n, const typename CplxT<R>::type* __restrict__ LU, i64 lda,
              typename CplxT<R>::type* __restrict__ B, i64 ldb, int mode, int* __restrict__ singular)
{
    __shared__ typename CplxT<R>::type s_x;
    zsweep<R>(n, LU, lda, B + (i64)blockIdx.x * ldb, mode, s_x, singular);
}

// One right-hand side per workgroup, n <= ZS_NMAX: both triangular solves on
// the vector in LDS.  Blocks of 16 rows: a thread loads its row's 16 entries of
// the block's columns, the first wave meanwhile solves the block (a row per
// lane, solved entries by DPP broadcast, one division an entry), then every row
// to come takes the block's product.  Bound: the block's chain of 16 divisions
// and one barrier pair per block.  mode as in zsweep; perm: row i of P A
// is row perm[i] of A.
constexpr int ZS_NMAX = 4096;
constexpr int ZS_NTH = 512;

template <typename R, int MODE>
__device__ __forceinline__ void zsolve_sweep(int n, const typename CplxT<R>::type* __restrict__ LU,
                                             i64 lda, typename CplxT<R>::type* s_b,
                                             int* __restrict__ singular)
{
    typedef typename CplxT<R>::type Z;
    constexpr bool fwd = MODE == 0 || MODE == 2, diag = MODE == 1 || MODE == 2;
    const int t = threadIdx.x, lane = t & 63, li = lane & 15;
    const int nb = (n + 15) >> 4;
    Z zero;
    zero.x = zero.y = R(0);
    // op(A)(i, 16 b + k), k < 16; columns past n and rows past the end as 0
    auto load = [&](int i, int b, Z (&a)[16]) __attribute__((always_inline)) {
        static_for<0, 16>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const int c = 16 * b + k;
            a[k] = zero;
            if (i >= 0 && i < n && c < n) a[k] = MODE < 2 ? LU[i + c * lda] : LU[c + i * lda];
        });
    };
    for (int q = 0; q < nb; ++q) {
        const int b = fwd ? q : nb - 1 - q;
        // rows to come: [r0, r1)
        const int r0 = fwd ? 16 * (b + 1) : 0, r1 = fwd ? n : 16 * b;
        Z a[16];
        load(r0 + t < r1 ? r0 + t : -1, b, a);
        if (t < 64) {
            const int r = 16 * b + li;
            // x: the entry less its products so far, formed anew in each step from
            // b less the sum of all but the last product (one fewer operation
            // on the chain than b less the whole sum)
            const Z bv = r < n ? s_b[r] : zero;
            Z x = bv, sum = zero, d[16], dd = zero;
            load(r, b, d);
            if constexpr (diag) {
                static_for<0, 16>([&](auto kc) __attribute__((always_inline)) {
                    constexpr int k = decltype(kc)::value;
                    if (li == k) dd = d[k];
                });
            }
            const bool dz = diag && r < n && dd.x == R(0) && dd.y == R(0);
            static_for<0, 16>([&](auto qc) __attribute__((always_inline)) {
                constexpr int k = fwd ? decltype(qc)::value : 15 - decltype(qc)::value;
                if constexpr (diag) {
                    if (li == k && r < n) {
                        if (dz) {
                            if (x.x != R(0) || x.y != R(0)) *singular = 1;
                            x = zero;
                        } else {
                            x = cdiv(x, dd);
                        }
                    }
                }
                const Z xk = row_bcast_z<k>(x);
                if (fwd ? li > k : li < k) {
                    const Z bs = csub(bv, sum);
                    x.x = fma(-d[k].x, xk.x, fma(d[k].y, xk.y, bs.x));
                    x.y = fma(-d[k].x, xk.y, fma(-d[k].y, xk.x, bs.y));
                    caddmul(sum, d[k], xk);
                }
            });
            if (lane < 16 && r < n) s_b[r] = x;
        }
        __syncthreads();
        const Z xv = 16 * b + li < n ? s_b[16 * b + li] : zero;
        for (int i0 = r0; i0 < r1; i0 += ZS_NTH) {
            const int i = i0 + t;
            if (i0 > r0) load(i < r1 ? i : -1, b, a);
            Z x = i < r1 ? s_b[i] : zero;
            R sr = R(0), si = R(0);          // minus the products, summed apart from x
            static_for<0, 4>([&](auto kc) __attribute__((always_inline)) {
                zbcast_fma4<4 * decltype(kc)::value>(sr, si, -xv.x, -xv.y, xv.y, a);
            });
            x.x += sr;
            x.y += si;
            if (i < r1) s_b[i] = x;
        }
        __syncthreads();
    }
}

template <typename R>
__global__ void __launch_bounds__(ZS_NTH)
zsolve_kernel(int trans, int n, const typename CplxT<R>::type* __restrict__ LU, i64 lda,
              const i64* __restrict__ perm, typename CplxT<R>::type* __restrict__ B, i64 ldb,
              int* __restrict__ singular)
{
    typedef typename CplxT<R>::type Z;
    __shared__ __attribute__((aligned(16))) Z s_b[ZS_NMAX];
    __shared__ Z s_x;
    __shared__ int s_sing;
    Z* b = B + (i64)blockIdx.x * ldb;
    const int t = threadIdx.x;
    for (int i = t; i < n; i += ZS_NTH) s_b[i] = trans ? b[i] : b[perm[i]];
    if (t == 0) s_sing = 0;
    __syncthreads();
    if (!trans) {
        zsolve_sweep<R, 0>(n, LU, lda, s_b, &s_sing);
        zsolve_sweep<R, 1>(n, LU, lda, s_b, &s_sing);
    } else {
        zsolve_sweep<R, 2>(n, LU, lda, s_b, &s_sing);
        zsolve_sweep<R, 3>(n, LU, lda, s_b, &s_sing);
    }
    // A zero entry takes no part in a substitution (src/TMV_TriDiv_V.cpp:187),
    // but a zero times an Inf or NaN of the factors does in a block of 16: a
    // solution with a NaN is found again by column sweeps, which skip it.
    int bad = 0;
    for (int i = t; i < n; i += ZS_NTH) bad |= s_b[i].x != s_b[i].x || s_b[i].y != s_b[i].y;
    if (__syncthreads_or(bad)) {
        for (int i = t; i < n; i += ZS_NTH) s_b[i] = trans ? b[i] : b[perm[i]];
        if (t == 0) s_sing = 0;
        __syncthreads();
#pragma clang loop unroll(disable)
        for (int mode = trans ? 2 : 0; mode < (trans ? 4 : 2); ++mode)
            zsweep<R>(n, LU, lda, s_b, mode, s_x, &s_sing);
    }
    if (t == 0 && s_sing) *singular = 1;
    for (int i = t; i < n; i += ZS_NTH) b[trans ? perm[i] : i] = s_b[i];
}

template <typename R>
int zgetrs_impl(int trans, i64 n, i64 nrhs, const R* LUr, i64 lda, const i64* piv, R* Br, i64 ldb,
                hipStream_t s)
{
    typedef typename CplxT<R>::type Z;
    if (n < 0 || nrhs < 0 || lda < (n > 0 ? n : 1) || ldb < (n > 0 ? n : 1)) return TMVX_ERR_ARG;
    if (n == 0 || nrhs == 0) return TMVX_OK;
    if (!LUr || !piv || !Br) return TMVX_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(LUr) % sizeof(Z) || reinterpret_cast<uintptr_t>(Br) % sizeof(Z))
        return TMVX_ERR_ARG;
    if (nrhs > 0x7fffffff) return TMVX_ERR_UNSUPPORTED;
    const Z* LU = reinterpret_cast<const Z*>(LUr);
    Z* B = reinterpret_cast<Z*>(Br);
    const bool in_lds = n <= ZS_NMAX;
    int* d_sing = nullptr;                   // the flag, then (n <= ZS_NMAX) the permutation
    if (hipMallocAsync((void**)&d_sing, 16 + (in_lds ? sizeof(i64) * (size_t)n : 0), s) !=
        hipSuccess)
        return TMVX_ERR_ALLOC;
    hipLaunchKernelGGL(set_int_kernel, dim3(1), dim3(1), 0, s, d_sing, 0);
    int rc = hip_status(hipGetLastError());
    const dim3 gp((unsigned)((nrhs + 63) / 64)), bp(64), gs((unsigned)nrhs), bs(256);
    if (rc == TMVX_OK && in_lds) {
        i64* perm = reinterpret_cast<i64*>(reinterpret_cast<char*>(d_sing) + 16);
        rc = piv_to_perm(n, piv, perm, s);
        if (rc == TMVX_OK) {
            hipLaunchKernelGGL(zsolve_kernel<R>, gs, dim3(ZS_NTH), 0, s, trans, (int)n, LU, lda,
                               perm, B, ldb, d_sing);
            rc = hip_status(hipGetLastError());
        }
    } else if (rc == TMVX_OK && !trans) {
        hipLaunchKernelGGL(zpermute_kernel<R>, gp, bp, 0, s, n, nrhs, B, ldb, piv, 0);
        hipLaunchKernelGGL(zsweep_kernel<R>, gs, bs, 0, s, n, LU, lda, B, ldb, 0, d_sing);
        hipLaunchKernelGGL(zsweep_kernel<R>, gs, bs, 0, s, n, LU, lda, B, ldb, 1, d_sing);
        rc = hip_status(hipGetLastError());
    } else if (rc == TMVX_OK) {
        hipLaunchKernelGGL(zsweep_kernel<R>, gs, bs, 0, s, n, LU, lda, B, ldb, 2, d_sing);
        hipLaunchKernelGGL(zsweep_kernel<R>, gs, bs, 0, s, n, LU, lda, B, ldb, 3, d_sing);
        hipLaunchKernelGGL(zpermute_kernel<R>, gp, bp, 0, s, n, nrhs, B, ldb, piv, 1);
        rc = hip_status(hipGetLastError());
    }
    int h_sing = 0;
    if (hipMemcpyAsync(&h_sing, d_sing, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess &&
        rc == TMVX_OK)
        rc = TMVX_ERR_HIP;
    hipFreeAsync(d_sing, s);
    if (hipStreamSynchronize(s) != hipSuccess && rc == TMVX_OK) rc = TMVX_ERR_HIP;
    if (rc == TMVX_OK && h_sing) rc = TMVX_ERR_SINGULAR;
    return rc;
}

} // namespace tmvx

using namespace tmvx;

extern "C" {

int tmvx_getrf_z(int64_t n, double* A, int64_t lda, int64_t* piv, int64_t* info, void* stream)
{ return zgetrf_impl<double>(n, A, lda, piv, info, (hipStream_t)stream); }

int tmvx_getrf_c(int64_t n, float* A, int64_t lda, int64_t* piv, int64_t* info, void* stream)
{ return zgetrf_impl<float>(n, A, lda, piv, info, (hipStream_t)stream); }

int tmvx_getrs_z(int trans, int64_t n, int64_t nrhs, const double* LU, int64_t lda,
                 const int64_t* piv, double* B, int64_t ldb, void* stream)
{ return zgetrs_impl<double>(trans, n, nrhs, LU, lda, piv, B, ldb, (hipStream_t)stream); }

int tmvx_getrs_c(int trans, int64_t n, int64_t nrhs, const float* LU, int64_t lda,
                 const int64_t* piv, float* B, int64_t ldb, void* stream)
{ return zgetrs_impl<float>(trans, n, nrhs, LU, lda, piv, B, ldb, (hipStream_t)stream); }

} // extern "C"

// ---------------------------------------------------------------------------
// Determinant and inverse from the complex factors.
// ---------------------------------------------------------------------------
namespace tmvx {

// out[0] = sum log|U_ii| (FP64), out[1..2] = det(P) * prod U_ii / |U_ii|
// (0 with out[0] = -inf when a diagonal is 0): LUDiv::logDet for complex T
// (src/TMV_LUD.cpp:145-156; DiagMatrix::logDet multiplies the signs z/|z|,
// src/TMV_DiagMatrix.cpp:59-90).  One workgroup of 256 threads.
template <typename R>
__global__ void __launch_bounds__(256)
zlogdet_kernel(i64 n, const typename CplxT<R>::type* __restrict__ LU, i64 lda,
               const i64* __restrict__ piv, double* __restrict__ out)
{
    __shared__ double s_l[256], s_re[256], s_im[256];
    __shared__ int s_neg[256], s_zero[256];
    const int t = threadIdx.x;
    double sum = 0.0, pr = 1.0, pi = 0.0;
    int neg = 0, zero = 0;
    for (i64 i = t; i < n; i += blockDim.x) {
        const double x = (double)LU[i + i * lda].x, y = (double)LU[i + i * lda].y;
        const double a = hypot(x, y);
        if (a == 0.0) zero = 1;
        else {
            sum += log(a);
            const double ur = x / a, ui = y / a;
            const double nr = pr * ur - pi * ui;
            pi = pr * ui + pi * ur;
            pr = nr;
        }
        if (piv[i] != i) neg ^= 1;
    }
    s_l[t] = sum; s_re[t] = pr; s_im[t] = pi; s_neg[t] = neg; s_zero[t] = zero;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (t < off) {
            s_l[t] += s_l[t + off];
            const double ar = s_re[t], ai = s_im[t], br = s_re[t + off], bi = s_im[t + off];
            s_re[t] = ar * br - ai * bi;
            s_im[t] = ar * bi + ai * br;
            s_neg[t] ^= s_neg[t + off];
            s_zero[t] |= s_zero[t + off];
        }
        __syncthreads();
    }
    if (t == 0) {
        const double sg = s_neg[0] ? -1.0 : 1.0;
        out[0] = s_zero[0] ? -INFINITY : s_l[0];
        out[1] = s_zero[0] ? 0.0 : sg * s_re[0];
        out[2] = s_zero[0] ? 0.0 : sg * s_im[0];
    }
}

template <typename R>
__global__ void zidentity_kernel(i64 n, typename CplxT<R>::type* __restrict__ X, i64 ldx)
{
    const i64 j = blockIdx.y;
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x) {
        typename CplxT<R>::type z;
        z.x = i == j ? R(1) : R(0);
        z.y = R(0);
        X[i + j * ldx] = z;
    }
}

template <typename R>
int zlogdet_impl(i64 n, const R* LUr, i64 lda, const i64* piv, double* logdet, double* sre,
                 double* sim, hipStream_t s)
{
    typedef typename CplxT<R>::type Z;
    if (n < 0 || lda < (n > 0 ? n : 1) || !logdet || !sre || !sim) return TMVX_ERR_ARG;
    if (n == 0) { *logdet = 0.0; *sre = 1.0; *sim = 0.0; return TMVX_OK; }
    if (!LUr || !piv) return TMVX_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(LUr) % sizeof(Z)) return TMVX_ERR_ARG;
    double* d = nullptr;
    if (hipMalloc((void**)&d, 3 * sizeof(double)) != hipSuccess) return TMVX_ERR_ALLOC;
    hipLaunchKernelGGL(zlogdet_kernel<R>, dim3(1), dim3(256), 0, s, n,
                       reinterpret_cast<const Z*>(LUr), lda, piv, d);
    int rc = hip_status(hipGetLastError());
    double h[3] = {0.0, 0.0, 0.0};
    if (rc == TMVX_OK && hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess)
        rc = TMVX_ERR_HIP;
    if (hipStreamSynchronize(s) != hipSuccess && rc == TMVX_OK) rc = TMVX_ERR_HIP;
    hipFree(d);
    *logdet = h[0];
    *sre = h[1];
    *sim = h[2];
    return rc;
}

template <typename R>
int zgetri_impl(i64 n, const R* LU, i64 lda, const i64* piv, R* Xr, i64 ldx, hipStream_t s)
{
    typedef typename CplxT<R>::type Z;
    if (n < 0 || lda < (n > 0 ? n : 1) || ldx < (n > 0 ? n : 1)) return TMVX_ERR_ARG;
    if (n == 0) return TMVX_OK;
    if (!LU || !piv || !Xr) return TMVX_ERR_ARG;
    if (n > 65535) return TMVX_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(Xr) % sizeof(Z)) return TMVX_ERR_ARG;
    const i64 gx = (n + 255) / 256;
    hipLaunchKernelGGL(zidentity_kernel<R>, dim3((unsigned)(gx < 64 ? gx : 64), (unsigned)n),
                       dim3(256), 0, s, n, reinterpret_cast<Z*>(Xr), ldx);
    TMVX_CHECK_LAUNCH();
    return zgetrs_impl<R>(0, n, n, LU, lda, piv, Xr, ldx, s);
}

} // namespace tmvx

extern "C" {

int tmvx_logdet_z(int64_t n, const double* LU, int64_t lda, const int64_t* piv, double* logdet,
                  double* sign_re, double* sign_im, void* stream)
{ return tmvx::zlogdet_impl<double>(n, LU, lda, piv, logdet, sign_re, sign_im, (hipStream_t)stream); }

int tmvx_getri_z(int64_t n, const double* LU, int64_t lda, const int64_t* piv, double* X,
                 int64_t ldx, void* stream)
{ return tmvx::zgetri_impl<double>(n, LU, lda, piv, X, ldx, (hipStream_t)stream); }

} // extern "C"
