// Batched LU of medium systems: one workgroup factors one system of
// n <= 1024 in place in global memory.
//
// Per system TMV's LU_Decompose (src/TMV_LUDecompose.cpp:217-407): largest
// |a|, first row on ties (src/TMV_Vector.cpp:473-504), the underflow rule (the
// column is zeroed from the diagonal down and interchanged with itself,
// src/TMV_LUDecompose.cpp:162-169), the column scaled by the pivot's
// reciprocal.
//
// Right-looking in panels of WL_NB = 32 columns:
//   panel: one row per thread, in registers (n <= the workgroup's threads).
//     Rows never move while the panel is factored (a thread carries its
//     row's position); per column each wave's best row writes itself to LDS
//     before the column's only barrier, then every wave picks the winner
//     among the waves' candidates and updates its rows;
//   interchanges + U12 = L11^-1 A12: one column per lane, the 32 rows in
//     registers, L11 read from LDS as broadcasts; U12 stays in LDS;
//   A22 -= L21 U12 on MFMA, 32 x 32 of A22 per wave, L21 read from L2, U12
//     from LDS.  The product is formed transposed, so that the 16 lanes of
//     an MFMA column hold 16 consecutive rows: A22 moves in 128-byte runs.
// The interchanges of the columns left of a panel (L's) are all applied at
// the end, one pass over the matrix (thread per row, the source row traced
// back through the interchange list), instead of a scattered pass per panel.
//
// Bound: the panel's chain of one barrier per column and the latency of
// the A22 tiles, with two workgroups per CU to overlap them; n^3 / (3 WL_NB)
// elements of A22 are read and written.
#include "tmvx_lu.h"
#include "tmvx_pivot.h"

#include <climits>
#include <cmath>

namespace tmvx {

constexpr int WL_NB = 32;        // panel width
constexpr int WL_CH = 256;       // trailing columns whose U12 is in LDS at once
constexpr int WL_LDU = WL_CH + 16;   // 16 elements of padding: the 4 lane groups of an
                                     // MFMA operand read rows k, k+1, .. without conflicts

template <typename T, int NTH>
__global__ void __launch_bounds__(NTH) __attribute__((amdgpu_waves_per_eu(NTH == 1024 ? 4 : 2)))
lu_wg_kernel(const int* __restrict__ order, const int32_t* __restrict__ nv, T* const* Av,
             int64_t* const* pivv, int32_t* __restrict__ info)
{
    constexpr int NW = NTH / 64, NB = WL_NB;
    constexpr int VN = Vec16<T>::n;
    typedef typename Vec16<T>::type VT;
    typedef typename Mfma<T>::v4 v4;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    __shared__ __attribute__((aligned(16))) T s_row[2][NW][NB];   // the waves' candidate rows
    __shared__ T s_v[2][NW];
    __shared__ int s_i[2][NW];
    __shared__ __attribute__((aligned(16))) T s_l[NB][NB];        // s_l[k][i] = L11(i, k)
    __shared__ __attribute__((aligned(16))) T s_u[NB][WL_LDU];    // U12 of one column chunk
    __shared__ int s_src[NB];     // panel row k comes from panel-relative row s_src[k]
    __shared__ int s_dst[NB];     // the row that was panel row k goes to s_dst[k]
    __shared__ int s_piv[NTH];    // the whole interchange list
    const int sys = order[blockIdx.x];
    const int n = nv[sys];
    T* __restrict__ A = Av[sys];
    const i64 ld = n;
    int first_zero = 0;

    for (int j = 0; j < n; j += NB) {
        const int m = n - j, jb = m < NB ? m : NB;
        // ---- panel ------------------------------------------------------
        const bool own = t < m;
        T row[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) row[c] = (own && c < jb) ? A[(j + t) + (j + c) * ld] : T(0);
        int pos = t;
        bool used = !own;
        // blocks of 8 columns, the block in hand in row[0..8): after block b
        // the row is rotated by 8, row[c] is column 8 b + c while that is < NB
        for (int b = 0; b < NB / 8; ++b) {
            static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
                constexpr int kk = decltype(kc)::value;
                const int k = 8 * b + kk;
                if (k >= jb) return;                                  // uniform
                constexpr int par = kk & 1;
                T v;
                int vi;
                lanes_argmax<64, T>(used ? T(-1) : T(fabs(row[kk])), pos, v, vi);
                if (lane == 0) { s_v[par][wave] = v; s_i[par][wave] = vi; }
                if (!used && pos == vi) {
                    static_for<0, NB / VN>([&](auto qc) __attribute__((always_inline)) {
                        constexpr int q = decltype(qc)::value * VN;
                        if constexpr (q + VN > kk) {
                            VT x;
                            static_for<0, VN>([&](auto uc) __attribute__((always_inline)) {
                                x[decltype(uc)::value] = row[q + decltype(uc)::value];
                            });
                            *reinterpret_cast<VT*>(&s_row[par][wave][q]) = x;
                        }
                    });
                }
                __syncthreads();
                T gv;
                int gi;
                const int ci = lane < NW ? s_i[par][lane] : INT_MAX;
                lanes_argmax<(NW > 8 ? 16 : 8)>(lane < NW ? s_v[par][lane] : T(-1), ci, gv, gi);
                const bool zero = !(gv >= tiny<T>());
                if (t == 0) s_piv[j + k] = j + (zero ? k : gi);
                if (zero) {
                    if (first_zero == 0) first_zero = j + k + 1;
                    if (!used) row[kk] = T(0);
                    if (!used && pos == k) used = true;
                } else {
                    const unsigned long long hw = __ballot(lane < NW && ci == gi);
                    const T* pr = &s_row[par][hw ? (int)__builtin_ctzll(hw) : 0][0];
                    if (!used && pos == gi) { used = true; pos = k; }
                    else if (!used && pos == k) pos = gi;
                    // rows already pivotal take multiplier 0 for their
                    // updates and keep their own column
                    const T l = row[kk] * (T(1) / pr[kk]);
                    if (!used) row[kk] = l;
                    const T lu = used ? T(0) : l;
                    static_for<0, NB / 8>([&](auto cc) __attribute__((always_inline)) {
                        constexpr int c0 = decltype(cc)::value * 8;
                        if (c0 >= NB - 8 * b) return;                 // uniform
                        static_for<0, 8 / VN>([&](auto qc) __attribute__((always_inline)) {
                            constexpr int q = c0 + decltype(qc)::value * VN;
                            if constexpr (q + VN > kk + 1) {
                                const VT u = *reinterpret_cast<const VT*>(pr + q);
                                static_for<0, VN>([&](auto uc) __attribute__((always_inline)) {
                                    constexpr int x = decltype(uc)::value;
                                    if constexpr (q + x > kk)
                                        if (!used) row[q + x] -= lu * u[x];
                                });
                            }
                        });
                    });
                }
            });
            T first[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) first[q] = row[q];
#pragma unroll
            for (int c = 0; c < NB - 8; ++c) row[c] = row[c + 8];
#pragma unroll
            for (int q = 0; q < 8; ++q) row[NB - 8 + q] = first[q];
        }
        // rows to their final positions; L11 and the row moves to LDS
        if (own) {
#pragma unroll
            for (int c = 0; c < NB; ++c)
                if (c < jb) A[(j + pos) + (j + c) * ld] = row[c];
            if (pos < NB) {
                s_src[pos] = t;
#pragma unroll
                for (int c = 0; c < NB; ++c) s_l[c][pos] = row[c];
            }
            if (t < NB) s_dst[t] = pos;
        }
        __syncthreads();
        if (m <= NB) break;

        // ---- interchanges, U12 and A22, WL_CH columns at a time ----------
        for (int cb = j + NB; cb < n; cb += WL_CH) {
            const int nc = n - cb < WL_CH ? n - cb : WL_CH;
            for (int c = t; c < WL_CH; c += NTH) {
                if (c >= nc) {              // read by edge tiles, never stored
#pragma unroll
                    for (int k = 0; k < NB; ++k) s_u[k][c] = T(0);
                    continue;
                }
                T* __restrict__ col = A + j + (cb + c) * ld;
                T x[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) x[k] = col[s_src[k]];
                // every gathered row has been read before a row is moved
                // over it; the panel's own rows are rewritten only below
                __builtin_amdgcn_s_waitcnt(0);
                static_for<0, NB / 8>([&](auto qc) __attribute__((always_inline)) {
                    constexpr int k0 = decltype(qc)::value * 8;
                    __asm__ volatile("" ::: "memory");
                    T old[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) old[k] = s_dst[k0 + k] >= NB ? col[k0 + k] : T(0);
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        if (s_dst[k0 + k] >= NB) col[s_dst[k0 + k]] = old[k];
                });
                static_for<0, NB>([&](auto kc) __attribute__((always_inline)) {
                    constexpr int k = decltype(kc)::value;
                    static_for<k + 1, NB>([&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        x[i] -= s_l[k][i] * x[k];
                    });
                    __asm__ volatile("" ::: "memory");   // L11's reads stay in their step
                });
#pragma unroll
                for (int k = 0; k < NB; ++k) { col[k] = x[k]; s_u[k][c] = x[k]; }
            }
            __syncthreads();
            const int li = lane & 15, g = lane >> 4;
            const int tm = (m - NB + 31) / 32, tn = (nc + 31) / 32;
            for (int tile = wave; tile < tm * tn; tile += NW) {
                const int r0 = j + NB + 32 * (tile % tm), c0 = 32 * (tile / tm);
                int rr[2];                  // rows past the end read the last one
                T lf[2][8], uf[2][8];
                static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    const int r = r0 + 16 * i + li;
                    rr[i] = r < n ? r : n - 1;
                });
                v4 acc[2][2];               // acc[jc][i]: columns c0 + 16 jc.., rows r0 + 16 i..
                static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                    static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                        static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
                            constexpr int q = decltype(rc)::value;
                            const int c = c0 + 16 * decltype(jc)::value + Mfma<T>::row(g, q);
                            acc[decltype(jc)::value][decltype(ic)::value][q] =
                                A[rr[decltype(ic)::value] + (cb + (c < nc ? c : nc - 1)) * ld];
                        });
                    });
                });
                static_for<0, 8>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        lf[i][s] = -A[rr[i] + (j + 4 * s + g) * ld];
                        uf[i][s] = s_u[4 * s + g][c0 + 16 * i + li];
                    });
                });
                static_for<0, 8>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                        static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                            constexpr int jj = decltype(jc)::value, i = decltype(ic)::value;
                            acc[jj][i] = Mfma<T>::mac(uf[jj][s], lf[i][s], acc[jj][i]);
                        });
                    });
                });
                static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                    static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                        static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
                            constexpr int q = decltype(rc)::value, i = decltype(ic)::value;
                            const int c = c0 + 16 * decltype(jc)::value + Mfma<T>::row(g, q);
                            if (r0 + 16 * i + li < n && c < nc)
                                A[rr[i] + (cb + c) * ld] = acc[decltype(jc)::value][i][q];
                        });
                    });
                });
            }
            __syncthreads();
        }
    }

    // ---- L's deferred interchanges, last panel first: row t takes the row
    // that the interchanges of all later panels bring to it -----------------
    int src = t;
    const int last = (n - 1) / NB * NB;           // first column of the last panel
    for (int j = last - NB; j >= 0; j -= NB) {
        const int k1 = j + NB, k2 = k1 + NB < n ? k1 + NB : n;
        for (int k = k2 - 1; k >= k1; --k) {
            const int p = s_piv[k];
            src = src == k ? p : src == p ? k : src;
        }
        const bool moves = t < n && src != t;
        T x[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) x[c] = moves ? A[src + (j + c) * ld] : T(0);
        __syncthreads();                          // every load before any store
        if (moves) {
#pragma unroll
            for (int c = 0; c < NB; ++c) A[t + (j + c) * ld] = x[c];
        }
    }
    for (int k = t; k < n; k += NTH) pivv[sys][k] = s_piv[k];
    if (t == 0) info[sys] = first_zero;
}

template <typename T>
int lu_wg_launch(int nmax, int count, const int* d_order, const int32_t* d_n, T* const* A,
                 int64_t* const* piv, int32_t* info, hipStream_t s)
{
    if (count <= 0) return TMVX_OK;
    if (nmax > 1024) return TMVX_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)count);
    if (nmax <= 256)
        hipLaunchKernelGGL((lu_wg_kernel<T, 256>), grid, dim3(256), 0, s, d_order, d_n, A, piv, info);
    else if (nmax <= 512)
        hipLaunchKernelGGL((lu_wg_kernel<T, 512>), grid, dim3(512), 0, s, d_order, d_n, A, piv, info);
    else
        hipLaunchKernelGGL((lu_wg_kernel<T, 1024>), grid, dim3(1024), 0, s, d_order, d_n, A, piv,
                           info);
    return hip_status(hipGetLastError());
}

template int lu_wg_launch<double>(int, int, const int*, const int32_t*, double* const*,
                                  int64_t* const*, int32_t*, hipStream_t);
template int lu_wg_launch<float>(int, int, const int*, const int32_t*, float* const*,
                                 int64_t* const*, int32_t*, hipStream_t);

} // namespace tmvx
