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
//   U12 = L11^-1 A12: one column per lane, its 32 pivot rows gathered into
//     registers, L11 read from LDS as broadcasts; U12 stays in LDS;
//   A22 -= L21 U12 on MFMA, 32 x 32 of A22 per wave, L21 read from L2, U12
//     from LDS; the interchanges are the row each update is read from.  The product is formed transposed, so that the 16 lanes of
//     an MFMA column hold 16 consecutive rows: A22 moves in 128-byte runs.
// The interchanges of the columns left of a panel (L's) are all applied at
// the end, one pass over the matrix (thread per row, the source row traced
// back through the interchange list), instead of a scattered pass per panel.
//
// Bound: the panel's chain of one barrier per column (0.8 us a column with
// two workgroups on the CU, most of it LDS traffic: every wave writes its
// candidate row and reads the winner's) and the latency of the A22 tiles;
// n^3 / (3 WL_NB) elements of A22 are read and written.  Measured, 512
// systems of n = 256 FP64: 0.63 ms (panels 0.20-0.22, U12 0.10, A22 0.18,
// L's interchanges 0.03), against 9.7 ms for rank-1 updates of the whole
// matrix in global memory with six barriers a column; 0.87 ms with the pivot
// search on floating-point maxima, a rotated panel row and the interchanges
// as a pass of their own.
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
    constexpr int NWP = NW <= 4 ? 4 : NW <= 8 ? 8 : 16;           // lanes that compare waves
    __shared__ __attribute__((aligned(16))) T s_row[2][NW][NB];   // the waves' candidate rows
    __shared__ unsigned s_hi[2][16], s_lo[2][16];                 // their keys and positions
    __shared__ int s_pos[2][16];
    __shared__ __attribute__((aligned(16))) T s_l[NB][NB];        // s_l[k][i] = L11(i, k)
    __shared__ __attribute__((aligned(16))) T s_u[NB][WL_LDU];    // U12 of one column chunk
    __shared__ short s_src[NB];   // panel row k comes from panel-relative row s_src[k]
    __shared__ short s_from[NTH]; // row r of the panel's moved rows comes from s_from[r]
    __shared__ short s_piv[NTH];  // the whole interchange list
    const int sys = order[blockIdx.x];
    const int n = nv[sys];
    T* __restrict__ A = Av[sys];
    const i64 ld = n;
    int first_zero = 0;
    if (t < 16) {                       // no candidate from waves that do not exist
        s_hi[0][t] = s_hi[1][t] = 0u;
        s_lo[0][t] = s_lo[1][t] = 0u;
        s_pos[0][t] = s_pos[1][t] = INT_MAX;
    }
    __syncthreads();

    for (int j = 0; j < n; j += NB) {
        const int m = n - j, jb = m < NB ? m : NB;
        // ---- panel ------------------------------------------------------
        const bool own = t < m;
        T row[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) row[c] = (own && c < jb) ? A[(j + t) + (j + c) * ld] : T(0);
        int pos = t;
        bool used = !own;
        // (a last panel narrower than NB runs its missing columns as zero
        // columns, with nothing recorded)
        static_for<0, NB>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value, par = k & 1;
            const unsigned hi = used ? 0u : mag_hi(row[k]), lo = mag_lo(row[k]);
            unsigned m;
            const int wl = lanes_best<64, T>(hi, lo, pos, m);
            if (lane == wl) {
                s_hi[par][wave] = m;
                s_lo[par][wave] = lo;
                s_pos[par][wave] = pos;
                static_for<k / VN, NB / VN>([&](auto qc) __attribute__((always_inline)) {
                    constexpr int q = decltype(qc)::value * VN;
                    VT x;
                    static_for<0, VN>([&](auto uc) __attribute__((always_inline)) {
                        x[decltype(uc)::value] = row[q + decltype(uc)::value];
                    });
                    *reinterpret_cast<VT*>(&s_row[par][wave][q]) = x;
                });
            }
            __syncthreads();
            unsigned gm;
            const int cpos = s_pos[par][lane & 15];
            const int ww = lanes_best<NWP, T>(s_hi[par][lane & 15], s_lo[par][lane & 15], cpos, gm);
            const bool zero = gm < mag_tiny<T>();                      // TMV_Underflow
            const int p = zero ? k : __builtin_amdgcn_readlane(cpos, ww);
            const T* pr = &s_row[par][ww][0];
            T u[NB];
            static_for<k / VN, NB / VN>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value * VN;
                const VT x = *reinterpret_cast<const VT*>(pr + q);
                static_for<0, VN>([&](auto uc) __attribute__((always_inline)) {
                    u[q + decltype(uc)::value] = x[decltype(uc)::value];
                });
            });
            if (t == 0 && k < jb) s_piv[j + k] = (short)(j + p);
            if (zero && first_zero == 0 && k < jb) first_zero = j + k + 1;
            if (zero && !used) row[k] = T(0);
            const bool isp = !used && pos == p;
            if (!used && pos == k) pos = p;
            if (isp) pos = k;
            used = used || isp;
            const T l = row[k] * (T(1) / u[k]);
            if (!used && !zero) {
                row[k] = l;
                static_for<k + 1, NB>([&](auto cc) __attribute__((always_inline)) {
                    constexpr int c = decltype(cc)::value;
                    row[c] -= l * u[c];
                });
            }
        });
        // rows to their final positions; L11 and the row moves to LDS
        if (own) {
#pragma unroll
            for (int c = 0; c < NB; ++c)
                if (c < jb) A[(j + pos) + (j + c) * ld] = row[c];
            if (pos < NB) {
                s_src[pos] = (short)t;
#pragma unroll
                for (int c = 0; c < NB; ++c) s_l[c][pos] = row[c];
            }
            s_from[pos] = (short)t;
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
                const T* __restrict__ col = A + j + (cb + c) * ld;
                T x[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) x[k] = col[s_src[k]];
                // (L11's column k is read when x[k - 4] is final: an opaque
                // dependency, or the reads would be hoisted to the top)
                int off = 0;
                static_for<0, NB>([&](auto kc) __attribute__((always_inline)) {
                    constexpr int k = decltype(kc)::value;
                    if constexpr (k >= 4 && k % 4 == 0) __asm__ volatile("" : "+v"(off) : "v"(x[k - 4]));
                    const T* lk = &s_l[k][0] + off;
                    static_for<k + 1, NB>([&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        x[i] -= lk[i] * x[k];
                    });
                });
#pragma unroll
                for (int k = 0; k < NB; ++k) s_u[k][c] = x[k];
            }
            __syncthreads();
            // A22: row r takes its update from the row that the interchanges
            // bring to it (one of the panel's own rows, unless it stays), so
            // the moves cost no pass of their own
            const int li = lane & 15, g = lane >> 4;
            const int tm = (m - NB + 31) / 32, tn = (nc + 31) / 32;
            for (int tile = wave; tile < tm * tn; tile += NW) {
                const int r0 = NB + 32 * (tile % tm), c0 = 32 * (tile / tm);
                int rr[2], fr[2];           // rows past the end read the last one
                T lf[2][8], uf[2][8];
                static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    const int r = r0 + 16 * i + li;
                    rr[i] = j + (r < m ? r : m - 1);
                    fr[i] = j + s_from[r < m ? r : m - 1];
                });
                v4 acc[2][2];               // acc[jc][i]: columns c0 + 16 jc.., rows r0 + 16 i..
                static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                    static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                        static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
                            constexpr int q = decltype(rc)::value;
                            const int c = c0 + 16 * decltype(jc)::value + Mfma<T>::row(g, q);
                            acc[decltype(jc)::value][decltype(ic)::value][q] =
                                A[fr[decltype(ic)::value] + (cb + (c < nc ? c : nc - 1)) * ld];
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
                            if (r0 + 16 * i + li < m && c < nc)
                                A[rr[i] + (cb + c) * ld] = acc[decltype(jc)::value][i][q];
                        });
                    });
                });
            }
            __syncthreads();
            // U12 over the panel's old rows, which A22 has taken by now
            for (int e = t; e < NB * nc; e += NTH)
                A[j + (e & (NB - 1)) + (cb + e / NB) * ld] = s_u[e & (NB - 1)][e / NB];
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
