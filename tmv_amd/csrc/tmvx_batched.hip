// Batched LU factorisation and solve of many small independent systems, and
// a batched GEMM over the same kind of ragged sizes.
//
// Counterpart, per system, of TMV's LU_Decompose + LU_LDivEq
// (src/TMV_LUDecompose.cpp:217-407, src/TMV_LUDiv.cpp:185-226) and MultMM
// (src/TMV_MultMM.cpp:404-477); TMV has no batched entry point, a caller
// loops over systems.  Here up to three launches, a workgroup or wave per system.
//
// Factor + solve kernels; a system of n <= 64 takes one wave, a larger one
// (n <= 128) a workgroup of two:
//   panel of up to 64 columns, a row per lane, in registers (panel64).  Rows
//     never move: a lane carries its row's position, so pivots, tie rule
//     (first maximum in the current row order) and underflow rule are TMV's
//     GEPP.  Columns go in blocks of 8.  Per column: the search on integer
//     keys (lanes_best), the best row's entries in the block to LDS (with
//     two waves, each wave's best row's, and a barrier), the update of the
//     block.  Per block: its 8 pivot rows to LDS at once, their U12 a column
//     per lane, and one rank-8 update of the columns to come, the rows of U12
//     read 16 entries per row of lanes and handed on by DPP broadcasts.  The
//     LDS is what this is built around: a write costs a wave ~30 cycles
//     whatever it carries, so a whole pivot row per column (up to 32 writes of
//     one lane each) took 3400 cycles a column at n = 64, most of them here;
//   n <= 64: that is the whole factorisation; the right-hand sides are
//     solved from the rows in registers, four at a time (n <= 32 is a kernel of
//     its own, whose registers let more waves in);
//   n > 64: the columns right of the panel, 16 to a wave: U12 by blocks of
//     16 rows and A22 -= L21 U12 on MFMA (tmvx_wg_solve.h), the interchanges
//     being where the rows are read from, the right-hand sides as one more
//     such chunk; then A22 (n - 64 <= 64) and its right-hand sides as a panel
//     of one wave, its interchanges on L21, and U11's part of the solution.
// A plan (made once per batch shape) orders the work list largest first.
// The launch allocates nothing and sets nothing on the host, so it can be
// captured in a hipGraph and replayed.
#include "tmvx_lu.h"
#include "tmvx_pivot.h"
#include "tmvx_wg_solve.h"
#include "../../include/tmvx_batched.h"

#include <algorithm>
#include <climits>
#include <cstdio>
#include <cstring>
#include <new>
#include <numeric>
#include <vector>

namespace tmvx {

template <typename T>
struct BatchArgs {
    const int4* slots;      // {system, n, nrhs, 0}, in work-list order
    T* const* A;            // n x n column-major, lda = n
    i64* const* piv;        // n interchanges, 0-based
    T* const* B;            // n x nrhs column-major, ldb = n (may be null if nrhs = 0)
    int* info;              // per system: 1-based first zero pivot, or 0
};

constexpr int BK_NW = 2;                // waves per workgroup system
constexpr int BK_NTH = 64 * BK_NW;
constexpr int BK_CH = 8;                // columns per block of the panel

// LDS of a panel of N columns, its rows in NW waves.
template <typename T, int N, int NW>
struct PanelLds {
    __attribute__((aligned(16))) T u[BK_CH][N];             // a block's pivot rows
    __attribute__((aligned(16))) T row[2][NW][BK_CH];       // candidates (column parity)
    __attribute__((aligned(16))) int4 key[2][4];            // {high, low key, position, 0}
    short piv[N];                       // interchange list
    short from[64 * NW];                // the row that the panel brings to each position
};

// row[c] := row[(c + BK_CH) mod N], and back.
template <typename T, int N>
__device__ __forceinline__ void rotate_row(T (&row)[N])
{
    T first[BK_CH];
#pragma unroll
    for (int q = 0; q < BK_CH; ++q) first[q] = row[q];
#pragma unroll
    for (int c = 0; c < N - BK_CH; ++c) row[c] = row[c + BK_CH];
#pragma unroll
    for (int q = 0; q < BK_CH; ++q) row[N - BK_CH + q] = first[q];
}
template <typename T, int N>
__device__ __forceinline__ void rotate_row_back(T (&row)[N])
{
    T last[BK_CH];
#pragma unroll
    for (int q = 0; q < BK_CH; ++q) last[q] = row[N - BK_CH + q];
#pragma unroll
    for (int c = N - 1; c >= BK_CH; --c) row[c] = row[c - BK_CH];
#pragma unroll
    for (int q = 0; q < BK_CH; ++q) row[q] = last[q];
}

// Factor columns [0, jb) (jb <= N) of m rows in place: thread t of NW waves
// holds row t in row[c], c < jb.  On return the row's final position in pos,
// for a pivot row the reciprocal of its pivot in rdiag, and in L.piv the
// interchanges, in first_zero (0 before) the 1-based first zero pivot.
template <int NW, typename T, int N>
__device__ __forceinline__ void panel_rows(T (&row)[N], int m, int jb, int t,
                                           PanelLds<T, N, NW>& L, int& pos, T& rdiag,
                                           int& first_zero)
{
    typedef typename Vec16<T>::type VT;
    constexpr int VN = Vec16<T>::n, CH = BK_CH;
    static_assert(CH == 8, "half a row of lanes");
    static_assert(NW <= 4, "waves whose candidates are compared");
    const int lane = t & 63, w = NW == 1 ? 0 : t >> 6;
    auto& U = L.u;
    auto sync = [&]() __attribute__((always_inline)) {
        if constexpr (NW > 1) __syncthreads();
        else WaveSync()();
    };
    // row[q0..q0+8) of this lane to p
    auto put8 = [&](auto qc, T* p) __attribute__((always_inline)) {
        constexpr int q0 = decltype(qc)::value;
        static_for<0, CH / VN>([&](auto vc) __attribute__((always_inline)) {
            constexpr int q = decltype(vc)::value * VN;
            VT x;
            static_for<0, VN>([&](auto uc) __attribute__((always_inline)) {
                x[decltype(uc)::value] = row[q0 + q + decltype(uc)::value];
            });
            *reinterpret_cast<VT*>(p + q) = x;
        });
    };
    pos = t;
    bool used = t >= m;
    // the block in hand is row[0..CH): after block b row[c] is column
    // CH b + c while that is < N
    const int nblk = (jb + CH - 1) / CH;
    for (int b = 0; b < nblk; ++b) {
        const int left = jb - CH * b;                  // columns from here on
        int mult = used ? 0 : CH;      // multipliers of this row for the block's pivot rows
        bool mine = false;             // became pivot row `mult` of the block
        static_for<0, CH>([&](auto kc) __attribute__((always_inline)) {
            constexpr int kk = decltype(kc)::value, par = kk & 1;
            if (kk < left) {                           // uniform
                const int k = CH * b + kk;
                const unsigned hi = used ? 0u : mag_hi(row[kk]), lo = mag_lo(row[kk]);
                unsigned gm;
                const int wl = lanes_best<64, T>(hi, lo, pos, gm);
                // every lane's reciprocal, beside the search; the pivot row's
                // takes the place of the pivot in what it publishes
                const T rcp = T(1) / row[kk];
                if (lane == wl) {
                    if constexpr (NW > 1) L.key[par][w] = int4{(int)gm, (int)lo, pos, 0};
                    put8(std::integral_constant<int, 0>{}, &L.row[par][w][0]);
                    L.row[par][w][kk] = rcp;
                }
                int p, ww = w;
                sync();
                if constexpr (NW > 1) {
                    const int4 c = L.key[par][lane & 3];
                    ww = lanes_best<4, T>((unsigned)c.x, (unsigned)c.y, c.z, gm);
                    p = __builtin_amdgcn_readlane(c.z, ww);
                } else {
                    p = __builtin_amdgcn_readlane(pos, wl);
                }
                const bool zero = gm < mag_tiny<T>();          // TMV_Underflow
                if (zero) p = k;
                const T uv = L.row[par][ww][lane & (CH - 1)];  // the pivot row's block entries
                if (t == 0) L.piv[k] = (short)p;
                if (zero && first_zero == 0) first_zero = k + 1;
                if (zero && !used) row[kk] = T(0);
                const bool isp = !used && pos == p;
                if (!used && pos == k) pos = p;
                if (isp) { pos = k; rdiag = zero ? T(0) : rcp; mult = kk; mine = true; }
                used = used || isp;
                if (!zero) {
                    // unmasked (the broadcasts need every lane): pivot rows
                    // take multiplier 0
                    const T l = row[kk] * row_bcast<kk>(uv);
                    if (!used) row[kk] = l;
                    const T nl = used ? T(0) : -l;
                    static_for<kk + 1, CH>([&](auto c1) __attribute__((always_inline)) {
                        constexpr int c = decltype(c1)::value;
                        row[c] = fma(row_bcast<c>(uv), nl, row[c]);
                    });
                }
            }
        });
        if (left > CH) {
            // pivot rows to LDS, U12 = L11^-1 A12 a column per lane (one wave)
            if (mine)
                static_for<0, N / CH>([&](auto cc) __attribute__((always_inline)) {
                    constexpr int c0 = decltype(cc)::value * CH;
                    if (c0 < left) put8(std::integral_constant<int, c0>{}, &U[mult][c0]);
                });
            sync();
            if (w == 0 && lane >= CH && lane < left) {
                // (the offsets here and below pass through empty asm
                // statements: all reads at once would spill the row)
                T x[CH];
                int off = 0;
                static_for<0, CH>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    if constexpr (i > 1) __asm__ volatile("" : "+v"(off) : "v"(x[i - 2]));
                    x[i] = U[i][lane];
                    const T* ui = &U[i][0] + off;
                    static_for<0, i>([&](auto jc) __attribute__((always_inline)) {
                        constexpr int j = decltype(jc)::value;
                        x[i] = fma(-ui[j], x[j], x[i]);
                    });
                    if (i > 0) U[i][lane] = x[i];
                });
            }
            sync();
            // rank-8 update; a pivot row of this block takes the rows before
            // its own (which is its row of U12), earlier ones nothing
            T nl[CH];
            static_for<0, CH>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                nl[i] = i < mult ? -row[i] : T(0);
            });
            int off = lane & 15;
            static_for<0, N / 16>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value;
                if (16 * q < left) {
                    T uv[CH];
                    if constexpr (q > 0) __asm__ volatile("" : "+v"(off) : "v"(row[16 * q - 1]));
                    static_for<0, CH>([&](auto ic) __attribute__((always_inline)) {
                        uv[decltype(ic)::value] = U[decltype(ic)::value][16 * q + off];
                    });
                    static_for<0, 2>([&](auto hc) __attribute__((always_inline)) {
                        constexpr int c0 = 16 * q + CH * decltype(hc)::value;
                        if constexpr (c0 >= CH)
                            if (c0 < left)
                                static_for<0, CH>([&](auto ic) __attribute__((always_inline)) {
                                    constexpr int i = decltype(ic)::value;
                                    bcast_fma8<decltype(hc)::value, c0>(row, uv[i], nl[i]);
                                });
                    });
                }
            });
            sync();                    // U is rewritten by the next block
        }
        rotate_row(row);
    }
    for (int b = nblk; b < N / CH; ++b) rotate_row(row);   // back to column order
}

// Right-hand sides of a system whose factors are the rows of one wave
// (n <= N): L^-1 P B, then U^-1 of it unless the matrix is singular, NR
// columns at a time.
template <int NR, typename T, int N>
__device__ __forceinline__ void solve_rows(T (&row)[N], int n, int nr, T* __restrict__ B,
                                           i64 ldb, int lane, int pos, T rdiag, bool singular)
{
    constexpr int CH = BK_CH;
    const bool own = lane < n;
    const int nblk = (n + CH - 1) / CH;
    auto lane_at = [&](int k) __attribute__((always_inline)) {    // of pivot row k
        return (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(own && pos == k));
    };
    for (int c0 = 0; c0 < nr; c0 += NR) {
        T y[NR];
#pragma unroll
        for (int q = 0; q < NR; ++q) y[q] = (own && c0 + q < nr) ? B[lane + (c0 + q) * ldb] : T(0);
        for (int b = 0; b < nblk; ++b) {
            static_for<0, CH>([&](auto kc) __attribute__((always_inline)) {
                constexpr int kk = decltype(kc)::value;
                const int k = CH * b + kk;
                if (k < n) {                           // uniform
                    const int wk = lane_at(k);
                    T yk[NR];
#pragma unroll
                    for (int q = 0; q < NR; ++q) yk[q] = readlane(y[q], wk);
                    if (own && pos > k) {
#pragma unroll
                        for (int q = 0; q < NR; ++q) y[q] = fma(-row[kk], yk[q], y[q]);
                    }
                }
            });
            rotate_row(row);
        }
        for (int b = nblk - 1; b >= 0; --b) {
            rotate_row_back(row);
            if (singular) continue;
            static_for<0, CH>([&](auto kc) __attribute__((always_inline)) {
                constexpr int kk = CH - 1 - decltype(kc)::value;
                const int k = CH * b + kk;
                if (k < n) {
                    const int wk = lane_at(k);
                    const T rd = readlane(rdiag, wk);
                    T xk[NR];
#pragma unroll
                    for (int q = 0; q < NR; ++q) {
                        const T yk = readlane(y[q], wk);
                        xk[q] = yk == T(0) ? T(0) : yk * rd;
                        if (lane == wk) y[q] = xk[q];
                    }
                    if (own && pos < k) {
#pragma unroll
                        for (int q = 0; q < NR; ++q) y[q] = fma(-row[kk], xk[q], y[q]);
                    }
                }
            });
        }
        if (own) {
#pragma unroll
            for (int q = 0; q < NR; ++q)
                if (c0 + q < nr) B[pos + (c0 + q) * ldb] = y[q];
        }
    }
}

// The rows of A (leading dimension ld, m rows, jb columns) into registers and
// back to their positions.
template <typename T, int N>
__device__ __forceinline__ void load_row(T (&row)[N], const T* A, i64 ld, int m, int jb, int r)
{
#pragma unroll
    for (int c = 0; c < N; ++c) row[c] = (c < jb && r < m) ? A[r + c * ld] : T(0);
}
template <typename T, int N>
__device__ __forceinline__ void store_row(const T (&row)[N], T* A, i64 ld, int m, int jb, int r,
                                          int pos)
{
    if (r >= m) return;
#pragma unroll
    for (int c = 0; c < N; ++c)
        if (c < jb) A[pos + c * ld] = row[c];
}

// System slots[blockIdx.x], n <= N, one wave.  (No loop over systems: what a
// loop keeps in registers from one to the next is more than there are.)
template <typename T, int N>
__global__ void __launch_bounds__(64)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) * N >= 512 ? 2 : sizeof(T) * N >= 256 ? 4 : 5)))
batched_lu_wave_kernel(BatchArgs<T> args)
{
    __shared__ PanelLds<T, N, 1> L;
    const int lane = threadIdx.x;
    const int4 sys = args.slots[blockIdx.x];
    // (readfirstlane: sizes in scalar registers, or every bound below
    // would be a vector compare and an exec mask)
    const int idx = __builtin_amdgcn_readfirstlane(sys.x);
    const int n = __builtin_amdgcn_readfirstlane(sys.y);
    const int nr = __builtin_amdgcn_readfirstlane(sys.z);
    T* A = args.A[idx];
    i64* piv = args.piv[idx];
    T* B = args.B ? args.B[idx] : nullptr;
    T row[N];
    int pos = 0, first_zero = 0;
    T rdiag = T(0);
    load_row(row, A, (i64)n, n, n, lane);
    panel_rows<1>(row, n, n, lane, L, pos, rdiag, first_zero);
    store_row(row, A, (i64)n, n, n, lane, pos);
    for (int k = lane; k < n; k += 64) piv[k] = L.piv[k];
    if (lane == 0) args.info[idx] = first_zero;
    // (a last right-hand side by itself as one column: a quarter of the work;
    // one after the other, not one or the other, for which the compiler saved
    // the rows to memory first, with no right-hand side too)
    const int nr4 = (nr & 3) == 1 ? nr - 1 : nr;
    solve_rows<4>(row, n, nr4, B, (i64)n, lane, pos, rdiag, first_zero != 0);
    if (nr4 < nr)
        solve_rows<1>(row, n, 1, B + nr4 * (i64)n, (i64)n, lane, pos, rdiag, first_zero != 0);
}

// System slots[blockIdx.x], 64 < n <= 128, a workgroup of two waves.
template <typename T>
__global__ void __launch_bounds__(BK_NTH) __attribute__((amdgpu_waves_per_eu(2)))
batched_lu_group_kernel(BatchArgs<T> args)
{
    typedef typename Mfma<T>::v4 v4;
    __shared__ union {
        PanelLds<T, 64, 2> p;
        PanelLds<T, 64, 1> q;
        WgSolveLds<T, 1> w[BK_NW];
    } sh;
    __shared__ short s_piv[128], s_from[128];
    __shared__ int s_fz;
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int4 sys = args.slots[blockIdx.x];
    const int idx = __builtin_amdgcn_readfirstlane(sys.x);
    const int n = __builtin_amdgcn_readfirstlane(sys.y);
    const int nr = __builtin_amdgcn_readfirstlane(sys.z);
    const i64 ld = n;
    T* A = args.A[idx];
    i64* piv = args.piv[idx];
    int first_zero = 0;
    // the first 64 columns
    {
        T row[64];
        int pos = 0;
        T rdiag = T(0);
        if (t < 8) sh.p.key[t >> 2][t & 3] = int4{0, 0, INT_MAX, 0};   // (waves 2 and 3)
        __syncthreads();
        load_row(row, A, ld, n, 64, t);
        panel_rows<2>(row, n, 64, t, sh.p, pos, rdiag, first_zero);
        store_row(row, A, ld, n, 64, t, pos);
        __syncthreads();
        if (t < 64) s_piv[t] = sh.p.piv[t];
        if (t < n) s_from[pos] = (short)t;
        __syncthreads();
    }
    // the other columns, 16 at a time per wave; the right-hand sides are
    // one more such chunk
    T* B = args.B ? args.B[idx] : nullptr;
    const int nch = (n - 64 + 15) >> 4;
    for (int ch = w; ch < nch + (nr > 0 ? 1 : 0); ch += BK_NW) {
        WgSolveLds<T, 1>& S = sh.w[w];
        T* __restrict__ C = ch < nch ? A + (64 + 16 * ch) * ld : B;
        const int left = ch < nch ? n - 64 - 16 * ch : nr, nc = left < 16 ? left : 16;
        const int src = s_from[lane];
        static_for<0, 16>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            S.x[lane][c] = c < nc ? C[src + c * ld] : T(0);
        });
        WaveSync()();
        wg_trsv<T, 1, false, true, true>(64, A, n, S, lane, WaveSync());
        // A22's rows come from where the interchanges bring them from
        for (int r0 = 64; r0 < n; r0 += 16) {
            const int rr = r0 + li < n ? r0 + li : n - 1, fr = s_from[rr];
            v4 acc;                 // transposed: column row(g, q), row r0 + li
            T lf[16];
            static_for<0, 4>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value;
                const int c = Mfma<T>::row(g, q);
                acc[q] = C[fr + (c < nc ? c : nc - 1) * ld];
            });
            static_for<0, 16>([&](auto sc) __attribute__((always_inline)) {
                constexpr int s = decltype(sc)::value;
                lf[s] = -A[rr + (4 * s + g) * ld];
            });
            static_for<0, 16>([&](auto sc) __attribute__((always_inline)) {
                constexpr int s = decltype(sc)::value;
                acc = Mfma<T>::mac(S.x[4 * s + g][li], lf[s], acc);
            });
            static_for<0, 4>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value;
                const int c = Mfma<T>::row(g, q);
                if (r0 + li < n && c < nc) C[rr + c * ld] = acc[q];
            });
        }
        static_for<0, 16>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            if (c < nc) C[lane + c * ld] = S.x[lane][c];
        });
        WaveSync()();
    }
    __syncthreads();
    // A22 and its right-hand sides by the first wave, A22's interchanges
    // on L21 by both
    const int m = n - 64;
    if (w == 0) {
        T row[64];
        int pos = 0, fz = 0;
        T rdiag = T(0);
        T* A22 = A + 64 + 64 * ld;
        load_row(row, A22, ld, m, m, lane);
        panel_rows<1>(row, m, m, lane, sh.q, pos, rdiag, fz);
        store_row(row, A22, ld, m, m, lane, pos);
        if (lane < m) {
            s_piv[64 + lane] = (short)(64 + sh.q.piv[lane]);
            s_from[pos] = (short)lane;
        }
        if (first_zero == 0 && fz != 0) first_zero = 64 + fz;
        if (lane == 0) {
            args.info[idx] = first_zero;
            s_fz = first_zero;
        }
        if (nr > 0)
            solve_rows<4>(row, m, nr, B + 64, ld, lane, pos, rdiag, first_zero != 0);
    }
    __syncthreads();
    if (t < n) piv[t] = s_piv[t];
    {
        const int src = lane < m ? 64 + s_from[lane] : 0;
        T* ap = A + 32 * w * ld;
        T x[32];
#pragma unroll
        for (int c = 0; c < 32; ++c) x[c] = lane < m ? ap[src + c * ld] : T(0);
        if (lane < m) {
#pragma unroll
            for (int c = 0; c < 32; ++c) ap[64 + lane + c * ld] = x[c];
        }
    }
    // the first 64 unknowns: U11 x1 = y1 - U12 x2
    if (nr > 0 && s_fz == 0 && w == 0) {
        WgSolveLds<T, 1>& S = sh.w[0];
        v4 acc[4];
        static_for<0, 4>([&](auto tc) __attribute__((always_inline)) {
            static_for<0, 4>([&](auto qc) __attribute__((always_inline)) {
                constexpr int i = decltype(tc)::value, q = decltype(qc)::value;
                // (columns past the last read it and are not stored)
                acc[i][q] = B[16 * i + Mfma<T>::row(g, q) + (li < nr ? li : nr - 1) * ld];
            });
        });
        for (int k0 = 0; k0 < m; k0 += 4) {
            const int k = k0 + g < m ? k0 + g : m - 1;
            const T xk = k0 + g < m ? B[64 + k + (li < nr ? li : nr - 1) * ld] : T(0);
            static_for<0, 4>([&](auto tc) __attribute__((always_inline)) {
                constexpr int i = decltype(tc)::value;
                const T u = A[16 * i + li + (64 + k) * ld];
                acc[i] = Mfma<T>::mac(k0 + g < m ? -u : T(0), xk, acc[i]);
            });
        }
        static_for<0, 4>([&](auto tc) __attribute__((always_inline)) {
            static_for<0, 4>([&](auto qc) __attribute__((always_inline)) {
                constexpr int i = decltype(tc)::value, q = decltype(qc)::value;
                S.x[16 * i + Mfma<T>::row(g, q)][li] = acc[i][q];
            });
        });
        WaveSync()();
        wg_trsv<T, 1, false, false, false>(64, A, n, S, lane, WaveSync());
        static_for<0, 16>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            if (c < nr) B[lane + c * ld] = S.x[lane][c];
        });
    }
}

// ---------------------------------------------------------------------------
// Batched solve with stored factors: a workgroup (n <= 64: a wave) per
// system, or, for more than WS_WG_MAX systems, one wave per system.
// ---------------------------------------------------------------------------
template <typename T, bool TRANS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
batched_getrs_kernel(int count, const int* __restrict__ nv, const int* __restrict__ nrhsv,
                     const T* const* __restrict__ LUv, const i64* const* __restrict__ pivv,
                     T* const* Bv)
{
    __shared__ WgSolveShared<T> sh;
    wg_getrs_batch<T, TRANS>(count, nv, nrhsv, LUv, pivv, (const T* const*)Bv, Bv, sh);
}

template <typename T>
__global__ void __launch_bounds__(256)
batched_getrs_wave_kernel(int trans, int count, const int* __restrict__ nv,
                     const int* __restrict__ nrhsv, const T* const* __restrict__ LUv,
                     const i64* const* __restrict__ pivv, T* const* __restrict__ Bv)
{
    const int lane = threadIdx.x & 63;
    const int gw = (int)((blockIdx.x * (i64)blockDim.x + threadIdx.x) >> 6);
    const int nwaves = (int)((gridDim.x * (i64)blockDim.x) >> 6);
    for (int sys = gw; sys < count; sys += nwaves) {
        const int n = nv[sys], nr = nrhsv[sys];
        if (n < 0 || n > WS_NMAX) continue;
        for (int c = 0; c < nr; ++c) {
            T* b = Bv[sys] + (i64)c * n;
            T x[WS_PR];
            wave_load(x, b, n, lane);
            wave_getrs(trans, n, LUv[sys], (i64)n, pivv[sys], x, lane);
            wave_store(x, b, n, lane);
        }
    }
}

// ---------------------------------------------------------------------------
// Batched GEMM C_i = alpha A_i B_i + beta C_i (m_i x k_i times k_i x n_i,
// column-major, packed: lda = m, ldb = k, ldc = m), one workgroup for one or
// four problems (batched_gemm_group), each wave a 32 x 32 block of C on MFMA.  The k index inside an
// MFMA step is permuted (k = k0 + 4g + s) so a lane reads 4 consecutive k
// of its B column in one load, and the block's rows are dealt to the two MFMA
// row tiles in turn (tile t, index i: row r0 + 2 i + t), so a lane reads and
// writes two adjacent rows at a time.  Loads go BG_P steps of 16 k ahead; rows
// and columns past the edge are clamped (what they hold is not stored).
// Bound: the latency of a problem's first loads, and for the larger ones the
// loads themselves (A and B are read once per 32 columns or rows of C).
// ---------------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 2)))
batched_gemm_kernel(int count, int grp, const int* __restrict__ mv, const int* __restrict__ nv,
                    const int* __restrict__ kv, T alpha, const T* const* __restrict__ Av,
                    const T* const* __restrict__ Bv, T beta, T* const* __restrict__ Cv)
{
    typedef typename Mfma<T>::v4 v4;
    typedef T Pair __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    typedef T Quad __attribute__((ext_vector_type(4), aligned(sizeof(T))));
    constexpr int BG_P = 2;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, g = lane >> 4;
    // problem idx's blocks are dealt to the waves from wave idx mod grp on
    for (i64 id = (i64)blockIdx.x * grp, q0 = 0; id + q0 < count;) {
        const int idx = (int)(id + q0), rot = (int)q0;
        if (++q0 == grp) { q0 = 0; id += (i64)gridDim.x * grp; }
        const int M = __builtin_amdgcn_readfirstlane(mv[idx]);
        const int N = __builtin_amdgcn_readfirstlane(nv[idx]);
        const int K = __builtin_amdgcn_readfirstlane(kv[idx]);
        const T* A = Av[idx];
        const T* B = Bv[idx];
        T* C = Cv[idx];
        const int nbm = (M + 31) / 32, nbn = (N + 31) / 32;
        // 16 k at a time; a single row has no pairs and takes its k by entry
        const int nfull = M >= 2 ? K / 16 : 0;
        for (int blk = (wave - rot) & 3; blk < nbm * nbn; blk += 4) {
            const int r0 = (blk % nbm) * 32, c0 = (blk / nbm) * 32;
            const int r = r0 + 2 * li;
            const int rp = r < M - 2 ? r : M >= 2 ? M - 2 : 0;     // the pair read
            const bool hi = r > rp;                 // row M - 1 alone: the pair's second
            const T* pa = A + rp + (i64)(4 * g) * M;
            const T* pb[2];
            static_for<0, 2>([&](auto tc) __attribute__((always_inline)) {
                constexpr int t = decltype(tc)::value;
                const int c = c0 + 16 * t + li;
                pb[t] = B + 4 * g + (i64)(c < N ? c : N - 1) * K;
            });
            v4 acc[2][2];
            static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                    acc[decltype(ic)::value][decltype(jc)::value] = v4{0, 0, 0, 0};
                });
            });
            Pair fa[BG_P][4];
            Quad fb[BG_P][2];
            auto load = [&](auto qc, int st) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value;
                static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    fa[q][s] = *reinterpret_cast<const Pair*>(pa + (i64)(16 * st + s) * M);
                });
                static_for<0, 2>([&](auto tc) __attribute__((always_inline)) {
                    constexpr int t = decltype(tc)::value;
                    fb[q][t] = *reinterpret_cast<const Quad*>(pb[t] + 16 * st);
                });
            };
            auto step = [&](const T (&a)[2][4], const T (&b)[2][4]) __attribute__((always_inline)) {
                static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    static_for<0, 2>([&](auto ic) __attribute__((always_inline)) {
                        constexpr int i = decltype(ic)::value;
                        static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                            constexpr int j = decltype(jc)::value;
                            acc[i][j] = Mfma<T>::mac(a[i][s], b[j][s], acc[i][j]);
                        });
                    });
                });
            };
            static_for<0, BG_P>([&](auto qc) __attribute__((always_inline)) {
                if (decltype(qc)::value < nfull) load(qc, decltype(qc)::value);
            });
            for (int kt = 0; kt < nfull; kt += BG_P)
                static_for<0, BG_P>([&](auto qc) __attribute__((always_inline)) {
                    constexpr int q = decltype(qc)::value;
                    if (kt + q >= nfull) return;                      // uniform
                    T a[2][4], b[2][4];
                    static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
                        constexpr int s = decltype(sc)::value;
                        a[0][s] = hi ? fa[q][s][1] : fa[q][s][0];
                        a[1][s] = fa[q][s][1];
                        b[0][s] = fb[q][0][s];
                        b[1][s] = fb[q][1][s];
                    });
                    if (kt + q + BG_P < nfull) load(qc, kt + q + BG_P);
                    step(a, b);
                });
            for (int k0 = 16 * nfull; k0 < K; k0 += 16) {             // K's remainder
                T a[2][4], b[2][4];
                static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    const int k = k0 + 4 * g + s;
                    static_for<0, 2>([&](auto tc) __attribute__((always_inline)) {
                        constexpr int t = decltype(tc)::value;
                        a[t][s] = (k < K && r + t < M) ? A[r + t + (i64)k * M] : T(0);
                        b[t][s] = k < K ? pb[t][k0 + s] : T(0);
                    });
                });
                step(a, b);
            }
            static_for<0, 2>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                const int c = c0 + 16 * j + li;
                static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
                    constexpr int q = decltype(rc)::value;
                    const int row = r0 + 2 * Mfma<T>::row(g, q);
                    if (row >= M || c >= N) return;
                    T* p = C + row + (i64)c * M;
                    const T v0 = alpha * acc[0][j][q], v1 = alpha * acc[1][j][q];
                    if (row + 1 < M) {
                        Pair* pp = reinterpret_cast<Pair*>(p);
                        Pair v = {v0, v1};
                        if (beta != T(0)) v += beta * *pp;
                        *pp = v;
                    } else {
                        *p = beta == T(0) ? v0 : v0 + beta * *p;
                    }
                });
            });
        }
    }
}

// Problems a workgroup: with enough of them to fill the chip, four, so that
// problems of one block (n <= 32) leave no wave idle; with fewer, one, so that
// the larger ones still spread over the CUs.  One a workgroup -> four (us):
//   FP64: 8191 of n = 1 27 -> 14, of n = 16 32 -> 18, of n = 32 46 -> 38;
//         4000 of n = 8 15 -> 10, of n = 128 500 -> 497; 2048 of n = 1 10.0 ->
//         9.6, of n = 100 218 -> 220; 1500 of n = 128 201 -> 244
//   FP32 (three workgroups a CU, not two): 8191 of n = 1 14 -> 10, of n = 128
//         565 -> 579; 6000 of n = 8 12.4 -> 9.8; 3000 of n = 8 8.5 -> 8.3, of
//         n = 100 197 -> 206
// Measured, one workgroup a problem with entry loads before: 20,000 of 8..128
// FP32 1.73 -> 0.82 ms; 4000 of n = 128 FP64 722 -> 497 us, FP32 615 -> 286.
template <typename T> static int batched_gemm_group(int64_t count)
{
    return count >= (sizeof(T) == 8 ? 2048 : 4096) ? 4 : 1;
}

// ---------------------------------------------------------------------------
// Host side: plans.
// ---------------------------------------------------------------------------

// One way of running a batch is left, a wave per system of n <= 64 (what a
// wave's registers hold) and a workgroup per larger one; the grid is the work
// list, largest first, so that it balances itself.  Measured, 20,000 systems
// of 8..128 with 1-4 right-hand sides, FP64: 6.80 ms with a 16 x 16 thread
// grid per system and two barriers a column -> 2.05 ms (n > 64 1.80, n <= 64
// 0.20, n <= 32 0.05); 10,000 of n = 64 3.09 -> 0.29 ms (FP32 2.85 -> 0.15),
// of n = 32 0.25 -> 0.10, of n = 128 6.24 -> 1.88.  A schedule that a caller
// forces (one of three, by the largest order that it gave to a wave) is
// checked and recorded, and changes nothing else.
constexpr int kSplitMax[] = {16, 32, 64};
constexpr int kNumSchedules = 3;
constexpr int kWaveRhsMax = 8;      // right-hand sides a forced split admits per wave

} // namespace tmvx

struct tmvx_batch_plan_s {
    int dtype = 0;
    int64_t count = 0;
    int ngroup = 0, nwave64 = 0;        // systems of a workgroup; of a wave, n > 32
    std::vector<int> h_n, h_nrhs;
    int* d_n = nullptr;
    int4* d_slots = nullptr;
    char desc[256] = {0};
};

namespace tmvx {

// The plan's text, with what was timed or forced.
static void plan_text(tmvx_batch_plan_s* p, const char* more)
{
    snprintf(p->desc, sizeof(p->desc), "n<=64 a wave, n<=128 a workgroup: %d + %d + %d systems%s",
             p->ngroup, p->nwave64, (int)p->count - p->ngroup - p->nwave64, more);
}

// Build the work list, largest first: systems with n <= 64 take a wave each,
// the rest a workgroup each.
static int plan_build(tmvx_batch_plan_s* p, hipStream_t s)
{
    const int64_t cnt = p->count;
    std::vector<int> order((size_t)cnt);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int b) { return p->h_n[a] > p->h_n[b]; });
    std::vector<int4> slots((size_t)cnt);
    for (int64_t i = 0; i < cnt; ++i) {
        const int k = order[i], n = p->h_n[k];
        slots[i] = int4{k, n, p->h_nrhs[k], 0};
        if (n > 64) ++p->ngroup;
        else if (n > 32) ++p->nwave64;
    }
    if (cnt > 0)
        TMVX_HIP(hipMemcpyAsync(p->d_slots, slots.data(), sizeof(int4) * (size_t)cnt,
                                hipMemcpyHostToDevice, s));
    TMVX_HIP(hipStreamSynchronize(s));
    plan_text(p, "");
    return TMVX_OK;
}

template <typename T>
static int batch_launch(const tmvx_batch_plan_s* p, T* const* A, i64* const* piv, T* const* B,
                        int* info, hipStream_t s)
{
    if (p->count == 0) return TMVX_OK;
    BatchArgs<T> args;
    args.A = A;
    args.piv = piv;
    args.B = B;
    args.info = info;
    // the largest systems first; a launch per form that has systems, a
    // workgroup per system (the hardware deals them out as they finish)
    const int g = p->ngroup, w64 = p->nwave64, w32 = (int)p->count - g - w64;
    args.slots = p->d_slots;
    if (g > 0)
        hipLaunchKernelGGL(batched_lu_group_kernel<T>, dim3((unsigned)g), dim3(BK_NTH), 0, s, args);
    args.slots += g;
    if (w64 > 0)
        hipLaunchKernelGGL((batched_lu_wave_kernel<T, 64>), dim3((unsigned)w64), dim3(64), 0, s,
                           args);
    args.slots += w64;
    if (w32 > 0)
        hipLaunchKernelGGL((batched_lu_wave_kernel<T, 32>), dim3((unsigned)w32), dim3(64), 0, s,
                           args);
    return hip_status(hipGetLastError());
}

// Synthetic batch of the plan's shape (uniform[-1,1] + n I, B uniform) for
// timing the plan.
__global__ void batch_diag_shift_kernel(int count, const int* nv, double* const* A64,
                                        float* const* A32)
{
    const int idx = blockIdx.x;
    if (idx >= count) return;
    const int n = nv[idx];
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        if (A64) A64[idx][i + (i64)i * n] += (double)n;
        if (A32) A32[idx][i + (i64)i * n] += (float)n;
    }
}
__global__ void f64_to_f32_kernel(i64 cnt, const double* in, float* out)
{
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < cnt) out[i] = (float)in[i];
}

static int plan_time(tmvx_batch_plan_s* p, hipStream_t s)
{
    const int64_t cnt = p->count;
    std::vector<i64> offA((size_t)cnt), offB((size_t)cnt), offP((size_t)cnt);
    i64 ta = 0, tb = 0, tp = 0;
    for (int64_t i = 0; i < cnt; ++i) {
        offA[i] = ta; ta += (i64)p->h_n[i] * p->h_n[i];
        offB[i] = tb; tb += (i64)p->h_n[i] * p->h_nrhs[i];
        offP[i] = tp; tp += p->h_n[i];
    }
    const size_t esz = p->dtype == 0 ? 8 : 4;
    const i64 ta1 = ta > 0 ? ta : 1, tb1 = tb > 0 ? tb : 1, tp1 = tp > 0 ? tp : 1;
    char *dA0 = nullptr, *dA = nullptr, *dB0 = nullptr, *dB = nullptr;
    i64* dP = nullptr;
    void** dptr = nullptr;        // [A | B | piv | A0] pointer arrays
    int* dinfo = nullptr;
    double* stage = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = TMVX_OK;
    if (hipMalloc((void**)&dA0, esz * ta1) != hipSuccess ||
        hipMalloc((void**)&dA, esz * ta1) != hipSuccess ||
        hipMalloc((void**)&dB0, esz * tb1) != hipSuccess ||
        hipMalloc((void**)&dB, esz * tb1) != hipSuccess ||
        hipMalloc((void**)&dP, sizeof(i64) * tp1) != hipSuccess ||
        hipMalloc((void**)&dptr, sizeof(void*) * 4 * cnt) != hipSuccess ||
        hipMalloc((void**)&dinfo, sizeof(int) * cnt) != hipSuccess ||
        hipMalloc((void**)&stage, sizeof(double) * std::max(ta1, tb1)) != hipSuccess)
        rc = TMVX_ERR_ALLOC;
    if (rc == TMVX_OK && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess))
        rc = TMVX_ERR_HIP;
    if (rc == TMVX_OK) {
        std::vector<void*> hp((size_t)(4 * cnt));
        for (int64_t i = 0; i < cnt; ++i) {
            hp[i] = dA + esz * offA[i];
            hp[cnt + i] = dB + esz * offB[i];
            hp[2 * cnt + i] = dP + offP[i];
            hp[3 * cnt + i] = dA0 + esz * offA[i];
        }
        if (hipMemcpy(dptr, hp.data(), sizeof(void*) * 4 * cnt, hipMemcpyHostToDevice) !=
            hipSuccess)
            rc = TMVX_ERR_HIP;
    }
    // Synthetic batch: uniform[-1,1] from a fixed seed, + n on the diagonal.
    auto fill = [&](uint64_t seed, i64 count, char* dst) -> int {
        if (count == 0) return TMVX_OK;
        double* tgt = p->dtype == 0 ? (double*)dst : stage;
        TMVX_TRY(tmvx_fill_uniform_f64(seed, 0, count, -1.0, 1.0, tgt, s));
        if (p->dtype == 1)
            hipLaunchKernelGGL(f64_to_f32_kernel, dim3((unsigned)((count + 255) / 256)),
                               dim3(256), 0, s, count, (const double*)stage, (float*)dst);
        return hip_status(hipGetLastError());
    };
    if (rc == TMVX_OK) rc = fill(0x7A15EED, ta, dA0);
    if (rc == TMVX_OK) rc = fill(0x7A15EEE, tb, dB0);
    if (rc == TMVX_OK && cnt > 0) {
        hipLaunchKernelGGL(batch_diag_shift_kernel, dim3((unsigned)cnt), dim3(128), 0, s,
                           (int)cnt, (const int*)p->d_n,
                           p->dtype == 0 ? (double* const*)(dptr + 3 * cnt) : nullptr,
                           p->dtype == 1 ? (float* const*)(dptr + 3 * cnt) : nullptr);
        rc = hip_status(hipGetLastError());
    }
    float best = 1e30f;
    for (int rep = 0; rep < 3 && rc == TMVX_OK; ++rep) {       // rep 0 warms up
        if (hipMemcpyAsync(dA, dA0, esz * ta, hipMemcpyDeviceToDevice, s) != hipSuccess ||
            hipMemcpyAsync(dB, dB0, esz * tb, hipMemcpyDeviceToDevice, s) != hipSuccess) {
            rc = TMVX_ERR_HIP;
            break;
        }
        hipEventRecord(e0, s);
        if (p->dtype == 0)
            rc = batch_launch<double>(p, (double* const*)dptr, (i64* const*)(dptr + 2 * cnt),
                                      (double* const*)(dptr + cnt), dinfo, s);
        else
            rc = batch_launch<float>(p, (float* const*)dptr, (i64* const*)(dptr + 2 * cnt),
                                     (float* const*)(dptr + cnt), dinfo, s);
        hipEventRecord(e1, s);
        if (hipEventSynchronize(e1) != hipSuccess) { rc = TMVX_ERR_HIP; break; }
        float ms = 0;
        hipEventElapsedTime(&ms, e0, e1);
        if (rep > 0) best = std::min(best, ms);
    }
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    hipFree(dA0); hipFree(dA); hipFree(dB0); hipFree(dB); hipFree(dP); hipFree(dptr);
    hipFree(dinfo); hipFree(stage);
    if (rc != TMVX_OK) return rc;
    char more[64];
    snprintf(more, sizeof(more), "; autotuned (one schedule): %.3f ms", best);
    plan_text(p, more);
    return TMVX_OK;
}

} // namespace tmvx

using namespace tmvx;

extern "C" {

int tmvx_batch_plan_create(int dtype, int64_t count, const int32_t* n_host,
                           const int32_t* nrhs_host, int tune, tmvx_batch_plan* plan,
                           void* stream)
{
    if (!plan) return TMVX_ERR_ARG;
    *plan = nullptr;
    if ((dtype != TMVX_BATCH_F64 && dtype != TMVX_BATCH_F32) || count < 0 || count > INT_MAX ||
        (count > 0 && !n_host))
        return TMVX_ERR_ARG;
    int maxn = 0, maxr = 0;
    for (int64_t i = 0; i < count; ++i) {
        const int ni = n_host[i], ri = nrhs_host ? nrhs_host[i] : 0;
        if (ni < 0 || ri < 0) return TMVX_ERR_ARG;
        maxn = std::max(maxn, ni);
        maxr = std::max(maxr, ri);
    }
    if (maxn > TMVX_BATCH_NMAX || maxr > TMVX_BATCH_RHSMAX) return TMVX_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    tmvx_batch_plan_s* p = new (std::nothrow) tmvx_batch_plan_s();
    if (!p) return TMVX_ERR_ALLOC;
    p->dtype = dtype;
    p->count = count;
    p->h_n.assign(n_host, n_host + count);
    p->h_nrhs.assign((size_t)count, 0);
    if (nrhs_host) p->h_nrhs.assign(nrhs_host, nrhs_host + count);
    const size_t c1 = (size_t)std::max<int64_t>(count, 1);
    int rc = TMVX_OK;
    if (hipMalloc((void**)&p->d_n, sizeof(int) * c1) != hipSuccess ||
        hipMalloc((void**)&p->d_slots, sizeof(int4) * c1) != hipSuccess)
        rc = TMVX_ERR_ALLOC;
    if (rc == TMVX_OK && count > 0 &&
        hipMemcpyAsync(p->d_n, p->h_n.data(), sizeof(int) * count, hipMemcpyHostToDevice, s) !=
            hipSuccess)
        rc = TMVX_ERR_HIP;
    if (rc == TMVX_OK) rc = plan_build(p, s);
    if (rc == TMVX_OK && tune && count > 0) rc = plan_time(p, s);
    if (rc != TMVX_OK) {
        tmvx_batch_plan_destroy(p);
        return rc;
    }
    *plan = p;
    return TMVX_OK;
}

int tmvx_batch_plan_destroy(tmvx_batch_plan p)
{
    if (!p) return TMVX_OK;
    hipFree(p->d_n);
    hipFree(p->d_slots);
    delete p;
    return TMVX_OK;
}

const char* tmvx_batch_plan_describe(tmvx_batch_plan p)
{
    return p ? p->desc : "";
}

int tmvx_batch_plan_set(tmvx_batch_plan p, int schedule, int split, int wgs_per_cu, void*)
{
    if (!p || schedule < 0 || schedule >= kNumSchedules || split < 0 || wgs_per_cu < 1 ||
        wgs_per_cu > 16)
        return TMVX_ERR_ARG;
    const int sp = std::min(split, kSplitMax[schedule]);
    for (int64_t i = 0; i < p->count; ++i)
        if (p->h_n[i] <= sp && p->h_nrhs[i] > kWaveRhsMax) return TMVX_ERR_UNSUPPORTED;
    char more[80];
    snprintf(more, sizeof(more), "; forced (no effect): schedule %d, split %d, %d/CU", schedule, sp,
             wgs_per_cu);
    plan_text(p, more);
    return TMVX_OK;
}

int tmvx_batch_schedule_count(void) { return kNumSchedules; }

int tmvx_gesv_batched_f64(tmvx_batch_plan p, double* const* A, int64_t* const* piv,
                          double* const* B, int32_t* info, void* stream)
{
    if (!p || p->dtype != TMVX_BATCH_F64) return TMVX_ERR_ARG;
    if (p->count > 0 && (!A || !piv || !info)) return TMVX_ERR_ARG;
    return batch_launch<double>(p, A, (i64* const*)piv, B, info, (hipStream_t)stream);
}

int tmvx_gesv_batched_f32(tmvx_batch_plan p, float* const* A, int64_t* const* piv,
                          float* const* B, int32_t* info, void* stream)
{
    if (!p || p->dtype != TMVX_BATCH_F32) return TMVX_ERR_ARG;
    if (p->count > 0 && (!A || !piv || !info)) return TMVX_ERR_ARG;
    return batch_launch<float>(p, A, (i64* const*)piv, B, info, (hipStream_t)stream);
}

extern "C++" template <typename T>
static int getrs_batched_launch(int trans, int64_t count, const int32_t* n, const int32_t* nrhs,
                                const T* const* LU, const int64_t* const* piv, T* const* B,
                                hipStream_t s)
{
    if (count < 0 || count > INT_MAX) return TMVX_ERR_ARG;
    if (count == 0) return TMVX_OK;
    if (!n || !nrhs || !LU || !piv || !B) return TMVX_ERR_ARG;
    const dim3 grid((unsigned)std::min<int64_t>(count, 2048)), block(256);
    if (count > WS_WG_MAX)           // 8192 waves; wave w takes systems w, w + 8192, ...
        hipLaunchKernelGGL(batched_getrs_wave_kernel<T>, dim3(2048), block, 0, s, trans,
                           (int)count, n, nrhs, LU, (const i64* const*)piv, B);
    else if (trans)
        hipLaunchKernelGGL((batched_getrs_kernel<T, true>), grid, block, 0, s, (int)count, n, nrhs,
                           LU, (const i64* const*)piv, B);
    else
        hipLaunchKernelGGL((batched_getrs_kernel<T, false>), grid, block, 0, s, (int)count, n, nrhs,
                           LU, (const i64* const*)piv, B);
    return hip_status(hipGetLastError());
}

int tmvx_getrs_batched_f64(int trans, int64_t count, const int32_t* n, const int32_t* nrhs,
                           const double* const* LU, const int64_t* const* piv, double* const* B,
                           void* stream)
{
    return getrs_batched_launch<double>(trans, count, n, nrhs, LU, piv, B, (hipStream_t)stream);
}

int tmvx_getrs_batched_f32(int trans, int64_t count, const int32_t* n, const int32_t* nrhs,
                           const float* const* LU, const int64_t* const* piv, float* const* B,
                           void* stream)
{
    return getrs_batched_launch<float>(trans, count, n, nrhs, LU, piv, B, (hipStream_t)stream);
}

int tmvx_gemm_batched_f64(int64_t count, const int32_t* m, const int32_t* n, const int32_t* k,
                          double alpha, const double* const* A, const double* const* B,
                          double beta, double* const* C, void* stream)
{
    if (count < 0 || count > INT_MAX) return TMVX_ERR_ARG;
    if (count == 0) return TMVX_OK;
    if (!m || !n || !k || !A || !B || !C) return TMVX_ERR_ARG;
    const int grp = batched_gemm_group<double>(count);
    const unsigned grid = (unsigned)std::min<int64_t>((count + grp - 1) / grp, 1 << 20);
    hipLaunchKernelGGL(batched_gemm_kernel<double>, dim3(grid), dim3(256), 0,
                       (hipStream_t)stream, (int)count, grp, m, n, k, alpha, A, B, beta, C);
    return hip_status(hipGetLastError());
}

int tmvx_gemm_batched_f32(int64_t count, const int32_t* m, const int32_t* n, const int32_t* k,
                          float alpha, const float* const* A, const float* const* B, float beta,
                          float* const* C, void* stream)
{
    if (count < 0 || count > INT_MAX) return TMVX_ERR_ARG;
    if (count == 0) return TMVX_OK;
    if (!m || !n || !k || !A || !B || !C) return TMVX_ERR_ARG;
    const int grp = batched_gemm_group<float>(count);
    const unsigned grid = (unsigned)std::min<int64_t>((count + grp - 1) / grp, 1 << 20);
    hipLaunchKernelGGL(batched_gemm_kernel<float>, dim3(grid), dim3(256), 0,
                       (hipStream_t)stream, (int)count, grp, m, n, k, alpha, A, B, beta, C);
    return hip_status(hipGetLastError());
}

} // extern "C"
