// Solves with stored LU factors of one small system (n <= WS_NMAX), by one
// workgroup or one wave, up to 16 right-hand sides at a time, for batches
// that leave the GPU short of waves.  Shared by the batched solve and the
// adjoint.
//
// A X = B: rows gathered through the interchange list, then unit-lower L and
// U (TMV LU_LDivEq, src/TMV_LUDiv.cpp:185-226).  A^T X = B: U^T, then L^T,
// then the rows scattered back (TMV LU_RDivEq on B^T, src/TMV_LUDiv.cpp:
// 369-410).  Entries are divided by U's diagonal, a zero entry stays zero
// (src/TMV_TriDiv_V.cpp:187).
//
// The triangle is walked in blocks of 16 rows.  The sums of products that the
// rows to come will take off their right-hand sides are MFMA accumulators (16
// rows x 16 right-hand sides each, the 16-row blocks dealt out to the waves);
// a solved block's product with the rows to come is one 16x16x16 MFMA step per
// block row, with the factor entries loaded a block ahead.  The diagonal block
// itself is a plain substitution, a right-hand side per lane, its entries
// broadcast from LDS.  A row's products are summed apart from its right-hand
// side and subtracted once: taken off one after another, each would be rounded
// at the size of the right-hand side (A^T X = B, n = 256, A uniform + n I:
// error 3.4 eps so, 0.36 eps apart, as the wave form's dot products), and each
// block's sum is formed by itself before it joins that of the blocks before.
// One barrier per block: the chain is 16 substitution steps per block
// instead of a wave-wide sweep (or a wave sum, for A^T) per row, and four
// waves stream the factors of one system.
#pragma once
#include "tmvx_wave_solve.h"

namespace tmvx {

// Batches of up to this many systems take the workgroup form; larger ones
// fill the GPU with a wave per system (tmvx_wave_solve.h), which keeps eight
// systems in flight where this form, by its LDS and registers, keeps two.
// Wave form -> workgroup form, FP64, transposed, one right-hand side (us):
//   512 systems:  n = 64 72 -> 42, n = 128 137 -> 63, n = 256 274 -> 145
//   640:          n = 64 73 -> 42, n = 128 138 -> 101, n = 256 278 -> 265
//   1024:         n = 64 73 -> 43, n = 128 138 -> 114, n = 200 220 -> 208,
//                 n = 256 281 -> 295 (four right-hand sides 1081 -> 301)
// and, untransposed, 2000 of n = 128 97 -> 224, 4000 of n = 65 91 -> 234.
constexpr int WS_WG_MAX = 1024;

constexpr int WS_RHS = 16;                 // right-hand sides per pass
constexpr int WS_TPW = 4;                  // 16-row blocks per wave

struct GroupSync {
    __device__ __forceinline__ void operator()() const { __syncthreads(); }
};
// Between the lanes of one wave: its LDS and memory accesses are in order, so
// only the compiler is held back.
struct WaveSync {
    __device__ __forceinline__ void operator()() const
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

// LDS of one system solved by NWV waves (n <= 64 NWV).
template <typename T, int NWV>
struct WgSolveLds {
    static constexpr int NMAX = 16 * WS_TPW * NWV;
    T x[NMAX][WS_RHS];
    T d[NMAX / 16][16][16];                // d[b][k][i] = op(A)(16 b + i, 16 b + k)
    T s[16][WS_RHS];                       // the next block's sums of products
    short src[NMAX];                       // row i of P A is row src[i] of A
    short piv[NMAX];
    int bad;                               // right-hand sides whose solution holds a NaN
};

// One triangular solve on L.x (rows past n are zero), A with leading
// dimension ld.  LOWER: op(A) is lower triangular (walked forward).
template <typename T, int NWV, bool TRANS, bool LOWER, bool UNIT, class Sync>
__device__ __forceinline__ void wg_trsv(int n, const T* __restrict__ A, int ld,
                                        WgSolveLds<T, NWV>& L, int tid, Sync sync)
{
    typedef typename Mfma<T>::v4 v4;
    const int lane = tid & 63, wave = NWV == 1 ? 0 : tid >> 6, li = lane & 15, g = lane >> 4;
    const int nb = (n + 15) >> 4;
    for (int e = tid; e < nb * 256; e += 64 * NWV) {
        const int b = e >> 8, i = 16 * b + (TRANS ? (e >> 4) & 15 : e & 15);
        const int k = 16 * b + (TRANS ? e & 15 : (e >> 4) & 15);
        L.d[b][k & 15][i & 15] = (i < n && k < n) ? (TRANS ? A[k + i * ld] : A[i + k * ld])
                                                  : (i == k ? T(1) : T(0));
    }
    for (int e = tid; e < 16 * WS_RHS; e += 64 * NWV) L.s[e / WS_RHS][e % WS_RHS] = T(0);
    // op(A)(16 tb + li, 16 b + k(s, g)), the MFMA k slot (s, g) holding
    // k = 4 s + g, or 4 g + s where k is the contiguous index of A
    auto frag = [&](int tb, int b, T (&f)[4]) __attribute__((always_inline)) {
        const int r = 16 * tb + li, rc = r < n ? r : n - 1;
        static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value;
            const int k = 16 * b + (TRANS ? 4 * g + s : 4 * s + g), kc = k < n ? k : n - 1;
            const T v = TRANS ? A[kc + rc * ld] : A[rc + kc * ld];
            f[s] = (r < n && k < n) ? v : T(0);
        });
    };
    auto later = [&](int tb, int b) __attribute__((always_inline)) {
        return LOWER ? (tb > b && tb < nb) : tb < b;
    };
    v4 acc[WS_TPW];
    T f[WS_TPW][4];
    const int first = LOWER ? 0 : nb - 1;
    static_for<0, WS_TPW>([&](auto tc) __attribute__((always_inline)) {
        constexpr int t = decltype(tc)::value;
        const int tb = wave + NWV * t;
        static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
            constexpr int r = decltype(rc)::value;
            acc[t][r] = T(0);
        });
        if (later(tb, first)) frag(tb, first, f[t]);
    });
    sync();                                   // L.d and L.s complete
    for (int q = 0; q < nb; ++q) {
        const int b = LOWER ? q : nb - 1 - q, bn = LOWER ? b + 1 : b - 1;
        if (NWV == 1 || wave == b % NWV) {
            // the block through LDS to one right-hand side per lane (every lane
            // group solves the same 16); x[k] is the sum of the block's own
            // products of row k, then its solution
            T x[16];
            static_for<0, 16>([&](auto kc) __attribute__((always_inline)) { x[decltype(kc)::value] = T(0); });
            // column k of the diagonal block, row k's right-hand side and its
            // sum so far are read one step before their use (the offset passes
            // through an empty asm statement with the previous entry, or all
            // the reads would be hoisted to the top)
            T d[16], bk = L.x[16 * b + (LOWER ? 0 : 15)][li], sk = L.s[LOWER ? 0 : 15][li];
            int off = 0;
            auto dcol = [&](auto kc, T (&c)[16]) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                static_for<0, 16>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    if constexpr ((LOWER ? i > k : i < k) || (!UNIT && i == k)) c[i] = (&L.d[b][k][i])[off];
                });
            };
            dcol(std::integral_constant<int, LOWER ? 0 : 15>{}, d);
            static_for<0, 16>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value, k = LOWER ? q : 15 - q;
                T dn[16], bn = T(0), sn = T(0);
                if constexpr (q > 0) __asm__ volatile("" : "+v"(off) : "v"(x[k]));
                if constexpr (q < 15) {
                    dcol(std::integral_constant<int, LOWER ? k + 1 : k - 1>{}, dn);
                    bn = (&L.x[16 * b + (LOWER ? k + 1 : k - 1)][li])[off];
                    sn = (&L.s[LOWER ? k + 1 : k - 1][li])[off];
                }
                x[k] = bk - (sk + x[k]);
                if constexpr (!UNIT) x[k] = x[k] == T(0) ? T(0) : x[k] / d[k];
                static_for<0, 16>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    if constexpr (LOWER ? i > k : i < k) x[i] = fma(d[i], x[k], x[i]);
                    if constexpr (q < 15) d[i] = dn[i];
                });
                bk = bn;
                sk = sn;
            });
            if (g == 0)
                static_for<0, 16>([&](auto kc) __attribute__((always_inline)) {
                    constexpr int k = decltype(kc)::value;
                    // (rows past n stay zero: the next sweep starts from them, and
                    // an Inf or NaN there would reach every row)
                    L.x[16 * b + k][li] = 16 * b + k < n ? x[k] : T(0);
                });
        }
        sync();
        if (bn < 0 || bn >= nb) break;
        // the next block first: its owner goes on with it
        T xb[4];
        static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
            constexpr int s = decltype(sc)::value;
            xb[s] = L.x[16 * b + (TRANS ? 4 * g + s : 4 * s + g)][li];
        });
        static_for<0, 2>([&](auto pc) __attribute__((always_inline)) {
            static_for<0, WS_TPW>([&](auto tc) __attribute__((always_inline)) {
                constexpr int t = decltype(tc)::value;
                const int tb = wave + NWV * t;
                if ((tb == bn) != (decltype(pc)::value == 0) || !later(tb, b)) return;   // uniform
                v4 p = {T(0), T(0), T(0), T(0)};
                static_for<0, 4>([&](auto sc) __attribute__((always_inline)) {
                    constexpr int s = decltype(sc)::value;
                    p = Mfma<T>::mac(f[t][s], xb[s], p);
                });
                acc[t] += p;
                if constexpr (decltype(pc)::value == 0)
                    static_for<0, 4>([&](auto rc) __attribute__((always_inline)) {
                        constexpr int r = decltype(rc)::value;
                        L.s[Mfma<T>::row(g, r)][li] = acc[t][r];
                    });
            });
        });
        static_for<0, WS_TPW>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value;
            const int tb = wave + NWV * t;
            if (later(tb, bn)) frag(tb, bn, f[t]);       // in flight during the next block
        });
        WaveSync()();                         // the owner's sums are in LDS for its own reads
    }
}

// Column c of L.x := U^-1 L^-1 P b by one wave, a column of LU at a time.
template <typename T, int NWV>
__device__ __forceinline__ void plain_getrs(int n, const T* __restrict__ LU, const T* b,
                                            WgSolveLds<T, NWV>& L, int c, int lane)
{
#pragma clang loop unroll(disable)
    for (int i = lane; i < n; i += 64) L.x[i][c] = b[(int)L.src[i]];
    WaveSync()();
#pragma clang loop unroll(disable)
    for (int q = 0; q < 2 * n; ++q) {
        const bool low = q < n;                    // L forward, then U backward
        const int k = low ? q : 2 * n - 1 - q;
        T x = L.x[k][c];
        if (!low && x != T(0)) {
            x = x / LU[k + k * n];
            L.x[k][c] = x;
        }
        if (x != T(0)) {
#pragma clang loop unroll(disable)
            for (int i = low ? k + 1 + lane : lane; i < (low ? n : k); i += 64)
                L.x[i][c] -= LU[i + k * n] * x;
        }
        WaveSync()();
    }
}

// X := A^-1 B (A^-T B) for nr right-hand sides, B and X n x nr with leading
// dimension n (X may be B).
template <typename T, int NWV, bool TRANS, class Sync>
__device__ __forceinline__ void wg_getrs(int n, int nr, const T* __restrict__ LU,
                                         const i64* __restrict__ piv, const T* B, T* X,
                                         WgSolveLds<T, NWV>& L, int tid, Sync sync)
{
    constexpr int NT = 64 * NWV;
    for (int i = tid; i < n; i += NT) {
        const i64 p = piv[i];
        L.piv[i] = (short)((p >= 0 && p < n) ? p : i);
    }
    sync();
    // the row that the interchanges, taken backwards, trace row i to
    for (int i = tid; i < n; i += NT) {
        int s = i;
        for (int k = n - 1; k >= 0; --k) {
            const int p = L.piv[k];
            s = s == k ? p : s == p ? k : s;
        }
        L.src[i] = (short)s;
    }
    sync();
    const int nb = (n + 15) >> 4;
    for (int c0 = 0; c0 < nr; c0 += WS_RHS) {
        const int nc = nr - c0 < WS_RHS ? nr - c0 : WS_RHS;
        for (int e = tid; e < nb * 256; e += NT) {
            const int i = e % (nb * 16), c = e / (nb * 16);    // (c < 16)
            T v = T(0);
            if (i < n && c < nc) v = B[(TRANS ? i : (int)L.src[i]) + (i64)(c0 + c) * n];
            L.x[i][c] = v;
        }
        if (tid == 0) L.bad = 0;
        sync();
        if constexpr (!TRANS) {
            wg_trsv<T, NWV, false, true, true>(n, LU, n, L, tid, sync);
            wg_trsv<T, NWV, false, false, false>(n, LU, n, L, tid, sync);
            // A NaN may come from a product that the substitution leaves out (a
            // zero entry takes no part in it, src/TMV_TriDiv_V.cpp:187, but a
            // zero times an Inf of the factors does in a matrix step): such
            // columns are solved again by plain column sweeps, a wave each.
            for (int e = tid; e < nc * n; e += NT) {
                const T v = L.x[e % n][e / n];
                if (v != v) atomicOr(&L.bad, 1 << (e / n));
            }
            sync();
            const int bad = __builtin_amdgcn_readfirstlane(L.bad);
            if (bad) {
                for (int c = NWV == 1 ? 0 : tid >> 6; c < nc; c += NWV)
                    if ((bad >> c) & 1) plain_getrs<T, NWV>(n, LU, B + (i64)(c0 + c) * n, L, c, tid & 63);
                sync();
            }
        } else {
            wg_trsv<T, NWV, true, true, false>(n, LU, n, L, tid, sync);
            wg_trsv<T, NWV, true, false, true>(n, LU, n, L, tid, sync);
        }
        for (int e = tid; e < nc * n; e += NT) {
            const int i = e % n, c = e / n;
            X[(TRANS ? (int)L.src[i] : i) + (i64)(c0 + c) * n] = L.x[i][c];
        }
        sync();
    }
}

// The systems of a batch, with a grid of one workgroup per system: workgroup
// i takes system i when 64 < n <= WS_NMAX, wave i of the grid system i when
// n <= 64 (larger ones are skipped).  No loop over systems: what a loop could
// keep in registers from one to the next is more than there are.
template <typename T>
union WgSolveShared {
    WgSolveLds<T, 4> g;
    WgSolveLds<T, 1> w[4];
};

template <typename T, bool TRANS>
__device__ __forceinline__ void wg_getrs_batch(int count, const int* __restrict__ nv,
                                               const int* __restrict__ nrhsv,
                                               const T* const* __restrict__ LUv,
                                               const i64* const* __restrict__ pivv,
                                               const T* const* Bv, T* const* Xv,
                                               WgSolveShared<T>& sh)
{
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    {
        const int sys = blockIdx.x;
        const int n = __builtin_amdgcn_readfirstlane(nv[sys]);
        const int nr = __builtin_amdgcn_readfirstlane(nrhsv[sys]);
        if (n > 64 && n <= WS_NMAX && nr > 0)
            wg_getrs<T, 4, TRANS>(n, nr, LUv[sys], pivv[sys], Bv[sys], Xv[sys], sh.g, tid,
                                  GroupSync());
    }
    if ((int)blockIdx.x * 4 >= count) return;
    __syncthreads();
    const int sys = (int)blockIdx.x * 4 + wave;
    if (sys >= count) return;
    const int n = __builtin_amdgcn_readfirstlane(nv[sys]);
    const int nr = __builtin_amdgcn_readfirstlane(nrhsv[sys]);
    if (n > 0 && n <= 64 && nr > 0)
        wg_getrs<T, 1, TRANS>(n, nr, LUv[sys], pivv[sys], Bv[sys], Xv[sys], sh.w[wave], tid & 63,
                              WaveSync());
}

} // namespace tmvx
