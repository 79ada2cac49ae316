// QR decomposition by Householder reflections and the least-squares /
// square solve with its factors (QR division).
//
// TMV's QR_Decompose(A, beta, det) (src/TMV_QRDecompose.cpp:603-650) stores
// the reflectors below the diagonal (first element 1, implicit), R on and
// above it, and beta (the reflectors' scale: H = I - beta v v^T).  Each
// reflector follows HouseholderReflect (src/TMV_Householder.cpp:46-180):
// scale by max |x|; y = -|x| when x0 > 0, else +|x|; v = x / (x0 - y) so
// that v(0) = 1; beta = (x0 - y)^2 / (|x|^2 - y x0); R(j, j) = y scale;
// an underflowing column becomes zero (beta = 0), and a column already zero
// below the diagonal needs no reflection (beta = 0).  QR division
// (QR_LDiv, src/TMV_QRDiv.cpp:33-94): y = Q^T b, x = R^-1 y(0:n).
//
// Up to QN_MMAX rows: panels of 8 columns, two launches each.
//   qr8_panel_kernel: one workgroup, its rows in registers (one to eight a
//     thread).  Per column two reductions over the workgroup: the scale max
//     |x|, then at once the norm, the dot products with the panel's later
//     columns and those with its earlier reflectors, from which the column of
//     T (LAPACK larft: H_0 .. H_7 = I - V T V^T) follows in the same kernel;
//   qr8_update_kernel: C := C - V (T^T (V^T C)), four columns a workgroup.
// The solve forms every panel's T in one launch and applies Q^T to a right-hand
// side in one workgroup, the vector in registers, a panel at a time.
// Bound: the two reductions a column (27 us a panel of 2000 rows: 3.4 us a
// column) and two launches per panel.  FP64 2000 x 500, decomposition and
// solve: 27.5 -> 3.3 ms (panels 13.9 -> 1.7, update 12.1 -> 1.2, Q^T b 0.2).
// More rows: 32-column panels by ONE workgroup in global memory, the compact WY
// update on the MFMA GEMM.
// Real types only.
#include "tmvx_wave_solve.h"
#include "tmvx_pivot.h"

#include <cfloat>
#include <cmath>

namespace tmvx {

constexpr int QR_NB = 32;        // panel width
constexpr int QR_NTH = 512;      // panel workgroup

template <typename T> struct QrLim;
template <> struct QrLim<double> { static constexpr double rmin = DBL_MIN; };
template <> struct QrLim<float> { static constexpr float rmin = FLT_MIN; };

// Sum (op = 0) or maximum (op = 1) of the workgroup's values v[0..K).
template <typename T, int K>
__device__ __forceinline__ void block_reduce(T (&v)[K], int op, T (*s_red)[K], int nk)
{
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    constexpr int NW = QR_NTH / 64;
    // static indices (a runtime index would put v in scratch memory)
#pragma unroll
    for (int q = 0; q < K; ++q)
        if (q < nk)
            for (int off = 32; off > 0; off >>= 1) {
                const T o = __shfl_xor(v[q], off);
                v[q] = op ? fmax(v[q], o) : v[q] + o;
            }
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < K; ++q)
            if (q < nk) s_red[wave][q] = v[q];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < K; ++q)
        if (q < nk) {
            T a = s_red[0][q];
            for (int w = 1; w < NW; ++w) a = op ? fmax(a, s_red[w][q]) : a + s_red[w][q];
            v[q] = a;
        }
    __syncthreads();                      // s_red is reused by the next call
}

// Reflectors for panel columns [j0, j1) of the m x n matrix; the panel's own
// later columns are updated as each reflector is formed.
template <typename T>
__global__ void __launch_bounds__(QR_NTH)
qr_panel_kernel(i64 m, T* __restrict__ A, i64 lda, i64 j0, i64 j1, T* __restrict__ beta)
{
    constexpr int NW = QR_NTH / 64;
    const int t = threadIdx.x;
    __shared__ T s_red[NW][QR_NB];
    __shared__ T s_w[QR_NB];
    for (i64 j = j0; j < j1; ++j) {
        T* x = A + j * lda;                 // column j; x[j] is x0
        // scale = max |x_i| over i >= j
        T mv[1] = {T(0)};
        for (i64 i = j + t; i < m; i += QR_NTH) mv[0] = fmax(mv[0], fabs(x[i]));
        block_reduce<T, 1>(mv, 1, reinterpret_cast<T(*)[1]>(s_red), 1);
        const T scale = mv[0];
        if (!(scale >= QrLim<T>::rmin)) {   // hopeless: the column becomes zero
            for (i64 i = j + t; i < m; i += QR_NTH) x[i] = T(0);
            if (t == 0) beta[j] = T(0);
            __syncthreads();
            continue;
        }
        const T invscale = T(1) / scale;
        T ns[1] = {T(0)};
        for (i64 i = j + 1 + t; i < m; i += QR_NTH) {
            const T a = x[i] * invscale;
            ns[0] += a * a;
        }
        block_reduce<T, 1>(ns, 0, reinterpret_cast<T(*)[1]>(s_red), 1);
        const T normsqx = ns[0];
        const T x0 = x[j];
        if (normsqx == T(0)) {              // H = I
            for (i64 i = j + 1 + t; i < m; i += QR_NTH) x[i] = T(0);
            if (t == 0) beta[j] = T(0);
            __syncthreads();
            continue;
        }
        const T x0s = x0 * invscale;
        const T normsq = normsqx + x0s * x0s;
        const T normx = sqrt(normsq);
        const T y = x0s > T(0) ? -normx : normx;
        const T v0 = x0s - y;
        const T b = (v0 * v0) / (normsq - y * x0s);
        const T sinv = (T(1) / v0) * invscale;
        for (i64 i = j + 1 + t; i < m; i += QR_NTH) x[i] *= sinv;
        __syncthreads();
        if (t == 0) { x[j] = y * scale; beta[j] = b; }
        // apply H = I - b v v^T to the panel's later columns
        const int nc = (int)(j1 - j - 1);
        if (nc > 0) {
            T dots[QR_NB];
            for (int c = 0; c < QR_NB; ++c) dots[c] = T(0);
            for (i64 i = j + 1 + t; i < m; i += QR_NTH) {
                const T vi = x[i];
#pragma unroll
                for (int c = 0; c < QR_NB; ++c)
                    if (c < nc) dots[c] += vi * A[i + (j + 1 + c) * lda];
            }
            block_reduce<T, QR_NB>(dots, 0, s_red, nc);
#pragma unroll
            for (int c = 0; c < QR_NB; ++c)       // dots[] is uniform after the reduction
                if (c < nc && t == c) s_w[c] = b * (A[j + (j + 1 + c) * lda] + dots[c]);   // v(0) = 1
            __syncthreads();
            if (t < nc) A[j + (j + 1 + t) * lda] -= s_w[t];
            for (i64 i = j + 1 + t; i < m; i += QR_NTH) {
                const T vi = x[i];
                for (int c = 0; c < nc; ++c) A[i + (j + 1 + c) * lda] -= s_w[c] * vi;
            }
        }
        __syncthreads();
    }
}

// V (m2 x jb, column-major, ld m2): the panel's reflectors with their unit
// first elements and zeros above.
template <typename T>
__global__ void qr_copy_v_kernel(i64 m2, int jb, const T* __restrict__ A, i64 lda, T* __restrict__ V)
{
    const int c = blockIdx.y;
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < m2; i += (i64)gridDim.x * blockDim.x)
        V[i + c * m2] = i < c ? T(0) : (i == c ? T(1) : A[i + (i64)c * lda]);
}

// T (jb x jb upper, column-major) of the compact WY form I - V T V^T from
// G = V^T V and beta (LAPACK larft, forward columnwise):
//   T(i, i) = beta_i,  T(0:i, i) = -beta_i T(0:i, 0:i) G(0:i, i).
template <typename T>
__global__ void qr_form_t_kernel(int jb, const T* __restrict__ G, const T* __restrict__ beta,
                                 T* __restrict__ Tm)
{
    __shared__ T s_t[QR_NB][QR_NB + 1];
    __shared__ T s_g[QR_NB][QR_NB + 1];
    const int t = threadIdx.x;
    for (int e = t; e < QR_NB * QR_NB; e += blockDim.x) {
        const int r = e % QR_NB, c = e / QR_NB;
        s_g[r][c] = (r < jb && c < jb) ? G[r + c * jb] : T(0);
        s_t[r][c] = T(0);
    }
    __syncthreads();
    for (int i = 0; i < jb; ++i) {
        const T bi = beta[i];
        if (t < i) {
            T acc = T(0);
            for (int q = t; q < i; ++q) acc += s_t[t][q] * s_g[q][i];   // T upper: q >= t
            s_t[t][i] = -bi * acc;
        }
        if (t == 0) s_t[i][i] = bi;
        __syncthreads();
    }
    for (int e = t; e < jb * jb; e += blockDim.x) {
        const int r = e % jb, c = e / jb;
        Tm[r + c * jb] = s_t[r][c];
    }
}

// C (m2 x nc, ld ldc) := (I - V T V^T)^T C for the panel's V (from A at
// column j0, m2 = m - j0 rows) and beta.  ws: m2*jb + 2*jb*jb + jb*nc
// elements.
template <typename T>
int qr_apply_block(i64 m2, int jb, const T* Apanel, i64 lda, const T* beta, T* C, i64 ldc, i64 nc,
                   T* ws, hipStream_t s)
{
    if (nc <= 0 || m2 <= 0 || jb <= 0) return TMVX_OK;
    T* V = ws;
    T* G = V + m2 * jb;
    T* Tm = G + (i64)jb * jb;
    T* W = Tm + (i64)jb * jb;
    const unsigned gx = (unsigned)((m2 + 255) / 256 < 1024 ? (m2 + 255) / 256 : 1024);
    hipLaunchKernelGGL(qr_copy_v_kernel<T>, dim3(gx, (unsigned)jb), dim3(256), 0, s, m2, jb, Apanel,
                       lda, V);
    TMVX_CHECK_LAUNCH();
    // G = V^T V (V^T is V read row-major)
    TMVX_TRY(gemm_launch<T>(1, 0, jb, jb, m2, T(1), V, m2, V, m2, T(0), G, jb, s));
    hipLaunchKernelGGL(qr_form_t_kernel<T>, dim3(1), dim3(64), 0, s, jb, G, beta, Tm);
    TMVX_CHECK_LAUNCH();
    // W = V^T C  (jb x nc)
    TMVX_TRY(gemm_launch<T>(1, 0, jb, nc, m2, T(1), V, m2, C, ldc, T(0), W, jb, s));
    // W := T^T W  (T^T is T read row-major); G's space holds the product
    T* W2 = G;
    if ((i64)jb * nc > (i64)jb * jb) {
        // G is only jb x jb: put the product after W instead
        W2 = W + (i64)jb * nc;
    }
    TMVX_TRY(gemm_launch<T>(1, 0, jb, nc, jb, T(1), Tm, jb, W, jb, T(0), W2, jb, s));
    // C -= V W2
    TMVX_TRY(gemm_launch<T>(0, 0, m2, nc, jb, T(-1), V, m2, W2, jb, T(1), C, ldc, s));
    return TMVX_OK;
}

static i64 qr_ws_elems(i64 m, i64 ncols)
{
    return m * QR_NB + 2 * (i64)QR_NB * QR_NB + 2 * (i64)QR_NB * ncols;
}

// ---- panels of 8 columns in registers --------------------------------------

constexpr int QN_NTH = 512;              // panel and solve workgroup
constexpr int QN_NW = QN_NTH / 64;
constexpr int QN_NB = 8;
constexpr int QN_RPT = 8;                // rows a thread holds at most
constexpr i64 QN_MMAX = (i64)QN_NTH * QN_RPT;
constexpr int QU_NTH = 256;              // update workgroup
constexpr int QU_CW = 4;                 // and its columns

// The wave's sum of v, in lane 63.
template <typename T> __device__ __forceinline__ T wave_sum63(T v)
{
    v = dpp_add<0xB1, 0xf>(v);
    v = dpp_add<0x4E, 0xf>(v);
    v = dpp_add<0x141, 0xf>(v);
    v = dpp_add<0x140, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);
    v = dpp_add<0x143, 0xc>(v);
    return v;
}

// Sums of v[0..8) over the workgroup of QN_NW waves: lane l returns that of
// v[l & 7].  One barrier; s (one per parity of the calls) holds the waves' sums.
template <typename T>
__device__ __forceinline__ T group_sum8(const T (&v)[8], T (&s)[QN_NW][8])
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    static_assert(QN_NW == 8, "a lane per wave and value");
    static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
        constexpr int c = decltype(cc)::value;
        const T x = wave_sum63(v[c]);
        if (lane == 63) s[wave][c] = x;
    });
    __syncthreads();
    T x = s[lane >> 3][lane & 7];
    x += __shfl_xor(x, 8);
    x += __shfl_xor(x, 16);
    x += __shfl_xor(x, 32);
    return x;
}

// Reflectors of columns [0, jb) of the m x jb panel A (jb <= 8, m <= RPT
// QN_NTH), their beta, and the 8 x 8 upper T of I - V T V^T (column-major,
// zeros past jb).
template <typename T, int RPT>
__global__ void __launch_bounds__(QN_NTH)
qr8_panel_kernel(int m, int jb, T* __restrict__ A, i64 lda, T* __restrict__ beta,
                 T* __restrict__ Tm)
{
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    __shared__ T s_mx[2][QN_NW];
    __shared__ T s_sum[2][QN_NW][8];
    __shared__ T s_prow[2][8];
    T row[RPT][8], trow[8];
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * QN_NTH;
        static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            row[q][c] = (r < m && c < jb) ? A[r + c * lda] : T(0);
        });
    });
    static_for<0, 8>([&](auto cc) __attribute__((always_inline)) { trow[decltype(cc)::value] = T(0); });
    static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, par = k & 1;
        if (k >= jb) return;                             // uniform
        // scale = max |x_r|, r >= k (row r is thread r mod QN_NTH's)
        T mx = t >= k ? T(fabs(row[0][k])) : T(0);
        static_for<1, RPT>([&](auto q_) __attribute__((always_inline)) {
            mx = fmax(mx, T(fabs(row[decltype(q_)::value][k])));
        });
        mx = dpp_max_step<0xB1, 0xf>(mx);
        mx = dpp_max_step<0x4E, 0xf>(mx);
        mx = dpp_max_step<0x141, 0xf>(mx);
        mx = dpp_max_step<0x140, 0xf>(mx);
        mx = dpp_max_step<0x142, 0xa>(mx);
        mx = dpp_max_step<0x143, 0xc>(mx);
        if (lane == 63) s_mx[par][wave] = mx;
        if (t == k)
            static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
                s_prow[par][decltype(cc)::value] = row[0][decltype(cc)::value];
            });
        __syncthreads();
        T scale = s_mx[par][lane & 7];
        scale = dpp_max_step<0xB1, 0xf>(scale);
        scale = dpp_max_step<0x4E, 0xf>(scale);
        scale = dpp_max_step<0x141, 0xf>(scale);
        scale = readlane(scale, 0);
        const T pv = s_prow[par][lane & 7];              // lane c: row k's column c
        if (!(scale >= QrLim<T>::rmin)) {                // hopeless: the column becomes zero
            static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                if (q > 0 || t >= k) row[q][k] = T(0);
            });
            if (t == 0) beta[k] = T(0);
            return;
        }
        const T invscale = T(1) / scale;
        // value c != k: sum over r > k of (x_r invscale) row[r][c]; value k: of
        // (x_r invscale)^2
        T sum[8];
        static_for<0, 8>([&](auto cc) __attribute__((always_inline)) { sum[decltype(cc)::value] = T(0); });
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            const T sx = (q > 0 || t > k) ? row[q][k] * invscale : T(0);
            static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
                constexpr int c = decltype(cc)::value;
                sum[c] = fma(sx, c == k ? sx : row[q][c], sum[c]);
            });
        });
        const T tot = group_sum8(sum, s_sum[par]);
        const T normsqx = row_bcast<k>(tot);
        if (normsqx == T(0)) {                           // H = I
            static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                if (q > 0 || t > k) row[q][k] = T(0);
            });
            if (t == 0) beta[k] = T(0);
            return;
        }
        const T x0s = row_bcast<k>(pv) * invscale;
        const T normsq = normsqx + x0s * x0s;
        const T normx = sqrt(normsq);
        const T y = x0s > T(0) ? -normx : normx;
        const T v0 = x0s - y;
        const T b = (v0 * v0) / (normsq - y * x0s);
        const T rv0 = T(1) / v0, sinv = rv0 * invscale;
        // dot products with v: lane c that of column c (later column or earlier
        // reflector), v(k) = 1.  The sums are those of v v0, up to sqrt(m) times
        // larger: where one overflows, all are formed again with v.
        T dot = fma(tot, rv0, pv);
        if (__builtin_amdgcn_ballot_w64(!(tot - tot == T(0)))) {          // uniform
            T again[8];
            static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
                constexpr int c = decltype(cc)::value;
                again[c] = T(0);
                static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                    constexpr int q = decltype(q_)::value;
                    const T vr = (q > 0 || t > k) ? row[q][k] * sinv : T(0);
                    again[c] = fma(vr, row[q][c], again[c]);
                });
            });
            dot = group_sum8(again, s_sum[par ^ 1]) + pv;
        }
        const T w = b * dot;
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            if (q > 0 || t > k) row[q][k] *= sinv;
        });
        static_for<k + 1, 8>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            const T wc = row_bcast<c>(w);
            static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                constexpr int q = decltype(q_)::value;
                if (q > 0 || t > k) row[q][c] = fma(-wc, row[q][k], row[q][c]);
                else if (t == k) row[q][c] -= wc;
            });
        });
        if (t == k) row[0][k] = y * scale;
        if (t == 0) beta[k] = b;
        // column k of T, row i in lane i
        T acc = T(0);
        static_for<0, k>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            acc = fma(trow[c], row_bcast<c>(dot), acc);
        });
        trow[k] = lane < k ? -b * acc : lane == k ? b : T(0);
    });
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * QN_NTH;
        static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            if (r < m && c < jb) A[r + c * lda] = row[q][c];
        });
    });
    if (t < 8)
        static_for<0, 8>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            Tm[t + 8 * c] = trow[c];
        });
}

// Entry (r, c) of a panel's V: unit diagonal, zeros above (and past jb).
template <typename T>
__device__ __forceinline__ T qr8_v(const T* __restrict__ A, i64 lda, int r, int c, int jb)
{
    return (r < c || c >= jb) ? T(0) : r == c ? T(1) : A[r + c * lda];
}

// C (m x nc) := (I - V T V^T)^T C, V the m x jb panel at A.
template <typename T>
__global__ void __launch_bounds__(QU_NTH)
qr8_update_kernel(int m, int jb, const T* __restrict__ A, i64 lda, const T* __restrict__ Tm,
                  T* __restrict__ C, i64 ldc, i64 nc)
{
    constexpr int NW = QU_NTH / 64;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    __shared__ T s_w[NW][8][QU_CW];
    __shared__ T s_w1[8][QU_CW], s_w2[8][QU_CW];
    const i64 cb = (i64)blockIdx.x * QU_CW;
    T* __restrict__ Cc = C + cb * ldc;
    const int ncc = nc - cb < QU_CW ? (int)(nc - cb) : QU_CW;
    T acc[8][QU_CW];
    static_for<0, 8 * QU_CW>([&](auto ec) __attribute__((always_inline)) {
        constexpr int e = decltype(ec)::value;
        acc[e / QU_CW][e % QU_CW] = T(0);
    });
    for (int r = t; r < m; r += QU_NTH) {
        T v[8], x[QU_CW];
        static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
            v[decltype(kc)::value] = qr8_v(A, lda, r, decltype(kc)::value, jb);
        });
        static_for<0, QU_CW>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            x[c] = Cc[r + (c < ncc ? c : 0) * ldc];
        });
        static_for<0, 8 * QU_CW>([&](auto ec) __attribute__((always_inline)) {
            constexpr int k = decltype(ec)::value / QU_CW, c = decltype(ec)::value % QU_CW;
            acc[k][c] = fma(v[k], x[c], acc[k][c]);
        });
    }
    static_for<0, 8 * QU_CW>([&](auto ec) __attribute__((always_inline)) {
        constexpr int k = decltype(ec)::value / QU_CW, c = decltype(ec)::value % QU_CW;
        const T x = wave_sum63(acc[k][c]);
        if (lane == 63) s_w[wave][k][c] = x;
    });
    __syncthreads();
    if (t < 8 * QU_CW) {
        T x = T(0);
        for (int q = 0; q < NW; ++q) x += s_w[q][t / QU_CW][t % QU_CW];
        s_w1[t / QU_CW][t % QU_CW] = x;
    }
    __syncthreads();
    if (t < 8 * QU_CW) {                                 // T^T W
        const int i = t / QU_CW, c = t % QU_CW;
        T x = T(0);
        for (int q = 0; q <= i; ++q) x = fma(Tm[q + 8 * i], s_w1[q][c], x);
        s_w2[i][c] = x;
    }
    __syncthreads();
    T w[8][QU_CW];
    static_for<0, 8 * QU_CW>([&](auto ec) __attribute__((always_inline)) {
        constexpr int k = decltype(ec)::value / QU_CW, c = decltype(ec)::value % QU_CW;
        w[k][c] = s_w2[k][c];
    });
    for (int r = t; r < m; r += QU_NTH) {
        T v[8], x[QU_CW];
        static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
            v[decltype(kc)::value] = qr8_v(A, lda, r, decltype(kc)::value, jb);
        });
        static_for<0, QU_CW>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            x[c] = Cc[r + (c < ncc ? c : 0) * ldc];
        });
        static_for<0, 8 * QU_CW>([&](auto ec) __attribute__((always_inline)) {
            constexpr int k = decltype(ec)::value / QU_CW, c = decltype(ec)::value % QU_CW;
            x[c] = fma(-v[k], w[k][c], x[c]);
        });
        static_for<0, QU_CW>([&](auto cc) __attribute__((always_inline)) {
            constexpr int c = decltype(cc)::value;
            if (c < ncc) Cc[r + c * ldc] = x[c];
        });
    }
}

// T of every panel of 8 columns of a factored m x n matrix: workgroup p that of
// columns [8 p, 8 p + 8), from G = V^T V (LAPACK larft, forward columnwise).
template <typename T>
__global__ void __launch_bounds__(QU_NTH)
qr8_form_t_kernel(i64 m, i64 n, const T* __restrict__ QR, i64 lda, const T* __restrict__ beta,
                  T* __restrict__ Tm)
{
    constexpr int NW = QU_NTH / 64, NP = 28;             // pairs q < i
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const i64 j0 = (i64)blockIdx.x * QN_NB;
    const int jb = n - j0 < QN_NB ? (int)(n - j0) : QN_NB, m2 = (int)(m - j0);
    const T* __restrict__ A = QR + j0 + j0 * lda;
    __shared__ T s_g[NW][NP];
    __shared__ T s_t[8][8];
    T g[NP];
    static_for<0, NP>([&](auto ec) __attribute__((always_inline)) { g[decltype(ec)::value] = T(0); });
    for (int r = t; r < m2; r += QU_NTH) {
        T v[8];
        static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
            v[decltype(kc)::value] = qr8_v(A, lda, r, decltype(kc)::value, jb);
        });
        static_for<1, 8>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            static_for<0, i>([&](auto qc) __attribute__((always_inline)) {
                constexpr int q = decltype(qc)::value, e = i * (i - 1) / 2 + q;
                g[e] = fma(v[q], v[i], g[e]);
            });
        });
    }
    static_for<0, NP>([&](auto ec) __attribute__((always_inline)) {
        constexpr int e = decltype(ec)::value;
        const T x = wave_sum63(g[e]);
        if (lane == 63) s_g[wave][e] = x;
    });
    if (t < 64) s_t[t >> 3][t & 7] = T(0);
    __syncthreads();
    if (t < 8) {
        for (int i = 0; i < jb; ++i) {
            const T b = beta[j0 + i];
            T acc = T(0);
            if (t < i)
                for (int q = t; q < i; ++q) {
                    T x = T(0);
                    for (int w = 0; w < NW; ++w) x += s_g[w][i * (i - 1) / 2 + q];
                    acc = fma(s_t[t][q], x, acc);
                }
            if (t < i) s_t[t][i] = -b * acc;
            if (t == i) s_t[i][i] = b;
            __builtin_amdgcn_wave_barrier();
        }
    }
    __syncthreads();
    if (t < 64) Tm[(i64)blockIdx.x * 64 + t] = s_t[t & 7][t >> 3];
}

// B(:, blockIdx.x) := Q^T B(:, blockIdx.x): the panels in turn, the column in
// registers, row t + q QN_NTH in thread t's slot q.  (FP32 with four rows a
// thread needs a few registers less than it takes for three workgroups a CU.)
template <typename T, int RPT>
__global__ void __launch_bounds__(QN_NTH)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) * RPT <= 16 ? 6 : sizeof(T) * RPT <= 32 ? 4 : 2)))
qr8_apply_kernel(int m, int n, const T* __restrict__ QR, i64 lda, const T* __restrict__ Tm,
                 T* __restrict__ B, i64 ldb)
{
    const int t = threadIdx.x, lane = t & 63;
    __shared__ T s_sum[2][QN_NW][8];
    T* __restrict__ b = B + (i64)blockIdx.x * ldb;
    T x[RPT];
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * QN_NTH;
        x[q] = r < m ? b[r] : T(0);
    });
    const int np = (n + QN_NB - 1) / QN_NB;
    for (int p = 0; p < np; ++p) {
        const int j0 = p * QN_NB, jb = n - j0 < QN_NB ? n - j0 : QN_NB;
        const T* __restrict__ A = QR + j0 + j0 * lda;
        T v[RPT][8], sum[8];
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            const int r = t + q * QN_NTH - j0;           // row of the panel
            static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                v[q][k] = (r >= 0 && r + j0 < m) ? qr8_v(A, lda, r, k, jb) : T(0);
            });
        });
        const T tk = lane < 64 ? Tm[(i64)p * 64 + lane] : T(0);   // T(lane & 7, lane >> 3)
        static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            sum[k] = T(0);
            static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                sum[k] = fma(v[decltype(q_)::value][k], x[decltype(q_)::value], sum[k]);
            });
        });
        const T w = group_sum8(sum, s_sum[p & 1]);       // lane l: W(l & 7)
        // T^T W: lane l has T(l & 7, l >> 3) W(l & 7); summed over l & 7 it is
        // entry l >> 3
        T z = tk * w;
        z = dpp_add<0xB1, 0xf>(z);
        z = dpp_add<0x4E, 0xf>(z);
        z = dpp_add<0x141, 0xf>(z);
        static_for<0, 8>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const T zk = readlane(z, 8 * k);
            static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
                x[decltype(q_)::value] = fma(-v[decltype(q_)::value][k], zk, x[decltype(q_)::value]);
            });
        });
        // the panel's own rows are finished: zeros in their place, as an Inf
        // would reach the others through its zero in V
        static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
            constexpr int q = decltype(q_)::value;
            const int r = t + q * QN_NTH;
            if ((unsigned)(r - j0) < (unsigned)jb) {
                b[r] = x[q];
                x[q] = T(0);
            }
        });
    }
    static_for<0, RPT>([&](auto q_) __attribute__((always_inline)) {
        constexpr int q = decltype(q_)::value;
        const int r = t + q * QN_NTH;
        if (r >= n && r < m) b[r] = x[q];
    });
}

template <typename T>
int geqrf_narrow(i64 m, i64 n, T* A, i64 lda, T* beta, T* Tm, hipStream_t s)
{
    for (i64 j0 = 0; j0 < n; j0 += QN_NB) {
        const int jb = (int)(n - j0 < QN_NB ? n - j0 : QN_NB), m2 = (int)(m - j0);
        T* P = A + j0 + j0 * lda;
        const int rpt = (m2 + QN_NTH - 1) / QN_NTH;
#define QN_PANEL(RPT)                                                                         \
    hipLaunchKernelGGL((qr8_panel_kernel<T, RPT>), dim3(1), dim3(QN_NTH), 0, s, m2, jb, P,     \
                       lda, beta + j0, Tm)
        if (rpt <= 1) QN_PANEL(1);
        else if (rpt <= 2) QN_PANEL(2);
        else if (rpt <= 4) QN_PANEL(4);
        else QN_PANEL(8);
#undef QN_PANEL
        const i64 nc = n - j0 - jb;
        if (nc > 0)
            hipLaunchKernelGGL(qr8_update_kernel<T>, dim3((unsigned)((nc + QU_CW - 1) / QU_CW)),
                               dim3(QU_NTH), 0, s, m2, jb, P, lda, Tm, P + (i64)jb * lda, lda, nc);
        TMVX_CHECK_LAUNCH();
    }
    return TMVX_OK;
}

// B := Q^T B for nrhs columns; Tm: 64 elements per panel.
template <typename T>
int qr8_apply_q(i64 m, i64 n, i64 nrhs, const T* QR, i64 lda, const T* beta, T* Tm, T* B, i64 ldb,
                hipStream_t s)
{
    const unsigned np = (unsigned)((n + QN_NB - 1) / QN_NB);
    hipLaunchKernelGGL(qr8_form_t_kernel<T>, dim3(np), dim3(QU_NTH), 0, s, m, n, QR, lda, beta, Tm);
    const int rpt = (int)((m + QN_NTH - 1) / QN_NTH);
#define QN_APPLY(RPT)                                                                         \
    hipLaunchKernelGGL((qr8_apply_kernel<T, RPT>), dim3((unsigned)nrhs), dim3(QN_NTH), 0, s,   \
                       (int)m, (int)n, QR, lda, Tm, B, ldb)
    if (rpt <= 1) QN_APPLY(1);
    else if (rpt <= 2) QN_APPLY(2);
    else if (rpt <= 4) QN_APPLY(4);
    else QN_APPLY(8);
#undef QN_APPLY
    return hip_status(hipGetLastError());
}

template <typename T>
int geqrf_impl(i64 m, i64 n, T* A, i64 lda, T* beta, hipStream_t s)
{
    if (m < 0 || n < 0 || m < n || lda < (m > 0 ? m : 1)) return TMVX_ERR_ARG;
    if (n == 0) return TMVX_OK;
    if (!A || !beta) return TMVX_ERR_ARG;
    T* ws = nullptr;
    if (hipMallocAsync((void**)&ws, sizeof(T) * (size_t)qr_ws_elems(m, n), s) != hipSuccess)
        return TMVX_ERR_ALLOC;
    int rc = TMVX_OK;
    if (m <= QN_MMAX) {                      // (the workspace holds a T)
        rc = geqrf_narrow<T>(m, n, A, lda, beta, ws, s);
        hipFreeAsync(ws, s);
        return rc;
    }
    for (i64 j0 = 0; j0 < n && rc == TMVX_OK; j0 += QR_NB) {
        const int jb = (int)(n - j0 < QR_NB ? n - j0 : QR_NB);
        hipLaunchKernelGGL(qr_panel_kernel<T>, dim3(1), dim3(QR_NTH), 0, s, m, A, lda, j0, j0 + jb,
                           beta);
        if ((rc = hip_status(hipGetLastError())) != TMVX_OK) break;
        rc = qr_apply_block<T>(m - j0, jb, A + j0 + j0 * lda, lda, beta + j0,
                               A + j0 + (j0 + jb) * lda, lda, n - j0 - jb, ws, s);
    }
    hipFreeAsync(ws, s);
    return rc;
}

__global__ void qr_diag_check_kernel(i64 n, const double* __restrict__ A, i64 lda, int* __restrict__ bad)
{
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        if (A[i + i * lda] == 0.0) *bad = 1;
}
__global__ void qr_diag_check_kernel_f(i64 n, const float* __restrict__ A, i64 lda, int* __restrict__ bad)
{
    for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (i64)gridDim.x * blockDim.x)
        if (A[i + i * lda] == 0.0f) *bad = 1;
}
__global__ void qr_set_int_kernel(int* p, int v) { *p = v; }

template <typename T>
int geqrs_impl(i64 m, i64 n, i64 nrhs, const T* QR, i64 lda, const T* beta, T* B, i64 ldb,
               hipStream_t s)
{
    if (m < 0 || n < 0 || m < n || nrhs < 0 || lda < (m > 0 ? m : 1) || ldb < (m > 0 ? m : 1))
        return TMVX_ERR_ARG;
    if (n == 0 || nrhs == 0) return TMVX_OK;
    if (!QR || !beta || !B) return TMVX_ERR_ARG;
    T* ws = nullptr;
    const size_t bytes = sizeof(T) * (size_t)qr_ws_elems(m, nrhs) + 64;
    if (hipMallocAsync((void**)&ws, bytes, s) != hipSuccess) return TMVX_ERR_ALLOC;
    int* d_bad = reinterpret_cast<int*>(reinterpret_cast<char*>(ws) + bytes - 64);
    int rc = TMVX_OK;
    // B := Q^T B = H_{n-1} ... H_0 B, a panel at a time (the narrow panels' T,
    // 8 n elements, fit the workspace's m QR_NB)
    const bool narrow = m <= QN_MMAX && nrhs <= 0x7fffffff;
    if (narrow) rc = qr8_apply_q<T>(m, n, nrhs, QR, lda, beta, ws, B, ldb, s);
    for (i64 j0 = 0; !narrow && j0 < n && rc == TMVX_OK; j0 += QR_NB) {
        const int jb = (int)(n - j0 < QR_NB ? n - j0 : QR_NB);
        rc = qr_apply_block<T>(m - j0, jb, QR + j0 + j0 * lda, lda, beta + j0, B + j0, ldb, nrhs,
                               ws, s);
    }
    // a zero diagonal of R: singular (TMV's triangular solve throws)
    if (rc == TMVX_OK) {
        hipLaunchKernelGGL(qr_set_int_kernel, dim3(1), dim3(1), 0, s, d_bad, 0);
        if constexpr (sizeof(T) == 8)
            hipLaunchKernelGGL(qr_diag_check_kernel, dim3((unsigned)((n + 255) / 256 < 256 ? (n + 255) / 256 : 256)),
                               dim3(256), 0, s, n, QR, lda, d_bad);
        else
            hipLaunchKernelGGL(qr_diag_check_kernel_f, dim3((unsigned)((n + 255) / 256 < 256 ? (n + 255) / 256 : 256)),
                               dim3(256), 0, s, n, QR, lda, d_bad);
        rc = hip_status(hipGetLastError());
    }
    int bad = 0;
    if (rc == TMVX_OK &&
        hipMemcpyAsync(&bad, d_bad, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess)
        rc = TMVX_ERR_HIP;
    if (rc == TMVX_OK && hipStreamSynchronize(s) != hipSuccess) rc = TMVX_ERR_HIP;
    if (rc == TMVX_OK && bad) rc = TMVX_ERR_SINGULAR;
    // X = R^-1 (Q^T B)(0:n)
    if (rc == TMVX_OK) {
        if constexpr (sizeof(T) == 8)
            rc = tmvx_trsm_f64(1, 0, 0, n, nrhs, QR, lda, B, ldb, s);
        else
            rc = tmvx_trsm_f32(1, 0, 0, n, nrhs, QR, lda, B, ldb, s);
    }
    hipFreeAsync(ws, s);
    return rc;
}

} // namespace tmvx

using namespace tmvx;

extern "C" {

int tmvx_geqrf_f64(int64_t m, int64_t n, double* A, int64_t lda, double* beta, void* stream)
{ return geqrf_impl<double>(m, n, A, lda, beta, (hipStream_t)stream); }
int tmvx_geqrf_f32(int64_t m, int64_t n, float* A, int64_t lda, float* beta, void* stream)
{ return geqrf_impl<float>(m, n, A, lda, beta, (hipStream_t)stream); }

int tmvx_geqrs_f64(int64_t m, int64_t n, int64_t nrhs, const double* QR, int64_t lda,
                   const double* beta, double* B, int64_t ldb, void* stream)
{ return geqrs_impl<double>(m, n, nrhs, QR, lda, beta, B, ldb, (hipStream_t)stream); }
int tmvx_geqrs_f32(int64_t m, int64_t n, int64_t nrhs, const float* QR, int64_t lda,
                   const float* beta, float* B, int64_t ldb, void* stream)
{ return geqrs_impl<float>(m, n, nrhs, QR, lda, beta, B, ldb, (hipStream_t)stream); }

} // extern "C"
