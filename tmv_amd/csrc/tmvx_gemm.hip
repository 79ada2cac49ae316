// GEMM entry points: configuration table, default choice per precision,
// and the C ABI (tmvx_gemm_f64 / tmvx_gemm_f32 and the tuning hooks).
#include "tmvx_gemm_decl.h"
#include "tmvx_gemm_cfgs.h"

namespace tmvx {

template <typename T> struct GemmTable;

#define TMVX_CFG_CASE(ID, BM, BN, BK, WM, WN, MW)                                   \
    case ID: return gemm_launch_cfg<GemmCfg<T, BM, BN, BK, WM, WN, MW>, T>(         \
                 ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
#define TMVX_CFG_NAME(ID, BM, BN, BK, WM, WN, MW)                                   \
    case ID: return #BM "x" #BN "x" #BK " waves " #WM "x" #WN " min/simd " #MW;
#define TMVX_CFG_COUNT(ID, BM, BN, BK, WM, WN, MW) +1

template <> struct GemmTable<double> {
    typedef double T;
    static constexpr int count = 0 TMVX_F64_CFGS(TMVX_CFG_COUNT);
    static int run(int cfg, int ta, int tb, i64 m, i64 n, i64 k, T alpha, const T* A,
                   i64 lda, const T* B, i64 ldb, T beta, T* C, i64 ldc, hipStream_t s)
    {
        switch (cfg) { TMVX_F64_CFGS(TMVX_CFG_CASE) default: return TMVX_ERR_ARG; }
    }
    static const char* name(int cfg)
    { switch (cfg) { TMVX_F64_CFGS(TMVX_CFG_NAME) default: return nullptr; } }
};

template <> struct GemmTable<float> {
    typedef float T;
    static constexpr int count = 0 TMVX_F32_CFGS(TMVX_CFG_COUNT);
    static int run(int cfg, int ta, int tb, i64 m, i64 n, i64 k, T alpha, const T* A,
                   i64 lda, const T* B, i64 ldb, T beta, T* C, i64 ldc, hipStream_t s)
    {
        switch (cfg) { TMVX_F32_CFGS(TMVX_CFG_CASE) default: return TMVX_ERR_ARG; }
    }
    static const char* name(int cfg)
    { switch (cfg) { TMVX_F32_CFGS(TMVX_CFG_NAME) default: return nullptr; } }
};

// Default configuration by shape, from what the configurations measured
// (table in tmvx_gemm_cfgs.h):
//   - fewer 64 x 64 tiles than CUs: 32 x 32 tiles, four times as many (512^3
//     FP64 26 -> 12 us; level with 64 x 64 at 1000^3, 256 tiles);
//   - 128 x 128 tiles with at least four full turns over the 256 CUs and at
//     most 3% of the last one idle, K deep enough that the traffic of C does
//     not count: the fewest LDS reads per product (8192^3 FP64 15.3 ms against
//     15.7; but 4.2 ms against 3.9 at 5000^3, 10% idle);
//   - else 128 x 64 where C is large, 64 x 64 below and for a short K:
//     several workgroups a CU hide each other's waits and the read and write
//     of C (8192 x 8192 x 128 FP32 278-289 us against 302).  The line lies
//     where 128 x 64 starts to win on some shapes; time of 64 x 64 over that
//     of 128 x 64, square column-major products, FP64 / FP32:
//       n     1777  2048         2500         3072         4096
//             1.06  1.00 / 0.98  0.88 / 0.87  0.90 / 0.91  0.99 / 1.02
//     and 1.00-1.04 above 16e6 entries.  Which is faster turns on how full
//     the last turn over the 256 CUs is, and FP32 with a row-major A gains
//     (3001 x 1777 x 2500: 1.04-1.06) where column-major loses: from the line
//     to 16e6 entries this costs about 3% (FP64) and 5% (FP32) on average
//     against the better of the two, and a line at 16e6 would cost 1%, but
//     4-6% on the shapes named here;
//   - in FP32 a row-major B takes 128 x 64 in place of 128 x 128 tiles
//     (4096^3: 1.05 ms against 1.22).
template <typename T> int default_cfg(int tb, i64 m, i64 n, i64 k)
{
    constexpr bool D = sizeof(T) == 8;
    constexpr int C64 = D ? 0 : 3, C128 = 1, C128x64 = 2, C32 = 4;
    const i64 t64 = ((m + 63) / 64) * ((n + 63) / 64);
    if (t64 < 256) return C32;
    const i64 t128 = ((m + 127) / 128) * ((n + 127) / 128);
    const i64 idle = (256 - t128 % 256) % 256;
    if (t128 >= 1024 && k >= 1024 && 32 * idle <= t128) return !D && tb ? C128x64 : C128;
    if (k <= 128) return C64;
    return (double)m * (double)n >= (D ? 4.0e6 : 5.0e6) ? C128x64 : C64;
}

// Scale C by beta (k == 0 or alpha == 0): C = beta * C, or 0 when beta == 0.
template <typename T>
__global__ void scale_kernel(i64 m, i64 n, T beta, T* C, i64 ldc)
{
    const i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    const i64 j = blockIdx.y;
    if (i < m && j < n) C[i + j * ldc] = beta == T(0) ? T(0) : beta * C[i + j * ldc];
}

template <typename T>
int gemm_run(int cfg, int ta, int tb, i64 m, i64 n, i64 k, T alpha, const T* A,
             i64 lda, const T* B, i64 ldb, T beta, T* C, i64 ldc, hipStream_t s)
{
    if (m < 0 || n < 0 || k < 0) return TMVX_ERR_ARG;
    if (m == 0 || n == 0) return TMVX_OK;
    if (ldc < m || lda < (ta ? k : m) || ldb < (tb ? n : k)) return TMVX_ERR_ARG;
    if (lda < 1 || ldb < 1) return TMVX_ERR_ARG;
    if (!C || (k > 0 && alpha != T(0) && (!A || !B))) return TMVX_ERR_ARG;
    if (k == 0 || alpha == T(0)) {
        if (beta == T(1)) return TMVX_OK;
        if (n > 65535) return TMVX_ERR_UNSUPPORTED;
        dim3 grid((unsigned)((m + 255) / 256), (unsigned)n);
        hipLaunchKernelGGL(scale_kernel<T>, grid, dim3(256), 0, s, m, n, beta, C, ldc);
        TMVX_CHECK_LAUNCH();
        return TMVX_OK;
    }
    if (cfg < 0) cfg = default_cfg<T>(tb, m, n, k);
    return GemmTable<T>::run(cfg, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}

template <typename T>
int gemm_launch(int ta, int tb, i64 m, i64 n, i64 k, T alpha, const T* A,
                i64 lda, const T* B, i64 ldb, T beta, T* C, i64 ldc,
                hipStream_t s)
{
    return gemm_run<T>(-1, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}

// Large FP32 trailing updates beside a panel take 128 x 64 tiles of 32 deep
// stages, one wave a SIMD: a panel's workgroups (two waves of 138 registers a
// SIMD) must find room on a CU before the chain goes on, and a chip filled to
// four waves a SIMD gives it late.  FP64 panels need a whole CU beside any
// tile, so the faster tile wins.
template <typename T>
int gemm_launch_beside(int ta, int tb, i64 m, i64 n, i64 k, T alpha, const T* A, i64 lda,
                       const T* B, i64 ldb, T beta, T* C, i64 ldc, hipStream_t s)
{
    const bool wide = sizeof(T) == 4 && k > 128 && (double)m * (double)n >= 1048576.0;
    return gemm_run<T>(wide ? 6 : -1, ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, s);
}

template int gemm_launch_beside<double>(int, int, i64, i64, i64, double, const double*, i64,
                                        const double*, i64, double, double*, i64, hipStream_t);
template int gemm_launch_beside<float>(int, int, i64, i64, i64, float, const float*, i64,
                                       const float*, i64, float, float*, i64, hipStream_t);
template int gemm_launch<double>(int, int, i64, i64, i64, double, const double*,
                                 i64, const double*, i64, double, double*, i64,
                                 hipStream_t);
template int gemm_launch<float>(int, int, i64, i64, i64, float, const float*,
                                i64, const float*, i64, float, float*, i64,
                                hipStream_t);

static bool layouts_ok(int la, int lb)
{
    return (la == TMVX_COLMAJOR || la == TMVX_ROWMAJOR) &&
           (lb == TMVX_COLMAJOR || lb == TMVX_ROWMAJOR);
}

} // namespace tmvx

extern "C" {

int tmvx_gemm_f64(int la, int lb, int64_t m, int64_t n, int64_t k, double alpha,
                  const double* A, int64_t lda, const double* B, int64_t ldb,
                  double beta, double* C, int64_t ldc, void* stream)
{
    if (!tmvx::layouts_ok(la, lb)) return TMVX_ERR_ARG;
    return tmvx::gemm_launch<double>(la, lb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                     (hipStream_t)stream);
}

int tmvx_gemm_f32(int la, int lb, int64_t m, int64_t n, int64_t k, float alpha,
                  const float* A, int64_t lda, const float* B, int64_t ldb,
                  float beta, float* C, int64_t ldc, void* stream)
{
    if (!tmvx::layouts_ok(la, lb)) return TMVX_ERR_ARG;
    return tmvx::gemm_launch<float>(la, lb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                    (hipStream_t)stream);
}

int tmvx_gemm_config_count(int elem_bytes)
{
    return elem_bytes == 8 ? tmvx::GemmTable<double>::count
         : elem_bytes == 4 ? tmvx::GemmTable<float>::count : 0;
}

const char* tmvx_gemm_config_name(int elem_bytes, int cfg)
{
    const char* s = elem_bytes == 8 ? tmvx::GemmTable<double>::name(cfg)
                  : elem_bytes == 4 ? tmvx::GemmTable<float>::name(cfg) : nullptr;
    return s ? s : "";
}

int tmvx_gemm_cfg_f64(int cfg, int la, int lb, int64_t m, int64_t n, int64_t k, double alpha,
                      const double* A, int64_t lda, const double* B, int64_t ldb,
                      double beta, double* C, int64_t ldc, void* stream)
{
    if (!tmvx::layouts_ok(la, lb) || cfg < 0 || cfg >= tmvx::GemmTable<double>::count)
        return TMVX_ERR_ARG;
    return tmvx::gemm_run<double>(cfg, la, lb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                  (hipStream_t)stream);
}

int tmvx_gemm_cfg_f32(int cfg, int la, int lb, int64_t m, int64_t n, int64_t k, float alpha,
                      const float* A, int64_t lda, const float* B, int64_t ldb,
                      float beta, float* C, int64_t ldc, void* stream)
{
    if (!tmvx::layouts_ok(la, lb) || cfg < 0 || cfg >= tmvx::GemmTable<float>::count)
        return TMVX_ERR_ARG;
    return tmvx::gemm_run<float>(cfg, la, lb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                                 (hipStream_t)stream);
}

} // extern "C"
