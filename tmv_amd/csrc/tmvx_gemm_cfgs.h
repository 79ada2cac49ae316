// GEMM tile-configuration tables: X(id, BM, BN, BK, WM, WN, min waves/SIMD).
// The tile does not show in the result: whatever BM, BN and BK, an entry of C
// is one MFMA chain over k, 16 at a time, the last ones filled up with zeros.
// The LU relies on it where it takes another tile beside a panel than alone.
// Measured on MI355X, column-major operands, beta != 0 (us):
//                       f64 0    1    2    4 | f32 0    1    2    3    4
//   512^3                  26   76   41   12 |    47   53   30   17    8
//   1000^3                 47  133   72   46 |    83   91   52   29   27
//   2048^3                251  254  251  308 |   144  161  150  142  164
//   4096^3               1924 1950 1912 2408 |  1069 1047 1052 1066 1245
//   8192^3    (ms)       15.8 15.3 15.7 19.1 |  8.30 8.04 8.14 8.36 9.99
//   8192 x 8192 x 256     639  813  620  883 |   541  463  389  385  513
#pragma once

#define TMVX_F64_CFGS(X)                    \
    X(0, 64, 64, 16, 2, 2, 4)               \
    X(1, 128, 128, 16, 4, 4, 1)             \
    X(2, 128, 64, 16, 4, 2, 4)              \
    X(3, 32, 64, 32, 2, 2, 2)               \
    X(4, 32, 32, 32, 2, 2, 2)               \
    X(5, 128, 128, 32, 4, 4, 1)

#define TMVX_F32_CFGS(X)                    \
    X(0, 128, 128, 32, 4, 4, 1)             \
    X(1, 128, 128, 16, 2, 2, 1)             \
    X(2, 128, 64, 16, 2, 2, 3)              \
    X(3, 64, 64, 16, 2, 2, 4)               \
    X(4, 32, 32, 32, 2, 2, 2)               \
    X(5, 64, 64, 32, 2, 2, 4)               \
    X(6, 128, 64, 32, 2, 2, 1)
