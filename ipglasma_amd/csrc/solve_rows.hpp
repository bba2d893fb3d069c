// solve_rows.hpp -- the root finder's 8x8 linear system (device and host build)
#pragma once
#include "su3.hpp"

IPG_HD bool solve_any(bool x) {
#ifdef __HIP_DEVICE_COMPILE__
    return __any(x);
#else
    return x;
#endif
}
// J y = F by Gaussian elimination with partial pivoting (first maximal pivot),
// J row-major, in registers; y replaces F.  Rows are exchanged by selects, and
// only when some lane of the wavefront has an exchange to make.
IPG_HD void solve_rows(double (&J)[64], double (&F)[8]) {
#pragma unroll
    for (int j = 0; j < 7; j++) {
        double best = fabs(J[9 * j]);
        int p = j;
#pragma unroll
        for (int r = j + 1; r < 8; r++)
            if (fabs(J[8 * r + j]) > best) {
                best = fabs(J[8 * r + j]);
                p = r;
            }
        if (solve_any(p != j)) {
#pragma unroll
            for (int r = j + 1; r < 8; r++) {
                const bool sw = r == p;
#pragma unroll
                for (int c = j; c < 8; c++) {
                    const double x = J[8 * j + c], y = J[8 * r + c];
                    J[8 * j + c] = sw ? y : x;
                    J[8 * r + c] = sw ? x : y;
                }
                const double x = F[j], y = F[r];
                F[j] = sw ? y : x;
                F[r] = sw ? x : y;
            }
        }
        // a reciprocal instead of a division a row; of a pivot below the normal
        // numbers, whose column has nothing larger, it would be infinite and the
        // step NaN instead of large
        const double inv = fabs(J[9 * j]) < 1e-300 ? 0. : 1. / J[9 * j];
#pragma unroll
        for (int r = j + 1; r < 8; r++) {
            const double f = J[8 * r + j] * inv;
#pragma unroll
            for (int c = j + 1; c < 8; c++) J[8 * r + c] -= f * J[8 * j + c];
            F[r] -= f * F[j];
        }
    }
#pragma unroll
    for (int r = 7; r >= 0; r--) {
        double t = F[r];
#pragma unroll
        for (int c = r + 1; c < 8; c++) t -= J[8 * r + c] * F[c];
        F[r] = t / J[9 * r];
    }
}
