// Host build of the root finder's linear solve (ipglasma_amd/csrc/solve_rows.hpp)
#include "../../ipglasma_amd/csrc/solve_rows.hpp"

// J row-major, y = J^-1 F
extern "C" void solve_rows_host(const double* J, const double* F, double* y) {
    double A[64], b[8];
    for (int k = 0; k < 64; k++) A[k] = J[k];
    for (int k = 0; k < 8; k++) b[k] = F[k];
    solve_rows(A, b);
    for (int k = 0; k < 8; k++) y[k] = b[k];
}
