// written_columns.cpp -- a program of the drop-in layer that writes columns: every
// off-diagonal column of the finest level becomes -1 (no entry), after which A x is
// 26 x.  Prints the least and the largest entry of A * 1.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "Extensions.hpp"
#include "hpcg.hpp"
#include "../../include/rochpcg_amd.h"

int main()
{
    Geometry* geom = new Geometry;
    GenerateGeometry(1, 0, 1, 0, 0, 0, 16, 24, 16, 1, 1, 1, geom);
    SparseMatrix A;
    InitializeSparseMatrix(A, geom);
    Vector b, x, xexact;
    GenerateProblem(A, &b, &x, &xexact);
    SetupHalo(A);
    CGData data;
    if(OptimizeProblem(A, data, b, x, xexact)) return 1;
    const long m = A.localNumberOfRows, n = (m + 127) / 128 * 128 * A.ell_width;
    std::vector<local_int_t> col(n), diag(m);
    if(hpcgx_memcpy_d2h(diag.data(), A.diag_idx, sizeof(local_int_t) * m)) return 2;
    std::fill(col.begin(), col.end(), -1);
    for(long r = 0; r < m; ++r) col[((r / 128) * A.ell_width + diag[r]) * 128 + r % 128] = (local_int_t)r;
    if(hpcgx_memcpy_h2d(A.ell_col_ind, col.data(), sizeof(local_int_t) * n)) return 3;
    if(HPCGX_ReadColumnsInPlace(A)) return 4;
    Vector y;
    HIPInitializeVector(y, A.localNumberOfRows);
    if(ComputeSPMV(A, xexact, y)) return 5;
    double sum, t = 0.0;
    bool opt = true;
    ComputeDotProduct(A.localNumberOfRows, y, y, sum, t, opt);   // waits for the product
    std::vector<double> h(m);
    if(hpcgx_memcpy_d2h(h.data(), y.d_values, sizeof(double) * m)) return 6;
    printf("%g %g\n", *std::min_element(h.begin(), h.end()), *std::max_element(h.begin(), h.end()));
    return 0;
}
