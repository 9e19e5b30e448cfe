// FP64 device linear algebra for B formation (see linalg.hip).
#pragma once
#include "common.hpp"

namespace nopt {
// C = alpha * A * op(B) + beta * C; op(B) = B (K x N, ldb) or, with transB,
// the transpose of B (N x K, ldb). Row-major; K at least 1.
hipError_t gemm_f64(bool transB, int M, int N, int K, double alpha, const double* A, long lda,
                    const double* B, long ldb, double beta, double* C, long ldc, hipStream_t s);
// In-place lower Cholesky A = L L^T (strict upper part zeroed); Xd gets the
// inverses of L's 64 x 64 diagonal blocks (chol_inverse_count(n) values).
// *d_info is set to j+1 for the first non-positive pivot j, else 0.
long chol_inverse_count(int n);
hipError_t cholesky_f64(double* A, long lda, int n, double* Xd, int* d_info, hipStream_t s);
// Rows r0 .. r1 (r0 a multiple of 64, r1 too or n) of B (n x ncol) <- those of
// L^-1 B for the factor and the inverses of cholesky_f64, the rows before r0
// being solved.
hipError_t trsm_lower_f64(const double* L, long ldl, int n, const double* Xd, double* B, long ldb, long ncol, int r0,
                          int r1, hipStream_t s);
}  // namespace nopt
