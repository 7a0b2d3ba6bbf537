// Large FP64 products on the int8 matrix cores (crt.hip).
#pragma once
#include "gi_context.h"

namespace gi {

// whether the int8 route is the faster one for an m x n x k product; `part`:
// share of the multiply-adds left by a triangular A
bool crt_pays(long long m, long long n, long long k, double part = 1.0);

// C (m x n, ldc) = beta C + alpha A B^T, A (m x k, lda) and B (n x k, ldb)
// column-major; tri: A is lower triangular (its upper part holds zeros).
// false, with C untouched, when an operand has rows that cannot be scaled (NaN,
// infinities, norms outside 1e-125..1e150), or when the work arrays cannot be had
// (int8_work_mb 0, a failed allocation): the caller's DGEMM then.
bool crt_gemm_nt(Context &C, long long m, long long n, long long k, double alpha, const double *A, long long lda,
                 const double *B, long long ldb, double beta, double *Cd, long long ldc, bool tri);

// the same with A(g, c) = X(g, p) X(g, q) of the orbital pair (p, q) =
// (pq[2 c], pq[2 c + 1]), halved for p = q, zero for p < 0
bool crt_pairs_nt(Context &C, long long m, long long n, long long k, double alpha, const double *X, long long ldx,
                  const int *pq, const double *B, long long ldb, double beta, double *Cd, long long ldc);

}  // namespace gi
