// direct.hpp -- one CSR product on host arrays without a plan (direct.cpp).
#pragma once

#include "internal.hpp"

namespace sblas {

// y = alpha*A*x + beta*y on the current device `device`; rp[0] = 0 and rp[m] =
// nnz are checked by the caller.  handled stays false, with nothing done, for
// calls that this path leaves to a plan: the v2 rule, empty sizes, a matrix
// beyond the context's memory, SBLAS_VARIANT, or a context in use by another
// thread.
int direct_csr(int device, int m, int n, int nnz, double alpha, const double *val, const int *rp,
               const int *col, const double *x, double beta, double *y, int kernel, int part_mode,
               spmv_ret &ret, bool &handled);

}  // namespace sblas
