// Batched Hermitian eigen-decomposition (small real matrices in LDS, the others
// by rocSOLVER's divide and conquer over host-threaded lanes); used by the
// block SVD.
#pragma once

#include "common.h"

namespace qlg {

// Largest order of the in-LDS solver (eigh_small.hip).  Four Gram matrices with
// singular values over seven decades, whole call, here and with the library's
// solver: order 8 0.08 and 0.28 ms, 16 0.16 and 0.59, 24 0.36 and 0.86, 32 0.46
// and 1.24.  It is the faster one up to order 64 (1.5 and 1.6 ms); the line lies
// at 32, and the block SVD's at 28 rows, so that truncated states stay what they
// are with the library's solver.  Where values are kept down to a few 1e-6 of
// the largest, any two solvers' states differ in the vectors of those: up to 28
// rows by at most 8e-11 (51 of 160 drawn states; both are up to 5e-11 from a
// dense SVD's), above by up to 4.9e-10.
constexpr int kSmallEigh = 32;
void launch_jacobi_eigh(double *a, double *w, int *info, int n, int batch, hipStream_t st);

// use_small: groups of real order up to kSmallEigh go to the in-LDS solver
void eigh_batched(Ctx &c, int dtype, int64_t ngroups, const qlg_eigh_group *groups, bool use_small = true);

}  // namespace qlg
