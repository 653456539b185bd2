// Batched Hermitian eigen-decomposition (small real matrices in LDS, the others
// by rocSOLVER's divide and conquer over host-threaded lanes); used by the
// block SVD.
#pragma once

#include "common.h"

namespace qlg {

// Largest order of the in-LDS solver (eigh_small.hip).  Four Gram matrices with
// singular values over seven decades, whole call: order 16 0.14 ms, 32 0.35,
// 48 0.85, 64 1.5; the library's solver 1.7 ms at order 96 and little less
// below.  The line lies at 32, and the block SVD's at 28 rows, because of the
// truncated states: where values are kept down to a few 1e-6 of the largest,
// the library's vectors of the small ones are off by up to 2e-10 (this solver's
// by a tenth of that); up to 28 rows the two truncated states agree to 7e-11.
constexpr int kSmallEigh = 32;
void launch_jacobi_eigh(double *a, double *w, int *info, int n, int batch, hipStream_t st);

// use_small: groups of real order up to kSmallEigh go to the in-LDS solver
void eigh_batched(Ctx &c, int dtype, int64_t ngroups, const qlg_eigh_group *groups, bool use_small = true);

}  // namespace qlg
