// Batched Hermitian eigen-decomposition (small real matrices in LDS, the others
// by rocSOLVER's divide and conquer over host-threaded lanes); used by the
// block SVD.
#pragma once

#include "common.h"

namespace qlg {

// Largest order of the in-LDS solver (eigh_small.hip).  Four Gram matrices with
// singular values over seven decades, whole call: order 16 0.14 ms, 32 0.35,
// 48 0.85, 64 1.5, 96 5.4; the library's solver takes 2.1 ms at order 112 and
// little less below, so the line lies between 64 and 96.
constexpr int kSmallEigh = 64;
void launch_jacobi_eigh(double *a, double *w, int *info, int n, int batch, hipStream_t st);

void eigh_batched(Ctx &c, int dtype, int64_t ngroups, const qlg_eigh_group *groups);

}  // namespace qlg
