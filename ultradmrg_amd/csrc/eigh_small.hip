// Eigen-decompositions of small real symmetric matrices, one workgroup each,
// entirely in LDS: the cyclic two-sided Jacobi method with the round-robin
// ordering (every round rotates n / 2 disjoint pairs).
//
// The block SVD of a short chain, or of the edge sectors of a large one, has
// Gram matrices of a few tens of rows.  The library's divide and conquer
// spends several launches per column on them (0.6 ms of kernels and over 1 ms
// of host time at order 32, whatever the batch); here a whole batch is one
// launch.  A sweep of a 20-site chain at D = 48, whose 36 updates are mostly
// such decompositions, went from 156 to 101 ms.  A round is bound by latency:
// the rotation angles (two reciprocal square roots and a reciprocal in
// sequence), two barriers and the LDS round trips between them; a matrix takes
// n - 1 rounds a sweep and 6 to 8 sweeps, spectra over many decades up to 16.
//
// Accuracy against the library's solver (means over random and graded matrices
// of order 32): residual 2.6e-15 |A| and 2.9e-15, orthonormality 6.3e-15 and
// 7.9e-15.  It takes rotate()'s form and an angle that keeps small rotations
// small: with c x - s y and divisions rounded to the last bit the two figures
// were 1.0e-14 and 2.8e-14.
//
// A pair is rotated while |a_pq| > 4 eps sqrt(|a_pp a_qq|) and above 1e-3 eps
// |A|_F: the Gram matrices' small eigenvalues keep their relative accuracy as
// long as the matrix itself does.  A matrix whose pairs stay above that for
// kSweeps sweeps (an indefinite one can, at rounding level) is accepted if its
// off-diagonal elements are within 16 eps |A|_F.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>

#include "common.h"
#include "eigh.h"

namespace qlg {

namespace {
constexpr double kEps = 2.220446049250313e-16;
constexpr int kSweeps = 24;

// reciprocal and reciprocal square root from the hardware estimates and Newton
// steps: a third of the latency of the IEEE sequences, which set a round's time
__device__ inline double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}
__device__ inline double rsqrt_(double x) {
  double r = __builtin_amdgcn_rsq(x);
  r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
  return fma(0.5 * r, fma(-x * r, r, 1.0), r);
}

// (x, y) <- (c x - s y, s x + c y), as corrections to x and y: with tau =
// s / (1 + c) the rounding errors are proportional to the angle, where those of
// c x - s y are an ulp of x whatever the angle and add up over hundreds of rounds
__device__ inline void rotate(double s, double tau, double &x, double &y) {
  const double x0 = x;
  x = fma(-s, fma(tau, x0, y), x0);
  y = fma(s, fma(-tau, y, x0), y);
}

template <class Op>
__device__ inline double block_reduce(double v, double *red, Op op) {
  const int tid = threadIdx.x;
  for (int o = 32; o; o >>= 1) v = op(v, __shfl_xor(v, o));
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = v;
  __syncthreads();
  v = red[0];
  for (int i = 1; i < (int)blockDim.x / 64; ++i) v = op(v, red[i]);
  return v;
}
__device__ inline double block_sum(double v, double *red) {
  return block_reduce(v, red, [](double x, double y) { return x + y; });
}
__device__ inline double block_max(double v, double *red) {
  return block_reduce(v, red, [](double x, double y) { return fmax(x, y); });
}
}  // namespace

// a: [batch][n][n] row-major symmetric; on return row j is eigenvector j, w
// the ascending eigenvalues; info[m] = 0, or 1 if matrix m did not converge.
// Dynamic LDS: A and V, [n][n + 1] doubles each.
__global__ __launch_bounds__(1024) void jacobi_eigh_kernel(double *__restrict__ a, double *__restrict__ w, int *__restrict__ info, int n) {
  extern __shared__ double lds[];
  __shared__ double red[16];   // one per wave
  __shared__ double rot[kSmallEigh / 2][3];   // sin theta, tan(theta / 2), tan theta
  __shared__ int pk[kSmallEigh / 2], qk[kSmallEigh / 2];
  __shared__ int rotated;
  const int ld = n + 1, tid = threadIdx.x, nt = blockDim.x;
  double *A = lds, *V = lds + n * ld;
  double *ga = a + (int64_t)blockIdx.x * n * n;
  double *gw = w + (int64_t)blockIdx.x * n;
  double big = 0.0;   // largest magnitude; infinite if any element is not finite
  for (int e = tid; e < n * n; e += nt) {
    const int i = e / n, j = e % n;
    // the row-major upper triangle is the input, as for the library's solver
    // (which takes the lower one of the same memory read column-major)
    const double v = ga[i <= j ? e : j * n + i];
    A[i * ld + j] = v;
    V[i * ld + j] = i == j ? 1.0 : 0.0;
    big = fmax(big, fabs(v) <= DBL_MAX ? fabs(v) : HUGE_VAL);
  }
  big = block_max(big, red);
  if (big > DBL_MAX) {   // NaN or infinity in the input: NaN out
    for (int e = tid; e < n * n; e += nt) ga[e] = big - big;
    for (int i = tid; i < n; i += nt) gw[i] = big - big;
    if (tid == 0) info[blockIdx.x] = 0;
    return;
  }
  // scaled by a power of two to a largest element in [1, 2), whatever the
  // input's range: no product below overflows, and no reciprocal meets a
  // denormal number
  const int ex = big > 0.0 ? ilogb(big) : 0;
  double fro = 0.0;
  for (int e = tid; e < n * n; e += nt) {   // (the thread's own elements)
    double &v = A[e / n * ld + e % n];
    v = ldexp(v, -ex);
    fro += v * v;
  }
  fro = sqrt(block_sum(fro, red));
  const int np = (n + 1) & ~1, half = np / 2;   // odd n: one index sits out each round
  const int lgh = half > 1 ? 32 - __clz(half - 1) : 0, lgn = n > 1 ? 32 - __clz(n - 1) : 0;
  const double floor_abs = 1e-3 * kEps * fro;
  int sweep = 0;
  bool done = n < 2;
  for (; !done && sweep < kSweeps; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int r = 0; r < np - 1; ++r) {
      // pair k of round r: position 0 is fixed, the others rotate by r
      auto at = [&](int pos) { return pos == 0 ? 0 : 1 + (pos - 1 + r) % (np - 1); };
      if (tid < half) {
        int p = at(tid), q = at(np - 1 - tid);
        if (p > q) {
          const int t = p;
          p = q;
          q = t;
        }
        double s = 0.0, tau = 0.0, t = 0.0;
        if (q < n) {
          const double app = A[p * ld + p], aqq = A[q * ld + q], apq = A[p * ld + q], m = fabs(apq);
          if (m > floor_abs && m > 4.0 * kEps * sqrt(fabs(app * aqq))) {
            // half of the angle 2 theta = atan(2 a_pq / (a_qq - a_pp)): cos^2 theta =
            // (1 + |cos 2 theta|) / 2, sin theta = |sin 2 theta| / (2 cos theta)
            const double d = aqq - app, r = rsqrt_(fma(d, d, 4.0 * apq * apq));
            const double cc = fma(0.5 * fabs(d), r, 0.5), rc = rsqrt_(cc);
            s = m * r * rc;
            if ((d >= 0.0) != (apq >= 0.0)) s = -s;
            tau = s * recip(fma(cc, rc, 1.0));   // tan(theta / 2)
            t = s * rc;
            rotated = 1;
          }
        }
        rot[tid][0] = s;
        rot[tid][1] = tau;
        rot[tid][2] = t;
        pk[tid] = p;
        qk[tid] = q;
      }
      __syncthreads();
      // A <- J^T A J on 2 x 2 blocks (pair k's rows, pair l's columns), and
      // rows p, q of V: one index space, so that every thread has an item
      const int na = half << lgh, nv = half << lgn;
      for (int e = tid; e < na + nv; e += nt) {
        if (e >= na) {
          const int k = (e - na) >> lgn, j = (e - na) & ((1 << lgn) - 1);
          const double s = rot[k][0], tau = rot[k][1];
          if (s == 0.0 || j >= n) continue;
          rotate(s, tau, V[pk[k] * ld + j], V[qk[k] * ld + j]);
          continue;
        }
        const int k = e >> lgh, l = e & ((1 << lgh) - 1);
        if (l >= half) continue;
        const double sk = rot[k][0], tk = rot[k][1], sl = rot[l][0], tl = rot[l][1];
        if (sk == 0.0 && sl == 0.0) continue;
        const int p = pk[k], q = qk[k], u = pk[l], v = qk[l];
        const bool hq = q < n, hv = v < n;   // (an index that sits out has s = 0)
        double x00 = A[p * ld + u], x01 = hv ? A[p * ld + v] : 0.0;
        double x10 = hq ? A[q * ld + u] : 0.0, x11 = hq && hv ? A[q * ld + v] : 0.0;
        if (k == l) {
          const double t = rot[k][2];
          x00 = fma(-t, x01, x00);
          x11 = fma(t, x01, x11);
          x01 = x10 = 0.0;
        } else {
          rotate(sk, tk, x00, x10);
          rotate(sk, tk, x01, x11);
          rotate(sl, tl, x00, x01);
          rotate(sl, tl, x10, x11);
        }
        A[p * ld + u] = x00;
        if (hv) A[p * ld + v] = x01;
        if (hq) A[q * ld + u] = x10;
        if (hq && hv) A[q * ld + v] = x11;
      }
      __syncthreads();
    }
    done = rotated == 0;
    __syncthreads();
  }
  int bad = 0;
  if (!done) {
    double off = 0.0;
    for (int e = tid; e < n * n; e += nt) {
      const int i = e / n, j = e % n;
      if (i != j) off += A[i * ld + j] * A[i * ld + j];
    }
    off = sqrt(block_sum(off, red));
    bad = !(off <= 16.0 * kEps * fro);
  }
  if (tid == 0) info[blockIdx.x] = bad;
  // ascending order: an eigenvalue's place is the number of smaller ones
  for (int i = tid >> 6; i < n; i += nt >> 6) {
    const double x = A[i * ld + i];
    int rank = 0;
    for (int j0 = 0; j0 < n; j0 += 64) {
      const int j = j0 + (tid & 63);
      const double y = j < n ? A[j * ld + j] : 0.0;
      rank += __popcll(__ballot(j < n && (y < x || (y == x && j < i))));
    }
    if ((tid & 63) == 0) gw[rank] = ldexp(x, ex);
    for (int j = tid & 63; j < n; j += 64) ga[rank * n + j] = V[i * ld + j];
  }
}

void launch_jacobi_eigh(double *a, double *w, int *info, int n, int batch, hipStream_t st) {
  QLG_CHECK(n >= 1 && n <= kSmallEigh, "small eigensolver: order out of range");
  const size_t lds = (size_t)2 * n * (n + 1) * sizeof(double);
  QLG_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(jacobi_eigh_kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              2 * kSmallEigh * (kSmallEigh + 1) * (int)sizeof(double)));
  // a thread per 2 x 2 block of A and pair of V's elements, up to 1024
  const int threads = n <= 16 ? 192 : n <= 24 ? 512 : 1024;
  hipLaunchKernelGGL(jacobi_eigh_kernel, dim3(batch), dim3(threads), lds, st, a, w, info, n);
  QLG_HIP(hipGetLastError());
}

}  // namespace qlg
