// Grouped FP64 GEMM on CDNA4 MFMA (v_mfma_f64_16x16x4_f64), in two kernels:
// direct_gemm_f64_kernel (further down) for the matvec's two contractions,
// whose operands the planner lays out for it, and grouped_gemm_f64_kernel for
// operands in any order (environment updates, contractions, the SVD's
// products) and for matvec plans whose spans the direct kernel cannot address.
//
// grouped_gemm_f64_kernel: one workgroup (4 wavefronts, 2x2) computes one BM x
// BN output tile of one task and walks the task's K-segments in order.
// BK-deep slices of A and B are staged through two LDS buffers (ping-pong): the
// raw buffer loads of slice i+1 are issued before the MFMAs of slice i and
// land in registers, which are written to the other LDS buffer afterwards, so
// each K step costs one barrier and the load latency hides behind the MFMA
// work.  Operands are read with raw buffer loads whose out-of-range elements
// come back as zero (tile_io.h), so the loads carry no branch and no select.
// Slices run as straight-line code, which lets the LDS fragment reads of one
// 4-deep sub-step overlap the MFMAs of the previous one (a segment's last
// slice is zero-filled past K and runs the same code).  Each wave owns a
// (BM/2) x (BN/2) sub-tile of 16x16 MFMA blocks; thin tiles (BN = 16, for
// tasks with few columns) stack the four waves along M.
//
// MFMA f64 16x16x4 operand layout (one double per lane):
//   A: lane l holds A[row = l % 16][k = l / 16]
//   B: lane l holds B[k = l / 16][col = l % 16]
//   D: lane l, register r holds D[row = l / 16 + 4 * r][col = l % 16]
//      (measured on gfx950 with an in-bounds probe of the builtin)
#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm.h"
#include "tile_io.h"

namespace qlg {

typedef double dbl4 __attribute__((ext_vector_type(4)));

namespace {
constexpr int PAD = 1;
}

template <int BM, int BN, int BK, bool CPLX>
__global__ __launch_bounds__(256, BM * BN * (CPLX ? 2 : 1) >= 128 * 128 ? 1 : 2) void grouped_gemm_f64_kernel(const GemmTile *__restrict__ tiles,
                                                               const GemmTask *__restrict__ tasks,
                                                               const GemmSeg *__restrict__ segs,
                                                               Slots slots, int ntiles) {
  // four waves: 2 x 2, or 4 x 1 for thin tiles (BN = 16)
  constexpr int WAVES_N = BN >= 32 ? 2 : 1, WAVES_M = 4 / WAVES_N;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;   // wave sub-tile
  constexpr int FM = WM / 16, FN = WN / 16;     // MFMA blocks per wave
  constexpr int A_PER = BM * BK / 256;          // A elements loaded per thread per slice
  constexpr int B_PER = BK * BN / 256;
  static_assert(A_PER >= 1 && B_PER >= 1, "tile too small for 256 threads");
  static_assert(WM >= 16 && WN >= 16, "wave sub-tile below one MFMA block");
  constexpr int NP = CPLX ? 2 : 1;              // real / imaginary planes
  constexpr uint32_t EB = CPLX ? 16u : 8u;      // element bytes
  __shared__ double As[2][NP][BK][BM + PAD];
  __shared__ double Bs[2][NP][BK][BN + PAD];

  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int wm0 = (wave / WAVES_N) * WM, wn0 = (wave % WAVES_N) * WN;
  if ((int)blockIdx.x >= ntiles) return;
  if (slots.skip && *slots.skip) return;   // the Krylov solve has stopped
  const GemmTile tl = tiles[blockIdx.x];
  if (tl.task < 0) return;  // padding slot of the XCD-balanced launch order
  const GemmTask tk = tasks[tl.task];
  const int M = tk.M, N = tk.N;

  dbl4 acc[NP][FM][FN];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[p][i][j] = dbl4{0.0, 0.0, 0.0, 0.0};

  double ra[NP][A_PER], rb[NP][B_PER];

  // element e of a slice: (m, k) of A and (k, n) of B, chosen so that
  // consecutive threads read consecutive addresses in either storage order.
  // The transposition flags are uniform, so the choice is a select on the
  // indices and every slice issues one straight sequence of loads.
  auto a_mk = [&](int i, bool ta, int &m, int &k) {
    const int e = tid + i * 256;
    m = ta ? e % BM : e / BK;
    k = ta ? e / BM : e % BK;
  };
  auto b_kn = [&](int i, bool tb, int &k, int &n) {
    const int e = tid + i * 256;
    n = tb ? e / BK : e % BN;
    k = tb ? e % BK : e / BN;
  };
  // Per-segment state of the slices being loaded: buffer descriptors, and
  // each element's offset at k0 = 0, its k within the slice and whether its
  // row / column lies inside the task.  A slice then costs one add, one
  // compare and one select per element.
  __amdgpu_buffer_rsrc_t ar, br;
  uint32_t astep = 1, bstep = 1;
  int segK = 0;
  uint32_t aoff[A_PER], boff[B_PER];
  int akk[A_PER], bkk[B_PER];
  bool ain[A_PER], bin[B_PER];
  auto setup = [&](const GemmSeg &sg) {
    ar = make_rsrc(slots.p[sg.a_slot] + sg.a_off * NP);
    br = make_rsrc(slots.p[sg.b_slot] + sg.b_off * NP);
    const uint32_t lda = (uint32_t)sg.lda, ldb = (uint32_t)sg.ldb;
    const bool ta = sg.flags & SEG_TRANS_A, tb = sg.flags & SEG_TRANS_B;
    segK = sg.K;
    astep = ta ? lda : 1u;
    bstep = tb ? 1u : ldb;
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      int m, k;
      a_mk(i, ta, m, k);
      const uint32_t gm = tl.m0 + m;
      aoff[i] = ta ? (uint32_t)k * lda + gm : gm * lda + (uint32_t)k;
      akk[i] = k;
      ain[i] = (int)gm < M;
    }
#pragma unroll
    for (int i = 0; i < B_PER; ++i) {
      int k, n;
      b_kn(i, tb, k, n);
      const uint32_t gn = tl.n0 + n;
      boff[i] = tb ? gn * ldb + (uint32_t)k : (uint32_t)k * ldb + gn;
      bkk[i] = k;
      bin[i] = (int)gn < N;
    }
  };
  auto load = [&](int k0) {
    const uint32_t ka = (uint32_t)k0 * astep, kb = (uint32_t)k0 * bstep;
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      const uint32_t off = (ain[i] && akk[i] + k0 < segK) ? (aoff[i] + ka) * EB : kOob;
      if constexpr (CPLX) {
        const double2 v = load_c128(ar, off);
        ra[0][i] = v.x;
        ra[1][i] = v.y;
      } else {
        ra[0][i] = load_f64(ar, off);
      }
    }
#pragma unroll
    for (int i = 0; i < B_PER; ++i) {
      const uint32_t off = (bin[i] && bkk[i] + k0 < segK) ? (boff[i] + kb) * EB : kOob;
      if constexpr (CPLX) {
        const double2 v = load_c128(br, off);
        rb[0][i] = v.x;
        rb[1][i] = v.y;
      } else {
        rb[0][i] = load_f64(br, off);
      }
    }
  };
  auto store = [&](int buf, uint8_t flags) {
    const bool ta = flags & SEG_TRANS_A, tb = flags & SEG_TRANS_B;
#pragma unroll
    for (int i = 0; i < A_PER; ++i) {
      int m, k;
      a_mk(i, ta, m, k);
      As[buf][0][k][m] = ra[0][i];
      if constexpr (CPLX) As[buf][1][k][m] = (flags & SEG_CONJ_A) ? -ra[1][i] : ra[1][i];
    }
#pragma unroll
    for (int i = 0; i < B_PER; ++i) {
      int k, n;
      b_kn(i, tb, k, n);
      Bs[buf][0][k][n] = rb[0][i];
      if constexpr (CPLX) Bs[buf][1][k][n] = (flags & SEG_CONJ_B) ? -rb[1][i] : rb[1][i];
    }
  };
  // one 4-deep sub-step of the staged slice
  auto step = [&](int buf, int kk) {
    double af[NP][FM], bf[NP][FN];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
#pragma unroll
      for (int i = 0; i < FM; ++i) af[p][i] = As[buf][p][kk + (lane >> 4)][wm0 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[p][j] = Bs[buf][p][kk + (lane >> 4)][wn0 + j * 16 + (lane & 15)];
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[0][i], bf[0][j], acc[0][i][j], 0, 0, 0);
        if constexpr (CPLX) {
          acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-af[1][i], bf[1][j], acc[0][i][j], 0, 0, 0);
          acc[1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[0][i], bf[1][j], acc[1][i][j], 0, 0, 0);
          acc[1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[1][i], bf[0][j], acc[1][i][j], 0, 0, 0);
        }
      }
  };

  const int s_end = tk.seg_begin + tk.seg_count;
  int s = tk.seg_begin;
  while (s < s_end && segs[s].K <= 0) ++s;
  if (s < s_end) {
    GemmSeg cur = segs[s];
    int k0 = 0, buf = 0;
    setup(cur);
    load(0);
    store(0, cur.flags);
    __syncthreads();
    while (true) {
      // iterator of the next slice; its loads stay in flight during this slice's MFMAs
      int ns = s, nk = k0 + BK;
      GemmSeg nxt = cur;
      if (nk >= cur.K) {
        ++ns;
        nk = 0;
        while (ns < s_end && segs[ns].K <= 0) ++ns;
        if (ns < s_end) nxt = segs[ns];
      }
      const bool more = ns < s_end;
      if (more) {
        if (ns != s) setup(nxt);
        load(nk);
      }
      // the staged slice is zero-filled past the segment's K, so a partial
      // slice runs the same straight-line code as a full one
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) step(buf, kk);
      if (!more) break;
      store(buf ^ 1, nxt.flags);
      __syncthreads();
      buf ^= 1;
      s = ns;
      k0 = nk;
      cur = nxt;
    }
  }

  // output row addresses: a row-address table or a plain row stride
  int64_t crow[FM][4];
  if (tk.c_rowtab) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tl.m0 + wm0 + i * 16 + (lane >> 4) + 4 * r;
        crow[i][r] = slots.crows[tk.c_row + min(row, M - 1)] - tk.c_off;
      }
  } else {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) crow[i][r] = (int64_t)(tl.m0 + wm0 + i * 16 + (lane >> 4) + 4 * r) * tk.ldc;
  }
  double *C = slots.p[tk.c_slot] + tk.c_off * NP;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = tl.n0 + wn0 + j * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tl.m0 + wm0 + i * 16 + (lane >> 4) + 4 * r;
        if (row < M && col < N) {
          const int64_t ix = crow[i][r] + col;
          if constexpr (CPLX)
            reinterpret_cast<double2 *>(C)[ix] = double2{acc[0][i][j][r], acc[1][i][j][r]};
          else
            C[ix] = acc[0][i][j][r];
        }
      }
    }
}

template <bool CPLX>
static void launch_shape(int bm, int bn, int bk, const GemmTile *tiles, const GemmTask *tasks, const GemmSeg *segs,
                         const Slots &slots, int ntiles, hipStream_t st) {
  dim3 grid(ntiles), block(256);
#define QLG_SHAPE(M_, N_, K_)                                                                                \
  if (bm == M_ && bn == N_ && bk == K_) {                                                                    \
    hipLaunchKernelGGL((grouped_gemm_f64_kernel<M_, N_, K_, CPLX>), grid, block, 0, st, tiles, tasks, segs,   \
                       slots, ntiles);                                                                       \
    return;                                                                                                  \
  }
  QLG_SHAPE(32, 32, 16)
  QLG_SHAPE(64, 32, 16)
  QLG_SHAPE(32, 64, 16)
  QLG_SHAPE(64, 64, 16)
  QLG_SHAPE(128, 64, 16)
  QLG_SHAPE(64, 128, 16)
  QLG_SHAPE(128, 128, 16)
  if constexpr (!CPLX) {  // two accumulator planes of complex tiles do not fit BK=32 double buffers
    QLG_SHAPE(64, 16, 16)
    QLG_SHAPE(128, 16, 16)
    QLG_SHAPE(32, 32, 32)
    QLG_SHAPE(64, 32, 32)
    QLG_SHAPE(32, 64, 32)
    QLG_SHAPE(64, 64, 32)
    QLG_SHAPE(128, 64, 32)
    QLG_SHAPE(64, 128, 32)
    QLG_SHAPE(64, 16, 32)
    QLG_SHAPE(128, 16, 32)
  }
#undef QLG_SHAPE
  throw Error(QLG_ERR_UNSUPPORTED, "unsupported FP64 tile shape");
}

// ---------------------------------------------------------------------------
// FP64 GEMM with operand fragments loaded straight from memory (the matvec's
// two contractions): C = A^T B with A stored [K x M] and B stored [K x N].
//
// A v_mfma_f64_16x16x4 takes 64 cycles, so a wave's matrix pipe is fed by few
// bytes per cycle: what bounds the matvec's tasks is the latency of the
// operand loads.  A lane loads exactly the operand values its MFMAs take,
// kDepth slices ahead, in registers: no LDS, no barrier, no per-element
// address arithmetic (the k offset of a slice is the load's scalar offset).
// Both operands are stored with k as the row index, so that the sixteen lanes
// that share a k read one contiguous run: with k contiguous the same lanes
// touch sixteen cache lines per load.
//
// Real data: two 16-wide blocks of a wave's tile are interleaved (lane l holds
// elements 2 (l % 16) and 2 (l % 16) + 1 of 32), so one 16-byte load feeds both.
// Such a load may reach one element past an odd-width operand's last column;
// the value lands in a row or column that is never stored, and the vectors'
// buffers carry that one element of slack.
//
// A workgroup's waves are WM x WN over the tile and WK over k: k-part w takes
// slices w, w + WK, ...; the parts are summed through LDS in order at the end.
// Small tiles use WK > 1, so that long-K tasks with few columns keep every
// SIMD busy.
//
// Measured per launch, LDS kernel -> this one (kernel trace): Hubbard D=2000
// (5.6 GFLOP each) stage 1 177 -> 145 us, stage 3 188 (and 17 for split-K's
// reduce) -> 137 us; dense 8 x (4096 x 4096 x 2048) 72 TFLOP/s.  The two-waves
// launch bound keeps the accumulators in vector registers: without it each
// slice moved them to and from the accumulation registers.  Counters of the
// two: MFMA pipe busy 0.56 and 0.65, waiting on memory 0.22 and 0.11 of the wave
// cycles, 1.7 and 3.0 waves per SIMD, padding to 16-wide blocks 1.10 and 1.19.
// ---------------------------------------------------------------------------
__device__ inline double2 load_pair(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  typedef double d2 __attribute__((ext_vector_type(2)));
  const d2 v = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
  return double2{v.x, v.y};
}

// position within the wave's tile of block i's element c (c < 16)
template <int F, bool CPLX>
__device__ inline int frag_pos(int i, int c) {
  if constexpr (CPLX || F % 2) return i * 16 + c;
  return (i / 2) * 32 + 2 * c + (i & 1);
}

// Fragments of F 16-wide blocks of one operand over a slice of KD rows;
// step t multiplies row k0 + 4 t + lane / 16.
template <int F, int KD, bool CPLX>
struct FragLoader {
  static constexpr bool PAIR = !CPLX && F % 2 == 0;
  static constexpr int NL = PAIR ? F / 2 : F;          // loads per k-step
  static constexpr uint32_t EB = CPLX ? 16u : 8u;
  struct Frag {
    double v[F][KD / 4][CPLX ? 2 : 1];
  };
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[NL];      // byte offset of the lane's element in slice 0, or kOob
  uint32_t kstep;        // bytes from row k to k + 1
  int kq, K;
  __device__ void setup(const void *base, int64_t ld, int Kseg, int x0, int X, int lane) {
    rs = make_rsrc(base);
    K = Kseg;
    kq = lane >> 4;
    kstep = (uint32_t)ld * EB;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int x = x0 + frag_pos<F, CPLX>(PAIR ? 2 * i : i, lane & 15);
      off[i] = x < X ? (uint32_t)kq * kstep + (uint32_t)x * EB : kOob;
    }
  }
  // loads past K return zeros without touching memory
  __device__ void load(Frag &f, int k0) const {
    const uint32_t s0 = k0 < K ? (uint32_t)k0 * kstep : 0u;   // masked loads keep a small scalar offset
#pragma unroll
    for (int t = 0; t < KD / 4; ++t) {
      const bool ok = k0 + 4 * t + kq < K;
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const uint32_t o = ok ? off[i] : kOob, so = s0 + 4u * t * kstep;
        if constexpr (CPLX) {
          const double2 x = load_pair(rs, o, so);
          f.v[i][t][0] = x.x;
          f.v[i][t][1] = x.y;
        } else if constexpr (PAIR) {
          const double2 x = load_pair(rs, o, so);
          f.v[2 * i][t][0] = x.x;
          f.v[2 * i + 1][t][0] = x.y;
        } else {
          f.v[i][t][0] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, o, so, 0));
        }
      }
    }
  }
};

template <int FM, int FN, int WM, int WN, int WK, int kDepth, bool CPLX>
__global__ __launch_bounds__(64 * WM * WN * WK, FM * FN * (CPLX ? 2 : 1) <= 8 ? 2 : 1) void direct_gemm_f64_kernel(const GemmTile *__restrict__ tiles,
                                                                            const GemmTask *__restrict__ tasks,
                                                                            const GemmSeg *__restrict__ segs,
                                                                            Slots slots, int ntiles) {
  constexpr int KD = CPLX ? 8 : 16;
  constexpr int NP = CPLX ? 2 : 1;
  using LA = FragLoader<FM, KD, CPLX>;
  using LB = FragLoader<FN, KD, CPLX>;
  if ((int)blockIdx.x >= ntiles) return;
  if (slots.skip && *slots.skip) return;   // the Krylov solve has stopped
  const GemmTile tl = tiles[blockIdx.x];
  if (tl.task < 0) return;  // padding slot of the XCD-balanced launch order
  const GemmTask tk = tasks[tl.task];
  const int M = tk.M, N = tk.N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wave / (WM * WN), wmn = wave % (WM * WN);
  const int m0 = tl.m0 + (wmn / WN) * FM * 16, n0 = tl.n0 + (wmn % WN) * FN * 16;

  dbl4 acc[NP][FM][FN];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[p][i][j] = dbl4{0.0, 0.0, 0.0, 0.0};

  typename LA::Frag fa[kDepth];
  typename LB::Frag fb[kDepth];
  for (int s = tk.seg_begin; s < tk.seg_begin + tk.seg_count; ++s) {
    const GemmSeg sg = segs[s];
    const int K = sg.K;
    if (K <= 0) continue;
    LA la;
    LB lb;
    la.setup(slots.p[sg.a_slot] + sg.a_off * NP, sg.lda, K, m0, M, lane);
    lb.setup(slots.p[sg.b_slot] + sg.b_off * NP, sg.ldb, K, n0, N, lane);
    const int ns = ((K + KD - 1) / KD - wk + WK - 1) / WK;   // this wave's slices
    auto fetch = [&](int d, int n) {
      la.load(fa[d], (n * WK + wk) * KD);
      lb.load(fb[d], (n * WK + wk) * KD);
      // keep the slices' loads in order: the wait before a slice's MFMAs then
      // leaves the later slices' loads in flight
      __builtin_amdgcn_sched_barrier(0);
    };
    // a slice's MFMAs; its k-steps from `left` on are past K (the last slice of
    // a short K is a good part of it)
    auto multiply = [&](int d, int left) {
#pragma unroll
      for (int t = 0; t < KD / 4; ++t) {
        if (4 * t >= left) break;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const double *a = fa[d].v[i][t], *b = fb[d].v[j][t];
            acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0], b[0], acc[0][i][j], 0, 0, 0);
            if constexpr (CPLX) {
              acc[0][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[1], b[1], acc[0][i][j], 0, 0, 0);
              acc[1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[0], b[1], acc[1][i][j], 0, 0, 0);
              acc[1][i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[1], b[0], acc[1][i][j], 0, 0, 0);
            }
          }
      }
    };
    auto left = [&](int n) { return K - (n * WK + wk) * KD; };
#pragma unroll
    for (int d = 0; d < kDepth; ++d) fetch(d, d);
    int n = 0;
    // straight-line rounds of kDepth slices (an exit inside the round would
    // make the compiler wait for every load at its top), then the rest
    for (; n + 2 * kDepth <= ns; n += kDepth)
#pragma unroll
      for (int d = 0; d < kDepth; ++d) {
        multiply(d, KD);
        fetch(d, n + d + kDepth);
      }
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      if (n + d < ns) multiply(d, left(n + d));
      if (n + d + kDepth < ns) fetch(d, n + d + kDepth);
    }
#pragma unroll
    for (int d = 0; d < kDepth - 1; ++d)
      if (n + d + kDepth < ns) multiply(d, left(n + d + kDepth));
  }

  // output row addresses: a row-address table or a plain row stride
  int64_t crow[FM][4];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + frag_pos<FM, CPLX>(i, (lane >> 4) + 4 * r);
      crow[i][r] = tk.c_rowtab ? slots.crows[tk.c_row + min(row, M - 1)] : tk.c_off + (int64_t)row * tk.ldc;
    }

  if constexpr (WK > 1) {   // sum the k parts, in order
    constexpr int R = NP * FM * FN * 4;
    __shared__ double red[(WK - 1) * WM * WN][R][64];
    if (wk > 0) {
      const int w = (wk - 1) * WM * WN + wmn;
#pragma unroll
      for (int r = 0; r < R; ++r) red[w][r][lane] = acc[r / (FM * FN * 4)][r / (FN * 4) % FM][r / 4 % FN][r % 4];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll 1
    for (int q = 0; q < WK - 1; ++q)
#pragma unroll
      for (int r = 0; r < R; ++r)
        acc[r / (FM * FN * 4)][r / (FN * 4) % FM][r / 4 % FN][r % 4] += red[q * WM * WN + wmn][r][lane];
  }

  double *C = slots.p[tk.c_slot];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + frag_pos<FM, CPLX>(i, (lane >> 4) + 4 * r);
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = n0 + frag_pos<FN, CPLX>(j, lane & 15);
        const int64_t ix = crow[i][r] + col;
        if constexpr (CPLX) {
          if (col < N) reinterpret_cast<double2 *>(C)[ix] = double2{acc[0][i][j][r], acc[1][i][j][r]};
        } else if constexpr (FN % 2 == 0) {   // blocks j, j + 1 hold neighbouring columns
          if (j & 1) continue;
          typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
          if (col + 1 < N)
            *reinterpret_cast<d2u *>(C + ix) = d2u{acc[0][i][j][r], acc[0][i][j + 1][r]};
          else if (col < N)
            C[ix] = acc[0][i][j][r];
        } else {
          if (col < N) C[ix] = acc[0][i][j][r];
        }
      }
    }
}

template <bool CPLX>
static void launch_direct(int bm, int bn, const GemmTile *tiles, const GemmTask *tasks, const GemmSeg *segs,
                          const Slots &slots, int ntiles, hipStream_t st) {
#define QLG_DIRECT(FM_, FN_, WM_, WN_, WK_, D_)                                                               \
  if (bm == FM_ * 16 * WM_ && bn == FN_ * 16 * WN_) {                                                         \
    hipLaunchKernelGGL((direct_gemm_f64_kernel<FM_, FN_, WM_, WN_, WK_, D_, CPLX>), dim3(ntiles),         \
                       dim3(64 * WM_ * WN_ * WK_), 0, st, tiles, tasks, segs, slots, ntiles);                 \
    return;                                                                                                   \
  }
  if constexpr (CPLX) {
    QLG_DIRECT(2, 2, 1, 1, 4, 2)
    QLG_DIRECT(2, 2, 2, 1, 2, 2)
    QLG_DIRECT(2, 2, 1, 2, 2, 2)
    QLG_DIRECT(2, 2, 2, 2, 1, 2)
  } else {
    QLG_DIRECT(2, 2, 1, 1, 4, 2)
    QLG_DIRECT(2, 2, 2, 1, 2, 3)
    QLG_DIRECT(2, 2, 1, 2, 2, 3)
    QLG_DIRECT(2, 2, 2, 2, 1, 3)
    QLG_DIRECT(4, 2, 2, 2, 1, 2)
    QLG_DIRECT(2, 4, 2, 2, 1, 2)
    QLG_DIRECT(4, 4, 2, 2, 1, 2)
    QLG_DIRECT(4, 1, 1, 1, 4, 2)
    QLG_DIRECT(4, 1, 2, 1, 2, 2)
  }
#undef QLG_DIRECT
  throw Error(QLG_ERR_UNSUPPORTED, "unsupported FP64 tile shape");
}

// Complex tiles end at 64 x 64: two accumulator planes of a 128-wide tile leave
// no registers for fragments in flight.  A plan pinned to a wider one
// (QLG_TILES) runs on the LDS kernel, which has it.
bool direct_gemm_shape(int bm, int bn, bool cplx) { return !cplx || (bm <= 64 && bn >= 32 && bn <= 64); }

void launch_direct_gemm_f64(int bm, int bn, bool cplx, const GemmTile *tiles, const GemmTask *tasks,
                            const GemmSeg *segs, const Slots &slots, int ntiles, hipStream_t st) {
  if (ntiles <= 0) return;
  cplx ? launch_direct<true>(bm, bn, tiles, tasks, segs, slots, ntiles, st)
       : launch_direct<false>(bm, bn, tiles, tasks, segs, slots, ntiles, st);
  QLG_HIP(hipGetLastError());
}

// Split-K reduction: every thread sums up to four elements of one task's
// partial panels in part order and writes them where the task's epilogue
// would (row table or row stride).
template <bool CPLX>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const RedTask *__restrict__ red,
                                                            const RedChunk *__restrict__ chunks, Slots slots,
                                                            int nchunks) {
  if ((int)blockIdx.x >= nchunks) return;
  if (slots.skip && *slots.skip) return;   // the Krylov solve has stopped
  const RedChunk ch = chunks[blockIdx.x];
  const RedTask t = red[ch.task];
  const int64_t panel = (int64_t)t.M * t.N;
  const double *W = slots.p[SLOT_W];
  double *C = slots.p[t.c_slot];
#pragma unroll
  for (int j = 0; j < kRedChunk / 256; ++j) {
    const int64_t e = (int64_t)ch.e0 + threadIdx.x + j * 256;
    if (e >= panel || e >= (int64_t)ch.e0 + kRedChunk) break;
    const int64_t r = e / t.N, c = e % t.N;
    const int64_t ix = (t.c_rowtab ? slots.crows[t.c_row + r] - t.c_off : r * t.ldc) + c + t.c_off;
    if constexpr (CPLX) {
      double2 acc = reinterpret_cast<const double2 *>(W)[t.wbase + e];
      for (int q = 1; q < t.parts; ++q) {
        const double2 v = reinterpret_cast<const double2 *>(W)[t.wbase + q * panel + e];
        acc.x += v.x;
        acc.y += v.y;
      }
      reinterpret_cast<double2 *>(C)[ix] = acc;
    } else {
      double acc = W[t.wbase + e];
      for (int q = 1; q < t.parts; ++q) acc += W[t.wbase + q * panel + e];
      C[ix] = acc;
    }
  }
}

void launch_splitk_reduce(bool cplx, const RedTask *red, const RedChunk *chunks, int nchunks, const Slots &slots,
                          hipStream_t st) {
  if (nchunks <= 0) return;
  if (cplx)
    hipLaunchKernelGGL(splitk_reduce_kernel<true>, dim3(nchunks), dim3(256), 0, st, red, chunks, slots, nchunks);
  else
    hipLaunchKernelGGL(splitk_reduce_kernel<false>, dim3(nchunks), dim3(256), 0, st, red, chunks, slots, nchunks);
  QLG_HIP(hipGetLastError());
}

int gemm_bk() {
  static int bk = [] {
    const char *v = std::getenv("QLG_BK");
    return (v && std::atoi(v) == 32) ? 32 : 16;
  }();
  return bk;
}

void launch_grouped_gemm_f64(int bm, int bn, bool cplx, const GemmTile *tiles, const GemmTask *tasks,
                             const GemmSeg *segs, const Slots &slots, int ntiles, hipStream_t st) {
  if (ntiles <= 0) return;
  const int bk = (cplx || bm * bn > 64 * 128) ? 16 : gemm_bk();
  if (cplx)
    launch_shape<true>(bm, bn, bk, tiles, tasks, segs, slots, ntiles, st);
  else
    launch_shape<false>(bm, bn, bk, tiles, tasks, segs, slots, ntiles, st);
  QLG_HIP(hipGetLastError());
}

}  // namespace qlg
