// Linear-solve path on the device: the reference's SolveEquation
// (SolveEquations/AlgebraicSolvers/SolveAlegbraicEquations.for:4) with its
// residual norms, PBCG, Gauss-Seidel and D-ILU solvers, and the Krylov
// solvers that carry the AMG preconditioner.
//
// Layout: every cell-indexed vector is FP64 in HBM; the ELL matrix keeps the
// reference's column-major anb(N,W), so slot j of consecutive cells is one
// contiguous stream and every thread's loads coalesce.  Gathers of x through
// the neighbour table are the only irregular accesses.
//
// Reductions are deterministic: each block reduces with wavefront shuffles in
// a fixed order into its own partial, and a one-block kernel combines the
// partials in index order.  A thread takes one row (four of a large system in
// the kernels that only sum): grids that stopped at
// 8192 workgroups gave some threads of 2.9 M tetrahedra two rows and others
// one, and k_spmv_dot took 66 us instead of 49.  Per
// cell, every sum is formed in the reference's slot order, so a sweep,
// residual or product of one cell is bitwise the reference's.
//
// Convergence never waits for the host: a one-block kernel updates the device
// flags (done, iteration count), and every iteration kernel returns
// immediately once done is set.  The same kernel posts the iteration count
// and done to pinned host memory, and the host launches iterations at most two
// ahead of the last one posted.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <mutex>
#include <stdexcept>

#include "fs_common.h"
#include "fs_kernels.h"
#include "fs_solve.h"

namespace fs {

// ---------------------------------------------------------------- scalars
enum Slot {
  S_IRES = 0, S_FRES, S_RRF, S_BKNUM, S_BKDEN, S_AKDEN, S_BK, S_AK,
  S_RHO, S_ALPHA, S_OMEGA, S_BETA, S_TS, S_TT, S_RV, S_RES_ABS, S_RES_MAX,
  S_RES_RMS, S_RES_SCALED, S_ACPHI, S_GAMMA, S_NSLOTS
};
enum Flag {
  F_DONE = 0, F_ITER = 1, F_ITMAX = 2, F_INNER = 4, F_GATE = 5,
  F_REJECT = 3,  // the initial guess, at the end the iterate, is dropped for zero
  F_BAD = 6,     // the input was refused: 2 = a non-finite ac or bc, 1 = a diagonal <= 0
                 // for a solver that divides by it
  F_NEEDPOS = 7, // set by the host when the solver divides by the diagonal
  F_NFLAGS = 8
};
static_assert(S_NSLOTS <= (int)(sizeof(SolveBox::scal) / sizeof(double)), "scalars of the box");

// The progress word of SolveBox: bit 0 done, bit 1 final (the scalars are
// there as well), bits 2-3 F_BAD, then the iteration count, and the solve's
// number in the upper 32 bits, so that a word of an earlier solve is not
// taken for this one's.
constexpr unsigned long long kBoxDone = 1, kBoxFinal = 2;
__device__ __forceinline__ void post_word(SolveBox *box, unsigned seq, const int *flags, unsigned long long final_bit) {
  const unsigned long long w = ((unsigned long long)seq << 32) | ((unsigned long long)(flags[F_ITER] & 0xfffffff) << 4) |
                               ((unsigned long long)flags[F_BAD] << 2) | final_bit | (flags[F_DONE] ? kBoxDone : 0);
  // the final post publishes the scalars beside it; the others are the word alone
  if (final_bit) __hip_atomic_store(&box->word, w, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  else __hip_atomic_store(&box->word, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
// F_INNER: the GMRES cycle in progress has finished its Arnoldi steps;
// F_GATE = F_DONE | F_INNER, the flag the cycle's kernels (and the V-cycle
// they call) test

constexpr int kFinBlock = 1024; // threads of the one-workgroup finalise kernels (256 where fin() says so)

static inline int grid_for(int n) { return xcd_grid(n); }
// one row per thread up to kPartials workgroups (the row loops of the reducing
// kernels stride by the grid beyond)
static inline int grid_red(int n) { return std::min(kPartials, xcd_grid(n)); }
// Kernels that only sum take four rows per thread, their loads first, from a
// million rows on: the reduction of a workgroup costs as much as its loads
// otherwise.  k_dot, one row against four, 125000 rows 2.80 and 3.08 us, 343000
// 3.40 and 3.44, 512000 3.84 and 3.80, 729000 4.52 and 4.32, 2.9 M 15.4 and 9.0;
// k_init_norms at 2.9 M 36 and 17.  The line lies past the tie, where a solve
// shows the gain (673000 cells of flow 0.5 % in noise of 0.9, 2.9 M rows 4 %).
constexpr int kSumRows = 4, kSumRowsFrom = 1000000;
static inline int sum_rows(int n) { return n >= kSumRowsFrom ? kSumRows : 1; }
static inline int grid_sum(int n) { return grid_red((n + sum_rows(n) - 1) / sum_rows(n)); }

// The Krylov products stream the FP64 matrix (read twice per iteration, too
// large to stay cached beside the vectors): non-temporal matrix loads.
constexpr bool kStreamMatrix = true;

// y = A*x in the order of dsprsax (PBCGMethod.for:324-329): diagonal first,
// then the off-diagonals in slot order.
__device__ __forceinline__ double ell_ax(int i, int n, int w, EllNbr nbr,
                                         const double *__restrict__ ac,
                                         const double *__restrict__ anb,
                                         const double *__restrict__ x) {
  const double s = ld_mat<kStreamMatrix>(&ac[i]) * x[i];
  return ell_fold<kStreamMatrix>(i, n, w, nbr, anb, x, s,
                             [](double acc, double a, double xk) { return acc + a * xk; });
}

// r = b - A*x in the order of CheckConvergence (CheckConvergenceRoutine.for:
// 23-34): b - ac*x first, then each off-diagonal subtracted in slot order.
__device__ __forceinline__ double ell_res(int i, int n, int w, EllNbr nbr,
                                          const double *__restrict__ ac,
                                          const double *__restrict__ anb,
                                          const double *__restrict__ b,
                                          const double *__restrict__ x) {
  const double r = b[i] - ld_mat<kStreamMatrix>(&ac[i]) * x[i];
  return ell_fold<kStreamMatrix>(i, n, w, nbr, anb, x, r,
                             [](double acc, double a, double xk) { return acc - a * xk; });
}

// y = A^T*x in the order of dsprstx (PBCGMethod.for:359-368): diagonal first,
// then the contributions of source rows in increasing row order.  tlin/tsrc
// list, per target cell, the linear anb index and source row of each
// transposed entry, pre-sorted by (row, slot).
// The sources go in batches like the slots of ell_fold: indices, then values
// and gathers, then the terms in order (one at a time, 40 products of 101050
// rows took 60 us more).
template <int B>
__device__ __forceinline__ double ell_atx_by(int i, int n, int wt, const int *__restrict__ tlin,
                                             const int *__restrict__ tsrc, const double *__restrict__ anb,
                                             const double *__restrict__ x, double s) {
  for (int j0 = 0; j0 < wt; j0 += B) {
    int l[B], k[B];
    double a[B], xv[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const size_t q = (size_t)min(j0 + u, wt - 1) * n + i;
      l[u] = tlin[q], k[u] = tsrc[q];
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      a[u] = anb[max(l[u], 0)];
      xv[u] = x[l[u] >= 0 ? k[u] : i];
    }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (j0 + u < wt && l[u] >= 0) s = s + a[u] * xv[u];
  }
  return s;
}
__device__ __forceinline__ double ell_atx(int i, int n, int wt, const int *__restrict__ tlin,
                                          const int *__restrict__ tsrc, const double *__restrict__ ac,
                                          const double *__restrict__ anb, const double *__restrict__ x) {
  const double s = ac[i] * x[i];
  return wt <= 4 ? ell_atx_by<4>(i, n, wt, tlin, tsrc, anb, x, s) : ell_atx_by<6>(i, n, wt, tlin, tsrc, anb, x, s);
}

// ---------------------------------------------------------------- kernels

// Initial residual norms of SolveEquation (CalculateResidualsRoutine.for:
// 19-67) with dphi = 0: r_i = bc_i.  Partials: sum|r|, max|r|, sum r^2,
// max|ac*fit|, and the input check: the largest of 0 (row fine), 1 (ac <= 0)
// and 2 (ac or bc not finite).
template <int ROWS>
__global__ void k_init_norms(int n, const double *__restrict__ ac, const double *__restrict__ bc,
                             const double *__restrict__ fit, double *__restrict__ part) {
  double s1 = 0.0, m1 = -1.0, s2 = 0.0, m2 = -1.0, bad = 0.0;
  for (int i0 = xcd_block() * kBlock * ROWS + threadIdx.x; i0 < n; i0 += gridDim.x * kBlock * ROWS) {
    double a[ROWS], b[ROWS], f[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const int i = min(i0 + u * kBlock, n - 1);
      a[u] = ac[i], b[u] = bc[i], f[u] = fit[i];
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      if (i0 + u * kBlock >= n) break;
      const double r = fabs(b[u]);
      s1 += r;
      m1 = fmax(m1, r);
      s2 += r * r;
      m2 = fmax(m2, fabs(a[u] * f[u]));
      bad = fmax(bad, !(isfinite(a[u]) && isfinite(b[u])) ? 2.0 : (a[u] > 0.0 ? 0.0 : 1.0));
    }
  }
  s1 = block_sum<kBlock>(s1);
  m1 = block_max<kBlock>(m1);
  s2 = block_sum<kBlock>(s2);
  m2 = block_max<kBlock>(m2);
  bad = block_max<kBlock>(bad);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s1;
    part[gridDim.x + blockIdx.x] = m1;
    part[2 * gridDim.x + blockIdx.x] = s2;
    part[3 * gridDim.x + blockIdx.x] = m2;
    part[4 * gridDim.x + blockIdx.x] = bad;
  }
}

// dphi = 0 (SolveAlegbraicEquations.for:47), unless the input was refused
__global__ void k_zero_start(int n, double *__restrict__ x, const int *__restrict__ flags) {
  if (flags[F_BAD]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

// x = 0 by a kernel (no memset node, so the sequence can be graph-captured)
__global__ void k_zero(int n, double *__restrict__ x) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

// L1 norm of the true residual bc - A*x (CheckConvergence).
__global__ void k_resid_l1(int n, int w, EllNbr nbr, const double *__restrict__ ac,
                           const double *__restrict__ anb, const double *__restrict__ b,
                           const double *__restrict__ x, double *__restrict__ part,
                           const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    s += fabs(ell_res(i, n, w, nbr, ac, anb, b, x));
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// r = b - A*x, also copied to r0; partial L1 of r.
// x *= gamma (the L2-optimal scaling of an initial guess)
__global__ void k_warm_scale(int n, double *__restrict__ x, const double *__restrict__ scal,
                             const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = scal[S_GAMMA] * x[i];
}

// a rejected initial guess becomes the zero start: x = 0
__global__ void k_warm_fix(int n, double *__restrict__ x, const int *__restrict__ flags) {
  if (!flags[F_REJECT]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = 0.0;
}

// p = z (first iteration) or z + beta*p
__global__ void k_cg_p(int n, const double *__restrict__ z, double *__restrict__ p,
                       const double *__restrict__ scal, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const bool first = flags[F_ITER] == 0;
  const double be = scal[S_BETA];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = first ? z[i] : z[i] + be * p[i];
}

// x += alpha p, r -= alpha q, partial L1(r)
__global__ void k_cg_update(int n, double *__restrict__ x, double *__restrict__ r,
                            const double *__restrict__ p, const double *__restrict__ q,
                            const double *__restrict__ scal, double *__restrict__ part,
                            const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const double al = scal[S_ALPHA];
  double a = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    x[i] = x[i] + al * p[i];
    const double ri = r[i] - al * q[i];
    r[i] = ri;
    a += fabs(ri);
  }
  a = block_sum<kBlock>(a);
  if (threadIdx.x == 0) part[blockIdx.x] = a;
}

__global__ void k_resid_vec(int n, int w, EllNbr nbr, const double *__restrict__ ac,
                            const double *__restrict__ anb, const double *__restrict__ b,
                            const double *__restrict__ x, double *__restrict__ r,
                            double *__restrict__ r0, double *__restrict__ part) {
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double v = ell_res(i, n, w, nbr, ac, anb, b, x);
    r[i] = v;
    if (r0) r0[i] = v;
    s += fabs(v);
  }
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_spmv(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                       const double *__restrict__ anb, const double *__restrict__ x,
                       double *__restrict__ y) {
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i < n) y[i] = ell_ax(i, n, w, nbr, ac, anb, x);
}

// PBCG start (PBCGMethod.for:147-161): r = bc - A*dphi, rr = r.
__global__ void k_pbcg_start(int n, const double *__restrict__ bc, double *__restrict__ r,
                             double *__restrict__ rr) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    const double v = bc[i] - r[i];
    r[i] = v;
    rr[i] = v;
  }
}

// bknum partials: sum (r*dc)*rr (PBCGMethod.for:163-170).
// z = dc*r (the reference's D-ILU asolve) or, with dc null, the
// preconditioned vector zp given (one AMG V-cycle)
__global__ void k_pbcg_bknum(int n, const double *__restrict__ r, const double *__restrict__ rr,
                             const double *__restrict__ dc, const double *__restrict__ zp,
                             double *__restrict__ part, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    s += (dc ? r[i] * dc[i] : zp[i]) * rr[i];
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// p = bk*p + r*dc, pp = bk*pp + rr*dc; on the first iteration p = r*dc,
// pp = rr*dc (PBCGMethod.for:172-192).
__global__ void k_pbcg_p(int n, const double *__restrict__ r, const double *__restrict__ rr,
                         const double *__restrict__ dc, const double *__restrict__ zp,
                         const double *__restrict__ zzp, double *__restrict__ p,
                         double *__restrict__ pp, const double *__restrict__ scal,
                         const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const double z = dc ? r[i] * dc[i] : zp[i], zz = dc ? rr[i] * dc[i] : zzp[i];
  if (flags[F_ITER] == 0) {
    p[i] = z;
    pp[i] = zz;
  } else {
    const double bk = scal[S_BK];
    p[i] = bk * p[i] + z;
    pp[i] = bk * pp[i] + zz;
  }
}

// z = A*p, zz = A^T*pp, akden partials = sum z*pp (PBCGMethod.for:195-205).
__global__ void k_pbcg_ap(int n, int w, int wt, EllNbr nbr,
                          const int *__restrict__ tlin, const int *__restrict__ tsrc,
                          const double *__restrict__ ac, const double *__restrict__ anb,
                          const double *__restrict__ p, const double *__restrict__ pp,
                          double *__restrict__ z, double *__restrict__ zz,
                          double *__restrict__ part, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double zi = ell_ax(i, n, w, nbr, ac, anb, p);
    z[i] = zi;
    zz[i] = ell_atx(i, n, wt, tlin, tsrc, ac, anb, pp);
    s += zi * pp[i];
  }
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// dphi += ak*p, r -= ak*z, rr -= ak*zz (PBCGMethod.for:207-213), and with dc
// the next iteration's bknum partials (those of k_pbcg_bknum): its launch and
// its finaliser's, two of eight in an iteration, go (101050 hexahedra, 40 iterations: 1.55 -> 1.40
// ms a solve).
__global__ void k_pbcg_axpy(int n, double *__restrict__ dphi, double *__restrict__ r,
                            double *__restrict__ rr, const double *__restrict__ p,
                            const double *__restrict__ z, const double *__restrict__ zz,
                            const double *__restrict__ dc, double *__restrict__ part,
                            const double *__restrict__ scal, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const double ak = scal[S_AK];
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    dphi[i] = dphi[i] + ak * p[i];
    const double ri = r[i] - ak * z[i], rri = rr[i] - ak * zz[i];
    r[i] = ri;
    rr[i] = rri;
    if (dc) s += ri * dc[i] * rri;
  }
  if (!dc) return;
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[gridDim.x + blockIdx.x] = s; // beside the residual's partials
}

// ---- level schedules of the natural-order triangular recurrences (the
// D-ILU diagonal, ILU's forward and backward substitutions).  The cells are
// sorted by dependency level, and everything a recurrence reads or writes is
// kept in that order: position t has up to D terms, term e at [e n + t], each
// naming the position it takes its value from.
//
// A level of a few hundred cells is far too short for a launch of its own
// (3.1-3.5 us each, 183 levels for 86k tetrahedra, 138 for 101k hexahedra),
// so a run of consecutive levels of at most kIluNarrow cells is worked by ONE
// workgroup with a workgroup barrier between the levels: 1.06 us a level, 194
// us a substitution of the tetrahedra instead of 600, 255 us for the
// hexahedra's diagonal instead of 910.  What one CU
// can fetch bounds it, hence the order: in cell order the values a level takes
// lie on a line of memory each (1.7 us a level of 470 tetrahedra, 10 us a
// level of 730 hexahedra with three gathered terms).  A wider level is left to
// a launch over the chip: beyond about 2000 cells one CU's share of the cache
// bandwidth costs more than the launch.
//
// steps: positions in order, each step at most a workgroup wide, twice the
// position plus 1 where a level ends (the dependents start there).  A step's
// own data do not depend on earlier levels and are loaded one step ahead,
// behind the loads of the values that do.
constexpr int kIluNarrow = 2048;
constexpr int kIluThreads = 1024;
constexpr int kIluTerms = 8; // most terms of a cell the runs carry in registers

// out[q] = in[idx[q]] (a vector, or the terms' matrix entries, into an order)
__global__ void k_gather(long long cnt, const int *__restrict__ idx, const double *__restrict__ in,
                         double *__restrict__ out, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const long long q = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (q < cnt) out[q] = in[idx[q]];
}

// x[cell[t]] += y[t]
__global__ void k_scatter_add(int n, const int *__restrict__ cell, const double *__restrict__ y,
                              double *__restrict__ x, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n) return;
  const int c = cell[t];
  x[c] = x[c] + y[t];
}

// The recurrences, position t with right-hand side r, terms (a, b) and the
// values y they take:
//   DIAG   v = r - a y b - ...,  y_t = 1/v: dc_j = 1/(ac_j - sum of
//          anb(j,i) dc_i anb(i,j)), terms in the reference's push order
//          (FactorizeUsingILU.for:23-75 in pull form)
//   FWD    v = r - a y - ...,    y_t = d v, and v kept: rc_j -= anb(j,i) (dc_i rc_i)
//   BWD    v = r - a y - ...,    y_t = d v: rc_i -= anb(i,j) rc_j, rc_i = dc_i rc_i
enum IluOp { ILU_DIAG = 0, ILU_FWD = 1, ILU_BWD = 2 };
struct IluArgs {
  int n;
  const int *src;       // positions of the terms' values, -1: no term
  const double *a, *b;  // the terms' matrix entries (b: DIAG only)
  const double *r, *d;  // right-hand side, D-ILU diagonal (not DIAG)
  double *y, *v;        // results; v: FWD only
};

template <int OP> __device__ __forceinline__ double ilu_term(double v, double a, double y, double b) {
  if constexpr (OP == ILU_DIAG) return v - a * y * b;
  else return v - a * y;
}
template <int OP> __device__ __forceinline__ void ilu_store(const IluArgs &A, int t, double v, double d) {
  A.y[t] = OP == ILU_DIAG ? 1.0 / v : d * v;
  if constexpr (OP == ILU_FWD) A.v[t] = v;
}

template <int OP, int D>
__global__ void __launch_bounds__(kIluThreads)
k_ilu_run(int ns, const int *__restrict__ steps, IluArgs A, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const int *__restrict__ src = A.src;
  const double *__restrict__ ta = A.a, *__restrict__ tb = A.b, *__restrict__ tr = A.r, *__restrict__ td = A.d;
  const double *y = A.y;
  struct Own { // one position's data: nothing earlier levels write
    bool on;
    int i[D];
    double a[D], b[D], r, d;
  };
  auto fetch = [&](int p0, int p1, Own &o) {
    const int t = p0 + (int)threadIdx.x;
    o.on = t < p1;
#pragma unroll
    for (int e = 0; e < D; ++e) o.i[e] = -1;
    if (!o.on) return;
#pragma unroll
    for (int e = 0; e < D; ++e) {
      const size_t q = (size_t)e * A.n + t;
      o.i[e] = src[q];
      o.a[e] = ta[q];
      if constexpr (OP == ILU_DIAG) o.b[e] = tb[q];
    }
    o.r = tr[t];
    if constexpr (OP != ILU_DIAG) o.d = td[t];
  };
  Own cur, nxt;
  int p0 = steps[0] >> 1, end = steps[1], next = ns > 1 ? steps[2] : end;
  fetch(p0, end >> 1, cur);
  for (int s = 0; s < ns; ++s) {
    const int after = s + 3 <= ns ? steps[s + 3] : next;
    double yv[D];
#pragma unroll
    for (int e = 0; e < D; ++e) yv[e] = cur.i[e] >= 0 ? y[cur.i[e]] : 0.0;
    fetch(end >> 1, next >> 1, nxt);
    if (cur.on) {
      double v = cur.r;
#pragma unroll
      for (int e = 0; e < D; ++e)
        if (cur.i[e] >= 0) v = ilu_term<OP>(v, cur.a[e], yv[e], cur.b[e]);
      ilu_store<OP>(A, p0 + (int)threadIdx.x, v, cur.d);
    }
    if (end & 1) __syncthreads();
    cur = nxt;
    p0 = end >> 1;
    end = next;
    next = after;
  }
}

// one wide level: positions p0 .. p1, nt terms
template <int OP>
__global__ void k_ilu_level(int p0, int p1, int nt, IluArgs A, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const int t = p0 + blockIdx.x * kBlock + threadIdx.x;
  if (t >= p1) return;
  double v = A.r[t];
  for (int e = 0; e < nt; ++e) {
    const size_t q = (size_t)e * A.n + t;
    const int i = A.src[q];
    if (i >= 0) v = ilu_term<OP>(v, A.a[q], A.y[i], OP == ILU_DIAG ? A.b[q] : 0.0);
  }
  ilu_store<OP>(A, t, v, OP == ILU_DIAG ? 0.0 : A.d[t]);
}

// One colour of a multicolour Gauss-Seidel sweep: dphi_i = (bc_i - sum
// anb*dphi_nb)/ac_i for the cells of the colour (SORMethod.for:22-36 per cell).
__global__ void k_gs_color(int cnt, const int *__restrict__ cells, int n, int w,
                           EllNbr nbr, const double *__restrict__ ac,
                           const double *__restrict__ anb, const double *__restrict__ bc,
                           double *__restrict__ x, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= cnt) return;
  const int i = cells[t];
  const double s = ell_fold(i, n, w, nbr, anb, (const double *)x, bc[i],
                                       [](double acc, double a, double xk) { return acc - a * xk; });
  x[i] = s / ac[i];
}

// The system in colour order: row t is that of cell cells[t], a colour's rows
// one after the other (ELL as before, the neighbours cell numbers).  In cell
// order a colour's rows are every third or fourth one of an irregular mesh, so
// each colour's launch fetched the lines of the whole matrix.
struct GsRows {
  const int *pos = nullptr, *nbr = nullptr;          // position of a cell; neighbours
  double *ac = nullptr, *anb = nullptr, *bc = nullptr;
};

__global__ void k_gs_rows(int n, int w, const double *__restrict__ ac, const double *__restrict__ anb,
                          const double *__restrict__ bc, GsRows g) {
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i >= n) return;
  const int t = g.pos[i];
  g.ac[t] = ac[i];
  g.bc[t] = bc[i];
  for (int j0 = 0; j0 < w; j0 += 4) {
    double a[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) a[u] = anb[(size_t)min(j0 + u, w - 1) * n + i];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (j0 + u < w) g.anb[(size_t)(j0 + u) * n + t] = a[u];
  }
}

__global__ void k_gs_order(int n, int w, const int *__restrict__ cells, const int *__restrict__ nbr,
                           int *__restrict__ pos, int *__restrict__ out) {
  const int t = xcd_block() * kBlock + threadIdx.x;
  if (t >= n) return;
  const int i = cells[t];
  pos[i] = t;
  for (int j = 0; j < w; ++j) out[(size_t)j * n + t] = nbr[(size_t)j * n + i];
}

// k_gs_color over rows t0 ... t0 + cnt - 1 of the colour order: the same
// values in the same order.
__global__ void k_gs_rows_color(int t0, int cnt, const int *__restrict__ cells, int n, int w, GsRows g,
                                double *__restrict__ x, const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  const int q = xcd_block() * kBlock + threadIdx.x;
  if (q >= cnt) return;
  const int t = t0 + q;
  const double s = ell_fold(t, n, w, EllNbr(g.nbr), (const double *)g.anb, (const double *)x, g.bc[t],
                            [](double acc, double a, double xk) { return acc - a * xk; });
  x[cells[t]] = s / g.ac[t];
}

// ---- generic vector kernels for the Krylov solvers

// partial sums of a*b
template <int ROWS>
__global__ void k_dot(int n, const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ part,
                      const int *__restrict__ flags) {
  if (flags && flags[F_DONE]) return;
  double s = 0.0;
  for (int i0 = xcd_block() * kBlock * ROWS + threadIdx.x; i0 < n; i0 += gridDim.x * kBlock * ROWS) {
    double av[ROWS], bv[ROWS];
#pragma unroll
    for (int u = 0; u < ROWS; ++u) {
      const int i = min(i0 + u * kBlock, n - 1);
      av[u] = a[i], bv[u] = b[i];
    }
#pragma unroll
    for (int u = 0; u < ROWS; ++u)
      if (i0 + u * kBlock < n) s += av[u] * bv[u];
  }
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// BiCGSTAB: p = r + beta*(p - omega*v)
__global__ void k_bicg_p(int n, const double *__restrict__ r, const double *__restrict__ v,
                         double *__restrict__ p, const double *__restrict__ scal,
                         const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  if (flags[F_ITER] == 0) {
    p[i] = r[i];
  } else {
    p[i] = r[i] + scal[S_BETA] * (p[i] - scal[S_OMEGA] * v[i]);
  }
}

// v = A*phat and partial (r0, v)
__global__ void k_spmv_dot(int n, int w, EllNbr nbr, const double *__restrict__ ac,
                           const double *__restrict__ anb, const double *__restrict__ x,
                           double *__restrict__ y, const double *__restrict__ d,
                           double *__restrict__ part, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double yi = ell_ax(i, n, w, nbr, ac, anb, x);
    y[i] = yi;
    s += yi * d[i];
  }
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// s = r - alpha*v
__global__ void k_bicg_s(int n, const double *__restrict__ r, const double *__restrict__ v,
                         double *__restrict__ s, const double *__restrict__ scal,
                         const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) s[i] = r[i] - scal[S_ALPHA] * v[i];
}

// t = A*shat, partials (t,s) and (t,t)
__global__ void k_spmv_dot_ts(int n, int w, EllNbr nbr,
                              const double *__restrict__ ac, const double *__restrict__ anb,
                              const double *__restrict__ x, double *__restrict__ t,
                              const double *__restrict__ s, double *__restrict__ part,
                              const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  double a0 = 0.0, a1 = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double ti = ell_ax(i, n, w, nbr, ac, anb, x);
    t[i] = ti;
    a0 += ti * s[i];
    a1 += ti * ti;
  }
  a0 = block_sum<kBlock>(a0);
  a1 = block_sum<kBlock>(a1);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = a0;
    part[gridDim.x + blockIdx.x] = a1;
  }
}

// x += alpha*phat + omega*shat; r = s - omega*t; partial L1(r)
// x += alpha phat + omega shat, r = s - omega t, with the partials of |r|_1
// and of the next iteration's rho = (r0, r) (the sum k_dot would form)
__global__ void k_bicg_update(int n, double *__restrict__ x, double *__restrict__ r,
                              const double *__restrict__ phat, const double *__restrict__ shat,
                              const double *__restrict__ s, const double *__restrict__ t,
                              const double *__restrict__ r0, const double *__restrict__ scal,
                              double *__restrict__ part, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const double al = scal[S_ALPHA], om = scal[S_OMEGA];
  double a = 0.0, d = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    x[i] = x[i] + al * phat[i] + om * shat[i];
    const double ri = s[i] - om * t[i];
    r[i] = ri;
    a += fabs(ri);
    d += r0[i] * ri;
  }
  a = block_sum<kBlock>(a);
  d = block_sum<kBlock>(d);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = a;
    part[gridDim.x + blockIdx.x] = d;
  }
}

// ---- the reference's ILU iteration (ILUMethod.for:4): rc = bc - A dphi with
// the diagonal first, into the forward substitution's order (pos), then the
// two level-scheduled substitutions with the operation order of the
// sequential loops
__global__ void k_ilu_resid(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                            const double *__restrict__ anb, const double *__restrict__ bc,
                            const double *__restrict__ dphi, const int *__restrict__ pos, double *__restrict__ r,
                            const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i >= n) return;
  r[pos[i]] = ell_fold(i, n, w, nbr, anb, dphi, -ac[i] * dphi[i] + bc[i],
                                  [](double acc, double a, double xk) { return acc - a * xk; });
}

// ---- restarted GMRES with right preconditioning (matrixSolverOMP.f90:48 is
// the reference's GMRES; this one keeps its Krylov basis and Hessenberg
// matrix on the device).  Classical Gram-Schmidt applied twice, all dot
// products FP64 over fixed partials.  gm[] holds the small state:
// H[(m+1) x m] column-major, then cs[m], sn[m], g[m+1], y[m], and the slots
// below.
enum GmSlot { GM_BETA = 0, GM_JEND, GM_TOL2, GM_NSLOT };
inline __host__ __device__ size_t gm_h(int) { return 0; }
inline __host__ __device__ size_t gm_cs(int m) { return (size_t)(m + 1) * m; }
inline __host__ __device__ size_t gm_sn(int m) { return gm_cs(m) + m; }
inline __host__ __device__ size_t gm_g(int m) { return gm_sn(m) + m; }
inline __host__ __device__ size_t gm_y(int m) { return gm_g(m) + m + 1; }
inline __host__ __device__ size_t gm_slot(int m) { return gm_y(m) + m; }
inline __host__ __device__ size_t gm_hpass(int m) { return gm_slot(m) + GM_NSLOT; }
inline __host__ __device__ size_t gm_size(int m) { return gm_hpass(m) + m + 1; }

__global__ void k_gm_spmv(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                          const double *__restrict__ anb, const double *__restrict__ x, double *__restrict__ y,
                          const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i < n) y[i] = ell_ax(i, n, w, nbr, ac, anb, x);
}

// part[j gridDim.x + block] = (V_j, w); blockIdx.y = j
__global__ void k_gm_dots(int n, const double *__restrict__ V, size_t ldv, const double *__restrict__ wv,
                          double *__restrict__ part, const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const double *vj = V + (size_t)blockIdx.y * ldv;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) s += vj[i] * wv[i];
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = s;
}

template <int BS = kFinBlock> __device__ double reduce_partials(const double *part, int np);

// hpass[j] = (V_j, w) from the partials; H[j][col] += hpass[j]; blockIdx.x = j
__global__ void k_gm_hfin(int np, int m, int col, const double *__restrict__ part, double *__restrict__ gm,
                          const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const int j = blockIdx.x;
  const double a = reduce_partials(part + (size_t)j * np, np);
  if (threadIdx.x == 0) {
    gm[gm_hpass(m) + j] = a;
    gm[gm_h(m) + (size_t)col * (m + 1) + j] += a;
  }
}

// w -= sum_{j < nv} hpass[j] V_j
__global__ void k_gm_maxpy(int n, int nv, int m, const double *__restrict__ V, size_t ldv,
                           const double *__restrict__ gm, double *__restrict__ wv, const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double s = wv[i];
  for (int j = 0; j < nv; ++j) s -= gm[gm_hpass(m) + j] * V[(size_t)j * ldv + i];
  wv[i] = s;
}

// partials of (w, w)
__global__ void k_gm_norm2(int n, const double *__restrict__ wv, double *__restrict__ part,
                           const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  double s = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) s += wv[i] * wv[i];
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// Column `col` of the Arnoldi relation: H[col+1][col] = ||w||, the previous
// Givens rotations, a new one, the residual estimate |g[col+1]|; ends the
// cycle's Arnoldi steps when the estimate meets the L2 target, the basis is
// full or w vanished.
__global__ void k_gm_col(int np, int m, int col, const double *__restrict__ part, double *__restrict__ gm,
                         int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const double hn = sqrt(reduce_partials(part, np));
  if (threadIdx.x != 0) return;
  double *H = gm + gm_h(m) + (size_t)col * (m + 1);
  double *cs = gm + gm_cs(m), *sn = gm + gm_sn(m), *g = gm + gm_g(m);
  H[col + 1] = hn;
  for (int i = 0; i < col; ++i) {
    const double a = H[i], b = H[i + 1];
    H[i] = cs[i] * a + sn[i] * b;
    H[i + 1] = -sn[i] * a + cs[i] * b;
  }
  const double a = H[col], b = H[col + 1];
  const double d = sqrt(a * a + b * b);
  const double c = d > 0.0 ? a / d : 1.0, s = d > 0.0 ? b / d : 0.0;
  cs[col] = c;
  sn[col] = s;
  H[col] = d;
  H[col + 1] = 0.0;
  const double gj = g[col];
  g[col] = c * gj;
  g[col + 1] = -s * gj;
  gm[gm_slot(m) + GM_JEND] = col + 1;
  gm[gm_hpass(m) + m] = hn; // the norm for the scaling of the next basis vector
  flags[F_ITER] = flags[F_ITER] + 1;
  if (!(fabs(g[col + 1]) > gm[gm_slot(m) + GM_TOL2]) || col + 1 == m || !(hn > 0.0) ||
      flags[F_ITER] >= flags[F_ITMAX]) {
    flags[F_INNER] = 1;
    flags[F_GATE] = 1;
  }
}

// v = w / ||w|| for the next basis vector
__global__ void k_gm_scale(int n, int m, const double *wv, double *v,
                           const double *__restrict__ gm, const int *__restrict__ flags) {
  if (flags[F_GATE]) return;
  const double inv = 1.0 / gm[gm_hpass(m) + m];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) v[i] = wv[i] * inv;
}

// y = H^{-1} g by back substitution over the cycle's jend columns
__global__ void k_gm_solve(int m, double *__restrict__ gm, const int *__restrict__ flags) {
  if (flags[F_DONE] || threadIdx.x != 0) return;
  const int je = (int)gm[gm_slot(m) + GM_JEND];
  const double *H = gm + gm_h(m), *g = gm + gm_g(m);
  double *y = gm + gm_y(m);
  for (int i = je - 1; i >= 0; --i) {
    double s = g[i];
    for (int k = i + 1; k < je; ++k) s -= H[(size_t)k * (m + 1) + i] * y[k];
    const double d = H[(size_t)i * (m + 1) + i];
    y[i] = d != 0.0 ? s / d : 0.0;
  }
}

// u = sum_{j < jend} y_j V_j
__global__ void k_gm_combine(int n, int m, const double *__restrict__ V, size_t ldv, const double *__restrict__ gm,
                             double *__restrict__ u, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int je = (int)gm[gm_slot(m) + GM_JEND];
  double s = 0.0;
  for (int j = 0; j < je; ++j) s += gm[gm_y(m) + j] * V[(size_t)j * ldv + i];
  u[i] = s;
}

__global__ void k_gm_addx(int n, double *__restrict__ x, const double *__restrict__ z, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = x[i] + z[i];
}

// r = b - A x with L1 and L2 partials
__global__ void k_gm_resid(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                           const double *__restrict__ anb, const double *__restrict__ b,
                           const double *__restrict__ x, double *__restrict__ r, double *__restrict__ part,
                           const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  double s1 = 0.0, s2 = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double v = b[i] - ell_ax(i, n, w, nbr, ac, anb, x);
    r[i] = v;
    s1 += fabs(v);
    s2 += v * v;
  }
  s1 = block_sum<kBlock>(s1);
  s2 = block_sum<kBlock>(s2);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = s1;
    part[gridDim.x + blockIdx.x] = s2;
  }
}

// start of a cycle: the reference's stop rule on the true L1 residual
// (CheckConvergenceRoutine.for semantics: fres <= rrf * ires), then
// beta = ||r||_2, g = (beta, 0, ...), H = 0, and the cycle's L2 target: the
// L2 residual scaled by the L1 reduction still needed, halved for safety
__global__ void k_gm_restart(int np, int m, const double *__restrict__ part, double *__restrict__ gm,
                             double *__restrict__ scal, int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const double l1 = reduce_partials(part, np);
  const double l2 = sqrt(reduce_partials(part + np, np));
  if (threadIdx.x != 0) return;
  scal[S_FRES] = l1;
  const bool done = !(l1 > scal[S_RRF] * scal[S_IRES] && flags[F_ITER] < flags[F_ITMAX]);
  flags[F_DONE] = done;
  flags[F_INNER] = 0;
  flags[F_GATE] = done;
  for (size_t k = 0; k < gm_cs(m); ++k) gm[gm_h(m) + k] = 0.0;
  double *g = gm + gm_g(m);
  g[0] = l2;
  for (int k = 1; k <= m; ++k) g[k] = 0.0;
  gm[gm_slot(m) + GM_BETA] = l2;
  gm[gm_slot(m) + GM_JEND] = 0;
  gm[gm_slot(m) + GM_TOL2] = l1 > 0.0 ? 0.5 * l2 * scal[S_RRF] * scal[S_IRES] / l1 : 0.0;
  if (!(l2 > 0.0)) {
    flags[F_DONE] = 1;
    flags[F_GATE] = 1;
  }
}

// v_0 = r / beta
__global__ void k_gm_v0(int n, int m, const double *__restrict__ r, double *__restrict__ v,
                        const double *__restrict__ gm, const int *__restrict__ flags) {
  if (flags[F_DONE]) return;
  const double inv = 1.0 / gm[gm_slot(m) + GM_BETA];
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) v[i] = r[i] * inv;
}

// ---------------------------------------------------------------- finalisers
enum FinOp {
  FIN_INIT_NORMS = 0, // res4, ires, done-before-start
  FIN_PBCG_BK,        // bknum, bk, bkden
  FIN_PBCG_AK,        // ak
  FIN_CONV,           // fres from partials, iteration count, done
  FIN_BICG_RHO,       // rho, beta
  FIN_BICG_ALPHA,     // alpha = rho/(r0,v)
  FIN_BICG_OMEGA,     // omega = (t,s)/(t,t)
  FIN_TRUE_RES,       // fres, and whether the iterate is dropped
  FIN_CG_RHO,         // rz = (r,z), beta
  FIN_CG_ALPHA,       // alpha = rz/(p,q)
  FIN_WARM,           // reject an initial guess whose L1 residual exceeds ires
  FIN_WARM_SCALE,     // gamma = (A x0, b)/(A x0, A x0)
  FIN_CONV_PBCG_BK,   // FIN_CONV, then (unless done) FIN_PBCG_BK of the next iteration
  FIN_CONV_BICG_RHO,  // FIN_CONV, then (unless done) FIN_BICG_RHO of the next iteration
  FIN_POST            // post the scalars and the final word
};

// what the initial finaliser sets up a solve with, and where it posts
struct SolveStart {
  double rrf;
  int itmax, itmax0; // of the loop; itmax0 < 1: done before it starts
  int needpos;       // the solver divides by the diagonal
  int drop;          // a diverged iterate is dropped at the end (FIN_TRUE_RES)
};
// A Krylov iterate whose true residual ends this many times above |bc|_1, that
// of the zero start, has diverged and is dropped.  A converged flow asks for
// that all the time: its singular p' system has round-off for a source, part of
// it outside the range, so the stop rule cannot be met and BiCGSTAB, CG and
// GMRES run to itmax, in every other solve to a residual above the first one,
// now and then 1e13 times.  Taken as a correction such an iterate threw a flow
// converged to 1e-15 back by up to 0.4, on an occasion that any change in the
// order of a sum moves.
constexpr double kDiverged = 100.0;
struct Post {
  SolveBox *box;
  unsigned seq;
};

// One workgroup of BS threads combines the np partials of a sum: a thread's
// partials i, i + BS, ... are loaded kFinR at a time, then
// folded in index order (the slots past np add +0.0, or take the max with the
// starting -1.0, which changes nothing).
constexpr int kFinR = 8;
template <int BS> struct Partials {
  double v[kFinR];
  __device__ __forceinline__ void load(const double *part, int np, int base) {
#pragma unroll
    for (int u = 0; u < kFinR; ++u) {
      const int i = base + u * BS;
      v[u] = i < np ? part[i] : 0.0;
    }
  }
  // the sum, the first kFinR BS partials being loaded
  __device__ __forceinline__ double sum(const double *part, int np) {
    double s = 0.0;
    for (int base = threadIdx.x;;) {
#pragma unroll
      for (int u = 0; u < kFinR; ++u) s += v[u];
      base += kFinR * BS;
      if (base >= np) break;
      load(part, np, base);
    }
    return block_sum<BS>(s);
  }
};
template <int BS> __device__ double reduce_partials(const double *part, int np) {
  Partials<BS> p;
  p.load(part, np, threadIdx.x);
  return p.sum(part, np);
}
template <int BS> __device__ double reduce_partials_max(const double *part, int np) {
  double s = -1.0;
  for (int base = threadIdx.x; base < np; base += kFinR * BS) {
    double v[kFinR];
#pragma unroll
    for (int u = 0; u < kFinR; ++u) {
      const int i = base + u * BS;
      v[u] = i < np ? part[i] : -1.0;
    }
#pragma unroll
    for (int u = 0; u < kFinR; ++u) s = fmax(s, v[u]);
  }
  return block_max<BS>(s);
}

// What a solve's scalars held before this kernel
struct FinState {
  double rho, alpha, omega, rrf, ires, bknum, bkden;
  int done, iter, itmax;
  __device__ FinState(const double *scal, const int *flags)
      : rho(scal[S_RHO]), alpha(scal[S_ALPHA]), omega(scal[S_OMEGA]), rrf(scal[S_RRF]), ires(scal[S_IRES]),
        bknum(scal[S_BKNUM]), bkden(scal[S_BKDEN]), done(flags[F_DONE]), iter(flags[F_ITER]), itmax(flags[F_ITMAX]) {}
};

// rho = (r0, r) and beta of BiCGSTAB after iter iterations.  Breakdown (rho or
// the last omega zero, or a non-finite beta, as on a singular system whose
// right-hand side carries round-off outside the range): stop with the current
// iterate.
__device__ void bicg_rho(double a, int iter, const FinState &in, double *__restrict__ scal, int *__restrict__ flags) {
  if (iter > 0) {
    const double beta = (a / in.rho) * (in.alpha / in.omega);
    if (in.omega == 0.0 || !isfinite(beta)) {
      flags[F_DONE] = 1;
      return;
    }
    scal[S_BETA] = beta;
  }
  scal[S_RHO] = a;
  if (a == 0.0) flags[F_DONE] = 1;
}

// One workgroup, so it lasts as long as its chain of loads: the solve's
// scalars and the partials are loaded together, and the done flag is tested
// after both.
template <int BS>
__global__ void __launch_bounds__(BS) k_fin(int op, int np, int n, int nf, const double *__restrict__ part,
                      double *__restrict__ scal, int *__restrict__ flags, SolveStart st, Post to) {
  const bool always = op == FIN_INIT_NORMS || op == FIN_TRUE_RES || op == FIN_POST;
  const FinState in(scal, flags);
  const bool two = op == FIN_BICG_OMEGA || op == FIN_WARM_SCALE || op == FIN_CONV_BICG_RHO ||
                   op == FIN_CONV_PBCG_BK;
  Partials<BS> first, second;
  if (op != FIN_POST) {
    first.load(part, np, threadIdx.x);
    if (two) second.load(part + np, np, threadIdx.x);
    in_register(first.v[0]);
  }
  if (!always && in.done) return;
  const double a = op == FIN_POST ? 0.0 : first.sum(part, np);
  double b = 0.0, c = 0.0, d = 0.0, e = 0.0;
  if (op == FIN_INIT_NORMS) {
    b = reduce_partials_max<BS>(part + np, np);
    c = reduce_partials<BS>(part + 2 * np, np);
    d = reduce_partials_max<BS>(part + 3 * np, np);
    e = reduce_partials_max<BS>(part + 4 * np, np);
  } else if (two) {
    b = second.sum(part + np, np);
  }
  if (threadIdx.x != 0) return;
  bool counted = false; // an iteration ended
  switch (op) {
  case FIN_INIT_NORMS: {
    for (int k = 0; k < S_NSLOTS; ++k) scal[k] = 0.0;
    for (int k = 0; k < F_NFLAGS; ++k) flags[k] = 0;
    scal[S_RRF] = st.rrf;
    flags[F_ITMAX] = st.itmax;
    flags[F_NEEDPOS] = st.needpos;
    scal[S_RES_ABS] = a;
    scal[S_RES_MAX] = b;
    scal[S_RES_RMS] = sqrt(c / n);
    scal[S_RES_SCALED] = (nf == 4) ? 0.0 : b / (d + 1.0e-15);
    scal[S_IRES] = a;
    scal[S_FRES] = a;
    flags[F_DONE] = !(a > st.rrf * a && 0 < st.itmax0);
    // refused input: nothing runs, the caller's arrays stay as they were
    flags[F_BAD] = e >= 2.0 ? 2 : (e >= 1.0 && st.needpos) ? 1 : 0;
    if (flags[F_BAD]) flags[F_DONE] = 1;
    counted = true;
    break;
  }
  case FIN_PBCG_BK: {
    scal[S_BKNUM] = a;
    if (in.iter > 0) scal[S_BK] = a / (in.bkden + 1.0e-10);
    scal[S_BKDEN] = a;
    break;
  }
  case FIN_PBCG_AK:
    scal[S_AKDEN] = a;
    scal[S_AK] = in.bknum / (a + 1.0e-10);
    break;
  case FIN_CONV: {
    counted = true;
    scal[S_FRES] = a;
    const int it = in.iter + 1;
    flags[F_ITER] = it;
    // NaN residuals end the loop as well
    flags[F_DONE] = !(a > in.rrf * in.ires && it < in.itmax);
    break;
  }
  case FIN_CONV_PBCG_BK: {
    counted = true;
    scal[S_FRES] = a;
    const int it = in.iter + 1;
    flags[F_ITER] = it;
    const bool more = a > in.rrf * in.ires && it < in.itmax;
    flags[F_DONE] = !more;
    if (more) {
      scal[S_BKNUM] = b;
      scal[S_BK] = b / (in.bkden + 1.0e-10);
      scal[S_BKDEN] = b;
    }
    break;
  }
  case FIN_BICG_RHO:
    bicg_rho(a, in.iter, in, scal, flags);
    break;
  case FIN_CONV_BICG_RHO: {
    counted = true;
    scal[S_FRES] = a;
    const int it = in.iter + 1;
    flags[F_ITER] = it;
    const bool more = a > in.rrf * in.ires && it < in.itmax;
    flags[F_DONE] = !more;
    if (more) bicg_rho(b, it, in, scal, flags);
    break;
  }
  case FIN_BICG_ALPHA:
    scal[S_RV] = a;
    scal[S_ALPHA] = (a != 0.0) ? in.rho / a : 0.0;
    break;
  case FIN_BICG_OMEGA:
    scal[S_TS] = a;
    scal[S_TT] = b;
    scal[S_OMEGA] = (b != 0.0) ? a / b : 0.0;
    break;
  case FIN_TRUE_RES: {
    const bool drop = st.drop && a > kDiverged * in.ires;
    flags[F_REJECT] = drop;
    scal[S_FRES] = drop ? in.ires : a;
    break;
  }
  case FIN_POST:
    break;
  case FIN_CG_RHO: {
    if (in.iter > 0) {
      const double beta = a / in.rho;
      if (!isfinite(beta)) {
        flags[F_DONE] = 1; // breakdown: keep the iterate
        break;
      }
      scal[S_BETA] = beta;
    }
    scal[S_RHO] = a;
    if (a == 0.0) flags[F_DONE] = 1;
    break;
  }
  case FIN_WARM:
    flags[F_REJECT] = !(a <= in.ires);
    break;
  case FIN_WARM_SCALE:
    scal[S_GAMMA] = (b > 0.0 && isfinite(a / b)) ? a / b : 0.0;
    break;
  case FIN_CG_ALPHA: {
    scal[S_RV] = a;
    const double alpha = (a != 0.0) ? in.rho / a : 0.0;
    const bool fine = a != 0.0 && isfinite(alpha);
    scal[S_ALPHA] = fine ? alpha : 0.0;
    if (!fine) flags[F_DONE] = 1;
    break;
  }
  }
  if (op == FIN_POST) {
    for (int k = 0; k < S_NSLOTS; ++k) to.box->scal[k] = scal[k];
    post_word(to.box, to.seq, flags, kBoxFinal);
  } else if (counted || (!always && flags[F_DONE])) {
    post_word(to.box, to.seq, flags, 0);
  }
}

// ---- Gauss-Seidel of a small system in one workgroup
//
// The whole solve after its initial norms: the sweeps of k_gs_color (the same
// values in the same order), the residual and the convergence test of every
// iteration, fit += dphi and the final post.  The iterate lives in LDS and a
// thread's R rows (in colour order, W slots) in registers, so that a colour
// costs its LDS gathers and a barrier instead of a launch and a chain of loads
// from memory.  4096 rows of six slots, two iterations: 18.6 us, where the
// fifteen launches it stands for took about 60.
constexpr int kGsOneThreads = 1024;
constexpr int kGsOneRows = 4 * kGsOneThreads;
constexpr int kGsOneColors = 8;
struct GsColors {
  int n, begin[kGsOneColors + 1];
};

template <int R, int W>
__global__ void __launch_bounds__(kGsOneThreads)
k_gs_one(int n, int w, GsColors col, const int *__restrict__ cells, const int *__restrict__ nbr,
         const double *__restrict__ ac, const double *__restrict__ anb, const double *__restrict__ bc,
         double *__restrict__ dphi, double *__restrict__ fit, double *__restrict__ scal, int *__restrict__ flags,
         Post to) {
  __shared__ double x[R * kGsOneThreads];
  __shared__ int s_more;
  const FinState in(scal, flags);
  const int bad = flags[F_BAD];
  const int tid = threadIdx.x;
  if (bad) { // refused: the caller's arrays stay as they were
    if (tid == 0) {
      for (int k = 0; k < S_NSLOTS; ++k) to.box->scal[k] = scal[k];
      post_word(to.box, to.seq, flags, kBoxFinal);
    }
    return;
  }
  // neighbours as two 16-bit cells; filled slots as bits W r + j of `filled`
  // (a cell may couple to itself: one cell between two periodic patches)
  static_assert(R * W <= 32 && R * kGsOneThreads <= 65536, "packed slots");
  int cell[R], color[R], k2[R][W / 2];
  unsigned filled = 0;
  double a[R][W], d[R], b[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int t = tid + r * kGsOneThreads;
    cell[r] = cells[min(t, n - 1)];
    color[r] = -1;
    for (int c = 0; c < col.n; ++c)
      if (t >= col.begin[c] && t < col.begin[c + 1]) color[r] = c;
    x[t] = 0.0;
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = cell[r];
    d[r] = ac[i], b[r] = bc[i];
    int k[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const size_t q = (size_t)min(j, w - 1) * n + i;
      k[j] = nbr[q], a[r][j] = anb[q];
    }
#pragma unroll
    for (int j = 0; j < W; ++j) {
      if (j < w && k[j] >= 0) filled |= 1u << (W * r + j);
      else k[j] = i;
    }
#pragma unroll
    for (int j = 0; j < W; j += 2) k2[r][j / 2] = k[j] | (k[j + 1] << 16);
  }
  // v - sum a x over the row's neighbours in slot order
  const auto fold = [&](int r, double v) {
    double xk[W];
#pragma unroll
    for (int j = 0; j < W; ++j) xk[j] = x[j & 1 ? (unsigned)k2[r][j / 2] >> 16 : k2[r][j / 2] & 0xffff];
#pragma unroll
    for (int j = 0; j < W; ++j)
      if (filled >> (W * r + j) & 1u) v = v - a[r][j] * xk[j];
    return v;
  };
  const auto sweep = [&](int c) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (color[r] == c) x[cell[r]] = fold(r, b[r]) / d[r];
    __syncthreads();
  };
  __syncthreads();
  int it = 0;
  double res = in.ires;
  if (!in.done)
    for (bool more = true; more;) {
      for (int c = it ? 1 : 0; c < col.n; ++c) sweep(c);
      for (int c = col.n - 2; c >= 0; --c) sweep(c);
      double s = 0.0;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (color[r] >= 0) s += fabs(fold(r, b[r] - d[r] * x[cell[r]]));
      s = block_sum<kGsOneThreads>(s);
      ++it;
      if (tid == 0) {
        res = s;
        s_more = s > in.rrf * in.ires && it < in.itmax; // NaN residuals end the loop as well
      }
      __syncthreads();
      more = s_more;
    }
  for (int i = tid; i < n; i += kGsOneThreads) {
    const double v = x[i];
    dphi[i] = v;
    fit[i] = fit[i] + v;
  }
  if (tid == 0) {
    scal[S_FRES] = res;
    flags[F_ITER] = it;
    flags[F_DONE] = 1;
    for (int k = 0; k < S_NSLOTS; ++k) to.box->scal[k] = scal[k];
    post_word(to.box, to.seq, flags, kBoxFinal);
  }
}

// Whether a Gauss-Seidel solve from zero runs in k_gs_one: whenever the rows
// fit the registers of one workgroup.  Solves of one to six iterations, launches
// against one workgroup: 64 rows 94 and 42 us, 1024 rows 99 and 43, 4096 rows
// 106 and 56 (two iterations), 161 and 68 (six), 3072 tetrahedra 139 and 55.
static bool gs_in_one(int n, int w, int colors) { return n <= kGsOneRows && w <= 6 && colors <= kGsOneColors; }

static void gs_one(fs_mesh *m, const std::vector<int> &begin, const int *cells, const double *ac, const double *anb,
                   const double *bc, double *dphi, double *fit) {
  const int n = m->n, w = m->w;
  GsColors col{(int)begin.size() - 1, {}};
  for (size_t c = 0; c < begin.size(); ++c) col.begin[c] = begin[c];
  const auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kGsOneThreads), 0, m->stream, n, w, col, cells, (const int *)m->d_nbr.p,
                       ac, anb, bc, dphi, fit, m->wk.scal, m->wk.flags, Post{m->box, m->seq});
  };
  if (n <= kGsOneThreads) w <= 4 ? go(k_gs_one<1, 4>) : go(k_gs_one<1, 6>);
  else if (n <= 2 * kGsOneThreads) w <= 4 ? go(k_gs_one<2, 4>) : go(k_gs_one<2, 6>);
  else w <= 4 ? go(k_gs_one<4, 4>) : go(k_gs_one<4, 6>);
}

// ---------------------------------------------------------------- host side

static void precompute_transpose(fs_mesh *m, std::vector<int> &tlin, std::vector<int> &tsrc, int &wt) {
  const int n = m->n, w = m->w;
  std::vector<int> deg(n, 0);
  for (int i = 0; i < n; ++i)
    for (int s = 0; s < m->h_nnbr[i]; ++s) {
      const int k = m->h_nbr[(size_t)s * n + i];
      if (k > 0 && k != i + 1) deg[k - 1]++;
    }
  wt = 1;
  for (int i = 0; i < n; ++i) wt = std::max(wt, deg[i]);
  tlin.assign((size_t)wt * n, -1);
  tsrc.assign((size_t)wt * n, 0);
  std::fill(deg.begin(), deg.end(), 0);
  for (int i = 0; i < n; ++i) // source rows ascending, slots ascending
    for (int s = 0; s < m->h_nnbr[i]; ++s) {
      const int k = m->h_nbr[(size_t)s * n + i];
      if (k > 0 && k != i + 1) {
        const int j = k - 1, t = deg[j]++;
        tlin[(size_t)t * n + j] = s * n + i;
        tsrc[(size_t)t * n + j] = i;
      }
    }
  (void)w;
}

// The order of a level-scheduled recurrence and the pieces it is launched in:
// runs of narrow levels (one workgroup each) and single wide levels.
struct IluPiece {
  int p0, p1;      // positions
  int steps, at;   // a run's step count and where its steps start; steps 0: a wide level
  int threads;     // of a run's workgroup
};
struct IluOrder {
  int terms = 0;   // most terms of a cell
  std::vector<IluPiece> pieces;
  std::vector<int> h_cell, h_pos; // cell of a position, position of a cell
  const int *cell = nullptr, *pos = nullptr, *steps = nullptr;
};

// Host integer arrays that go to the device together: one allocation, one
// copy, one wait.
struct IntPool {
  std::vector<int> h;
  std::vector<std::pair<const int **, size_t>> where;
  DevBuf<int> d;
  void put(const std::vector<int> &v, const int **out) {
    where.push_back({out, h.size()});
    h.insert(h.end(), v.begin(), v.end());
  }
  void upload(hipStream_t s) {
    if (h.empty()) h.push_back(0);
    d.upload(h, s);
    FS_HIP_THROW(hipStreamSynchronize(s)); // h ends here
    for (auto &w : where) *w.first = d.p + w.second;
    std::vector<int>().swap(h);
    where.clear();
  }
};

// Sorts the cells by dependency level (src[ptr[i]..] are the cells that cell i
// waits for; up: higher cells first) and cuts the levels into pieces.
static void ilu_order(fs_mesh *m, const std::vector<int> &ptr, const std::vector<int> &src, bool up, IluOrder &O,
                      IntPool &pool) {
  const int n = m->n;
  std::vector<int> level(n, 0), level_ptr, cells(n, 0);
  int maxl = 0;
  O.terms = 0;
  for (int q = 0; q < n; ++q) {
    const int i = up ? n - 1 - q : q; // dependencies are processed first
    int l = 0;
    for (int t = ptr[i]; t < ptr[i + 1]; ++t) l = std::max(l, level[src[t]] + 1);
    level[i] = l;
    maxl = std::max(maxl, l);
    O.terms = std::max(O.terms, ptr[i + 1] - ptr[i]);
  }
  level_ptr.assign(maxl + 2, 0);
  for (int i = 0; i < n; ++i) level_ptr[level[i] + 1]++;
  for (int l = 0; l <= maxl; ++l) level_ptr[l + 1] += level_ptr[l];
  std::vector<int> fill(level_ptr.begin(), level_ptr.end() - 1), steps;
  for (int i = 0; i < n; ++i) cells[fill[level[i]]++] = i;
  O.pieces.clear();
  for (int l = 0; l <= maxl;) {
    auto width = [&](int k) { return level_ptr[k + 1] - level_ptr[k]; };
    IluPiece P{level_ptr[l], level_ptr[l + 1], 0, 0, 0};
    if (width(l) > kIluNarrow || O.terms > kIluTerms) {
      ++l;
    } else {
      int e = l, widest = 0;
      for (; e <= maxl && width(e) <= kIluNarrow; ++e) widest = std::max(widest, width(e));
      P.p1 = level_ptr[e];
      P.threads = std::min(kIluThreads, (widest + 63) / 64 * 64);
      P.at = (int)steps.size();
      steps.push_back(2 * P.p0);
      for (; l < e; ++l)
        for (int p = level_ptr[l]; p < level_ptr[l + 1]; p += P.threads) {
          const int q = std::min(p + P.threads, level_ptr[l + 1]);
          steps.push_back(2 * q + (q == level_ptr[l + 1] ? 1 : 0));
        }
      P.steps = (int)steps.size() - P.at - 1;
    }
    O.pieces.push_back(P);
  }
  if (steps.empty()) steps.push_back(0);
  O.h_pos.assign(n, 0);
  for (int t = 0; t < n; ++t) O.h_pos[cells[t]] = t;
  O.h_cell = std::move(cells);
  pool.put(O.h_cell, &O.cell);
  pool.put(O.h_pos, &O.pos);
  pool.put(steps, &O.steps);
}

// terms a position of an order has room for: what its kernel (4, 6 or 8
// terms, or any number a level at a time) reads
static int ilu_width(const IluOrder &O) {
  const int nt = std::max(O.terms, 1);
  return nt <= 4 ? 4 : nt <= 6 ? 6 : std::max(nt, kIluTerms);
}

// list[ptr[cell of t] + e] at [e n + t], through map if given; absent terms
// get `none`
static void ilu_terms(fs_mesh *m, const IluOrder &O, const std::vector<int> &ptr, const std::vector<int> &list,
                      const int *map, int none, IntPool &pool, const int **out) {
  const int n = m->n;
  std::vector<int> h((size_t)ilu_width(O) * n, none);
  for (int t = 0; t < n; ++t) {
    const int c = O.h_cell[t];
    for (int q = ptr[c]; q < ptr[c + 1]; ++q) h[(size_t)(q - ptr[c]) * n + t] = map ? map[list[q]] : list[q];
  }
  pool.put(h, out);
}

// The schedule of the D-ILU diagonal: emulates the loops of
// FactorizeUsingILU.for:29-75 to list, per cell, the terms of its diagonal in
// the order the reference applies them.
struct IluDiag {
  bool ready = false;
  IluOrder order;
  const int *ta = nullptr, *ti = nullptr, *tb = nullptr; // the terms' anb entries and positions
  double *a = nullptr, *b = nullptr, *r = nullptr, *y = nullptr; // those entries, ac and the result in the order
  IntPool ints;
  DevBuf<double> mem;
};

static void precompute_ilu(fs_mesh *m, IluDiag &F) {
  const int n = m->n, w = m->w;
  const size_t total = (size_t)n * w;
  std::vector<int> to, A0, I0, B0; // the terms as the loops reach them, and their cells
  for (int i1 = 1; i1 <= n; ++i1) {
    if (i1 == n - 1) continue; // FactorizeUsingILU.for:36
    const int i3 = m->h_nnbr[i1 - 1];
    for (int j2 = 1; j2 <= i3; ++j2) {
      const int j4 = m->h_nbr[(size_t)(j2 - 1) * n + (i1 - 1)];
      if (!(j4 > i1 && j4 <= n)) continue;
      const int j3 = m->h_nnbr[j4 - 1];
      int i2 = 0, i4 = -1;
      while (i2 <= j3 && i4 != i1) {
        i2 = i2 + 1;
        const size_t lin = (size_t)(i2 - 1) * n + (j4 - 1);
        i4 = lin < total ? m->h_nbr[lin] : 0;
      }
      if (i4 == i1) {
        to.push_back(j4 - 1);
        A0.push_back((i2 - 1) * n + (j4 - 1));
        I0.push_back(i1 - 1);
        B0.push_back((j2 - 1) * n + (i1 - 1));
      }
    }
  }
  // by cell, each cell's terms in the order reached
  std::vector<int> ptr(n + 1, 0), A(to.size()), I(to.size()), B(to.size());
  for (int j : to) ptr[j + 1]++;
  for (int j = 0; j < n; ++j) ptr[j + 1] += ptr[j];
  std::vector<int> at(ptr.begin(), ptr.end() - 1);
  for (size_t q = 0; q < to.size(); ++q) {
    const int k = at[to[q]]++;
    A[k] = A0[q];
    I[k] = I0[q];
    B[k] = B0[q];
  }
  ilu_order(m, ptr, I, false, F.order, F.ints);
  ilu_terms(m, F.order, ptr, A, nullptr, 0, F.ints, &F.ta);
  ilu_terms(m, F.order, ptr, I, F.order.h_pos.data(), -1, F.ints, &F.ti);
  ilu_terms(m, F.order, ptr, B, nullptr, 0, F.ints, &F.tb);
  F.ints.upload(m->stream);
  const size_t nt = (size_t)ilu_width(F.order) * n;
  F.mem.alloc(2 * nt + 2 * (size_t)n);
  F.a = F.mem.p;
  F.b = F.a + nt;
  F.r = F.b + nt;
  F.y = F.r + n;
  F.ready = true;
}

// Greedy colouring in cell order: each cell takes the smallest colour not
// used by an already coloured neighbour.
void greedy_colors(int n, int w, const int *nbr0, std::vector<int> &ptr, std::vector<int> &cells) {
  std::vector<int> col(n, -1);
  int nc = 0;
  std::vector<int> used;
  for (int i = 0; i < n; ++i) {
    used.assign(nc + 1, 0);
    for (int j = 0; j < w; ++j) {
      const int k = nbr0[(size_t)j * n + i];
      if (k >= 0 && col[k] >= 0) used[col[k]] = 1;
    }
    int c = 0;
    while (c < nc && used[c]) ++c;
    col[i] = c;
    if (c == nc) ++nc;
  }
  ptr.assign(nc + 1, 0);
  for (int i = 0; i < n; ++i) ptr[col[i] + 1]++;
  for (int c = 0; c < nc; ++c) ptr[c + 1] += ptr[c];
  cells.resize(n);
  std::vector<int> fill(ptr.begin(), ptr.end() - 1);
  for (int i = 0; i < n; ++i) cells[fill[col[i]]++] = i;
}

// Level-scheduled triangular sweeps of the reference's ILU iteration
// (ILUMethod.for:45-140): per cell the contributions in the reference's
// order, cells grouped in dependency levels.
struct IluSweep {
  bool ready = false;
  struct Half {
    IluOrder order;
    const int *src = nullptr, *lin = nullptr; // the terms' positions and anb entries
    const int *from_diag = nullptr;           // position in the diagonal's order
    double *a = nullptr, *r = nullptr, *d = nullptr, *y = nullptr; // entries, right-hand side, diagonal, result
  } fwd, bwd;
  const int *fwd_of_bwd = nullptr;            // position in the forward order of each backward one
  double *v = nullptr;                        // the forward result
  IntPool ints;
  DevBuf<double> mem;
};

struct SolveWork {
  IluDiag diag;
  IluSweep ilu;
  int gm_m = 0;
  DevBuf<double> gm_V, gm_state, gm_part;
  int wt = 1;
  DevBuf<int> tlin, tsrc;
  std::vector<int> color_ptr;
  DevBuf<int> color_cells;
  bool gs_rows = false;   // Gauss-Seidel reads its rows in colour order (gs_by_rows()):
  DevBuf<int> gs_ints;    // the buffers of GsRows
  DevBuf<double> gs_vals;
  GsRows gs;
  DevBuf<double> dc;
};

static SolveWork &work(fs_mesh *m) {
  static_assert(sizeof(SolveWork) > 0, "");
  return *reinterpret_cast<SolveWork *>(m->solve_work);
}

// Lists of the forward substitution (ILUMethod.for:45-93: rc(j) -=
// anb(j, slot of i) * dc(i) * rc(i) for the lower neighbours i of j, i
// increasing) and of the backward one (:97-138: rc(i) -= anb(i, j2) * rc(j)
// for the upper neighbours j of i in slot order), with their levels.
static void precompute_ilu_sweep(fs_mesh *m, const IluDiag &diag, IluSweep &S) {
  const int n = m->n;
  const std::vector<int> &nb = m->h_nbr, &nn = m->h_nnbr;
  std::vector<std::vector<int>> flin(n), fsrc(n);
  for (int i1 = 1; i1 <= n; ++i1) {
    for (int j2 = 1; j2 <= nn[i1 - 1]; ++j2) {
      const int j1 = nb[(size_t)(j2 - 1) * n + (i1 - 1)];
      if (!(j1 != 0 && j1 > i1 && j1 <= n)) continue;
      const int j3 = nn[j1 - 1];
      int i2 = 0, k = 0;
      while (i2 + 1 <= j3 && k != i1) {
        i2 = i2 + 1;
        k = nb[(size_t)(i2 - 1) * n + (j1 - 1)];
      }
      if (k != 0 && k == i1) {
        flin[j1 - 1].push_back((i2 - 1) * n + (j1 - 1));
        fsrc[j1 - 1].push_back(i1 - 1);
      }
    }
  }
  std::vector<int> fptr(n + 1, 0), fl, fs, bptr(n + 1, 0), bl, bs;
  for (int j = 0; j < n; ++j) {
    fptr[j + 1] = fptr[j] + (int)flin[j].size();
    fl.insert(fl.end(), flin[j].begin(), flin[j].end());
    fs.insert(fs.end(), fsrc[j].begin(), fsrc[j].end());
  }
  for (int i1 = 1; i1 <= n; ++i1) {
    if (i1 < n)
      for (int j2 = 1; j2 <= nn[i1 - 1]; ++j2) {
        const int j = nb[(size_t)(j2 - 1) * n + (i1 - 1)];
        if (j > i1) {
          bl.push_back((j2 - 1) * n + (i1 - 1));
          bs.push_back(j - 1);
        }
      }
    bptr[i1] = (int)bl.size();
  }
  auto half = [&](IluSweep::Half &H, const std::vector<int> &ptr, const std::vector<int> &lin,
                  const std::vector<int> &src, bool up) {
    ilu_order(m, ptr, src, up, H.order, S.ints);
    ilu_terms(m, H.order, ptr, src, H.order.h_pos.data(), -1, S.ints, &H.src);
    ilu_terms(m, H.order, ptr, lin, nullptr, 0, S.ints, &H.lin);
    std::vector<int> from(n);
    for (int t = 0; t < n; ++t) from[t] = diag.order.h_pos[H.order.h_cell[t]];
    S.ints.put(from, &H.from_diag);
  };
  half(S.fwd, fptr, fl, fs, false);
  half(S.bwd, bptr, bl, bs, true);
  std::vector<int> fb(n);
  for (int t = 0; t < n; ++t) fb[t] = S.fwd.order.h_pos[S.bwd.order.h_cell[t]];
  S.ints.put(fb, &S.fwd_of_bwd);
  S.ints.upload(m->stream);
  const size_t nf = (size_t)ilu_width(S.fwd.order) * n, nb2 = (size_t)ilu_width(S.bwd.order) * n;
  S.mem.alloc(nf + nb2 + 7 * (size_t)n);
  double *at = S.mem.p;
  for (IluSweep::Half *H : {&S.fwd, &S.bwd}) {
    H->a = at;
    H->r = H->a + (H == &S.fwd ? nf : nb2);
    H->d = H->r + n;
    H->y = H->d + n;
    at = H->y + n;
  }
  S.v = at;
  S.ready = true;
}

// Whether Gauss-Seidel copies its system into colour order (one pass over the
// matrix, read and written) and then reads a colour's rows from there: with
// three colours and more, on rows that overflow the L2s.  A solve of about
// three iterations in cell order and in colour order, four colours of
// tetrahedra: 105456 rows 187 and 191 us, 235824 rows 235 and 193, 663552 rows
// 337 and 271, 2919840 rows 920 and 650.  With the two colours of hexahedra a
// colour reads its half of the lines twice at worst and the copy pays little:
// 262144 rows 154 and 158 us, 2048383 rows 450 and 433.
constexpr size_t kGsRowsSlots = 800000;
static bool gs_by_rows(int n, int w, int colors) { return colors >= 3 && (size_t)n * w >= kGsRowsSlots; }

// The buffers of a system in colour order, and its neighbours.
static void prepare_gs_rows(fs_mesh *m, SolveWork &sw) {
  const size_t n = m->n, w = m->w;
  sw.gs_ints.alloc((w + 1) * n);
  sw.gs_vals.alloc((w + 2) * n);
  int *ip = sw.gs_ints.p;
  double *vp = sw.gs_vals.p;
  hipLaunchKernelGGL(k_gs_order, dim3(grid_for(m->n)), dim3(kBlock), 0, m->stream, m->n, m->w, sw.color_cells.p,
                     m->d_nbr.p, ip, ip + n);
  sw.gs = GsRows{ip, ip + n, vp, vp + 2 * n, vp + n};
}

int mesh_prepare_solver(fs_mesh *m) {
  auto *sw = new SolveWork();
  m->solve_work = sw;
  std::vector<int> tlin, tsrc;
  precompute_transpose(m, tlin, tsrc, sw->wt);
  sw->tlin.upload(tlin, m->stream);
  sw->tsrc.upload(tsrc, m->stream);
  // the solve without allocation may ask for the D-ILU diagonal; a larger
  // mesh schedules it with its first PBCG or ILU solve
  if (m->n <= FS_NOALLOC_MAX_CELLS) precompute_ilu(m, sw->diag);
  std::vector<int> nbr0((size_t)m->n * m->w);
  for (size_t t = 0; t < nbr0.size(); ++t) nbr0[t] = m->h_nbr_dev[t];
  std::vector<int> cells;
  greedy_colors(m->n, m->w, nbr0.data(), sw->color_ptr, cells);
  sw->color_cells.upload(cells, m->stream);
  // (a mesh numbered colour by colour is in that order as it is)
  sw->gs_rows = gs_by_rows(m->n, m->w, (int)sw->color_ptr.size() - 1) && !std::is_sorted(cells.begin(), cells.end());
  // the solve without allocation may ask for the rows; a larger mesh gets them
  // with its first Gauss-Seidel solve (a flow's pressure mesh never: 68 bytes a
  // tetrahedron)
  if (sw->gs_rows && m->n <= FS_NOALLOC_MAX_CELLS) prepare_gs_rows(m, *sw);
  sw->dc.alloc(m->n);
  for (auto &v : m->v) v.alloc(m->n);
  m->partial.alloc(5 * kPartials);
  m->scal.alloc(S_NSLOTS);
  m->flags.alloc(F_NFLAGS);
  FS_HIP_THROW(hipHostMalloc((void **)&m->box, sizeof(SolveBox), hipHostMallocDefault));
  memset(m->box, 0, sizeof(SolveBox));
  for (int k = 0; k < 12; ++k) m->wk.v[k] = m->v[k].p;
  m->wk.dc = sw->dc.p;
  m->wk.partial = m->partial.p;
  m->wk.scal = m->scal.p;
  m->wk.flags = m->flags.p;
  m->nnz = 0;
  for (int i = 0; i < m->n; ++i)
    for (int j = 0; j < m->w; ++j)
      if (m->h_nbr_dev[(size_t)j * m->n + i] >= 0) ++m->nnz;
  FS_HIP_THROW(hipStreamSynchronize(m->stream));
  return 0;
}

int kernel_clock_start(fs_mesh *m, int site_mask, int capacity) {
  KernelClock &c = m->kclock;
  const int valid = (1 << FS_CLOCK_SPMV) | (1 << FS_CLOCK_FINE_SWEEP);
  if (site_mask & ~valid) {
    set_error("fs_kernel_clock_start: unknown site in mask " + std::to_string(site_mask));
    return -1;
  }
  if (site_mask == 0) {
    c.sites = 0;
    return 0;
  }
  if (capacity < 1 || capacity > (1 << 20)) {
    set_error("fs_kernel_clock_start: capacity must lie in [1, 2^20]");
    return -1;
  }
  while ((int)c.ev.size() < 2 * capacity) {
    hipEvent_t e;
    FS_HIP(hipEventCreate(&e));
    c.ev.push_back(e);
  }
  c.sites = site_mask;
  c.cap = capacity;
  c.c = KernelClock::Counts{};
  c.site.assign(capacity, 0);
  c.bytes.assign(capacity, 0.0);
  return 0;
}

int kernel_clock_read(fs_mesh *m, int site, double *out) {
  KernelClock &c = m->kclock;
  if (site < 1 || site > 3) {
    set_error("fs_kernel_clock_read: unknown site " + std::to_string(site));
    return -1;
  }
  FS_HIP(hipStreamSynchronize(m->stream));
  long long k = 0;
  double ms = 0.0, by = 0.0;
  for (int u = 0; u < c.c.used; ++u) {
    if (c.site[u] != site) continue;
    float t = 0.f;
    FS_HIP(hipEventElapsedTime(&t, c.ev[2 * u], c.ev[2 * u + 1]));
    ms += t;
    by += c.bytes[u];
    ++k;
  }
  out[0] = (double)k;
  out[1] = k ? ms / k : 0.0;
  out[2] = k ? by / k : 0.0;
  out[3] = (double)c.c.dropped[site & 3];
  return 0;
}

int kernel_clock_clear(fs_mesh *m) {
  KernelClock &c = m->kclock;
  FS_HIP(hipStreamSynchronize(m->stream));
  c.c = KernelClock::Counts{};
  return 0;
}

int kernel_clock_stride(fs_mesh *m, int stride) {
  if (stride < 1 || stride > 1024) {
    set_error("fs_kernel_clock_stride: stride must lie in [1, 1024]");
    return -1;
  }
  m->kclock.stride = stride;
  for (long long &k : m->kclock.c.seen) k = 0;
  return 0;
}

void kernel_clock_release(fs_mesh *m) {
  for (hipEvent_t e : m->kclock.ev) (void)hipEventDestroy(e);
  m->kclock = KernelClock{};
}

void mesh_release_solver(fs_mesh *m) {
  kernel_clock_release(m);
  delete reinterpret_cast<SolveWork *>(m->solve_work);
  m->solve_work = nullptr;
  if (m->box) (void)hipHostFree(m->box);
  m->box = nullptr;
}

static void gather(fs_mesh *m, size_t cnt, const int *idx, const double *in, double *out, const int *flags = nullptr) {
  if (cnt == 0) return;
  hipLaunchKernelGGL(k_gather, dim3((unsigned)((cnt + kBlock - 1) / kBlock)), dim3(kBlock), 0, m->stream,
                     (long long)cnt, idx, in, out, flags);
}

// a recurrence over its order
template <int OP> static void ilu_pieces(fs_mesh *m, const IluOrder &O, const IluArgs &A, const int *flags) {
  for (const IluPiece &P : O.pieces) {
    if (P.steps == 0) {
      hipLaunchKernelGGL(k_ilu_level<OP>, dim3(grid_for(P.p1 - P.p0)), dim3(kBlock), 0, m->stream, P.p0, P.p1, O.terms,
                         A, flags);
      continue;
    }
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(1), dim3(P.threads), 0, m->stream, P.steps, O.steps + P.at, A,
                         flags);
    };
    if (O.terms <= 4) run(k_ilu_run<OP, 4>);
    else if (O.terms <= 6) run(k_ilu_run<OP, 6>);
    else run(k_ilu_run<OP, kIluTerms>);
  }
}

// D-ILU diagonal on the device (exact reference order), in its schedule's
// order in F.y and, with dc, in cell order
static void ilu_factor(fs_mesh *m, const double *ac, const double *anb, double *dc) {
  IluDiag &F = work(m).diag;
  if (!F.ready) precompute_ilu(m, F);
  const IluOrder &O = F.order;
  const size_t n = m->n, nt = (size_t)O.terms * n;
  gather(m, nt, F.ta, anb, F.a);
  gather(m, nt, F.tb, anb, F.b);
  gather(m, n, O.cell, ac, F.r);
  ilu_pieces<ILU_DIAG>(m, O, IluArgs{m->n, F.ti, F.a, F.b, F.r, nullptr, F.y, nullptr}, nullptr);
  if (dc) gather(m, n, O.pos, F.y, dc);
}

// the matrix and the diagonal in the orders of the two substitutions
static void ilu_pack(fs_mesh *m, const double *anb) {
  SolveWork &sw = work(m);
  for (IluSweep::Half *H : {&sw.ilu.fwd, &sw.ilu.bwd}) {
    gather(m, (size_t)H->order.terms * m->n, H->lin, anb, H->a);
    gather(m, m->n, H->from_diag, sw.diag.y, H->d);
  }
}

// one ILU iteration from the residual in the forward order (fwd.r):
// dphi += U^-1 L^-1 r
static void ilu_apply(fs_mesh *m, double *dphi, const int *flags) {
  IluSweep &S = work(m).ilu;
  IluSweep::Half &f = S.fwd, &b = S.bwd;
  ilu_pieces<ILU_FWD>(m, f.order, IluArgs{m->n, f.src, f.a, nullptr, f.r, f.d, f.y, S.v}, flags);
  gather(m, m->n, S.fwd_of_bwd, S.v, b.r, flags);
  ilu_pieces<ILU_BWD>(m, b.order, IluArgs{m->n, b.src, b.a, nullptr, b.r, b.d, b.y, nullptr}, flags);
  hipLaunchKernelGGL(k_scatter_add, dim3(grid_for(m->n)), dim3(kBlock), 0, m->stream, m->n, b.order.cell, b.y, dphi,
                     flags);
}

static void fin(fs_mesh *m, FinOp op, int np, int nf, SolveStart st = SolveStart{}) {
  // few partials: a workgroup of 256 starts and reduces sooner (396 partials, with
  // the plain posts: 4.1 us a launch in workgroups of 1024, 2.7 in 256)
  const bool few = np <= 256 * kFinR;
  hipLaunchKernelGGL(few ? k_fin<256> : k_fin<kFinBlock>, dim3(1), dim3(few ? 256 : kFinBlock), 0, m->stream, (int)op, np,
                     m->n, nf, m->wk.partial, m->wk.scal, m->wk.flags, st, Post{m->box, m->seq});
}

static void host_flags(fs_mesh *m, int *fl) {
  FS_HIP_THROW(hipMemcpyAsync(fl, m->wk.flags, sizeof(int) * F_NFLAGS, hipMemcpyDeviceToHost, m->stream));
  FS_HIP_THROW(hipStreamSynchronize(m->stream));
}

// The progress of the solve in flight as posted so far (0: nothing yet).
static unsigned long long box_word(const fs_mesh *m) {
  const unsigned long long w = __atomic_load_n(&m->box->word, __ATOMIC_ACQUIRE);
  return (unsigned)(w >> 32) == m->seq ? w : 0;
}
static int box_iterations(unsigned long long w) { return (int)(w >> 4 & 0xfffffff); }
static int box_bad(unsigned long long w) { return (int)(w >> 2 & 3); }

bool solve_done(const fs_mesh *m) { return box_word(m) & kBoxDone; }

// Waits for a post that pred accepts.  Ends with the stream in any case: the
// stream is asked now and then, and a stream that has failed, or has nothing
// left to run that could post, raises an error.
template <class P> static unsigned long long box_wait(fs_mesh *m, P pred) {
  for (unsigned long long w;;) {
    for (int k = 0; k < 2000; ++k) {
      if (pred(w = box_word(m))) return w;
#if defined(__x86_64__)
      __builtin_ia32_pause();
#endif
    }
    const hipError_t e = hipStreamQuery(m->stream);
    if (e == hipErrorNotReady) {
      (void)hipGetLastError();
      continue;
    }
    FS_HIP_THROW(e);
    if (pred(w = box_word(m))) return w;
    throw std::runtime_error("the stream ended without the solve's post");
  }
}

unsigned long long box_wait_final(fs_mesh *m) {
  return box_wait(m, [](unsigned long long w) { return (w & kBoxFinal) != 0; });
}

// Runs `body` until the device posts done, at most itmax times, two iterations
// ahead of the last one posted (at most FS_OPT_CHECK_EVERY - 1), so that the
// stream is never empty; the iterations launched past the last one run idle:
// their kernels return at once, and bodies of many launches stop where they
// see done posted.  One ahead leaves gaps where an iteration takes the host
// as long as the device (24 launches of 3 us on 4096 cells).  Waiting for
// copied flags after batches of the previous solve's iteration count cost a
// synchronisation of about 20 us a batch and up to check_every idle iterations.
template <class F> static void run_iterations(fs_mesh *m, int itmax, F body) {
  const int ahead = std::min(2, m->check_every - 1);
  for (int k = 0; k < itmax; ++k) {
    const unsigned long long w = box_wait(m, [&](unsigned long long v) {
      return (v & kBoxDone) || (v ? box_iterations(v) : -1) + ahead >= k;
    });
    if (w & kBoxDone) break;
    if (m->kclock.sites) m->kclock.before.push_back(m->kclock.c);
    body();
  }
}

// the launches of iterations past the converged one returned at once
static void clock_iterations(fs_mesh *m, int iters) {
  KernelClock &c = m->kclock;
  if (iters < (int)c.before.size()) c.c = c.before[iters];
  c.before.clear();
}

// x0 *= (A x0, b)/(A x0, A x0): the scaling of an initial guess with the
// smallest L2 residual (0 when A x0 = 0), so the guess is never worse than
// a zero start in that norm.  v is scratch.
static void scale_guess(fs_mesh *m, const double *ac, const double *anb, const double *bc, double *x, double *v) {
  const int n = m->n, gr = grid_red(n);
  hipStream_t s = m->stream;
  hipLaunchKernelGGL(k_spmv_dot_ts, dim3(gr), dim3(kBlock), 0, s, n, m->w, EllNbr(m->d_nbr.p, m->d_nbr16.p), ac, anb, x,
                     v, bc, m->wk.partial, m->wk.flags);
  fin(m, FIN_WARM_SCALE, gr, 4);
  hipLaunchKernelGGL(k_warm_scale, dim3(grid_for(n)), dim3(kBlock), 0, s, n, x, m->wk.scal, m->wk.flags);
}

// ---------------------------------------------------------------- projection
// Projection of the right-hand side onto earlier solutions (Fischer, "Projection
// techniques for iterative solution of Ax = b with successive right-hand
// sides", CMAME 163, 1998): x0 = sum_a c_a x_a with the c that minimise
// |b - A x0|_2, i.e. G c = h with G_ab = (A x_a, A x_b), h_a = (A x_a, b).

constexpr int kProjGrid = 2048; // blocks of the Gram pass: 14 partial rows fit the partial buffer

struct ProjVecs {
  const double *p[kProjMax];
};
struct ProjCoef {
  double c[kProjMax];
};

// Partials of the upper triangle of G and of h, row u of the order
// (G_00, h_0, G_01, ..., G_11, h_1, ...) at part[u * gridDim.x + block].
template <int K>
__global__ void __launch_bounds__(kBlock) k_proj_gram(int n, ProjVecs y, const double *__restrict__ b,
                                                      double *__restrict__ part) {
  constexpr int NS = K * (K + 1) / 2 + K;
  double s[NS];
#pragma unroll
  for (int u = 0; u < NS; ++u) s[u] = 0.0;
  for (int i = xcd_block() * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    double v[K];
#pragma unroll
    for (int a = 0; a < K; ++a) v[a] = y.p[a][i];
    const double bi = b[i];
    int u = 0;
#pragma unroll
    for (int a = 0; a < K; ++a) {
#pragma unroll
      for (int c = a; c < K; ++c) s[u++] += v[a] * v[c];
      s[u++] += v[a] * bi;
    }
  }
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const double t = block_sum<kBlock>(s[u]);
    if (threadIdx.x == 0) part[(size_t)u * gridDim.x + blockIdx.x] = t;
  }
}

// extra[u] of the box = sum of row u of the partials, in a fixed order
__global__ void __launch_bounds__(kBlock) k_proj_fin(int ns, int gp, const double *__restrict__ part, Post to) {
  for (int u = 0; u < ns; ++u) {
    double t = 0.0;
    for (int j = threadIdx.x; j < gp; j += kBlock) t += part[(size_t)u * gp + j];
    t = block_sum<kBlock>(t);
    if (threadIdx.x == 0) to.box->extra[u] = t;
  }
  if (threadIdx.x == 0)
    __hip_atomic_store(&to.box->word, ((unsigned long long)to.seq << 32) | kBoxFinal, __ATOMIC_RELEASE,
                       __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ void k_proj_comb(int n, int k, ProjVecs x, ProjCoef c, double *__restrict__ out) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int a = 0; a < k; ++a) s += c.c[a] * x.p[a][i];
  out[i] = s;
}

int project_guess(fs_mesh *m, const double *ac, const double *anb, const double *bc, const double *const *X, int k,
                  double *x0) {
  if (k > kProjMax) k = kProjMax;
  if (k <= 0) return 0;
  const int n = m->n;
  hipStream_t s = m->stream;
  ProjVecs yv{}, xv{};
  for (int a = 0; a < k; ++a) {
    yv.p[a] = m->wk.v[a];
    xv.p[a] = X[a];
    hipLaunchKernelGGL(k_spmv, dim3(grid_for(n)), dim3(kBlock), 0, s, n, m->w, m->d_nbr.p, ac, anb, X[a],
                       m->wk.v[a]);
  }
  const int ns = k * (k + 1) / 2 + k;
  double *part = m->wk.partial;
  switch (k) {
  case 1: hipLaunchKernelGGL(k_proj_gram<1>, dim3(kProjGrid), dim3(kBlock), 0, s, n, yv, bc, part); break;
  case 2: hipLaunchKernelGGL(k_proj_gram<2>, dim3(kProjGrid), dim3(kBlock), 0, s, n, yv, bc, part); break;
  case 3: hipLaunchKernelGGL(k_proj_gram<3>, dim3(kProjGrid), dim3(kBlock), 0, s, n, yv, bc, part); break;
  default: hipLaunchKernelGGL(k_proj_gram<4>, dim3(kProjGrid), dim3(kBlock), 0, s, n, yv, bc, part); break;
  }
  ++m->seq; // a post of its own
  hipLaunchKernelGGL(k_proj_fin, dim3(1), dim3(kBlock), 0, s, ns, kProjGrid, part, Post{m->box, m->seq});
  static_assert(kProjMax * (kProjMax + 1) / 2 + kProjMax <= (int)(sizeof(SolveBox::extra) / sizeof(double)), "Gram sums");
  box_wait_final(m);
  const double *g = m->box->extra;
  double G[kProjMax][kProjMax] = {}, h[kProjMax] = {};
  for (int a = 0, u = 0; a < k; ++a) {
    for (int c = a; c < k; ++c) G[a][c] = G[c][a] = g[u++];
    h[a] = g[u++];
  }
  // Cholesky of G over the vectors in order; a vector whose part outside
  // the span of those before it is below 1e-10 of its norm (or not finite)
  // is left out, so the earliest vectors (the latest solutions) are kept
  double L[kProjMax][kProjMax] = {}, z[kProjMax] = {};
  bool use[kProjMax] = {};
  int used = 0;
  for (int j = 0; j < k; ++j) {
    double d = G[j][j];
    for (int p = 0; p < j; ++p) d -= L[j][p] * L[j][p];
    if (!(G[j][j] > 0.0) || !std::isfinite(G[j][j]) || !(d > 1e-10 * G[j][j])) continue;
    use[j] = true;
    ++used;
    L[j][j] = std::sqrt(d);
    for (int i = j + 1; i < k; ++i) {
      double t = G[i][j];
      for (int p = 0; p < j; ++p) t -= L[i][p] * L[j][p];
      L[i][j] = t / L[j][j];
    }
  }
  for (int j = 0; j < k; ++j) {
    if (!use[j]) continue;
    double t = h[j];
    for (int p = 0; p < j; ++p) t -= L[j][p] * z[p];
    z[j] = t / L[j][j];
  }
  ProjCoef cf{};
  for (int j = k - 1; j >= 0; --j) {
    if (!use[j]) continue;
    double t = z[j];
    for (int i = j + 1; i < k; ++i) t -= L[i][j] * cf.c[i];
    cf.c[j] = t / L[j][j];
  }
  hipLaunchKernelGGL(k_proj_comb, dim3(grid_for(n)), dim3(kBlock), 0, s, n, k, xv, cf, x0);
  return used;
}

int solve_device(fs_mesh *m, int nf, double *fit, double rrf, int itmax, int solver, int lmg,
                 const double *ac, const double *anb, const double *bc, double *dphi, double *res4,
                 fs_solve_stats *st, bool warm, bool sync) {
  const int n = m->n, w = m->w;
  hipStream_t s = m->stream;
  auto t0 = std::chrono::steady_clock::now();
  const int gr = grid_red(n), ge = grid_for(n), gs = grid_sum(n);
  double *part = m->wk.partial, *scal = m->wk.scal;
  int *flags = m->wk.flags;
  const int *nbr = m->d_nbr.p;
  const EllNbr nb(m->d_nbr.p, m->d_nbr16.p); // the row loops of the hot kernels
  SolveWork &sw = work(m);

  if (solver < FS_SOR || solver > FS_CG || solver == FS_DIRECT) {
    set_error("unsupported solver code " + std::to_string(solver) +
              (solver == FS_DIRECT ? " ('direct' is the host's dense LU)" : ""));
    return -3;
  }
  // Gauss-Seidel, D-ILU (also PBCG's preconditioner) and every multigrid
  // smoother divide by the diagonal
  SolveStart start{rrf, lmg == FS_MG_SOLVER ? m->mg_maxcycles : itmax, itmax, 0, 0};
  start.needpos = (lmg != FS_MG_OFF || solver == FS_SOR || solver == FS_ILU || solver == FS_PBCG) ? 1 : 0;
  ++m->seq;
  m->kclock.before.clear();
  const int ncalls_mg = m->ncalls_mg;
  hipLaunchKernelGGL(sum_rows(n) == 1 ? k_init_norms<1> : k_init_norms<kSumRows>, dim3(gs), dim3(kBlock), 0, s, n, ac, bc, fit, part);
  fin(m, FIN_INIT_NORMS, gs, nf, start);
  const bool one = solver == FS_SOR && !warm && lmg != FS_MG_SOLVER && gs_in_one(n, w, (int)sw.color_ptr.size() - 1);
  if (!warm && !one) hipLaunchKernelGGL(k_zero_start, dim3(ge), dim3(kBlock), 0, s, n, dphi, (const int *)flags);
  auto refuse = [](int bad) {
    set_error(bad == 2 ? "a coefficient ac or source bc is not finite"
                       : "a diagonal coefficient ac <= 0, which this solver divides by");
    return bad == 2 ? -4 : -1;
  };
  if (lmg != FS_MG_OFF && amg_will_build(m)) {
    // the hierarchy is built from the operator: refuse bad input before that
    const int bad = box_bad(box_wait(m, [](unsigned long long w) { return w != 0; }));
    if (bad) return refuse(bad);
  }

  double *V0 = m->wk.v[0], *V1 = m->wk.v[1], *V2 = m->wk.v[2], *V3 = m->wk.v[3], *V4 = m->wk.v[4],
         *V5 = m->wk.v[5], *V6 = m->wk.v[6], *V7 = m->wk.v[7];

  // An initial guess, whatever the solver: scaled to its multiple with the
  // smallest L2 residual, then dropped for the zero start when its L1
  // residual still exceeds that of the zero start (|bc|_1).  Every solver
  // below starts from dphi as it stands, so the guess can only change the
  // iteration count, never the stop rule.
  if (warm) {
    scale_guess(m, ac, anb, bc, dphi, V3);
    hipLaunchKernelGGL(k_resid_l1, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, part, flags);
    fin(m, FIN_WARM, gr, nf);
    hipLaunchKernelGGL(k_warm_fix, dim3(ge), dim3(kBlock), 0, s, n, dphi, (const int *)flags);
  }

  if (lmg == FS_MG_SOLVER) {
    amg_solve(m, ac, anb, bc, dphi, solver, warm);
  } else if (solver == FS_PBCG) {
    // r=V0 rr=V1 p=V2 pp=V3 z=V4 zz=V5 (PBCG1.F90:4)
    ilu_factor(m, ac, anb, m->wk.dc);
    hipLaunchKernelGGL(k_spmv, dim3(ge), dim3(kBlock), 0, s, n, w, nbr, ac, anb, dphi, V0);
    hipLaunchKernelGGL(k_pbcg_start, dim3(ge), dim3(kBlock), 0, s, n, bc, V0, V1);
    hipLaunchKernelGGL(k_spmv, dim3(ge), dim3(kBlock), 0, s, n, w, nbr, ac, anb, V0, V1);
    // with FS_MG_PRECOND the D-ILU asolve is replaced by one AMG V-cycle for
    // both r and rr (the transpose preconditioner is the cycle itself: exact
    // for symmetric operators such as p', an approximation otherwise)
    const bool pre = (lmg == FS_MG_PRECOND);
    const double alpha = m->mg_alpha > 0.0 ? m->mg_alpha : 1.7;
    if (pre) amg_prepare(m, ac, anb, alpha);
    const double *dc = pre ? nullptr : m->wk.dc;
    const auto bknum = [&]() {
      hipLaunchKernelGGL(k_pbcg_bknum, dim3(gr), dim3(kBlock), 0, s, n, V0, V1, dc, V6, part, flags);
      fin(m, FIN_PBCG_BK, gr, nf);
    };
    if (!pre) bknum(); // every later one comes with the update
    run_iterations(m, itmax, [&]() {
      if (pre) {
        amg_apply(m, V0, V6, flags, alpha);
        amg_apply(m, V1, V7, flags, alpha);
        bknum();
      }
      hipLaunchKernelGGL(k_pbcg_p, dim3(ge), dim3(kBlock), 0, s, n, V0, V1, dc, V6, V7, V2, V3, scal, flags);
      hipLaunchKernelGGL(k_pbcg_ap, dim3(gr), dim3(kBlock), 0, s, n, w, sw.wt, nb, sw.tlin.p,
                         sw.tsrc.p, ac, anb, V2, V3, V4, V5, part, flags);
      fin(m, FIN_PBCG_AK, gr, nf);
      hipLaunchKernelGGL(k_pbcg_axpy, dim3(gr), dim3(kBlock), 0, s, n, dphi, V0, V1, V2, V4, V5, dc, part, scal, flags);
      hipLaunchKernelGGL(k_resid_l1, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, part, flags);
      fin(m, pre ? FIN_CONV : FIN_CONV_PBCG_BK, gr, nf);
    });
  } else if (one) {
    gs_one(m, sw.color_ptr, sw.color_cells.p, ac, anb, bc, dphi, fit);
  } else if (solver == FS_SOR) {
    // multicolour symmetric Gauss-Seidel: colours forward then backward.  A
    // colour is an independent set, so its update reads only the other
    // colours, and a colour swept twice in a row would recompute the same
    // values bitwise: the backward pass starts at colour nc-2, and every
    // forward pass after the first at colour 1 (the residual check between
    // iterations leaves x alone).
    bool first = true;
    const bool rows = sw.gs_rows;
    if (rows && !sw.gs.pos) prepare_gs_rows(m, sw);
    if (rows) hipLaunchKernelGGL(k_gs_rows, dim3(ge), dim3(kBlock), 0, s, n, w, ac, anb, bc, sw.gs);
    const auto color = [&](int c) {
      const int b = sw.color_ptr[c], e = sw.color_ptr[c + 1];
      if (rows)
        hipLaunchKernelGGL(k_gs_rows_color, dim3(grid_for(e - b)), dim3(kBlock), 0, s, b, e - b, sw.color_cells.p, n, w,
                           sw.gs, dphi, flags);
      else
        hipLaunchKernelGGL(k_gs_color, dim3(grid_for(e - b)), dim3(kBlock), 0, s, e - b, sw.color_cells.p + b, n, w, nb,
                           ac, anb, bc, dphi, flags);
    };
    run_iterations(m, itmax, [&]() {
      const int nc = (int)sw.color_ptr.size() - 1;
      for (int c = first ? 0 : 1; c < nc; ++c) {
        if (solve_done(m)) return; // the rest would return at once
        color(c);
      }
      for (int c = nc - 2; c >= 0; --c) color(c);
      first = false;
      hipLaunchKernelGGL(k_resid_l1, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, part, flags);
      fin(m, FIN_CONV, gr, nf);
    });
  } else if (solver == FS_BICGS) {
    // right-preconditioned BiCGSTAB; r=V0 r0=V1 p=V2 v=V3 s=V4 t=V5 phat=V6 shat=V7
    const bool pre = (lmg == FS_MG_PRECOND);
    const double alpha = m->mg_alpha > 0.0 ? m->mg_alpha : 1.7;
    if (pre) amg_prepare(m, ac, anb, alpha);
    // algorithmic bytes of y = A x with the (r0, y) partials: ac, the
    // neighbour words (4 per slot, or 4 per pair of slots), anb, x, y, r0
    const double ib = nb.d16 ? 4.0 * ((w + 1) / 2) : 4.0 * w;
    const double spmv_bytes = 8.0 * n + ib * n + 8.0 * m->nnz + 24.0 * n;
    hipLaunchKernelGGL(k_resid_vec, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, V0, V1, part);
    hipLaunchKernelGGL(k_zero, dim3(ge), dim3(kBlock), 0, s, n, V3);
    // rho of the first iteration; every later rho comes with the update
    hipLaunchKernelGGL(sum_rows(n) == 1 ? k_dot<1> : k_dot<kSumRows>, dim3(gs), dim3(kBlock), 0, s, n, V1, V0, part, flags);
    fin(m, FIN_BICG_RHO, gs, nf);
    run_iterations(m, itmax, [&]() {
      hipLaunchKernelGGL(k_bicg_p, dim3(ge), dim3(kBlock), 0, s, n, V0, V3, V2, scal, flags);
      if (pre) amg_apply(m, V2, V6, flags, alpha);
      const double *ph = pre ? V6 : V2;
      timed_launch(m, FS_CLOCK_SPMV, spmv_bytes, k_spmv_dot, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, ph,
                   V3, (const double *)V1, part, (const int *)flags);
      fin(m, FIN_BICG_ALPHA, gr, nf);
      if (solve_done(m)) return;
      hipLaunchKernelGGL(k_bicg_s, dim3(ge), dim3(kBlock), 0, s, n, V0, V3, V4, scal, flags);
      if (pre) amg_apply(m, V4, V7, flags, alpha);
      const double *sh = pre ? V7 : V4;
      hipLaunchKernelGGL(k_spmv_dot_ts, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, sh, V5, V4, part, flags);
      fin(m, FIN_BICG_OMEGA, gr, nf);
      hipLaunchKernelGGL(k_bicg_update, dim3(gr), dim3(kBlock), 0, s, n, dphi, V0, ph, sh, V4, V5, (const double *)V1,
                         scal, part, flags);
      fin(m, FIN_CONV_BICG_RHO, gr, nf);
    });
  } else if (solver == FS_CG) {
    // preconditioned conjugate gradient; r=V0 z=V1 p=V2 q=V3
    const bool pre = (lmg == FS_MG_PRECOND);
    const double alpha = m->mg_alpha > 0.0 ? m->mg_alpha : 1.7;
    if (pre) amg_prepare(m, ac, anb, alpha);
    // y = A p with the (p, y) partials: ac, nbr, anb, p, y
    const double spmv_bytes = 8.0 * n + (nb.d16 ? 4.0 * ((w + 1) / 2) : 4.0 * w) * n + 8.0 * m->nnz + 16.0 * n;
    hipLaunchKernelGGL(k_resid_vec, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, V0, nullptr,
                       part);
    run_iterations(m, itmax, [&]() {
      const double *z = V0;
      if (pre) {
        amg_apply(m, V0, V1, flags, alpha);
        z = V1;
      }
      hipLaunchKernelGGL(sum_rows(n) == 1 ? k_dot<1> : k_dot<kSumRows>, dim3(gs), dim3(kBlock), 0, s, n, V0, z, part, flags);
      fin(m, FIN_CG_RHO, gs, nf);
      hipLaunchKernelGGL(k_cg_p, dim3(ge), dim3(kBlock), 0, s, n, z, V2, scal, flags);
      timed_launch(m, FS_CLOCK_SPMV, spmv_bytes, k_spmv_dot, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, V2,
                   V3, (const double *)V2, part, (const int *)flags);
      fin(m, FIN_CG_ALPHA, gr, nf);
      hipLaunchKernelGGL(k_cg_update, dim3(gr), dim3(kBlock), 0, s, n, dphi, V0, V2, V3, scal, part, flags);
      fin(m, FIN_CONV, gr, nf);
    });
  } else if (solver == FS_GMRES) {
    // restarted GMRES(m), right-preconditioned: basis V (m+1 vectors), z = M^-1 v_j
    // (V10), u = V y (V11), r (V0); the cycle ends when its L2 estimate meets the
    // target, the basis is full or itmax is reached; the stop rule is checked on
    // the true L1 residual at every restart
    const bool pre = (lmg == FS_MG_PRECOND);
    const double alpha = m->mg_alpha > 0.0 ? m->mg_alpha : 1.7;
    if (pre) amg_prepare(m, ac, anb, alpha);
    const int gmm = std::max(1, std::min(64, m->gmres_m));
    if (sw.gm_m != gmm || sw.gm_V.n < (size_t)(gmm + 1) * n) {
      sw.gm_V.alloc((size_t)(gmm + 1) * n);
      sw.gm_state.alloc(gm_size(gmm));
      sw.gm_part.alloc((size_t)(gmm + 1) * kPartials);
      sw.gm_m = gmm;
    }
    double *V = sw.gm_V.p, *gm = sw.gm_state.p, *gp = sw.gm_part.p;
    double *Z = m->wk.v[10], *U = m->wk.v[11];
    const size_t ldv = (size_t)n;
    auto restart = [&]() {
      hipLaunchKernelGGL(k_gm_resid, dim3(gr), dim3(kBlock), 0, s, n, w, nbr, ac, anb, bc, dphi, V0, part, flags);
      hipLaunchKernelGGL(k_gm_restart, dim3(1), dim3(kFinBlock), 0, s, gr, gmm, part, gm, scal, flags);
      hipLaunchKernelGGL(k_gm_v0, dim3(ge), dim3(kBlock), 0, s, n, gmm, V0, V, gm, flags);
    };
    restart();
    int fl[F_NFLAGS];
    host_flags(m, fl);
    while (!fl[F_DONE]) {
      for (int j = 0; j < gmm; ++j) {
        const double *vj = V + (size_t)j * ldv;
        double *wv = V + (size_t)(j + 1) * ldv;
        const double *zj = vj;
        if (pre) {
          amg_apply(m, vj, Z, flags + F_GATE, alpha);
          zj = Z;
        }
        hipLaunchKernelGGL(k_gm_spmv, dim3(ge), dim3(kBlock), 0, s, n, w, nbr, ac, anb, zj, wv, flags);
        for (int pass = 0; pass < 2; ++pass) {
          hipLaunchKernelGGL(k_gm_dots, dim3(gr, j + 1), dim3(kBlock), 0, s, n, V, ldv, wv, gp, flags);
          hipLaunchKernelGGL(k_gm_hfin, dim3(j + 1), dim3(kFinBlock), 0, s, gr, gmm, j, gp, gm, flags);
          hipLaunchKernelGGL(k_gm_maxpy, dim3(ge), dim3(kBlock), 0, s, n, j + 1, gmm, V, ldv, gm, wv, flags);
        }
        hipLaunchKernelGGL(k_gm_norm2, dim3(gr), dim3(kBlock), 0, s, n, wv, gp, flags);
        hipLaunchKernelGGL(k_gm_col, dim3(1), dim3(kFinBlock), 0, s, gr, gmm, j, gp, gm, flags);
        hipLaunchKernelGGL(k_gm_scale, dim3(ge), dim3(kBlock), 0, s, n, gmm, wv, wv, gm, flags);
      }
      hipLaunchKernelGGL(k_gm_solve, dim3(1), dim3(64), 0, s, gmm, gm, flags);
      hipLaunchKernelGGL(k_gm_combine, dim3(ge), dim3(kBlock), 0, s, n, gmm, V, ldv, gm, U, flags);
      const double *zu = U;
      if (pre) {
        amg_apply(m, U, Z, flags, alpha);
        zu = Z;
      }
      hipLaunchKernelGGL(k_gm_addx, dim3(ge), dim3(kBlock), 0, s, n, dphi, zu, flags);
      restart();
      host_flags(m, fl);
    }
  } else if (solver == FS_ILU) {
    // the reference's ILU iteration: exact D-ILU diagonal, then per iteration
    // the residual and the two level-scheduled substitutions
    ilu_factor(m, ac, anb, nullptr);
    if (!sw.ilu.ready) precompute_ilu_sweep(m, sw.diag, sw.ilu);
    ilu_pack(m, anb);
    IluSweep &S = sw.ilu;
    run_iterations(m, itmax, [&]() {
      hipLaunchKernelGGL(k_ilu_resid, dim3(ge), dim3(kBlock), 0, s, n, w, nbr, ac, anb, bc, dphi, S.fwd.order.pos,
                         S.fwd.r, flags);
      ilu_apply(m, dphi, flags);
      hipLaunchKernelGGL(k_resid_l1, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, part, flags);
      fin(m, FIN_CONV, gr, nf);
    });
  } else {
    set_error("unsupported solver code " + std::to_string(solver));
    return -3;
  }
  (void)V5;
  (void)V6;
  (void)V7;

  // true final residual, fit += dphi (:180).  The sweeps, ILU and PBCG end on
  // the true residual of the same dphi: formed again it would be the same bits.
  const bool ends_true = lmg != FS_MG_SOLVER && (solver == FS_SOR || solver == FS_ILU || solver == FS_PBCG) && !warm;
  start.drop = lmg != FS_MG_SOLVER && (solver == FS_BICGS || solver == FS_CG || solver == FS_GMRES);
  const auto true_residual = [&]() {
    hipLaunchKernelGGL(k_resid_l1, dim3(gr), dim3(kBlock), 0, s, n, w, nb, ac, anb, bc, dphi, part, nullptr);
    fin(m, FIN_TRUE_RES, gr, nf, start);
  };
  if (!ends_true) true_residual();
  if (!one) {
    add_inplace(m, fit, dphi);
    fin(m, FIN_POST, 0, nf);
  }
  unsigned long long last = box_wait_final(m);
  if (ends_true && box_iterations(last) == 0 && !box_bad(last)) {
    // nothing was iterated, so nothing has looked at anb yet
    ++m->seq;
    true_residual();
    fin(m, FIN_POST, 0, nf);
    last = box_wait_final(m);
  }
  const int iters = box_iterations(last);
  clock_iterations(m, iters);
  // for the caller's own streams and copies: everything above is complete
  if (sync) FS_HIP(hipStreamSynchronize(s));
  if (box_bad(last)) {
    m->ncalls_mg = ncalls_mg; // a refused call does not count towards the next aggregation
    return refuse(box_bad(last));
  }
  const double *h_out = m->box->scal;
  if (res4) {
    res4[0] = h_out[S_RES_ABS];
    res4[1] = h_out[S_RES_MAX];
    res4[2] = h_out[S_RES_RMS];
    res4[3] = h_out[S_RES_SCALED];
  }
  if (st) {
    st->iterations = iters;
    st->levels = (lmg != FS_MG_OFF) ? amg_levels(m) : 1;
    st->initial_l1 = h_out[S_IRES];
    st->final_l1 = h_out[S_FRES];
    st->seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  }
  const bool converged = !(h_out[S_FRES] > rrf * h_out[S_IRES]);
  if (std::isnan(h_out[S_FRES])) {
    set_error("residual is NaN");
    return -4;
  }
  return converged ? 0 : 1;
}

// fit += dphi, unless the input was refused; a dropped dphi becomes zero
__global__ void k_add(int n, double *__restrict__ a, double *__restrict__ b, const int *__restrict__ flags) {
  if (flags[F_BAD]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  if (flags[F_REJECT]) b[i] = 0.0;
  else a[i] = a[i] + b[i];
}

void run_cycles(fs_mesh *m, int np, int itmax, const std::function<void()> &body) {
  run_iterations(m, itmax, [&]() {
    body();
    fin(m, FIN_CONV, np, 4);
  });
}

void add_inplace(fs_mesh *m, double *a, double *b) {
  hipLaunchKernelGGL(k_add, dim3(grid_for(m->n)), dim3(kBlock), 0, m->stream, m->n, a, b, m->wk.flags);
}

} // namespace fs

// ---- kernel timing for the roofline figure: the ELL product y = A*x of the
// Krylov loop (k_spmv_dot), launched reps times between two events on the
// mesh's stream.
namespace fs {
int time_spmv(fs_mesh *m, const double *ac, const double *anb, const double *x, const double *dot_with,
              double *y, int reps, double *avg_ms) {
  const int n = m->n, w = m->w, gr = grid_red(n);
  hipEvent_t e0, e1;
  FS_HIP(hipEventCreate(&e0));
  FS_HIP(hipEventCreate(&e1));
  int h_fl[F_NFLAGS] = {0, 0, 1, 0};
  FS_HIP(hipMemcpyAsync(m->wk.flags, h_fl, sizeof(h_fl), hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_spmv_dot, dim3(gr), dim3(kBlock), 0, m->stream, n, w, EllNbr(m->d_nbr.p, m->d_nbr16.p), ac, anb, x,
                     y, dot_with, m->wk.partial, m->wk.flags);
  FS_HIP(hipEventRecord(e0, m->stream));
  for (int r = 0; r < reps; ++r)
    hipLaunchKernelGGL(k_spmv_dot, dim3(gr), dim3(kBlock), 0, m->stream, n, w, EllNbr(m->d_nbr.p, m->d_nbr16.p), ac, anb,
                       x, y, dot_with, m->wk.partial, m->wk.flags);
  FS_HIP(hipEventRecord(e1, m->stream));
  FS_HIP(hipEventSynchronize(e1));
  float ms = 0.f;
  FS_HIP(hipEventElapsedTime(&ms, e0, e1));
  *avg_ms = ms / reps;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return 0;
}
} // namespace fs

// ---- the solve without allocation: its scratch in one static device array.
// Layout (doubles, every slice 256-byte aligned): 8 work vectors and the D-ILU
// diagonal of kNoallocMaxCells each, the reduction partials, the scalar slots,
// the flags.
namespace fs {
constexpr int kNoallocMaxCells = FS_NOALLOC_MAX_CELLS;
constexpr size_t kNoallocVec = (size_t)kNoallocMaxCells;
constexpr size_t kNoallocPartial = 5 * (size_t)8192;
static_assert(kNoallocMaxCells / kBlock + 8 <= 8192, "partials of the largest mesh without allocation");
constexpr size_t kNoallocScal = 64, kNoallocFlags = 64;
static_assert(S_NSLOTS <= (int)kNoallocScal && F_NFLAGS * sizeof(int) <= kNoallocFlags * sizeof(double),
              "scalar and flag slices");
static_assert(kNoallocVec % 32 == 0 && kNoallocPartial % 32 == 0, "256-byte slices");
constexpr size_t kNoallocDoubles = 9 * kNoallocVec + kNoallocPartial + kNoallocScal + kNoallocFlags;
static_assert(kNoallocDoubles * sizeof(double) == FS_NOALLOC_SCRATCH_BYTES, "size stated in fsamd.h");
} // namespace fs

static __device__ __align__(256) double scratch[fs::kNoallocDoubles];

namespace fs {
// The device address of `scratch` on each device, taken once per device with
// that device current (each GPU holds its own copy of the array).
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[64] = {nullptr};

static double *scratch_on(int dev) {
  if (dev < 0 || dev >= 64) throw std::runtime_error("device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    double *ptr = nullptr;
    FS_HIP_THROW(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) throw std::runtime_error("hipGetSymbolAddress returned no address for the scratch array");
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}

int solve_device_noalloc(fs_mesh *m, int nf, double *fit, double rrf, int itmax, int solver, int lmg,
                         const double *ac, const double *anb, const double *bc, double *dphi, double *res4,
                         fs_solve_stats *st) {
  if (m->n > kNoallocMaxCells) {
    set_error("fs_solve_equation_device_noalloc: " + std::to_string(m->n) + " cells exceed the scratch array's " +
              std::to_string(kNoallocMaxCells));
    return -1;
  }
  if (lmg != FS_MG_OFF) {
    set_error("fs_solve_equation_device_noalloc: LMultigrid must be 0 (the AMG hierarchy is allocated)");
    return -1;
  }
  if (solver != FS_SOR && solver != FS_PBCG && solver != FS_BICGS && solver != FS_CG) {
    set_error("fs_solve_equation_device_noalloc: solver must be SOR, PBCG, BICGS or CG (ILU builds its "
              "substitution schedule and GMRES its basis on first use)");
    return -3;
  }
  int cur = 0;
  FS_HIP(hipGetDevice(&cur));
  if (cur != m->device) {
    set_error("fs_solve_equation_device_noalloc: the mesh's device " + std::to_string(m->device) +
              " is not the current device " + std::to_string(cur));
    return -1;
  }
  double *base = scratch_on(cur);
  fs_mesh::Scratch saved = m->wk, sc{};
  for (int k = 0; k < 8; ++k) sc.v[k] = base + (size_t)k * kNoallocVec;
  for (int k = 8; k < 12; ++k) sc.v[k] = nullptr; // the multigrid and GMRES vectors are not used
  sc.dc = base + 8 * kNoallocVec;
  sc.partial = base + 9 * kNoallocVec;
  sc.scal = sc.partial + kNoallocPartial;
  sc.flags = reinterpret_cast<int *>(sc.scal + kNoallocScal);
  m->wk = sc;
  int rc;
  try {
    rc = solve_device(m, nf, fit, rrf, itmax, solver, lmg, ac, anb, bc, dphi, res4, st, false);
  } catch (...) {
    m->wk = saved;
    throw;
  }
  m->wk = saved;
  return rc;
}
} // namespace fs

extern "C" int fs_solve_equation_device_noalloc(fs_mesh *m, int nf, double *d_fit, double rrf, int itmax, int solver,
                                                int lmultigrid, const double *d_ac, const double *d_anb,
                                                const double *d_bc, double *d_dphi, double *res4,
                                                fs_solve_stats *stats) {
  if (!m || !d_fit || !d_ac || !d_anb || !d_bc || !d_dphi) {
    fs::set_error("fs_solve_equation_device_noalloc: NULL argument");
    return -1;
  }
  try {
    return fs::solve_device_noalloc(m, nf, d_fit, rrf, itmax, solver, lmultigrid, d_ac, d_anb, d_bc, d_dphi, res4,
                                    stats);
  } catch (const std::exception &e) {
    fs::set_error(e.what());
    return -2;
  }
}
