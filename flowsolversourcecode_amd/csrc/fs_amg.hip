// Aggregation algebraic multigrid on the device.
//
// Setup (host, sequential, run once and then every reAgglomorate calls):
// the greedy seed aggregation of AgglomorateALevelAlgebraicly
// (SolveEquations/AlgebraicMultiGrid/AgglomorateALevelAlgebraicly.for:48-331),
// coarse connectivity in the reference's insertion order (:733-787) and the
// level loop of AgglomorateGrid.for:36-44.  The maps are integer and
// bit-exact with the reference's Parents / Children / ElementParent /
// ElementNeighborMG arrays.
//
// Per call (device): Galerkin operators A_c = P^T A P with the reference's
// summation order (AssembleElementBasedAgglomoratedLHS.for:29-150), one
// thread per coarse matrix entry over a precomputed contribution list, so the
// FP64 coarse operators are bitwise the reference's acMG/anbMG.
//
// Cycle (device): the additive-correction V-cycle of MultiGridCycle.for:32-47
// with restriction = sum of member residuals in fine-cell order
// (AssembleNodeAndElementBasedAgglomoratedRHS.for:25-33) and prolongation =
// injection (CorrectSolutionOnFinerLevel.for:17-24), optionally scaled by an
// over-correction factor alpha (FS_OPT_MG_ALPHA; 1 = the reference).  The
// reference's sequential SOR smoother becomes damped Jacobi (or multicolour
// symmetric Gauss-Seidel), so cycle iterates differ while the converged
// solution does not.  Each visit of a coarse level starts from a zero
// correction, the standard V-cycle.  The coarsest level (at most 64 cells) is
// solved directly in FP64.  The hierarchy can be held in FP32
// (FS_OPT_MG_FP32): Galerkin sums stay FP64 and are rounded once to FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cmath>
#include <cstring>
#include <stdexcept>

#include "fs_common.h"
#include "fs_kernels.h"
#include "fs_solve.h"

namespace fs {

namespace {

inline int gfor(int n) { return xcd_grid(n); }

// ------------------------------------------------------------ host setup
struct HostLevel {
  int n = 0, w = 0;
  std::vector<int> nbr;  // 1-based, 0 = none, [j*n + i]
  std::vector<int> nnbr;
  std::vector<double> ac, anb;
  std::vector<int> parent;                 // 1-based, to the next level
  std::vector<int> seed, nchild;           // of this level's aggregates
  std::vector<std::vector<int>> children;  // insertion order
};

int max_children(int ilevel) { // AgglomorateALevelAlgebraicly.for:79-105
  if (ilevel == 2) return 8;
  if (ilevel == 3) return 4;
  if (ilevel == 4) return 3;
  return 2;
}

void finish_level(HostLevel &f, HostLevel &c, const std::vector<int> &parents, const std::vector<int> &seeds,
                  const std::vector<std::vector<int>> &kids, int nc);

void aggregate(HostLevel &f, HostLevel &c, int ilevel) {
  const int nf = f.n, maxch = max_children(ilevel);
  const double ratiomin = 0.5, tiny = 1.0e-15;
  std::vector<double> maxanb(nf);
  for (int i = 0; i < nf; ++i) {
    double m = -1.0;
    for (int j = 0; j < f.nnbr[i]; ++j) m = std::fmax(m, -f.anb[(size_t)j * nf + i]);
    maxanb[i] = m;
  }
  std::vector<int> parents(nf, 0);
  std::vector<std::vector<int>> kids(1);
  std::vector<int> seeds(1, 0);
  int ip = 1;
  for (int s1 = 1; s1 <= nf; ++s1) {
    if (parents[s1 - 1] != 0) continue;
    parents[s1 - 1] = ip;
    if ((int)kids.size() <= ip) {
      kids.resize(ip + 1);
      seeds.resize(ip + 1, 0);
    }
    kids[ip].clear();
    int nb = 0;
    for (int l = 0; l < f.nnbr[s1 - 1]; ++l) {
      const int inb = f.nbr[(size_t)l * nf + s1 - 1];
      if (inb == 0 || parents[inb - 1] != 0) continue;
      const double ratio = -f.anb[(size_t)l * nf + s1 - 1] / std::fmax(maxanb[s1 - 1], tiny);
      if (ratio > ratiomin && nb < maxch) {
        parents[inb - 1] = ip;
        kids[ip].push_back(inb);
        ++nb;
      }
    }
    const int nb2 = nb;
    for (int cl = 0; cl < nb2; ++cl) {
      const int ich = kids[ip][cl];
      for (int l = 0; l < f.nnbr[ich - 1]; ++l) {
        const int inb = f.nbr[(size_t)l * nf + ich - 1];
        if (inb == 0 || parents[inb - 1] != 0) continue;
        const double ratio = -f.anb[(size_t)l * nf + ich - 1] / std::fmax(maxanb[ich - 1], tiny);
        if (ratio > ratiomin && nb < maxch) {
          parents[inb - 1] = ip;
          ++nb;
          kids[ip].push_back(inb);
        }
      }
    }
    if (nb == 0) {
      parents[s1 - 1] = 0;
    } else {
      seeds[ip] = s1;
      ++ip;
    }
  }
  for (int io = 1; io <= nf; ++io) {
    if (parents[io - 1] == 0) {
      double strength = 0.0;
      bool placed = false;
      for (int l = 0; l < f.nnbr[io - 1]; ++l) {
        const int inb = f.nbr[(size_t)l * nf + io - 1];
        if (inb == 0) continue;
        if (parents[inb - 1] != 0 && !placed) {
          const double ratio = -f.anb[(size_t)l * nf + io - 1] / maxanb[inb - 1];
          if (strength < ratio) {
            placed = true;
            strength = ratio;
            const int p = parents[inb - 1];
            parents[io - 1] = p;
            kids[p].push_back(io);
          }
        }
      }
    }
    if (parents[io - 1] == 0) { // isolated orphan: aggregate without a seed
      parents[io - 1] = ip;
      if ((int)kids.size() <= ip) {
        kids.resize(ip + 1);
        seeds.resize(ip + 1, 0);
      }
      kids[ip].clear();
      seeds[ip] = 0;
      ++ip;
    }
  }
  finish_level(f, c, parents, seeds, kids, ip - 1);
}

// The coarse level of an aggregation: parents (1-based) of the fine cells,
// seed and children (in insertion order) of aggregates 1..nc; the coarse
// neighbour lists in the order the fine cells and their slots reach them.
void finish_level(HostLevel &f, HostLevel &c, const std::vector<int> &parents, const std::vector<int> &seeds,
                  const std::vector<std::vector<int>> &kids, int nc) {
  const int nf = f.n;
  std::vector<std::vector<int>> cn(nc + 1);
  int wmax = 1;
  for (int e = 1; e <= nf; ++e)
    for (int l = 0; l < f.nnbr[e - 1]; ++l) {
      const int inb = f.nbr[(size_t)l * nf + e - 1];
      if (inb == 0) continue;
      const int p = parents[e - 1], q = parents[inb - 1];
      if (p == q) continue;
      auto &lst = cn[p];
      if (std::find(lst.begin(), lst.end(), q) == lst.end()) {
        lst.push_back(q);
        wmax = std::max(wmax, (int)lst.size());
      }
    }
  f.parent = parents;
  c.n = nc;
  c.w = wmax;
  c.nbr.assign((size_t)nc * wmax, 0);
  c.nnbr.assign(nc, 0);
  c.seed.assign(nc, 0);
  c.nchild.assign(nc, 0);
  c.children.assign(nc, {});
  for (int p = 1; p <= nc; ++p) {
    c.seed[p - 1] = seeds[p];
    c.children[p - 1] = kids[p];
    c.nchild[p - 1] = (int)kids[p].size();
    c.nnbr[p - 1] = (int)cn[p].size();
    for (size_t k = 0; k < cn[p].size(); ++k) c.nbr[k * nc + p - 1] = cn[p][k];
  }
  c.ac.assign(nc, 0.0);
  c.anb.assign((size_t)nc * wmax, 0.0);
}

// Off-diagonal couplings of a level as compressed rows (the diagonal is not
// needed to judge strength).
struct Couplings {
  int n = 0;
  std::vector<int> rp, col;
  std::vector<double> val;
};

Couplings couplings_of(const HostLevel &f) {
  Couplings A;
  A.n = f.n;
  A.rp.assign(f.n + 1, 0);
  for (int i = 0; i < f.n; ++i) {
    for (int l = 0; l < f.nnbr[i]; ++l) {
      const int j = f.nbr[(size_t)l * f.n + i];
      if (j <= 0) continue;
      A.col.push_back(j - 1);
      A.val.push_back(f.anb[(size_t)l * f.n + i]);
    }
    A.rp[i + 1] = (int)A.col.size();
  }
  return A;
}

// One pass of pairwise matching: each unmatched cell, in order, is paired
// with the unmatched neighbour of its strongest negative coupling among those
// at least `beta` times the row's strongest (Notay's pairwise aggregation);
// a cell without one stays alone.  agg[i] = 0-based pair number.
int pair_pass(const Couplings &A, double beta, std::vector<int> &agg) {
  const int n = A.n;
  agg.assign(n, -1);
  int na = 0;
  for (int i = 0; i < n; ++i) {
    if (agg[i] >= 0) continue;
    double mx = 0.0;
    for (int k = A.rp[i]; k < A.rp[i + 1]; ++k) mx = std::fmax(mx, -A.val[k]);
    int best = -1;
    double bv = 0.0;
    for (int k = A.rp[i]; k < A.rp[i + 1]; ++k) {
      const int j = A.col[k];
      const double sv = -A.val[k];
      if (j == i || agg[j] >= 0 || !(sv > 0.0) || sv < beta * mx) continue;
      if (sv > bv) {
        bv = sv;
        best = j;
      }
    }
    agg[i] = na;
    if (best >= 0) agg[best] = na;
    ++na;
  }
  return na;
}

// The couplings between pairs: the fine couplings summed over pair members,
// those inside a pair dropped.
Couplings pair_couplings(const Couplings &A, const std::vector<int> &agg, int na) {
  std::vector<std::vector<int>> mem(na);
  for (int i = 0; i < A.n; ++i) mem[agg[i]].push_back(i);
  Couplings B;
  B.n = na;
  B.rp.assign(na + 1, 0);
  std::vector<int> where(na, -1);
  std::vector<int> touched;
  for (int p = 0; p < na; ++p) {
    touched.clear();
    for (int i : mem[p])
      for (int k = A.rp[i]; k < A.rp[i + 1]; ++k) {
        const int q = agg[A.col[k]];
        if (q == p) continue;
        if (where[q] < 0) {
          where[q] = (int)B.col.size();
          B.col.push_back(q);
          B.val.push_back(0.0);
          touched.push_back(q);
        }
        B.val[where[q]] += A.val[k];
      }
    for (int q : touched) where[q] = -1;
    B.rp[p + 1] = (int)B.col.size();
  }
  return B;
}

// Aggregation by `passes` pairwise passes (aggregates of up to 2^passes
// cells).  Aggregates are numbered in the order of their first fine cell,
// which is also their seed; the other members follow in increasing order.
void aggregate_pairwise(HostLevel &f, HostLevel &c, int passes) {
  const double beta = 0.25;
  const Couplings A = couplings_of(f);
  std::vector<int> agg;
  int nc = pair_pass(A, beta, agg);
  if (passes > 1) {
    const Couplings B = pair_couplings(A, agg, nc);
    std::vector<int> agg2;
    nc = pair_pass(B, beta, agg2);
    for (int i = 0; i < f.n; ++i) agg[i] = agg2[agg[i]];
  }
  std::vector<int> ren(nc, 0);
  int t = 0;
  std::vector<int> parents(f.n);
  for (int i = 0; i < f.n; ++i) {
    if (ren[agg[i]] == 0) ren[agg[i]] = ++t;
    parents[i] = ren[agg[i]];
  }
  std::vector<int> seeds(nc + 1, 0);
  std::vector<std::vector<int>> kids(nc + 1);
  for (int i = 0; i < f.n; ++i) {
    const int p = parents[i];
    if (seeds[p] == 0) seeds[p] = i + 1;
    else kids[p].push_back(i + 1);
  }
  finish_level(f, c, parents, seeds, kids, nc);
}

// Galerkin contribution lists of level c in the reference's order and the
// host values (for the aggregation of the next level).
void galerkin_lists(const HostLevel &f, HostLevel &c, std::vector<int> &ptr,
                    std::vector<long long> &src) {
  const int nc = c.n, wc = c.w, nf = f.n;
  std::vector<std::vector<long long>> lists((size_t)nc * (wc + 1));
  for (int p = 1; p <= nc; ++p) {
    auto &dl = lists[p - 1];
    double acc = 0.0;
    const int nmem = c.nchild[p - 1] + 1;
    for (int mm = 0; mm < nmem; ++mm) {
      const int e = (mm == 0) ? c.seed[p - 1] : c.children[p - 1][mm - 1];
      if (e <= 0) continue;
      dl.push_back(e - 1);
      acc = acc + f.ac[e - 1];
      for (int l = 0; l < f.nnbr[e - 1]; ++l) {
        const int inb = f.nbr[(size_t)l * nf + e - 1];
        if (inb <= 0) continue;
        const int q = f.parent[inb - 1];
        if (q <= 0) continue;
        const size_t lin = (size_t)l * nf + e - 1;
        const double a = f.anb[lin];
        if (q == p) {
          dl.push_back((long long)nf + (long long)lin);
          acc = acc + a;
        } else {
          for (int k = 0; k < c.nnbr[p - 1]; ++k)
            if (c.nbr[(size_t)k * nc + p - 1] == q) {
              lists[(size_t)nc + (size_t)k * nc + p - 1].push_back((long long)nf + (long long)lin);
              c.anb[(size_t)k * nc + p - 1] = c.anb[(size_t)k * nc + p - 1] + a;
            }
        }
      }
    }
    c.ac[p - 1] = acc;
  }
  ptr.assign(lists.size() + 1, 0);
  src.clear();
  for (size_t e = 0; e < lists.size(); ++e) {
    ptr[e + 1] = ptr[e] + (int)lists[e].size();
    src.insert(src.end(), lists[e].begin(), lists[e].end());
  }
  if (src.empty()) src.push_back(0);
}

// ------------------------------------------------------------ device kernels

// coarse entry e of level c = sum of its contributions (FP64), then stored
// in both precisions when the hierarchy runs in FP32
__global__ void k_galerkin(int ne, int nc, const int *__restrict__ ptr,
                           const int *__restrict__ src, int nf,
                           const double *__restrict__ acf, const double *__restrict__ anbf,
                           double *__restrict__ acc_out, double *__restrict__ anbc,
                           float *__restrict__ ac32, float *__restrict__ anb32,
                           const int *__restrict__ csr_pos, double *__restrict__ val64,
                           float *__restrict__ val32) {
  const int e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= ne) return;
  // contributions in list order, loaded in batches (sources, then values)
  const int t0 = ptr[e], t1 = ptr[e + 1];
  double a = 0.0;
  constexpr int B = 4;
  for (int t = t0; t < t1; t += B) {
    int sv[B];
    double v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) sv[u] = src[min(t + u, t1 - 1)];
#pragma unroll
    for (int u = 0; u < B; ++u) v[u] = sv[u] < nf ? acf[sv[u]] : anbf[sv[u] - nf];
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (t + u < t1) a = a + v[u];
  }
  if (e < nc) {
    acc_out[e] = a;
    if (ac32) ac32[e] = (float)a;
  } else {
    anbc[e - nc] = a;
    if (anb32) anb32[e - nc] = (float)a;
    // the same value at its place in the row-major CSR copy of the level
    const int q = csr_pos[e - nc];
    if (q >= 0) {
      val64[q] = a;
      if (val32) val32[q] = (float)a;
    }
  }
}

template <class T>
__global__ void k_to(int n, const double *__restrict__ a, T *__restrict__ b) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) b[i] = (T)a[i];
}

// ------------------------------------------------------------ cycle kernels
// Grid-wide kernels for the levels above the tail.  Every kernel returns at
// once when the Krylov loop has set its done flag, so the batches launched
// after convergence cost only their launch.

// The level kernels load their matrix as ordinary (cached) data: a level's
// matrix is re-read by every sweep of a cycle and partly stays in the
// Infinity Cache between them (non-temporal loads here took the 128^3 fine
// sweep from 4.7 to 4.1 TB/s).
constexpr bool kStreamLevel = false;

// The done flag, as a load that waits for nothing and is waited for with the
// loads that follow it (a null test around it would wait there); any is any
// readable address of the kernel.
__device__ __forceinline__ int done_flag(const int *flags, const void *any) {
  const int v = *(flags ? flags : (const int *)any);
  return flags ? v : 0;
}

// The prolongation of a level's correction into the next finer level: the
// kernel that forms a coarse cell's value adds alpha times it to the cell's
// members (x[mem[q]], q in [mptr[p], mptr[p+1])).  Every finer cell belongs to
// one coarse cell, so no two threads touch one value, and the sum is that of
// a pass of its own (k_prolong) without that pass's launch (3.4 us, 28 of them
// in the channel's F-cycle), and without the parent lookup of every neighbour
// that forming it in the finer level's first sweep took (finest level of 128^3
// hexahedra: 28.8 us instead of 16.9).  Not on the large levels in sliced
// ELL, whose lanes would each walk a list of their own: 342k cells with 2.0M
// members took 35 us, the plain sweep and k_prolong take 13 and 8.
template <class T> struct Scatter {
  const int *mptr, *mem; // members of the level's cells in the next finer level
  T *x;                  // the finer level's iterate
  T alpha;
};

// A cell's part of the scatter on LPR lanes: the first 16 members' values are
// loaded beside the row's own operands, before the cell's value is known.
template <int LPR, class T> struct ScatterRow {
  static constexpr int B = LPR < 16 ? 16 / LPR : 1;
  int q, q1, id[B];
  T xv[B];
  // begin: the first member of this lane; end: the members' end
  __device__ __forceinline__ void members(const Scatter<T> &sc, int begin, int end) {
    q = begin;
    q1 = end;
#pragma unroll
    for (int u = 0; u < B; ++u) id[u] = sc.mem[min(q + u * LPR, q1 - 1)];
  }
  __device__ __forceinline__ void values(const Scatter<T> &sc) {
#pragma unroll
    for (int u = 0; u < B; ++u) xv[u] = sc.x[id[u]];
  }
  __device__ __forceinline__ void add(const Scatter<T> &sc, T v) {
    const T a = sc.alpha * v;
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (q + u * LPR < q1) sc.x[id[u]] = xv[u] + a;
    for (int k = q + B * LPR; k < q1; k += LPR) {
      const int i = sc.mem[k];
      sc.x[i] = sc.x[i] + a;
    }
  }
};

// sum_j anb_ij x_j over the slots of row i, spread over LPR consecutive
// lanes and combined with shuffles
template <int LPR, class T>
__device__ __forceinline__ T row_offdiag(int i, int lane, int n, int w, EllNbr nbr,
                                         const T *__restrict__ anb, const T *x) {
  if (LPR == 1)
    return ell_fold<kStreamLevel>(i, n, w, nbr, anb, x, T(0), [](T acc, T a, T xk) { return acc + a * xk; });
  T s = T(0);
  for (int j = lane; j < w; j += LPR) {
    const int k = nbr.i32[(size_t)j * n + i];
    if (k >= 0) s += anb[(size_t)j * n + i] * x[k];
  }
#pragma unroll
  for (int off = LPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, LPR);
  return s;
}

// One damped-Jacobi sweep xn = x + omega*(b - A x)/ac of the finest level.
// TO = double writes the FP64 result of the cycle directly.
template <int LPR, class T, class TO>
__global__ void __launch_bounds__(kBlock)
k_sweep(int n, int w, EllNbr nbr, const T *__restrict__ ac, const T *__restrict__ anb,
        const T *__restrict__ b, const T *x, T omega, TO *xn, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int t = xcd_block() * kBlock + threadIdx.x;
  const int i = t / LPR, lane = t % LPR;
  const bool ok = i < n;
  const T s = row_offdiag<LPR, T>(ok ? i : 0, lane, ok ? n : 1, ok ? w : 0, nbr, anb, x);
  if (ok && lane == 0) {
    const T xi = x[i];
    xn[i] = (TO)(xi + omega * (b[i] - ac[i] * xi - s) / ac[i]);
  }
}

// r = b - A x
template <int LPR, class T>
__global__ void __launch_bounds__(kBlock)
k_resid(int n, int w, EllNbr nbr, const T *__restrict__ ac, const T *__restrict__ anb,
        const T *__restrict__ b, const T *__restrict__ x, T *__restrict__ r, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int t = xcd_block() * kBlock + threadIdx.x;
  const int i = t / LPR, lane = t % LPR;
  const bool ok = i < n;
  const T s = row_offdiag<LPR, T>(ok ? i : 0, lane, ok ? n : 1, ok ? w : 0, nbr, anb, x);
  if (ok && lane == 0) r[i] = b[i] - ac[i] * x[i] - s;
}

// ---- coarse levels in row-major CSR (no padding; a row's entries are
// contiguous, so the LPR lanes of a row read one segment)
//
// The levels between the finest and the dense map are too small to use the
// chip's bandwidth: a launch on them lasts as long as its chain of dependent
// loads, about 0.7 us each.  So a row's entries go in batches of kCsrBatch per
// lane (columns and values, then the gathers: one round for up to
// kCsrBatch LPR entries), the done flag is read beside the first loads
// instead of ahead of them, and what a kernel needs after its sum is loaded
// before it.  On the levels of 2.9 M tetrahedra k_resid_restrict_csr went from
// 5.7 to 4.4 us, k_sweep_csr from 4.1 to 3.4 (16 lanes) and from 5.8 to 4.8 (8
// lanes, prolongating), k_dense_apply from 5.1 to 4.6.
constexpr int kCsrBatch = 4;
template <int LPR, class T, class V> struct CsrRow {
  int q, q1, c[kCsrBatch];
  V a[kCsrBatch];
  T xv[kCsrBatch];
  // entries q0 + lane, q0 + lane + LPR, ... of a row's [q0, end)
  __device__ __forceinline__ void entries(int at, int end, const int *__restrict__ col, const V *__restrict__ val) {
    q = at;
    q1 = end;
#pragma unroll
    for (int u = 0; u < kCsrBatch; ++u) {
      const int e = max(min(q + u * LPR, q1 - 1), 0);
      c[u] = col[e];
      a[u] = val[e];
    }
  }
  __device__ __forceinline__ void gather(const T *x) {
#pragma unroll
    for (int u = 0; u < kCsrBatch; ++u) xv[u] = x[c[u]];
  }
  __device__ __forceinline__ T sum(T s) const {
#pragma unroll
    for (int u = 0; u < kCsrBatch; ++u)
      if (q + u * LPR < q1) s += a[u] * xv[u];
    return s;
  }
  // the row's sum on all of its lanes, the first batch being gathered
  __device__ __forceinline__ T finish(const int *__restrict__ col, const V *__restrict__ val, const T *x) {
    T s = sum(T(0));
    while (q + kCsrBatch * LPR < q1) {
      entries(q + kCsrBatch * LPR, q1, col, val);
      gather(x);
      s = sum(s);
    }
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, LPR);
    return s;
  }
};

// SC: the level's last sweep, which also prolongates its result
template <int LPR, class T, bool SC>
__global__ void __launch_bounds__(kBlock)
k_sweep_csr(int n, const int *__restrict__ rp, const int *__restrict__ col, const T *__restrict__ val,
            const T *__restrict__ ac, const T *__restrict__ b, const T *x, T omega, T *xn, Scatter<T> sc,
            const int *__restrict__ flags) {
  const int done = done_flag(flags, rp);
  const int t = xcd_block() * kBlock + threadIdx.x;
  const int i = min(t / LPR, n - 1), lane = t % LPR;
  const bool ok = t / LPR < n;
  int q0 = rp[i], q1 = rp[i + 1], m0 = 0, m1 = 0;
  const T ai = ac[i], bi = b[i], xi = x[i];
  if (SC) m0 = sc.mptr[i], m1 = sc.mptr[i + 1];
  in_register(q0);
  if (done) return;
  CsrRow<LPR, T, T> row;
  ScatterRow<LPR, T> to;
  row.entries(q0 + lane, q1, col, val);
  if (SC) to.members(sc, m0 + lane, m1);
  row.gather(x);
  if (SC) to.values(sc);
  const T s = row.finish(col, val, x);
  if (!ok) return;
  const T v = xi + omega * (bi - ai * xi - s) / ai; // the same on the row's lanes
  if (lane == 0) xn[i] = v;
  if (SC) to.add(sc, v);
}

// ---- large coarse levels in sliced ELL: slices of 64 rows (one wavefront),
// one row per lane, a slice's entries column-major (entry k of the slice's
// lane l at ptr[s] + 64 k + l, so a wavefront's loads of entry k coalesce),
// padded to the slice's longest row with zero values whose column is the row
// itself.  row[] maps a slot to its row (-1: past the end); rows are sorted by
// length within windows of 256 rows so that a slice's rows have similar
// lengths.  Each lane sums its row's entries in CSR order.
// P16: the columns as 16-bit offsets from the row, two entries to a word (entry
// 2p of a lane in the low half of word p, 2p + 1 in the high half, a slice's
// length then even): 6 bytes an FP32 entry instead of 8 on levels that are bound
// by them (a solve on 2.1 M hexahedra 11.10 -> 10.90 ms, on 2.9 M tetrahedra 18.75
// -> 18.40).
template <class T, bool P16>
__device__ __forceinline__ T sell_offdiag(int slot, int lane, int i, const int *__restrict__ ptr,
                                          const int *__restrict__ col, const T *__restrict__ val, const T *x) {
  const int sl = slot >> 6, p0 = ptr[sl], q0 = p0 + lane, len = (ptr[sl + 1] - p0) >> 6;
  constexpr int B = 4; // entries per batch: columns first, then values and gathers
  T s = T(0);
  for (int k0 = 0; k0 < len; k0 += B) {
    int c[B];
    T v[B], xv[B];
    if (P16) {
#pragma unroll
      for (int u = 0; u < B; u += 2) {
        const int w = col[(p0 >> 1) + lane + (min((k0 + u) >> 1, (len >> 1) - 1) << 6)];
        c[u] = i + (short)(w & 0xffff);
        c[u + 1] = i + (w >> 16);
      }
    } else {
#pragma unroll
      for (int u = 0; u < B; ++u) c[u] = col[q0 + (min(k0 + u, len - 1) << 6)];
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
      v[u] = val[q0 + (min(k0 + u, len - 1) << 6)];
      xv[u] = x[c[u]];
    }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (k0 + u < len) s += v[u] * xv[u];
  }
  return s;
}

template <class T, bool P16>
__global__ void __launch_bounds__(kBlock)
k_sweep_sell(int nslots, const int *__restrict__ ptr, const int *__restrict__ row, const int *__restrict__ col,
             const T *__restrict__ val, const T *__restrict__ ac, const T *__restrict__ b, const T *x, T omega, T *xn,
             const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int t = xcd_block() * kBlock + threadIdx.x;
  if (t >= nslots) return;
  const int i = row[t];
  if (i < 0) return;
  const T s = sell_offdiag<T, P16>(t, t & 63, i, ptr, col, val, x);
  const T xi = x[i];
  xn[i] = xi + omega * (b[i] - ac[i] * xi - s) / ac[i];
}

// r = b - A x on a sliced-ELL level
template <class T, bool P16>
__global__ void __launch_bounds__(kBlock)
k_resid_sell(int nslots, const int *__restrict__ ptr, const int *__restrict__ row, const int *__restrict__ col,
             const T *__restrict__ val, const T *__restrict__ ac, const T *__restrict__ b, const T *__restrict__ x,
             T *__restrict__ r, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int t = xcd_block() * kBlock + threadIdx.x;
  if (t >= nslots) return;
  const int i = row[t];
  if (i < 0) return;
  const T s = sell_offdiag<T, P16>(t, t & 63, i, ptr, col, val, x);
  r[i] = b[i] - ac[i] * x[i] - s;
}

// Residual of a coarse level summed straight into the next level's
// right-hand side: b_c[p] = sum over the members i of p of (b_i - A_i x);
// the coarse level's first sweep as k_restrict (mode 1: x_c = omega
// b_c/ac_c, 2: x_c = 0, 0: untouched).  Each coarse cell has MPR groups of
// LPR lanes (all in one wavefront): group g works through members g, g+MPR,
// ... in increasing order, its LPR lanes through each member row together,
// and the groups' sums are combined in a fixed butterfly, so the result is
// deterministic and a coarse cell waits on ceil(members / MPR) member rows
// instead of all of them.
// rows[q] is the range of member q's entries, beside mem[q].
template <int LPR, int MPR, class T>
__global__ void __launch_bounds__(kBlock)
k_resid_restrict_csr(int nc, const int *__restrict__ mptr, const int *__restrict__ mem, const int2 *__restrict__ rows,
                     const int *__restrict__ col, const T *__restrict__ val, const T *__restrict__ ac,
                     const T *__restrict__ b, const T *__restrict__ x, T *__restrict__ bc, const T *__restrict__ acc,
                     T *__restrict__ xc, T omega, int mode, const int *__restrict__ flags) {
  constexpr int G = LPR * MPR;
  static_assert(64 % G == 0 && kBlock % 64 == 0, "a coarse cell's lanes must share a wavefront");
  const int done = done_flag(flags, mptr);
  const int t = xcd_block() * kBlock + threadIdx.x;
  const int p = min(t / G, nc - 1), lane = t % LPR, grp = (t % G) / LPR;
  int q0 = mptr[p], q1 = mptr[p + 1];
  const T ap = mode == 1 ? acc[p] : T(1);
  in_register(q0);
  if (done) return;
  T sum = T(0);
  for (int q = q0 + grp; q < q1; q += MPR) { // the same trip count on the LPR lanes of a group
    const int i = mem[q];
    const int2 e = rows[q];
    const T bi = b[i], ai = ac[i], xi = x[i];
    CsrRow<LPR, T, T> row;
    row.entries(e.x + lane, e.y, col, val);
    row.gather(x);
    const T s = row.finish(col, val, x);
    sum = sum + (bi - ai * xi - s);
  }
#pragma unroll
  for (int off = LPR; off < G; off <<= 1) sum += __shfl_xor(sum, off, G);
  if (t < nc * G && lane == 0 && grp == 0) {
    bc[p] = sum;
    if (mode == 1) xc[p] = omega * sum / ap;
    else if (mode == 2) xc[p] = T(0);
  }
}

// Entry of the cycle on the finest level: b = (T)rhs (when the hierarchy is
// FP32; b may be null in FP64) and the first sweep from a zero start,
// x = omega*b/ac, or x = 0 when no pre-smoothing sweep is asked for.
template <class T>
__global__ void k_enter(int n, const T *__restrict__ ac, const double *__restrict__ rhs, T *__restrict__ b,
                        T *__restrict__ x, T omega, int sweep, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i >= n) return;
  const T bi = (T)rhs[i];
  if (b) b[i] = bi;
  x[i] = sweep ? omega * bi / ac[i] : T(0);
}

// Entry of the cycle fused with the residual of its first sweep, for one
// pre-sweep on the finest level: b = (T)rhs, x = omega*b/ac, r = b - A x,
// where the neighbours' x_j = omega*(T)rhs_j/ac_j are formed from their
// right-hand sides (x is pointwise in b), so no second pass is needed.  The
// values are those of k_enter followed by k_resid.
template <class T>
__global__ void __launch_bounds__(kBlock)
k_enter_resid(int n, int w, EllNbr nbr, const T *__restrict__ ac, const T *__restrict__ anb,
              const double *__restrict__ rhs, T *__restrict__ b, T *__restrict__ x, T *__restrict__ r, T omega,
              const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i >= n) return;
  const T bi = (T)rhs[i];
  if (b) b[i] = bi;
  const T xi = omega * bi / ac[i];
  x[i] = xi;
  const T s = ell_fold_get<kStreamLevel>(
      i, n, w, nbr, anb, [=](int k) { return omega * (T)rhs[k] / ac[k]; }, T(0),
      [](T acc, T a, T xk) { return acc + a * xk; });
  r[i] = bi - ac[i] * xi - s;
}

// Entry of the cycle and its first two sweeps, for two pre-sweeps and more on
// the finest level: b = (T)rhs and the second sweep from x = omega*b/ac, whose
// values are formed as in k_enter_resid.  The values are those of k_enter
// followed by k_sweep, in one launch (64x64 cells: 1.06 -> 1.02 ms a solve).
template <class T>
__global__ void __launch_bounds__(kBlock)
k_enter_sweep(int n, int w, EllNbr nbr, const T *__restrict__ ac, const T *__restrict__ anb,
              const double *__restrict__ rhs, T *__restrict__ b, T *__restrict__ x, T omega,
              const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i >= n) return;
  const T bi = (T)rhs[i], ai = ac[i];
  if (b) b[i] = bi;
  const T xi = omega * bi / ai;
  const T s = ell_fold_get<kStreamLevel>(
      i, n, w, nbr, anb, [=](int k) { return omega * (T)rhs[k] / ac[k]; }, T(0),
      [](T acc, T a, T xk) { return acc + a * xk; });
  x[i] = xi + omega * (bi - ai * xi - s) / ai;
}

// Residual of the finest level summed straight into the next level's
// right-hand side, with ENTER the entry of the cycle as well (k_enter_resid):
// kFineGroup lanes per coarse cell, lane g through its members g, g +
// kFineGroup, ..., combined in a fixed butterfly; mode as in k_restrict.  On a
// small mesh a pass is its launch and its chain of loads, and this saves one
// of each per cycle.
constexpr int kFineGroup = 8;
template <class T, bool ENTER>
__global__ void __launch_bounds__(kBlock)
k_fine_restrict(int nc, const int *__restrict__ mptr, const int *__restrict__ mem, int n, int w, EllNbr nbr,
                const T *__restrict__ ac, const T *__restrict__ anb, const double *__restrict__ rhs, const T *bin,
                T *bout, const T *xin, T *xout, T *__restrict__ bc, const T *__restrict__ acc, T *__restrict__ xc,
                T omega, int mode, const int *__restrict__ flags) {
  const int done = done_flag(flags, mptr);
  const int t = xcd_block() * kBlock + threadIdx.x;
  const int p = min(t / kFineGroup, nc - 1), g = t % kFineGroup;
  int q0 = mptr[p], q1 = mptr[p + 1];
  const T ap = mode == 1 ? acc[p] : T(1);
  in_register(q0);
  if (done) return;
  const bool ok = t < nc * kFineGroup;
  T sum = T(0);
  if (ok)
    for (int q = q0 + g; q < q1; q += kFineGroup) {
      const int i = mem[q];
      const T ai = ac[i];
      const auto add = [](T a0, T a, T xk) { return a0 + a * xk; };
      if (ENTER) {
        const T bi = (T)rhs[i], xi = omega * bi / ai;
        const T s = ell_fold_get<kStreamLevel>(
            i, n, w, nbr, anb, [=](int k) { return omega * (T)rhs[k] / ac[k]; }, T(0), add);
        if (bout) bout[i] = bi;
        xout[i] = xi;
        sum = sum + (bi - ai * xi - s);
      } else {
        const T bi = bin[i], xi = xin[i];
        const T s = ell_fold<kStreamLevel>(i, n, w, nbr, anb, xin, T(0), add);
        sum = sum + (bi - ai * xi - s);
      }
    }
#pragma unroll
  for (int off = 1; off < kFineGroup; off <<= 1) sum += __shfl_xor(sum, off, kFineGroup);
  if (ok && g == 0) {
    bc[p] = sum;
    if (mode == 1) xc[p] = omega * sum / ap;
    else if (mode == 2) xc[p] = T(0);
  }
}

// Restriction b_c[p] = sum of the member residuals in increasing fine-cell
// order; mode 1 also takes the coarse level's first sweep from a zero start
// (x_c = omega*b_c/ac_c), mode 2 sets x_c = 0, mode 0 leaves x_c alone.
template <class T>
__global__ void k_restrict(int nc, const int *__restrict__ mptr, const int *__restrict__ mem,
                           const T *__restrict__ rf, T *__restrict__ bc, const T *__restrict__ acc,
                           T *__restrict__ xc, T omega, int mode, const int *__restrict__ flags) {
  const int done = done_flag(flags, mptr);
  const int p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= nc) return;
  int q0 = mptr[p], q1 = mptr[p + 1];
  in_register(q0);
  if (done) return;
  T s = T(0);
  // members in batches: their indices, then their residuals, then the sum
  // in member order
  constexpr int B = 8;
  for (int q = q0; q < q1; q += B) {
    int id[B];
    T v[B];
#pragma unroll
    for (int u = 0; u < B; ++u) id[u] = mem[min(q + u, q1 - 1)];
#pragma unroll
    for (int u = 0; u < B; ++u) v[u] = rf[id[u]];
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (q + u < q1) s = s + v[u];
  }
  bc[p] = s;
  if (mode == 1) xc[p] = omega * s / acc[p];
  else if (mode == 2) xc[p] = T(0);
}

// out = x + alpha*xc[parent] (out may be x)
template <class T, class TO>
__global__ void k_prolong(int nf, const int *__restrict__ parent, const T *__restrict__ xc, const T *x,
                          T alpha, TO *out, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = xcd_block() * kBlock + threadIdx.x;
  if (i < nf) out[i] = (TO)(x[i] + alpha * xc[parent[i]]);
}

template <class T, class TO>
__global__ void k_convert(int n, const T *__restrict__ x, TO *__restrict__ out, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) out[i] = (TO)x[i];
}

template <class T>
__global__ void k_zero(int n, T *__restrict__ x, const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = T(0);
}

// one colour of a multicolour Gauss-Seidel sweep, in place
template <class T>
__global__ void k_gsc(int cnt, const int *__restrict__ cells, int n, int w, const int *__restrict__ nbr,
                      const T *__restrict__ ac, const T *__restrict__ anb, const T *__restrict__ b, T *x,
                      const int *__restrict__ flags) {
  if (flags && flags[0]) return;
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= cnt) return;
  const int i = cells[t];
  const T s = ell_fold(i, n, w, nbr, anb, (const T *)x, b[i], [](T acc, T a, T xk) { return acc - a * xk; });
  x[i] = s / ac[i];
}

// AMG-as-solver residual: r = b - A x and partial L1(r)
__global__ void k_amg_res(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                          const double *__restrict__ anb, const double *__restrict__ b,
                          const double *__restrict__ x, double *__restrict__ r, double *__restrict__ part,
                          const int *__restrict__ flags) {
  if (flags[0]) return;
  double s = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    const double v = ell_fold(i, n, w, nbr, anb, x, b[i] - ac[i] * x[i],
                                         [](double acc, double a, double xk) { return acc - a * xk; });
    r[i] = v;
    s += fabs(v);
  }
  s = block_sum<kBlock>(s);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_add2(int n, double *__restrict__ x, const double *__restrict__ c,
                       const int *__restrict__ flags) {
  if (flags[0]) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) x[i] = x[i] + c[i];
}

// ------------------------------------------------------------ small levels
// The cycle below the first small level is one fixed linear map x = C b (it
// starts every level from zero and never tests anything), so it is formed
// once per operator as a dense matrix and applied as a matrix-vector product.
// Column j is the cycle's answer to the j-th unit vector: k_dense_level forms
// all columns of a level from the level's sparse operator and the dense map of
// the level below it.  Maps are FP64 for every hierarchy: they hold the inverse
// of the coarsest operator, which on a nearly singular system is one large
// constant and, below its FP32 rounding, the part that corrects.  A product is
// bound by one round of loads (1190 cells: 11 MB, spread over the chip) and takes
// 5.0 us (828 cells 3.9, 1939 cells 9.0; with FP32 maps 4.7, 4.6, 6.5), where one
// workgroup that walked the levels in LDS took 13-25 us per visit, 8 to 30 visits
// per Krylov iteration; forming the maps takes 60-210 us per operator.  2.1 M
// hexahedra take 531 us a BiCGSTAB iteration (519 with FP32 maps), 2.9 M
// tetrahedra 549 us a CG iteration (545).
constexpr int kDirectMax = 64;               // coarsest levels up to this size are solved directly
constexpr int kDenseThreads = 512;
constexpr int kDenseRows = 8;                // rows of a product's workgroup
// cells of the largest map.  FP64 hierarchies: 16 MB, half of what the L2s hold;
// FP32 ones up to 34 MB, where the map is even with the level's own launches
// around the map below (1939 cells under 2.1 M hexahedra: 531 us an iteration
// and 528).
inline int dense_max(bool fp32) { return fp32 ? 2048 : 1448; }

// A map is stored in strips of kDenseRows rows, each strip column by column,
// so that a strip is one contiguous run of memory: entry (i, j) of an n x n map.
__host__ __device__ __forceinline__ size_t dense_at(int i, int j, int n) {
  return ((size_t)(i / kDenseRows) * n + j) * kDenseRows + i % kDenseRows;
}
// values of a map of n cells (the last strip is padded)
inline size_t dense_size(int n) { return (size_t)((n + kDenseRows - 1) / kDenseRows) * kDenseRows * n; }

typedef double doublex2 __attribute__((ext_vector_type(2)));
constexpr int kDenseColumns = 2;             // columns a workgroup of k_dense_level forms together

// The map of a level, K = 2 columns per workgroup: `pre` damped-Jacobi sweeps from
// zero on the unit vectors, the restricted residual through the map Cc of the
// next level (nc cells), alpha times the result prolongated, `post` sweeps.
// Cc null: the sweeps alone (a coarsest level too large for the direct solve).
// The vectors live in LDS, K to a 16-byte element, and the level's rows come
// from L2 once per pass for all K, in the hierarchy's precision (the pass is
// bound by those reads: 1939 cells 148 us; one column a workgroup from FP64 rows
// took 314, four columns, whose LDS leaves one workgroup a CU, no less).  After one
// sweep from zero the residual reaches only the aggregates next to the unit's
// cell, so the coarse map is applied to the nonzero entries alone.
template <class A>
__global__ void __launch_bounds__(kDenseThreads)
k_dense_level(int n, int w, const int *__restrict__ nbr, const A *__restrict__ anb,
              const A *__restrict__ ac, const int *__restrict__ parent, int nc, const int *__restrict__ mptr,
              const int *__restrict__ mem, const double *__restrict__ Cc, int pre, int post, double omega,
              double alpha, double *__restrict__ C) {
  constexpr int K = kDenseColumns;
  typedef double T;
  typedef doublex2 V;
  static_assert(sizeof(V) == K * sizeof(T), "columns of a vector element");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  V *x = (V *)lds, *y = x + n, *rc = y + n;
  int *list = (int *)(rc + nc);
  __shared__ int s_cnt;
  const int j0 = blockIdx.x * K;
  auto unit = [&](int i) {
    V e;
#pragma unroll
    for (int k = 0; k < K; ++k) e[k] = i == j0 + k ? T(1) : T(0);
    return e;
  };
  // y = x + omega (e - A x)/ac, or the residual e - A x; one row a lane, its
  // slots in batches
  auto pass = [&](bool jac) {
    constexpr int B = 8;
    for (int i = threadIdx.x; i < n; i += kDenseThreads) {
      V sum = T(0);
      for (int s0 = 0; s0 < w; s0 += B) {
        int k[B];
        T a[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const size_t at = (size_t)min(s0 + u, w - 1) * n + i;
          k[u] = nbr[at];
          a[u] = anb[at];
        }
#pragma unroll
        for (int u = 0; u < B; ++u)
          if (s0 + u < w && k[u] >= 0) sum = sum + a[u] * x[k[u]];
      }
      const T a = ac[i];
      const V r = unit(i) - a * x[i] - sum;
      y[i] = jac ? x[i] + omega * r / a : r;
    }
    __syncthreads();
    if (jac) {
      V *t = x;
      x = y;
      y = t;
    }
  };
  for (int i = threadIdx.x; i < n; i += kDenseThreads) {
    V v = T(0);
    if (pre > 0) v = omega * unit(i) / ac[i];
    x[i] = v;
  }
  __syncthreads();
  for (int k = 1; k < pre; ++k) pass(true);
  if (Cc) {
    pass(false);
    for (int p = threadIdx.x; p < nc; p += kDenseThreads) {
      V s = T(0);
      for (int q = mptr[p]; q < mptr[p + 1]; ++q) s = s + y[mem[q]];
      rc[p] = s;
    }
    __syncthreads();
    if (threadIdx.x < 64) { // the entries nonzero for any column, in order
      int cnt = 0;
      for (int p0 = 0; p0 < nc; p0 += 64) {
        const int p = p0 + (int)threadIdx.x;
        bool nz = false;
        if (p < nc)
#pragma unroll
          for (int k = 0; k < K; ++k) nz = nz || rc[p][k] != T(0);
        const unsigned long long m = __ballot(nz);
        if (nz) list[cnt + __popcll(m & ((1ull << threadIdx.x) - 1ull))] = p;
        cnt += __popcll(m);
      }
      if (threadIdx.x == 0) s_cnt = cnt;
    }
    __syncthreads();
    const int cnt = s_cnt;
    for (int p = threadIdx.x; p < nc; p += kDenseThreads) {
      V s = T(0);
      for (int q = 0; q < cnt; ++q) s = s + Cc[dense_at(p, list[q], nc)] * rc[list[q]];
      y[p] = s; // the residuals are summed: y is free
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kDenseThreads) x[i] = x[i] + alpha * y[parent[i]];
    __syncthreads();
    for (int k = 0; k < post; ++k) pass(true);
  }
  // K columns of one row are K kDenseRows values: lanes run over a strip's
  // rows first
  const int values = (n + kDenseRows - 1) / kDenseRows * kDenseRows * K;
  for (int t = threadIdx.x; t < values; t += kDenseThreads) {
    const int i = t / (kDenseRows * K) * kDenseRows + t % kDenseRows, k = t / kDenseRows % K;
    if (i < n && j0 + k < n) C[dense_at(i, j0 + k, n)] = x[i][k];
  }
}

// x = C b (ACC: x += C b), the products and sums in FP64, and with SC the
// prolongation of x.  A workgroup owns a strip of kDenseRows rows, whose
// entries its threads load 16 bytes at a time in address order, all of a
// thread's loads before the first product; the partial sums are combined in a
// fixed order.
template <class T, bool ACC, bool SC>
__global__ void __launch_bounds__(kDenseThreads)
k_dense_apply(int n, const double *__restrict__ C, const T *__restrict__ b, T *__restrict__ x,
              const int *__restrict__ parent, Scatter<T> sc, const int *__restrict__ flags) {
  constexpr int K = 2, LPC = kDenseRows / K, W = kDenseThreads / 64, B = 8; // lanes per column
  typedef doublex2 V;
  __shared__ double part[W][kDenseRows];
  __shared__ T xs[kDenseRows];
  const int i0 = blockIdx.x * kDenseRows, cnt = n * LPC; // 16-byte elements of the strip
  const V *strip = (const V *)(C + (size_t)i0 * n);
  const int done = done_flag(flags, C); // tested before the stores
  // the strip's members: this thread's first one is loaded beside the products
  const int m0 = SC ? sc.mptr[i0] + (int)threadIdx.x : 0, m1 = SC ? sc.mptr[min(i0 + kDenseRows, n)] : 0;
  int mf = 0, mp = 0;
  T mx = T(0);
  V c[B];
  T v[B];
  const auto fetch = [&](int e0) {
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int e = min(e0 + u * kDenseThreads, cnt - 1);
      c[u] = strip[e];
      v[u] = b[e / LPC];
    }
  };
  fetch(threadIdx.x);
  if (SC) mf = sc.mem[min(m0, m1 - 1)];
  double acc[K];
#pragma unroll
  for (int k = 0; k < K; ++k) acc[k] = 0.0;
  const auto add = [&](int e0) {
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (e0 + u * kDenseThreads < cnt)
#pragma unroll
        for (int k = 0; k < K; ++k) acc[k] += c[u][k] * (double)v[u];
  };
  if (SC) mp = parent[mf] - i0, mx = sc.x[mf];
  add(threadIdx.x);
  for (int e0 = threadIdx.x + B * kDenseThreads; e0 < cnt; e0 += B * kDenseThreads) {
    fetch(e0);
    add(e0);
  }
  if (done) return;
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int off = LPC; off < 64; off <<= 1)
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] += __shfl_xor(acc[k], off, 64);
  if (lane < LPC)
#pragma unroll
    for (int k = 0; k < K; ++k) part[wid][lane * K + k] = acc[k];
  __syncthreads();
  const int r = i0 + (int)threadIdx.x;
  if (threadIdx.x < kDenseRows && r < n) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < W; ++k) s += part[k][threadIdx.x];
    const T v = ACC ? (T)((double)x[r] + s) : (T)s;
    x[r] = v;
    if (SC) xs[threadIdx.x] = v;
  }
  if constexpr (SC) {
    __syncthreads();
    if (m0 < m1) sc.x[mf] = mx + sc.alpha * xs[mp];
    for (int q = m0 + kDenseThreads; q < m1; q += kDenseThreads) {
      const int f = sc.mem[q];
      sc.x[f] = sc.x[f] + sc.alpha * xs[parent[f] - i0];
    }
  }
}

// FP64 inverse of the coarsest operator by Gauss-Jordan elimination without
// pivoting (the coarse operators are diagonally dominant), one workgroup,
// n <= kDirectMax.  A singular operator with zero row sums (the pure
// Neumann p' problem, null space = constants) is solved with its last
// unknown pinned to zero: the result is the inverse of the leading (n-1)x(n-1) block,
// bordered by zeros, a symmetric generalised inverse.  A zero or non-finite
// pivot leaves it 0 (no coarse correction) rather than garbage.
constexpr int kInvThreads = 256;
__global__ void __launch_bounds__(kInvThreads)
k_coarse_inverse(int n, int w, const int *__restrict__ nbr, const double *__restrict__ ac,
                 const double *__restrict__ anb, double *__restrict__ C) {
  __shared__ double M[kDirectMax * kDirectMax];
  __shared__ double rowk[kDirectMax], colk[kDirectMax];
  __shared__ int s_m, s_fail;
  const int nn = n * n;
  for (int e = threadIdx.x; e < nn; e += blockDim.x) {
    const int i = e / n, k = e % n;
    M[e] = (i == k) ? ac[i] : 0.0;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    s_m = n - 1;
    s_fail = 0;
  }
  __syncthreads();
  // one row a thread, its off-diagonals in slot order (a level's neighbours
  // are distinct); singularity test on the row sums
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    double rs = ac[i];
    for (int j = 0; j < w; ++j) {
      const int k = nbr[(size_t)j * n + i];
      if (k >= 0) {
        const double a = anb[(size_t)j * n + i];
        M[i * n + k] += a;
        rs += a;
      }
    }
    if (!(fabs(rs) <= 1.0e-9 * fabs(ac[i]))) s_m = n; // every writer stores the same value
  }
  __syncthreads();
  const int m = s_m;
  for (int k = 0; k < m; ++k) {
    const double p = M[k * n + k];
    if (!(fabs(p) > 0.0) || !isfinite(p)) {
      if (threadIdx.x == 0) s_fail = 1;
      break; // p is read from LDS by every thread: the branch is uniform
    }
    for (int j = threadIdx.x; j < m; j += blockDim.x) {
      rowk[j] = (j == k) ? 1.0 / p : M[k * n + j] / p;
      colk[j] = M[j * n + k];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < m * m; e += blockDim.x) {
      const int i = e / m, j = e % m;
      if (i == k) M[k * n + j] = rowk[j];
      else M[i * n + j] = ((j == k) ? 0.0 : M[i * n + j]) - colk[i] * rowk[j];
    }
    __syncthreads();
  }
  __syncthreads();
  const bool fail = s_fail != 0;
  for (int e = threadIdx.x; e < nn; e += blockDim.x) {
    const int i = e / n, j = e % n;
    C[dense_at(i, j, n)] = (!fail && i < m && j < m) ? M[i * n + j] : 0.0;
  }
}

} // namespace

// ------------------------------------------------------------ hierarchy
struct DLevel {
  int n = 0, w = 0;
  const int *nbr = nullptr;      // device, 0-based/-1
  const int *nbr16 = nullptr;    // level 0: the mesh's packed 16-bit offsets, if any
  DevBuf<int> nbr_own;
  const double *ac64 = nullptr, *anb64 = nullptr;
  DevBuf<double> ac64_own, anb64_own;
  DevBuf<float> ac32, anb32;
  DevBuf<double> x64, b64, r64, t64;
  DevBuf<float> x32, b32, r32, t32;
  std::vector<int> color_ptr;
  DevBuf<int> color_cells;
  DevBuf<int> parent;            // 0-based parent in the next level
  DevBuf<int> mptr, mem;         // members of this level's aggregates (coarse)
  DevBuf<int2> mrow;             // beside mem: the member's entries in the finer level's CSR
  DevBuf<int> gptr;
  DevBuf<int> gsrc;               // 32-bit: fine n + n w stays below 2^31
  int gne = 0;
  // levels >= 1: row-major CSR copy of the off-diagonals for the grid-wide
  // Jacobi kernels (values written by k_galerkin through csr_pos)
  long long nnz = 0;
  DevBuf<int> csr_rp, csr_col, csr_pos;
  DevBuf<double> val64;
  DevBuf<float> val32;
  DevBuf<double> dense; // small levels: the map of the cycle from this level down
  // large levels: sliced ELL instead (val64/val32 then hold the sliced
  // layout and csr_pos points into it)
  bool sell = false, sell16 = false; // sell16: sell_col as 16-bit offsets (k_sweep_sell)
  int sell_slots = 0;
  DevBuf<int> sell_ptr, sell_row, sell_col;
};

constexpr int kSellWindow = 256; // rows sorted by length within windows of this size

// Sliced-ELL image of a CSR level: slot order, slice offsets, columns, and
// the map from CSR entry to sliced entry.
static void build_sell(int n, bool even, const std::vector<int> &rp, const std::vector<int> &col, std::vector<int> &ptr,
                       std::vector<int> &row, std::vector<int> &scol, std::vector<int> &csr2sell) {
  std::vector<int> order(n);
  for (int i = 0; i < n; ++i) order[i] = i;
  for (int w0 = 0; w0 < n; w0 += kSellWindow) {
    const int w1 = std::min(n, w0 + kSellWindow);
    std::stable_sort(order.begin() + w0, order.begin() + w1,
                     [&](int a, int b) { return rp[a + 1] - rp[a] > rp[b + 1] - rp[b]; });
  }
  const int ns = (n + 63) / 64;
  row.assign((size_t)ns * 64, -1);
  ptr.assign(ns + 1, 0);
  for (int s = 0; s < ns; ++s) {
    int len = 0;
    for (int l = 0; l < 64 && s * 64 + l < n; ++l) {
      const int r = order[s * 64 + l];
      row[(size_t)s * 64 + l] = r;
      len = std::max(len, rp[r + 1] - rp[r]);
    }
    if (even) len += len & 1;
    ptr[s + 1] = ptr[s] + 64 * len;
  }
  scol.assign(std::max(ptr[ns], 1), 0);
  csr2sell.assign(std::max<size_t>(col.size(), 1), -1);
  for (int s = 0; s < ns; ++s) {
    const int len = (ptr[s + 1] - ptr[s]) / 64;
    for (int l = 0; l < 64; ++l) {
      const int r = row[(size_t)s * 64 + l];
      for (int k = 0; k < len; ++k) {
        const int q = ptr[s] + 64 * k + l;
        if (r < 0) scol[q] = 0;
        else if (k < rp[r + 1] - rp[r]) {
          scol[q] = col[rp[r] + k];
          csr2sell[rp[r] + k] = q;
        } else {
          scol[q] = r; // padding: zero value times the row's own x
        }
      }
    }
  }
}

// The levels whose cycle is held as a dense map (k_dense_level), for one
// precision of the hierarchy.  ts: the first level of at most mg_tail_cells
// cells (and at most dense_max()), the bottom of the cycle pattern;
// levels when there is none.  dl: the level the map is applied on, ts or the
// level above it when that one's map fits as well.
struct DenseTail {
  int ts = -1, dl = -1;
};

struct Hierarchy {
  std::vector<HostLevel> host;   // maps for export / tests
  std::vector<DLevel> lev;
  int calls = 0;
  bool fp32 = false;
  DenseTail tail;
};

static void build_hierarchy(fs_mesh *m, const double *ac, const double *anb) {
  auto H = std::make_shared<Hierarchy>();
  hipStream_t s = m->stream;
  const int n = m->n, w = m->w;
  HostLevel L0;
  L0.n = n;
  L0.w = w;
  L0.nbr = m->h_nbr;
  L0.nnbr = m->h_nnbr;
  L0.ac.resize(n);
  L0.anb.resize((size_t)n * w);
  FS_HIP_THROW(hipMemcpyAsync(L0.ac.data(), ac, sizeof(double) * n, hipMemcpyDeviceToHost, s));
  FS_HIP_THROW(hipMemcpyAsync(L0.anb.data(), anb, sizeof(double) * n * w, hipMemcpyDeviceToHost, s));
  FS_HIP_THROW(hipStreamSynchronize(s));
  H->host.push_back(std::move(L0));
  std::vector<std::vector<int>> gptrs(1);
  std::vector<std::vector<long long>> gsrcs(1);
  int nl = 1;
  while (nl < m->mg_maxlevels && H->host[nl - 1].n > 2 * m->mg_minparents) {
    HostLevel c;
    if (m->mg_agg == 0) aggregate(H->host[nl - 1], c, nl + 1);
    else aggregate_pairwise(H->host[nl - 1], c, m->mg_agg);
    std::vector<int> gp;
    std::vector<long long> gs;
    galerkin_lists(H->host[nl - 1], c, gp, gs);
    H->host.push_back(std::move(c));
    gptrs.push_back(std::move(gp));
    gsrcs.push_back(std::move(gs));
    ++nl;
  }
  H->lev.resize(nl);
  std::vector<int> rp_f; // row starts of the finer level's CSR
  for (int l = 0; l < nl; ++l) {
    DLevel &D = H->lev[l];
    HostLevel &h = H->host[l];
    D.n = h.n;
    D.w = h.w;
    std::vector<int> nbr0((size_t)h.n * h.w);
    for (int i = 0; i < h.n; ++i)
      for (int j = 0; j < h.w; ++j) {
        const int k = h.nbr[(size_t)j * h.n + i];
        nbr0[(size_t)j * h.n + i] = (j < h.nnbr[i] && k > 0) ? k - 1 : -1;
      }
    if (l == 0) {
      D.nbr = m->d_nbr.p;
      D.nbr16 = m->d_nbr16.p;
    } else {
      D.nbr_own.upload(nbr0, s);
      D.nbr = D.nbr_own.p;
      D.ac64_own.alloc(h.n);
      D.anb64_own.alloc((size_t)h.n * h.w);
      D.ac64 = D.ac64_own.p;
      D.anb64 = D.anb64_own.p;
      D.gptr.upload(gptrs[l], s);
      {
        std::vector<int> g32(gsrcs[l].size());
        for (size_t t = 0; t < g32.size(); ++t) {
          if (gsrcs[l][t] > INT32_MAX) throw std::runtime_error("AMG level too large for 32-bit Galerkin sources");
          g32[t] = (int)gsrcs[l][t];
        }
        D.gsrc.upload(g32, s);
      }
      D.gne = (int)gptrs[l].size() - 1;
      // members in increasing fine order
      const HostLevel &f = H->host[l - 1];
      std::vector<int> mptr(h.n + 1, 0), mem(f.n, 0);
      for (int i = 0; i < f.n; ++i) mptr[f.parent[i]]++;
      for (int p = 0; p < h.n; ++p) mptr[p + 1] += mptr[p];
      std::vector<int> fill(mptr.begin(), mptr.end() - 1);
      for (int i = 0; i < f.n; ++i) mem[fill[f.parent[i] - 1]++] = i;
      D.mptr.upload(mptr, s);
      D.mem.upload(mem, s);
      if (l > 1) {
        std::vector<int2> mrow(f.n);
        for (int q = 0; q < f.n; ++q) mrow[q] = make_int2(rp_f[mem[q]], rp_f[mem[q] + 1]);
        D.mrow.upload(mrow, s);
      }
      std::vector<int> rp(h.n + 1, 0), col, pos((size_t)h.n * h.w, -1);
      for (int i = 0; i < h.n; ++i) {
        for (int j = 0; j < h.w; ++j) {
          const int k = nbr0[(size_t)j * h.n + i];
          if (k < 0) continue;
          pos[(size_t)j * h.n + i] = (int)col.size();
          col.push_back(k);
        }
        rp[i + 1] = (int)col.size();
      }
      D.nnz = (long long)col.size();
      // a level that runs grid-wide (larger than the tail) and has at least
      // mg_sell_rows rows keeps its operator in sliced ELL
      D.sell = m->mg_sell_rows > 0 && h.n >= m->mg_sell_rows && h.n > m->mg_tail_cells;
      size_t nval = std::max<size_t>(col.size(), 1);
      if (D.sell) {
        std::vector<int> sptr, srow, scol, c2s;
        D.sell16 = true; // if every offset fits
        for (int i = 0; i < h.n && D.sell16; ++i)
          for (int q = rp[i]; q < rp[i + 1]; ++q) D.sell16 = D.sell16 && std::abs(col[q] - i) <= INT16_MAX;
        build_sell(h.n, D.sell16, rp, col, sptr, srow, scol, c2s);
        for (auto &q : pos)
          if (q >= 0) q = c2s[q];
        D.sell_slots = (int)srow.size();
        D.sell_ptr.upload(sptr, s);
        D.sell_row.upload(srow, s);
        nval = scol.size();
        if (D.sell16) {
          std::vector<int> words(std::max<size_t>(nval / 2, 1), 0);
          for (size_t sl = 0; sl + 1 < sptr.size(); ++sl)
            for (int q = sptr[sl]; q < sptr[sl + 1]; ++q) {
              const int k = (q - sptr[sl]) >> 6, l = q & 63, r = srow[sl * 64 + l];
              const int d = r < 0 ? 0 : (scol[q] - r) & 0xffff;
              words[(sptr[sl] >> 1) + ((k >> 1) << 6) + l] |= k & 1 ? d << 16 : d;
            }
          D.sell_col.upload(words, s);
        } else {
          D.sell_col.upload(scol, s);
        }
      }
      if (col.empty()) col.push_back(0);
      D.csr_rp.upload(rp, s);
      D.csr_col.upload(col, s);
      D.csr_pos.upload(pos, s);
      rp_f = std::move(rp);
      D.val64.alloc(nval);
      D.val32.alloc(nval);
      // padded sliced entries are never written by the Galerkin kernel
      FS_HIP_THROW(hipMemsetAsync(D.val64.p, 0, sizeof(double) * nval, s));
      FS_HIP_THROW(hipMemsetAsync(D.val32.p, 0, sizeof(float) * nval, s));
    }
    if (l + 1 < nl) {
      std::vector<int> par0(h.n);
      for (int i = 0; i < h.n; ++i) par0[i] = h.parent[i] - 1;
      D.parent.upload(par0, s);
    }
    std::vector<int> cells;
    greedy_colors(h.n, h.w, nbr0.data(), D.color_ptr, cells);
    D.color_cells.upload(cells, s);
    D.x64.alloc(h.n);
    D.b64.alloc(h.n);
    D.r64.alloc(h.n);
    D.t64.alloc(h.n);
    D.x32.alloc(h.n);
    D.b32.alloc(h.n);
    D.r32.alloc(h.n);
    D.t32.alloc(h.n);
    D.ac32.alloc(h.n);
    D.anb32.alloc((size_t)h.n * h.w);
  }
  FS_HIP_THROW(hipStreamSynchronize(s));
  m->amg = H;
}

// multicolour symmetric Gauss-Seidel only where it is cheap: few colours,
// narrow rows
static bool use_gs(const fs_mesh *m, const DLevel &D) {
  return m->mg_smoother == 1 && (int)D.color_ptr.size() - 1 <= 4 && D.w <= 8;
}

// sweeps on the levels below the finest, and on a coarsest level too large
// for the direct solve
static int coarse_pre(const fs_mesh *m) { return m->mg_cpre >= 0 ? m->mg_cpre : m->mg_pre; }
static int coarse_post(const fs_mesh *m) { return m->mg_cpost >= 0 ? m->mg_cpost : m->mg_post; }
static int coarsest_sweeps(const fs_mesh *m) { return std::max(m->mg_coarse_sweeps, 1); }

// The dense maps of the small levels, from the coarsest up to the one applied.
static void build_dense(fs_mesh *m, Hierarchy &H, double alpha) {
  hipStream_t s = m->stream;
  const int nl = (int)H.lev.size(), most = dense_max(H.fp32);
  DenseTail &dt = H.tail;
  dt.ts = nl;
  for (int l = 1; l < nl; ++l)
    if (H.lev[l].n <= std::min(m->mg_tail_cells, most)) {
      dt.ts = l;
      break;
    }
  dt.dl = dt.ts;
  if (dt.ts >= nl) return;
  if (dt.ts > 1) {
    const DLevel &U = H.lev[dt.ts - 1];
    if (U.n <= most && !U.sell && !use_gs(m, U)) dt.dl = dt.ts - 1;
  }
  for (int l = nl - 1; l >= dt.dl; --l) {
    DLevel &D = H.lev[l];
    D.dense.alloc(dense_size(D.n));
    const bool last = l == nl - 1;
    if (last && D.n <= kDirectMax) {
      hipLaunchKernelGGL(k_coarse_inverse, dim3(1), dim3(kInvThreads), 0, s, D.n, D.w, D.nbr, D.ac64, D.anb64,
                         D.dense.p);
      continue;
    }
    DLevel *U = last ? nullptr : &H.lev[l + 1];
    const int nc = last ? 0 : U->n, pre = last ? coarsest_sweeps(m) : coarse_pre(m), post = last ? 0 : coarse_post(m);
    const size_t lds = sizeof(doublex2) * (2 * (size_t)D.n + nc) + sizeof(int) * (size_t)nc;
    const auto form = [&](auto kernel, const auto *anb, const auto *ac) {
      // the largest maps ask for more than the default dynamic LDS window
      if (lds > 64 * 1024)
        FS_HIP_THROW(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
      hipLaunchKernelGGL(kernel, dim3((D.n + kDenseColumns - 1) / kDenseColumns), dim3(kDenseThreads), (unsigned)lds, s,
                         D.n, D.w, D.nbr, anb, ac, D.parent.p, nc, last ? nullptr : U->mptr.p,
                         last ? nullptr : U->mem.p, last ? nullptr : (const double *)U->dense.p, pre, post,
                         m->mg_omega, alpha, D.dense.p);
      FS_HIP_THROW(hipGetLastError()); // a refused launch (LDS request) must not pass silently
    };
    if (H.fp32) form(k_dense_level<float>, (const float *)D.anb32.p, (const float *)D.ac32.p);
    else form(k_dense_level<double>, (const double *)D.anb64, (const double *)D.ac64);
  }
}

bool amg_will_build(const fs_mesh *m) {
  return !m->amg || (m->mg_reagg > 0 && m->ncalls_mg % m->mg_reagg == 0) || m->amg->lev.empty() ||
         m->amg->lev[0].n != m->n;
}

void amg_prepare(fs_mesh *m, const double *ac, const double *anb, double alpha) {
  if (amg_will_build(m)) build_hierarchy(m, ac, anb);
  m->ncalls_mg++;
  Hierarchy &H = *m->amg;
  H.fp32 = m->mg_fp32 != 0;
  hipStream_t s = m->stream;
  DLevel &L0 = H.lev[0];
  L0.ac64 = ac;
  L0.anb64 = anb;
  if (H.fp32) {
    hipLaunchKernelGGL(k_to<float>, dim3(gfor(L0.n)), dim3(kBlock), 0, s, L0.n, ac, L0.ac32.p);
    hipLaunchKernelGGL(k_to<float>, dim3(gfor(L0.n * L0.w)), dim3(kBlock), 0, s, L0.n * L0.w, anb,
                       L0.anb32.p);
  }
  for (size_t l = 1; l < H.lev.size(); ++l) {
    DLevel &F = H.lev[l - 1], &C = H.lev[l];
    hipLaunchKernelGGL(k_galerkin, dim3(gfor(C.gne)), dim3(kBlock), 0, s, C.gne, C.n, C.gptr.p,
                       C.gsrc.p, F.n, F.ac64, F.anb64, C.ac64_own.p, C.anb64_own.p,
                       H.fp32 ? C.ac32.p : nullptr, H.fp32 ? C.anb32.p : nullptr, C.csr_pos.p, C.val64.p,
                       H.fp32 ? C.val32.p : nullptr);
  }
  build_dense(m, H, alpha);
}

int amg_levels(fs_mesh *m) { return m->amg ? (int)m->amg->lev.size() : 1; }

template <class T> struct LV {
  static T *x(DLevel &d);
  static T *b(DLevel &d);
  static T *r(DLevel &d);
  static T *t(DLevel &d);
  static const T *ac(DLevel &d);
  static const T *anb(DLevel &d);
  static const T *val(DLevel &d);
};
template <> struct LV<double> {
  static double *x(DLevel &d) { return d.x64.p; }
  static double *b(DLevel &d) { return d.b64.p; }
  static double *r(DLevel &d) { return d.r64.p; }
  static double *t(DLevel &d) { return d.t64.p; }
  static const double *ac(DLevel &d) { return d.ac64; }
  static const double *anb(DLevel &d) { return d.anb64; }
  static const double *val(DLevel &d) { return d.val64.p; }
};
template <> struct LV<float> {
  static float *x(DLevel &d) { return d.x32.p; }
  static float *b(DLevel &d) { return d.b32.p; }
  static float *r(DLevel &d) { return d.r32.p; }
  static float *t(DLevel &d) { return d.t32.p; }
  static const float *ac(DLevel &d) { return d.ac32.p; }
  static const float *anb(DLevel &d) { return d.anb32.p; }
  static const float *val(DLevel &d) { return d.val32.p; }
};

// lanes per row of a coarse level's CSR kernels by its mean row length
static int csr_lpr(const DLevel &D) {
  const double a = D.n ? (double)D.nnz / D.n : 0.0;
  return a <= 6.0 ? 4 : a <= 16.0 ? 8 : 16;
}

// residual of coarse level D restricted into C (plus C's first sweep): 8 member
// groups per coarse cell of 4 lanes (rows of up to 6 entries) or 8 lanes each
// (with 16 lanes, and so 4 groups, wide rows took longer)
template <class T>
static void launch_resid_restrict(fs_mesh *m, DLevel &D, DLevel &C, const T *b, const T *x, T om, int mode,
                                  const int *flags) {
  const auto go = [&](auto kernel, int lanes) {
    hipLaunchKernelGGL(kernel, dim3(gfor(C.n * lanes)), dim3(kBlock), 0, m->stream, C.n, C.mptr.p, C.mem.p, C.mrow.p,
                       D.csr_col.p, LV<T>::val(D), LV<T>::ac(D), b, x, LV<T>::b(C), LV<T>::ac(C), LV<T>::x(C), om,
                       mode, flags);
  };
  if (csr_lpr(D) == 4) go(k_resid_restrict_csr<4, 8, T>, 4 * 8);
  else go(k_resid_restrict_csr<8, 8, T>, 8 * 8);
}

// one damped-Jacobi sweep on a coarse grid-wide level in CSR, lanes per row by
// row width; with sc the prolongation of the result into the finer level
template <class T, bool SC>
static void launch_sweep_csr(fs_mesh *m, DLevel &D, const T *b, const T *x, T om, T *xn, Scatter<T> sc,
                             const int *flags) {
  hipStream_t s = m->stream;
  const T *ac = LV<T>::ac(D), *val = LV<T>::val(D);
  const int *rp = D.csr_rp.p, *col = D.csr_col.p;
  switch (csr_lpr(D)) {
  case 4:
    hipLaunchKernelGGL((k_sweep_csr<4, T, SC>), dim3(gfor(D.n * 4)), dim3(kBlock), 0, s, D.n, rp, col, val, ac, b, x,
                       om, xn, sc, flags);
    break;
  case 8:
    hipLaunchKernelGGL((k_sweep_csr<8, T, SC>), dim3(gfor(D.n * 8)), dim3(kBlock), 0, s, D.n, rp, col, val, ac, b, x,
                       om, xn, sc, flags);
    break;
  default:
    hipLaunchKernelGGL((k_sweep_csr<16, T, SC>), dim3(gfor(D.n * 16)), dim3(kBlock), 0, s, D.n, rp, col, val, ac, b,
                       x, om, xn, sc, flags);
  }
}

// one damped-Jacobi sweep on the finest level, through the kernel clock (site
// FS_CLOCK_FINE_SWEEP) with its algorithmic bytes: ac, b, x, the result, the
// neighbour indices and the off-diagonal values
template <class T, class TO>
static void launch_sweep_fine(fs_mesh *m, DLevel &D, const T *b, const T *x, T om, TO *xn, const int *flags) {
  hipStream_t s = m->stream;
  const T *ac = LV<T>::ac(D), *anb = LV<T>::anb(D);
  const double bytes = (double)D.n * (3.0 * sizeof(T) + sizeof(TO)) +
                       (D.nbr16 ? 4.0 * ((D.w + 1) / 2) : 4.0 * D.w) * D.n + (double)sizeof(T) * m->nnz;
  const EllNbr nb(D.nbr, D.nbr16);
  auto go = [&](auto kernel, int lpr) {
    timed_launch(m, FS_CLOCK_FINE_SWEEP, bytes, kernel, dim3(gfor(D.n * lpr)), dim3(kBlock), 0, s, D.n, D.w, nb, ac, anb,
                 b, x, om, xn, flags);
  };
  if (D.w <= 8) go(k_sweep<1, T, TO>, 1);
  else if (D.w <= 16) go(k_sweep<4, T, TO>, 4);
  else if (D.w <= 32) go(k_sweep<8, T, TO>, 8);
  else go(k_sweep<16, T, TO>, 16);
}

// a sweep on any grid-wide level, nothing prolongated
template <class T>
static void launch_sweep(fs_mesh *m, DLevel &D, int level, const T *b, const T *x, T om, T *xn, const int *flags) {
  if (level == 0)
    launch_sweep_fine<T, T>(m, D, b, x, om, xn, flags);
  else if (D.sell)
    hipLaunchKernelGGL((D.sell16 ? k_sweep_sell<T, true> : k_sweep_sell<T, false>), dim3(gfor(D.sell_slots)),
                       dim3(kBlock), 0, m->stream, D.sell_slots, D.sell_ptr.p, D.sell_row.p, D.sell_col.p,
                       LV<T>::val(D), LV<T>::ac(D), b, x, om, xn, flags);
  else
    launch_sweep_csr<T, false>(m, D, b, x, om, xn, Scatter<T>{}, flags);
}

template <class T>
static void launch_resid(fs_mesh *m, DLevel &D, const T *b, const T *x, T *r, const int *flags) {
  hipStream_t s = m->stream;
  const T *ac = LV<T>::ac(D), *anb = LV<T>::anb(D);
  if (D.sell) {
    hipLaunchKernelGGL((D.sell16 ? k_resid_sell<T, true> : k_resid_sell<T, false>), dim3(gfor(D.sell_slots)),
                       dim3(kBlock), 0, s, D.sell_slots, D.sell_ptr.p, D.sell_row.p, D.sell_col.p, LV<T>::val(D), ac,
                       b, x, r, flags);
    return;
  }
  const EllNbr nb(D.nbr, D.nbr16);
  if (D.w <= 8)
    hipLaunchKernelGGL((k_resid<1, T>), dim3(gfor(D.n)), dim3(kBlock), 0, s, D.n, D.w, nb, ac, anb, b, x, r, flags);
  else if (D.w <= 16)
    hipLaunchKernelGGL((k_resid<4, T>), dim3(gfor(D.n * 4)), dim3(kBlock), 0, s, D.n, D.w, nb, ac, anb, b, x, r,
                       flags);
  else if (D.w <= 32)
    hipLaunchKernelGGL((k_resid<8, T>), dim3(gfor(D.n * 8)), dim3(kBlock), 0, s, D.n, D.w, nb, ac, anb, b, x, r,
                       flags);
  else
    hipLaunchKernelGGL((k_resid<16, T>), dim3(gfor(D.n * 16)), dim3(kBlock), 0, s, D.n, D.w, nb, ac, anb, b, x, r,
                       flags);
}

template <class T>
static void gs_sweeps(fs_mesh *m, DLevel &D, const T *b, T *x, int sweeps, const int *flags) {
  hipStream_t s = m->stream;
  const T *ac = LV<T>::ac(D), *anb = LV<T>::anb(D);
  const int nc = (int)D.color_ptr.size() - 1;
  // symmetric sweeps; a colour is an independent set, so a colour swept
  // twice in a row (the last of a forward pass, the first of the next
  // forward pass) would recompute the same values and is swept once
  for (int sw = 0; sw < sweeps; ++sw) {
    for (int c = sw == 0 ? 0 : 1; c < nc; ++c) {
      const int bb = D.color_ptr[c], e = D.color_ptr[c + 1];
      hipLaunchKernelGGL(k_gsc<T>, dim3(gfor(e - bb)), dim3(kBlock), 0, s, e - bb, D.color_cells.p + bb, D.n,
                         D.w, D.nbr, ac, anb, b, x, flags);
    }
    for (int c = nc - 2; c >= 0; --c) {
      const int bb = D.color_ptr[c], e = D.color_ptr[c + 1];
      hipLaunchKernelGGL(k_gsc<T>, dim3(gfor(e - bb)), dim3(kBlock), 0, s, e - bb, D.color_cells.p + bb, D.n,
                         D.w, D.nbr, ac, anb, b, x, flags);
    }
  }
}

// Remaining pre-smoothing sweeps after the first (which the entry or the
// restriction kernel took); returns the buffer that holds the result.
template <class T>
static T *pre_smooth(fs_mesh *m, DLevel &D, int level, const T *b, int sweeps, T om, T *&other, const int *flags) {
  T *cur = LV<T>::x(D), *oth = LV<T>::t(D);
  if (use_gs(m, D)) {
    gs_sweeps<T>(m, D, b, cur, sweeps, flags); // x was zeroed by the caller
  } else {
    for (int k = 1; k < sweeps; ++k) {
      launch_sweep<T>(m, D, level, b, cur, om, oth, flags);
      std::swap(cur, oth);
    }
  }
  other = oth;
  return cur;
}

// Post-smoothing sweeps of a level whose iterate x already holds the coarse
// correction.  Level 0 (out given) ends in out; a coarser level in a buffer,
// which is returned, and with up given its result is prolongated into up (the
// next finer level's iterate).
template <class T>
static T *post_smooth(fs_mesh *m, DLevel &D, int level, const T *b, T *x, T *other, int sweeps, T om, T al, DLevel *F,
                      T *up, double *out, const int *flags) {
  hipStream_t s = m->stream;
  const bool gs = use_gs(m, D);
  T *cur = x, *oth = other;
  bool written = false; // the last sweep wrote out, or prolongated
  if (gs) {
    gs_sweeps<T>(m, D, b, x, sweeps, flags);
  } else {
    for (int k = 0; k < sweeps; ++k) {
      const bool last = k + 1 == sweeps;
      if (last && level == 0) {
        launch_sweep_fine<T, double>(m, D, b, cur, om, out, flags);
        return cur;
      }
      if (last && up && !D.sell) {
        launch_sweep_csr<T, true>(m, D, b, cur, om, oth, Scatter<T>{D.mptr.p, D.mem.p, up, al}, flags);
        written = true;
      } else {
        launch_sweep<T>(m, D, level, b, cur, om, oth, flags);
      }
      std::swap(cur, oth);
    }
  }
  if (level == 0)
    hipLaunchKernelGGL((k_convert<T, double>), dim3(gfor(D.n)), dim3(kBlock), 0, s, D.n, cur, out, flags);
  else if (up && !written)
    hipLaunchKernelGGL((k_prolong<T, T>), dim3(gfor(F->n)), dim3(kBlock), 0, s, F->n, F->parent.p, cur, up, al, up,
                       flags);
  return cur;
}

// Whether the finest level's residual is summed into the next level by one
// kernel (k_fine_restrict) instead of a pass over its rows and k_restrict:
// up to 150000 rows.  A coarse cell's members lie apart, so the fused kernel
// gathers its rows where the pass streams them: that is hidden while a launch
// waits on latency, and shows above.  Whole solves, two passes against fused:
// 64x64 cells 1.02 -> 0.96 ms, 40^3 hexahedra 1.69 -> 1.63 (FP32) and 2.01 ->
// 1.85 (FP64), 54^3 (157464 rows) 2.05 -> 2.05 and 2.48 -> 2.21, 60^3 2.49 ->
// 2.70, 74^3 3.48 -> 3.53 and 4.22 -> 4.38; tetrahedra 105456 rows 2.68 ->
// 2.60, 663552 rows 6.52 -> 6.71.
constexpr int kFineRestrictRows = 150000;
static bool fuse_fine_restrict(const fs_mesh *m, const DLevel &D) {
  return D.n <= kFineRestrictRows && D.w <= 8 && !use_gs(m, D);
}

// out = M^{-1} rhs: one V-cycle on the hierarchy held in precision T.  The
// first sweep of each level is fused into the kernel that produces its
// right-hand side, the prolongation into the kernel that finishes the coarser
// level, the FP64 output into the last sweep; the levels from the tail's
// applied level down are one dense product.  out must not alias rhs.
template <class T>
static void vcycle(fs_mesh *m, const double *rhs, double *out, double alpha, const int *flags) {
  if (solve_done(m)) return; // its kernels would return at once
  Hierarchy &H = *m->amg;
  hipStream_t s = m->stream;
  const int L = (int)H.lev.size();
  const int ts = H.tail.ts, dl = H.tail.dl;
  const T om = (T)m->mg_omega, al = (T)alpha;
  const int pre0 = m->mg_pre, post0 = m->mg_post;
  const int cpre = coarse_pre(m), cpost = coarse_post(m), coarse = coarsest_sweeps(m);
  const bool fp64 = sizeof(T) == 8;

  DLevel &D0 = H.lev[0];
  const T *b0 = fp64 ? (const T *)rhs : LV<T>::b(D0);
  // level 0 with no coarser level: smoothing only
  if (L == 1) {
    const bool gs = use_gs(m, D0);
    hipLaunchKernelGGL(k_enter<T>, dim3(gfor(D0.n)), dim3(kBlock), 0, s, D0.n, LV<T>::ac(D0), rhs,
                       fp64 ? nullptr : LV<T>::b(D0), LV<T>::x(D0), om, gs ? 0 : 1, flags);
    T *oth = nullptr;
    T *x = pre_smooth<T>(m, D0, 0, b0, coarse, om, oth, flags);
    hipLaunchKernelGGL((k_convert<T, double>), dim3(gfor(D0.n)), dim3(kBlock), 0, s, D0.n, x, out, flags);
    return;
  }
  std::vector<T *> res(L, nullptr), oth(L, nullptr);
  const bool dense = dl < L;
  const int bot = dense ? dl : L - 1;    // the level below the grid-wide ones
  const int top = ts < L ? ts : L - 1;   // levels of the cycle pattern above its bottom
  // the restriction from level l into l + 1 also starts level l + 1: mode 0
  // hands it to the dense product, 1 makes the first Jacobi sweep from zero,
  // 2 zeroes it (Gauss-Seidel)
  auto mode_from = [&](int l) {
    if (dense && l + 1 == dl) return 0;                       // the dense product takes over
    if (l + 1 == L - 1) return 1;                             // grid-wide coarsest: `coarse` sweeps
    return (!use_gs(m, H.lev[l + 1]) && cpre > 0) ? 1 : 2;
  };
  const EllNbr nb0(D0.nbr, D0.nbr16);
  const bool fine = fuse_fine_restrict(m, D0);
  auto fine_restrict = [&](auto kernel, const T *b, const T *x) {
    DLevel &C = H.lev[1];
    hipLaunchKernelGGL(kernel, dim3(gfor(C.n * kFineGroup)), dim3(kBlock), 0, s, C.n, C.mptr.p, C.mem.p, D0.n, D0.w,
                       nb0, LV<T>::ac(D0), LV<T>::anb(D0), rhs, b, fp64 ? nullptr : LV<T>::b(D0), x, LV<T>::x(D0),
                       LV<T>::b(C), LV<T>::ac(C), LV<T>::x(C), om, mode_from(0), flags);
  };
  auto restrict_from = [&](int l, const T *b, const T *x) {
    DLevel &D = H.lev[l], &C = H.lev[l + 1];
    const int mode = mode_from(l);
    if (l == 0 && fine) {
      fine_restrict(k_fine_restrict<T, false>, b, x);
    } else if (l > 0 && !use_gs(m, D) && !D.sell) {
      launch_resid_restrict<T>(m, D, C, b, x, om, mode, flags);
    } else {
      launch_resid<T>(m, D, b, x, LV<T>::r(D), flags);
      hipLaunchKernelGGL(k_restrict<T>, dim3(gfor(C.n)), dim3(kBlock), 0, s, C.n, C.mptr.p, C.mem.p, LV<T>::r(D),
                         LV<T>::b(C), LV<T>::ac(C), LV<T>::x(C), om, mode, flags);
    }
  };
  auto dense_apply = [&](bool acc, bool up, const T *b) {
    DLevel &D = H.lev[dl], &F = H.lev[dl - 1];
    const Scatter<T> sc{D.mptr.p, D.mem.p, up ? res[dl - 1] : nullptr, al};
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((D.n + kDenseRows - 1) / kDenseRows), dim3(kDenseThreads), 0, s, D.n,
                         (const double *)D.dense.p, b, LV<T>::x(D), F.parent.p, sc, flags);
    };
    if (acc) {
      if (up) go(k_dense_apply<T, true, true>);
      else go(k_dense_apply<T, true, false>);
    } else {
      if (up) go(k_dense_apply<T, false, true>);
      else go(k_dense_apply<T, false, false>);
    }
  };
  // the bottom level from zero; up: its result is prolongated into the level
  // above
  auto bottom = [&](bool up) {
    DLevel &D = H.lev[bot];
    if (dense) {
      dense_apply(false, up, LV<T>::b(D));
      res[bot] = LV<T>::x(D);
      return;
    }
    // the restriction took the first of the coarse sweeps
    T *o = nullptr;
    T *x = pre_smooth<T>(m, D, bot, LV<T>::b(D), coarse, om, o, flags);
    if (up)
      hipLaunchKernelGGL((k_prolong<T, T>), dim3(gfor(H.lev[bot - 1].n)), dim3(kBlock), 0, s, H.lev[bot - 1].n,
                         H.lev[bot - 1].parent.p, x, res[bot - 1], al, res[bot - 1], flags);
    res[bot] = x;
  };
  // post-smoothing from the bottom up to level stop (level 0 writes out);
  // every level's result goes on into the next finer one, but for level stop's
  auto ascend = [&](int stop) {
    for (int l = bot - 1; l >= stop; --l) {
      DLevel &D = H.lev[l];
      T *up = l > stop ? res[l - 1] : nullptr;
      res[l] = post_smooth<T>(m, D, l, l == 0 ? b0 : LV<T>::b(D), res[l], oth[l], l == 0 ? post0 : cpost, om, al,
                              l > 0 ? &H.lev[l - 1] : nullptr, up, out, flags);
      if (l > 0) oth[l] = res[l] == LV<T>::x(D) ? LV<T>::t(D) : LV<T>::x(D);
    }
  };
  // a second coarse-grid correction of level l1 >= 1 (F and W cycles):
  // pre-sweeps from its current iterate, then a fresh descent (every coarser
  // level from zero) to the bottom.  On the dense level itself this is one
  // more cycle from the iterate it has: x += C (b - A x).
  auto redescend = [&](int l1, bool up) {
    DLevel &D = H.lev[l1];
    const T *b = LV<T>::b(D);
    if (l1 == bot) {
      launch_resid<T>(m, D, b, res[l1], LV<T>::r(D), flags);
      dense_apply(true, up, LV<T>::r(D));
      return;
    }
    T *cur = res[l1], *o = oth[l1];
    if (use_gs(m, D)) {
      gs_sweeps<T>(m, D, b, cur, cpre, flags);
    } else {
      for (int k = 0; k < cpre; ++k) {
        launch_sweep<T>(m, D, l1, b, cur, om, o, flags);
        std::swap(cur, o);
      }
    }
    res[l1] = cur;
    oth[l1] = o;
    restrict_from(l1, b, cur);
    for (int l = l1 + 1; l < bot; ++l) {
      DLevel &Dl = H.lev[l];
      res[l] = pre_smooth<T>(m, Dl, l, LV<T>::b(Dl), cpre, om, oth[l], flags);
      restrict_from(l, LV<T>::b(Dl), res[l]);
    }
    bottom(up);
  };

  // one Jacobi pre-sweep on the finest level: the entry and the residual of
  // that sweep in one kernel
  const bool fuse0 = !use_gs(m, D0) && pre0 == 1 && bot > 0;
  // two Jacobi pre-sweeps or more: the entry and the first two in one kernel
  const bool enter2 = !use_gs(m, D0) && pre0 >= 2;
  if (enter2) {
    hipLaunchKernelGGL(k_enter_sweep<T>, dim3(gfor(D0.n)), dim3(kBlock), 0, s, D0.n, D0.w, nb0, LV<T>::ac(D0),
                       LV<T>::anb(D0), rhs, fp64 ? nullptr : LV<T>::b(D0), LV<T>::x(D0), om, flags);
  } else if (!fuse0) {
    const bool gs = use_gs(m, D0);
    hipLaunchKernelGGL(k_enter<T>, dim3(gfor(D0.n)), dim3(kBlock), 0, s, D0.n, LV<T>::ac(D0), rhs,
                       fp64 ? nullptr : LV<T>::b(D0), LV<T>::x(D0), om, (!gs && pre0 > 0) ? 1 : 0, flags);
  }
  for (int l = 0; l < bot; ++l) {
    DLevel &D = H.lev[l];
    const T *b = l == 0 ? b0 : LV<T>::b(D);
    const int npre = l == 0 ? pre0 - (enter2 ? 1 : 0) : cpre;
    if (l == 0 && fuse0) {
      res[0] = LV<T>::x(D0);
      oth[0] = LV<T>::t(D0);
      if (fine) {
        fine_restrict(k_fine_restrict<T, true>, nullptr, nullptr);
        continue;
      }
      DLevel &C = H.lev[1];
      hipLaunchKernelGGL(k_enter_resid<T>, dim3(gfor(D0.n)), dim3(kBlock), 0, s, D0.n, D0.w, nb0, LV<T>::ac(D0),
                         LV<T>::anb(D0), rhs, fp64 ? nullptr : LV<T>::b(D0), LV<T>::x(D0), LV<T>::r(D0), om, flags);
      hipLaunchKernelGGL(k_restrict<T>, dim3(gfor(C.n)), dim3(kBlock), 0, s, C.n, C.mptr.p, C.mem.p, LV<T>::r(D0),
                         LV<T>::b(C), LV<T>::ac(C), LV<T>::x(C), om, mode_from(0), flags);
      continue;
    }
    res[l] = pre_smooth<T>(m, D, l, b, npre, om, oth[l], flags);
    restrict_from(l, b, res[l]);
  }
  // F and W cycles (FS_OPT_MG_CYCLE 1, 2) in the pattern of the reference's
  // fMultiGridCycle and wMultiGridCycle (MultiGridCycle.for:84-127, 162-220):
  // back up to level l1 and down again, for l1 from the deepest level above
  // the tail up to level 1, and for W once more from level 2 down to the
  // deepest; the levels from the tail's first level down count as one
  std::vector<int> again;
  if (m->mg_cycle >= 1)
    for (int l1 = top - 1; l1 >= 1; --l1) again.push_back(l1);
  if (m->mg_cycle == 2)
    for (int l1 = 2; l1 <= top - 1; ++l1) again.push_back(l1);
  // the bottom's result goes up unless the next correction is the bottom's own
  auto goes_up = [&](size_t k) { return k >= again.size() || again[k] != bot; };
  if (solve_done(m)) return; // the rest would return at once
  bottom(goes_up(0));
  for (size_t k = 0; k < again.size(); ++k) {
    if (solve_done(m)) return;
    if (again[k] != bot) ascend(again[k]);
    redescend(again[k], goes_up(k + 1));
  }
  ascend(0);
}

void amg_apply(fs_mesh *m, const double *rhs, double *out, const int *flags, double alpha) {
  if (m->amg->fp32) vcycle<float>(m, rhs, out, alpha, flags);
  else vcycle<double>(m, rhs, out, alpha, flags);
}

// The reference's multigrid solve loop (AlgebraicMultiGridMainRoutine.for:
// 371-416): cycles while the fine L1 residual exceeds rrf*ires and at most
// MaxMultiGridCycles; each cycle corrects with one V-cycle of the residual.
void amg_solve(fs_mesh *m, const double *ac, const double *anb, const double *bc, double *dphi,
               int solver, bool warm) {
  (void)solver;
  // additive correction as in the reference unless asked otherwise
  const double alpha = m->mg_alpha > 0.0 ? m->mg_alpha : 1.0;
  amg_prepare(m, ac, anb, alpha);
  hipStream_t s = m->stream;
  const int n = m->n;
  double *r = m->wk.v[8], *c = m->wk.v[9];
  int *flags = m->wk.flags;
  const int gr = std::min(kPartials, gfor(n));
  // the first cycle's right-hand side: bc (dphi = 0), or the residual of the
  // initial guess
  if (warm)
    hipLaunchKernelGGL(k_amg_res, dim3(gr), dim3(kBlock), 0, s, n, m->w, m->d_nbr.p, ac, anb, bc, dphi, r,
                       m->wk.partial, (const int *)flags);
  const double *rhs = warm ? r : bc;
  run_cycles(m, gr, m->mg_maxcycles, [&]() {
    amg_apply(m, rhs, c, flags, alpha);
    hipLaunchKernelGGL(k_add2, dim3(gfor(n)), dim3(kBlock), 0, s, n, dphi, c, flags);
    hipLaunchKernelGGL(k_amg_res, dim3(gr), dim3(kBlock), 0, s, n, m->w, m->d_nbr.p, ac, anb,
                       bc, dphi, r, m->wk.partial, flags);
    rhs = r;
  });
}

int amg_export(fs_mesh *m, int level, int *dims, int *parent, int *seed, int *nchild,
               int *child_ptr, int *child, int *nbr, int *nnbr, double *ac, double *anb) {
  if (!m->amg || level < 0 || level >= (int)m->amg->host.size()) return -1;
  const HostLevel &h = m->amg->host[level];
  DLevel &D = m->amg->lev[level];
  int nch = 0;
  for (int p = 0; p < (int)h.children.size(); ++p) nch += (int)h.children[p].size();
  if (dims) {
    dims[0] = h.n;
    dims[1] = h.w;
    dims[2] = nch;
    dims[3] = (int)m->amg->lev.size();
    dims[4] = (int)D.color_ptr.size() - 1;
  }
  if (parent && !h.parent.empty()) std::copy(h.parent.begin(), h.parent.end(), parent);
  if (seed && !h.seed.empty()) std::copy(h.seed.begin(), h.seed.end(), seed);
  if (nchild && !h.nchild.empty()) std::copy(h.nchild.begin(), h.nchild.end(), nchild);
  if (child_ptr && child && !h.children.empty()) {
    int t = 0;
    child_ptr[0] = 0;
    for (int p = 0; p < h.n; ++p) {
      for (int c : h.children[p]) child[t++] = c;
      child_ptr[p + 1] = t;
    }
  }
  if (nbr) std::copy(h.nbr.begin(), h.nbr.end(), nbr);
  if (nnbr) std::copy(h.nnbr.begin(), h.nnbr.end(), nnbr);
  // coefficients: the device operators of the last prepare call for coarse
  // levels (level 0 belongs to the caller and may be gone: host copy of setup)
  if (level == 0) {
    if (ac) std::copy(h.ac.begin(), h.ac.end(), ac);
    if (anb) std::copy(h.anb.begin(), h.anb.end(), anb);
  } else {
    if (ac) FS_HIP_THROW(hipMemcpy(ac, D.ac64_own.p, sizeof(double) * h.n, hipMemcpyDeviceToHost));
    if (anb)
      FS_HIP_THROW(hipMemcpy(anb, D.anb64_own.p, sizeof(double) * h.n * h.w, hipMemcpyDeviceToHost));
  }
  return 0;
}

} // namespace fs
