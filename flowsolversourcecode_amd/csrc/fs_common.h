// Internal declarations shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "fsamd.h"

namespace fs {

void set_error(const std::string &msg);

#define FS_HIP(call)                                                          \
  do {                                                                        \
    hipError_t e_ = (call);                                                   \
    if (e_ != hipSuccess) {                                                   \
      ::fs::set_error(std::string(#call) + ": " + hipGetErrorString(e_));     \
      return -2;                                                              \
    }                                                                         \
  } while (0)

#define FS_HIP_THROW(call)                                                    \
  do {                                                                        \
    hipError_t e_ = (call);                                                   \
    if (e_ != hipSuccess)                                                     \
      throw std::runtime_error(std::string(#call) + ": " +                    \
                               hipGetErrorString(e_));                        \
  } while (0)

constexpr int kBlock = 256;     // threads per block for streaming kernels
// Most partials of a reduction: one row per thread up to 8.4 M rows.  The
// partials of a kernel lie gridDim.x apart, k-th sum at part[k gridDim.x + b].
constexpr int kPartials = 32768;

// Workgroups for n threads of kBlock, a multiple of 8 beyond a few (the extra
// ones find nothing to do) so that xcd_block() can give each XCD one
// contiguous range; left as it comes, seven grids of eight stayed in
// round-robin order, where every L2 fetches every other's neighbours.
inline int xcd_grid(long long n) {
  const int g = (int)((n + kBlock - 1) / kBlock);
  return g < 1 ? 1 : g < 64 ? g : (g + 7) & ~7;
}

// Device buffer owning a hipMalloc allocation.
template <class T> struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf &) = delete;
  DevBuf &operator=(const DevBuf &) = delete;
  DevBuf(DevBuf &&o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  DevBuf &operator=(DevBuf &&o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      n = o.n;
      o.p = nullptr;
      o.n = 0;
    }
    return *this;
  }
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  void alloc(size_t count) {
    if (count <= n && p) return;
    release();
    FS_HIP_THROW(hipMalloc(&p, sizeof(T) * (count ? count : 1)));
    n = count;
  }
  void upload(const T *h, size_t count, hipStream_t s) {
    alloc(count);
    FS_HIP_THROW(hipMemcpyAsync(p, h, sizeof(T) * count, hipMemcpyHostToDevice, s));
  }
  void upload(const std::vector<T> &h, hipStream_t s) { upload(h.data(), h.size(), s); }
};

struct Hierarchy; // fs_amg.hip

// What a solve tells the host without a copy or a synchronisation: pinned
// host memory that the one-block finalise kernels write.  `word` is the
// progress of the solve with the number in its upper half (post_word in
// fs_solve.hip); scal and extra are complete when it carries the final bit.
struct SolveBox {
  unsigned long long word;
  double scal[24];
  double extra[16];
};

// Per-launch HIP-event timing of one kernel site of the solve loops: events
// are recorded by the dispatch itself (hipExtLaunchKernelGGL).  How many
// iterations past the last one were launched (they return at once) is a matter
// of the host's timing, so a solve ends by setting the counts back to where
// they stood before those: what is counted did its work, and is the same
// every time.
struct KernelClock {
  struct Counts {
    int used = 0;                      // records
    int dropped[4] = {0, 0, 0, 0};     // launches beyond the capacity
    long long seen[4] = {0, 0, 0, 0};  // launches of each site since the start
  };
  int sites = 0, cap = 0;  // sites: bit (1 << site) per armed site
  int stride = 1;          // time every stride-th launch of a site
  Counts c;
  std::vector<Counts> before;  // the counts before each iteration of the solve in progress
  std::vector<hipEvent_t> ev;  // 2 per record
  std::vector<int> site;
  std::vector<double> bytes;
};

} // namespace fs

struct fs_mesh {
  int n = 0, w = 0;
  int device = 0;           // the device current at fs_mesh_create
  hipStream_t stream = nullptr;
  bool own_stream = true;   // false: the stream belongs to another context
  std::vector<int> h_nbr;   // reference layout, 1-based, 0 = boundary
  std::vector<int> h_nnbr;
  std::vector<int> h_nbr_dev; // 0-based, -1 = none (the device layout)
  fs::DevBuf<int> d_nbr;    // 0-based, -1 = none (slots past nnbr as well)
  fs::DevBuf<int> d_nbr16;  // the same as int16 offsets k - i (0 = none), two
                            // slots per word, when every offset fits
  fs::DevBuf<int> d_mir;    // transpose map, linear anb index or -1
  // face topology (optional)
  int nif = 0, nfaces_total = 0;
  std::vector<int> h_owner, h_neigh;
  fs::DevBuf<int> d_owner, d_neigh, d_iown, d_inbr;
  fs::DevBuf<int> d_face_code;  // per (cell, slot): face*4 + role
  // work vectors
  fs::DevBuf<double> v[12];
  fs::DevBuf<double> partial;  // 5 sums' partials
  fs::DevBuf<double> scal;     // scalar slots
  fs::DevBuf<int> flags;       // [0] done, [1] iterations
  fs::SolveBox *box = nullptr; // pinned; what the finalise kernels post to the host
  unsigned seq = 0;            // the solve the posts belong to
  // The scratch the solve uses: the mesh's buffers above, or slices of the
  // library's static device array for the duration of a
  // fs_solve_equation_device_noalloc call.
  struct Scratch {
    double *v[12];
    double *dc;       // D-ILU diagonal
    double *partial;
    double *scal;
    int *flags;
  } wk{};
  // options
  int mg_pre = 2, mg_post = 2, mg_maxcycles = 30, mg_maxlevels = 10;
  int mg_minparents = 10, mg_reagg = 300, mg_fp32 = 0, mg_smoother = 0;
  int mg_agg = 0;           // FS_OPT_MG_AGGREGATION
  int mg_cycle = 0;         // FS_OPT_MG_CYCLE: 0 V, 1 F, 2 W
  int warm_prev = 0;        // FS_OPT_WARM_PREVIOUS (read by the SIMPLE case)
  double mg_omega = 0.8;
  int mg_tail_cells = 1024, mg_coarse_sweeps = 16;
  int mg_cpre = -1, mg_cpost = -1; // sweeps on the coarse levels (-1: as on the finest)
  int mg_sell_rows = 100000;       // coarse levels at least this large use sliced ELL
  double mg_alpha = 0.0;           // over-correction (0: 1 as solver, 1.7 as preconditioner)
  int gmres_m = 30, check_every = 8;
  int ncalls_mg = 0;
  long long nnz = 0;                    // off-diagonal entries of the ELL pattern
  fs::KernelClock kclock;
  void *solve_work = nullptr;           // fs_solve.hip
  std::shared_ptr<fs::Hierarchy> amg;   // fs_amg.hip
};
