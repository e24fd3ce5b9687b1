// Learned warm start for the p' solve: a message-passing network over the
// cell graph, trained and run with hand-written kernels.  The dense layers
// run on the matrix cores (v_mfma_f32_16x16x32_bf16: BF16 operands, FP32
// accumulation); the message aggregation is a gather over the ELL slots,
// bound by memory like the solver's own kernels.  No counterpart in the
// reference; the definition is stated in include/fsamd_learn.h.
//
// Storage: weights FP32 master + BF16 copies in the layouts the matrix cores
// read (K contiguous per lane: forward Wt[out][in], backward Wb[in][out]);
// activations BF16 [cell][64] (128-byte rows); gradients of activations FP32.
// Every reduction runs over fixed per-block partials in a fixed order, so a
// step is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "fs_common.h"
#include "fs_kernels.h"
#include "fs_mpnn.h"
#include "fs_solve.h"

namespace fs {
namespace {

constexpr int kH = 64;     // hidden width
constexpr int kF = 8;      // input features (4 used, padded)
constexpr int kIn = 2 * kH; // input width of a message-passing layer
constexpr int kMaxLayers = 8;
constexpr int kStatBlocks = 64;
constexpr int kTile = 16;      // cells of a matrix-core tile
constexpr int kTiles = 2;      // tiles a wavefront of the dense kernels works through
constexpr int kRowsFwd = 4 * kTiles * kTile; // cells per block of the dense kernels
constexpr int kStage = 64;     // cells the weight-gradient kernel stages at a time
constexpr int kChunk = 256;    // cells per block (and partial gradient) of the gradient kernels

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef unsigned char u8x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

inline int cdiv(long long a, int b) { return (int)((a + b - 1) / b); }
// blocks of the gradient kernels for a batch of Bn cells.  Their workspace is
// sized for the largest batch so far, so this must not fall as Bn grows: the
// chunk is the same for every batch (blocks of more cells above 131072 cells
// saved 1-2 % of a step: 557 and 571 us at 135168, 3.52 and 3.56 ms at 1048576).
inline int grad_blocks(long long Bn) { return cdiv(Bn, kChunk); }

// float -> bfloat16 bits, round to nearest even (NaN kept quiet)
__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u && (u & 0x7fffffu)) return (unsigned short)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

__device__ __forceinline__ bf16x8 load_bf8(const unsigned short *p) {
  const uint4 v = *reinterpret_cast<const uint4 *>(p);
  return __builtin_bit_cast(bf16x8, v);
}

// ---------------------------------------------------------------- features
// per (sample, block) partial sums of b^2, ac, vol, x
constexpr int kStats = 5; // per sample: s_b, s_a, mean vol, mean x, mean xp

template <class T>
__global__ void k_stats(int N, const int *__restrict__ ids, const T *__restrict__ b, const T *__restrict__ ac,
                        const T *__restrict__ vol, const T *__restrict__ x, const T *__restrict__ xp,
                        double *__restrict__ part) {
  const int s = blockIdx.y, id = ids[s];
  const size_t base = (size_t)id * N;
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0, a4 = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock) {
    const double bi = (double)b[base + i];
    a0 += bi * bi;
    a1 += (double)ac[base + i];
    a2 += (double)vol[base + i];
    if (x) a3 += (double)x[base + i];
    if (xp) a4 += (double)xp[base + i];
  }
  a0 = block_sum<kBlock>(a0);
  a1 = block_sum<kBlock>(a1);
  a2 = block_sum<kBlock>(a2);
  a3 = block_sum<kBlock>(a3);
  a4 = block_sum<kBlock>(a4);
  if (threadIdx.x == 0) {
    double *p = part + ((size_t)s * gridDim.x + blockIdx.x) * kStats;
    p[0] = a0;
    p[1] = a1;
    p[2] = a2;
    p[3] = a3;
    p[4] = a4;
  }
}

// scal[s] = {s_b, s_a, mean vol, mean x, mean xp}; one wavefront per sample:
// the partials are loaded together and each quantity is summed in block order
// by a thread of its own
__global__ void __launch_bounds__(64)
k_stats_fin(int N, int nb, const double *__restrict__ part, double *__restrict__ scal) {
  __shared__ double v[kStatBlocks * kStats];
  const int s = blockIdx.x, q = threadIdx.x;
  for (int k = threadIdx.x; k < nb * kStats; k += 64) v[k] = part[(size_t)s * nb * kStats + k];
  __syncthreads();
  if (q >= kStats) return;
  double a = 0.0;
  for (int k = 0; k < nb; ++k) a += v[k * kStats + q];
  scal[s * kStats + q] = q == 0 ? sqrt(a / N) + 1e-300 : a / N;
}

// X0, edge weights E[j][c] and the normalised target of the batch cells
template <class T>
__global__ void k_feat(int N, int W, int Bn, const int *__restrict__ ids, const int *__restrict__ nbr0,
                       const T *__restrict__ b, const T *__restrict__ ac, const T *__restrict__ anb,
                       const T *__restrict__ vol, const T *__restrict__ x, const T *__restrict__ xp,
                       const double *__restrict__ scal, float *__restrict__ X0, float *__restrict__ E,
                       float *__restrict__ Tg) {
  const int c = blockIdx.x * kBlock + threadIdx.x;
  if (c >= Bn) return;
  const int s = c / N, i = c - s * N, id = ids[s];
  const size_t base = (size_t)id * N;
  const double *sc = scal + (size_t)s * kStats;
  const double sb = sc[0], sa = sc[1], vm = sc[2], xm = sc[3], xpm = sc[4];
  const double aci = (double)ac[base + i];
  int nn = 0;
  for (int j = 0; j < W; ++j) {
    const int k = nbr0[(size_t)j * N + i];
    float e = 0.f;
    if (k >= 0) {
      ++nn;
      e = (float)(-(double)anb[((size_t)id * W + j) * N + i] / aci);
    }
    E[(size_t)j * Bn + c] = e;
  }
  float *xr = X0 + (size_t)c * kF;
  xr[0] = (float)((double)b[base + i] / sb);
  xr[1] = (float)(aci / sa);
  xr[2] = (float)((double)nn / W);
  xr[3] = (float)((double)vol[base + i] / vm);
  xr[4] = xp ? (float)(((double)xp[base + i] - xpm) * sa / sb) : 0.f;
  xr[5] = xr[6] = xr[7] = 0.f;
  if (Tg) Tg[c] = x ? (float)(((double)x[base + i] - xm) * sa / sb) : 0.f;
}

// ---------------------------------------------------------------- forward
// H0 = bf16(relu(X0 We + be)); thread per (cell, 8 outputs)
__global__ void k_enc(int Bn, const float *__restrict__ X0, const float *__restrict__ weq,
                      const float *__restrict__ be, unsigned short *__restrict__ H0) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const int c = (int)(t >> 3), g = (int)(t & 7);
  if (c >= Bn) return;
  const float *xr = X0 + (size_t)c * kF;
  u16x8 out;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int o = g * 8 + q;
    float z = 0.f;
#pragma unroll
    for (int f = 0; f < kF; ++f) z += xr[f] * weq[f * kH + o];
    z += be[o];
    out[q] = f2bf(fmaxf(z, 0.f));
  }
  *reinterpret_cast<u16x8 *>(H0 + (size_t)c * kH + g * 8) = out;
}

// M[c] = bf16(sum_j E[j][c] H[nbr_j(c)]); thread per (cell, 8 features)
__global__ void k_agg(int N, int W, int Bn, const int *__restrict__ nbr0, const float *__restrict__ E,
                      const unsigned short *__restrict__ H, unsigned short *__restrict__ M) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const int c = (int)(t >> 3), g = (int)(t & 7);
  if (c >= Bn) return;
  const int s = c / N, i = c - s * N;
  float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int j = 0; j < W; ++j) {
    const int k = nbr0[(size_t)j * N + i];
    if (k < 0) continue;
    const float e = E[(size_t)j * Bn + c];
    const u16x8 h = *reinterpret_cast<const u16x8 *>(H + ((size_t)s * N + k) * kH + g * 8);
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] += e * bf2f(h[q]);
  }
  u16x8 out;
#pragma unroll
  for (int q = 0; q < 8; ++q) out[q] = f2bf(acc[q]);
  *reinterpret_cast<u16x8 *>(M + (size_t)c * kH + g * 8) = out;
}

// z = [H M] W + b on the matrix cores; Hn = bf16(H + relu(z)); mask = z > 0.
// The product is formed transposed (rows: the 64 outputs, columns: 16 cells),
// so that a lane holds four consecutive outputs of one cell and its state,
// result and mask move 8, 8 and 4 bytes at a time; a wavefront keeps the
// layer's weights in registers (64) for its kTiles tiles.  65536 cells:
// 13.9 us (one cell column a lane, 2-byte accesses: 16.4 us).
__global__ void __launch_bounds__(256)
k_dense_fwd(int Bn, const unsigned short *__restrict__ H, const unsigned short *__restrict__ M,
            const unsigned short *__restrict__ wt, const float *__restrict__ bias, unsigned short *__restrict__ Hn,
            unsigned char *__restrict__ mask) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, kg = lane >> 4;
  bf16x8 wv[4][4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) wv[ks][mt] = load_bf8(wt + (size_t)(mt * 16 + (lane & 15)) * kIn + ks * 32 + kg * 8);
  const int c0 = blockIdx.x * kRowsFwd + wave * kTiles * kTile + (lane & 15);
  bf16x8 xv[kTiles][4];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const size_t row = (size_t)min(c0 + t * kTile, Bn - 1); // cells past the end repeat the last one
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      xv[t][ks] = load_bf8((ks < 2 ? H + row * kH + ks * 32 : M + row * kH + (ks - 2) * 32) + kg * 8);
  }
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const int c = c0 + t * kTile;
    floatx4 acc[4];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[ks][mt], xv[t][ks], acc[mt], 0, 0, 0);
    if (c >= Bn) continue;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      const int o = mt * 16 + kg * 4;
      const size_t at = (size_t)c * kH + o;
      const floatx4 bo = *reinterpret_cast<const floatx4 *>(bias + o);
      const u16x4 h = *reinterpret_cast<const u16x4 *>(H + at);
      u16x4 hn;
      u8x4 mk;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float z = acc[mt][r] + bo[r];
        hn[r] = f2bf(bf2f(h[r]) + fmaxf(z, 0.f));
        mk[r] = z > 0.f;
      }
      *reinterpret_cast<u16x4 *>(Hn + at) = hn;
      *reinterpret_cast<u8x4 *>(mask + at) = mk;
    }
  }
}

// y = H wd + bd per cell, partial sums of y per (sample, block)
__global__ void k_decode(int N, int Bn, const unsigned short *__restrict__ H, const float *__restrict__ wdq,
                         const float *__restrict__ bdp, float *__restrict__ Y, double *__restrict__ part) {
  const int s = blockIdx.y;
  const float bd = *bdp;
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock) {
    const int c = s * N + i;
    const unsigned short *h = H + (size_t)c * kH;
    float y = 0.f;
#pragma unroll 8
    for (int o = 0; o < kH; ++o) y += bf2f(h[o]) * wdq[o];
    y += bd;
    Y[c] = y;
    acc += y;
  }
  acc = block_sum<kBlock>(acc);
  if (threadIdx.x == 0) part[(size_t)s * gridDim.x + blockIdx.x] = acc;
  (void)Bn;
}

// ymean[s] from the partials, loaded together and summed in block order
__global__ void __launch_bounds__(64)
k_mean_fin(int N, int nb, const double *__restrict__ part, double *__restrict__ ymean) {
  static_assert(kStatBlocks <= 64, "one partial a lane");
  __shared__ double v[64];
  const int s = blockIdx.x;
  v[threadIdx.x] = (int)threadIdx.x < nb ? part[(size_t)s * nb + threadIdx.x] : 0.0;
  __syncthreads();
  if (threadIdx.x != 0) return;
  double a = 0.0;
  for (int k = 0; k < nb; ++k) a += v[k];
  ymean[s] = a / N;
}

// yc = y - mean; loss partials and dy = 2 (yc - t)/total (training), or the
// prediction x = yc s_b/s_a (inference, out != null)
__global__ void k_loss(int N, const double *__restrict__ ymean, const double *__restrict__ scal,
                       float *__restrict__ Y, const float *__restrict__ Tg, float *__restrict__ DY, double inv_total,
                       double *__restrict__ part, double *__restrict__ out) {
  const int s = blockIdx.y;
  const double ym = ymean[s];
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < N; i += gridDim.x * kBlock) {
    const int c = s * N + i;
    const float yc = (float)((double)Y[c] - ym);
    Y[c] = yc;
    if (out) {
      out[(size_t)s * N + i] = (double)yc * scal[s * kStats] / scal[s * kStats + 1];
    } else {
      const double d = (double)yc - (double)Tg[c];
      acc += d * d;
      DY[c] = (float)(2.0 * d * inv_total);
    }
  }
  if (!out) {
    acc = block_sum<kBlock>(acc);
    if (threadIdx.x == 0) part[(size_t)s * gridDim.x + blockIdx.x] = acc;
  }
}

// ---------------------------------------------------------------- backward
// four of a row's activation gradients and, with mask, the layer's dz =
// bf16(mask ? dH : 0) formed from them
__device__ __forceinline__ void store_dh(size_t at, floatx4 d, float *__restrict__ dH,
                                         const unsigned char *__restrict__ mask, unsigned short *__restrict__ DZ) {
  *reinterpret_cast<floatx4 *>(dH + at) = d;
  if (!mask) return;
  const u8x4 m = *reinterpret_cast<const u8x4 *>(mask + at);
  u16x4 z;
#pragma unroll
  for (int q = 0; q < 4; ++q) z[q] = f2bf(m[q] ? d[q] : 0.f);
  *reinterpret_cast<u16x4 *>(DZ + at) = z;
}

// dH[c][o] = dy[c] wd[o], and dz of the last layer; thread per (cell, 4 outputs)
__global__ void k_dec_bwd(int Bn, const float *__restrict__ DY, const float *__restrict__ wdq, float *__restrict__ dH,
                          const unsigned char *__restrict__ mask, unsigned short *__restrict__ DZ) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const int c = (int)(t >> 4), o = (int)(t & 15) * 4;
  if (c >= Bn) return;
  const float dy = DY[c];
  floatx4 d;
#pragma unroll
  for (int q = 0; q < 4; ++q) d[q] = dy * wdq[o + q];
  store_dh((size_t)c * kH + o, d, dH, mask, DZ);
}

// Decoder gradient: per-block sums out[blk][o] = sum of dy[c] H[c][o] over the
// block's cells, out[blk][64] = sum of dy[c].  Block: 256 threads = 4 cell
// lanes x 64 columns, the loads of 8 cells in flight.
__global__ void k_dec_grad(int Bn, const float *__restrict__ DY, const unsigned short *__restrict__ H,
                           float *__restrict__ out) {
  const int o = threadIdx.x & 63, r = threadIdx.x >> 6;
  const int c0 = blockIdx.x * kChunk, c1 = min(Bn, c0 + kChunk);
  float s = 0.f, sa = 0.f;
  constexpr int B = 8;
  for (int cb = c0 + r; cb < c1; cb += 4 * B) {
    float dy[B], h[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const int c = min(cb + 4 * u, c1 - 1);
      dy[u] = DY[c];
      h[u] = bf2f(H[(size_t)c * kH + o]);
    }
#pragma unroll
    for (int u = 0; u < B; ++u)
      if (cb + 4 * u < c1) {
        s += dy[u] * h[u];
        sa += dy[u];
      }
  }
  __shared__ float red[4][kH + 1];
  red[r][o] = s;
  if (o == 0) red[r][kH] = sa;
  __syncthreads();
  for (int k = threadIdx.x; k <= kH; k += 256)
    out[(size_t)blockIdx.x * (kH + 1) + k] = red[0][k] + red[1][k] + red[2][k] + red[3][k];
}

// D = dz W^T on the matrix cores: [Bn x 64] x [64 x 128] -> FP32 [Bn x 128],
// formed transposed like k_dense_fwd (16-byte stores; 65536 cells: 12.6 us,
// 14.9 us with 4-byte stores and the weights loaded for every tile).
__global__ void __launch_bounds__(256)
k_dense_bwd_x(int Bn, const unsigned short *__restrict__ DZ, const unsigned short *__restrict__ wb,
              float *__restrict__ D) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, kg = lane >> 4;
  bf16x8 wv[2][8];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) wv[ks][mt] = load_bf8(wb + (size_t)(mt * 16 + (lane & 15)) * kH + ks * 32 + kg * 8);
  const int c0 = blockIdx.x * kRowsFwd + wave * kTiles * kTile + (lane & 15);
  bf16x8 zv[kTiles][2];
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const size_t row = (size_t)min(c0 + t * kTile, Bn - 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) zv[t][ks] = load_bf8(DZ + row * kH + ks * 32 + kg * 8);
  }
#pragma unroll
  for (int t = 0; t < kTiles; ++t) {
    const int c = c0 + t * kTile;
    floatx4 acc[8];
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) acc[mt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mt = 0; mt < 8; ++mt)
        acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[ks][mt], zv[t][ks], acc[mt], 0, 0, 0);
    if (c >= Bn) continue;
#pragma unroll
    for (int mt = 0; mt < 8; ++mt)
      *reinterpret_cast<floatx4 *>(D + (size_t)c * kIn + mt * 16 + kg * 4) = acc[mt];
  }
}

// dH_prev[c] = dH[c] + D[c][0:64] + sum over neighbours k of c of
// e_{k,c} D[k][64:128] (the transpose of the aggregation; e_{k,c} is the
// weight of c in k's row, found through the mirror slot), and dz of the layer
// below (mask, DZ; none below the first)
__global__ void k_agg_t(int N, int W, int Bn, const int *__restrict__ nbr0, const int *__restrict__ mir,
                        const float *__restrict__ E, const float *__restrict__ dH, const float *__restrict__ D,
                        float *__restrict__ dHp, const unsigned char *__restrict__ mask,
                        unsigned short *__restrict__ DZ) {
  const long long t = (long long)blockIdx.x * kBlock + threadIdx.x;
  const int c = (int)(t >> 4), g = (int)(t & 15) * 4;
  if (c >= Bn) return;
  const int s = c / N, i = c - s * N;
  const floatx4 h = *reinterpret_cast<const floatx4 *>(dH + (size_t)c * kH + g);
  floatx4 acc = h + *reinterpret_cast<const floatx4 *>(D + (size_t)c * kIn + g);
  for (int j = 0; j < W; ++j) {
    const int k = nbr0[(size_t)j * N + i];
    if (k < 0) continue;
    const int jm = mir[(size_t)j * N + i];
    const size_t ck = (size_t)s * N + k;
    const float e = E[(size_t)jm * Bn + ck];
    acc += e * *reinterpret_cast<const floatx4 *>(D + ck * kIn + kH + g);
  }
  store_dh((size_t)c * kH + g, acc, dHp, mask, DZ);
}

// Partial dW = [H M]^T dz and db = column sums of dz over the block's cells,
// out[blk] = {dW[in][o], db[o]}, FP32.  The matrix cores contract over cells,
// so both operands are needed feature-major: the block stages kStage cells at
// a time in LDS, each thread transposing one 8 cells x 8 features tile in
// registers (16-byte loads and LDS stores; the next stage's loads are in
// flight behind the products).  Wave w owns input features 32w..32w+31 (2 x 4
// output tiles).  65536 cells: 9.5 us (2-byte staging of 32 cells: 53.6 us,
// and another 20 us for the column sums).
constexpr int kStageStride = kStage + 8; // bf16 elements per staged row: 16-byte rows, spread over the banks
constexpr int kGradW = kIn * kH + kH;    // values of a layer's gradient (W, b)

__global__ void __launch_bounds__(256)
k_dense_bwd_w(int Bn, const unsigned short *__restrict__ H, const unsigned short *__restrict__ M,
              const unsigned short *__restrict__ DZ, float *__restrict__ out) {
  __shared__ __attribute__((aligned(16))) unsigned short st[(kIn + kH) * kStageStride];
  __shared__ float bred[4][kH];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, kg = lane >> 4;
  const int c0 = blockIdx.x * kChunk, c1 = min(Bn, c0 + kChunk);
  // the thread's tile: cells 8 cg.., feature group fg of [H | M | dz]
  const int cg = threadIdx.x & 7, fg = threadIdx.x >> 3;
  const bool loads = fg < (kIn + kH) / 8;
  const unsigned short *src = fg < 8 ? H + fg * 8 : fg < 16 ? M + (fg - 8) * 8 : DZ + (fg - 16) * 8;
  uint4 w[8];
  auto fetch = [&](int cs) {
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int c = cs + cg * 8 + r;
      w[r] = uint4{0u, 0u, 0u, 0u};
      if (loads && c < c1) w[r] = *reinterpret_cast<const uint4 *>(src + (size_t)c * kH);
    }
  };
  floatx4 acc[2][4];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = floatx4{0.f, 0.f, 0.f, 0.f};
  float bs = 0.f;
  fetch(c0);
  for (int cs = c0; cs < c1; cs += kStage) {
    __syncthreads(); // the last stage has been read
    if (loads) {
      auto word = [&](int r, int q) { return q == 0 ? w[r].x : q == 1 ? w[r].y : q == 2 ? w[r].z : w[r].w; };
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        unsigned lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const unsigned a = word(2 * k, q), b = word(2 * k + 1, q);
          lo[k] = (a & 0xffffu) | (b << 16);
          hi[k] = (a >> 16) | (b & 0xffff0000u);
        }
        unsigned short *dst = st + (size_t)(fg * 8 + 2 * q) * kStageStride + cg * 8;
        *reinterpret_cast<uint4 *>(dst) = uint4{lo[0], lo[1], lo[2], lo[3]};
        *reinterpret_cast<uint4 *>(dst + kStageStride) = uint4{hi[0], hi[1], hi[2], hi[3]};
      }
    }
    __syncthreads();
    if (cs + kStage < c1) fetch(cs + kStage);
    const unsigned short *zs = st + (size_t)kIn * kStageStride;
#pragma unroll
    for (int ks = 0; ks < kStage / 32; ++ks) {
      bf16x8 bv[4];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) bv[nt] = load_bf8(zs + (nt * 16 + (lane & 15)) * kStageStride + ks * 32 + kg * 8);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const bf16x8 a = load_bf8(st + (wave * 32 + mt * 16 + (lane & 15)) * kStageStride + ks * 32 + kg * 8);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv[nt], acc[mt][nt], 0, 0, 0);
      }
    }
    // column sums: lane o, every fourth cell per wave
#pragma unroll
    for (int k = 0; k < kStage / 4; ++k) bs += bf2f(zs[lane * kStageStride + 4 * k + wave]);
  }
  bred[wave][lane] = bs;
  __syncthreads();
  float *dst = out + (size_t)blockIdx.x * kGradW;
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int o = nt * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int f = wave * 32 + mt * 16 + kg * 4 + r;
        dst[f * kH + o] = acc[mt][nt][r];
      }
    }
  if (threadIdx.x < kH)
    dst[kIn * kH + threadIdx.x] =
        bred[0][threadIdx.x] + bred[1][threadIdx.x] + bred[2][threadIdx.x] + bred[3][threadIdx.x];
}

// encoder gradient partials: out[blk][f][o] = sum X0[c][f] dz0[c][o] (f < 8),
// out[blk][8][o] = sum dz0[c][o], dz0 = (H0 > 0) ? dH : 0
__global__ void k_enc_bwd(int Bn, const float *__restrict__ X0, const unsigned short *__restrict__ H0,
                          const float *__restrict__ dH, float *__restrict__ out) {
  const int o = threadIdx.x & 63, r = threadIdx.x >> 6;
  const int c0 = blockIdx.x * kChunk, c1 = min(Bn, c0 + kChunk);
  static_assert(kF == 8, "features in two 16-byte loads");
  float s[kF + 1];
#pragma unroll
  for (int f = 0; f <= kF; ++f) s[f] = 0.f;
  constexpr int B = 8; // cells in flight
  for (int cb = c0 + r; cb < c1; cb += 4 * B) {
    float dz[B];
    floatx4 xa[B], xb[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
      const size_t c = (size_t)min(cb + 4 * u, c1 - 1);
      const float h = bf2f(H0[c * kH + o]), d = dH[c * kH + o];
      dz[u] = h > 0.f && cb + 4 * u < c1 ? d : 0.f;
      xa[u] = *reinterpret_cast<const floatx4 *>(X0 + c * kF);
      xb[u] = *reinterpret_cast<const floatx4 *>(X0 + c * kF + 4);
    }
#pragma unroll
    for (int u = 0; u < B; ++u) {
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        s[f] += xa[u][f] * dz[u];
        s[4 + f] += xb[u][f] * dz[u];
      }
      s[kF] += dz[u];
    }
  }
  __shared__ float red[4][kF + 1][kH];
#pragma unroll
  for (int f = 0; f <= kF; ++f) red[r][f][o] = s[f];
  __syncthreads();
  if (r == 0)
    for (int f = 0; f <= kF; ++f)
      out[((size_t)blockIdx.x * (kF + 1) + f) * kH + o] = red[0][f][o] + red[1][f][o] + red[2][f][o] + red[3][f][o];
}

// dst[k] = sum over the nb blocks' partials part[b][k] in block order, k < K.  A
// block sums 32 columns: its threads load kReduceRows rows of them together
// into LDS, where one thread a column adds them up one after the other: 3.6-6.5
// us for 256 blocks (one thread a column over all rows: 60 us).
constexpr int kReduceRows = 256;
__global__ void __launch_bounds__(kBlock)
k_reduce(int nb, int K, const float *__restrict__ part, float *__restrict__ dst) {
  constexpr int C = 32, G = kBlock / C;
  __shared__ float v[kReduceRows][C];
  const int kk = threadIdx.x % C, g = threadIdx.x / C, k = blockIdx.x * C + kk;
  float s = 0.f;
  for (int b0 = 0; b0 < nb; b0 += kReduceRows) {
    const int rows = min(kReduceRows, nb - b0);
    if (k < K) {
      float r[kReduceRows / G];
#pragma unroll
      for (int u = 0; u < kReduceRows / G; ++u) r[u] = part[(size_t)(b0 + min(g + u * G, rows - 1)) * K + k];
#pragma unroll
      for (int u = 0; u < kReduceRows / G; ++u) v[g + u * G][kk] = r[u];
    }
    __syncthreads();
    if (g == 0 && k < K) {
      int b = 0;
      for (; b + 16 <= rows; b += 16) {
        float t[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = v[b + u][kk];
#pragma unroll
        for (int u = 0; u < 16; ++u) s += t[u];
      }
      for (; b < rows; ++b) s += v[b][kk];
    }
    __syncthreads();
  }
  if (g == 0 && k < K) dst[k] = s;
}

__global__ void k_adam(int n, float *__restrict__ th, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, float lr, float c1, float c2) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = 0.9f * m[i] + 0.1f * gi;
  const float vi = 0.999f * v[i] + 0.001f * gi * gi;
  m[i] = mi;
  v[i] = vi;
  th[i] = th[i] - lr * (mi / c1) / (sqrtf(vi / c2) + 1e-8f);
}

// BF16 copies of the weights in the layouts the kernels read
__global__ void k_quant(int L, const float *__restrict__ th, float *__restrict__ weq, unsigned short *__restrict__ wt,
                        unsigned short *__restrict__ wb, float *__restrict__ wdq) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const int per = kIn * kH;
  if (i < kF * kH) weq[i] = bf2f(f2bf(th[i]));
  if (i < kH) wdq[i] = bf2f(f2bf(th[kF * kH + kH + L * (per + kH) + i]));
  if (i >= L * per) return;
  const int l = i / per, r = i - l * per, k = r / kH, o = r - k * kH;
  const unsigned short q = f2bf(th[kF * kH + kH + l * (per + kH) + r]);
  wt[(size_t)l * per + o * kIn + k] = q;
  wb[(size_t)l * per + k * kH + o] = q;
}

__global__ void k_to_f32(long long n, const double *__restrict__ a, float *__restrict__ b) {
  const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}

} // namespace
} // namespace fs

// ====================================================================== host
struct fs_mpnn {
  int N = 0, W = 0, L = 3, P = 0, cap = 0, count = 0, steps = 0;
  bool use_prev = false;  // fifth input: the previous p' solution
  hipStream_t s = nullptr;
  std::vector<int> h_nbr0;
  fs::DevBuf<int> nbr0, mir, ids;
  fs::DevBuf<float> theta, grad, am, av, weq, wdq;
  fs::DevBuf<unsigned short> wt, wb;
  fs::DevBuf<float> ds_b, ds_x, ds_ac, ds_anb, ds_vol, ds_xp;
  // batch work buffers (grown on demand)
  long long bn_cap = 0;
  fs::DevBuf<double> part, scal, ymean;
  fs::DevBuf<float> X0, E, Tg, Y, DY, dH, dH2, D, gpart;
  std::vector<fs::DevBuf<unsigned short>> Hs, Ms;
  std::vector<fs::DevBuf<unsigned char>> masks;
  fs::DevBuf<unsigned short> DZ;
  std::vector<double> h_part;
};

namespace fs {

int mpnn_offset_W(int l) { return kF * kH + kH + l * (kIn * kH + kH); }

static void mpnn_grow(fs_mpnn *n, int B) {
  const long long Bn = (long long)B * n->N;
  n->ids.alloc(B);
  n->part.alloc((size_t)B * kStatBlocks * kStats);
  n->scal.alloc((size_t)B * kStats);
  n->ymean.alloc(B);
  if (Bn <= n->bn_cap) return;
  n->X0.alloc(Bn * kF);
  n->E.alloc(Bn * n->W);
  n->Tg.alloc(Bn);
  n->Y.alloc(Bn);
  n->DY.alloc(Bn);
  n->dH.alloc(Bn * kH);
  n->dH2.alloc(Bn * kH);
  n->D.alloc(Bn * kIn);
  n->DZ.alloc(Bn * kH);
  n->Hs.resize(n->L + 1);
  n->Ms.resize(n->L);
  n->masks.resize(n->L);
  for (auto &h : n->Hs) h.alloc(Bn * kH);
  for (auto &m : n->Ms) m.alloc(Bn * kH);
  for (auto &m : n->masks) m.alloc(Bn * kH);
  n->gpart.alloc((size_t)grad_blocks(Bn) * kGradW);
  n->bn_cap = Bn;
}

static void quantize(fs_mpnn *n) {
  hipLaunchKernelGGL(k_quant, dim3(cdiv((long long)n->L * kIn * kH, kBlock)), dim3(kBlock), 0, n->s, n->L,
                     n->theta.p, n->weq.p, n->wt.p, n->wb.p, n->wdq.p);
}

// Forward over the batch already described by ids / features.  Returns the
// number of stat blocks per sample.
template <class T>
static void mpnn_forward(fs_mpnn *n, int B, const T *b, const T *ac, const T *anb, const T *vol, const T *x,
                         const T *xp) {
  hipStream_t s = n->s;
  const int N = n->N, W = n->W;
  const int Bn = B * N;
  const int nb = std::min(kStatBlocks, cdiv(N, kBlock));
  if (!n->use_prev) xp = nullptr;
  hipLaunchKernelGGL(k_stats<T>, dim3(nb, B), dim3(kBlock), 0, s, N, n->ids.p, b, ac, vol, x, xp, n->part.p);
  hipLaunchKernelGGL(k_stats_fin, dim3(B), dim3(64), 0, s, N, nb, n->part.p, n->scal.p);
  hipLaunchKernelGGL(k_feat<T>, dim3(cdiv(Bn, kBlock)), dim3(kBlock), 0, s, N, W, Bn, n->ids.p, n->nbr0.p, b, ac,
                     anb, vol, x, xp, n->scal.p, n->X0.p, n->E.p, x ? n->Tg.p : nullptr);
  hipLaunchKernelGGL(k_enc, dim3(cdiv((long long)Bn * 8, kBlock)), dim3(kBlock), 0, s, Bn, n->X0.p, n->weq.p,
                     n->theta.p + kF * kH, n->Hs[0].p);
  for (int l = 0; l < n->L; ++l) {
    hipLaunchKernelGGL(k_agg, dim3(cdiv((long long)Bn * 8, kBlock)), dim3(kBlock), 0, s, N, W, Bn, n->nbr0.p, n->E.p,
                       n->Hs[l].p, n->Ms[l].p);
    hipLaunchKernelGGL(k_dense_fwd, dim3(cdiv(Bn, kRowsFwd)), dim3(256), 0, s, Bn, n->Hs[l].p, n->Ms[l].p,
                       n->wt.p + (size_t)l * kIn * kH, n->theta.p + mpnn_offset_W(l) + kIn * kH, n->Hs[l + 1].p,
                       n->masks[l].p);
  }
  hipLaunchKernelGGL(k_decode, dim3(nb, B), dim3(kBlock), 0, s, N, Bn, n->Hs[n->L].p, n->wdq.p,
                     n->theta.p + n->P - 1, n->Y.p, n->part.p);
  hipLaunchKernelGGL(k_mean_fin, dim3(B), dim3(64), 0, s, N, nb, n->part.p, n->ymean.p);
}

// The batch's loss partials and, with want_grad, the gradient into n->grad, on
// the network's stream.
static void mpnn_loss_grad(fs_mpnn *n, const int *ids, int B, bool want_grad) {
  hipStream_t s = n->s;
  for (int k = 0; k < B; ++k)
    if (ids[k] < 0 || ids[k] >= n->count) throw std::runtime_error("sample id out of range");
  mpnn_grow(n, B);
  FS_HIP_THROW(hipMemcpyAsync(n->ids.p, ids, sizeof(int) * B, hipMemcpyHostToDevice, s));
  const int N = n->N, Bn = B * N;
  mpnn_forward<float>(n, B, n->ds_b.p, n->ds_ac.p, n->ds_anb.p, n->ds_vol.p, n->ds_x.p, n->ds_xp.p);
  const int nb = std::min(kStatBlocks, cdiv(N, kBlock));
  hipLaunchKernelGGL(k_loss, dim3(nb, B), dim3(kBlock), 0, s, N, n->ymean.p, n->scal.p, n->Y.p, n->Tg.p, n->DY.p,
                     1.0 / Bn, n->part.p, (double *)nullptr);
  if (!want_grad) return;
  const int L = n->L, nbc = grad_blocks(Bn);
  if ((size_t)nbc * kGradW > n->gpart.n) throw std::runtime_error("gradient workspace too small for the batch");
  float *g = n->grad.p;
  auto reduce = [&](int K, float *dst) {
    hipLaunchKernelGGL(k_reduce, dim3(cdiv(K, 32)), dim3(kBlock), 0, s, nbc, K, n->gpart.p, dst);
  };
  // decoder (wd and bd are the last parameters)
  hipLaunchKernelGGL(k_dec_grad, dim3(nbc), dim3(256), 0, s, Bn, n->DY.p, n->Hs[L].p, n->gpart.p);
  reduce(kH + 1, g + mpnn_offset_W(L));
  const unsigned quads = cdiv((long long)Bn * (kH / 4), kBlock);
  hipLaunchKernelGGL(k_dec_bwd, dim3(quads), dim3(kBlock), 0, s, Bn, n->DY.p, n->wdq.p, n->dH.p, n->masks[L - 1].p,
                     n->DZ.p);
  float *dH = n->dH.p, *dH2 = n->dH2.p;
  for (int l = L - 1; l >= 0; --l) {
    hipLaunchKernelGGL(k_dense_bwd_w, dim3(nbc), dim3(256), 0, s, Bn, n->Hs[l].p, n->Ms[l].p, n->DZ.p,
                       n->gpart.p);
    reduce(kGradW, g + mpnn_offset_W(l));
    hipLaunchKernelGGL(k_dense_bwd_x, dim3(cdiv(Bn, kRowsFwd)), dim3(256), 0, s, Bn, n->DZ.p,
                       n->wb.p + (size_t)l * kIn * kH, n->D.p);
    hipLaunchKernelGGL(k_agg_t, dim3(quads), dim3(kBlock), 0, s, N, n->W, Bn, n->nbr0.p, n->mir.p, n->E.p, dH, n->D.p,
                       dH2, l > 0 ? n->masks[l - 1].p : nullptr, n->DZ.p);
    std::swap(dH, dH2);
  }
  hipLaunchKernelGGL(k_enc_bwd, dim3(nbc), dim3(256), 0, s, Bn, n->X0.p, n->Hs[0].p, dH, n->gpart.p);
  reduce((kF + 1) * kH, g);
}

// The loss of the batch just evaluated; waits for the stream.
static double mpnn_loss(fs_mpnn *n, int B) {
  const int nb = std::min(kStatBlocks, cdiv(n->N, kBlock));
  n->h_part.resize((size_t)B * nb);
  FS_HIP_THROW(hipMemcpyAsync(n->h_part.data(), n->part.p, sizeof(double) * B * nb, hipMemcpyDeviceToHost, n->s));
  FS_HIP_THROW(hipStreamSynchronize(n->s));
  double loss = 0.0;
  for (double v : n->h_part) loss += v;
  return loss / ((double)B * n->N);
}

} // namespace fs

using fs::set_error;

#define MPNN_GUARD_BEGIN try {
#define MPNN_GUARD_END                                                        \
  }                                                                           \
  catch (const std::exception &e) {                                           \
    set_error(e.what());                                                      \
    return -2;                                                                \
  }

extern "C" {

int fs_mpnn_create(int n_cells, int width, const int *elem_nbr, int layers, int use_prev, unsigned long long seed,
                   int capacity, fs_mpnn **out) {
  MPNN_GUARD_BEGIN
  if (!out || !elem_nbr || n_cells <= 0 || width <= 0 || layers < 1 || layers > fs::kMaxLayers || capacity < 0 ||
      (use_prev != 0 && use_prev != 1)) {
    set_error("fs_mpnn_create: invalid arguments");
    return -1;
  }
  *out = nullptr;
  for (long long t = 0; t < (long long)n_cells * width; ++t)
    if (elem_nbr[t] < 0 || elem_nbr[t] > n_cells) {
      set_error("fs_mpnn_create: ElementNeighbor entry out of range at linear index " + std::to_string(t));
      return -1;
    }
  auto n = std::make_unique<fs_mpnn>();
  n->N = n_cells;
  n->W = width;
  n->L = layers;
  n->use_prev = use_prev != 0;
  n->P = fs::mpnn_offset_W(layers) + fs::kH + 1;
  FS_HIP(hipStreamCreate(&n->s));
  // 0-based neighbours and the mirror slots (slot of i in the list of nbr_j(i))
  n->h_nbr0.resize((size_t)n_cells * width);
  for (size_t t = 0; t < n->h_nbr0.size(); ++t) n->h_nbr0[t] = elem_nbr[t] - 1;
  std::vector<int> mir(n->h_nbr0.size(), -1);
  for (int i = 0; i < n_cells; ++i)
    for (int j = 0; j < width; ++j) {
      const int k = n->h_nbr0[(size_t)j * n_cells + i];
      if (k < 0) continue;
      for (int q = 0; q < width; ++q)
        if (n->h_nbr0[(size_t)q * n_cells + k] == i) {
          mir[(size_t)j * n_cells + i] = q;
          break;
        }
      if (mir[(size_t)j * n_cells + i] < 0) {
        set_error("fs_mpnn_create: neighbour lists are not symmetric (cell " + std::to_string(i + 1) + ")");
        (void)hipStreamDestroy(n->s);
        return -1;
      }
    }
  n->nbr0.upload(n->h_nbr0, n->s);
  n->mir.upload(mir, n->s);
  // He initialisation
  std::vector<float> th(n->P, 0.f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> nd(0.0, 1.0);
  for (int i = 0; i < fs::kF * fs::kH; ++i) th[i] = (float)(nd(rng) * std::sqrt(2.0 / fs::kF));
  for (int l = 0; l < layers; ++l)
    for (int i = 0; i < fs::kIn * fs::kH; ++i) th[fs::mpnn_offset_W(l) + i] = (float)(nd(rng) * std::sqrt(2.0 / fs::kIn));
  for (int i = 0; i < fs::kH; ++i) th[fs::mpnn_offset_W(layers) + i] = (float)(nd(rng) * std::sqrt(1.0 / fs::kH));
  n->theta.upload(th, n->s);
  n->grad.alloc(n->P);
  n->am.alloc(n->P);
  n->av.alloc(n->P);
  FS_HIP(hipMemsetAsync(n->grad.p, 0, sizeof(float) * n->P, n->s));
  FS_HIP(hipMemsetAsync(n->am.p, 0, sizeof(float) * n->P, n->s));
  FS_HIP(hipMemsetAsync(n->av.p, 0, sizeof(float) * n->P, n->s));
  n->weq.alloc(fs::kF * fs::kH);
  n->wdq.alloc(fs::kH);
  n->wt.alloc((size_t)layers * fs::kIn * fs::kH);
  n->wb.alloc((size_t)layers * fs::kIn * fs::kH);
  fs::quantize(n.get());
  n->cap = capacity;
  const size_t cn = (size_t)std::max(capacity, 1) * n_cells;
  n->ds_b.alloc(cn);
  n->ds_x.alloc(cn);
  n->ds_ac.alloc(cn);
  n->ds_vol.alloc(cn);
  n->ds_xp.alloc(cn);
  n->ds_anb.alloc(cn * width);
  FS_HIP(hipStreamSynchronize(n->s));
  *out = n.release();
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_destroy(fs_mpnn *n) {
  if (!n) return 0;
  (void)hipStreamSynchronize(n->s);
  hipStream_t s = n->s;
  delete n;
  if (s) (void)hipStreamDestroy(s);
  return 0;
}

int fs_mpnn_param_count(fs_mpnn *n) { return n ? n->P : -1; }

int fs_mpnn_get_params(fs_mpnn *n, double *theta, int count) {
  MPNN_GUARD_BEGIN
  if (!n || !theta || count != n->P) {
    set_error("fs_mpnn_get_params: NULL argument or count != fs_mpnn_param_count");
    return -1;
  }
  std::vector<float> h(n->P);
  FS_HIP(hipMemcpyAsync(h.data(), n->theta.p, sizeof(float) * n->P, hipMemcpyDeviceToHost, n->s));
  FS_HIP(hipStreamSynchronize(n->s));
  for (int i = 0; i < n->P; ++i) theta[i] = h[i];
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_set_params(fs_mpnn *n, const double *theta, int count) {
  MPNN_GUARD_BEGIN
  if (!n || !theta || count != n->P) {
    set_error("fs_mpnn_set_params: NULL argument or count != fs_mpnn_param_count");
    return -1;
  }
  std::vector<float> h(n->P);
  for (int i = 0; i < n->P; ++i) h[i] = (float)theta[i];
  FS_HIP(hipMemcpyAsync(n->theta.p, h.data(), sizeof(float) * n->P, hipMemcpyHostToDevice, n->s));
  FS_HIP(hipMemsetAsync(n->am.p, 0, sizeof(float) * n->P, n->s));
  FS_HIP(hipMemsetAsync(n->av.p, 0, sizeof(float) * n->P, n->s));
  n->steps = 0;
  fs::quantize(n);
  FS_HIP(hipStreamSynchronize(n->s));
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_add_samples(fs_mpnn *n, int ns, const double *b, const double *x, const double *ac, const double *anb,
                        const double *vol, const double *x_prev) {
  MPNN_GUARD_BEGIN
  if (!n || ns < 0 || !b || !x || !ac || !anb || !vol) {
    set_error("fs_mpnn_add_samples: invalid arguments");
    return -1;
  }
  if (n->count + ns > n->cap) {
    set_error("fs_mpnn_add_samples: dataset capacity exceeded");
    return -1;
  }
  const size_t N = n->N, off = (size_t)n->count * N, cnt = (size_t)ns * N;
  fs::DevBuf<double> tmp;
  tmp.alloc(cnt * n->W);
  auto put = [&](const double *src, float *dst, size_t m) {
    FS_HIP_THROW(hipMemcpyAsync(tmp.p, src, sizeof(double) * m, hipMemcpyHostToDevice, n->s));
    hipLaunchKernelGGL(fs::k_to_f32, dim3(fs::cdiv((long long)m, fs::kBlock)), dim3(fs::kBlock), 0, n->s, (long long)m,
                       tmp.p, dst);
    FS_HIP_THROW(hipStreamSynchronize(n->s));
  };
  put(b, n->ds_b.p + off, cnt);
  put(x, n->ds_x.p + off, cnt);
  put(ac, n->ds_ac.p + off, cnt);
  put(vol, n->ds_vol.p + off, cnt);
  put(anb, n->ds_anb.p + off * n->W, cnt * n->W);
  if (x_prev) put(x_prev, n->ds_xp.p + off, cnt);
  else FS_HIP(hipMemsetAsync(n->ds_xp.p + off, 0, sizeof(float) * cnt, n->s));
  FS_HIP(hipStreamSynchronize(n->s));
  n->count += ns;
  return n->count;
  MPNN_GUARD_END
}

int fs_mpnn_sample_count(fs_mpnn *n) { return n ? n->count : -1; }

int fs_mpnn_get_sample(fs_mpnn *n, int k, double *b, double *x, double *ac, double *anb, double *vol,
                       double *x_prev) {
  MPNN_GUARD_BEGIN
  if (!n || k < 0 || k >= n->count) {
    set_error("fs_mpnn_get_sample: sample out of range");
    return -1;
  }
  const size_t N = n->N;
  std::vector<float> h(N * n->W);
  auto get = [&](const float *src, double *dst, size_t m) {
    if (!dst) return;
    FS_HIP_THROW(hipMemcpyAsync(h.data(), src, sizeof(float) * m, hipMemcpyDeviceToHost, n->s));
    FS_HIP_THROW(hipStreamSynchronize(n->s));
    for (size_t i = 0; i < m; ++i) dst[i] = h[i];
  };
  get(n->ds_b.p + k * N, b, N);
  get(n->ds_x.p + k * N, x, N);
  get(n->ds_ac.p + k * N, ac, N);
  get(n->ds_vol.p + k * N, vol, N);
  get(n->ds_anb.p + k * N * n->W, anb, N * n->W);
  get(n->ds_xp.p + k * N, x_prev, N);
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_loss_grad(fs_mpnn *n, const int *ids, int batch, double *loss, double *grad) {
  MPNN_GUARD_BEGIN
  if (!n || !ids || batch < 1 || !loss) {
    set_error("fs_mpnn_loss_grad: invalid arguments");
    return -1;
  }
  fs::mpnn_loss_grad(n, ids, batch, grad != nullptr);
  *loss = fs::mpnn_loss(n, batch);
  if (grad) {
    std::vector<float> h(n->P);
    FS_HIP(hipMemcpyAsync(h.data(), n->grad.p, sizeof(float) * n->P, hipMemcpyDeviceToHost, n->s));
    FS_HIP(hipStreamSynchronize(n->s));
    for (int i = 0; i < n->P; ++i) grad[i] = h[i];
  }
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_train_step(fs_mpnn *n, const int *ids, int batch, double lr, double *loss) {
  MPNN_GUARD_BEGIN
  if (!n || !ids || batch < 1 || !(lr > 0.0)) {
    set_error("fs_mpnn_train_step: invalid arguments");
    return -1;
  }
  fs::mpnn_loss_grad(n, ids, batch, true);
  n->steps++;
  const float c1 = 1.f - std::pow(0.9f, (float)n->steps), c2 = 1.f - std::pow(0.999f, (float)n->steps);
  hipLaunchKernelGGL(fs::k_adam, dim3(fs::cdiv(n->P, fs::kBlock)), dim3(fs::kBlock), 0, n->s, n->P, n->theta.p,
                     n->grad.p, n->am.p, n->av.p, (float)lr, c1, c2);
  fs::quantize(n);
  const double l = fs::mpnn_loss(n, batch); // the step's only wait
  if (loss) *loss = l;
  return 0;
  MPNN_GUARD_END
}

int fs_mpnn_predict(fs_mpnn *n, const double *b, const double *ac, const double *anb, const double *vol,
                    const double *x_prev, double *x) {
  MPNN_GUARD_BEGIN
  if (!n || !b || !ac || !anb || !vol || !x) {
    set_error("fs_mpnn_predict: NULL argument");
    return -1;
  }
  const size_t N = n->N;
  fs::DevBuf<double> db, dac, danb, dvol, dx, dxp;
  db.upload(b, N, n->s);
  dac.upload(ac, N, n->s);
  danb.upload(anb, N * n->W, n->s);
  dvol.upload(vol, N, n->s);
  if (x_prev) dxp.upload(x_prev, N, n->s);
  dx.alloc(N);
  const int rc = fs::mpnn_predict_device(n, n->s, db.p, dac.p, danb.p, dvol.p, x_prev ? dxp.p : nullptr, dx.p);
  if (rc < 0) return rc;
  FS_HIP(hipMemcpyAsync(x, dx.p, sizeof(double) * N, hipMemcpyDeviceToHost, n->s));
  FS_HIP(hipStreamSynchronize(n->s));
  return 0;
  MPNN_GUARD_END
}

} // extern "C"

namespace fs {

int mpnn_predict_device(fs_mpnn *n, hipStream_t stream, const double *b, const double *ac, const double *anb,
                        const double *vol, const double *xp, double *x) {
  // run on the caller's stream
  hipStream_t own = n->s;
  n->s = stream;
  try {
    mpnn_grow(n, 1);
    const int zero = 0;
    FS_HIP_THROW(hipMemcpyAsync(n->ids.p, &zero, sizeof(int), hipMemcpyHostToDevice, stream));
    mpnn_forward<double>(n, 1, b, ac, anb, vol, (const double *)nullptr, xp);
    const int nb = std::min(kStatBlocks, cdiv(n->N, kBlock));
    hipLaunchKernelGGL(k_loss, dim3(nb, 1), dim3(kBlock), 0, stream, n->N, n->ymean.p, n->scal.p, n->Y.p,
                       (const float *)nullptr, (float *)nullptr, 0.0, n->part.p, x);
  } catch (...) {
    n->s = own;
    throw;
  }
  n->s = own;
  return 0;
}

bool mpnn_matches(fs_mpnn *n, int n_cells, int width, const std::vector<int> &nbr0) {
  return n && n->N == n_cells && n->W == width && n->h_nbr0 == nbr0;
}

// append one device system (FP64) to the dataset; false when full
bool mpnn_capture(fs_mpnn *n, hipStream_t stream, const double *b, const double *x, const double *ac,
                  const double *anb, const double *vol, const double *xp) {
  if (!n || n->count >= n->cap) return false;
  const size_t N = n->N, off = (size_t)n->count * N;
  auto put = [&](const double *src, float *dst, size_t m) {
    hipLaunchKernelGGL(k_to_f32, dim3(cdiv((long long)m, kBlock)), dim3(kBlock), 0, stream, (long long)m, src, dst);
  };
  put(b, n->ds_b.p + off, N);
  put(x, n->ds_x.p + off, N);
  put(ac, n->ds_ac.p + off, N);
  put(vol, n->ds_vol.p + off, N);
  put(xp, n->ds_xp.p + off, N);
  put(anb, n->ds_anb.p + off * n->W, N * n->W);
  n->count++;
  return true;
}

} // namespace fs
