// Learned eddy-viscosity closure: packing, training and data kernels.
//
// Training is deterministic: tlbm_mlp_grad writes one partial gradient vector
// per 64-sample workgroup, tlbm_mlp_adam sums the partials in a fixed order
// and applies Adam (torch.optim.Adam update rule, as in the reference's
// train_eddy_viscosity_model, src/tensorlbm/ai/train.py:382-435).
//
// Data: the DNS populations are block-averaged by an integer factor
// (the 3-D form of ai/pipeline.py:93-107 _coarsen_mean) into rho, u_i and
// <u_i u_j>; the samples are the resolved strain (periodic central
// differences, ai/dataset.py:41-72 in 3-D) and the sub-grid eddy viscosity
// nu = max(0, -tau_ij S_ij / (2 S_kl S_kl)), tau_ij = <u_i u_j> - <u_i><u_j>.
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <mutex>

#include "../../include/tlbm_hip.h"
#include "collide.hpp"
#include "mlp.hpp"
#include "store.hpp"

namespace tlbm {

using namespace mlp;

constexpr int GRAD_BS = 64;  // samples per workgroup in the gradient kernel

// ---------------------------------------------------------------------------
// packing: fp32 parameters -> matrix-core operand blob
// ---------------------------------------------------------------------------

// fp16 bits of v, round to nearest even
__device__ __forceinline__ uint16_t f16_bits(float v) { return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v)); }

// bf16 bits of v, round to nearest even
__device__ __forceinline__ uint16_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }

// operand bits of v in the blob's type, and v rounded to that type
template <bool BF16>
__device__ __forceinline__ uint16_t op_bits(float v) {
  return BF16 ? bf16_bits(v) : f16_bits(v);
}
template <bool BF16>
__device__ __forceinline__ float op_round(float v) {
  return BF16 ? static_cast<float>(static_cast<__bf16>(v)) : static_cast<float>(static_cast<_Float16>(v));
}

template <bool BF16>
__global__ __launch_bounds__(64) void k_mlp_pack(const float* __restrict__ p, Packed* __restrict__ out) {
  const int l = threadIdx.x;
  const int h = l >> 5, i = l & 31;
  for (int e = 0; e < 8; ++e) {
    if (e < NIN) {
      out->a1[l][e] = op_bits<BF16>(p[OW1 + i * NIN + e]);
    } else {  // bias at K 7 (hi, lanes < 32) and K 15 (lo, lanes >= 32)
      const float b = p[OB1 + i];
      out->a1[l][e] = op_bits<BF16>(h == 0 ? b : b - op_round<BF16>(b));
    }
    for (int s = 0; s < 2; ++s) out->a2[s][l][e] = op_bits<BF16>(p[OW2 + i * NH + w2_col(s, h, e)]);
  }
  if (l < 32) {
    const int hh = l >> 4, r = l & 15;
    out->b1c[hh][r] = p[OB1 + c_row(hh, r)];
    out->b2c[hh][r] = p[OB2 + c_row(hh, r)];
    out->w3c[hh][r] = p[OW3 + c_row(hh, r)];
  }
  if (l == 0) {
    out->b3 = p[OB3];
    for (int e = 0; e < NIN; ++e) {
      out->mean[e] = p[OMEAN + e];
      out->istd[e] = p[OISTD + e];
    }
    out->pad = 0.0f;
  }
}

// ---------------------------------------------------------------------------
// fp32 forward (prediction) and gradient
// ---------------------------------------------------------------------------

// One lane per sample, the whole network unrolled: activations in registers, weights
// by scalar loads (their index is uniform).  With rolled loops over a per-lane
// activation array the array lived in scratch memory (13,107 samples: 17.4 us).
__global__ __launch_bounds__(256) void k_mlp_predict(const float* __restrict__ p, const float* __restrict__ x,
                                                     uint64_t n, float* __restrict__ y) {
  const uint64_t s = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  float xh[NIN], h1[NH];
#pragma unroll
  for (int e = 0; e < NIN; ++e) xh[e] = (x[s * NIN + e] - p[OMEAN + e]) * p[OISTD + e];
#pragma unroll
  for (int i = 0; i < NH; ++i) {
    float a = p[OB1 + i];
#pragma unroll
    for (int e = 0; e < NIN; ++e) a += p[OW1 + i * NIN + e] * xh[e];
    h1[i] = fmaxf(a, 0.0f);
  }
  float z3 = p[OB3];
#pragma unroll 4
  for (int i = 0; i < NH; ++i) {
    float a = p[OB2 + i];
#pragma unroll
    for (int j = 0; j < NH; ++j) a += p[OW2 + i * NH + j] * h1[j];
    z3 += p[OW3 + i] * fmaxf(a, 0.0f);
  }
  y[s] = softplus(z3);
}

// Gradient of 64 samples per workgroup into partials[block].  Lane = sample, and each
// of the four waves carries a quarter of the hidden units through the forward and the
// backward pass, so that all four SIMDs of a CU work (with one wave running all units
// and its activation arrays in scratch memory, 4096 samples took 25 us).  The parameters are
// staged into LDS in one round of loads beside the sample's own (read where they are
// used, by scalar loads, each layer waited for several round trips: 10 us); every lane
// of a wave reads the same weight, an LDS broadcast.  Activations and deltas go
// through LDS as [unit][sample].  The weight gradients are products
// delta^T activation over the 64 samples: fp32 matrix-core tiles (16 x 16, exact fp32
// products and accumulation), whose operands the LDS pitch of 68 floats serves without
// bank conflicts (bank 4 unit + sample).
//   A: lane -> row lane % 16, k = lane / 16;  B: column lane % 16, k = lane / 16;
//   D: rows 4 (lane / 16) + r, column lane % 16.
// idx (optional) names the rows of x and t to take, so a minibatch needs no copy.
constexpr int GP = 68;  // LDS pitch of a unit's 64 samples
static_assert(OW2 % 4 == 0 && NH % 4 == 0, "four weights of a row of W2 are 16-byte aligned in LDS");
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <class FA, class FB>
__device__ __forceinline__ f32x4 grad_tile(int lane, const FA& a, const FB& b) {
  f32x4 d = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int k = 0; k < GRAD_BS; k += 4) {
    const int sm = k + (lane >> 4);
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(a(lane & 15, sm), b(lane & 15, sm), d, 0, 0, 0);
  }
  return d;
}

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__global__ __launch_bounds__(256) void k_mlp_grad(const float* __restrict__ p, const float* __restrict__ x,
                                                  const float* __restrict__ t, const int64_t* __restrict__ idx,
                                                  uint64_t n, float inv_n, float* __restrict__ partials) {
  constexpr int U = NH / 4;  // hidden units per wave
  __shared__ float s_xb[8][GP];  // normalised inputs, then a row of ones (the bias column)
  __shared__ float s_h1[NH][GP], s_d1[NH][GP], s_h2[NH][GP], s_d2[NH][GP];
  __shared__ float s_z3[4][GRAD_BS], s_d3[GRAD_BS];
  __shared__ __align__(16) float s_p[(NTOTAL + 3) / 4 * 4];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int u0 = w * U;
  const uint64_t s = uint64_t(blockIdx.x) * GRAD_BS + lane;
  const bool ok = s < n;
  const uint64_t row = ok ? (idx != nullptr ? uint64_t(idx[s]) : s) : 0;
  float pv[(NTOTAL + 255) / 256];
#pragma unroll
  for (int k = 0; k < (NTOTAL + 255) / 256; ++k) {
    const int i = int(threadIdx.x) + 256 * k;
    pv[k] = i < NTOTAL ? p[i] : 0.0f;
  }
  const float target = ok ? t[row] : 0.0f;
  float xh[NIN];
#pragma unroll
  for (int e = 0; e < NIN; ++e) xh[e] = ok ? x[row * NIN + e] : 0.0f;
#pragma unroll
  for (int k = 0; k < (NTOTAL + 255) / 256; ++k) {
    const int i = int(threadIdx.x) + 256 * k;
    if (i < NTOTAL) s_p[i] = pv[k];
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < NIN; ++e) xh[e] = (xh[e] - s_p[OMEAN + e]) * s_p[OISTD + e];
  if (w == 0) {
#pragma unroll
    for (int e = 0; e < NIN; ++e) s_xb[e][lane] = xh[e];
    s_xb[NIN][lane] = 1.0f;
  }
  float z1[U], z2[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int i = u0 + u;
    float a = s_p[OB1 + i];
#pragma unroll
    for (int e = 0; e < NIN; ++e) a += s_p[OW1 + i * NIN + e] * xh[e];
    z1[u] = a;
    s_h1[i][lane] = fmaxf(a, 0.0f);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) z2[u] = s_p[OB2 + u0 + u];
#pragma unroll
  for (int j = 0; j < NH; j += 4) {
    const float h0 = s_h1[j][lane], h1 = s_h1[j + 1][lane], h2 = s_h1[j + 2][lane], h3 = s_h1[j + 3][lane];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const f32x4 wt = *reinterpret_cast<const f32x4*>(&s_p[OW2 + (u0 + u) * NH + j]);
      z2[u] = fmaf(wt[3], h3, fmaf(wt[2], h2, fmaf(wt[1], h1, fmaf(wt[0], h0, z2[u]))));
    }
  }
  float part = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float h = fmaxf(z2[u], 0.0f);
    s_h2[u0 + u][lane] = h;
    part += s_p[OW3 + u0 + u] * h;
  }
  s_z3[w][lane] = part;
  __syncthreads();
  const float z3 = s_p[OB3] + ((s_z3[0][lane] + s_z3[1][lane]) + (s_z3[2][lane] + s_z3[3][lane]));
  const float res = ok ? softplus(z3) - target : 0.0f;
  // dL/dz3 = 2 (y - t)/N * softplus'(z3): sigmoid(beta z3), 1 where softplus returns z3 (beta z3 > 20)
  const float bz = fmaxf(BETA * z3, -60.0f);
  const float d3 = 2.0f * res * inv_n * (bz > 20.0f ? 1.0f : 1.0f / (1.0f + __expf(-bz)));
  if (w == 0) s_d3[lane] = d3;
#pragma unroll
  for (int u = 0; u < U; ++u) s_d2[u0 + u][lane] = z2[u] > 0.0f ? d3 * s_p[OW3 + u0 + u] : 0.0f;
  __syncthreads();
  float d1[U];
#pragma unroll
  for (int u = 0; u < U; ++u) d1[u] = 0.0f;
#pragma unroll 8
  for (int i = 0; i < NH; ++i) {
    const float d = s_d2[i][lane];
#pragma unroll
    for (int u = 0; u < U; u += 4) {
      const f32x4 wt = *reinterpret_cast<const f32x4*>(&s_p[OW2 + i * NH + u0 + u]);
#pragma unroll
      for (int e = 0; e < 4; ++e) d1[u + e] = fmaf(d, wt[e], d1[u + e]);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) s_d1[u0 + u][lane] = z1[u] > 0.0f ? d1[u] : 0.0f;
  __syncthreads();

  float* out = partials + uint64_t(blockIdx.x) * (NPARAM + 1);
  const int c = lane & 15, r0 = 4 * (lane >> 4);
  {  // W2: one quadrant per wave
    const int i0 = 16 * (w >> 1), j0 = 16 * (w & 1);
    const f32x4 d = grad_tile(lane, [&](int i, int sm) { return s_d2[i0 + i][sm]; },
                              [&](int j, int sm) { return s_h1[j0 + j][sm]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) out[OW2 + (i0 + r0 + r) * NH + j0 + c] = d[r];
  }
  const int i0 = 16 * (w & 1);
  if (w < 2) {  // W1 and b1 (column 7: the ones); then the output weights
    f32x4 d = grad_tile(lane, [&](int i, int sm) { return s_d1[i0 + i][sm]; },
                        [&](int j, int sm) { return j < 8 ? s_xb[j][sm] : 0.0f; });
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = i0 + r0 + r;
      if (c < NIN) out[OW1 + i * NIN + c] = d[r];
      if (c == NIN) out[OB1 + i] = d[r];
    }
    d = grad_tile(lane, [&](int i, int sm) { return s_h2[i0 + i][sm]; },
                  [&](int j, int sm) { return j == 0 ? s_d3[sm] : 0.0f; });
    if (c == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) out[OW3 + i0 + r0 + r] = d[r];
    }
  } else {  // b2, b3 and the loss
    const f32x4 d = grad_tile(lane, [&](int i, int sm) { return s_d2[i0 + i][sm]; },
                              [&](int j, int) { return j == 0 ? 1.0f : 0.0f; });
    if (c == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) out[OB2 + i0 + r0 + r] = d[r];
    }
    const float sum = wave_sum64(w == 2 ? d3 : res * res * inv_n);
    if (lane == 0) out[w == 2 ? OB3 : NPARAM] = sum;
  }
}

// One workgroup: sum the per-workgroup partials in a fixed order, clip the global
// gradient norm (torch.nn.utils.clip_grad_norm_ rule: scale by min(1, clip / (|g| +
// 1e-6)), ai/train.py:401-405), then one Adam step.  The partials are read four
// columns to a thread and three interleaved sets of rows at a time, so that a CU has
// 1011 sixteen-byte loads in flight per row triple (one four-byte column per thread
// and all rows in turn took 32 us for 64 partials).  loss_sum, when given, receives
// += loss * weight in double (an epoch's running loss).
constexpr int ADAM_THREADS = 1024;
constexpr int COLS4 = (NPARAM + 1 + 3) / 4;           // 337
constexpr int ROW_SETS = ADAM_THREADS / COLS4;        // 3
static_assert(2 * ADAM_THREADS > NPARAM, "two entries per thread cover the gradient and the loss");
static_assert(ROW_SETS == 3, "sums of three row sets");
// rows are 4-byte aligned (an odd number of float pairs apart)
struct __attribute__((packed, aligned(4))) Row4 {
  float v[4];
};

__global__ __launch_bounds__(ADAM_THREADS) void k_mlp_adam(float* __restrict__ p, const float* __restrict__ partials,
                                                           int nblk, float* __restrict__ m, float* __restrict__ v,
                                                           float lr, float b1, float b2, float eps, float bc1,
                                                           float bc2, float clip, float* __restrict__ loss_out,
                                                           float* __restrict__ grad_out,
                                                           double* __restrict__ loss_sum, double weight) {
  __shared__ float s_g[ROW_SETS][4 * COLS4];
  __shared__ float s_red[ADAM_THREADS / 64];
  const int tid = threadIdx.x;
  const bool update = lr != 0.0f;
  float pk[2] = {}, mk[2] = {}, vk[2] = {};
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int k = tid + r * ADAM_THREADS;
    if (update && k < NPARAM) {
      pk[r] = p[k];
      mk[r] = m[k];
      vk[r] = v[k];
    }
  }
  const int set = tid / COLS4, col = 4 * (tid % COLS4);
  if (set < ROW_SETS) {
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const float* src = partials + col;
    if (col + 4 <= NPARAM + 1) {
#pragma unroll 8
      for (int b = set; b < nblk; b += ROW_SETS) {
        const Row4 q = *reinterpret_cast<const Row4*>(src + uint64_t(b) * (NPARAM + 1));
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] += q.v[e];
      }
    } else {  // the last columns of a row
      for (int b = set; b < nblk; b += ROW_SETS)
        for (int e = 0; col + e <= NPARAM; ++e) a[e] += src[uint64_t(b) * (NPARAM + 1) + e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) s_g[set][col + e] = a[e];
  }
  __syncthreads();
  float g[2];
  float sq = 0.0f;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int k = tid + r * ADAM_THREADS;
    g[r] = k <= NPARAM ? (s_g[0][k] + s_g[1][k]) + s_g[2][k] : 0.0f;
    if (k < NPARAM) sq += g[r] * g[r];
  }
  sq = wave_sum64(sq);
  if ((tid & 63) == 0) s_red[tid >> 6] = sq;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < ADAM_THREADS / 64; ++i) total += s_red[i];
  const float norm = sqrtf(total);
  const float scale = clip > 0.0f ? fminf(1.0f, clip / (norm + 1e-6f)) : 1.0f;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int k = tid + r * ADAM_THREADS;
    if (k == NPARAM) {
      if (loss_out) *loss_out = g[r];
      if (loss_sum) *loss_sum += double(g[r]) * weight;
    }
    if (k >= NPARAM) continue;
    if (grad_out) grad_out[k] = g[r];
    if (!update) continue;
    const float gk = g[r] * scale;
    mk[r] = b1 * mk[r] + (1.0f - b1) * gk;
    vk[r] = b2 * vk[r] + (1.0f - b2) * gk * gk;
    m[k] = mk[r];
    v[k] = vk[r];
    p[k] = pk[r] - lr * (mk[r] / bc1) / (sqrtf(vk[r] / bc2) + eps);
  }
}

// The partials' column sums by as many CUs as there are 64-column strips, into row 0
// of `sum`: one CU reads memory written by the others at some 25 GB/s (16.6 us for 64
// partials in k_mlp_adam), 22 of them in one round trip.  Four row sets per column,
// each in row order, added in a fixed order.
__global__ __launch_bounds__(256) void k_mlp_reduce(const float* __restrict__ partials, int nblk,
                                                    float* __restrict__ sum) {
  __shared__ float s_part[4][64];
  const int c = threadIdx.x & 63, set = threadIdx.x >> 6;
  const int k = int(blockIdx.x) * 64 + c;
  float a = 0.0f;
  if (k <= NPARAM) {
#pragma unroll 16
    for (int b = set; b < nblk; b += 4) a += partials[uint64_t(b) * (NPARAM + 1) + k];
  }
  s_part[set][c] = a;
  __syncthreads();
  if (set == 0 && k <= NPARAM) sum[k] = (s_part[0][c] + s_part[1][c]) + (s_part[2][c] + s_part[3][c]);
}

// Gradient partials of tlbm_mlp_train_step_noalloc: up to NOALLOC_MAX_BLOCKS workgroups of
// GRAD_BS samples, (NPARAM + 1) floats each (2.76 MB), one copy per GPU for the life of the
// process.  k_mlp_grad writes every entry of the blocks a call launches before k_mlp_adam
// reads them, so nothing is cleared between calls.
constexpr int NOALLOC_MAX_BLOCKS = TLBM_MLP_NOALLOC_MAX_SAMPLES / GRAD_BS;
static_assert(NOALLOC_MAX_BLOCKS * GRAD_BS == TLBM_MLP_NOALLOC_MAX_SAMPLES, "whole blocks");
static __device__ __align__(256) float scratch[NOALLOC_MAX_BLOCKS * (NPARAM + 1)];

// ---------------------------------------------------------------------------
// DNS -> LES data
// ---------------------------------------------------------------------------

struct Lay {
  int64_t sq, sz, sy;
  int nx, ny, nz;
};

// out: 10 fields of the coarse grid: rho, u_x, u_y, u_z, <uxux> <uyuy> <uzuz> <uxuy> <uxuz> <uyuz>
//
// A workgroup owns `cells` coarse cells of one coarse row, one lane per fine column
// (lanes a multiple of r; lanes beyond 512 columns loop), so every load of a wave is
// contiguous.  A lane adds its column's r x r fine cells in FP64, then the r columns
// of a coarse cell meet in LDS.  With one lane per coarse cell each load instruction
// touched r times the cache lines: 288^3 fp32, r = 3: 503 us, now 315 us (5.85 TB/s;
// 351 us with plain loads).
constexpr int COARSEN_LANES = 512;

// element x of a row that is uniform over the wave: scalar base, 32-bit lane offset;
// the populations are read once, so past the caches
template <typename T>
__device__ __forceinline__ T ld_row(const T* row, uint32_t x) {
  using G = __attribute__((address_space(1))) const T;
  return __builtin_nontemporal_load((G*)(reinterpret_cast<const char*>(row) + x * uint32_t(sizeof(T))));
}

template <class L, int S>
__global__ __launch_bounds__(COARSEN_LANES) void k_coarsen(const void* __restrict__ fv, Lay lay, int r, int cells,
                                                           float* __restrict__ out) {
  using ST = Store<S>;
  extern __shared__ double s_acc[];  // [10][blockDim.x]
  const typename ST::T* f = static_cast<const typename ST::T*>(fv);
  const int cx = lay.nx / r, cy = lay.ny / r, cz = lay.nz / r;
  const int nbx = (cx + cells - 1) / cells;
  const int X0 = int(blockIdx.x % uint32_t(nbx)) * cells;
  const uint32_t row = blockIdx.x / uint32_t(nbx);
  const int Y = int(row % uint32_t(cy)), Z = int(row / uint32_t(cy));
  const int here = min(cells, cx - X0);        // coarse cells of this workgroup
  const int lanes = min(r, COARSEN_LANES);     // lanes of one coarse cell
  const int t = threadIdx.x;
  double acc[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (t < here * lanes) {
    for (int dx = t % lanes; dx < r; dx += lanes) {
      const uint32_t x = uint32_t(X0 + t / lanes) * uint32_t(r) + uint32_t(dx);
      for (int dz = 0; dz < r; ++dz)
        for (int dy = 0; dy < r; ++dy) {
          const typename ST::T* base = f + int64_t(Z * r + dz) * lay.sz + int64_t(Y * r + dy) * lay.sy;
          typename ST::C v[L::Q];
#pragma unroll
          for (int q = 0; q < L::Q; ++q) v[q] = ST::template get<L>(ld_row(base + int64_t(q) * lay.sq, x), q);
          const Macro<typename ST::C> mc = macro<L>(v);
          const double ux = mc.ux, uy = mc.uy, uz = mc.uz;
          acc[0] += mc.rho;
          acc[1] += ux;
          acc[2] += uy;
          acc[3] += uz;
          acc[4] += ux * ux;
          acc[5] += uy * uy;
          acc[6] += uz * uz;
          acc[7] += ux * uy;
          acc[8] += ux * uz;
          acc[9] += uy * uz;
        }
    }
  }
#pragma unroll
  for (int k = 0; k < 10; ++k) s_acc[k * int(blockDim.x) + t] = acc[k];
  __syncthreads();
  const uint64_t nc = uint64_t(cx) * cy * cz;
  const double inv = 1.0 / (double(r) * r * r);
  for (int i = t; i < 10 * here; i += int(blockDim.x)) {
    const int k = i / here, c = i - k * here;
    double a = 0.0;
    for (int l = 0; l < lanes; ++l) a += s_acc[k * int(blockDim.x) + c * lanes + l];
    out[uint64_t(k) * nc + uint64_t(row) * cx + uint64_t(X0 + c)] = float(a * inv);
  }
}

__global__ __launch_bounds__(256) void k_sgs_samples(const float* __restrict__ fld, int nx, int ny, int nz,
                                                     float* __restrict__ feats, float* __restrict__ labels) {
  const uint64_t nc = uint64_t(nx) * ny * nz;
  const uint64_t c = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  const int x = int(c % nx), y = int((c / nx) % ny), z = int(c / (uint64_t(nx) * ny));
  const int xp = x == nx - 1 ? 0 : x + 1, xm = x == 0 ? nx - 1 : x - 1;
  const int yp = y == ny - 1 ? 0 : y + 1, ym = y == 0 ? ny - 1 : y - 1;
  const int zp = z == nz - 1 ? 0 : z + 1, zm = z == 0 ? nz - 1 : z - 1;
  auto at = [&](int k, int zz, int yy, int xx) {
    return double(fld[uint64_t(k) * nc + (uint64_t(zz) * ny + yy) * nx + xx]);
  };
  double g[3][3];  // g[i][j] = d u_i / d x_j
  for (int i = 0; i < 3; ++i) {
    g[i][0] = 0.5 * (at(1 + i, z, y, xp) - at(1 + i, z, y, xm));
    g[i][1] = 0.5 * (at(1 + i, z, yp, x) - at(1 + i, z, ym, x));
    g[i][2] = 0.5 * (at(1 + i, zp, y, x) - at(1 + i, zm, y, x));
  }
  const int ci[6] = {0, 1, 2, 0, 0, 1}, cj[6] = {0, 1, 2, 1, 2, 2};
  const double ux = at(1, z, y, x), uy = at(2, z, y, x), uz = at(3, z, y, x);
  const double um[3] = {ux, uy, uz};
  double ss = 0.0, ts = 0.0;
  for (int k = 0; k < 6; ++k) {
    const int i = ci[k], j = cj[k];
    const double s = 0.5 * (g[i][j] + g[j][i]);
    const double tau = at(4 + k, z, y, x) - um[i] * um[j];
    const double w = i == j ? 1.0 : 2.0;
    ss += w * s * s;
    ts += w * tau * s;
    feats[c * NIN + k] = float(s);
  }
  feats[c * NIN + 6] = float(sqrt(2.0 * ss));
  const double nu = -ts / (2.0 * (ss > 1e-30 ? ss : 1e-30));
  labels[c] = float(nu > 0.0 ? nu : 0.0);
}

}  // namespace tlbm

// ===========================================================================
// C ABI
// ===========================================================================

using namespace tlbm;

namespace tlbm {
int set_error(int code, const char* msg);  // tlbm.hip: shared tlbm_last_error() channel
}

namespace {

int cfail(int code, const char* msg) { return tlbm::set_error(code, msg); }

int claunch(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    char buf[256];
    snprintf(buf, sizeof(buf), "%s: %s", what, hipGetErrorString(e));
    return tlbm::set_error(TLBM_ERR_HIP, buf);
  }
  return TLBM_OK;
}

// Device address of `scratch` on the current device.  Host code must never pass the array's
// name to a kernel: on the host it is a stand-in, not the device copy's address.  Looked up once
// per device (each GPU holds its own copy at its own address) and kept.
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
float* g_scratch[MAX_DEVICES] = {};

int scratch_ptr(float** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return cfail(TLBM_ERR_HIP, "hipGetDevice failed");
  if (dev < 0 || dev >= MAX_DEVICES) return cfail(TLBM_ERR_UNSUPPORTED, "device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(tlbm::scratch));
    if (e != hipSuccess || p == nullptr) {
      char buf[256];
      snprintf(buf, sizeof(buf), "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
      return tlbm::set_error(TLBM_ERR_HIP, buf);
    }
    g_scratch[dev] = static_cast<float*>(p);
  }
  *out = g_scratch[dev];
  return TLBM_OK;
}

}  // namespace

extern "C" {

int tlbm_mlp_sizes(int64_t* nparam, int64_t* ntotal, int64_t* packed_bytes, int64_t* batch_block) {
  if (nparam) *nparam = mlp::NPARAM;
  if (ntotal) *ntotal = mlp::NTOTAL;
  if (packed_bytes) *packed_bytes = int64_t(sizeof(mlp::Packed));
  if (batch_block) *batch_block = GRAD_BS;
  return TLBM_OK;
}

int tlbm_mlp_pack(const float* params, void* packed, tlbm_stream_t stream) {
  if (!params || !packed) return cfail(TLBM_ERR_INVALID, "null pointer");
  hipLaunchKernelGGL(k_mlp_pack<false>, dim3(1), dim3(64), 0, (hipStream_t)stream, params, (mlp::Packed*)packed);
  return claunch("k_mlp_pack");
}

int tlbm_mlp_pack_bf16(const float* params, void* packed, tlbm_stream_t stream) {
  if (!params || !packed) return cfail(TLBM_ERR_INVALID, "null pointer");
  hipLaunchKernelGGL(k_mlp_pack<true>, dim3(1), dim3(64), 0, (hipStream_t)stream, params, (mlp::Packed*)packed);
  return claunch("k_mlp_pack");
}

int tlbm_mlp_predict(const float* params, const float* x, int64_t n, float* y, tlbm_stream_t stream) {
  if (n < 0) return cfail(TLBM_ERR_SHAPE, "negative sample count");
  if (n == 0) return TLBM_OK;
  if (!params || !x || !y) return cfail(TLBM_ERR_INVALID, "null pointer");
  const uint32_t nb = uint32_t((uint64_t(n) + 255) / 256);
  hipLaunchKernelGGL(k_mlp_predict, dim3(nb), dim3(256), 0, (hipStream_t)stream, params, x, uint64_t(n), y);
  return claunch("k_mlp_predict");
}

int tlbm_mlp_grad(const float* params, const float* x, const float* t, int64_t n, float* partials,
                  tlbm_stream_t stream) {
  if (n <= 0) return cfail(TLBM_ERR_SHAPE, "need at least one sample");
  if (!params || !x || !t || !partials) return cfail(TLBM_ERR_INVALID, "null pointer");
  const uint64_t nb = (uint64_t(n) + GRAD_BS - 1) / GRAD_BS;
  if (nb >= (uint64_t(1) << 31)) return cfail(TLBM_ERR_SHAPE, "batch too large");
  hipLaunchKernelGGL(k_mlp_grad, dim3(uint32_t(nb)), dim3(256), 0, (hipStream_t)stream, params, x, t,
                     (const int64_t*)nullptr, uint64_t(n), 1.0f / float(n), partials);
  return claunch("k_mlp_grad");
}

int tlbm_mlp_adam(float* params, const float* partials, int nblocks, float* m, float* v, int step, float lr,
                  float beta1, float beta2, float eps, float clip_norm, float* loss_out, float* grad_out,
                  tlbm_stream_t stream) {
  if (nblocks <= 0 || step < 1) return cfail(TLBM_ERR_INVALID, "need nblocks > 0 and step >= 1");
  if (!params || !partials || (lr != 0.0f && (!m || !v))) return cfail(TLBM_ERR_INVALID, "null pointer");
  const float bc1 = 1.0f - powf(beta1, float(step));
  const float bc2 = 1.0f - powf(beta2, float(step));
  hipLaunchKernelGGL(k_mlp_adam, dim3(1), dim3(ADAM_THREADS), 0, (hipStream_t)stream, params, partials, nblocks, m,
                     v, lr, beta1, beta2, eps, bc1, bc2, clip_norm, loss_out, grad_out, (double*)nullptr, 0.0);
  return claunch("k_mlp_adam");
}

int tlbm_mlp_train_step_noalloc(float* params, const float* x, const float* t, int64_t n, float* m, float* v,
                                int step, float lr, float beta1, float beta2, float eps, float clip_norm,
                                float* loss_out, float* grad_out, tlbm_stream_t stream) {
  if (n <= 0) return cfail(TLBM_ERR_SHAPE, "need at least one sample");
  if (n > TLBM_MLP_NOALLOC_MAX_SAMPLES) {
    char buf[160];
    snprintf(buf, sizeof(buf), "%lld samples exceed the no-allocation limit of %d per call", (long long)n,
             TLBM_MLP_NOALLOC_MAX_SAMPLES);
    return cfail(TLBM_ERR_SHAPE, buf);
  }
  if (step < 1) return cfail(TLBM_ERR_INVALID, "need step >= 1");
  if (!params || !x || !t || (lr != 0.0f && (!m || !v))) return cfail(TLBM_ERR_INVALID, "null pointer");
  float* partials = nullptr;
  const int rc = scratch_ptr(&partials);
  if (rc != TLBM_OK) return rc;
  const int nb = int((n + GRAD_BS - 1) / GRAD_BS);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_mlp_grad, dim3(uint32_t(nb)), dim3(256), 0, s, params, x, t, (const int64_t*)nullptr,
                     uint64_t(n), 1.0f / float(n), partials);
  const int rg = claunch("k_mlp_grad");
  if (rg != TLBM_OK) return rg;
  const float bc1 = 1.0f - powf(beta1, float(step));
  const float bc2 = 1.0f - powf(beta2, float(step));
  hipLaunchKernelGGL(k_mlp_adam, dim3(1), dim3(ADAM_THREADS), 0, s, params, partials, nb, m, v, lr, beta1, beta2,
                     eps, bc1, bc2, clip_norm, loss_out, grad_out, (double*)nullptr, 0.0);
  return claunch("k_mlp_adam");
}

int tlbm_mlp_train_epoch(float* params, const float* x, const float* t, const int64_t* order, int64_t n,
                         int64_t batch, float* workspace, float* m, float* v, int step, float lr, float beta1,
                         float beta2, float eps, float clip_norm, double* loss_sum, tlbm_stream_t stream) {
  if (n <= 0 || batch <= 0) return cfail(TLBM_ERR_SHAPE, "need at least one sample and a positive minibatch");
  if (step < 1) return cfail(TLBM_ERR_INVALID, "need step >= 1");
  if (!params || !x || !t || !order || !workspace || !m || !v || !loss_sum)
    return cfail(TLBM_ERR_INVALID, "null pointer");
  const int64_t rows = (batch + GRAD_BS - 1) / GRAD_BS;
  if (rows >= (int64_t(1) << 31) || (n + batch - 1) / batch >= (int64_t(1) << 31) - step)
    return cfail(TLBM_ERR_SHAPE, "batch too large");
  hipStream_t s = (hipStream_t)stream;
  float* partials = workspace + (NPARAM + 1);
  for (int64_t at = 0; at < n; at += batch, ++step) {
    const int64_t nb = n - at < batch ? n - at : batch;
    const int nblk = int((nb + GRAD_BS - 1) / GRAD_BS);
    hipLaunchKernelGGL(k_mlp_grad, dim3(uint32_t(nblk)), dim3(256), 0, s, params, x, t, order + at, uint64_t(nb),
                       1.0f / float(nb), partials);
    hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + 64) / 64), dim3(256), 0, s, partials, nblk, workspace);
    const float bc1 = 1.0f - powf(beta1, float(step));
    const float bc2 = 1.0f - powf(beta2, float(step));
    hipLaunchKernelGGL(k_mlp_adam, dim3(1), dim3(ADAM_THREADS), 0, s, params, workspace, 1, m, v, lr, beta1, beta2,
                       eps, bc1, bc2, clip_norm, (float*)nullptr, (float*)nullptr, loss_sum, double(nb));
  }
  return claunch("tlbm_mlp_train_epoch");
}

int tlbm_coarsen_moments(int lattice, int store, const void* f, const int64_t* strides, int nz, int ny, int nx,
                         int factor, float* out, tlbm_stream_t stream) {
  if (!f || !out) return cfail(TLBM_ERR_INVALID, "null pointer");
  if (nz < 1 || ny < 1 || nx < 1) return cfail(TLBM_ERR_SHAPE, "grid dims must be >= 1");
  if (factor < 1 || nx % factor || ny % factor || nz % factor)
    return cfail(TLBM_ERR_SHAPE, "grid dims must be multiples of the coarsening factor");
  if (lattice != TLBM_D3Q19 && lattice != TLBM_D3Q27) return cfail(TLBM_ERR_UNSUPPORTED, "3-D lattices only");
  const int64_t N = int64_t(nz) * ny * nx;
  Lay lay{strides ? strides[0] : N, strides ? strides[1] : int64_t(ny) * nx, strides ? strides[2] : nx, nx, ny, nz};
  // a coarse row in as few workgroups as 512 lanes allow, all alike
  const int lanes = factor < COARSEN_LANES ? factor : COARSEN_LANES;
  const int cx = nx / factor, most = COARSEN_LANES / lanes;
  const int cells = (cx + (cx + most - 1) / most - 1) / ((cx + most - 1) / most);
  const uint64_t nb = uint64_t((cx + cells - 1) / cells) * uint64_t(ny / factor) * uint64_t(nz / factor);
  if (nb >= (uint64_t(1) << 31)) return cfail(TLBM_ERR_SHAPE, "too many workgroups");
  const int threads = (cells * lanes + 63) / 64 * 64;
  const size_t lds = size_t(10) * threads * sizeof(double);
  hipStream_t s = (hipStream_t)stream;
#define TLBM_COARSEN(LT, SK) \
  hipLaunchKernelGGL((k_coarsen<LT, SK>), dim3(uint32_t(nb)), dim3(threads), lds, s, f, lay, factor, cells, out)
  if (lattice == TLBM_D3Q19) {
    switch (store) {
      case TLBM_STORE_F32: TLBM_COARSEN(D3Q19, ST_F32); break;
      case TLBM_STORE_F64: TLBM_COARSEN(D3Q19, ST_F64); break;
      case TLBM_STORE_F16_DEV: TLBM_COARSEN(D3Q19, ST_F16_DEV); break;
      default: return cfail(TLBM_ERR_DTYPE, "coarsening takes fp32, fp64 or fp16-deviation populations");
    }
  } else {
    switch (store) {
      case TLBM_STORE_F32: TLBM_COARSEN(D3Q27, ST_F32); break;
      case TLBM_STORE_F64: TLBM_COARSEN(D3Q27, ST_F64); break;
      default: return cfail(TLBM_ERR_DTYPE, "coarsening takes fp32 or fp64 D3Q27 populations");
    }
  }
#undef TLBM_COARSEN
  return claunch("k_coarsen");
}

int tlbm_sgs_samples(const float* fields, int nz, int ny, int nx, float* feats, float* labels, tlbm_stream_t stream) {
  if (!fields || !feats || !labels) return cfail(TLBM_ERR_INVALID, "null pointer");
  if (nx < 3 || ny < 3 || nz < 3) return cfail(TLBM_ERR_SHAPE, "coarse grid needs at least 3 cells per axis");
  const uint64_t nc = uint64_t(nx) * ny * nz;
  hipLaunchKernelGGL(k_sgs_samples, dim3(uint32_t((nc + 255) / 256)), dim3(256), 0, (hipStream_t)stream, fields, nx,
                     ny, nz, feats, labels);
  return claunch("k_sgs_samples");
}

}  // extern "C"
