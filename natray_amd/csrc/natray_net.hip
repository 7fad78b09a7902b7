// The CG warm-start network: a 4-layer 3D convolution net on 16^3 tiles of cells, with
// hand-written BF16 MFMA kernels (v_mfma_f32_16x16x32_bf16, FP32 accumulate) for the forward
// pass and both gradients, and the training step (masked MSE, Adam) on the GPU.
//
// Layers: conv 3^3 C0 -> 16, ReLU, conv 16 -> 16, ReLU, conv 16 -> 16, ReLU, conv 16 -> 1.
// Tiles are independent, zero-padded at their faces. Activations are NDHWC per tile: voxel
// v = 256 x + 16 y + z of the 16^3 tile, channels contiguous, stored as BF16 with 8 or 16
// channels (the 2 input channels and the 1 output channel are padded with zeros).
//
// A convolution is an implicit GEMM: rows are voxels, K runs over (tap, input channel) with
// k = tap * Cin + c (tap = 9 (dx + 1) + 3 (dy + 1) + (dz + 1)), columns are output channels.
// One wave computes the 16 voxels of a z-row against 16 output channels: lane l holds voxel
// l % 16 and the 8 consecutive k of group l / 16 of each 32-wide K step (8 channels of one
// tap: one 16-byte load), and gets rows 4 (l / 16) .. + 3 of column l % 16 back.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "natray.h"
#include "natray_net.h"

namespace natray {
namespace net {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int TILE = 16;
constexpr int VOX = TILE * TILE * TILE;  // 4096
constexpr int TAPS = 27;

__host__ __device__ constexpr int ksteps(int cin) { return (TAPS * cin + 31) / 32; }

// Y[t][v][n] = act(bias[n] + sum_k X[t][v + off(tap)][c] W[k][n]) for n < 16, with W in the
// MFMA B layout `wb` (ksteps(CIN) x 4 groups x 16 columns x 8 values, see k_pack). `yf` (FP32,
// 16 channels), `y1` (FP32, channel 0 alone) or `yb` (BF16, 16 channels) receives the result;
// with `gate` (BF16, 16 channels), 0 where it is not positive: the ReLU's gradient.
//
// A work item is XP = 2 output x-planes of one tile (32 z-rows). Its input slab, planes
// x0 - 1 .. x0 + 2 with y and z from -1 to 16, is staged in LDS with zeros outside the tile, so
// the A fragments are plain 16-byte LDS reads at lane-constant offsets (no bounds tests); a
// staged voxel holds CIN channels padded to VS so that the 16 lanes of a row, 48 bytes apart
// for CIN = 16, fall in distinct banks. The weights stay in registers (B fragments, one per
// K step). Each wave runs two z-rows at a time, two independent MFMA chains. Work items are
// strided over the grid; the tile count is `tiles`, or min(*tiles_dev, tiles) when tiles_dev is
// given (a count only the device knows when the work is enqueued).
constexpr int XP = 2;
constexpr int SLAB = (XP + 2) * 18 * 18;

template <int CIN>
struct ConvShape {
  static constexpr int VS = CIN == 16 ? 24 : 8;  // bf16 per staged voxel
  static constexpr int KS = ksteps(CIN);
};

template <int CIN>
__global__ __launch_bounds__(256) void k_conv(const __bf16* __restrict__ X, const bf16x8* __restrict__ wb,
                                              const float* __restrict__ bias, int relu, const __bf16* __restrict__ gate,
                                              __bf16* __restrict__ yb, float* __restrict__ yf, float* __restrict__ y1,
                                              int tiles, const uint32_t* __restrict__ tiles_dev) {
  using Sh = ConvShape<CIN>;
  constexpr int VS = Sh::VS, KS = Sh::KS, CH = CIN / 8;  // 16-byte chunks of data per staged voxel
  constexpr int PER_THREAD = (SLAB * CH + 255) / 256;
  __shared__ __attribute__((aligned(16))) __bf16 slab[SLAB * VS];
  const int nt = tiles_dev ? (int)min(*tiles_dev, (uint32_t)tiles) : tiles;
  const int items = nt * (TILE / XP);
  if ((int)blockIdx.x >= items) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int g = lane >> 4, col = lane & 15;
  bf16x8 w[KS];
  int off[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    w[s] = wb[s * 64 + lane];
    const int k = s * 32 + g * 8, tap = k / CIN, c0 = k % CIN;
    const int dx = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dz = tap % 3 - 1;
    // K padding (tap 27) reads a valid slab address and is replaced by zeros below.
    off[s] = tap < TAPS ? ((dx * 18 + dy) * 18 + dz) * VS + c0 : 0;
  }
  // Only the last step can hold K padding (tap 27).
  const bool last_ok = ((KS - 1) * 32 + g * 8) / CIN < TAPS;
  bf16x8 zero;
#pragma unroll
  for (int j = 0; j < 8; ++j) zero[j] = (__bf16)0.0f;
  const float bcol = bias ? bias[col] : 0.0f;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int t = item / (TILE / XP), x0 = (item % (TILE / XP)) * XP;
    const __bf16* Xt = X + (size_t)t * VOX * CIN;
    // Every load of the slab is issued before the first LDS store (the padding of a staged
    // voxel beyond CIN channels is never read and stays unwritten).
    bf16x8 val[PER_THREAD];
#pragma unroll
    for (int k = 0; k < PER_THREAD; ++k) {
      const int i = threadIdx.x + 256 * k;
      const int v = i / CH, j = i % CH;
      const int px = v / 324, py = (v / 18) % 18, pz = v % 18;
      const int x = x0 - 1 + px, y = py - 1, z = pz - 1;
      val[k] = zero;
      if (i < SLAB * CH && (unsigned)x < TILE && (unsigned)y < TILE && (unsigned)z < TILE)
        val[k] = *reinterpret_cast<const bf16x8*>(Xt + (size_t)((x * TILE + y) * TILE + z) * CIN + 8 * j);
    }
    __syncthreads();  // the previous item's reads of the slab are done
#pragma unroll
    for (int k = 0; k < PER_THREAD; ++k) {
      const int i = threadIdx.x + 256 * k;
      if (i < SLAB * CH) *reinterpret_cast<bf16x8*>(slab + (i / CH) * VS + 8 * (i % CH)) = val[k];
    }
    __syncthreads();
    for (int r = wave; r < XP * TILE; r += 8) {
      f32x4 acc[2];
      int base[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int rr = r + 4 * h, xo = rr / TILE, y = rr % TILE;
        base[h] = (((xo + 1) * 18 + (y + 1)) * 18 + (col + 1)) * VS;
        acc[h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int s = 0; s < KS; ++s) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          bf16x8 a = *reinterpret_cast<const bf16x8*>(slab + base[h] + off[s]);
          if (s == KS - 1 && !last_ok) a = zero;
          acc[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[s], acc[h], 0, 0, 0);
        }
      }
      // acc[h][i] is voxel z = 4 g + i of row r + 4 h, output channel col.
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int rr = r + 4 * h, row = (x0 + rr / TILE) * TILE + rr % TILE;
        const size_t vox0 = (size_t)t * VOX + (size_t)row * TILE + 4 * g;
        if (y1) {
          f32x4 v = acc[h];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] += bcol;
            if (relu) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
          }
          if (col == 0) *reinterpret_cast<f32x4*>(y1 + vox0) = v;
          continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[h][i] + bcol;
          if (relu) v = v > 0.0f ? v : 0.0f;
          const size_t o = (vox0 + i) * 16 + col;
          if (gate && !((float)gate[o] > 0.0f)) v = 0.0f;
          if (yf) yf[o] = v;
          if (yb) yb[o] = (__bf16)v;
        }
      }
    }
  }
}

// Packs FP32 weights W[tap][cin_real][cout_real] into the MFMA B layout of a layer with cin
// input and 16 output channels (zeros where the padding is), BF16. With `flip`, packs the
// weights of the input-gradient convolution instead: W'[tap][n][c] = W[26 - tap][c][n], whose
// input channels are the layer's outputs (cin = 16) and outputs its inputs.
struct PackJob {
  const float* W;
  int cin_real, cout_real, cin, flip;
  bf16x8* wb;
};
struct PackJobs {
  PackJob job[7];
};
constexpr int PACK_MAX = (ksteps(16) * 64 + 255) / 256;  // workgroups of the largest job
// One job per gridDim.y.
__global__ void k_pack(PackJobs jobs) {
  const PackJob& jb = jobs.job[blockIdx.y];
  const float* __restrict__ W = jb.W;
  const int cin_real = jb.cin_real, cout_real = jb.cout_real, cin = jb.cin, flip = jb.flip;
  bf16x8* __restrict__ wb = jb.wb;
  const int ks = ksteps(cin);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;  // (s, lane)
  if (i >= ks * 64) return;
  const int s = i / 64, lane = i % 64, g = lane >> 4, n = lane & 15;
  bf16x8 out;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int k = s * 32 + g * 8 + j, tap = k / cin, c = k % cin;
    float w = 0.0f;
    if (tap < TAPS) {
      if (!flip) {
        if (c < cin_real && n < cout_real) w = W[((size_t)tap * cin_real + c) * cout_real + n];
      } else {
        // c is the layer's output channel, n its input channel.
        if (c < cout_real && n < cin_real) w = W[((size_t)(TAPS - 1 - tap) * cin_real + n) * cout_real + c];
      }
    }
    out[j] = (__bf16)w;
  }
  wb[i] = out;
}

// dZ = dY where the layer's ReLU output was positive (all of dY without ReLU), as BF16. For the check
// of one layer, whose dY is given; in training k_conv's gate does this where dY is made.
__global__ void k_relu_back(const float* __restrict__ dY, const __bf16* __restrict__ Y, int relu, __bf16* __restrict__ dZ,
                            size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float g = dY[i];
    dZ[i] = (__bf16)((!relu || (float)Y[i] > 0.0f) ? g : 0.0f);
  }
}

// Partial sums over voxels of X[v + off(tap)][c] dZ[v][n] (the weights' gradient) and of dZ[v][n]
// (the bias's), on MFMA with K over voxels: rows are 16 consecutive k = tap CIN + c, columns n.
// A work item is XP x-planes of a tile, as in k_conv; a workgroup walks items blockIdx.x,
// + gridDim.x, ... and leaves its sums in part[blockIdx.x][k][n], the bias's behind them, which
// k_grad_fold adds up in workgroup order.
//
// Eight consecutive voxels of a fragment lie along z, so the item's inputs are staged channel by
// channel with z fastest, once per dz: each fragment is then one aligned 16-byte LDS read. (With
// every fragment gathered from global memory two bytes at a time and its sums added to the
// gradient with atomics, a layer took 36 us at 32 tiles, and its bias 16 in a kernel of its own;
// now 10 together.)
template <int CIN>
struct WgradShape {
  static constexpr int ROWS = (TAPS * CIN + 15) / 16;       // 16-row blocks
  static constexpr int CS = (XP + 2) * 18 * TILE + 8;       // bf16 per channel and dz (padded: banks)
  static constexpr int NS = XP * TILE * TILE + 8;           // bf16 per column of dZ
  static constexpr int PART = TAPS * CIN * 16 + 16;         // floats per workgroup
  static constexpr int WAVES = 8;
  static constexpr int PER = (ROWS + 1 + WAVES - 1) / WAVES;  // row blocks per wave, the bias's among them
};
template <int CIN>
__global__ __launch_bounds__(512) void k_conv_wgrad(const __bf16* __restrict__ X, const __bf16* __restrict__ dZ,
                                                    float* __restrict__ part, int tiles) {
  using Sh = WgradShape<CIN>;
  __shared__ __attribute__((aligned(16))) __bf16 xt[3 * CIN * Sh::CS];
  __shared__ __attribute__((aligned(16))) __bf16 zt[16 * Sh::NS];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
  const int items = tiles * (TILE / XP);
  f32x4 acc[Sh::PER];
  int at[Sh::PER];  // the fragment's row in xt at output plane 0, row 0; -1 padding, -2 the bias
#pragma unroll
  for (int q = 0; q < Sh::PER; ++q) {
    acc[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int rb = wave + Sh::WAVES * q, k = rb * 16 + m, tap = k / CIN, c = k % CIN;
    at[q] = -1;
    if (rb < Sh::ROWS && tap < TAPS) at[q] = ((tap % 3) * CIN + c) * Sh::CS + ((tap / 9) * 18 + (tap / 3) % 3) * TILE;
    if (rb == Sh::ROWS) at[q] = -2;
  }
  bf16x8 zero, ones;
#pragma unroll
  for (int j = 0; j < 8; ++j) zero[j] = (__bf16)0.0f, ones[j] = (__bf16)1.0f;
  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int t = item / (TILE / XP), x0 = (item % (TILE / XP)) * XP;
    const __bf16* Xt = X + (size_t)t * VOX * CIN;
    const __bf16* Zt = dZ + ((size_t)t * VOX + (size_t)x0 * TILE * TILE) * 16;
    __syncthreads();  // the previous item's reads are done
    // Planes x0 - 1 .. x0 + XP, rows y = -1 .. 16, voxel z of copy dz = X[z + dz - 1].
    constexpr int CH = CIN / 8, ROWVOX = (XP + 2) * 18 * TILE;
    for (int i = threadIdx.x; i < ROWVOX * CH; i += 512) {
      const int j = i % CH, v = i / CH, z = v % TILE, py = (v / TILE) % 18, px = v / (TILE * 18);
      const int x = x0 - 1 + px, y = py - 1;
      bf16x8 val = zero;
      if ((unsigned)x < TILE && (unsigned)y < TILE)
        val = *reinterpret_cast<const bf16x8*>(Xt + (size_t)((x * TILE + y) * TILE + z) * CIN + 8 * j);
      const int row = (px * 18 + py) * TILE;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int c = 8 * j + e;
        xt[(0 * CIN + c) * Sh::CS + row + (z + 1) % TILE] = z + 1 < TILE ? val[e] : (__bf16)0.0f;
        xt[(1 * CIN + c) * Sh::CS + row + z] = val[e];
        xt[(2 * CIN + c) * Sh::CS + row + (z + TILE - 1) % TILE] = z > 0 ? val[e] : (__bf16)0.0f;
      }
    }
    for (int i = threadIdx.x; i < XP * TILE * TILE * 2; i += 512) {
      const int j = i & 1, v = i >> 1;
      const bf16x8 val = *reinterpret_cast<const bf16x8*>(Zt + (size_t)v * 16 + 8 * j);
#pragma unroll
      for (int e = 0; e < 8; ++e) zt[(8 * j + e) * Sh::NS + v] = val[e];
    }
    __syncthreads();
    // 32 voxels a step: rows y and y + 1 of output plane xo, group g taking 8 voxels along z.
    for (int s = 0; s < XP * TILE / 2; ++s) {
      const int xo = s / (TILE / 2), y = s % (TILE / 2) * 2 + (g >> 1), z0 = (g & 1) * 8;
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(zt + m * Sh::NS + (xo * TILE + y) * TILE + z0);
#pragma unroll
      for (int q = 0; q < Sh::PER; ++q) {
        if (wave + Sh::WAVES * q > Sh::ROWS) continue;
        bf16x8 a = at[q] == -2 ? ones : zero;
        if (at[q] >= 0) a = *reinterpret_cast<const bf16x8*>(xt + at[q] + (xo * 18 + y) * TILE + z0);
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[q], 0, 0, 0);
      }
    }
  }
  // acc[q][i]: row rb * 16 + 4 g + i, column m.
  float* out = part + (size_t)blockIdx.x * Sh::PART;
#pragma unroll
  for (int q = 0; q < Sh::PER; ++q) {
    const int rb = wave + Sh::WAVES * q;
    if (rb < Sh::ROWS) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = rb * 16 + 4 * g + i;
        if (k < TAPS * CIN) out[k * 16 + m] = acc[q][i];
      }
    } else if (rb == Sh::ROWS && g == 0) {
      out[TAPS * CIN * 16 + m] = acc[q][0];
    }
  }
}

// Adds up the workgroups' partial sums of each layer's gradient, and the loss's into loss[0], in
// a fixed order: a workgroup per 16 outputs, thread t taking partials t / 16, + 16, ...
struct FoldJob {
  const float* part;
  int groups, stride, cin, cin_real, cout_real;
  float *dW, *db;
};
struct FoldJobs {
  FoldJob job[4];
  const float* loss_part;
  int loss_parts;
  float* loss;
};
constexpr int FOLD_BLOCKS = TAPS * 16 + 1;  // rows of outputs of the largest layer
__global__ __launch_bounds__(256) void k_grad_fold(FoldJobs jobs) {
  const FoldJob& jb = jobs.job[blockIdx.y];
  __shared__ float w[4][16];
  const int lane = threadIdx.x & 63, n = lane & 15;
  const int k = blockIdx.x, rows = TAPS * jb.cin;  // row `rows` is the bias
  if (k <= rows) {
    float s = 0.0f;
#pragma unroll 4
    for (int q = threadIdx.x >> 4; q < jb.groups; q += 16) s += jb.part[(size_t)q * jb.stride + k * 16 + n];
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (lane < 16) w[threadIdx.x >> 6][n] = s;
    __syncthreads();
    if (threadIdx.x < 16u && n < jb.cout_real) {
      s = (w[0][n] + w[1][n]) + (w[2][n] + w[3][n]);
      const int tap = k / jb.cin, c = k % jb.cin;
      if (k == rows)
        jb.db[n] = s;
      else if (c < jb.cin_real)
        jb.dW[((size_t)tap * jb.cin_real + c) * jb.cout_real + n] = s;
    }
  }
  if (jobs.loss && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 64u) {
    float s = 0.0f;
    for (int i = lane; i < jobs.loss_parts; i += 64) s += jobs.loss_part[i];
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) jobs.loss[0] = s;
  }
}

// A workgroup's share of the loss (all 256 threads call it).
__device__ __forceinline__ void loss_part(float s, float inv_count, float* __restrict__ part) {
  __shared__ float w[4];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((w[0] + w[1]) + (w[2] + w[3])) * inv_count;
}
// The gradient g at channel 0 of a voxel's BF16 record, zeros in the others.
__device__ __forceinline__ void store_dz(__bf16* __restrict__ dz, size_t v, float g) {
  bf16x8 lo, hi;
#pragma unroll
  for (int j = 0; j < 8; ++j) lo[j] = hi[j] = (__bf16)0.0f;
  lo[0] = (__bf16)g;
  reinterpret_cast<bf16x8*>(dz)[2 * v] = lo;
  reinterpret_cast<bf16x8*>(dz)[2 * v + 1] = hi;
}

// Masked mean squared error of `pred` against `target`: each workgroup's share of the loss to
// part, and dZ = 2 (pred - target) mask / count on channel 0.
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ pred, const float* __restrict__ target,
                                             const float* __restrict__ mask, float inv_count, __bf16* __restrict__ dz,
                                             float* __restrict__ part, size_t voxels) {
  float s = 0.0f;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x) {
    const float e = (pred[v] - target[v]) * mask[v];
    s += e * e;
    store_dz(dz, v, 2.0f * e * inv_count);
  }
  loss_part(s, inv_count, part);
}

// The scaled residual of a guess on each tile: e_v = x_v - (A o)_v on water voxels (diag_v > 0),
// with (A o)_v = diag_v o_v - sum of o_u over the water neighbours u of v inside the tile (bit
// 2 axis + 1 of nbm for the + side, 2 axis for the - side; axes x, y, z are voxel strides 256,
// 16, 1); x is input channel 0 (FP32, [voxel][2]) and o is `pred`. Writes e, and each workgroup's
// share of the mean of e^2 over the water voxels to part. (Every wave adding its share to one word
// took 29 us at 32 tiles; now 5.)
__device__ __forceinline__ float tile_stencil(const float* __restrict__ f, size_t v, uint32_t bits) {
  const int z = (int)(v & 15), y = (int)((v >> 4) & 15), x = (int)((v >> 8) & 15);
  float s = 0.0f;
  if ((bits & 1u) && x > 0) s += f[v - 256];
  if ((bits & 2u) && x < 15) s += f[v + 256];
  if ((bits & 4u) && y > 0) s += f[v - 16];
  if ((bits & 8u) && y < 15) s += f[v + 16];
  if ((bits & 16u) && z > 0) s += f[v - 1];
  if ((bits & 32u) && z < 15) s += f[v + 1];
  return s;
}
__global__ __launch_bounds__(256) void k_res_e(const float* __restrict__ pred, const float* __restrict__ x,
                                               const float* __restrict__ diag, const uint32_t* __restrict__ nbm,
                                               float inv_count, float* __restrict__ e, float* __restrict__ part, size_t voxels) {
  float s = 0.0f;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x) {
    float ev = 0.0f;
    if (diag[v] > 0.0f) ev = x[v * 2] - (diag[v] * pred[v] - tile_stencil(pred, v, nbm[v]));
    e[v] = ev;
    s += ev * ev;
  }
  loss_part(s, inv_count, part);
}
// d loss / d o = -2 A e / count on water voxels (A is symmetric), as dZ's channel 0.
__global__ void k_res_grad(const float* __restrict__ e, const float* __restrict__ diag, const uint32_t* __restrict__ nbm,
                           float inv_count, __bf16* __restrict__ dz, size_t voxels) {
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x) {
    float g = 0.0f;
    if (diag[v] > 0.0f) g = -2.0f * inv_count * (diag[v] * e[v] - tile_stencil(e, v, nbm[v]));
    store_dz(dz, v, g);
  }
}

// Adam (Kingma and Ba, 2015) on n parameters with bias-corrected moments.
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       int n, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi / c1) / (__builtin_sqrtf(vi / c2) + eps);
}

}  // namespace net
}  // namespace natray

// ---- host side -------------------------------------------------------------------------------

namespace natray {
namespace net {

// FP32 [voxels][2] -> BF16 [voxels][8], zero padded, 16 bytes a store.
__global__ __launch_bounds__(256) void k_input(const float2* __restrict__ src, bf16x8* __restrict__ dst, size_t voxels) {
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x) {
    const float2 s = src[v];
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (__bf16)0.0f;
    o[0] = (__bf16)s.x;
    o[1] = (__bf16)s.y;
    dst[v] = o;
  }
}
// FP32 [voxels][cin_real] -> BF16 [voxels][cin] with zero padding.
__global__ void k_to_bf16(const float* __restrict__ src, int cin_real, int cin, __bf16* __restrict__ dst, size_t voxels) {
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x)
    for (int c = 0; c < cin; ++c) dst[v * cin + c] = (__bf16)(c < cin_real ? src[v * cin_real + c] : 0.0f);
}
// The first cout_real channels of FP32 [voxels][16] into [voxels][cout_real].
__global__ void k_take(const float* __restrict__ src, int cout_real, float* __restrict__ dst, size_t voxels) {
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x)
    for (int c = 0; c < cout_real; ++c) dst[v * cout_real + c] = src[v * 16 + c];
}
// FP32 [voxels][cout_real] into [voxels][16], zero padded.
__global__ void k_pad16(const float* __restrict__ src, int cout_real, float* __restrict__ dst, size_t voxels) {
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < voxels; v += (size_t)gridDim.x * blockDim.x)
    for (int c = 0; c < 16; ++c) dst[v * 16 + c] = c < cout_real ? src[v * cout_real + c] : 0.0f;
}

struct Layer {
  int cin_real, cout_real, cin, relu;
  size_t w_off, b_off;  // into the parameter vector
};

// W1 27x2x16, b1 16, W2 27x16x16, b2 16, W3 27x16x16, b3 16, W4 27x16x1, b4 1.
constexpr Layer LAYERS[4] = {
    {2, 16, 8, 1, 0, 864},
    {16, 16, 16, 1, 880, 880 + 6912},
    {16, 16, 16, 1, 880 + 6928, 880 + 6928 + 6912},
    {16, 1, 16, 0, 880 + 2 * 6928, 880 + 2 * 6928 + 432},
};
static_assert(880 + 2 * 6928 + 433 == NATRAY_NET_PARAMS, "parameter layout");

}  // namespace net
}  // namespace natray

using namespace natray::net;

struct natray_net {
  uint32_t max_tiles = 0;
  float* p = nullptr;     // parameters (FP32 master copy)
  float* g = nullptr;     // their gradients
  float* m = nullptr;     // Adam moments
  float* v = nullptr;
  bf16x8* wb[4] = {};     // packed forward weights
  bf16x8* wt[4] = {};     // packed input-gradient weights (layers 2..4)
  __bf16* in = nullptr;   // [T][4096][8]
  __bf16* act[3] = {};    // [T][4096][16] outputs of layers 1..3
  float* out = nullptr;   // [T][4096] output of layer 4
  __bf16* dz[2] = {};     // [T][4096][16] gradient w.r.t. a layer's output through the ReLU, BF16:
                          // a layer's and the one below's
  float* part = nullptr;  // the workgroups' partial gradients, layer by layer (part_off)
  float* lpart = nullptr; // LOSS_PARTS: the workgroups' shares of the loss
  float* target = nullptr;
  float* mask = nullptr;
  float* resid = nullptr;  // [T][4096] residual of the residual loss
  float* stage = nullptr;  // [T][4096][2] FP32 staging of inputs and outputs
  float* loss = nullptr;
  std::vector<void*> allocs;
  uint32_t steps = 0;
  bool packed = false;
  hipStream_t stream = nullptr;
};

namespace {

thread_local std::string g_net_err;

int nfail(int code, const std::string& msg) {
  g_net_err = msg;
  return code;
}

#define NCHK(x)                                                                                       \
  do {                                                                                                \
    hipError_t e_ = (x);                                                                              \
    if (e_ != hipSuccess) return nfail(NATRAY_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

template <class T>
int nalloc(natray_net* n, T** ptr, size_t count) {
  void* q = nullptr;
  hipError_t e = hipMalloc(&q, (count ? count : 1) * sizeof(T));
  if (e != hipSuccess) return nfail(NATRAY_E_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  n->allocs.push_back(q);
  *ptr = static_cast<T*>(q);
  return NATRAY_OK;
}

// Workgroups of k_conv_wgrad (its LDS leaves one per CU), and of the loss kernels.
constexpr uint32_t WGRAD_GROUPS = 256, LOSS_PARTS = 512;
constexpr size_t part_size(int cin) {
  return (size_t)WGRAD_GROUPS * (cin == 8 ? WgradShape<8>::PART : WgradShape<16>::PART);
}
constexpr size_t part_off(int l) { return l == 0 ? 0 : part_size(8) + (size_t)(l - 1) * part_size(16); }
unsigned grid_for(size_t items) { return (unsigned)std::min<size_t>((items + 255) / 256, 4096); }

int pack(natray_net* n) {
  PackJobs jobs{};
  int k = 0;
  for (int l = 0; l < 4; ++l) {
    const Layer& L = LAYERS[l];
    jobs.job[k++] = PackJob{n->p + L.w_off, L.cin_real, L.cout_real, L.cin, 0, n->wb[l]};
    if (l > 0) jobs.job[k++] = PackJob{n->p + L.w_off, L.cin_real, L.cout_real, 16, 1, n->wt[l]};
  }
  hipLaunchKernelGGL(k_pack, dim3(PACK_MAX, k), dim3(256), 0, n->stream, jobs);
  NCHK(hipGetLastError());
  n->packed = true;
  return NATRAY_OK;
}

// A convolution over `tiles` tiles: one workgroup per work item (2 x-planes), up to 2 per CU
// (the LDS slab of a 16-channel input takes 62 KB).
void launch_conv(int cin, uint32_t tiles, hipStream_t stream, const __bf16* X, const bf16x8* wb, const float* bias, int relu,
                 const __bf16* gate, __bf16* yb, float* yf, float* y1, const uint32_t* tiles_dev) {
  const unsigned grid = (unsigned)std::min<uint32_t>(tiles * (TILE / XP), 512u);
  if (cin == 8)
    hipLaunchKernelGGL(k_conv<8>, dim3(grid), dim3(256), 0, stream, X, wb, bias, relu, gate, yb, yf, y1, (int)tiles, tiles_dev);
  else
    hipLaunchKernelGGL(k_conv<16>, dim3(grid), dim3(256), 0, stream, X, wb, bias, relu, gate, yb, yf, y1, (int)tiles, tiles_dev);
}

// The weights' and bias's partial gradients of a layer; returns the workgroups that left one.
uint32_t launch_wgrad(int cin, uint32_t tiles, hipStream_t stream, const __bf16* X, const __bf16* dz, float* part) {
  const uint32_t groups = std::min<uint32_t>(tiles * (TILE / XP), WGRAD_GROUPS);
  if (cin == 8)
    hipLaunchKernelGGL(k_conv_wgrad<8>, dim3(groups), dim3(512), 0, stream, X, dz, part, (int)tiles);
  else
    hipLaunchKernelGGL(k_conv_wgrad<16>, dim3(groups), dim3(512), 0, stream, X, dz, part, (int)tiles);
  return groups;
}

int forward(natray_net* n, uint32_t tiles, const uint32_t* tiles_dev = nullptr) {
  if (!n->packed) {
    int e = pack(n);
    if (e) return e;
  }
  const __bf16* x = n->in;
  for (int l = 0; l < 4; ++l) {
    const Layer& L = LAYERS[l];
    launch_conv(L.cin, tiles, n->stream, x, n->wb[l], n->p + L.b_off, L.relu, nullptr, l < 3 ? n->act[l] : nullptr, nullptr,
                l == 3 ? n->out : nullptr, tiles_dev);
    if (l < 3) x = n->act[l];
  }
  NCHK(hipGetLastError());
  return NATRAY_OK;
}

// Gradients of the loss of the last forward: the masked MSE against n->target, or with
// `residual` the scaled residual with the operator in n->target (diagonal) and n->mask
// (neighbour bits). The parameters' gradients go to n->g.
int backward(natray_net* n, uint32_t tiles, float inv_count, bool residual = false) {
  const size_t vox = (size_t)tiles * VOX;
  const unsigned lgrid = std::min(grid_for(vox), (unsigned)LOSS_PARTS);
  __bf16* dz = n->dz[0];
  if (!residual) {
    hipLaunchKernelGGL(k_mse, dim3(lgrid), dim3(256), 0, n->stream, n->out, n->target, n->mask, inv_count, dz, n->lpart, vox);
  } else {
    const uint32_t* bits = reinterpret_cast<const uint32_t*>(n->mask);
    hipLaunchKernelGGL(k_res_e, dim3(lgrid), dim3(256), 0, n->stream, n->out, n->stage, n->target, bits, inv_count,
                       n->resid, n->lpart, vox);
    hipLaunchKernelGGL(k_res_grad, dim3(grid_for(vox)), dim3(256), 0, n->stream, n->resid, n->target, bits, inv_count, dz,
                       vox);
  }
  FoldJobs jobs{};
  for (int l = 3; l >= 0; --l) {
    const Layer& L = LAYERS[l];
    float* part = n->part + part_off(l);
    const uint32_t groups = launch_wgrad(L.cin, tiles, n->stream, l > 0 ? n->act[l - 1] : n->in, dz, part);
    jobs.job[l] = FoldJob{part, (int)groups, L.cin == 8 ? WgradShape<8>::PART : WgradShape<16>::PART, L.cin, L.cin_real,
                          L.cout_real, n->g + L.w_off, n->g + L.b_off};
    if (l > 0) {
      // The input's gradient through the ReLU of the layer below.
      __bf16* below = dz == n->dz[0] ? n->dz[1] : n->dz[0];
      launch_conv(16, tiles, n->stream, dz, n->wt[l], nullptr, 0, n->act[l - 1], below, nullptr, nullptr, nullptr);
      dz = below;
    }
  }
  jobs.loss_part = n->lpart;
  jobs.loss_parts = (int)lgrid;
  jobs.loss = n->loss;
  hipLaunchKernelGGL(k_grad_fold, dim3(FOLD_BLOCKS, 4), dim3(256), 0, n->stream, jobs);
  NCHK(hipGetLastError());
  return NATRAY_OK;
}

int upload_input(natray_net* n, const float* input, uint32_t tiles) {
  const size_t vox = (size_t)tiles * VOX;
  NCHK(hipMemcpyAsync(n->stage, input, vox * 2 * 4, hipMemcpyHostToDevice, n->stream));
  hipLaunchKernelGGL(k_input, dim3(grid_for(vox)), dim3(256), 0, n->stream, reinterpret_cast<const float2*>(n->stage),
                     reinterpret_cast<bf16x8*>(n->in), vox);
  NCHK(hipGetLastError());
  return NATRAY_OK;
}

}  // namespace

namespace natray {
namespace net {
int forward_device(natray_net* n, uint32_t tiles, const uint32_t* tiles_dev, void* stream) {
  hipStream_t keep = n->stream;
  n->stream = static_cast<hipStream_t>(stream);
  int e = forward(n, std::min(tiles, n->max_tiles), tiles_dev);
  n->stream = keep;
  return e;
}
void* input_buffer(natray_net* n) { return n->in; }
const float* output_buffer(natray_net* n) { return n->out; }
uint32_t max_tiles(natray_net* n) { return n->max_tiles; }
}  // namespace net
}  // namespace natray

extern "C" {

const char* natray_net_last_error(void) { return g_net_err.c_str(); }

int natray_net_create(uint32_t max_tiles, uint64_t seed, natray_net** out) {
  if (!out || max_tiles == 0 || max_tiles > (1u << 16)) return nfail(NATRAY_E_ARG, "max_tiles must be 1..65536");
  natray_net* n = new natray_net();
  n->max_tiles = max_tiles;
  auto bail = [&](int code) {
    for (void* q : n->allocs) (void)hipFree(q);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
    return code;
  };
  const size_t vox = (size_t)max_tiles * VOX;
  int e = 0;
  if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) return bail(nfail(NATRAY_E_HIP, "stream"));
  if ((e = nalloc(n, &n->p, NATRAY_NET_PARAMS)) || (e = nalloc(n, &n->g, NATRAY_NET_PARAMS)) ||
      (e = nalloc(n, &n->m, NATRAY_NET_PARAMS)) || (e = nalloc(n, &n->v, NATRAY_NET_PARAMS)) ||
      (e = nalloc(n, &n->in, vox * 8)) || (e = nalloc(n, &n->act[0], vox * 16)) || (e = nalloc(n, &n->act[1], vox * 16)) ||
      (e = nalloc(n, &n->act[2], vox * 16)) || (e = nalloc(n, &n->out, vox)) || (e = nalloc(n, &n->dz[0], vox * 16)) ||
      (e = nalloc(n, &n->dz[1], vox * 16)) || (e = nalloc(n, &n->part, part_off(4))) || (e = nalloc(n, &n->lpart, LOSS_PARTS)) || (e = nalloc(n, &n->target, vox)) || (e = nalloc(n, &n->mask, vox)) ||
      (e = nalloc(n, &n->stage, vox * 2)) || (e = nalloc(n, &n->loss, 1)) || (e = nalloc(n, &n->resid, vox)))
    return bail(e);
  for (int l = 0; l < 4; ++l) {
    if ((e = nalloc(n, &n->wb[l], (size_t)ksteps(LAYERS[l].cin) * 64))) return bail(e);
    if (l > 0 && (e = nalloc(n, &n->wt[l], (size_t)ksteps(16) * 64))) return bail(e);
  }
  // He-uniform weights (bound sqrt(6 / fan_in)) from a splitmix64 stream; the last layer is
  // scaled by 0.1 so an untrained net predicts corrections near zero. Biases start at zero.
  std::vector<float> h(NATRAY_NET_PARAMS, 0.0f);
  uint64_t s = seed;
  auto next = [&]() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  for (int l = 0; l < 4; ++l) {
    const Layer& L = LAYERS[l];
    const double bound = std::sqrt(6.0 / (TAPS * L.cin_real)) * (l == 3 ? 0.1 : 1.0);
    for (size_t i = 0; i < (size_t)TAPS * L.cin_real * L.cout_real; ++i) h[L.w_off + i] = (float)((2.0 * next() - 1.0) * bound);
  }
  if (hipMemcpy(n->p, h.data(), h.size() * 4, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(n->m, 0, NATRAY_NET_PARAMS * 4) != hipSuccess || hipMemset(n->v, 0, NATRAY_NET_PARAMS * 4) != hipSuccess ||
      hipMemset(n->in, 0, vox * 8 * sizeof(__bf16)) != hipSuccess)
    return bail(nfail(NATRAY_E_HIP, "initialising the network"));
  *out = n;
  return NATRAY_OK;
}

void natray_net_destroy(natray_net* n) {
  if (!n) return;
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  for (void* q : n->allocs) (void)hipFree(q);
  if (n->stream) (void)hipStreamDestroy(n->stream);
  delete n;
}

int natray_net_params(natray_net* n, float* out) {
  if (!n || !out) return nfail(NATRAY_E_ARG, "null argument");
  NCHK(hipStreamSynchronize(n->stream));
  NCHK(hipMemcpy(out, n->p, NATRAY_NET_PARAMS * 4, hipMemcpyDeviceToHost));
  return NATRAY_OK;
}

int natray_net_set_params(natray_net* n, const float* in) {
  if (!n || !in) return nfail(NATRAY_E_ARG, "null argument");
  NCHK(hipStreamSynchronize(n->stream));
  NCHK(hipMemcpy(n->p, in, NATRAY_NET_PARAMS * 4, hipMemcpyHostToDevice));
  n->packed = false;
  return NATRAY_OK;
}

int natray_net_grads(natray_net* n, float* out) {
  if (!n || !out) return nfail(NATRAY_E_ARG, "null argument");
  NCHK(hipStreamSynchronize(n->stream));
  NCHK(hipMemcpy(out, n->g, NATRAY_NET_PARAMS * 4, hipMemcpyDeviceToHost));
  return NATRAY_OK;
}

int natray_net_forward(natray_net* n, const float* input, uint32_t tiles, float* output) {
  if (!n || !input || !output) return nfail(NATRAY_E_ARG, "null argument");
  if (tiles == 0 || tiles > n->max_tiles) return nfail(NATRAY_E_ARG, "tiles must be 1..max_tiles");
  int e = upload_input(n, input, tiles);
  if (e) return e;
  if ((e = forward(n, tiles))) return e;
  const size_t vox = (size_t)tiles * VOX;
  NCHK(hipMemcpyAsync(output, n->out, vox * 4, hipMemcpyDeviceToHost, n->stream));
  NCHK(hipStreamSynchronize(n->stream));
  return NATRAY_OK;
}

int natray_net_train_step(natray_net* n, const float* input, const float* target, const float* mask, uint32_t tiles,
                          float lr, float* loss) {
  if (!n || !input || !target || !mask) return nfail(NATRAY_E_ARG, "null argument");
  if (tiles == 0 || tiles > n->max_tiles) return nfail(NATRAY_E_ARG, "tiles must be 1..max_tiles");
  const size_t vox = (size_t)tiles * VOX;
  int e = upload_input(n, input, tiles);
  if (e) return e;
  NCHK(hipMemcpyAsync(n->target, target, vox * 4, hipMemcpyHostToDevice, n->stream));
  NCHK(hipMemcpyAsync(n->mask, mask, vox * 4, hipMemcpyHostToDevice, n->stream));
  if ((e = forward(n, tiles))) return e;
  // The GPU runs the forward pass meanwhile.
  double count = 0.0;
  for (size_t i = 0; i < vox; ++i) count += mask[i];
  if ((e = backward(n, tiles, count > 0.0 ? (float)(1.0 / count) : 0.0f))) return e;
  if (lr > 0.0f) {
    n->steps += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)n->steps), c2 = 1.0f - std::pow(b2, (float)n->steps);
    hipLaunchKernelGGL(k_adam, dim3((NATRAY_NET_PARAMS + 255) / 256), dim3(256), 0, n->stream, n->p, n->g, n->m, n->v,
                       NATRAY_NET_PARAMS, lr, b1, b2, 1e-8f, c1, c2);
    NCHK(hipGetLastError());
    n->packed = false;
  }
  float h = 0.0f;
  NCHK(hipMemcpyAsync(&h, n->loss, 4, hipMemcpyDeviceToHost, n->stream));
  NCHK(hipStreamSynchronize(n->stream));
  if (loss) *loss = h;
  return NATRAY_OK;
}

int natray_net_train_step_residual(natray_net* n, const float* input, const float* diag, const uint32_t* nbm,
                                   uint32_t tiles, float lr, float* loss) {
  if (!n || !input || !diag || !nbm) return nfail(NATRAY_E_ARG, "null argument");
  if (tiles == 0 || tiles > n->max_tiles) return nfail(NATRAY_E_ARG, "tiles must be 1..max_tiles");
  const size_t vox = (size_t)tiles * VOX;
  int e = upload_input(n, input, tiles);
  if (e) return e;
  NCHK(hipMemcpyAsync(n->target, diag, vox * 4, hipMemcpyHostToDevice, n->stream));
  NCHK(hipMemcpyAsync(n->mask, nbm, vox * 4, hipMemcpyHostToDevice, n->stream));
  if ((e = forward(n, tiles))) return e;
  // The GPU runs the forward pass meanwhile.
  size_t count = 0;
  for (size_t i = 0; i < vox; ++i) count += diag[i] > 0.0f ? 1u : 0u;
  if ((e = backward(n, tiles, count ? (float)(1.0 / (double)count) : 0.0f, true))) return e;
  if (lr > 0.0f) {
    n->steps += 1;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - std::pow(b1, (float)n->steps), c2 = 1.0f - std::pow(b2, (float)n->steps);
    hipLaunchKernelGGL(k_adam, dim3((NATRAY_NET_PARAMS + 255) / 256), dim3(256), 0, n->stream, n->p, n->g, n->m, n->v,
                       NATRAY_NET_PARAMS, lr, b1, b2, 1e-8f, c1, c2);
    NCHK(hipGetLastError());
    n->packed = false;
  }
  float h = 0.0f;
  NCHK(hipMemcpyAsync(&h, n->loss, 4, hipMemcpyDeviceToHost, n->stream));
  NCHK(hipStreamSynchronize(n->stream));
  if (loss) *loss = h;
  return NATRAY_OK;
}

int natray_net_layer_check(uint32_t cin_real, uint32_t cout_real, int relu, const float* X, const float* W, const float* b,
                           const float* dY, uint32_t tiles, float* Y, float* dX, float* dW, float* db) {
  if (!X || !W || !b || !dY || !Y || !dX || !dW || !db || tiles == 0 || tiles > 64) return nfail(NATRAY_E_ARG, "bad argument");
  if (!((cin_real == 2 || cin_real == 16) && (cout_real == 16 || cout_real == 1)))
    return nfail(NATRAY_E_ARG, "layer shapes are (2 or 16) -> (16 or 1)");
  const int cin = cin_real == 2 ? 8 : 16;
  const size_t vox = (size_t)tiles * VOX, nw = (size_t)TAPS * cin_real * cout_real;
  std::vector<void*> a;
  auto al = [&](size_t bytes) -> void* {
    void* q = nullptr;
    if (hipMalloc(&q, bytes ? bytes : 16) != hipSuccess) return nullptr;
    a.push_back(q);
    return q;
  };
  auto done = [&](int code) {
    (void)hipDeviceSynchronize();
    for (void* q : a) (void)hipFree(q);
    return code;
  };
  float* dXf = (float*)al(vox * cin_real * 4);
  float* dWd = (float*)al(nw * 4);
  float* dbd = (float*)al(16 * 4);
  float* bd = (float*)al(16 * 4);
  float* stage = (float*)al(vox * 16 * 4);
  __bf16* xb = (__bf16*)al(vox * cin * 2);
  __bf16* yb = (__bf16*)al(vox * 16 * 2);
  float* yf = (float*)al(vox * 16 * 4);
  float* g = (float*)al(vox * 16 * 4);
  __bf16* dz = (__bf16*)al(vox * 16 * 2);
  float* dxf = (float*)al(vox * 16 * 4);
  bf16x8* wb = (bf16x8*)al((size_t)ksteps(cin) * 64 * 16);
  bf16x8* wt = (bf16x8*)al((size_t)ksteps(16) * 64 * 16);
  float* part = (float*)al(part_size(cin) * 4);
  if (a.size() != 14) return done(nfail(NATRAY_E_NOMEM, "hipMalloc"));
  const unsigned grid = grid_for(vox);
  std::vector<float> bb(16, 0.0f);
  for (uint32_t i = 0; i < cout_real; ++i) bb[i] = b[i];
  if (hipMemcpy(dWd, W, nw * 4, hipMemcpyHostToDevice) || hipMemcpy(bd, bb.data(), 64, hipMemcpyHostToDevice) ||
      hipMemcpy(stage, X, vox * cin_real * 4, hipMemcpyHostToDevice))
    return done(nfail(NATRAY_E_HIP, "upload"));
  hipLaunchKernelGGL(k_to_bf16, dim3(grid), dim3(256), 0, 0, stage, (int)cin_real, cin, xb, vox);
  PackJobs pj{};
  pj.job[0] = PackJob{dWd, (int)cin_real, (int)cout_real, cin, 0, wb};
  pj.job[1] = PackJob{dWd, (int)cin_real, (int)cout_real, 16, 1, wt};
  hipLaunchKernelGGL(k_pack, dim3(PACK_MAX, 2), dim3(256), 0, 0, pj);
  launch_conv(cin, tiles, 0, xb, wb, bd, relu, nullptr, yb, yf, nullptr, nullptr);
  // The one-channel output as the network's last layer writes it, or the first channels of 16.
  if (cout_real == 1)
    launch_conv(cin, tiles, 0, xb, wb, bd, relu, nullptr, nullptr, nullptr, stage, nullptr);
  else
    hipLaunchKernelGGL(k_take, dim3(grid), dim3(256), 0, 0, yf, (int)cout_real, stage, vox);
  if (hipMemcpy(Y, stage, vox * cout_real * 4, hipMemcpyDeviceToHost)) return done(nfail(NATRAY_E_HIP, "download Y"));
  // Backward from dY.
  if (hipMemcpy(stage, dY, vox * cout_real * 4, hipMemcpyHostToDevice)) return done(nfail(NATRAY_E_HIP, "upload dY"));
  hipLaunchKernelGGL(k_pad16, dim3(grid), dim3(256), 0, 0, stage, (int)cout_real, g, vox);
  hipLaunchKernelGGL(k_relu_back, dim3(grid_for(vox * 16)), dim3(256), 0, 0, g, yb, relu, dz, vox * 16);
  const uint32_t groups = launch_wgrad(cin, tiles, 0, xb, dz, part);
  FoldJobs fj{};
  fj.job[0] = FoldJob{part, (int)groups, cin == 8 ? WgradShape<8>::PART : WgradShape<16>::PART, cin, (int)cin_real,
                      (int)cout_real, dWd, dbd};
  hipLaunchKernelGGL(k_grad_fold, dim3(FOLD_BLOCKS, 1), dim3(256), 0, 0, fj);
  launch_conv(16, tiles, 0, dz, wt, nullptr, 0, nullptr, nullptr, dxf, nullptr, nullptr);
  hipLaunchKernelGGL(k_take, dim3(grid), dim3(256), 0, 0, dxf, (int)cin_real, dXf, vox);
  if (hipGetLastError() != hipSuccess) return done(nfail(NATRAY_E_HIP, "layer kernels"));
  if (hipMemcpy(dX, dXf, vox * cin_real * 4, hipMemcpyDeviceToHost) || hipMemcpy(dW, dWd, nw * 4, hipMemcpyDeviceToHost) ||
      hipMemcpy(db, dbd, cout_real * 4, hipMemcpyDeviceToHost))
    return done(nfail(NATRAY_E_HIP, "download gradients"));
  return done(NATRAY_OK);
}

}  // extern "C"
