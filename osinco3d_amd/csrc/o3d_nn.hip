// Learned warm start for the Poisson solve: a 3D U-Net-lite on MI355X.
//
// Layout: activations are channels-last [voxel][channel] BF16 (voxel = x +
// nx*(y + ny*z)), so the 8 consecutive channels an MFMA lane needs are one
// 16-byte load.  Gradients of activations are FP32 (accumulated), weight
// gradients and master weights FP32.
//
// 3x3x3 convolutions are implicit GEMMs on v_mfma_f32_16x16x32_bf16:
//   M = 16 consecutive voxels (one wave), N = 16 output channels per tile,
//   K = 27 taps x C_in, flattened as k = tap*C_in + c and zero-padded to a
//   multiple of 32; lane l supplies A[m = l%16][k = 8(l/16)..+7] (one voxel,
//   8 channels of one tap) and B[k][n = l%16] (8 weights of one output
//   channel), and receives C[m = 4(l/16)+i][n = l%16].
// The data gradient is the same kernel with the weights transposed and the
// taps mirrored (periodic padding makes the adjoint of the convolution the
// convolution with the flipped kernel).  The weight gradient is a GEMM on the
// same instruction whose K dimension is the voxels; it reads channel-major
// copies of its operands (runs of 8 voxels along x) and reduces over slabs
// of voxels in a fixed order.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>
#include <string>
#include <vector>

#include "../../include/o3d.h"
#include "../../include/o3d_nn.h"
#include "o3d_common.h"
#include "o3d_nn.h"
#include "o3d_sor.h"

namespace o3d {
namespace nn {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kSlope = 0.1f;  // leaky-ReLU slope

__device__ __forceinline__ int wrapi(int q, int n) { return q < 0 ? q + n : (q >= n ? q - n : q); }
__device__ __forceinline__ float act_f(float v) { return v > 0.f ? v : kSlope * v; }
__device__ __forceinline__ float dact(float y) { return y > 0.f ? 1.f : kSlope; }

// ----------------------------------------------------------------- convolution
template <typename TO>
struct ConvArgs {
  const bf16 *x;      // [V][ci]
  const bf16 *w;      // [co][kp]  k = tap*ci + c, zero padded
  const float *bias;  // [co] or null
  const bf16 *skip;   // [V][co] or null, added before the activation
  TO *y;              // [V][co]
  int nx, ny, nz;
  int lci, ci, co, kp;
  int act;            // 1: leaky ReLU
};

// One wave computes 16*MV consecutive voxels (linear order, so coarse levels
// with nx < 16 work too) for 16*NT output channels: MV x NT MFMA tiles share
// each loaded A fragment across NT output tiles and each B fragment across MV
// voxel tiles.
template <typename TO, int NT, int MV>
__global__ void __launch_bounds__(256) conv_kernel(const ConvArgs<TO> a) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int V = a.nx * a.ny * a.nz;
  const int vbase = (blockIdx.x * 4 + wv) * 16 * MV;
  if (vbase >= V) return;  // no barriers in this kernel
  const int co0 = blockIdx.y * 16 * NT;
  const int g = lane >> 4, l16 = lane & 15;
  f32x4 acc[MV][NT];
#pragma unroll
  for (int m = 0; m < MV; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ktot = 27 * a.ci;
  const int nchunk = a.kp >> 5;
  // A-operand voxels of this lane, one per voxel tile.
  int xm[MV], ym[MV], zm[MV];
  bool vin[MV];
#pragma unroll
  for (int m = 0; m < MV; ++m) {
    const int vm = vbase + 16 * m + l16;
    vin[m] = vm < V;
    xm[m] = vm % a.nx;
    ym[m] = (vm / a.nx) % a.ny;
    zm[m] = vm / (a.nx * a.ny);
  }
  const bf16 *wrow[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wrow[n] = a.w + (size_t)(co0 + 16 * n + l16) * a.kp;
  for (int kc = 0; kc < nchunk; ++kc) {
    const int k0 = (kc << 5) + (g << 3);
    bf16x8 bv[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) bv[n] = *(const bf16x8 *)(wrow[n] + k0);
    const bool kin = k0 < ktot;
    const int t = k0 >> a.lci;
    const int c0 = k0 & (a.ci - 1);
    const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
#pragma unroll
    for (int m = 0; m < MV; ++m) {
      bf16x8 av;
      if (kin && vin[m]) {
        const int vx = wrapi(xm[m] + dx, a.nx), vy = wrapi(ym[m] + dy, a.ny),
                  vz = wrapi(zm[m] + dz, a.nz);
        av = *(const bf16x8 *)(a.x + (size_t)(vx + a.nx * (vy + a.ny * vz)) * a.ci + c0);
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) av[q] = (bf16)0.f;
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
        acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[n], acc[m][n], 0, 0, 0);
    }
  }
#pragma unroll
  for (int m = 0; m < MV; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int c = co0 + 16 * n + l16;
      const float b = a.bias ? a.bias[c] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vox = vbase + 16 * m + 4 * g + i;
        if (vox >= V) continue;
        const size_t o = (size_t)vox * a.co + c;
        float v = acc[m][n][i] + b;
        if (a.skip) v += (float)a.skip[o];
        if (a.act) v = act_f(v);
        a.y[o] = (TO)v;
      }
    }
}

// The same implicit GEMM for the coarse grids, whose few voxel tiles would
// leave most of the machine idle: a block of KW waves owns one tile of 16
// consecutive voxels and 16*NT output channels and splits the K chunks among
// its waves (wave w takes chunks w, w + KW, ...); the waves' FP32
// accumulators are added in LDS, in wave order, and the block's threads
// apply bias, skip and activation to the sums.
template <typename TO, int NT, int KW>
__global__ void __launch_bounds__(64 * KW) conv_kw_kernel(const ConvArgs<TO> a) {
  __shared__ float red[KW][NT][4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int V = a.nx * a.ny * a.nz;
  const int vbase = blockIdx.x * 16;
  const int co0 = blockIdx.y * 16 * NT;
  const int g = lane >> 4, l16 = lane & 15;
  f32x4 acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int ktot = 27 * a.ci;
  const int nchunk = a.kp >> 5;
  const int vm = vbase + l16;
  const bool vin = vm < V;
  const int xm = vm % a.nx, ym = (vm / a.nx) % a.ny, zm = vm / (a.nx * a.ny);
  const bf16 *wrow[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) wrow[n] = a.w + (size_t)(co0 + 16 * n + l16) * a.kp;
  for (int kc = wv; kc < nchunk; kc += KW) {
    const int k0 = (kc << 5) + (g << 3);
    bf16x8 bv[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) bv[n] = *(const bf16x8 *)(wrow[n] + k0);
    const int t = k0 >> a.lci;
    const int c0 = k0 & (a.ci - 1);
    bf16x8 av;
    if (k0 < ktot && vin) {
      const int vx = wrapi(xm + t % 3 - 1, a.nx), vy = wrapi(ym + (t / 3) % 3 - 1, a.ny),
                vz = wrapi(zm + t / 9 - 1, a.nz);
      av = *(const bf16x8 *)(a.x + (size_t)(vx + a.nx * (vy + a.ny * vz)) * a.ci + c0);
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) av[q] = (bf16)0.f;
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
      acc[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv[n], acc[n], 0, 0, 0);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wv][n][i][lane] = acc[n][i];
  __syncthreads();
  for (int e = threadIdx.x; e < NT * 4 * 64; e += 64 * KW) {
    const int n = e >> 8, i = (e >> 6) & 3, ln = e & 63;
    const int vox = vbase + 4 * (ln >> 4) + i;
    if (vox >= V) continue;
    float v = red[0][n][i][ln];
#pragma unroll
    for (int w = 1; w < KW; ++w) v += red[w][n][i][ln];
    const int c = co0 + 16 * n + (ln & 15);
    const size_t o = (size_t)vox * a.co + c;
    if (a.bias) v += a.bias[c];
    if (a.skip) v += (float)a.skip[o];
    if (a.act) v = act_f(v);
    a.y[o] = (TO)v;
  }
}

// The same implicit GEMM with its operands staged through LDS, for the fine
// levels.  A block owns a brick of 16 (x) x TY (y) x 4 (z) voxels and all
// 16*NT output channels of its blockIdx.y group; wave w computes the z plane
// w of the brick, TY voxel tiles of 16 (one per x row).
//  * Input: the brick and its one-voxel periodic halo (18 x (TY+2) x 6
//    voxels, every input channel) are loaded once, coalesced, as [channel
//    group of 8][voxel] 16-byte entries, so the 16 lanes that supply one
//    MFMA A fragment (16 consecutive x voxels, 8 channels of one tap) read
//    256 contiguous bytes: one pass over the 64 banks.  Each input value is
//    read once from L2 instead of once per tap.  With UP the input is the
//    grid of half the size, upsampled 2x (nearest) as it is staged, which is
//    the decoder's up-sampling fused into the convolution that consumes it.
//  * Weights: slices of SK K-chunks of the block's 16*NT rows (as many as
//    fit in 48 KB of LDS next to the input tile, at least 8: one slice for
//    16 input channels), loaded cooperatively; the first slice's loads are
//    issued with the input tile's, before one barrier.  Rows are padded by
//    16 bytes so the 16 lanes reading one B fragment (16 rows, same k) hit
//    distinct banks.  The K loop then waits on LDS only, not on a global
//    load per chunk.
// Needs nx % 16 == 0, ny % TY == 0, nz % 4 == 0 and ci == CI (UP: even
// dimensions, x of (nx/2, ny/2, nz/2) voxels).
template <typename TO, int NT, int TY, int CI, bool UP>
__global__ void __launch_bounds__(256) conv_lds_kernel(const ConvArgs<TO> a) {
  constexpr int HX = 18, HY = TY + 2, HZ = 6, NV = HX * HY * HZ, NG = CI / 8;
  // K chunks per weight slice: as many as fit in 48 KB of LDS with the
  // input tile (three blocks per CU), at least 8, at most all of them.
  constexpr int KCH = (27 * CI + 31) / 32;
  constexpr int SKF = ((48 * 1024 - NG * NV * 16) / (NT * 16 * 16) - 1) / 4;
  constexpr int SK = (SKF > 8 ? SKF : 8) < KCH ? (SKF > 8 ? SKF : 8) : KCH;
  static_assert(SK >= 1, "no room for a weight slice");
  constexpr int WROW = SK * 4 + 1;   // 16-byte entries per padded weight row
  __shared__ bf16x8 tile[NG * NV];
  __shared__ bf16x8 wts[NT * 16 * WROW];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int ntx = a.nx >> 4, nty = a.ny / TY;
  const int bx = (int)blockIdx.x % ntx, byz = (int)blockIdx.x / ntx;
  const int x0 = bx * 16, y0 = (byz % nty) * TY, z0 = (byz / nty) * 4;
  const int sx = UP ? a.nx >> 1 : a.nx, sy = UP ? a.ny >> 1 : a.ny;
  for (int e = threadIdx.x; e < NG * NV; e += 256) {
    const int cg = e / NV, v = e - cg * NV;
    const int hx = v % HX, hy = (v / HX) % HY, hz = v / (HX * HY);
    int gx = wrapi(x0 + hx - 1, a.nx), gy = wrapi(y0 + hy - 1, a.ny),
        gz = wrapi(z0 + hz - 1, a.nz);
    if (UP) {
      gx >>= 1;
      gy >>= 1;
      gz >>= 1;
    }
    tile[e] = *(const bf16x8 *)(a.x + (size_t)(gx + sx * (gy + (size_t)sy * gz)) * CI + cg * 8);
  }
  const int co0 = blockIdx.y * 16 * NT;
  f32x4 acc[TY][NT];
#pragma unroll
  for (int m = 0; m < TY; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int ktot = 27 * CI;
  const int nchunk = a.kp >> 5;
  for (int s0 = 0; s0 < nchunk; s0 += SK) {
    if (s0 > 0) __syncthreads();  // every wave is done with the previous slice
    for (int v = threadIdx.x; v < NT * 16 * SK * 4; v += 256) {
      const int row = v / (SK * 4), c8 = v - row * (SK * 4);
      const int k = s0 * 32 + c8 * 8;
      bf16x8 w8;
      if (k < a.kp) {
        w8 = *(const bf16x8 *)(a.w + (size_t)(co0 + row) * a.kp + k);
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) w8[q] = (bf16)0.f;
      }
      wts[row * WROW + c8] = w8;
    }
    __syncthreads();  // the slice (and, the first time, the input tile) is in LDS
    const int ce = min(SK, nchunk - s0);
    for (int c = 0; c < ce; ++c) {
      const int k0 = ((s0 + c) << 5) + (g << 3);
      bf16x8 bv[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) bv[n] = wts[(16 * n + l16) * WROW + c * 4 + g];
      bf16x8 av[TY];
      if (k0 < ktot) {
        const int t = k0 / CI, cg = (k0 % CI) >> 3;
        const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = t / 9 - 1;
        const int base = cg * NV + (l16 + 1 + dx) + HX * ((1 + dy) + HY * (wv + 1 + dz));
#pragma unroll
        for (int m = 0; m < TY; ++m) av[m] = tile[base + HX * m];
      } else {
#pragma unroll
        for (int m = 0; m < TY; ++m)
#pragma unroll
          for (int q = 0; q < 8; ++q) av[m][q] = (bf16)0.f;
      }
#pragma unroll
      for (int m = 0; m < TY; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[m], bv[n], acc[m][n], 0, 0, 0);
    }
  }
  // Epilogue through LDS, one 16-channel output tile at a time: each wave
  // writes its accumulators as [row m][voxel][channel] floats over the input
  // tile (no longer read), then every lane forms 8 consecutive channels of
  // one voxel, so the skip is read and the result written as 16-byte
  // vectors instead of one 2- or 4-byte access per value.  Same operations
  // per value, in the same order, as a per-value epilogue.
  const int z = z0 + wv;
  static_assert(TY * 16 * 16 * 4 * 4 <= NG * NV * 16, "epilogue does not fit the tile");
  float *ob = reinterpret_cast<float *>(tile) + wv * (TY * 16 * 16);
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    __syncthreads();  // the tile (first pass) or the previous pass is done with
#pragma unroll
    for (int m = 0; m < TY; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) ob[(m * 16 + 4 * g + i) * 16 + l16] = acc[m][n][i];
    __syncthreads();
    for (int t = lane; t < TY * 16 * 2; t += 64) {
      const int m = t >> 5, v16 = (t >> 1) & 15, c8 = t & 1;
      const int c = co0 + 16 * n + 8 * c8;
      const int vox = x0 + v16 + a.nx * (y0 + m + a.ny * z);
      const size_t o = (size_t)vox * a.co + c;
      const float *src = ob + (m * 16 + v16) * 16 + 8 * c8;
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = src[q] + (a.bias ? a.bias[c + q] : 0.f);
      if (a.skip) {
        const bf16x8 sk = *(const bf16x8 *)(a.skip + o);
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] += (float)sk[q];
      }
      if (a.act) {
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = act_f(v[q]);
      }
      if constexpr (std::is_same<TO, float>::value) {
        f32x4 *yo = (f32x4 *)(a.y + o);
        yo[0] = f32x4{v[0], v[1], v[2], v[3]};
        yo[1] = f32x4{v[4], v[5], v[6], v[7]};
      } else {
        bf16x8 w;
#pragma unroll
        for (int q = 0; q < 8; ++q) w[q] = (bf16)v[q];
        *(bf16x8 *)(a.y + o) = w;
      }
    }
  }
}

// LDS bricks of a grid (TY rows per brick) and whether the grid tiles.
inline long long lds_bricks(int nx, int ny, int nz, int ty) {
  if (nx % 16 || ny % ty || nz % 4) return 0;
  return (long long)(nx / 16) * (ny / ty) * (nz / 4);
}

// Shape of the LDS-staged kernel for a convolution: rows per brick (4 while
// that leaves >= 512 blocks, else 1 while >= 256) and output tiles per block
// (the natural 16*NT channels, at most 2 tiles for LDS); ty = 0 when it does
// not apply (64 input channels: one-row bricks only; 128: never; coarser
// grids split the K chunks among the waves of a block, conv_kw_kernel,
// which measured faster there: the 64^3 network's forward pass took 0.246 ms
// with its 16^3 layers staged through LDS one output tile per block, 0.228
// ms with them on conv_kw_kernel).
struct LdsPlan {
  int ty = 0, nt = 0;
};
inline LdsPlan lds_plan(int nx, int ny, int nz, int ci, int co) {
  LdsPlan p;
  if (ci != 16 && ci != 32 && ci != 64) return p;
  const int nat = std::min(2, co >= 64 ? 4 : (co >= 32 ? 2 : 1));
  const long long b4 = ci <= 32 ? lds_bricks(nx, ny, nz, 4) : 0;
  const long long b1 = lds_bricks(nx, ny, nz, 1);
  if (b4 * (co / (16 * nat)) >= 512) {
    p.ty = 4;
    p.nt = nat;
  } else if (b1 * (co / (16 * nat)) >= 256) {
    p.ty = 1;
    p.nt = nat;
  }
  return p;
}

template <typename TO, int NT, int CI, bool UP>
void launch_conv_lds(const ConvArgs<TO> &a, int ty, hipStream_t s) {
  const int gy = a.co / (16 * NT);
  if constexpr (CI <= 32) {
    if (ty == 4) {
      conv_lds_kernel<TO, NT, 4, CI, UP>
          <<<dim3((unsigned)lds_bricks(a.nx, a.ny, a.nz, 4), gy), 256, 0, s>>>(a);
      return;
    }
  }
  conv_lds_kernel<TO, NT, 1, CI, UP>
      <<<dim3((unsigned)lds_bricks(a.nx, a.ny, a.nz, 1), gy), 256, 0, s>>>(a);
}

template <typename TO, bool UP>
void launch_conv_lds_any(const ConvArgs<TO> &a, LdsPlan p, hipStream_t s) {
  if (a.ci == 16 && p.nt == 1) launch_conv_lds<TO, 1, 16, UP>(a, p.ty, s);
  else if (a.ci == 16) launch_conv_lds<TO, 2, 16, UP>(a, p.ty, s);
  else if (a.ci == 32 && p.nt == 1) launch_conv_lds<TO, 1, 32, UP>(a, p.ty, s);
  else if (a.ci == 32) launch_conv_lds<TO, 2, 32, UP>(a, p.ty, s);
  else if (p.nt == 1) launch_conv_lds<TO, 1, 64, UP>(a, p.ty, s);
  else launch_conv_lds<TO, 2, 64, UP>(a, p.ty, s);
}

// Blocks a convolution launches with one 16-voxel tile per wave.
inline int conv_blocks(int V, int co) {
  const int nt = co >= 64 ? 4 : (co >= 32 ? 2 : 1);
  return ((V + 63) / 64) * (co / (16 * nt));
}

// Waves per block of the coarse-grid kernel.
constexpr int kConvKW = 8;

template <typename TO, int NT>
hipError_t launch_conv_nt(const ConvArgs<TO> &a, int V, hipStream_t s) {
  // Four voxel tiles per wave (four independent gathers per K chunk) once
  // the grid still has >= 1024 blocks (4096 waves); one tile per wave while
  // it has >= 1024 blocks that way; on coarser grids, the K chunks split
  // among the waves of a block.
  constexpr int kMV = 4;
  const int gy = a.co / (16 * NT);
  if ((long long)((V + 64 * kMV - 1) / (64 * kMV)) * gy >= 1024) {
    dim3 grid((V + 64 * kMV - 1) / (64 * kMV), gy);
    conv_kernel<TO, NT, kMV><<<grid, 256, 0, s>>>(a);
  } else if (conv_blocks(V, a.co) >= 1024) {
    dim3 grid((V + 63) / 64, gy);
    conv_kernel<TO, NT, 1><<<grid, 256, 0, s>>>(a);
  } else {
    dim3 grid((V + 15) / 16, gy);
    conv_kw_kernel<TO, NT, kConvKW><<<grid, 64 * kConvKW, 0, s>>>(a);
  }
  return hipGetLastError();
}

template <typename TO>
hipError_t launch_conv(const ConvArgs<TO> &a, hipStream_t s) {
  const int V = a.nx * a.ny * a.nz;
  const int nt = a.co >= 64 ? 4 : (a.co >= 32 ? 2 : 1);
  // Fine levels (16, 32 or 64 input channels, enough blocks): the LDS-staged
  // kernel.
  const LdsPlan lp = lds_plan(a.nx, a.ny, a.nz, a.ci, a.co);
  if (lp.ty) {
    launch_conv_lds_any<TO, false>(a, lp, s);
    return hipGetLastError();
  }
  if (nt == 4) return launch_conv_nt<TO, 4>(a, V, s);
  if (nt == 2) return launch_conv_nt<TO, 2>(a, V, s);
  return launch_conv_nt<TO, 1>(a, V, s);
}

// Weight gradient: dW[co][tap*ci + c] = sum_v dz[v][co] * x[v + off(tap)][c],
// a GEMM with M = co, N = 27 ci and the voxels as K.  An MFMA lane supplies 8
// consecutive K values of one row or column, which channels-last storage
// keeps a channel vector apart, so both operands are first copied
// channel-major, a row of nx voxels as nr = ceil(nx / 8) runs of 8:
//   dzt[co][row][nr * 8]        zero past nx (those K values add nothing)
//   xt[ci][row][(nr + 2) * 8]   one run before and after the row, holding the
//                               periodic neighbours x = -1 and x = nx (else 0)
// The 27 taps of a run then are 9 rows (dy, dz) of xt, each read once as the
// aligned 16-byte run and the two 4-byte words beside it; the three x shifts
// are register funnel shifts of those.
struct Runs {
  int nx, ny, nz, nr;
  int rows() const { return ny * nz; }
  size_t dz_plane() const { return (size_t)ny * nz * nr * 8; }
  size_t x_plane() const { return (size_t)ny * nz * (nr + 2) * 8; }
};

// The 8x8 transpose of one run: v[e][c] (voxel e, channel c) to channel c's
// run of 8 voxels.
__device__ __forceinline__ bf16x8 run_of(const bf16x8 *v, int c) {
  bf16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = v[e][c];
  return o;
}

// The copy of x, 256 threads of which this is number idx.
__device__ __forceinline__ void x_runs(const bf16 *__restrict__ x, bf16 *__restrict__ xt,
                                       const Runs &R, int C, int idx) {
  const int G = C >> 3, nh = R.nr + 2;
  if (idx >= R.ny * R.nz * nh * G) return;
  const int cg = idx % G, q = idx / G;
  const int r = q % nh, row = q / nh;
  bf16x8 v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int i = 8 * (r - 1) + e;
    if (i >= -1 && i <= R.nx) {
      v[e] = *(const bf16x8 *)(x + ((size_t)row * R.nx + wrapi(i, R.nx)) * C + 8 * cg);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) v[e][c] = (bf16)0.f;
    }
  }
  const size_t plane = (size_t)R.ny * R.nz * nh * 8;
  bf16 *o = xt + (size_t)8 * cg * plane + ((size_t)row * nh + r) * 8;
#pragma unroll
  for (int c = 0; c < 8; ++c) *(bf16x8 *)(o + c * plane) = run_of(v, c);
}

// A block of 4 waves owns one 16-channel tile of ci and WC of co (wave w:
// co tile w % WC) and the K chunks (4 runs, 32 voxels) of slab blockIdx.y;
// the 4 / WC waves of a co tile take every (4 / WC)-th chunk and their
// accumulators (27 taps x 4 registers) are added in LDS in wave order.  The
// operands come straight from L1/L2: a chunk is 28 loads of up to 16 bytes
// per lane for 27 MFMAs; their latency at two waves per SIMD bounds it.
// Against the previous kernel (one thread per weight, a scalar product per
// voxel) the 14 layers of a 128x96x64 network take 0.76 ms instead of 64.9 ms,
// those of a 32^3 network 0.16 ms instead of 6.7 ms.
template <int WC>
__global__ void __launch_bounds__(256) wgrad_kernel(const bf16 *__restrict__ dzt,
                                                    const bf16 *__restrict__ xt,
                                                    float *__restrict__ part, Runs R, int ci,
                                                    int co, int per) {
  constexpr int WK = 4 / WC;
  __shared__ f32x4 red[WK > 1 ? 27 * 64 : 1];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int nct = ci >> 4;
  const int c0 = (blockIdx.x % nct) * 16;
  const int o0 = ((blockIdx.x / nct) * WC + wv % WC) * 16;
  const int nh = R.nr + 2, nruns = R.ny * R.nz * R.nr;
  const size_t zp = (size_t)R.ny * R.nz * R.nr * 8, xp = (size_t)R.ny * R.nz * nh * 8;
  const bf16 *A = dzt + (size_t)(o0 + l16) * zp;
  const bf16 *B = xt + (size_t)(c0 + l16) * xp;
  const int nchunk = (nruns + 3) >> 2;
  const int k0 = blockIdx.y * per, k1 = min(nchunk, k0 + per);
  f32x4 acc[27];
#pragma unroll
  for (int t = 0; t < 27; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  for (int k = k0 + wv / WC; k < k1; k += WK) {
    const int q = 4 * k + g;
    bf16x8 av;
#pragma unroll
    for (int e = 0; e < 8; ++e) av[e] = (bf16)0.f;
    if (q < nruns) av = *(const bf16x8 *)(A + (size_t)q * 8);
    const int qq = min(q, nruns - 1);
    const int row = qq / R.nr, r = qq - row * R.nr;
    const int z = row / R.ny, y = row - z * R.ny;
    u32x4 d[9];
    unsigned lo[9], hi[9];
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      const int yy = wrapi(y + s % 3 - 1, R.ny), zz = wrapi(z + s / 3 - 1, R.nz);
      const bf16 *b = B + ((size_t)(zz * R.ny + yy) * nh + r + 1) * 8;
      d[s] = *(const u32x4 *)b;
      lo[s] = *(const unsigned *)(b - 2);
      hi[s] = *(const unsigned *)(b + 8);
    }
#pragma unroll
    for (int s = 0; s < 9; ++s) {
      // Elements -1..6 (dx = -1) and 1..8 (dx = 1) of the run 0..7.
      const unsigned m0 = __builtin_amdgcn_alignbit(d[s][0], lo[s], 16);
      const unsigned m1 = __builtin_amdgcn_alignbit(d[s][1], d[s][0], 16);
      const unsigned m2 = __builtin_amdgcn_alignbit(d[s][2], d[s][1], 16);
      const unsigned m3 = __builtin_amdgcn_alignbit(d[s][3], d[s][2], 16);
      const unsigned m4 = __builtin_amdgcn_alignbit(hi[s], d[s][3], 16);
      const bf16x8 bm = __builtin_bit_cast(bf16x8, u32x4{m0, m1, m2, m3});
      const bf16x8 bz = __builtin_bit_cast(bf16x8, d[s]);
      const bf16x8 bp = __builtin_bit_cast(bf16x8, u32x4{m1, m2, m3, m4});
      acc[3 * s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bm, acc[3 * s], 0, 0, 0);
      acc[3 * s + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bz, acc[3 * s + 1], 0, 0, 0);
      acc[3 * s + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bp, acc[3 * s + 2], 0, 0, 0);
    }
  }
  if constexpr (WK > 1) {
#pragma unroll 1
    for (int w = 1; w < WK; ++w) {
      for (int c = 0; c < WC; ++c) {
        __syncthreads();
        if (wv == w * WC + c) {
#pragma unroll
          for (int t = 0; t < 27; ++t) red[t * 64 + lane] = acc[t];
        }
        __syncthreads();
        if (wv == c) {
#pragma unroll
          for (int t = 0; t < 27; ++t) acc[t] += red[t * 64 + lane];
        }
      }
    }
  }
  if (wv >= WC) return;
  // acc[t][i] = dW[o0 + 4g + i][t][c0 + l16]
  float *out = part + (size_t)blockIdx.y * co * 27 * ci;
#pragma unroll
  for (int t = 0; t < 27; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[((size_t)(o0 + 4 * g + i) * 27 + t) * ci + c0 + l16] = acc[t][i];
}

// Waves of a weight gradient block across the co tiles, and its slabs: about
// 768 blocks (three per CU; two are resident at 230 registers), at least two chunks
// per wave, and at most 16 MB of partial sums (a slab of the 128 x 128 layer
// alone is 1.8 MB).
struct WgradPlan {
  int wc, tiles, slabs, per;
};
inline WgradPlan wgrad_plan(const Runs &R, int ci, int co) {
  WgradPlan p;
  p.wc = co >= 64 ? 4 : (co >= 32 ? 2 : 1);
  p.tiles = (ci / 16) * (co / (16 * p.wc));
  const int chunks = (R.rows() * R.nr + 3) / 4;
  const int entries = co * 27 * ci;
  int slabs = std::min((768 + p.tiles - 1) / p.tiles, (4 << 20) / entries);
  slabs = std::max(1, std::min(slabs, chunks / (2 * (4 / p.wc))));
  p.per = (chunks + slabs - 1) / slabs;
  p.slabs = (chunks + p.per - 1) / p.per;
  return p;
}

// dst[e] += sum_s part[s][e] of every weight, bias and head gradient in one launch:
// 64 entries per block, the slabs dealt to its 4 waves, the waves' sums added in wave
// order.  (A launch per set was 29 of them, 2.8 us each for a 32^3 network.)
struct ReduceSet {
  const float *part;
  float *dst;
  int nparts, entries, block0;  // first block of the set
};
constexpr int kReduceSets = 29;
struct ReduceSets {
  ReduceSet s[kReduceSets];
  int n, blocks;
};
__global__ void __launch_bounds__(256) reduce_parts_kernel(const ReduceSets a) {
  __shared__ float sw[4][64];
  int m = 0;
  while (m + 1 < a.n && (int)blockIdx.x >= a.s[m + 1].block0) ++m;
  const ReduceSet &t = a.s[m];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int e = ((int)blockIdx.x - t.block0) * 64 + lane;
  const int entries = t.entries, nparts = t.nparts;
  const float *part = t.part;
  float s = 0.f;
  if (e < entries) {
#pragma unroll 8
    for (int p = wv; p < nparts; p += 4) s += part[(size_t)p * entries + e];
  }
  sw[wv][lane] = s;
  __syncthreads();
  if (wv == 0 && e < entries)
    t.dst[e] += ((sw[0][lane] + sw[1][lane]) + sw[2][lane]) + sw[3][lane];
}

// ------------------------------------------------------- elementwise pieces
// x[v] = (in[0][v], in[1][v], 0, ..., 0), C a multiple of 8 (16-byte stores).
__global__ void pack_input_kernel(const float *__restrict__ in, bf16 *__restrict__ x, int V,
                                  int C) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  bf16x8 *row = (bf16x8 *)(x + (size_t)v * C);
  bf16x8 z;
#pragma unroll
  for (int q = 0; q < 8; ++q) z[q] = (bf16)0.f;
  bf16x8 h = z;
  h[0] = (bf16)in[v];
  h[1] = (bf16)in[V + v];
  row[0] = h;
  for (int g = 1; g < C / 8; ++g) row[g] = z;
}

// The first convolution in the forward pass: only 2 of its 16 (padded)
// input channels are non-zero, so its K is made dense: k = 2*tap + channel
// over the 54 real pairs, zero-padded to 64 (two MFMA K-chunks instead of
// the padded layout's 14).  A wave computes kFirstTiles tiles of 16
// consecutive voxels x 16 output channels (the block's weight staging
// serves 64 * kFirstTiles voxels); lane (l16, g) gathers, per chunk, the
// two channels of taps 16*chunk + 4g .. +3 of voxel l16 straight from the
// network's FP32 input planes (the 16 lanes of a tap read 16 consecutive
// floats), rounded to BF16 as the packed input holds them.  The dense
// weights are staged in LDS from the padded layout (rows padded by 16
// bytes: the 16 lanes of a B fragment hit distinct banks); bias and leaky
// ReLU follow.
constexpr int kFirstTiles = 4;
__global__ void __launch_bounds__(256) conv_first_kernel(const float *__restrict__ in,
                                                         const bf16 *__restrict__ w,
                                                         const float *__restrict__ bias,
                                                         bf16 *__restrict__ y, int nx, int ny,
                                                         int nz, int kp) {
  __shared__ bf16 wd[16][64 + 8];
  for (int e = threadIdx.x; e < 16 * 64; e += blockDim.x) {
    const int co = e >> 6, k = e & 63;
    wd[co][k] = k < 54 ? w[(size_t)co * kp + (k >> 1) * 16 + (k & 1)] : (bf16)0.f;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int g = lane >> 4, l16 = lane & 15;
  const int V = nx * ny * nz;
  const float b = bias[l16];
  for (int tt = 0; tt < kFirstTiles; ++tt) {
    const int vbase = ((blockIdx.x * 4 + wv) * kFirstTiles + tt) * 16;
    if (vbase >= V) return;  // after the kernel's only barrier
    const int vm = vbase + l16;
    const bool vin = vm < V;
    const int i = vm % nx, j = (vm / nx) % ny, k = vm / (nx * ny);
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      bf16x8 av;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int t = 16 * kc + 4 * g + q;
        bf16x2 pr;
        pr[0] = pr[1] = (bf16)0.f;
        if (t < 27 && vin) {
          const int vx = wrapi(i + t % 3 - 1, nx), vy = wrapi(j + (t / 3) % 3 - 1, ny),
                    vz = wrapi(k + t / 9 - 1, nz);
          const size_t u = (size_t)vx + (size_t)nx * (vy + (size_t)ny * vz);
          pr[0] = (bf16)in[u];
          pr[1] = (bf16)in[(size_t)V + u];
        }
        av[2 * q] = pr[0];
        av[2 * q + 1] = pr[1];
      }
      const bf16x8 bv = *(const bf16x8 *)&wd[l16][32 * kc + 8 * g];
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, acc, 0, 0, 0);
    }
    // acc[q] = C[voxel vbase + 4g + q][channel l16]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int vox = vbase + 4 * g + q;
      if (vox < V) y[(size_t)vox * 16 + l16] = (bf16)act_f(acc[q] + b);
    }
  }
}

// 2x average pooling onto the grid (nx/2, ny/2, nz/2): one thread per
// coarse voxel and group of 8 channels (16-byte loads and stores), each
// channel's 8 children summed in the same order.
__global__ void pool_fwd_kernel(const bf16 *__restrict__ in, bf16 *__restrict__ out, int nx,
                                int ny, int nz, int C) {
  const int mx = nx / 2, my = ny / 2, mz = nz / 2;
  const int G = C / 8;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)mx * my * mz * G) return;
  const int cg = idx % G;
  const int v = idx / G;
  const int i = v % mx, j = (v / mx) % my, k = v / (mx * my);
  bf16x8 ch[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int u = (2 * i + (q & 1)) + nx * ((2 * j + ((q >> 1) & 1)) + ny * (2 * k + (q >> 2)));
    ch[q] = *(const bf16x8 *)(in + (size_t)u * C + 8 * cg);
  }
  bf16x8 o;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    float s = 0.f;
#pragma unroll
    for (int q = 0; q < 8; ++q) s += (float)ch[q][c];
    o[c] = (bf16)(0.125f * s);
  }
  *(bf16x8 *)(out + (size_t)v * C + 8 * cg) = o;
}

// g_in (fine, FP32) += g_out(coarse)/8, four channels per thread.
__global__ void __launch_bounds__(256) pool_bwd_kernel(const float *__restrict__ gout,
                                                       float *__restrict__ gin, int nx, int ny,
                                                       int nz, int C) {
  const int G = C >> 2;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= nx * ny * nz * G) return;
  const int cg = idx % G, v = idx / G;
  const int i = v % nx, j = (v / nx) % ny, k = v / (nx * ny);
  const int p = i / 2 + (nx / 2) * (j / 2 + (ny / 2) * (k / 2));
  f32x4 *o = (f32x4 *)gin + idx;
  *o = *o + 0.125f * *((const f32x4 *)gout + (size_t)p * G + cg);
}

// nearest up-sampling: fine (nx, ny, nz) from coarse (nx/2, ...), one thread
// per fine voxel and group of 8 channels.
__global__ void up_fwd_kernel(const bf16 *__restrict__ in, bf16 *__restrict__ out, int nx,
                              int ny, int nz, int C) {
  const int G = C / 8;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)nx * ny * nz * G) return;
  const int cg = idx % G;
  const int v = idx / G;
  const int i = v % nx, j = (v / nx) % ny, k = v / (nx * ny);
  const int p = i / 2 + (nx / 2) * (j / 2 + (ny / 2) * (k / 2));
  *(bf16x8 *)(out + (size_t)v * C + 8 * cg) = *(const bf16x8 *)(in + (size_t)p * C + 8 * cg);
}

// g_in (coarse) = sum of the 8 fine children, four channels per thread.
__global__ void __launch_bounds__(256) up_bwd_kernel(const float *__restrict__ gout,
                                                     float *__restrict__ gin, int nx, int ny,
                                                     int nz, int C) {
  const int mx = nx / 2, my = ny / 2, mz = nz / 2;
  const int G = C >> 2;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= mx * my * mz * G) return;
  const int cg = idx % G, v = idx / G;
  const int i = v % mx, j = (v / mx) % my, k = v / (mx * my);
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int u = (2 * i + (q & 1)) + nx * ((2 * j + ((q >> 1) & 1)) + ny * (2 * k + (q >> 2)));
    s += *((const f32x4 *)gout + (size_t)u * G + cg);
  }
  *((f32x4 *)gin + idx) = s;
}

// d = g act'(y) in every layout its readers take, in one pass: gskip = d
// (when given), dz = bf16(d) channels-last (when given: the data gradient
// reads it), dzt = bf16(d) in runs (the weight gradient), and the block's
// bias gradient sums into part[block][C].  A thread owns one run of 8 voxels
// and 8 channels; its sums stay in registers over its runs, then go through
// the wave and the block in a fixed order.  (The previous kernel added every
// value to an LDS word per channel: 45.5 us for 16 channels of 128x96x64,
// now 37.6 us including the channel-major copy, and no gradient buffer needs
// clearing.)
// The blocks from nact on copy the layer's input x channel-major (x_runs): the
// weight gradient needs both, neither fills the chip on the coarse levels, and a
// launch costs as much as either does there.
__global__ void __launch_bounds__(256) act_bwd_kernel(const float *__restrict__ g,
                                                      const bf16 *__restrict__ y,
                                                      bf16 *__restrict__ dz,
                                                      float *__restrict__ gskip,
                                                      bf16 *__restrict__ dzt,
                                                      float *__restrict__ part, Runs R, int C,
                                                      int nact, const bf16 *__restrict__ x,
                                                      bf16 *__restrict__ xt, int ci) {
  if ((int)blockIdx.x >= nact) {
    x_runs(x, xt, R, ci, ((int)blockIdx.x - nact) * 256 + (int)threadIdx.x);
    return;
  }
  __shared__ float sb[4][128];
  const int G = C >> 3;
  const int n = R.ny * R.nz * R.nr * G;
  const size_t plane = (size_t)R.ny * R.nz * R.nr * 8;
  float db[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) db[c] = 0.f;
  // The stride is a multiple of G (a power of two up to 16), so a thread's
  // channels stay the same.
  const int cg = threadIdx.x & (G - 1);
  for (int idx = blockIdx.x * 256 + threadIdx.x; idx < n; idx += nact * 256) {
    const int q = idx / G;
    const int row = q / R.nr, r = q - row * R.nr;
    bf16x8 h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = 8 * r + e;
      if (i < R.nx) {
        const size_t o = ((size_t)row * R.nx + i) * C + 8 * cg;
        const f32x4 g0 = *(const f32x4 *)(g + o), g1 = *(const f32x4 *)(g + o + 4);
        const bf16x8 yv = *(const bf16x8 *)(y + o);
        float d[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          d[c] = (c < 4 ? g0[c] : g1[c - 4]) * dact((float)yv[c]);
          h[e][c] = (bf16)d[c];
          db[c] += d[c];
        }
        if (dz) *(bf16x8 *)(dz + o) = h[e];
        if (gskip) {
          *(f32x4 *)(gskip + o) = f32x4{d[0], d[1], d[2], d[3]};
          *(f32x4 *)(gskip + o + 4) = f32x4{d[4], d[5], d[6], d[7]};
        }
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) h[e][c] = (bf16)0.f;
      }
    }
    bf16 *t = dzt + (size_t)8 * cg * plane + (size_t)q * 8;
#pragma unroll
    for (int c = 0; c < 8; ++c) *(bf16x8 *)(t + c * plane) = run_of(h, c);
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    for (int o = 32; o >= G; o >>= 1) db[c] += __shfl_xor(db[c], o, O3D_WAVE);
    if (lane < G) sb[wv][8 * cg + c] = db[c];
  }
  __syncthreads();
  if ((int)threadIdx.x < C)
    part[(size_t)blockIdx.x * C + threadIdx.x] =
        ((sb[0][threadIdx.x] + sb[1][threadIdx.x]) + sb[2][threadIdx.x]) + sb[3][threadIdx.x];
}

// out[v] = sum_c wh[c] d0[v][c] + bh + id[v]: the network learns a
// correction to its second input plane (the previous increment).
// C a multiple of 8: 16-byte loads of d0, the channels summed in order.
__global__ void head_fwd_kernel(const bf16 *__restrict__ d0, const float *__restrict__ wh,
                                const float *__restrict__ id, float *__restrict__ out, int V,
                                int C) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= V) return;
  float s = wh[C];
  const bf16x8 *row = (const bf16x8 *)(d0 + (size_t)v * C);
  for (int gq = 0; gq < C / 8; ++gq) {
    const bf16x8 h = row[gq];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += wh[8 * gq + q] * (float)h[q];
  }
  out[v] = s + id[v];
}

// Gradients of the head: gd0[v][c] = dout[v] wh[c], and the block's sums of
// dout d0[.][c] and of dout into part[block][17] (register sums per thread,
// then wave and block in a fixed order).
__global__ void __launch_bounds__(256) head_bwd_kernel(const float *__restrict__ dout,
                                                       const bf16 *__restrict__ d0,
                                                       const float *__restrict__ wh,
                                                       float *__restrict__ gd0,
                                                       float *__restrict__ part, int V) {
  __shared__ float sw[4][17];
  float acc[17], w[16];
#pragma unroll
  for (int c = 0; c < 17; ++c) acc[c] = 0.f;
#pragma unroll
  for (int c = 0; c < 16; ++c) w[c] = wh[c];
  for (int v = blockIdx.x * 256 + threadIdx.x; v < V; v += gridDim.x * 256) {
    const float d = dout[v];
    const bf16x8 *row = (const bf16x8 *)(d0 + (size_t)v * 16);
    f32x4 *o = (f32x4 *)(gd0 + (size_t)v * 16);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bf16x8 x = row[h];
#pragma unroll
      for (int c = 0; c < 8; ++c) acc[8 * h + c] += d * (float)x[c];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int b = 8 * h + 4 * f;
        o[2 * h + f] = f32x4{d * w[b], d * w[b + 1], d * w[b + 2], d * w[b + 3]};
      }
    }
    acc[16] += d;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 17; ++c) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc[c] += __shfl_xor(acc[c], o, O3D_WAVE);
    if (lane == 0) sw[wv][c] = acc[c];
  }
  __syncthreads();
  const int c = threadIdx.x;
  if (c < 17)
    part[(size_t)blockIdx.x * 17 + c] = ((sw[0][c] + sw[1][c]) + sw[2][c]) + sw[3][c];
}

__global__ void __launch_bounds__(256) mse_kernel(const float *__restrict__ out,
                                                  const float *__restrict__ tgt, float scale,
                                                  float *__restrict__ dout, double *part, int V) {
  __shared__ double sc[4];
  double s = 0.0;
  for (int v = blockIdx.x * blockDim.x + threadIdx.x; v < V; v += gridDim.x * blockDim.x) {
    const float d = out[v] - tgt[v];
    s += (double)d * d;
    if (dout) dout[v] = scale * 2.f * d / (float)V;
  }
  s = block_sum<4>(s, sc);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void adam_kernel(float *w, const float *g, float *m, float *v, size_t n, float lr,
                            float b1, float b2, float eps, float c1, float c2) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 copies of one conv layer's master weights W[co][27*ci]:
// forward layout wf[co][kpf] and backward layout wb[ci][kpb] with
// wb[c][t'*co + o] = W[o][(26 - t')*ci + c].
__global__ void sync_weights_kernel(const float *W, bf16 *wf, bf16 *wb, int ci, int co, int kpf,
                                    int kpb) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int nf = co * kpf, nb = ci * kpb;
  if (e < nf) {
    const int o = e / kpf, k = e % kpf;
    wf[e] = (bf16)(k < 27 * ci ? W[(size_t)o * 27 * ci + k] : 0.f);
  }
  if (e < nb) {
    const int c = e / kpb, k = e % kpb;
    float v = 0.f;
    if (k < 27 * co) {
      const int tp = k / co, o = k % co;
      v = W[(size_t)o * 27 * ci + (26 - tp) * ci + c];
    }
    wb[e] = (bf16)v;
  }
}

// ------------------------------------------------------------------ network
struct Conv {
  int ci, co, level;
  size_t woff, boff;  // offsets into the flat parameter array
  int kpf, kpb;
  bf16 *wf = nullptr, *wb = nullptr;
};

int ilog2(int v) {
  int l = 0;
  while ((1 << l) < v) ++l;
  return l;
}

struct Net {
  int nx[4], ny[4], nz[4];
  size_t V[4];
  std::vector<Conv> conv;
  size_t nparam = 0, head_off = 0;
  float *W = nullptr, *G = nullptr, *M = nullptr, *Vv = nullptr;  // FP32 master, grad, Adam
  bf16 *wbuf = nullptr;  // BF16 copies of all conv weights
  // activations (bf16)
  bf16 *xin, *e0a, *e0, *p1, *e1a, *e1, *p2, *e2a, *e2, *p3, *e3a, *e3, *u2, *d2a, *d2, *u1,
      *d1a, *d1, *u0, *d0a, *d0;
  bf16 *dz = nullptr;      // scratch for act gradients (largest level)
  bf16 *dzt = nullptr, *xt = nullptr;  // the weight gradient's operands in runs
  float *gbuf = nullptr;   // FP32 activation gradients (one arena)
  float *g_d0, *g_d0a, *g_u0, *g_d1, *g_d1a, *g_u1, *g_d2, *g_d2a, *g_u2, *g_e3, *g_e3a, *g_p3,
      *g_e2, *g_e2a, *g_p2, *g_e1, *g_e1a, *g_p1, *g_e0, *g_e0a;
  float *part = nullptr;   // partial sums of the gradients (owns dzt and xt)
  // Of each layer's weights and bias, and of the head: summed at the end of a
  // backward pass.
  float *wpart[14], *bpart[15];
  ReduceSets sets;
  double *mse_part = nullptr;
  double *hpart = nullptr;
  void *act_arena = nullptr;
  hipEvent_t ev[2];
  double last_ms = 0.0, last_flops = 0.0;
  // u0 / u1 (the up-sampled d1 / d2) not formed by the last forward pass:
  // its convolutions 12 / 10 read d1 / d2 up-sampled as they staged them.
  bool up_stale[2] = {false, false};
  // The input of the last forward pass (its caller keeps it for the
  // backward pass), not yet packed into xin.
  const float *fwd_in = nullptr;
  bool xin_stale = false;
  std::vector<void *> allocs;

  ~Net() {
    for (void *p : allocs) (void)hipFree(p);
    if (act_arena) (void)hipFree(act_arena);
    if (gbuf) (void)hipFree(gbuf);
    if (part) (void)hipFree(part);
    if (hpart) (void)hipHostFree(hpart);
    (void)hipEventDestroy(ev[0]);
    (void)hipEventDestroy(ev[1]);
  }
};

#define NNCHK(...)                                                                       \
  do {                                                                                   \
    hipError_t e_ = (__VA_ARGS__);                                                       \
    if (e_ != hipSuccess) return o3d::set_error(hipGetErrorString(e_));                  \
  } while (0)
#define NCHK(x)              \
  do {                       \
    int r_ = (x);            \
    if (r_ != 0) return r_;  \
  } while (0)


void build_layers(Net &n) {
  // (ci, co, level): encoder, bottleneck, decoder (14 convolutions).
  const int spec[14][3] = {{16, 16, 0},  {16, 16, 0},  {16, 32, 1},  {32, 32, 1},  {32, 64, 2},
                           {64, 64, 2},  {64, 128, 3}, {128, 128, 3}, {128, 64, 2}, {64, 64, 2},
                           {64, 32, 1},  {32, 32, 1},  {32, 16, 0},  {16, 16, 0}};
  size_t off = 0;
  for (auto &s : spec) {
    Conv c;
    c.ci = s[0];
    c.co = s[1];
    c.level = s[2];
    c.woff = off;
    off += (size_t)c.co * 27 * c.ci;
    c.boff = off;
    off += c.co;
    c.kpf = ((27 * c.ci + 31) / 32) * 32;
    c.kpb = ((27 * c.co + 31) / 32) * 32;
    n.conv.push_back(c);
  }
  n.head_off = off;
  off += 17;
  n.nparam = off;
}

Runs runs_of(const Net &n, int level) {
  return {n.nx[level], n.ny[level], n.nz[level], (n.nx[level] + 7) / 8};
}

// Blocks of the bias and head gradient kernels, at most (their partial sums).
constexpr int kBiasBlocks = 1024;
// Blocks of act_bwd_kernel that work on a layer's output, and of head_bwd_kernel.
int act_blocks(const Runs &R, int co) {
  return std::min(kBiasBlocks, (R.rows() * R.nr * (co / 8) + 255) / 256);
}
int head_blocks(const Net &n) { return (int)std::min<size_t>(kBiasBlocks, (n.V[0] + 255) / 256); }

int alloc_activations(Net &n, int nx, int ny, int nz) {
  if (nx % 8 || ny % 8 || nz % 8)
    return o3d::set_error("network grid: every axis must be a multiple of 8");
  for (int l = 0; l < 4; ++l) {
    n.nx[l] = nx >> l;
    n.ny[l] = ny >> l;
    n.nz[l] = nz >> l;
    n.V[l] = (size_t)n.nx[l] * n.ny[l] * n.nz[l];
  }
  if (n.act_arena) { (void)hipFree(n.act_arena); n.act_arena = nullptr; }
  n.fwd_in = nullptr;  // a backward pass needs a forward pass on the new grid
  n.xin_stale = false;
  n.up_stale[0] = n.up_stale[1] = false;
  if (n.gbuf) { (void)hipFree(n.gbuf); n.gbuf = nullptr; }
  if (n.part) { (void)hipFree(n.part); n.part = nullptr; }
  // bf16 activations: channels per level.
  struct A { bf16 **p; int level, ch; };
  const A acts[] = {{&n.xin, 0, 16}, {&n.e0a, 0, 16}, {&n.e0, 0, 16}, {&n.p1, 1, 16},
                    {&n.e1a, 1, 32}, {&n.e1, 1, 32},  {&n.p2, 2, 32}, {&n.e2a, 2, 64},
                    {&n.e2, 2, 64},  {&n.p3, 3, 64},  {&n.e3a, 3, 128}, {&n.e3, 3, 128},
                    {&n.u2, 2, 128}, {&n.d2a, 2, 64}, {&n.d2, 2, 64}, {&n.u1, 1, 64},
                    {&n.d1a, 1, 32}, {&n.d1, 1, 32},  {&n.u0, 0, 32}, {&n.d0a, 0, 16},
                    {&n.d0, 0, 16}, {&n.dz, 0, 32}};
  size_t total = 0;
  for (const A &a : acts) total += ((n.V[a.level] * a.ch * sizeof(bf16) + 255) / 256) * 256;
  NNCHK(o3d::device_malloc(&n.act_arena, total));
  char *p = (char *)n.act_arena;
  for (const A &a : acts) {
    *a.p = (bf16 *)p;
    p += ((n.V[a.level] * a.ch * sizeof(bf16) + 255) / 256) * 256;
  }
  struct G { float **p; int level, ch; };
  const G grads[] = {{&n.g_d0, 0, 16}, {&n.g_d0a, 0, 16}, {&n.g_u0, 0, 32}, {&n.g_d1, 1, 32},
                     {&n.g_d1a, 1, 32}, {&n.g_u1, 1, 64}, {&n.g_d2, 2, 64}, {&n.g_d2a, 2, 64},
                     {&n.g_u2, 2, 128}, {&n.g_e3, 3, 128}, {&n.g_e3a, 3, 128}, {&n.g_p3, 3, 64},
                     {&n.g_e2, 2, 64}, {&n.g_e2a, 2, 64}, {&n.g_p2, 2, 32}, {&n.g_e1, 1, 32},
                     {&n.g_e1a, 1, 32}, {&n.g_p1, 1, 16}, {&n.g_e0, 0, 16}, {&n.g_e0a, 0, 16}};
  total = 0;
  for (const G &g : grads) total += ((n.V[g.level] * g.ch * 4 + 255) / 256) * 256;
  NNCHK(o3d::device_malloc((void **)&n.gbuf, total));
  p = (char *)n.gbuf;
  for (const G &g : grads) {
    *g.p = (float *)p;
    p += ((n.V[g.level] * g.ch * 4 + 255) / 256) * 256;
  }
  // The weight gradient's operands, for its largest layer, and every layer's partial
  // sums.
  size_t zt = 0, xt = 0;
  auto up = [](size_t bytes) { return (bytes + 255) / 256 * 256; };
  size_t wb[14], bb[15];
  total = 0;
  for (int li = 0; li < 14; ++li) {
    const Conv &c = n.conv[li];
    const Runs R = runs_of(n, c.level);
    const WgradPlan w = wgrad_plan(R, c.ci, c.co);
    zt = std::max(zt, R.dz_plane() * c.co);
    xt = std::max(xt, R.x_plane() * c.ci);
    wb[li] = up((size_t)w.slabs * c.co * 27 * c.ci * 4);
    bb[li] = up((size_t)act_blocks(R, c.co) * c.co * 4);
    total += wb[li] + bb[li];
  }
  bb[14] = up((size_t)head_blocks(n) * 17 * 4);
  total += bb[14] + up(zt * sizeof(bf16)) + up(xt * sizeof(bf16));
  p = nullptr;
  NNCHK(o3d::device_malloc((void **)&p, total));
  n.part = (float *)p;
  for (int li = 0; li < 15; ++li) {
    if (li < 14) { n.wpart[li] = (float *)p; p += wb[li]; }
    n.bpart[li] = (float *)p;
    p += bb[li];
  }
  n.dzt = (bf16 *)p;
  n.xt = (bf16 *)(p + up(zt * sizeof(bf16)));
  return 0;
}

hipStream_t st() { return o3d::current_stream(); }

int sync_weights(Net &n) {
  for (const Conv &c : n.conv) {
    const int e = std::max(c.co * c.kpf, c.ci * c.kpb);
    sync_weights_kernel<<<(e + 255) / 256, 256, 0, st()>>>(n.W + c.woff, c.wf, c.wb, c.ci, c.co,
                                                           c.kpf, c.kpb);
  }
  NNCHK(hipGetLastError());
  return 0;
}

// Deterministic He-style initialisation (splitmix64 -> uniform); the head
// starts small so the untrained network returns about its identity input.
void init_params(std::vector<float> &w, const Net &n, uint64_t seed) {
  uint64_t s = seed;
  auto next = [&]() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) / 9007199254740992.0;
  };
  std::fill(w.begin(), w.end(), 0.f);
  for (size_t li = 0; li < n.conv.size(); ++li) {
    const Conv &c = n.conv[li];
    const int fan_in = 27 * (li == 0 ? 2 : c.ci);
    const double bound = sqrt(6.0 / fan_in) * 0.8;
    for (int o = 0; o < c.co; ++o)
      for (int t = 0; t < 27; ++t)
        for (int ci = 0; ci < c.ci; ++ci) {
          if (li == 0 && ci >= 2) continue;  // padded input channels stay zero
          w[c.woff + (size_t)o * 27 * c.ci + t * c.ci + ci] = (float)((2 * next() - 1) * bound);
        }
  }
  for (int c = 0; c < 16; ++c) w[n.head_off + c] = (float)((2 * next() - 1) * 0.02);
}

// The first convolution from the network's FP32 input planes.
int conv_first_fwd(Net &n, const float *in, bf16 *y) {
  const Conv &c = n.conv[0];
  if (c.ci != 16 || c.co != 16) return o3d::set_error("first convolution: 16 -> 16 expected");
  const int V = (int)n.V[c.level];
  conv_first_kernel<<<(V + 64 * kFirstTiles - 1) / (64 * kFirstTiles), 256, 0, st()>>>(
      in, c.wf, n.W + c.boff, y,
                                                       n.nx[c.level], n.ny[c.level],
                                                       n.nz[c.level], c.kpf);
  NNCHK(hipGetLastError());
  n.last_flops += 54.0 * 2 * c.co * (double)V;  // the two real input channels
  return 0;
}

int conv_fwd(Net &n, int li, const bf16 *x, const bf16 *skip, bf16 *y) {
  const Conv &c = n.conv[li];
  ConvArgs<bf16> a;
  a.x = x; a.w = c.wf; a.bias = n.W + c.boff; a.skip = skip; a.y = y;
  a.nx = n.nx[c.level]; a.ny = n.ny[c.level]; a.nz = n.nz[c.level];
  a.lci = ilog2(c.ci); a.ci = c.ci; a.co = c.co; a.kp = c.kpf;
  a.act = 1;
  NNCHK(launch_conv<bf16>(a, st()));
  n.last_flops += 54.0 * c.ci * c.co * (double)n.V[c.level];
  return 0;
}

// Convolution li of the decoder on xc up-sampled 2x (nearest), fused into
// the LDS-staged kernel's staging; false (nothing launched) when that kernel
// does not apply to the layer's grid.
bool conv_fwd_up(Net &n, int li, const bf16 *xc, const bf16 *skip, bf16 *y, int *rc) {
  const Conv &c = n.conv[li];
  const int L = c.level;
  const LdsPlan lp = lds_plan(n.nx[L], n.ny[L], n.nz[L], c.ci, c.co);
  *rc = 0;
  if (!lp.ty) return false;
  ConvArgs<bf16> a;
  a.x = xc; a.w = c.wf; a.bias = n.W + c.boff; a.skip = skip; a.y = y;
  a.nx = n.nx[L]; a.ny = n.ny[L]; a.nz = n.nz[L];
  a.lci = ilog2(c.ci); a.ci = c.ci; a.co = c.co; a.kp = c.kpf;
  a.act = 1;
  launch_conv_lds_any<bf16, true>(a, lp, st());
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) *rc = o3d::set_error(hipGetErrorString(e));
  n.last_flops += 54.0 * c.ci * c.co * (double)n.V[L];
  return true;
}

// Adds a set to those the end of the backward pass sums.
void reduce_parts(Net &n, const float *part, int nparts, int entries, float *dst) {
  n.sets.s[n.sets.n++] = {part, dst, nparts, entries, n.sets.blocks};
  n.sets.blocks += (entries + 63) / 64;
}

// Backward of y = act(conv(x) + b + skip): gy (FP32) -> dz; gskip = dz;
// db, dW += ...; gx = conv^T(dz) when gx is given.
int conv_bwd(Net &n, int li, const float *gy, const bf16 *y, const bf16 *x, float *gskip,
             float *gx) {
  const Conv &c = n.conv[li];
  const int L = c.level;
  const Runs R = runs_of(n, L);
  const int blocks = act_blocks(R, c.co);
  const int xw = (R.rows() * (R.nr + 2) * (c.ci / 8) + 255) / 256;
  act_bwd_kernel<<<blocks + xw, 256, 0, st()>>>(gy, y, gx ? n.dz : nullptr, gskip, n.dzt,
                                                n.bpart[li], R, c.co, blocks, x, n.xt, c.ci);
  NNCHK(hipGetLastError());
  reduce_parts(n, n.bpart[li], blocks, c.co, n.G + c.boff);
  // Weight gradient.
  float *part = n.wpart[li];
  const WgradPlan w = wgrad_plan(R, c.ci, c.co);
  const dim3 g1(w.tiles, w.slabs);
  if (w.wc == 4) wgrad_kernel<4><<<g1, 256, 0, st()>>>(n.dzt, n.xt, part, R, c.ci, c.co, w.per);
  else if (w.wc == 2)
    wgrad_kernel<2><<<g1, 256, 0, st()>>>(n.dzt, n.xt, part, R, c.ci, c.co, w.per);
  else
    wgrad_kernel<1><<<g1, 256, 0, st()>>>(n.dzt, n.xt, part, R, c.ci, c.co, w.per);
  NNCHK(hipGetLastError());
  reduce_parts(n, part, w.slabs, c.co * 27 * c.ci, n.G + c.woff);
  if (gx) {
    ConvArgs<float> a;
    a.x = n.dz; a.w = c.wb; a.bias = nullptr; a.skip = nullptr; a.y = gx;
    a.nx = n.nx[L]; a.ny = n.ny[L]; a.nz = n.nz[L];
    a.lci = ilog2(c.co); a.ci = c.co; a.co = c.ci; a.kp = c.kpb;
    a.act = 0;
    NNCHK(launch_conv<float>(a, st()));
  }
  return 0;
}

int elem_blocks(size_t n) { return (int)((n + 255) / 256); }

int forward(Net &n, const float *in, float *out) {
  n.last_flops = 0.0;
  NNCHK(hipEventRecord(n.ev[0], st()));
  // The packed BF16 input (the first layer's weight gradient reads it) is
  // formed only when a backward pass follows.
  n.fwd_in = in;
  n.xin_stale = true;
  NCHK(conv_first_fwd(n, in, n.e0a));
  NCHK(conv_fwd(n, 1, n.e0a, nullptr, n.e0));
  pool_fwd_kernel<<<elem_blocks(n.V[1] * 2), 256, 0, st()>>>(n.e0, n.p1, n.nx[0], n.ny[0],
                                                               n.nz[0], 16);
  NCHK(conv_fwd(n, 2, n.p1, nullptr, n.e1a));
  NCHK(conv_fwd(n, 3, n.e1a, nullptr, n.e1));
  pool_fwd_kernel<<<elem_blocks(n.V[2] * 4), 256, 0, st()>>>(n.e1, n.p2, n.nx[1], n.ny[1],
                                                               n.nz[1], 32);
  NCHK(conv_fwd(n, 4, n.p2, nullptr, n.e2a));
  NCHK(conv_fwd(n, 5, n.e2a, nullptr, n.e2));
  pool_fwd_kernel<<<elem_blocks(n.V[3] * 8), 256, 0, st()>>>(n.e2, n.p3, n.nx[2], n.ny[2],
                                                               n.nz[2], 64);
  NCHK(conv_fwd(n, 6, n.p3, nullptr, n.e3a));
  NCHK(conv_fwd(n, 7, n.e3a, nullptr, n.e3));
  up_fwd_kernel<<<elem_blocks(n.V[2] * 16), 256, 0, st()>>>(n.e3, n.u2, n.nx[2], n.ny[2],
                                                              n.nz[2], 128);
  NCHK(conv_fwd(n, 8, n.u2, n.e2, n.d2a));
  NCHK(conv_fwd(n, 9, n.d2a, nullptr, n.d2));
  int rc = 0;
  n.up_stale[1] = conv_fwd_up(n, 10, n.d2, n.e1, n.d1a, &rc);
  NCHK(rc);
  if (!n.up_stale[1]) {
    up_fwd_kernel<<<elem_blocks(n.V[1] * 8), 256, 0, st()>>>(n.d2, n.u1, n.nx[1], n.ny[1],
                                                               n.nz[1], 64);
    NCHK(conv_fwd(n, 10, n.u1, n.e1, n.d1a));
  }
  NCHK(conv_fwd(n, 11, n.d1a, nullptr, n.d1));
  n.up_stale[0] = conv_fwd_up(n, 12, n.d1, n.e0, n.d0a, &rc);
  NCHK(rc);
  if (!n.up_stale[0]) {
    up_fwd_kernel<<<elem_blocks(n.V[0] * 4), 256, 0, st()>>>(n.d1, n.u0, n.nx[0], n.ny[0],
                                                               n.nz[0], 32);
    NCHK(conv_fwd(n, 12, n.u0, n.e0, n.d0a));
  }
  NCHK(conv_fwd(n, 13, n.d0a, nullptr, n.d0));
  head_fwd_kernel<<<elem_blocks(n.V[0]), 256, 0, st()>>>(n.d0, n.W + n.head_off, in + n.V[0],
                                                          out, (int)n.V[0], 16);
  NNCHK(hipGetLastError());
  NNCHK(hipEventRecord(n.ev[1], st()));
  return 0;
}

int backward(Net &n, const float *dout) {
  // Every activation gradient is written by its first reader's pass and only
  // added to by pool_bwd_kernel, so none needs clearing.
  const int hb = head_blocks(n);
  n.sets.n = n.sets.blocks = 0;
  head_bwd_kernel<<<hb, 256, 0, st()>>>(dout, n.d0, n.W + n.head_off, n.g_d0, n.bpart[14],
                                        (int)n.V[0]);
  NNCHK(hipGetLastError());
  reduce_parts(n, n.bpart[14], hb, 17, n.G + n.head_off);
  NCHK(conv_bwd(n, 13, n.g_d0, n.d0, n.d0a, nullptr, n.g_d0a));
  if (n.up_stale[0]) {  // the forward pass read d1 up-sampled without forming u0
    up_fwd_kernel<<<elem_blocks(n.V[0] * 4), 256, 0, st()>>>(n.d1, n.u0, n.nx[0], n.ny[0],
                                                               n.nz[0], 32);
    NNCHK(hipGetLastError());
    n.up_stale[0] = false;
  }
  NCHK(conv_bwd(n, 12, n.g_d0a, n.d0a, n.u0, n.g_e0, n.g_u0));
  up_bwd_kernel<<<elem_blocks(n.V[1] * 8), 256, 0, st()>>>(n.g_u0, n.g_d1, n.nx[0], n.ny[0],
                                                             n.nz[0], 32);
  NCHK(conv_bwd(n, 11, n.g_d1, n.d1, n.d1a, nullptr, n.g_d1a));
  if (n.up_stale[1]) {
    up_fwd_kernel<<<elem_blocks(n.V[1] * 8), 256, 0, st()>>>(n.d2, n.u1, n.nx[1], n.ny[1],
                                                               n.nz[1], 64);
    NNCHK(hipGetLastError());
    n.up_stale[1] = false;
  }
  NCHK(conv_bwd(n, 10, n.g_d1a, n.d1a, n.u1, n.g_e1, n.g_u1));
  up_bwd_kernel<<<elem_blocks(n.V[2] * 16), 256, 0, st()>>>(n.g_u1, n.g_d2, n.nx[1], n.ny[1],
                                                             n.nz[1], 64);
  NCHK(conv_bwd(n, 9, n.g_d2, n.d2, n.d2a, nullptr, n.g_d2a));
  NCHK(conv_bwd(n, 8, n.g_d2a, n.d2a, n.u2, n.g_e2, n.g_u2));
  up_bwd_kernel<<<elem_blocks(n.V[3] * 32), 256, 0, st()>>>(n.g_u2, n.g_e3, n.nx[2], n.ny[2],
                                                              n.nz[2], 128);
  NCHK(conv_bwd(n, 7, n.g_e3, n.e3, n.e3a, nullptr, n.g_e3a));
  NCHK(conv_bwd(n, 6, n.g_e3a, n.e3a, n.p3, nullptr, n.g_p3));
  pool_bwd_kernel<<<elem_blocks(n.V[2] * 16), 256, 0, st()>>>(n.g_p3, n.g_e2, n.nx[2], n.ny[2],
                                                               n.nz[2], 64);
  NCHK(conv_bwd(n, 5, n.g_e2, n.e2, n.e2a, nullptr, n.g_e2a));
  NCHK(conv_bwd(n, 4, n.g_e2a, n.e2a, n.p2, nullptr, n.g_p2));
  pool_bwd_kernel<<<elem_blocks(n.V[1] * 8), 256, 0, st()>>>(n.g_p2, n.g_e1, n.nx[1], n.ny[1],
                                                               n.nz[1], 32);
  NCHK(conv_bwd(n, 3, n.g_e1, n.e1, n.e1a, nullptr, n.g_e1a));
  NCHK(conv_bwd(n, 2, n.g_e1a, n.e1a, n.p1, nullptr, n.g_p1));
  pool_bwd_kernel<<<elem_blocks(n.V[0] * 4), 256, 0, st()>>>(n.g_p1, n.g_e0, n.nx[0], n.ny[0],
                                                               n.nz[0], 16);
  NCHK(conv_bwd(n, 1, n.g_e0, n.e0, n.e0a, nullptr, n.g_e0a));
  if (n.xin_stale) {
    pack_input_kernel<<<elem_blocks(n.V[0]), 256, 0, st()>>>(n.fwd_in, n.xin, (int)n.V[0], 16);
    NNCHK(hipGetLastError());
    n.xin_stale = false;
  }
  NCHK(conv_bwd(n, 0, n.g_e0a, n.e0a, n.xin, nullptr, nullptr));
  reduce_parts_kernel<<<n.sets.blocks, 256, 0, st()>>>(n.sets);
  NNCHK(hipGetLastError());
  return 0;
}

}  // namespace nn
}  // namespace o3d

using namespace o3d::nn;

extern "C" int o3d_nn_create(int nx, int ny, int nz, unsigned long long seed, void **out) {
  if (!out) return o3d::set_error("NULL argument");
  Net *n = new Net();
  build_layers(*n);
  int rc = 0;
  auto al = [&](void **p, size_t bytes) {
    if (rc) return;
    if (o3d::device_malloc(p, bytes) != hipSuccess) { rc = o3d::set_error("hipMalloc failed"); return; }
    n->allocs.push_back(*p);
    if (hipMemset(*p, 0, bytes) != hipSuccess) rc = o3d::set_error("hipMemset failed");
  };
  al((void **)&n->W, n->nparam * 4);
  al((void **)&n->G, n->nparam * 4);
  al((void **)&n->M, n->nparam * 4);
  al((void **)&n->Vv, n->nparam * 4);
  size_t wb = 0;
  for (const Conv &c : n->conv) wb += (size_t)c.co * c.kpf + (size_t)c.ci * c.kpb;
  al((void **)&n->wbuf, wb * sizeof(bf16));
  al((void **)&n->mse_part, 1024 * sizeof(double));
  if (!rc && hipHostMalloc((void **)&n->hpart, 1024 * sizeof(double)) != hipSuccess)
    rc = o3d::set_error("hipHostMalloc failed");
  if (!rc && (hipEventCreate(&n->ev[0]) != hipSuccess || hipEventCreate(&n->ev[1]) != hipSuccess))
    rc = o3d::set_error("hipEventCreate failed");
  if (!rc) {
    bf16 *p = n->wbuf;
    for (Conv &c : n->conv) {
      c.wf = p; p += (size_t)c.co * c.kpf;
      c.wb = p; p += (size_t)c.ci * c.kpb;
    }
    std::vector<float> h(n->nparam);
    init_params(h, *n, seed);
    if (hipMemcpy(n->W, h.data(), n->nparam * 4, hipMemcpyHostToDevice) != hipSuccess)
      rc = o3d::set_error("hipMemcpy failed");
  }
  if (!rc) rc = alloc_activations(*n, nx, ny, nz);
  if (!rc) rc = sync_weights(*n);
  if (!rc && hipStreamSynchronize(st()) != hipSuccess) rc = o3d::set_error("sync failed");
  if (rc) { delete n; return rc; }
  *out = n;
  return 0;
}

extern "C" int o3d_nn_destroy(void *nn) {
  if (nn) {
    (void)hipStreamSynchronize(st());
    delete (Net *)nn;
  }
  return 0;
}

extern "C" int o3d_nn_resize(void *nn, int nx, int ny, int nz) {
  if (!nn) return o3d::set_error("NULL network");
  Net &n = *(Net *)nn;
  if (n.nx[0] == nx && n.ny[0] == ny && n.nz[0] == nz) return 0;
  NNCHK(hipStreamSynchronize(st()));
  return alloc_activations(n, nx, ny, nz);
}

extern "C" int o3d_nn_num_params(void *nn, long long *np) {
  if (!nn || !np) return o3d::set_error("NULL argument");
  *np = (long long)((Net *)nn)->nparam;
  return 0;
}

extern "C" int o3d_nn_get_params(void *nn, float *out) {
  if (!nn || !out) return o3d::set_error("NULL argument");
  Net &n = *(Net *)nn;
  NNCHK(hipMemcpyAsync(out, n.W, n.nparam * 4, hipMemcpyDefault, st()));
  NNCHK(hipStreamSynchronize(st()));
  return 0;
}

extern "C" int o3d_nn_set_params(void *nn, const float *in) {
  if (!nn || !in) return o3d::set_error("NULL argument");
  Net &n = *(Net *)nn;
  NNCHK(hipMemcpyAsync(n.W, in, n.nparam * 4, hipMemcpyDefault, st()));
  NCHK(sync_weights(n));
  NNCHK(hipStreamSynchronize(st()));
  return 0;
}

extern "C" int o3d_nn_get_grads(void *nn, float *out) {
  if (!nn || !out) return o3d::set_error("NULL argument");
  Net &n = *(Net *)nn;
  NNCHK(hipMemcpyAsync(out, n.G, n.nparam * 4, hipMemcpyDefault, st()));
  NNCHK(hipStreamSynchronize(st()));
  return 0;
}

extern "C" int o3d_nn_zero_grad(void *nn) {
  if (!nn) return o3d::set_error("NULL network");
  Net &n = *(Net *)nn;
  NNCHK(hipMemsetAsync(n.G, 0, n.nparam * 4, st()));
  return 0;
}

extern "C" int o3d_nn_forward(void *nn, const float *in, float *out) {
  if (!nn || !in || !out) return o3d::set_error("NULL argument");
  return forward(*(Net *)nn, in, out);
}

extern "C" int o3d_nn_backward(void *nn, const float *dout) {
  if (!nn || !dout) return o3d::set_error("NULL argument");
  return backward(*(Net *)nn, dout);
}

extern "C" int o3d_nn_mse(void *nn, const float *out, const float *target, float scale,
                          float *dout, double *loss) {
  if (!nn || !out || !target) return o3d::set_error("NULL argument");
  Net &n = *(Net *)nn;
  const int V = (int)n.V[0];
  const int blocks = std::min(1024, (V + 255) / 256);
  mse_kernel<<<blocks, 256, 0, st()>>>(out, target, scale, dout, n.mse_part, V);
  NNCHK(hipGetLastError());
  if (loss) {
    NNCHK(hipMemcpyAsync(n.hpart, n.mse_part, blocks * sizeof(double), hipMemcpyDeviceToHost,
                         st()));
    NNCHK(hipStreamSynchronize(st()));
    double s = 0.0;
    for (int b = 0; b < blocks; ++b) s += n.hpart[b];
    *loss = s / V;
  }
  return 0;
}

extern "C" int o3d_nn_adam_step(void *nn, float lr, float beta1, float beta2, float eps, int t) {
  if (!nn) return o3d::set_error("NULL network");
  Net &n = *(Net *)nn;
  const float c1 = 1.f - powf(beta1, (float)t), c2 = 1.f - powf(beta2, (float)t);
  adam_kernel<<<elem_blocks(n.nparam), 256, 0, st()>>>(n.W, n.G, n.M, n.Vv, n.nparam, lr, beta1,
                                                        beta2, eps, c1, c2);
  NNCHK(hipGetLastError());
  return sync_weights(n);
}

extern "C" int o3d_nn_last_timing(void *nn, double *ms, double *flops) {
  if (!nn) return o3d::set_error("NULL network");
  Net &n = *(Net *)nn;
  float t = 0.f;
  NNCHK(hipEventSynchronize(n.ev[1]));
  NNCHK(hipEventElapsedTime(&t, n.ev[0], n.ev[1]));
  if (ms) *ms = t;
  if (flops) *flops = n.last_flops;
  return 0;
}

