// Multigrid V-cycles for the coarse-grid correction of the warm starts.
//
// No counterpart in the reference (its pressure solve is SOR from the
// previous pressure).  In the mixed forms the residual of the warm-start
// guess is averaged over 2^3 blocks, this module solves the 7-point Poisson
// problem of those averages (spacing 2h) approximately, and the solver adds
// the trilinear interpolation of the result to the guess.  The SOR solve
// that follows still decides convergence (same stop rule), so the
// correction only changes where SOR starts.  The grids are small (128^3 and
// below at 256^3) and the launch count dominates: a level above the last takes
// one launch per sweep, the levels of at most 16^3 cells run as one V-cycle in
// one block's LDS, and a larger last level takes two sweeps per launch or, where
// its rows are too wide for that, one launch per colour.
#include <algorithm>
#include <utility>

#include "o3d_mg.h"

namespace o3d {

size_t mg_plan(MgHierarchy &H, const int m0[3], const double h[3], const int per[3]) {
  H = MgHierarchy();
  for (int a = 0; a < 3; ++a) H.per[a] = per[a];
  int m[3] = {m0[0], m0[1], m0[2]};
  double hh[3] = {h[0], h[1], h[2]};
  size_t floats = 0;
  for (int l = 0; l < kMgMaxLevels; ++l) {
    for (int a = 0; a < 3; ++a) {
      H.m[l][a] = m[a];
      H.c[l][a] = 1.0 / (hh[a] * hh[a]);
    }
    const size_t cells = (size_t)m[0] * m[1] * m[2];
    floats += 3 * cells;
    H.levels = l + 1;
    const bool halvable = m[0] % 2 == 0 && m[1] % 2 == 0 && m[2] % 2 == 0 && m[0] >= 4 &&
                          m[1] >= 4 && m[2] >= 4;
    if (cells <= 64 || !halvable) break;
    for (int a = 0; a < 3; ++a) {
      m[a] /= 2;
      hh[a] *= 2.0;
    }
  }
  return floats;
}

void mg_bind(MgHierarchy &H, float *base) {
  for (int l = 0; l < H.levels; ++l) {
    const size_t cells = (size_t)H.m[l][0] * H.m[l][1] * H.m[l][2];
    H.u[l] = base;
    H.f[l] = base + cells;
    H.r[l] = base + 2 * cells;
    base += 3 * cells;
  }
}

namespace {

// Neighbour along an axis of m cells: periodic wrap, or the cell-centred
// mirror (the ghost cell equals the edge cell).
__device__ __forceinline__ int mg_nb(int q, int m, int per) {
  if (q < 0) return per ? q + m : 0;
  if (q >= m) return per ? q - m : m - 1;
  return q;
}

struct MgGrid {
  int mx, my, mz, px, py, pz;
  float cx, cy, cz;
  float diag, invd;  // -2 (cx + cy + cz) and its reciprocal
};

// Weighted sum of the 6 neighbours (32-bit offsets: mg_plan keeps every
// level below 2^31 cells).
__device__ __forceinline__ float mg_lap_off(const float *u, const MgGrid &g, int i, int j, int k) {
  const int pl = g.mx * g.my;
  const int jr = g.mx * j, kp = pl * k;
  const float sx = u[kp + jr + mg_nb(i - 1, g.mx, g.px)] + u[kp + jr + mg_nb(i + 1, g.mx, g.px)];
  const float sy = u[kp + g.mx * mg_nb(j - 1, g.my, g.py) + i] +
                   u[kp + g.mx * mg_nb(j + 1, g.my, g.py) + i];
  const float sz = u[pl * mg_nb(k - 1, g.mz, g.pz) + jr + i] +
                   u[pl * mg_nb(k + 1, g.mz, g.pz) + jr + i];
  return g.cx * sx + g.cy * sy + g.cz * sz;
}

// Gauss-Seidel update of cell (i, j, k) at linear index q.
__device__ __forceinline__ void mg_relax(float *u, const float *f, const MgGrid &g, int i, int j,
                                         int k, int q) {
  u[q] = (f[q] - mg_lap_off(u, g, i, j, k)) * g.invd;
}

// The same update from the neighbour sums (the operation order of
// mg_lap_off and mg_relax, so both give the same value).
__device__ __forceinline__ float mg_relax_value(float fq, float sx, float sy, float sz,
                                                const MgGrid &g) {
  return (fq - (g.cx * sx + g.cy * sy + g.cz * sz)) * g.invd;
}

// The residual f - L u averaged over the 8 children of coarse cell (I, J, K),
// the fine level's axes even: the children's own cells and the faces around
// them are loaded once (20 loads of one or two cells, against 7 per child).
__device__ __forceinline__ float mg_child_mean(const float *u, const float *f, const MgGrid &g,
                                               int I, int J, int K) {
  const int i = 2 * I, j = 2 * J, k = 2 * K, pl = g.mx * g.my;
  const int xm = mg_nb(i - 1, g.mx, g.px), xp = mg_nb(i + 2, g.mx, g.px);
  const int ry[4] = {g.mx * mg_nb(j - 1, g.my, g.py), g.mx * j, g.mx * (j + 1),
                     g.mx * mg_nb(j + 2, g.my, g.py)};
  const int rz[4] = {pl * mg_nb(k - 1, g.mz, g.pz), pl * k, pl * (k + 1),
                     pl * mg_nb(k + 2, g.mz, g.pz)};
  auto pair = [&](const float *a, int y, int z) {
    return *reinterpret_cast<const float2 *>(a + (i + ry[y] + rz[z]));
  };
  float2 c[4][4];  // [z][y], the rows that hold children or face them
#pragma unroll
  for (int z = 0; z < 4; ++z)
#pragma unroll
    for (int y = 0; y < 4; ++y)
      if ((y == 1 || y == 2) || (z == 1 || z == 2)) c[z][y] = pair(u, y, z);
  float s = 0.f;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const int y = 1 + (n & 1), z = 1 + (n >> 1);
    const int row = ry[y] + rz[z];
    const float2 v = c[z][y], ff = pair(f, y, z);
    const float l = u[row + xm], r = u[row + xp];
    const float2 ya = c[z][y - 1], yb = c[z][y + 1], za = c[z - 1][y], zb = c[z + 1][y];
    s += ff.x - ((g.cx * (l + v.y) + g.cy * (ya.x + yb.x) + g.cz * (za.x + zb.x)) + g.diag * v.x);
    s += ff.y - ((g.cx * (v.x + r) + g.cy * (ya.y + yb.y) + g.cz * (za.y + zb.y)) + g.diag * v.y);
  }
  return 0.125f * s;
}

// Trilinear interpolation of the coarse field uc (cx, cy, cz cells) at the 8
// fine cells of coarse cell (I, J, K), v[2 * (2 * dz + dy) + dx].  Along an
// axis a fine cell lies a quarter of a coarse cell from its own coarse cell's
// centre: weight 1/4 of the neighbour on its side (periodic wraps, others
// clamp).  Lines along x first, then y, then z; 27 loads for 8 cells.
__device__ __forceinline__ void mg_interp_cell(const float *uc, int I, int J, int K, int cx,
                                               int cy, int cz, int px, int py, int pz,
                                               float v[8]) {
  const int x[3] = {mg_nb(I - 1, cx, px), I, mg_nb(I + 1, cx, px)};
  const int y[3] = {cx * mg_nb(J - 1, cy, py), cx * J, cx * mg_nb(J + 1, cy, py)};
  const int pl = cx * cy;
  const int z[3] = {pl * mg_nb(K - 1, cz, pz), pl * K, pl * mg_nb(K + 1, cz, pz)};
  // Weight of the upper coarse cell for the lower and upper fine cell.
  const float x0 = !px && I == 0 ? 0.f : 0.75f, x1 = !px && I == cx - 1 ? 0.f : 0.25f;
  const float y0 = !py && J == 0 ? 0.f : 0.75f, y1 = !py && J == cy - 1 ? 0.f : 0.25f;
  const float z0 = !pz && K == 0 ? 0.f : 0.75f, z1 = !pz && K == cz - 1 ? 0.f : 0.25f;
  float p[3][4];  // per coarse plane, the 4 fine cells of (dy, dx)
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    float l[3], r[3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      const float *q = uc + (y[b] + z[c]);
      const float a0 = q[x[0]], a1 = q[x[1]], a2 = q[x[2]];
      l[b] = (1.f - x0) * a0 + x0 * a1;
      r[b] = (1.f - x1) * a1 + x1 * a2;
    }
    p[c][0] = (1.f - y0) * l[0] + y0 * l[1];
    p[c][1] = (1.f - y0) * r[0] + y0 * r[1];
    p[c][2] = (1.f - y1) * l[1] + y1 * l[2];
    p[c][3] = (1.f - y1) * r[1] + y1 * r[2];
  }
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    v[n] = (1.f - z0) * p[0][n] + z0 * p[1][n];
    v[4 + n] = (1.f - z1) * p[1][n] + z1 * p[2][n];
  }
}

// ------------------------------------------------------ fused level kernels
// One whole red-black sweep of a level with everything around it in one
// launch, for levels with every axis even.  A block stages a tile of 32 x 8 x
// TZ cells with a halo of 2 in LDS, relaxes red on the tile and one cell
// around it, then black on the tile, so neighbouring blocks recompute the halo
// instead of meeting between the colours; the result goes to another array.
//   ZERO      the level starts from u = 0 (nothing is read, and red is f / diag)
//   PROLONG   u += the interpolated coarse correction before the sweep
//   RESTRICT  (with ZERO) the averaged residual after the sweep goes to fc
// Same updates in the same order as mg_smooth_kernel, mg_restrict_kernel and
// mg_prolong_kernel, so the values are the same.  What bounds the levels is the
// number of launches (3 to 4 us each below 128^3) and, at 128^3, the work per
// cell of the tile and halo (a thread stages whole columns, so the index
// arithmetic is once per column: with it per cell the kernel took twice as
// long).  A V(1, 1) level was 8 launches and is 2: 128^3, from zero with
// restriction 30 -> 10 us, with prolongation 23 -> 13 us; 64^3 12 -> 4.7 and
// 10.5 -> 5.0 us; a plain sweep of 128^3 14.6 -> 10.6 us.
constexpr int kSwX = 32, kSwY = 8, kSwNT = 512;

template <int TZ, bool ZERO, bool PROLONG, bool RESTRICT>
__global__ void __launch_bounds__(kSwNT) mg_sweep_kernel(float *__restrict__ uo,
                                                         const float *__restrict__ u,
                                                         const float *__restrict__ f,
                                                         const float *__restrict__ uc,
                                                         float *__restrict__ fc, MgGrid g,
                                                         int ntx, int nty) {
  static_assert(!RESTRICT || ZERO, "the residual's black halo needs red on a halo of 2");
  constexpr int LX = kSwX + 4, LY = kSwY + 4, LZ = TZ + 4, LP = LX * LY;  // u, halo of 2
  constexpr int HF = ZERO ? 2 : 1;                                        // f's halo
  constexpr int FX = kSwX + 2 * HF, FY = kSwY + 2 * HF, FZ = TZ + 2 * HF, FP = FX * FY;
  constexpr int CX = kSwX / 2 + 4, CY = kSwY / 2 + 4, CZ = TZ / 2 + 4;
  static_assert(LP <= kSwNT && CX * CY <= kSwNT, "one column per thread");
  __shared__ float su[LZ * LP];
  __shared__ float sf[FZ * FP];
  __shared__ float sc[PROLONG ? CZ * CY * CX : 1];
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int bx = t % ntx, r = t / ntx, by = r % nty, bz = r / nty;
  const int x0 = bx * kSwX, y0 = by * kSwY, z0 = bz * TZ;
  const int tid = threadIdx.x;
  const int plane = g.mx * g.my;
  // Stored cell of cell q (periodic image; elsewhere any cell of the level,
  // for positions that no cell of the tile reads).
  auto img = [](int q, int m, int per) {
    if (q < 0) q = per ? q + m : 0;
    if (q >= m) q = per ? q - m : m - 1;
    return min(max(q, 0), m - 1);
  };
  // A thread stages one column of each array; z is the same for the block.
  if (tid < FP) {
    const int lx = tid % FX, ly = tid / FX;
    const float *fp = f + img(x0 - HF + lx, g.mx, g.px) + g.mx * img(y0 - HF + ly, g.my, g.py);
    float v[FZ];
#pragma unroll
    for (int lz = 0; lz < FZ; ++lz) v[lz] = fp[(size_t)plane * img(z0 - HF + lz, g.mz, g.pz)];
#pragma unroll
    for (int lz = 0; lz < FZ; ++lz) {
      sf[tid + FP * lz] = v[lz];
      // Red of the first sweep from zero; x0, y0, z0 and the halo are even.
      if (ZERO) su[tid + FP * lz] = ((lx + ly + lz) & 1) == 0 ? v[lz] * g.invd : 0.f;
    }
  }
  if (!ZERO) {
    const int lx = tid % LX, ly = tid / LX;
    const int gi = x0 - 2 + lx, gj = y0 - 2 + ly;
    const float *up = u + img(gi, g.mx, g.px) + g.mx * img(gj, g.my, g.py);
    float v[LZ];
    if (tid < LP) {
#pragma unroll
      for (int lz = 0; lz < LZ; ++lz) v[lz] = up[(size_t)plane * img(z0 - 2 + lz, g.mz, g.pz)];
    }
    if (PROLONG) {
      if (tid < CX * CY) {
        const int cx = g.mx >> 1, cy = g.my >> 1, cz = g.mz >> 1;
        const float *cp = uc + img(x0 / 2 - 2 + tid % CX, cx, g.px) +
                          cx * img(y0 / 2 - 2 + tid / CX, cy, g.py);
#pragma unroll
        for (int lz = 0; lz < CZ; ++lz)
          sc[tid + CX * CY * lz] = cp[(size_t)(cx * cy) * img(z0 / 2 - 2 + lz, cz, g.pz)];
      }
      __syncthreads();
    }
    if (tid < LP) {
      // Lower coarse cell (local) and weight of the upper one (mg_interp_cell).
      const int X = (lx + 1) >> 1, Y = (ly + 1) >> 1;
      float wx = (lx & 1) ? 0.25f : 0.75f, wy = (ly & 1) ? 0.25f : 0.75f;
      if (!g.px && (gi <= 0 || gi >= g.mx - 1)) wx = 0.f;
      if (!g.py && (gj <= 0 || gj >= g.my - 1)) wy = 0.f;
      float c[CZ];
      if (PROLONG) {
#pragma unroll
        for (int Z = 0; Z < CZ; ++Z) {
          const float *a = sc + X + CX * (Y + CY * Z);
          c[Z] = (1.f - wy) * ((1.f - wx) * a[0] + wx * a[1]) +
                 wy * ((1.f - wx) * a[CX] + wx * a[CX + 1]);
        }
      }
#pragma unroll
      for (int lz = 0; lz < LZ; ++lz) {
        float w = v[lz];
        if (PROLONG) {
          const int gk = z0 - 2 + lz, Z = (lz + 1) >> 1;
          float wz = (lz & 1) ? 0.25f : 0.75f;
          if (!g.pz && (gk <= 0 || gk >= g.mz - 1)) wz = 0.f;
          w += (1.f - wz) * c[Z] + wz * c[Z + 1];
        }
        su[tid + LP * lz] = w;
      }
    }
  }
  __syncthreads();
  // Offsets of the neighbours of a cell of su, the cell itself (the mirror)
  // past an edge of an axis that does not wrap.
  auto below = [](int q, int per, int d) { return !per && q == 0 ? 0 : -d; };
  auto above = [](int q, int m, int per, int d) { return !per && q == m - 1 ? 0 : d; };
  // A colour on the tile and one cell around it: a thread takes one pair of
  // columns (17 pairs x 10 rows) on every third plane.
  auto relax = [&](int colour) {
    constexpr int HX = kSwX / 2 + 1, HY = kSwY + 2, HC = HX * HY, ZG = kSwNT / HC;
    if (tid >= HC * ZG) return;
    const int zg = tid / HC, q = tid - zg * HC;
    const int ly = 1 + q / HX, lxp = 1 + 2 * (q % HX);
    const int ym = below(y0 - 2 + ly, g.py, LX), yp = above(y0 - 2 + ly, g.my, g.py, LX);
#pragma unroll
    for (int n = 0; n < (TZ + 2 + ZG - 1) / ZG; ++n) {
      const int lz = 1 + zg + n * ZG;
      if (lz > TZ + 2) break;
      const int lx = lxp + ((1 + ly + lz + colour) & 1);
      const int i = x0 - 2 + lx, k = z0 - 2 + lz;
      float *c = su + lx + LX * ly + LP * lz;
      const float sx = c[below(i, g.px, 1)] + c[above(i, g.mx, g.px, 1)];
      const float sy = c[ym] + c[yp];
      const float sz = c[below(k, g.pz, LP)] + c[above(k, g.mz, g.pz, LP)];
      *c = mg_relax_value(sf[lx - 2 + HF + FX * (ly - 2 + HF) + FP * (lz - 2 + HF)], sx, sy, sz,
                          g);
    }
  };
  if (!ZERO) {
    relax(0);
    __syncthreads();
  }
  if (RESTRICT) {
    relax(1);
    __syncthreads();
    constexpr int NC = kSwX / 2 * (kSwY / 2) * (TZ / 2);
    if (tid < NC) {
      const int I = tid % (kSwX / 2), J = tid / (kSwX / 2) % (kSwY / 2),
                K = tid / (kSwX / 2 * (kSwY / 2));
      float s = 0.f;
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        const int lx = 2 + 2 * I + (n & 1), ly = 2 + 2 * J + ((n >> 1) & 1),
                  lz = 2 + 2 * K + (n >> 2);
        const int i = x0 - 2 + lx, j = y0 - 2 + ly, k = z0 - 2 + lz;
        const float *c = su + lx + LX * ly + LP * lz;
        // Even children have no upper edge, odd ones no lower edge.
        const float sx = c[n & 1 ? -1 : below(i, g.px, 1)] + c[n & 1 ? above(i, g.mx, g.px, 1) : 1];
        const float sy = c[n & 2 ? -LX : below(j, g.py, LX)] +
                         c[n & 2 ? above(j, g.my, g.py, LX) : LX];
        const float sz = c[n & 4 ? -LP : below(k, g.pz, LP)] +
                         c[n & 4 ? above(k, g.mz, g.pz, LP) : LP];
        s += sf[lx + FX * ly + FP * lz] -
             ((g.cx * sx + g.cy * sy + g.cz * sz) + g.diag * *c);
      }
      const int ci = x0 / 2 + I, cj = y0 / 2 + J, ck = z0 / 2 + K;
      if (2 * ci < g.mx && 2 * cj < g.my && 2 * ck < g.mz)
        fc[ci + (g.mx >> 1) * (cj + (g.my >> 1) * ck)] = 0.125f * s;
    }
  }
  // The tile's cells: a column of every second plane per thread, so the colour
  // is the column's.
  const int lx = 2 + tid % kSwX, ly = 2 + tid / kSwX % kSwY, zb = tid / (kSwX * kSwY);
  const int i = x0 - 2 + lx, j = y0 - 2 + ly;
  if (i >= g.mx || j >= g.my) return;
  const int xm = below(i, g.px, 1), xp = above(i, g.mx, g.px, 1);
  const int ym = below(j, g.py, LX), yp = above(j, g.my, g.py, LX);
  const bool black = !RESTRICT && ((lx + ly + zb) & 1);
  float *o = uo + i + (size_t)g.mx * j;
#pragma unroll
  for (int n = 0; n < TZ / 2; ++n) {
    const int lz = 2 + zb + 2 * n, k = z0 - 2 + lz;
    if (k >= g.mz) break;
    const float *c = su + lx + LX * ly + LP * lz;
    float v = *c;
    if (black) {  // from the finished red
      const float sz = c[below(k, g.pz, LP)] + c[above(k, g.mz, g.pz, LP)];
      v = mg_relax_value(sf[lx - 2 + HF + FX * (ly - 2 + HF) + FP * (lz - 2 + HF)],
                         c[xm] + c[xp], c[ym] + c[yp], sz, g);
    }
    o[(size_t)plane * k] = v;
  }
}

// One colour of a red-black Gauss-Seidel sweep, one thread per cell of that
// colour (mx even: every row holds mx / 2 cells of each colour).  The
// smoothing, restriction and prolongation kernels take their blocks in
// XCD-aware order (xcd_tile): each XCD works on a contiguous run of planes
// and finds most neighbour planes in its own L2 (at 256^3: the 128^3
// prolongation 10.2 -> 8.0 us, restriction 10.1 -> 9.7 us, smoothing 7.5 ->
// 7.2 us).  The pooling kernels only stream and keep the plain order.
__global__ void __launch_bounds__(256) mg_smooth_kernel(float *__restrict__ u,
                                                        const float *__restrict__ f, MgGrid g,
                                                        int colour) {
  const int hx = g.mx >> 1;
  const int p = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (p >= hx * g.my * g.mz) return;
  const int row = p / hx, t = p - row * hx;
  const int k = row / g.my, j = row - k * g.my;
  const int i = 2 * t + ((j + k + colour) & 1);
  mg_relax(u, f, g, i, j, k, i + g.mx * row);
}

// Two cells of one colour are neighbours (an odd axis that wraps): cells 0 and m - 1
// of such an axis.  Relaxed in place, which of them reads the other's new value would
// depend on waves and blocks that nothing orders, and with it the free constant of the
// solution (by some 1e-3 of it) from run to run.  So every kernel of a level whose
// colours meet reads all cells of a colour before it writes any of them: the values do
// not depend on the kernel, its tiles or the block's size.  (One wave does so by
// itself, and so did in practice the launches per colour and small blocks, whose loads
// are all on their way before the first store.)  A V(2, 2) cycle where they meet / where
// no axis wraps: a last level of 20 x 15 x 9 cells in one block 82 / 73 us (one barrier
// more per colour), 36 x 9 x 13 in rows 322 / 268 us, 104 x 87 x 33 by launches per
// colour 442 / 424 us.
__device__ __host__ __forceinline__ bool mg_colours_meet(const MgGrid &g) {
  return ((g.mx & g.px) | (g.my & g.py) | (g.mz & g.pz)) & 1;
}

// One colour of a sweep where the colours meet: the new values go to uo.  un holds the
// other colour's latest values (uo itself for the second colour of a sweep), u the
// values before the sweep; a neighbour of the cell's own colour (across the wrap, or
// the cell itself at a mirrored edge) is read from u.
__global__ void __launch_bounds__(256) mg_smooth_meet_kernel(float *uo, const float *un,
                                                             const float *u,
                                                             const float *__restrict__ f,
                                                             MgGrid g, int colour) {
  const int hx = (g.mx + 1) >> 1;
  const int p = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (p >= hx * g.my * g.mz) return;
  const int row = p / hx, t = p - row * hx;
  const int k = row / g.my, j = row - k * g.my;
  const int i = 2 * t + ((j + k + colour) & 1);
  if (i >= g.mx) return;
  const int pl = g.mx * g.my, q = i + g.mx * row;
  const int xm = mg_nb(i - 1, g.mx, g.px), xp = mg_nb(i + 1, g.mx, g.px);
  const int ym = mg_nb(j - 1, g.my, g.py), yp = mg_nb(j + 1, g.my, g.py);
  const int zm = mg_nb(k - 1, g.mz, g.pz), zp = mg_nb(k + 1, g.mz, g.pz);
  // The value d places from the cell, across so many indices of an axis.
  auto at = [&](int across, int d) { return ((across & 1) ? un : u)[q + d]; };
  const float sx = at(xm - i, xm - i) + at(xp - i, xp - i);
  const float sy = at(ym - j, g.mx * (ym - j)) + at(yp - j, g.mx * (yp - j));
  const float sz = at(zm - k, pl * (zm - k)) + at(zp - k, pl * (zp - k));
  uo[q] = mg_relax_value(f[q], sx, sy, sz, g);
}

// The same in place for mx odd: one thread per cell, the other colour idle.
__global__ void __launch_bounds__(256) mg_smooth_any_kernel(float *__restrict__ u,
                                                            const float *__restrict__ f,
                                                            MgGrid g, int colour) {
  const int idx = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (idx >= g.mx * g.my * g.mz) return;
  const int row = idx / g.mx, i = idx - row * g.mx;
  const int k = row / g.my, j = row - k * g.my;
  if (((i + j + k) & 1) != colour) return;
  mg_relax(u, f, g, i, j, k, idx);
}

// fc = the residual of the fine level averaged over the 8 children of each
// coarse cell.
__global__ void __launch_bounds__(256) mg_restrict_kernel(float *__restrict__ fc,
                                                          const float *__restrict__ u,
                                                          const float *__restrict__ f, MgGrid g) {
  const int cx = g.mx >> 1, cy = g.my >> 1, cz = g.mz >> 1;
  const int idx = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (idx >= cx * cy * cz) return;
  const int crow = idx / cx, I = idx - crow * cx;
  const int K = crow / cy, J = crow - K * cy;
  fc[idx] = mg_child_mean(u, f, g, I, J, K);
}

// u += trilinear interpolation of the coarse correction uc, one thread per
// coarse cell.
__global__ void __launch_bounds__(256) mg_prolong_kernel(float *__restrict__ u,
                                                         const float *__restrict__ uc, int mx,
                                                         int my, int mz, int px, int py, int pz) {
  const int cx = mx >> 1, cy = my >> 1, cz = mz >> 1;
  const int p = xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (p >= cx * cy * cz) return;
  const int row = p / cx, I = p - row * cx;
  const int K = row / cy, J = row - K * cy;
  float v[8];
  mg_interp_cell(uc, I, J, K, cx, cy, cz, px, py, pz, v);
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const size_t fr = (size_t)(2 * J + (n & 1)) + (size_t)my * (2 * K + (n >> 1));
    float2 *o = reinterpret_cast<float2 *>(u + (size_t)mx * fr) + I;
    float2 w = *o;
    w.x += v[2 * n];
    w.y += v[2 * n + 1];
    *o = w;
  }
}

// The coarsest level: `sweeps` red-black Gauss-Seidel sweeps from u = 0 by
// one block, the level staged in LDS.
__global__ void __launch_bounds__(1024) mg_coarsest_kernel(float *__restrict__ u,
                                                           const float *__restrict__ f, MgGrid g,
                                                           int sweeps) {
  __shared__ float su[kMgCoarsestCells], sf[kMgCoarsestCells];
  const int n = g.mx * g.my * g.mz;
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    su[q] = 0.f;
    sf[q] = f[q];
  }
  __syncthreads();
  // The cells of this thread and their neighbours, worked out once (a V-cycle over 9 x
  // 15 x 24 cells, y and z mirrored, 383 -> 81 us).
  const bool meet = mg_colours_meet(g);
  constexpr int kPer = kMgCoarsestCells / 1024;
  int nb[kPer][6], col[kPer];
  float fq[kPer], v[kPer];
#pragma unroll
  for (int s = 0; s < kPer; ++s) {
    const int q = threadIdx.x + s * blockDim.x;
    col[s] = -1;
    fq[s] = 0.f;
    if (q >= n) continue;
    const int row = q / g.mx, i = q - row * g.mx;
    const int k = row / g.my, j = row - k * g.my;
    const int pl = g.mx * g.my;
    nb[s][0] = q - i + mg_nb(i - 1, g.mx, g.px);
    nb[s][1] = q - i + mg_nb(i + 1, g.mx, g.px);
    nb[s][2] = q + g.mx * (mg_nb(j - 1, g.my, g.py) - j);
    nb[s][3] = q + g.mx * (mg_nb(j + 1, g.my, g.py) - j);
    nb[s][4] = q + pl * (mg_nb(k - 1, g.mz, g.pz) - k);
    nb[s][5] = q + pl * (mg_nb(k + 1, g.mz, g.pz) - k);
    col[s] = (i + j + k) & 1;
    fq[s] = sf[q];
  }
  for (int sw = 0; sw < sweeps; ++sw)
    for (int colour = 0; colour < 2; ++colour) {
#pragma unroll
      for (int s = 0; s < kPer; ++s)
        if (col[s] == colour) {
          v[s] = mg_relax_value(fq[s], su[nb[s][0]] + su[nb[s][1]], su[nb[s][2]] + su[nb[s][3]],
                                su[nb[s][4]] + su[nb[s][5]], g);
          if (!meet) su[threadIdx.x + s * blockDim.x] = v[s];
        }
      __syncthreads();
      if (!meet) continue;
#pragma unroll
      for (int s = 0; s < kPer; ++s)
        if (col[s] == colour) su[threadIdx.x + s * blockDim.x] = v[s];
      __syncthreads();
    }
  for (int q = threadIdx.x; q < n; q += blockDim.x) u[q] = su[q];
}

// The levels from `first` down, all of at most kMgCoarsestCells cells, as
// one V-cycle by one block in LDS: f of the first level in, u of the first
// level out (from u = 0).  Same smoother, residual, restriction and
// prolongation as the per-level kernels.  Each thread keeps the coordinates
// of its cells of one colour in registers for the sweeps of a level.
constexpr int kMgSmallLevels = 4;
constexpr int kMgSmallCells = 4096 + 512 + 64 + 8;
constexpr int kMgSmallThreads = 1024;
constexpr int kMgSmallPer = kMgCoarsestCells / 2 / kMgSmallThreads;
struct MgSmall {
  int levels;
  MgGrid g[kMgSmallLevels];
  int off[kMgSmallLevels];  // offsets of each level in the LDS arrays
  int nu1, nu2, coarse_sweeps;
};

// p / n for the cell counts of the small levels (p < 2^16): exact, since
// (p + 1/2) / n is at least 1 / (2 n) away from an integer, far more than the
// rounding of the two float operations; an integer division by a run-time n
// is some 20 instructions.
struct SmallDiv {
  int n;
  float inv;
  __device__ __forceinline__ explicit SmallDiv(int n_) : n(n_), inv(1.0f / (float)n_) {}
  __device__ __forceinline__ int div(int p) const { return (int)(((float)p + 0.5f) * inv); }
};

__device__ __forceinline__ void lds_smooth(float *u, const float *f, const MgGrid &g,
                                           int sweeps) {
  const bool meet = mg_colours_meet(g);
  if (g.mx & 1) {
    const int n = g.mx * g.my * g.mz;
    constexpr int kPer = kMgCoarsestCells / kMgSmallThreads;
    for (int s = 0; s < sweeps; ++s)
      for (int colour = 0; colour < 2; ++colour) {
        float v[kPer];
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
          const int q = threadIdx.x + c * kMgSmallThreads;
          if (q >= n) continue;
          const int row = q / g.mx, i = q - row * g.mx;
          const int k = row / g.my, j = row - k * g.my;
          v[c] = u[q];
          if (((i + j + k) & 1) != colour) continue;
          v[c] = (f[q] - mg_lap_off(u, g, i, j, k)) * g.invd;
          if (!meet) u[q] = v[c];
        }
        __syncthreads();
        if (!meet) continue;
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
          const int q = threadIdx.x + c * kMgSmallThreads;
          if (q < n) u[q] = v[c];
        }
        __syncthreads();
      }
    return;
  }
  // Per cell pair of this thread: its offset and, for both of its cells, the
  // neighbours' (the y and z neighbours lie in the rows beside).
  const int hx = g.mx >> 1, nh = hx * g.my * g.mz, pl = g.mx * g.my;
  const SmallDiv dx(hx), dy(g.my);
  int base[kMgSmallPer], oxl[kMgSmallPer], oxr[kMgSmallPer], oym[kMgSmallPer], oyp[kMgSmallPer],
      ozm[kMgSmallPer], ozp[kMgSmallPer];
#pragma unroll
  for (int s = 0; s < kMgSmallPer; ++s) {
    const int p = threadIdx.x + s * kMgSmallThreads;
    const int row = dx.div(p), t = p - row * hx, k = dy.div(row), j = row - k * g.my;
    base[s] = (2 * t + g.mx * row) * 2 + ((j + k) & 1);
    oxl[s] = mg_nb(2 * t - 1, g.mx, g.px) - 2 * t;
    oxr[s] = mg_nb(2 * t + 2, g.mx, g.px) - 2 * t;
    oym[s] = g.mx * (mg_nb(j - 1, g.my, g.py) - j);
    oyp[s] = g.mx * (mg_nb(j + 1, g.my, g.py) - j);
    ozm[s] = pl * (mg_nb(k - 1, g.mz, g.pz) - k);
    ozp[s] = pl * (mg_nb(k + 1, g.mz, g.pz) - k);
  }
  for (int sw = 0; sw < sweeps; ++sw)
    for (int colour = 0; colour < 2; ++colour) {
      float v[kMgSmallPer];
#pragma unroll
      for (int s = 0; s < kMgSmallPer; ++s)
        if (threadIdx.x + s * kMgSmallThreads < nh) {
          const int right = (base[s] + colour) & 1, l = base[s] >> 1, q = l + right;
          const float sx = u[right ? l : l + oxl[s]] + u[right ? l + oxr[s] : l + 1];
          v[s] = mg_relax_value(f[q], sx, u[q + oym[s]] + u[q + oyp[s]],
                                u[q + ozm[s]] + u[q + ozp[s]], g);
          if (!meet) u[q] = v[s];
        }
      __syncthreads();
      if (!meet) continue;
#pragma unroll
      for (int s = 0; s < kMgSmallPer; ++s)
        if (threadIdx.x + s * kMgSmallThreads < nh)
          u[(base[s] >> 1) + ((base[s] + colour) & 1)] = v[s];
      __syncthreads();
    }
}

// `sweeps` red-black sweeps of a level of at most 64 cells by wave 0, one
// cell per lane in registers, the neighbours fetched across lanes: no block
// barrier per colour.  The same updates in the same order as lds_smooth.
// Called by every thread of the block (it ends with the block barrier).
__device__ __forceinline__ void wave_smooth(float *u, const float *f, const MgGrid &g,
                                            int sweeps) {
  if (threadIdx.x < O3D_WAVE) {
    const int n = g.mx * g.my * g.mz;
    const int q = threadIdx.x;
    const bool act = q < n;
    int i = 0, j = 0, k = 0;
    if (act) {
      const int row = q / g.mx;
      i = q - row * g.mx;
      k = row / g.my;
      j = row - k * g.my;
    }
    // Neighbour lanes (inactive lanes read their own).
    const int rj = g.mx * (j + g.my * k);
    const int lxm = act ? rj + mg_nb(i - 1, g.mx, g.px) : q;
    const int lxp = act ? rj + mg_nb(i + 1, g.mx, g.px) : q;
    const int lym = act ? i + g.mx * (mg_nb(j - 1, g.my, g.py) + g.my * k) : q;
    const int lyp = act ? i + g.mx * (mg_nb(j + 1, g.my, g.py) + g.my * k) : q;
    const int lzm = act ? i + g.mx * (j + g.my * mg_nb(k - 1, g.mz, g.pz)) : q;
    const int lzp = act ? i + g.mx * (j + g.my * mg_nb(k + 1, g.mz, g.pz)) : q;
    const int col = (i + j + k) & 1;
    float uq = act ? u[q] : 0.f;
    const float fq = act ? f[q] : 0.f;
    for (int sw = 0; sw < sweeps; ++sw)
      for (int colour = 0; colour < 2; ++colour) {
        const float sx = __shfl(uq, lxm) + __shfl(uq, lxp);
        const float sy = __shfl(uq, lym) + __shfl(uq, lyp);
        const float sz = __shfl(uq, lzm) + __shfl(uq, lzp);
        if (act && col == colour) uq = mg_relax_value(fq, sx, sy, sz, g);
      }
    if (act) u[q] = uq;
  }
  __syncthreads();
}

__global__ void __launch_bounds__(kMgSmallThreads) mg_small_vcycle_kernel(
    float *__restrict__ u_out, const float *__restrict__ f_in, MgSmall S) {
  __shared__ __align__(16) float su[kMgSmallCells], sf[kMgSmallCells];
  const int n0 = S.g[0].mx * S.g[0].my * S.g[0].mz;
  for (int q = threadIdx.x; q < n0; q += kMgSmallThreads) {
    sf[q] = f_in[q];
    su[q] = 0.f;
  }
  __syncthreads();
  // Down: smooth, then the averaged residual as the next level's f.  (One copy of
  // the code for all levels: every launch meets it cold, and with a copy per level
  // 24x16x8 cells took 21.4 us, now 19.8.)
#pragma unroll 1
  for (int l = 0; l < kMgSmallLevels - 1; ++l) {
    if (l >= S.levels - 1) break;
    const MgGrid &g = S.g[l], &c = S.g[l + 1];
    float *u = su + S.off[l];
    const float *f = sf + S.off[l];
    lds_smooth(u, f, g, S.nu1);
    const int nc = c.mx * c.my * c.mz;
    const SmallDiv dx(c.mx), dy(c.my);
    for (int q = threadIdx.x; q < nc; q += kMgSmallThreads) {
      const int crow = dx.div(q), I = q - crow * c.mx;
      const int K = dy.div(crow), J = crow - K * c.my;
      sf[S.off[l + 1] + q] = mg_child_mean(u, f, g, I, J, K);
      su[S.off[l + 1] + q] = 0.f;
    }
    __syncthreads();
  }
  // Coarsest.
#pragma unroll 1
  for (int l = 1; l < kMgSmallLevels; ++l)
    if (l == S.levels - 1) {
      const MgGrid &g = S.g[l];
      if (g.mx * g.my * g.mz <= O3D_WAVE)
        wave_smooth(su + S.off[l], sf + S.off[l], g, S.coarse_sweeps);
      else
        lds_smooth(su + S.off[l], sf + S.off[l], g, S.coarse_sweeps);
    }
  // Up: prolong, smooth.
#pragma unroll 1
  for (int l = kMgSmallLevels - 2; l >= 0; --l) {
    if (l >= S.levels - 1) continue;
    const MgGrid &g = S.g[l], &c = S.g[l + 1];
    float *u = su + S.off[l];
    const float *uc = su + S.off[l + 1];
    const int np = c.mx * c.my * c.mz;
    const SmallDiv dx(c.mx), dy(c.my);
    for (int q = threadIdx.x; q < np; q += kMgSmallThreads) {
      const int row = dx.div(q), I = q - row * c.mx;
      const int K = dy.div(row), J = row - K * c.my;
      float v[8];
      mg_interp_cell(uc, I, J, K, c.mx, c.my, c.mz, g.px, g.py, g.pz, v);
#pragma unroll
      for (int n = 0; n < 4; ++n) {
        float *o = u + 2 * I + g.mx * (2 * J + (n & 1) + g.my * (2 * K + (n >> 1)));
        o[0] += v[2 * n];
        o[1] += v[2 * n + 1];
      }
    }
    __syncthreads();
    lds_smooth(u, sf + S.off[l], g, S.nu2);
  }
  for (int q = threadIdx.x; q < n0; q += kMgSmallThreads) u_out[q] = su[q];
}

// Two sweeps of a last level too large for one block, per launch.  The rows of a
// tile of 8 x 8 (y, z) and a halo of 4 lie in LDS, whole in x (at most kBtX cells), and
// four half sweeps shrink the halo.  A halo row is the stored row it is an image of and
// keeps that row's colours, and a colour is read before it is written where two of its
// cells meet (mg_colours_meet), so every tile computes the same values: those of the
// launches per colour.  A thread takes a pair of cells (2t, 2t + 1), one of
// each colour.  A launch per colour, 120 of them for 60 sweeps, is bound by the launches
// at the sizes met here.  A V(1, 1) cycle over a last level, launches per colour / this:
// 21^3 433 / 281 us, 25^3 407 / 298, 31^3 407 / 329.
constexpr int kBtX = 40, kBtT = 8, kBtL = kBtT + 8, kBtNT = 1024;
constexpr int kBtPer = kBtL * kBtL * (kBtX / 2) / kBtNT;
template <bool ZERO>
__global__ void __launch_bounds__(kBtNT) mg_bottom_kernel(float *__restrict__ uo,
                                                          const float *__restrict__ u,
                                                          const float *__restrict__ f, MgGrid g,
                                                          int nty) {
  constexpr int L = kBtL;
  __shared__ float su[L * L * kBtX];
  __shared__ int img[2][L];  // stored row of a local y, z; -1 outside
  const int y0 = (int)(blockIdx.x % nty) * kBtT, z0 = (int)(blockIdx.x / nty) * kBtT;
  const int tid = threadIdx.x;
  if (tid < 2 * L) {
    const int a = tid / L, l = tid % L;
    const int q = (a ? z0 : y0) + l - 4, m = a ? g.mz : g.my;
    img[a][l] = (a ? g.pz : g.py) ? ((q % m) + m) % m : (q < 0 || q >= m ? -1 : q);
  }
  __syncthreads();
  const int hp = (g.mx + 1) >> 1, slots = hp * L * L;
  const bool meet = mg_colours_meet(g);
  // Per slot: LDS place of its left cell, row offsets of the y and z neighbours (0: the
  // mirror), the x neighbours' offsets of both cells, the rows' distance to the edge.
  int at[kBtPer], ym[kBtPer], yp[kBtPer], zm[kBtPer], zp[kBtPer], xl[kBtPer], xr[kBtPer],
      par[kBtPer], rim[kBtPer];
  float f0[kBtPer], f1[kBtPer];
#pragma unroll
  for (int s = 0; s < kBtPer; ++s) {
    const int q = tid + s * kBtNT;
    rim[s] = -1;
    at[s] = ym[s] = yp[s] = zm[s] = zp[s] = xl[s] = xr[s] = par[s] = 0;
    f0[s] = f1[s] = 0.f;
    if (q >= slots) continue;
    const int row = q / hp, t = q - row * hp, ly = row % L, lz = row / L;
    const int y = img[0][ly], z = img[1][lz];
    if (y < 0 || z < 0) continue;
    const int x = 2 * t;
    at[s] = row * kBtX + x;
    const size_t o = x + (size_t)g.mx * (y + (size_t)g.my * z);
    const bool two = x + 1 < g.mx;
    su[at[s]] = ZERO ? 0.f : u[o];
    f0[s] = f[o];
    if (two) {
      su[at[s] + 1] = ZERO ? 0.f : u[o + 1];
      f1[s] = f[o + 1];
    }
    ym[s] = !g.py && y == 0 ? 0 : -kBtX;
    yp[s] = !g.py && y == g.my - 1 ? 0 : kBtX;
    zm[s] = !g.pz && z == 0 ? 0 : -L * kBtX;
    zp[s] = !g.pz && z == g.mz - 1 ? 0 : L * kBtX;
    // Before the left cell, after the last one of the pair.
    xl[s] = x > 0 ? -1 : (g.px ? g.mx - 1 : 0);
    const int last = two ? x + 1 : x;
    xr[s] = last < g.mx - 1 ? last + 1 - x : (g.px ? -x : last - x);
    par[s] = ((y + z) & 1) | (two ? 2 : 0);
    rim[s] = min(min(ly, L - 1 - ly), min(lz, L - 1 - lz));
  }
  __syncthreads();
#pragma unroll 1
  for (int h = 0; h < 4; ++h) {
    float v[kBtPer];
#pragma unroll
    for (int s = 0; s < kBtPer; ++s) {
      const int right = (par[s] + h) & 1;
      if (rim[s] > h && (!right || (par[s] & 2))) {
        const float *c = su + at[s] + right;
        const bool two = par[s] & 2;
        const float a = right ? c[-1] : c[xl[s]];
        const float b = right ? c[xr[s] - 1] : (two ? c[1] : c[xr[s]]);
        v[s] = mg_relax_value(right ? f1[s] : f0[s], a + b, c[ym[s]] + c[yp[s]],
                              c[zm[s]] + c[zp[s]], g);
        if (!meet) su[at[s] + right] = v[s];
      }
    }
    __syncthreads();
    if (!meet) continue;
#pragma unroll
    for (int s = 0; s < kBtPer; ++s) {
      const int right = (par[s] + h) & 1;
      if (rim[s] > h && (!right || (par[s] & 2))) su[at[s] + right] = v[s];
    }
    __syncthreads();
  }
#pragma unroll
  for (int s = 0; s < kBtPer; ++s) {
    if (rim[s] < 4) continue;
    const int row = at[s] / kBtX, x = at[s] - row * kBtX;
    const int y = y0 + row % L - 4, z = z0 + row / L - 4;
    if (y >= g.my || z >= g.mz) continue;
    float *o = uo + x + (size_t)g.mx * (y + (size_t)g.my * z);
    o[0] = su[at[s]];
    if (par[s] & 2) o[1] = su[at[s] + 1];
  }
}

MgGrid grid_of(const MgHierarchy &H, int l) {
  MgGrid g;
  g.mx = H.m[l][0]; g.my = H.m[l][1]; g.mz = H.m[l][2];
  g.px = H.per[0]; g.py = H.per[1]; g.pz = H.per[2];
  g.cx = (float)H.c[l][0]; g.cy = (float)H.c[l][1]; g.cz = (float)H.c[l][2];
  g.diag = -2.f * (g.cx + g.cy + g.cz);
  g.invd = 1.f / g.diag;
  return g;
}

unsigned blocks_for(long long threads) { return (unsigned)((threads + 255) / 256); }

hipError_t smooth(MgHierarchy &H, int l, int sweeps, hipStream_t s) {
  const MgGrid g = grid_of(H, l);
  const long long n = (long long)g.mx * g.my * g.mz;
  if (mg_colours_meet(g)) {
    // A sweep goes from H.u[l] into H.r[l], which then trade places.
    const unsigned blocks = blocks_for((long long)((g.mx + 1) / 2) * g.my * g.mz);
    for (int q = 0; q < sweeps; ++q) {
      for (int colour = 0; colour < 2; ++colour)
        mg_smooth_meet_kernel<<<blocks, 256, 0, s>>>(H.r[l], colour ? H.r[l] : H.u[l], H.u[l],
                                                     H.f[l], g, colour);
      std::swap(H.u[l], H.r[l]);
    }
    return hipGetLastError();
  }
  for (int q = 0; q < sweeps; ++q)
    for (int colour = 0; colour < 2; ++colour) {
      if (g.mx & 1)
        mg_smooth_any_kernel<<<blocks_for(n), 256, 0, s>>>(H.u[l], H.f[l], g, colour);
      else
        mg_smooth_kernel<<<blocks_for(n / 2), 256, 0, s>>>(H.u[l], H.f[l], g, colour);
    }
  return hipGetLastError();
}

// The levels from l down fit one block's LDS (every level at most
// kMgCoarsestCells cells, the sum at most kMgSmallCells), and every level
// above the last is halvable (mx even).
bool small_from(const MgHierarchy &H, int l) {
  if (H.levels - l > kMgSmallLevels) return false;
  size_t tot = 0;
  for (int q = l; q < H.levels; ++q) {
    const size_t c = (size_t)H.m[q][0] * H.m[q][1] * H.m[q][2];
    if (c > (size_t)kMgCoarsestCells) return false;
    tot += c;
  }
  return tot <= (size_t)kMgSmallCells;
}
// One sweep of level l from H.u[l] into H.r[l], which then trade places.  Tiles
// of 8 planes, or of 4 while 8 would leave CUs without a block.
template <bool ZERO, bool PROLONG, bool RESTRICT>
hipError_t sweep(MgHierarchy &H, int l, hipStream_t s) {
  const MgGrid g = grid_of(H, l);
  const int ntx = (g.mx + kSwX - 1) / kSwX, nty = (g.my + kSwY - 1) / kSwY;
  const float *uc = PROLONG ? H.u[l + 1] : nullptr;
  float *fc = RESTRICT ? H.f[l + 1] : nullptr;
  if ((long long)ntx * nty * ((g.mz + 7) / 8) >= 512)
    mg_sweep_kernel<8, ZERO, PROLONG, RESTRICT><<<ntx * nty * ((g.mz + 7) / 8), kSwNT, 0, s>>>(
        H.r[l], H.u[l], H.f[l], uc, fc, g, ntx, nty);
  else
    mg_sweep_kernel<4, ZERO, PROLONG, RESTRICT><<<ntx * nty * ((g.mz + 3) / 4), kSwNT, 0, s>>>(
        H.r[l], H.u[l], H.f[l], uc, fc, g, ntx, nty);
  std::swap(H.u[l], H.r[l]);
  return hipGetLastError();
}

__global__ void mg_zero_kernel(float *u, int n) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < n) u[idx] = 0.f;
}

hipError_t clear_level(const MgHierarchy &H, int l, hipStream_t s) {
  const int n = H.m[l][0] * H.m[l][1] * H.m[l][2];
  mg_zero_kernel<<<blocks_for(n), 256, 0, s>>>(H.u[l], n);
  return hipGetLastError();
}

// An even number of sweeps of the last level, two per launch.
hipError_t bottom(MgHierarchy &H, int l, int sweeps, bool zero, hipStream_t s) {
  const MgGrid g = grid_of(H, l);
  const int nty = (g.my + kBtT - 1) / kBtT, blocks = nty * ((g.mz + kBtT - 1) / kBtT);
  for (int q = 0; q < sweeps; q += 2) {
    if (zero && q == 0)
      mg_bottom_kernel<true><<<blocks, kBtNT, 0, s>>>(H.r[l], H.u[l], H.f[l], g, nty);
    else
      mg_bottom_kernel<false><<<blocks, kBtNT, 0, s>>>(H.r[l], H.u[l], H.f[l], g, nty);
    std::swap(H.u[l], H.r[l]);
  }
  return hipGetLastError();
}

// A V(nu1, nu2) cycle from level l down; zero: u starts from 0 (its array need
// not be cleared).
hipError_t vcycle(MgHierarchy &H, int l, int nu1, int nu2, bool zero, hipStream_t s) {
  const MgGrid g = grid_of(H, l);
  const int n = g.mx * g.my * g.mz;
  hipError_t e = hipSuccess;
  if (l > 0 && H.levels - l >= 2 && small_from(H, l)) {
    MgSmall S;
    S.levels = H.levels - l;
    int off = 0;
    for (int q = 0; q < S.levels; ++q) {
      S.g[q] = grid_of(H, l + q);
      S.off[q] = off;
      off += H.m[l + q][0] * H.m[l + q][1] * H.m[l + q][2];
    }
    S.nu1 = nu1;
    S.nu2 = nu2;
    S.coarse_sweeps = 10;
    mg_small_vcycle_kernel<<<1, kMgSmallThreads, 0, s>>>(H.u[l], H.f[l], S);
    return hipGetLastError();
  }
  if (l == H.levels - 1) {
    // At most 64 cells when the axes halve that far: one wave, 30 sweeps.
    if (n <= kMgCoarsestCells) {
      const int threads = n <= 64 ? 64 : 1024;
      mg_coarsest_kernel<<<1, threads, 0, s>>>(H.u[l], H.f[l], g, n <= 64 ? 30 : 60);
      return hipGetLastError();
    }
    if (g.mx <= kBtX) return bottom(H, l, 60, zero, s);
    if (zero && (e = clear_level(H, l, s)) != hipSuccess) return e;
    return smooth(H, l, 60, s);
  }
  // Every axis of a level above the last is even.
  int pre = nu1;
  bool restricted = false;
  if (zero && pre == 1) {
    if ((e = sweep<true, false, true>(H, l, s)) != hipSuccess) return e;
    restricted = true;
    pre = 0;
  } else if (zero && pre > 1) {
    if ((e = sweep<true, false, false>(H, l, s)) != hipSuccess) return e;
    --pre;
  } else if (zero) {
    if ((e = clear_level(H, l, s)) != hipSuccess) return e;
  }
  for (; pre > 0; --pre)
    if ((e = sweep<false, false, false>(H, l, s)) != hipSuccess) return e;
  if (!restricted) {
    mg_restrict_kernel<<<blocks_for(n / 8), 256, 0, s>>>(H.f[l + 1], H.u[l], H.f[l], g);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if ((e = vcycle(H, l + 1, nu1, nu2, true, s)) != hipSuccess) return e;
  if (nu2 < 1) {
    mg_prolong_kernel<<<blocks_for(n / 8), 256, 0, s>>>(H.u[l], H.u[l + 1], g.mx, g.my, g.mz,
                                                        g.px, g.py, g.pz);
    return hipGetLastError();
  }
  if ((e = sweep<false, true, false>(H, l, s)) != hipSuccess) return e;
  for (int q = 1; q < nu2; ++q)
    if ((e = sweep<false, false, false>(H, l, s)) != hipSuccess) return e;
  return hipSuccess;
}

// Per-block sums of f (at most kMgMeanBlocks blocks), then f -= their total / n:
// the coarse problem made compatible with its null space (the constants).
constexpr int kMgMeanBlocks = 256;
__global__ void __launch_bounds__(256) mg_sum_kernel(const float *__restrict__ f, int n,
                                                     double *__restrict__ part) {
  __shared__ double sc[4];
  double s = 0.0;
  // 32 loads in flight, added in order (256x192x128 cells 26 us with 8, now 6.8).
  const int step = gridDim.x * 256;
  for (long long i0 = blockIdx.x * 256 + threadIdx.x; i0 < n; i0 += 32ll * step) {
    float v[32];
#pragma unroll
    for (int q = 0; q < 32; ++q) {
      const long long i = i0 + (long long)q * step;
      v[q] = f[min(i, (long long)n - 1)];
    }
#pragma unroll
    for (int q = 0; q < 32; ++q)
      if (i0 + (long long)q * step < n) s += (double)v[q];
  }
  s = block_sum<4>(s, sc);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void __launch_bounds__(256) mg_center_kernel(float *__restrict__ f, int n,
                                                        const double *__restrict__ part,
                                                        int nparts) {
  __shared__ double sc[4];
  double s = threadIdx.x < nparts ? part[threadIdx.x] : 0.0;
  s = block_sum<4>(s, sc);
  const float m = (float)(s / n);
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) f[i] -= m;
}

__global__ void __launch_bounds__(256) mg_pool_split_kernel(const float *__restrict__ r,
                                                            float *__restrict__ f0, int nx,
                                                            int ny, int nz) {
  const int mx = nx / 2, my = ny / 2, mz = nz / 2;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= mx * my * mz) return;
  const int I = idx % mx, J = (idx / mx) % my, K = idx / (mx * my);
  const size_t hx = (size_t)(nx / 2), half = (size_t)nx * ny * nz / 2;
  float t = 0.f;
  // Cells 2I and 2I+1 of a row are one red and one black node, both entry I
  // of their colour's row.
  for (int q = 0; q < 4; ++q) {
    const size_t row = (size_t)(2 * J + (q & 1)) + (size_t)ny * (2 * K + (q >> 1));
    t += r[hx * row + I] + r[half + hx * row + I];
  }
  f0[idx] = 0.125f * t;
}

// The trilinear interpolation of the level-0 solution onto the fine grid, one
// thread per coarse cell, 64 x 4 of them per block and blockIdx.z = the plane.
// SPLIT: stored colour-split (the first FP32 correction solve's starting
// iterate; a pair of cells (2c, 2c + 1) of a row is one red and one black cell,
// both entry c); else added to the FP64 field q.  A thread per pair of fine
// cells was bound by its arithmetic (97 % VALU busy): 512x384x256 split 94 us.
template <bool SPLIT>
__global__ void __launch_bounds__(256) mg_prolong_top_kernel(float *__restrict__ e,
                                                             double *__restrict__ q,
                                                             const float *__restrict__ u0,
                                                             int nx, int ny, int nz, int px,
                                                             int py, int pz) {
  const int cx = nx / 2, cy = ny / 2;
  const int I = blockIdx.x * 64 + threadIdx.x;
  const int J = blockIdx.y * 4 + threadIdx.y, K = blockIdx.z;
  if (I >= cx || J >= cy) return;
  float v[8];
  mg_interp_cell(u0, I, J, K, cx, cy, nz / 2, px, py, pz, v);
  const size_t half = (size_t)cx * ny * nz;
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const size_t row = (size_t)(2 * J + (n & 1)) + (size_t)ny * (2 * K + (n >> 1));
    if (SPLIT) {
      // Red cell: i = 2 I + (j + k) % 2.
      const bool odd = ((n & 1) + (n >> 1)) & 1;
      e[cx * row + I] = odd ? v[2 * n + 1] : v[2 * n];
      e[half + cx * row + I] = odd ? v[2 * n] : v[2 * n + 1];
    } else {
      double2 *o = reinterpret_cast<double2 *>(q + (size_t)nx * row) + I;
      double2 w = *o;
      w.x = w.x + (double)v[2 * n];
      w.y = w.y + (double)v[2 * n + 1];
      *o = w;
    }
  }
}

}  // namespace

hipError_t mg_pool_split(const float *r, float *f0, int nx, int ny, int nz, hipStream_t s) {
  if (nx % 2 || ny % 2 || nz % 2) return hipErrorInvalidValue;
  const int nc = (nx / 2) * (ny / 2) * (nz / 2);
  mg_pool_split_kernel<<<(nc + 255) / 256, 256, 0, s>>>(r, f0, nx, ny, nz);
  return hipGetLastError();
}

hipError_t mg_prolong_split(float *e, const float *u0, int nx, int ny, int nz, const int per[3],
                            hipStream_t s) {
  if (nx % 2 || ny % 2 || nz % 2) return hipErrorInvalidValue;
  const dim3 grid((nx / 2 + 63) / 64, (ny / 2 + 3) / 4, nz / 2);
  mg_prolong_top_kernel<true><<<grid, dim3(64, 4), 0, s>>>(e, nullptr, u0, nx, ny, nz, per[0],
                                                           per[1], per[2]);
  return hipGetLastError();
}

hipError_t mg_prolong_add(double *q, const float *u0, int nx, int ny, int nz, const int per[3],
                          hipStream_t s) {
  if (nx % 2 || ny % 2 || nz % 2) return hipErrorInvalidValue;
  const dim3 grid((nx / 2 + 63) / 64, (ny / 2 + 3) / 4, nz / 2);
  mg_prolong_top_kernel<false><<<grid, dim3(64, 4), 0, s>>>(nullptr, q, u0, nx, ny, nz, per[0],
                                                            per[1], per[2]);
  return hipGetLastError();
}

hipError_t mg_seed_from_level1(const MgHierarchy &H, hipStream_t s) {
  if (H.levels < 2) return hipErrorInvalidValue;
  const MgGrid g = grid_of(H, 0);
  const int n0 = g.mx * g.my * g.mz;
  mg_zero_kernel<<<(n0 + 255) / 256, 256, 0, s>>>(H.u[0], n0);
  mg_prolong_kernel<<<blocks_for(n0 / 8), 256, 0, s>>>(H.u[0], H.u[1], g.mx, g.my, g.mz, g.px,
                                                       g.py, g.pz);
  return hipGetLastError();
}

hipError_t mg_solve(MgHierarchy &H, int cycles, int nu1, int nu2, hipStream_t s,
                    bool from_zero) {
  if (H.levels < 1) return hipErrorInvalidValue;
  if ((long long)H.m[0][0] * H.m[0][1] * H.m[0][2] >= (1LL << 31)) return hipErrorInvalidValue;
  const int n0 = H.m[0][0] * H.m[0][1] * H.m[0][2];
  if (!(H.per[0] && H.per[1] && H.per[2]) && n0 >= 2) {
    // With a mirrored axis the fine residual need not have zero mean (an
    // rhs the mirror cannot satisfy); only its zero-mean part is solvable
    // here.  On all-periodic grids the mean is zero up to rounding.  The
    // level-0 residual array is free: restriction forms residuals on the fly.
    // At most n0 / 2 partials: they fit the n0 floats of that array.
    double *part = reinterpret_cast<double *>(H.r[0]);
    const int nb = std::max(1, std::min(kMgMeanBlocks, n0 / 2));
    mg_sum_kernel<<<nb, 256, 0, s>>>(H.f[0], n0, part);
    mg_center_kernel<<<std::min(1024, (n0 + 255) / 256), 256, 0, s>>>(H.f[0], n0, part, nb);
  }
  hipError_t e = hipGetLastError();
  if (cycles < 1 && from_zero) e = clear_level(H, 0, s);
  for (int c = 0; c < cycles && e == hipSuccess; ++c)
    e = vcycle(H, 0, nu1, nu2, from_zero && c == 0, s);
  return e;
}

}  // namespace o3d
