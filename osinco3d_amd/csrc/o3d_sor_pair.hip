// Red-black SOR, two iterations per launch (MI355X).
//
// The iterate and the rhs are in colour-split storage (o3d_sor.h): entry c of a
// row's two halves is the pair of nodes (2c, 2c + 1).  A launch reads one
// buffer and writes the other, so two iterations read the iterate and the rhs
// once and write the iterate once; a launch per colour, updating it in place,
// reads three of the four half arrays and writes one four times over.
//
// A block owns a tile of pairs x rows and a chunk of planes and computes the
// four half sweeps (red, black, red, black) on the tile plus a halo that
// loses one node per half sweep: 4 nodes in x and y, 4 planes below, 3 above.
// It marches in z: step t runs red on plane t, black on t - 1, red on t - 2
// and black on t - 3, each from the planes the previous half sweep has just
// left, so a plane lives for 8 steps in registers and meets memory twice.  A
// thread keeps its column of pairs on RY rows: z neighbours are its own
// registers, the x neighbour beside the pair comes from the next lane by DPP,
// and only the first and last row of each thread's RY pass through LDS (one
// barrier per step).  Ghost nodes (periodic images, mirror images) load from
// their image and evolve exactly as it does, so no boundary case is left in
// the march.  Every half sweep is the point update of sor_kernel in its
// operation order: the iterates are identical.
//
// The stop rule looks at dmax after every iteration, so the second iteration
// of a pair is a guess that the first does not end the solve or change omega.
// The next launch checks it; when it was wrong the source buffer still holds
// the iterate before the pair, and that launch runs the first iteration (or
// the pair with the right omegas) again.  With idyn = 1 that costs a launch per change
// of omega, of which solves have few: 400 iterations from omega 1.5 or 1.99 take 53.0
// to 53.2 us each at FP64 256^3 (52.8 with idyn = 0), 12.0 at 128^3 (11.6), 6.7 to 6.9
// at 64^3 (6.4).
//
// What bounds it: small grids by the plane step, 0.85 us (0.95 us with the
// tests of the first steps as branches inside the march, which kept the
// compiler from interleaving the half sweeps: 64^3 16.7 -> 15.2 us a launch);
// large ones by memory, at 4.3 TB/s (FP64, FP32 4.9) of the traffic that reaches the
// fabric, 1.16 (1.26) times the algorithmic bytes at 256^3 (the
// same kernel without its arithmetic takes as long), and there by the halos,
// which neighbouring tiles find in their XCD's L2 only while they march side by
// side.  So tiles are handed to the XCDs in
// contiguous runs (FP32 256^3: 90 us per launch in the plain order, 54 us so),
// one block runs per CU (FP64 256^3: 105 us with one block of 384 threads per
// CU, 131 us with two), loads are issued two planes ahead (three: no gain), and
// every second launch marches from the other end, towards what the last one
// left in the Infinity Cache (FP32 512x384x256 173 -> 156 us, FP64 320^3 199 ->
// 188).  Per two iterations, launches of
// one colour in place / this kernel: FP64 128^3 36.7 / 24.2 us
// (23 since the launch's maxima go by DPP), 256^3 186 / 106, 512x384x256 696 / 306;
// FP32 256^3 98 / 54, 384x256x128 93 / 38, 512x384x256 327 / 156 (the figures hold the
// host's share of a batch of launches, about 3 us).
#include <algorithm>
#include <utility>

#include "o3d_sor.h"

namespace o3d {

namespace {

// Lanes (pairs) per row, rows per thread, threads per block and LDS asked for
// beyond what the block uses (it sets how many blocks share a CU).
template <typename T, int SHAPE>
struct PairShape;
template <>
struct PairShape<double, 0> {
  static constexpr int LX = 32, RY = 2, NT = 384, PAD = 40000;
};
template <>
struct PairShape<double, 1> {
  static constexpr int LX = 32, RY = 2, NT = 512, PAD = 20000;
};
template <>
struct PairShape<float, 0> {
  static constexpr int LX = 32, RY = 2, NT = 768, PAD = 30000;
};
template <>
struct PairShape<float, 1> {
  static constexpr int LX = 64, RY = 4, NT = 512, PAD = 0;
};

constexpr int kPairRing = 8;  // planes t - 4 .. t + 2 and the one being loaded
constexpr int kPairSlots = 64, kPairStride = 16;  // dmax words per iteration
constexpr int kPairSets = 4;                      // launches in the dmax ring

template <int K>
struct PIC { static constexpr int value = K; };

// Image of node q of an axis of n nodes for q in [-4, n + 4] (n >= 6);
// positions further out belong to idle rows and lanes of a partial tile.
__device__ __forceinline__ int pair_ghost(int q, int n, int periodic) {
  if (q > n + 4) return n - 1;
  if (periodic) return q < 0 ? q + n : (q >= n ? q - n : q);
  return q < 0 ? -q : (q > n - 1 ? 2 * (n - 1) - q : q);
}

// xcd_tile for any number of blocks: block b runs on XCD b % 8, and each XCD
// gets one contiguous run of tiles (the grids here are seldom a multiple of 8,
// and the tiles' halos are half of what they load).
__device__ __forceinline__ int pair_tile(int b, int nb) {
  const int x = b & 7, q = nb >> 3, r = nb & 7;
  return x * q + min(x, r) + (b >> 3);
}

// The value of the lane before (DIR = 0) or after (DIR = 1) this one.
template <int DIR>
__device__ __forceinline__ float lane_next(float v) {
  constexpr int ctrl = DIR == 0 ? 0x138 : 0x130;  // wave_shr:1, wave_shl:1
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), ctrl, 0xf, 0xf, true));
}
template <int DIR>
__device__ __forceinline__ double lane_next(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  constexpr int ctrl = DIR == 0 ? 0x138 : 0x130;
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), ctrl, 0xf, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) |
                                          (unsigned)lo));
}

// max(m, |d|), m for a NaN d, as one instruction (fmax would first
// canonicalise its operands).
__device__ __forceinline__ float max_abs(float m, float d) {
  float r;
  asm("v_max_f32 %0, %1, |%2|" : "=v"(r) : "v"(m), "v"(d));
  return r;
}
__device__ __forceinline__ double max_abs(double m, double d) {
  double r;
  asm("v_max_f64 %0, %1, |%2|" : "=v"(r) : "v"(m), "v"(d));
  return r;
}

// num / A.  FP64 divides as the reference does: from the correctly rounded reciprocal
// invA, the quotient, its exact remainder by fma and the quotient corrected by it are
// correctly rounded (Markstein's theorem), as long as the remainder is a normal number
// or exact: for |num| above 2^-968.  Below, the last bit may differ from num / A; such
// a numerator is a sum of pressures and rhs all under 1e-291.  Zero, infinite and NaN
// numerators by div_fixup.  FP32 multiplies by 1 / A.
__device__ __forceinline__ double pair_div(double num, double A, double invA) {
  const double q = num * invA;
  const double r = __builtin_fma(-q, A, num);
  return __builtin_amdgcn_div_fixup(__builtin_fma(r, invA, q), A, num);
}
__device__ __forceinline__ float pair_div(float num, float, float invA) { return num * invA; }

template <typename T>
__device__ __forceinline__ T pload(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

template <typename T>
__device__ __forceinline__ void pstore(T v, __amdgpu_buffer_rsrc_t r, unsigned voff,
                                       unsigned soff) {
  if constexpr (sizeof(T) == 8) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), r, voff, soff, 0);
  } else {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
  }
}

template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pair_rsrc(const T *p, int n) {
  // At most INT_MAX bytes (sor_buffer_fits, checked by the launcher).
  return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0,
                                           (int)((long long)n * (long long)sizeof(T)), 0x00020000);
}

// What one launch does: iterations it0 .. it0 + n - 1 from buffer src.
struct PairStep {
  bool done;       // the solve is over: the launch does nothing
  int it0, n, src;
  double d_prev, om_a, om_b;
  // When done.
  int reason, sweeps, result;
  double dlast, omega;
};

// The reference's loop tail after iteration q with update d1 (the one before
// it d0): true when the solve ends; om becomes omega of iteration q + 1.
// Same rules and order as sor_decide_with of the single-iteration kernels.
template <typename T>
__device__ __forceinline__ bool pair_tail(int q, double d1, double d0, const SorPairArgs<T> &a,
                                          double &om, int &reason) {
  reason = -1;
  if (d1 < a.eps) reason = 0;
  else if (fabs(d0 - d1) < a.eps_stag) reason = 1;
  // No eps or stagnation exit inside the Gauss-Seidel opening.
  if (reason >= 0) return q > a.gs;
  if (q > 1 && a.idyn == 1) {
    if (d1 > d0) om = om * (2.0 - a.factor);
    else if (d1 < 0.1 * d0) om = fmin(om * a.factor, 2.0);
  }
  if (q + 1 > a.kmax) { reason = 2; return true; }
  return false;
}

// The next action from the previous launch's (P) and its two dmax values.
template <typename T>
__device__ __forceinline__ PairStep pair_decide(const SorSched &P, double da, double db,
                                                const SorPairArgs<T> &a) {
  PairStep s{};
  s.src = P.src;
  s.it0 = P.it0;
  s.om_a = P.om_a;
  s.d_prev = P.d_prev;
  if (P.n > 0) {
    double om = P.om_a;
    int reason;
    const bool stop = pair_tail(P.it0, da, P.it0 == 1 ? 1609.0 : P.d_prev, a, om, reason);
    if (stop && P.n == 2) {  // one iteration too many: the first alone
      s.n = 1;
      s.om_b = s.om_a;
      return s;
    }
    // The pair with its own omegas (bits: a NaN omega is no change either).
    if (!stop && P.n == 2 && __double_as_longlong(om) != __double_as_longlong(P.om_b)) {
      s.n = 2;
      s.om_b = om;
      return s;
    }
    int q = P.it0;
    double d = da;
    bool end = stop;
    if (!stop && P.n == 2) {
      ++q;
      d = db;
      end = pair_tail(q, db, da, a, om, reason);
    }
    s.src = 1 - P.src;
    if (end) {
      s.done = true;
      s.reason = reason;
      s.sweeps = q;
      s.result = s.src;
      s.dlast = d;
      s.omega = om;
      return s;
    }
    s.it0 = q + 1;
    s.om_a = om;
    s.d_prev = d;
  }
  s.om_b = s.om_a;
  s.n = s.it0 + 1 <= a.kmax ? 2 : 1;
  return s;
}

// What block 0 leaves of the launch's action: the result of the solve, or the
// next launch's view of this one and its cleared dmax slots.
template <typename T>
__device__ __forceinline__ void pair_record(const PairStep &s, const SorPairArgs<T> &a, int tid,
                                            int threads) {
  SorState *st = a.st;
  if (s.done) {
    if (tid == 0) {
      st->done = 1;
      st->reason = s.reason;
      st->exit_iter = s.reason == 2 ? a.kmax + 1 : s.sweeps;
      st->sweeps = s.sweeps;
      st->result = s.result;
      st->dmax_final = s.dlast;
      st->omega_final = s.omega;
    }
    return;
  }
  if (tid == 0) {
    st->sched[(a.launch + 1) & 1] = {s.it0, s.n, s.src, 0, s.d_prev, s.om_a, s.om_b};
    st->sweeps = s.it0 + s.n - 1;
  }
  unsigned long long *next =
      a.dslot + (size_t)((a.launch + 1) % kPairSets) * 2 * kPairSlots * kPairStride;
  for (int q = tid; q < 2 * kPairSlots; q += threads) next[(size_t)q * kPairStride] = 0ull;
}

// The block's dmax of both iterations into the launch's slots.
template <int NT, typename T>
__device__ __forceinline__ void pair_dmax(T ma, T mb, double (&scr)[2][NT / O3D_WAVE],
                                          const SorPairArgs<T> &a, int tid) {
  const double va = wave_max((double)ma), vb = wave_max((double)mb);
  if (tid % O3D_WAVE == 0) {
    scr[0][tid / O3D_WAVE] = va;
    scr[1][tid / O3D_WAVE] = vb;
  }
  __syncthreads();
  if (tid < 2) {
    double v = scr[tid][0];
#pragma unroll
    for (int q = 1; q < NT / O3D_WAVE; ++q) v = fmax(v, scr[tid][q]);
    if (v != 0.0)
      atomicMax(&a.dslot[((size_t)(a.launch % kPairSets) * 2 * kPairSlots +
                          (size_t)tid * kPairSlots + blockIdx.x % kPairSlots) * kPairStride],
                (unsigned long long)__double_as_longlong(v));
  }
}

template <int... K, typename F>
__device__ __forceinline__ bool pair_group(std::integer_sequence<int, K...>, int m, int last,
                                           F &&f) {
  return ((m + K <= last && (f(m + K, PIC<K>{}), true)) && ...);
}

// FLIP: the march runs through the planes backwards in an even number of them
// (virtual plane v is plane nz - 1 - v, of the other parity).
template <typename T, int SHAPE, int FLIP>
__global__ void __launch_bounds__((PairShape<T, SHAPE>::NT))
    sor_pair_kernel(const SorPairArgs<T> a) {
  using Shape = PairShape<T, SHAPE>;
  constexpr int LX = Shape::LX, RY = Shape::RY, NT = Shape::NT;
  constexpr int NG = NT / LX, TY = NG * RY, NR = kPairRing;
  static_assert(RY % 2 == 0 && TY % 2 == 0, "row parities are compile-time constants");
  // First and last row of every thread's RY: old black, new red, new black,
  // second red of the planes the next step reads; [0] the last rows, [1] the
  // first ones.  One guard group on each side.
  __shared__ T ex[2][4][2][NG + 2][LX];
  __shared__ double scr[2][NT / O3D_WAVE];
  const int tid = threadIdx.x;
  const int lane = tid % LX, g = tid / LX;
  SorState *st = a.st;
  const int over = st->done;
  const SorSched P = st->sched[a.launch & 1];
  const unsigned long long *ds =
      a.dslot + (size_t)((a.launch + kPairSets - 1) % kPairSets) * 2 * kPairSlots * kPairStride;
  const size_t wl = (size_t)__lane_id() * kPairStride;
  const unsigned long long dwa = ds[wl], dwb = ds[(size_t)kPairSlots * kPairStride + wl];

  const int nx = a.nx, ny = a.ny, nz = a.nz, hx = nx / 2;
  const int tile = pair_tile(blockIdx.x, gridDim.x);
  const int tix = tile % a.ntx, rr = tile / a.ntx;
  // Every second launch marches the other way: what the last one touched last
  // (and the Infinity Cache still holds) is read first.
  const bool rev = a.launch & 1;
  const int tiy = rr % a.nty, tiz = rev ? a.ntz - 1 - rr / a.nty : rr / a.nty;
  const int c0 = tix * (LX - 4), y0 = tiy * (TY - 8), z0 = tiz * a.zc;
  const int z1 = min(z0 + a.zc, nz);
  const T ox = T(a.ox), oy = T(a.oy), oz = T(a.oz), A = T(a.A), invA = T(a.invA);

  // Entries of the left and right node of this thread's pair, per row (they
  // differ only for mirror images, whose two nodes lie in two pairs).
  const int c = c0 - 2 + lane;
  const int eL = pair_ghost(2 * c, nx, a.per[0]) >> 1;
  const int eR = pair_ghost(2 * c + 1, nx, a.per[0]) >> 1;
  const int jb = y0 - 4 + g * RY;
  unsigned vL[RY], vR[RY];
  bool own[RY];
#pragma unroll
  for (int r = 0; r < RY; ++r) {
    const int row = hx * pair_ghost(jb + r, ny, a.per[1]);
    vL[r] = (unsigned)(row + eL) * (unsigned)sizeof(T);
    vR[r] = (unsigned)(row + eR) * (unsigned)sizeof(T);
    const int lr = g * RY + r;
    own[r] = lane >= 2 && lane < LX - 2 && c < hx && lr >= 4 && lr < TY - 4 && jb + r < ny;
  }
  const int n = nx * ny * nz;
  const unsigned planeB = (unsigned)(hx * ny) * (unsigned)sizeof(T);
  const unsigned halfB = planeB * (unsigned)nz;
  // The source buffer as long as no pair was taken back; the first loads go
  // out before the decision that may change it.
  int src = a.launch & 1;
  __amdgpu_buffer_rsrc_t rin = pair_rsrc(a.buf[src], n);
  const __amdgpu_buffer_rsrc_t rrh = pair_rsrc(a.rhs, n);

  // Ring slot of plane z0 - 4 + q is q % 8; z0 and the tile's first row are
  // even, so the parity of row + plane is (r + q) & 1.
  T R[NR][RY], B[NR][RY], fR[NR][RY], fB[NR][RY];
#pragma unroll
  for (int q = 0; q < NR; ++q)
#pragma unroll
    for (int r = 0; r < RY; ++r) R[q][r] = B[q][r] = fR[q][r] = fB[q][r] = T(0);
  // Byte offset of plane z0 - 4 + q (at most nz + 4; the image as in
  // pair_ghost, without branches).
  const int zs = a.per[2] ? 1 : -1, zlo = a.per[2] ? nz : 0, zhi = a.per[2] ? -nz : 2 * (nz - 1);
  auto zsoff = [&](int q) {
    const int z = z0 - 4 + q, im = zs * z + (z < 0 ? zlo : zhi);
    const int v = z < 0 || z >= nz ? im : z;
    return planeB * (unsigned)(rev ? nz - 1 - v : v);
  };
  auto load_p = [&](int q, auto SL) __attribute__((always_inline)) {
    constexpr int sl = decltype(SL)::value % NR;
    const unsigned so = zsoff(q);
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      const bool odd = (r + sl + FLIP) & 1;
      R[sl][r] = pload<T>(rin, odd ? vR[r] : vL[r], so);
      B[sl][r] = pload<T>(rin, odd ? vL[r] : vR[r], so + halfB);
    }
  };
  auto load_f = [&](int q, auto SL) __attribute__((always_inline)) {
    constexpr int sl = decltype(SL)::value % NR;
    const unsigned so = zsoff(q);
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      const bool odd = (r + sl + FLIP) & 1;
      fR[sl][r] = pload<T>(rrh, odd ? vR[r] : vL[r], so);
      fB[sl][r] = pload<T>(rrh, odd ? vL[r] : vR[r], so + halfB);
    }
  };
  T dA[RY], dB[RY];
#pragma unroll
  for (int r = 0; r < RY; ++r) dA[r] = dB[r] = T(0);

  // One half sweep of plane slot sl: X (this colour) from Y (the other), with
  // the rows beside the thread's own from LDS; CNT: the plane counts for dmax.
  auto half = [&](auto SL, auto COL, T(&X)[NR][RY], T(&Y)[NR][RY], const T(&F)[NR][RY], T lo,
                  T hi, T w, T w1, auto CNT, T(&dm)[RY]) __attribute__((always_inline)) {
    constexpr int sl = decltype(SL)::value % NR, sm = (sl + NR - 1) % NR, sp = (sl + 1) % NR;
    constexpr int col = decltype(COL)::value;
    T d[RY];
#pragma unroll
    for (int r = 0; r < RY; ++r) {
      // Node on the left of its pair: its other x neighbour is in the pair
      // before; on the right: in the pair after.
      const bool right = ((r + sl + col + FLIP) & 1) != 0;
      const T side = right ? lane_next<1>(Y[sl][r]) : lane_next<0>(Y[sl][r]);
      const T ym = r == 0 ? lo : Y[sl][r == 0 ? 0 : r - 1];
      const T yp = r == RY - 1 ? hi : Y[sl][r == RY - 1 ? r : r + 1];
      const T num = -ox * (side + Y[sl][r]) - oy * (ym + yp) - oz * (Y[sm][r] + Y[sp][r]) +
                    F[sl][r];
      const T pn = pair_div(num, A, invA);
      d[r] = pn - X[sl][r];
      X[sl][r] = w1 * X[sl][r] + w * pn;
    }
    if constexpr (decltype(CNT)::value) {
#pragma unroll
      for (int r = 0; r < RY; ++r) dm[r] = max_abs(dm[r], d[r]);
    }
  };
  // First and last rows of the four planes the step after step m reads.
  auto publish = [&](int b, auto K) __attribute__((always_inline)) {
    constexpr int k = decltype(K)::value;
    constexpr int s0 = (k + 2) % NR, s1 = (k + 1) % NR, s2 = k % NR, s3 = (k + NR - 1) % NR;
    ex[b][0][0][g + 1][lane] = B[s0][RY - 1];
    ex[b][0][1][g + 1][lane] = B[s0][0];
    ex[b][1][0][g + 1][lane] = R[s1][RY - 1];
    ex[b][1][1][g + 1][lane] = R[s1][0];
    ex[b][2][0][g + 1][lane] = B[s2][RY - 1];
    ex[b][2][1][g + 1][lane] = B[s2][0];
    ex[b][3][0][g + 1][lane] = R[s3][RY - 1];
    ex[b][3][1][g + 1][lane] = R[s3][0];
  };

  // The guard groups feed rows outside the tile's valid region only; they
  // hold zeros.
  for (int q = tid; q < 2 * 4 * 2 * 2 * LX; q += NT) {
    const int l = q % LX, e = q / LX;
    ex[e & 1][(e >> 1) & 3][(e >> 3) & 1][(e >> 4) ? NG + 1 : 0][l] = T(0);
  }
  load_p(0, PIC<0>{});
  load_p(1, PIC<1>{});
  load_f(1, PIC<1>{});
  load_p(2, PIC<2>{});

  if (over) return;
  PairStep s = pair_decide(P, wave_max(__longlong_as_double((long long)dwa)),
                           wave_max(__longlong_as_double((long long)dwb)), a);
  // Equal in every lane; in scalar registers, as the buffer descriptors and
  // the branches of the march need them.
  s.done = __builtin_amdgcn_readfirstlane((int)s.done) != 0;
  s.n = __builtin_amdgcn_readfirstlane(s.n);
  s.src = __builtin_amdgcn_readfirstlane(s.src);
  if (blockIdx.x == 0) pair_record(s, a, tid, NT);
  if (s.done) return;
  if (s.src != src) {
    src = s.src;
    rin = pair_rsrc(a.buf[src], n);
    load_p(0, PIC<0>{});
    load_p(1, PIC<1>{});
    load_p(2, PIC<2>{});
  }
  const __amdgpu_buffer_rsrc_t rout = pair_rsrc(a.buf[1 - src], n);
  const double oma = s.it0 <= a.gs ? 1.0 : s.om_a, omb = s.it0 + 1 <= a.gs ? 1.0 : s.om_b;
  const T wa = T(oma), wa1 = T(1.0 - oma), wb = T(omb), wb1 = T(1.0 - omb);
  const bool two = s.n == 2;
  publish(0, PIC<NR - 1>{});  // before step 0: its red reads plane slot 1's black
  __syncthreads();

  // Step m: t = z0 - 3 + m, slot of plane t is (m + 1) % 8.
  const int last = z1 - z0 + 5;
  // FIRST: steps 0 .. NR - 1, whose later half sweeps have not reached a plane
  // with valid inputs yet: those do not count for dmax and are not stored.  From
  // then on every half sweep updates nodes of the grid (the chunk's own or, at
  // its end, the next one's, whose updates are the same there).
  auto step = [&](int m, auto K, auto FIRST, auto TWO) __attribute__((always_inline)) {
    constexpr int k = decltype(K)::value;
    constexpr bool first = decltype(FIRST)::value != 0, two = decltype(TWO)::value != 0;
    load_p(m + 3, PIC<k + 3>{});
    load_f(m + 2, PIC<k + 2>{});
    const int b = m & 1;
    T lo[4], hi[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      lo[q] = ex[b][q][0][g][lane];
      hi[q] = ex[b][q][1][g + 2][lane];
    }
    half(PIC<k + 1>{}, PIC<0>{}, R, B, fR, lo[0], hi[0], wa, wa1, PIC<1>{}, dA);
    half(PIC<k>{}, PIC<1>{}, B, R, fB, lo[1], hi[1], wa, wa1,
         PIC<!first || k >= 2>{}, dA);
    if constexpr (two) {
      half(PIC<k + NR - 1>{}, PIC<0>{}, R, B, fR, lo[2], hi[2], wb, wb1,
           PIC<!first || k >= 4>{}, dB);
      half(PIC<k + NR - 2>{}, PIC<1>{}, B, R, fB, lo[3], hi[3], wb, wb1,
           PIC<!first || k >= 6>{}, dB);
    }
    publish(1 - b, K);
    if constexpr (!first || k >= 6) {
      constexpr int sl = (k + NR - 2) % NR;
      const unsigned so = planeB * (unsigned)(rev ? nz - 1 - (z0 - 6 + m) : z0 - 6 + m);
#pragma unroll
      for (int r = 0; r < RY; ++r)
        if (own[r]) {
          pstore(R[sl][r], rout, vL[r], so);
          pstore(B[sl][r], rout, vL[r], so + halfB);
        }
    }
    __syncthreads();
  };
  auto march = [&](auto TWO) __attribute__((always_inline)) {
    auto head = [&](int m, auto K) __attribute__((always_inline)) { step(m, K, PIC<1>{}, TWO); };
    auto body = [&](int m, auto K) __attribute__((always_inline)) { step(m, K, PIC<0>{}, TWO); };
    if (!pair_group(std::make_integer_sequence<int, NR>{}, 0, last, head)) return;
    for (int m = NR; pair_group(std::make_integer_sequence<int, NR>{}, m, last, body); m += NR) {
    }
  };
  if (two) march(PIC<1>{});
  else march(PIC<0>{});

  T ma = T(0), mb = T(0);
#pragma unroll
  for (int r = 0; r < RY; ++r)
    if (own[r]) {
      ma = dA[r] > ma ? dA[r] : ma;
      mb = dB[r] > mb ? dB[r] : mb;
    }
  pair_dmax<NT>(ma, mb, scr, a, tid);
}

// ------------------------------------------------------------- small grids
// The same two iterations of a tile at rest: a block holds its tile and the
// halo of 4 in registers, a thread a column of ZG planes of pairs, and every
// half sweep updates all of it.  Where the march's first and last steps outweigh
// its planes (a launch is never below 11 plane steps) this is the shorter one: a
// launch is one round of loads and four half sweeps, however few planes there are.
// Values, stop rule and records are sor_pair_kernel's.
//   Neighbours: z from the thread's own registers, across threads and in y from
// the colour's copy in LDS (one barrier per half sweep), x by DPP.  A wave holds
// four rows of one parity, so that the side of a pair its node lies on is the same
// in the whole wave; their LDS rows lie side by side (no bank conflicts).
//   Half sweep h updates the tile and 3 - h nodes around it; planes outside are
// left out, rows and lanes outside evolve unread.
//   What bounds it: one round of loads, the stop decision and the block maximum, then
// the vector units, 16 waves on a CU for 5 times the tile's own nodes.
// Per launch, march / this: FP64 32^3 11.2 / 9.0 us, 64^3 12.4 / 10.1; FP32 32^3 12.6 / 8.0, 64^3 11.4 / 8.6.  A second round of blocks doubles it
// (80^3 FP64 14.4 / 19): the line is one block per CU (tile_tiling).
template <int ZG>
struct TileShape {
  static constexpr int LX = 16, LY = 16, LZ = 4 * ZG, NT = 4 * LX * LY;
  static constexpr int OX = LX - 4, OY = LY - 8, OZ = LZ - 8;  // pairs, rows, planes
};

template <typename T, int ZG>
__global__ void __launch_bounds__((TileShape<ZG>::NT)) sor_tile_kernel(const SorPairArgs<T> a) {
  using S = TileShape<ZG>;
  constexpr int LX = S::LX, LY = S::LY, LZ = S::LZ, NT = S::NT;
  constexpr int PL = LX * LY;  // pairs of a plane
  static_assert(ZG >= 4 && ZG % 2 == 0, "the halo of 4 planes ends inside the outer groups");
  __shared__ T ex[2][LZ][PL];
  __shared__ double scr[2][NT / O3D_WAVE];
  const int tid = threadIdx.x;
  const int lane = tid % LX;
  // Rows of wave w of a group: parity w & 1, four of them from 8 (w >> 1) on.
  const int zg = __builtin_amdgcn_readfirstlane(tid / PL);
  const int w = __builtin_amdgcn_readfirstlane(tid / O3D_WAVE) & 3, par = w & 1;
  const int row = 8 * (w >> 1) + 2 * ((tid / LX) & 3) + par;
  SorState *st = a.st;
  const int over = st->done;
  const SorSched P = st->sched[a.launch & 1];
  const unsigned long long *ds =
      a.dslot + (size_t)((a.launch + kPairSets - 1) % kPairSets) * 2 * kPairSlots * kPairStride;
  const size_t wl = (size_t)__lane_id() * kPairStride;
  const unsigned long long dwa = ds[wl], dwb = ds[(size_t)kPairSlots * kPairStride + wl];

  const int nx = a.nx, ny = a.ny, nz = a.nz, hx = nx / 2;
  const int tile = pair_tile(blockIdx.x, gridDim.x);
  const int tix = tile % a.ntx, rr = tile / a.ntx;
  const int c0 = tix * S::OX, y0 = rr % a.nty * S::OY, z0 = rr / a.nty * S::OZ;
  const T ox = T(a.ox), oy = T(a.oy), oz = T(a.oz), A = T(a.A), invA = T(a.invA);

  const int c = c0 - 2 + lane, y = y0 - 4 + row;
  const int rowo = hx * pair_ghost(y, ny, a.per[1]);
  const int eL = pair_ghost(2 * c, nx, a.per[0]) >> 1, eR = pair_ghost(2 * c + 1, nx, a.per[0]) >> 1;
  const unsigned vL = (unsigned)(rowo + eL) * (unsigned)sizeof(T);
  const unsigned vR = (unsigned)(rowo + eR) * (unsigned)sizeof(T);
  const bool own = lane >= 2 && lane < LX - 2 && c < hx && row >= 4 && row < LY - 4 && y < ny;
  const int n = nx * ny * nz;
  const unsigned planeB = (unsigned)(hx * ny) * (unsigned)sizeof(T);
  const unsigned halfB = planeB * (unsigned)nz;
  int src = a.launch & 1;
  __amdgpu_buffer_rsrc_t rin = pair_rsrc(a.buf[src], n);
  const __amdgpu_buffer_rsrc_t rrh = pair_rsrc(a.rhs, n);
  // Planes zb + k, k < ZG.  The parity of row + plane of plane k is par + k: z0
  // and y0 are even.
  const int zb = z0 - 4 + zg * ZG;
  T R[ZG], B[ZG], fR[ZG], fB[ZG];
  const unsigned v0 = par ? vR : vL, v1 = par ? vL : vR;  // red, black node, even k
  auto load_p = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < ZG; ++k) {
      const unsigned so = planeB * (unsigned)pair_ghost(zb + k, nz, a.per[2]);
      R[k] = pload<T>(rin, k & 1 ? v1 : v0, so);
      B[k] = pload<T>(rin, k & 1 ? v0 : v1, so + halfB);
    }
  };
  load_p();
#pragma unroll
  for (int k = 0; k < ZG; ++k) {
    const unsigned so = planeB * (unsigned)pair_ghost(zb + k, nz, a.per[2]);
    fR[k] = pload<T>(rrh, k & 1 ? v1 : v0, so);
    fB[k] = pload<T>(rrh, k & 1 ? v0 : v1, so + halfB);
  }
  if (over) return;
  PairStep s = pair_decide(P, wave_max(__longlong_as_double((long long)dwa)),
                           wave_max(__longlong_as_double((long long)dwb)), a);
  s.done = __builtin_amdgcn_readfirstlane((int)s.done) != 0;
  s.n = __builtin_amdgcn_readfirstlane(s.n);
  s.src = __builtin_amdgcn_readfirstlane(s.src);
  if (blockIdx.x == 0) pair_record(s, a, tid, NT);
  if (s.done) return;
  if (s.src != src) {
    src = s.src;
    rin = pair_rsrc(a.buf[src], n);
    load_p();
  }
  const __amdgpu_buffer_rsrc_t rout = pair_rsrc(a.buf[1 - src], n);
  const double oma = s.it0 <= a.gs ? 1.0 : s.om_a, omb = s.it0 + 1 <= a.gs ? 1.0 : s.om_b;

  // LDS place of a row: the rows of one parity are contiguous.
  auto place = [&](int r) { return ((r & 1) * (LY / 2) + (r >> 1)) * LX + lane; };
  const int me = place(row), lo = place(max(row - 1, 0)), hi = place(min(row + 1, LY - 1));
  T dA = T(0), dB = T(0);
  // Half sweep H of this group (GRP 0: the lowest, 2: the highest, 1: between), of
  // rows of parity PAR: X (this colour) from Y (the other).
  auto half = [&](auto H, auto GRP, auto PAR, T(&X)[ZG], const T(&Y)[ZG], const T(&F)[ZG], T om,
                  T om1, T &dm) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value, grp = decltype(GRP)::value;
    constexpr int klo = grp == 0 ? 1 + h : 0, khi = grp == 2 ? ZG - 2 - h : ZG - 1;
    constexpr int olo = grp == 0 ? 4 : 0, ohi = grp == 2 ? ZG - 5 : ZG - 1;
    const T(*e)[PL] = ex[1 - (h & 1)];
    T ym[ZG], yp[ZG], zl = T(0), zh = T(0);
#pragma unroll
    for (int k = klo; k <= khi; ++k) {
      ym[k] = e[zg * ZG + k][lo];
      yp[k] = e[zg * ZG + k][hi];
    }
    if constexpr (klo == 0) zl = e[zg * ZG - 1][me];
    if constexpr (khi == ZG - 1) zh = e[zg * ZG + ZG][me];
#pragma unroll
    for (int k = klo; k <= khi; ++k) {
      const bool right = ((decltype(PAR)::value + k + h) & 1) != 0;
      const T side = right ? lane_next<1>(Y[k]) : lane_next<0>(Y[k]);
      const T zm = k == 0 ? zl : Y[k == 0 ? 0 : k - 1];
      const T zp = k == ZG - 1 ? zh : Y[k == ZG - 1 ? k : k + 1];
      const T num = -ox * (side + Y[k]) - oy * (ym[k] + yp[k]) - oz * (zm + zp) + F[k];
      const T pn = pair_div(num, A, invA);
      if (k >= olo && k <= ohi) dm = max_abs(dm, zb + k < nz ? pn - X[k] : T(0));
      X[k] = om1 * X[k] + om * pn;
      if constexpr (h < 3) ex[h & 1][zg * ZG + k][me] = X[k];
    }
  };
  auto sweep = [&](auto H, T om, T om1, T &dm) __attribute__((always_inline)) {
    auto go = [&](auto GRP) __attribute__((always_inline)) {
      constexpr int h = decltype(H)::value;
      if constexpr (h & 1) {
        if (par) half(H, GRP, PIC<1>{}, B, R, fB, om, om1, dm);
        else half(H, GRP, PIC<0>{}, B, R, fB, om, om1, dm);
      } else {
        if (par) half(H, GRP, PIC<1>{}, R, B, fR, om, om1, dm);
        else half(H, GRP, PIC<0>{}, R, B, fR, om, om1, dm);
      }
    };
    if (zg == 0) go(PIC<0>{});
    else if (zg == 3) go(PIC<2>{});
    else go(PIC<1>{});
    if constexpr (decltype(H)::value < 3) __syncthreads();
  };
#pragma unroll
  for (int k = 0; k < ZG; ++k) ex[1][zg * ZG + k][me] = B[k];
  __syncthreads();
  sweep(PIC<0>{}, T(oma), T(1.0 - oma), dA);
  sweep(PIC<1>{}, T(oma), T(1.0 - oma), dA);
  if (s.n == 2) {
    sweep(PIC<2>{}, T(omb), T(1.0 - omb), dB);
    sweep(PIC<3>{}, T(omb), T(1.0 - omb), dB);
  }
  if (own) {
#pragma unroll
    for (int k = 0; k < ZG; ++k) {
      const int q = zg * ZG + k;
      if (q < 4 || q >= LZ - 4 || zb + k >= nz) continue;
      const unsigned so = planeB * (unsigned)(zb + k);
      pstore(R[k], rout, vL, so);
      pstore(B[k], rout, vL, so + halfB);
    }
  }
  pair_dmax<NT>(own ? dA : T(0), own ? dB : T(0), scr, a, tid);
}

// Whole iterations of a grid that fits one block's LDS, as many as the solve
// takes (at most kBlockIters per launch, the state carried on in `sched`).  A
// launch of the march costs 11 us however small its grid; here an iteration is two
// barriers and the stop rule's block maximum.  A thread keeps PER pairs in
// registers and, of each, the LDS places of its neighbours (16 bits each); every
// half sweep reads the other colour from LDS, which bounds it together with the
// FP64 unit of the one CU.
// Same updates in the same order as sor_pair_kernel, and its stop rule after every
// iteration.
constexpr int kBlockNT = 1024, kBlockIters = 512;

template <typename T, int PER>
__global__ void __launch_bounds__(kBlockNT) sor_block_kernel(const SorPairArgs<T> a) {
  constexpr int NP = PER * kBlockNT;
  __shared__ T ex[2][NP];  // black, red
  __shared__ double scr[2][kBlockNT / O3D_WAVE];
  SorState *st = a.st;
  if (st->done) return;
  const SorSched P = st->sched[a.launch & 1];
  const int src = P.src;
  const int tid = threadIdx.x;
  const int nx = a.nx, ny = a.ny, nz = a.nz, hx = nx / 2, np = hx * ny * nz;
  const T ox = T(a.ox), oy = T(a.oy), oz = T(a.oz), A = T(a.A), invA = T(a.invA);
  const T *in = a.buf[src];
  T R[PER], B[PER], fR[PER], fB[PER];
  // Entries of the other colour: y - 1 | y + 1, z - 1 | z + 1, the x neighbour
  // outside the pair of the red | of the black node.
  unsigned oy2[PER], oz2[PER], os2[PER];
#pragma unroll
  for (int m = 0; m < PER; ++m) {
    const int p = tid + m * kBlockNT;
    R[m] = B[m] = fR[m] = fB[m] = T(0);
    oy2[m] = oz2[m] = os2[m] = 0;
    if (p >= np) continue;
    R[m] = in[p];
    B[m] = in[np + p];
    fR[m] = a.rhs[p];
    fB[m] = a.rhs[np + p];
    const int row = p / hx, c = p - row * hx, k = row / ny, j = row - k * ny;
    const int yb = c + hx * ny * k, zb = c + hx * j;
    oy2[m] = (unsigned)(yb + hx * pair_ghost(j - 1, ny, a.per[1])) |
             (unsigned)(yb + hx * pair_ghost(j + 1, ny, a.per[1])) << 16;
    oz2[m] = (unsigned)(zb + hx * ny * pair_ghost(k - 1, nz, a.per[2])) |
             (unsigned)(zb + hx * ny * pair_ghost(k + 1, nz, a.per[2])) << 16;
    const unsigned l = (unsigned)(hx * row + (pair_ghost(2 * c - 1, nx, a.per[0]) >> 1));
    const unsigned r = (unsigned)(hx * row + (pair_ghost(2 * c + 2, nx, a.per[0]) >> 1));
    os2[m] = (j + k) & 1 ? r | l << 16 : l | r << 16;
    ex[0][p] = B[m];
  }
  __syncthreads();
  T dm = T(0);
  // One colour, X, from the other one, Y (e: its LDS copy).
  auto half = [&](auto COL, T(&X)[PER], const T(&Y)[PER], const T(&F)[PER], T w, T w1)
      __attribute__((always_inline)) {
    constexpr int col = decltype(COL)::value;
    const T *e = ex[col];
    T *o = ex[1 - col];
#pragma unroll
    for (int m = 0; m < PER; ++m) {
      const int p = tid + m * kBlockNT;
      // Keeps the unpacked places out of registers of their own across iterations.
      asm("" : "+v"(oy2[m]), "+v"(oz2[m]), "+v"(os2[m]));
      const T side = e[col ? os2[m] >> 16 : os2[m] & 0xffffu];
      const T num = -ox * (side + Y[m]) - oy * (e[oy2[m] & 0xffffu] + e[oy2[m] >> 16]) -
                    oz * (e[oz2[m] & 0xffffu] + e[oz2[m] >> 16]) + F[m];
      const T pn = pair_div(num, A, invA);
      const T d = pn - X[m];
      X[m] = w1 * X[m] + w * pn;
      if (p < np) {
        dm = max_abs(dm, d);
        o[p] = X[m];
      }
    }
    __syncthreads();
  };
  int it = P.it0, reason = -1;
  double om = P.om_a, dprev = P.d_prev;
  bool end = false;
  for (int q = 0; q < kBlockIters; ++q) {
    const double w = it <= a.gs ? 1.0 : om;
    dm = T(0);
    half(PIC<0>{}, R, B, fR, T(w), T(1.0 - w));
    // The maximum of the last iteration's other buffer has been read.
    half(PIC<1>{}, B, R, fB, T(w), T(1.0 - w));
    const double v = wave_max((double)dm);
    if (tid % O3D_WAVE == 0) scr[q & 1][tid / O3D_WAVE] = v;
    __syncthreads();
    const double d = wave_max(scr[q & 1][tid % (kBlockNT / O3D_WAVE)]);
    end = pair_tail(it, d, it == 1 ? 1609.0 : dprev, a, om, reason);
    dprev = d;
    ++it;
    if (end) break;
  }
  T *out = a.buf[1 - src];
#pragma unroll
  for (int m = 0; m < PER; ++m) {
    const int p = tid + m * kBlockNT;
    if (p < np) {
      out[p] = R[m];
      out[np + p] = B[m];
    }
  }
  if (tid == 0) {
    st->sweeps = it - 1;
    if (end) {
      st->done = 1;
      st->reason = reason;
      st->exit_iter = reason == 2 ? a.kmax + 1 : it - 1;
      st->result = 1 - src;
      st->dmax_final = dprev;
      st->omega_final = om;
    } else {
      st->sched[(a.launch + 1) & 1] = {it, 0, 1 - src, 0, dprev, om, om};
    }
  }
}

// One colour of a Gauss-Seidel sweep (omega = 1) in place, the updates of
// sor_pair_kernel, with 64-bit addresses and no stop rule: the multigrid smoother of
// grids beyond what buffer descriptors address (2 GiB of FP32).  One thread per node of
// the colour; memory bounds it.
template <typename T>
__global__ void __launch_bounds__(256) gs_split_kernel(T *__restrict__ x,
                                                       const T *__restrict__ y,
                                                       const T *__restrict__ rhs, int colour,
                                                       int nx, int ny, int nz, int px, int py,
                                                       int pz, T ox, T oy, T oz, T A, T invA) {
  const int hx = nx / 2;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= (size_t)hx * ny * nz) return;
  const int row = (int)(e / hx), c = (int)(e - (size_t)row * hx);
  const int k = row / ny, j = row - k * ny;
  const bool right = ((j + k + colour) & 1) != 0;
  const size_t plane = (size_t)hx * ny, yb = plane * k + c, zb = (size_t)hx * j + c;
  const int out = pair_ghost(right ? 2 * c + 2 : 2 * c - 1, nx, px) >> 1;
  const T side = y[(size_t)row * hx + out];
  const T ym = y[yb + (size_t)hx * pair_ghost(j - 1, ny, py)];
  const T yp = y[yb + (size_t)hx * pair_ghost(j + 1, ny, py)];
  const T zm = y[zb + plane * pair_ghost(k - 1, nz, pz)];
  const T zp = y[zb + plane * pair_ghost(k + 1, nz, pz)];
  const T num = -ox * (side + y[e]) - oy * (ym + yp) - oz * (zm + zp) + rhs[e];
  x[e] = T(0) * x[e] + T(1) * pair_div(num, A, invA);
}

__global__ void __launch_bounds__(256) sor_pair_init_kernel(SorState *st, double omega,
                                                            unsigned long long *dslot,
                                                            int words) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < words) dslot[i] = 0ull;
  if (i == 0) {
    st->omega_final = omega;
    st->dmax_final = 0.0;
    st->done = 0;
    st->exit_iter = 0;
    st->reason = -1;
    st->sweeps = 0;
    st->result = 0;
    st->sched[0] = {1, 0, 0, 0, 1609.0, omega, omega};
  }
}

// Concurrent blocks of the kernel on this device.
template <typename T, int SHAPE>
int pair_slots() {
  static const int slots = [] {
    int per_cu = 0, dev = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, sor_pair_kernel<T, SHAPE, 0>, PairShape<T, SHAPE>::NT,
            PairShape<T, SHAPE>::PAD) != hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
      (void)hipGetLastError();
      return 256;
    }
    return std::max(1, per_cu * cus);
  }();
  return slots;
}

// Tiles of one shape: the even chunk of planes with the least
// rounds * (planes + 6 of the pipeline + 3 of prologue), the plane steps of the
// launch, which it returns.
template <typename T, int SHAPE>
double pair_tiling(SorPairArgs<T> &a) {
  using Shape = PairShape<T, SHAPE>;
  constexpr int OX = Shape::LX - 4, OY = Shape::NT / Shape::LX * Shape::RY - 8;
  a.shape = SHAPE;
  a.ntx = (a.nx / 2 + OX - 1) / OX;
  a.nty = (a.ny + OY - 1) / OY;
  const long long layer = (long long)a.ntx * a.nty;
  const int slots = pair_slots<T, SHAPE>();
  double best = 1e300;
  for (int zc = 2; zc < a.nz + 2; zc += 2) {
    const int ntz = (a.nz + zc - 1) / zc;
    const long long rounds = (layer * ntz + slots - 1) / slots;
    const double cost = (double)rounds * (zc + 9.0);
    if (cost < best - 1e-9) {
      best = cost;
      a.zc = zc;
      a.ntz = ntz;
    }
  }
  return best;
}

// Tiles of sor_tile_kernel where they are one round of blocks (its comment has the
// figures of both sides).
constexpr int kTileShape = 16;
template <typename T, int ZG>
bool tile_tiling(SorPairArgs<T> &a) {
  using S = TileShape<ZG>;
  const int ntx = (a.nx / 2 + S::OX - 1) / S::OX, nty = (a.ny + S::OY - 1) / S::OY,
            ntz = (a.nz + S::OZ - 1) / S::OZ;
  if ((long long)ntx * nty * ntz > 256) return false;
  a.shape = kTileShape + ZG;
  a.ntx = ntx;
  a.nty = nty;
  a.ntz = ntz;
  a.zc = S::OZ;
  return true;
}

template <typename T, int SHAPE>
void pair_launch(const SorPairArgs<T> &a, hipStream_t s) {
  using Shape = PairShape<T, SHAPE>;
  const int blocks = a.ntx * a.nty * a.ntz;
  if ((a.launch & 1) && a.nz % 2 == 0)
    sor_pair_kernel<T, SHAPE, 1><<<blocks, Shape::NT, Shape::PAD, s>>>(a);
  else
    sor_pair_kernel<T, SHAPE, 0><<<blocks, Shape::NT, Shape::PAD, s>>>(a);
}

}  // namespace

size_t sor_pair_slot_words() { return (size_t)kPairSets * 2 * kPairSlots * kPairStride; }

// Both buffers and the rhs stay in the 256 MB of the Infinity Cache.
template <typename T>
bool pair_cached(const SorPairArgs<T> &a) {
  return 3ll * (long long)sizeof(T) * a.nx * a.ny * a.nz <= (256ll << 20);
}

// FP64: 8 waves own 24 of 32 rows, 6 waves 16 of 24, for a plane step of 0.90 and
// 0.86 us, so 8 waves take fewer steps in most grids; beyond the cache the smaller
// tile's halos are found in L2 more often.  Per launch, 6 / 8 waves: 64^3 15.4 /
// 16.1 us, 128^3 26.0 / 24.2, 192^3 49.5 / 39.9, 208^3 59 / 49, then 256^3 106 /
// 114, 320^3 188 / 198, 512x384x256 306 / 378.
template <>
void sor_pair_tiling<double>(SorPairArgs<double> &a) {
  if (tile_tiling<double, 4>(a)) return;
  const double six = 0.86 * pair_tiling<double, 0>(a);
  if (!pair_cached(a)) return;
  SorPairArgs<double> b = a;
  if (0.90 * pair_tiling<double, 1>(b) < six) a = b;
}
// FP32: the narrow tile in the cache, the wide one (longer rows, fewer x halos)
// beyond.  Per
// launch, narrow / wide: 192^3 31.5 / 32.3 us, 256^3 53.8 / 64.4, 384x256x128
// 39.8 / 49.5, then 288^3 96.9 / 87.1, 320^3 114 / 107, 512x384x256 219 / 174.
template <>
void sor_pair_tiling<float>(SorPairArgs<float> &a) {
  if (tile_tiling<float, 4>(a)) return;
  if (pair_cached(a)) pair_tiling<float, 0>(a);
  else pair_tiling<float, 1>(a);
}

// Grids of sor_block_kernel, whose launch runs the whole solve: pairs per thread, 0
// for larger grids.  Per iteration, march / block: FP64 8^3 5.5 / 0.67 us, 16^3
// 5.6 / 1.55, 20x20x16 5.6 / 2.5; 8 pairs of doubles spill (24^3 5.6 / 5.3, without
// the launches' gaps).  FP32 16^3 5.4 / 0.45, 24x20x20 5.6 / 0.88, 24^3 5.9 / 2.1.
constexpr int kBlockShape = 8;
template <typename T>
static int block_per(const SorPairArgs<T> &a) {
  const long long pairs = (long long)(a.nx / 2) * a.ny * a.nz;
  for (int per = 2; per <= 32 / (int)sizeof(T); per *= 2)
    if (pairs <= (long long)per * kBlockNT) return per;
  return 0;
}
template <typename T>
bool sor_whole(SorPairArgs<T> &a) {
  if (!block_per(a)) return false;
  a.shape = kBlockShape;
  a.ntx = a.nty = a.ntz = 1;
  a.zc = 2;
  return true;
}

template <typename T>
hipError_t launch_sor_pair_init(const SorPairArgs<T> &a, double omega, hipStream_t s) {
  const int words = (int)sor_pair_slot_words();
  sor_pair_init_kernel<<<(words + 255) / 256, 256, 0, s>>>(a.st, omega, a.dslot, words);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_sor_pair(const SorPairArgs<T> &a, hipStream_t s) {
  if (a.nx % 2 != 0 || a.nx < 6 || a.ny < 6 || a.nz < 6 ||
      a.zc % 2 != 0 || !sor_buffer_fits<T, T>(a.nx, a.ny, a.nz))
    return hipErrorInvalidValue;
  if (a.shape == kBlockShape) {
    const int per = block_per(a);
    if (per == 2) sor_block_kernel<T, 2><<<1, kBlockNT, 0, s>>>(a);
    else if (per == 4) sor_block_kernel<T, 4><<<1, kBlockNT, 0, s>>>(a);
    else if (per == 0) return hipErrorInvalidValue;
    if constexpr (sizeof(T) == 4) {
      if (per == 8) sor_block_kernel<T, 8><<<1, kBlockNT, 0, s>>>(a);
    }
  } else if (a.shape == kTileShape + 4) {
    sor_tile_kernel<T, 4><<<a.ntx * a.nty * a.ntz, TileShape<4>::NT, 0, s>>>(a);
  } else if (a.shape == 1) pair_launch<T, 1>(a, s);
  else pair_launch<T, 0>(a, s);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_gs_split(const SorPairArgs<T> &a, T *field, int sweeps, hipStream_t s) {
  if (a.nx % 2 != 0 || a.nx < 6 || a.ny < 6 || a.nz < 6) return hipErrorInvalidValue;
  const size_t half = (size_t)(a.nx / 2) * a.ny * a.nz;
  T *c[2] = {field, field + half};
  const T *f[2] = {a.rhs, a.rhs + half};
  for (int q = 0; q < 2 * sweeps; ++q)
    gs_split_kernel<T><<<(unsigned)((half + 255) / 256), 256, 0, s>>>(
        c[q & 1], c[1 - (q & 1)], f[q & 1], q & 1, a.nx, a.ny, a.nz, a.per[0], a.per[1], a.per[2],
        T(a.ox), T(a.oy), T(a.oz), T(a.A), T(a.invA));
  return hipGetLastError();
}

template hipError_t launch_gs_split<float>(const SorPairArgs<float> &, float *, int, hipStream_t);
template bool sor_whole<float>(SorPairArgs<float> &);
template bool sor_whole<double>(SorPairArgs<double> &);
template hipError_t launch_sor_pair_init<float>(const SorPairArgs<float> &, double, hipStream_t);
template hipError_t launch_sor_pair_init<double>(const SorPairArgs<double> &, double,
                                                 hipStream_t);
template hipError_t launch_sor_pair<float>(const SorPairArgs<float> &, hipStream_t);
template hipError_t launch_sor_pair<double>(const SorPairArgs<double> &, hipStream_t);

}  // namespace o3d
