// The coarse end of the multigrid cycle in one workgroup (gfx950): every
// level small enough runs from LDS, in FP64, interpreting the host-built
// cycle program.
#pragma once

#include <type_traits>

#include "hf_cycle.hpp"

namespace hf {

enum TailKind : uint8_t { T_SMOOTH = 0, T_RESTRICT = 1, T_PROLONG = 2 };
struct alignas(8) TailOp {
  uint8_t kind;
  uint8_t level;  // counted from the tail's first level
  uint8_t reverse;
  uint8_t retain;
  uint16_t sweeps;
  uint16_t pad;
};

// What bounds the tail is latency: a 2x2x2 coarsest level runs 48 dependent
// colour passes of a handful of cells, and every instruction that runs once
// is fetched cold.  So everything an op needs is laid out once per
// coefficient refresh in the order it is read (the blob below) and read
// through few dependent steps: the kernel copies the blob's head to LDS
// while it loads the first level's x and b, an op's geometry and the coarse
// levels' coefficients then come from LDS, a smoothing keeps its cells'
// coefficients and neighbour positions in registers, levels of up to 64
// cells are smoothed by one wavefront without workgroup barriers, the
// update's division by D runs on a stored reciprocal (tail_divide), and the
// code is kept short (one pass body for both colours, loops where unrolling
// saves nothing).  A launch of the V(2,2) tail of a 64^3 grid (8^3 and below)
// takes 18.8 us, of a 512x256x256 one (16x8x8 and below) 28.9 us, and a visit
// of the Chebyshev F-cycle on 64^3 27.1 us; reading coefficients, geometry
// and boundary modes where they are used took 28.3, 40.2 and 41.5 us.  A
// pass of the coarsest level takes 370 cycles (930 with its branches).
//
// Cells of a level are worked on in slot order: colour 0 in natural order,
// then colour 1, so that a colour pass keeps whole wavefronts busy; x, b and
// r in LDS stay in natural order.
//
// Blob: a TailGeo per level, then per level, coarsest first, its coefficients
// by slot (kTailCoefs arrays of `cells` doubles) and its tables by slot
// (kTailTables arrays of `cells` 16-bit values).
enum TailCoef : int {
  kTailD = 0,
  kTailXl,
  kTailXh,
  kTailYl,
  kTailYh,
  kTailZl,
  kTailZh,
  kTailInv,  // 1 / D, or 0 where tail_divide may not use it
  kTailVol,  // fluid volume (0 on solid cells)
  kTailCoefs
};
enum TailTable : int {
  kTailCell = 0,  // natural cell index
  kTailNb = 1,    // six neighbours (x-lo, x-hi, y-lo, ...): natural index
  kTailIjk = 7,   // i, j, k
  // prolongation, per axis: the two coarse planes' offsets in the coarse
  // level (the second kTailNone where one plane serves)
  kTailLow = 10,
  kTailHigh = 13,
  kTailTables = 16
};
// Dirichlet neighbour (reads +0), or no second coarse plane
constexpr uint16_t kTailNone = 0xffffu;

struct TailGeo {
  int nx, ny, nz, cells;
  int colour0;       // cells of colour 0
  int coarsen_mask;
  int fused;         // 0: an odd periodic extent (separated colour passes)
  int cheb;          // Chebyshev-Jacobi smoothing (else red-black)
  int work;          // offset (doubles) of x in LDS; b and r follow
  int image;         // offset (doubles) of the coefficients in the blob
  double volume;     // sum of fluid volumes
};
constexpr int kTailGeoDoubles = sizeof(TailGeo) / sizeof(double);
static_assert(kTailGeoDoubles == 6, "kTailOverhead below and tail_geo()");

constexpr int kTailThreads = 1024;
constexpr int kTailMaxCells = 3072;  // three cells per thread, at most
// (a level of at most 3072 cells has at most twelve levels below it, and an
// F-cycle through those takes fewer ops than this)
constexpr int kTailMaxLevels = 16;
constexpr int kTailMaxOps = 512;
constexpr int64_t kTailLdsBytes = 156 * 1024;
// LDS doubles beside x, b, r: slots 0 (+0) and 1 (spare), the geometry and
// the ops
constexpr int kTailSlots = 2;
constexpr int64_t kTailOverhead =
    kTailSlots + kTailMaxLevels * 6 + kTailMaxOps;
// what x, b and r of the tail levels may take together, 2730 cells (the
// coarsest alone must fit)
constexpr int64_t kTailWorkBytes = 64 * 1024;
static_assert(kTailWorkBytes + 8 * kTailOverhead <= kTailLdsBytes,
              "the geometry and the ops fit beside the largest work space");

// Doubles of one level's image.
__host__ __device__ constexpr int64_t tail_image_doubles(int64_t cells) {
  const int64_t n = kTailCoefs * cells + kTailTables / 4 * cells;
  return n + (n & 1);  // images start at even offsets (16-byte copies)
}

// Chebyshev-Jacobi stage factors of the tail's Chebyshev levels, stage s:
// direction d = pf[s] d + rf[s] (b - A x) / D (d = rf[0] (b - A x) / D at
// s = 0).  The host fills them with the recurrence of the grid levels.
constexpr int kTailChebStages = 16;
struct TailCheb {
  double rf[kTailChebStages];
  double pf[kTailChebStages];
};

// n / d correctly rounded, given y = 1 / d correctly rounded (or y = 0: the
// plain division): two Newton corrections of n y, each with its remainder
// exact in an FMA, the second of which rounds correctly (Markstein,
// "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990).  The remainders are exact while n and d stay away from
// the ends of the exponent range; elsewhere the division itself is taken.
// The five dependent operations replace the eleven of a division, on a chain
// that nothing else overlaps.
__device__ __forceinline__ double tail_reciprocal(double d) {
  return d >= 0x1p-100 && d <= 0x1p100 ? 1.0 / d : 0.0;
}

__device__ __forceinline__ double tail_divide(double n, double d, double y) {
  double q = n * y;
  q = fma(fma(-q, d, n), y, q);
  q = fma(fma(-q, d, n), y, q);
  q = n == 0.0 ? n : q;  // d > 0: the sign of zero is n's
  // 2^-900 <= |n| < 2^901 by its exponent field, or zero
  const uint32_t e = (static_cast<uint32_t>(__double2hiint(n)) >> 20) & 0x7ffu;
  const bool plain = (y == 0.0) | ((e - 123u > 1800u) & (n != 0.0));
  if (__builtin_expect(__any(plain), 0)) q = plain ? n / d : q;
  return q;
}

// Coefficients of every tail level into the blob, by slot (one block per 256
// slots of a level, blockIdx.y = level), and the levels' volumes into their
// geometry.
struct TailPack {
  Lv<double> L[kTailMaxLevels];
  double volume[kTailMaxLevels];
};

__global__ void k_tail_pack(TailPack a, double* blob) {
  const int level = blockIdx.y;
  TailGeo* geo = reinterpret_cast<TailGeo*>(blob) + level;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s == 0) geo->volume = a.volume[level];
  const int cells = geo->cells;
  if (s >= cells) return;
  const Lv<double>& L = a.L[level];
  double* out = blob + geo->image;
  const uint16_t* table =
      reinterpret_cast<const uint16_t*>(out + kTailCoefs * cells);
  const int c = table[kTailCell * cells + s];
  const int j = table[(kTailIjk + 1) * cells + s];
  const int k = table[(kTailIjk + 2) * cells + s];
  const StencilCoef<double> f = stencil_coef<double>(L, j, k, c);
  out[kTailD * cells + s] = f.d;
  out[kTailXl * cells + s] = f.xl;
  out[kTailXh * cells + s] = f.xh;
  out[kTailYl * cells + s] = f.yl;
  out[kTailYh * cells + s] = f.yh;
  out[kTailZl * cells + s] = f.zl;
  out[kTailZh * cells + s] = f.zh;
  out[kTailInv * cells + s] = tail_reciprocal(f.d);
  out[kTailVol * cells + s] = L.vol[c];
}

struct TailRun {
  const double* blob;
  double* x0;  // first level's x, b and fluid flags in memory
  const double* b0;
  const uint8_t* act0;
  int cells0;
  MeanRef mean;        // pending constant projection of b0 (at: null, none)
  int work;        // LDS doubles of x, b, r (and slots 0 and 1)
  int head;        // doubles of the blob copied to LDS
  int resident;    // first level whose image is in that head
  const TailOp* ops;
  int nops;
  int zero_x;      // x of the first level starts from zero
  int null_space;
  TailCheb cheb;
};

extern __shared__ double tail_lds[];

// Coefficient array `which` and table `which` of a level, slot s, from LDS
// or from memory.
struct TailImage {
  const double* memory;
  int lds;  // offset in LDS, or -1
  int cells;
  __device__ __forceinline__ double coef(int which, int s) const {
    return lds >= 0 ? tail_lds[lds + which * cells + s]
                    : memory[which * cells + s];
  }
  __device__ __forceinline__ int table(int which, int s) const {
    const int at = which * cells + s;
    return lds >= 0 ? reinterpret_cast<const uint16_t*>(
                          tail_lds + lds + kTailCoefs * cells)[at]
                    : reinterpret_cast<const uint16_t*>(
                          memory + kTailCoefs * cells)[at];
  }
};

__device__ __forceinline__ TailImage tail_image(const TailRun& a, int level,
                                                const TailGeo& g) {
  TailImage im;
  im.memory = a.blob + g.image;
  im.lds = level >= a.resident ? a.work + g.image : -1;
  im.cells = g.cells;
  return im;
}

// The geometry of a level from the LDS copy, in scalar registers.
__device__ __forceinline__ TailGeo tail_geo(const TailRun& a, int level) {
  const double* at = tail_lds + a.work + level * kTailGeoDoubles;
  const int* w = reinterpret_cast<const int*>(at);
  auto s = [w](int n) { return __builtin_amdgcn_readfirstlane(w[n]); };
  TailGeo g;
  g.nx = s(0);
  g.ny = s(1);
  g.nz = s(2);
  g.cells = s(3);
  g.colour0 = s(4);
  g.coarsen_mask = s(5);
  g.fused = s(6);
  g.cheb = s(7);
  g.work = s(8);
  g.image = s(9);
  g.volume = at[5];
  return g;
}

// Orders a pass's LDS accesses before the next one's.  One wavefront's
// accesses complete in order: its lanes only need the compiler to keep that
// order.
template <bool kOneWave>
__device__ __forceinline__ void tail_sync() {
  if constexpr (kOneWave) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// What a smoothing pass updates: red-black passes (src/solver_mg.cpp:
// 3149-3222), red-black passes from the values before the pass (the
// separated route of :3262-3307 on an odd periodic extent), or
// Chebyshev-Jacobi stages (:2916-3090).
enum TailMode : int { kTailRb = 0, kTailSeparated = 1, kTailCheb = 2 };

// Smoothing of one level, then the retained defect in r.  A thread owns kM
// slots, kTailThreads apart, with their x and b in registers; a pass has no
// branch: threads without a cell of the pass's colour store the x they hold
// (threads without a cell at all, into the spare slot 1 of LDS).  kOneWave:
// at most 64 cells, called by the first wavefront alone.
template <int kM, bool kOneWave, int kMode>
__device__ __forceinline__ void tail_smooth(const TailGeo& g,
                                            const TailImage& im,
                                            const TailOp& op,
                                            const TailCheb& cheb) {
  double d[kM], f[kM][6], inv[kM], dir[kM], x[kM], b[kM];
  int at[kM], nb[kM][6], colour[kM];
  // (the image's place is uniform: one branch, every load issued before any
  // is used)
  auto load = [&](const double* coef, const uint16_t* table) {
#pragma unroll
    for (int q = 0; q < kM; ++q) {
      const int s = static_cast<int>(threadIdx.x) + kTailThreads * q;
      colour[q] = s < g.colour0 ? 0 : 1;
      const int slot = s < g.cells ? s : 0;
      d[q] = coef[kTailD * g.cells + slot];
#pragma unroll
      for (int n = 0; n < 6; ++n) f[q][n] = coef[(kTailXl + n) * g.cells + slot];
      inv[q] = coef[kTailInv * g.cells + slot];
      at[q] = table[kTailCell * g.cells + slot];
#pragma unroll
      for (int n = 0; n < 6; ++n)
        nb[q][n] = table[(kTailNb + n) * g.cells + slot];
    }
  };
  if (im.lds >= 0)
    load(tail_lds + im.lds, reinterpret_cast<const uint16_t*>(
                                tail_lds + im.lds + kTailCoefs * g.cells));
  else
    load(im.memory, reinterpret_cast<const uint16_t*>(im.memory +
                                                      kTailCoefs * g.cells));
  const int bo = g.cells, ro = 2 * g.cells;
  bool mine[kM];
#pragma unroll
  for (int q = 0; q < kM; ++q) {
    mine[q] = static_cast<int>(threadIdx.x) + kTailThreads * q < g.cells;
    at[q] += g.work;
    x[q] = tail_lds[at[q]];
    b[q] = tail_lds[at[q] + bo];
    dir[q] = 0.0;
#pragma unroll
    for (int n = 0; n < 6; ++n)  // lds[0] = +0
      nb[q][n] = nb[q][n] == kTailNone ? 0 : g.work + nb[q][n];
  }
  // b - A x at an owned cell, A x in the reference order
  auto residual = [&](int q) -> double {
    double v = d[q] * x[q];
#pragma unroll
    for (int n = 0; n < 6; ++n) v -= f[q][n] * tail_lds[nb[q][n]];
    return b[q] - v;
  };
  auto store = [&]() {
#pragma unroll
    for (int q = 0; q < kM; ++q) tail_lds[mine[q] ? at[q] : 1] = x[q];
  };
  // wavefronts without a cell of the pass only keep step
  const int wave0 =
      __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) & ~63);
  auto busy = [&](int active) -> bool {
    if constexpr (kOneWave) return true;
    bool any = false;
#pragma unroll
    for (int q = 0; q < kM; ++q) {
      const int s = wave0 + kTailThreads * q;
      any = any || (active == 0 ? s < g.colour0
                                : s + kWave > g.colour0 && s < g.cells);
    }
    return any;
  };
  if constexpr (kMode == kTailCheb) {
#pragma unroll 1
    for (int stage = 0; stage < op.sweeps; ++stage) {
      const double rf = cheb.rf[stage], pf = cheb.pf[stage];
      const bool work = busy(0) || busy(1);
      if (work) {
#pragma unroll
        for (int q = 0; q < kM; ++q) {
          const double scaled = tail_divide(rf * residual(q), d[q], inv[q]);
          dir[q] = stage == 0 ? scaled : pf * dir[q] + scaled;
          x[q] = x[q] + dir[q];
        }
      }
      tail_sync<kOneWave>();
      if (work) store();
      tail_sync<kOneWave>();
    }
  } else {
    const double omega = 0.72;
#pragma unroll 1
    for (int pass = 0; pass < 2 * op.sweeps; ++pass) {
      const int active = (pass ^ op.reverse) & 1;
      const bool work = busy(active);
      if (work) {
#pragma unroll
        for (int q = 0; q < kM; ++q) {
          const double xn =
              x[q] + tail_divide(omega * residual(q), d[q], inv[q]);
          x[q] = colour[q] == active ? xn : x[q];
        }
        if constexpr (kMode == kTailRb) store();
      }
      if constexpr (kMode == kTailSeparated) {
        tail_sync<kOneWave>();
        if (work) store();
      }
      tail_sync<kOneWave>();
    }
  }
  if (op.retain) {
#pragma unroll
    for (int q = 0; q < kM; ++q)
      tail_lds[mine[q] ? at[q] + ro : 1] = residual(q);
  }
}

template <int kM, bool kOneWave>
__device__ __forceinline__ void tail_smooth_mode(const TailGeo& g,
                                                 const TailImage& im,
                                                 const TailOp& op,
                                                 const TailCheb& cheb) {
  if (g.cheb)
    tail_smooth<kM, kOneWave, kTailCheb>(g, im, op, cheb);
  else if (g.fused)
    tail_smooth<kM, kOneWave, kTailRb>(g, im, op, cheb);
  else
    tail_smooth<kM, kOneWave, kTailSeparated>(g, im, op, cheb);
}

// Restriction (src/solver_mg.cpp:3633-3720): coarse b = the children's r
// summed in dz, dy, dx order, coarse x = 0; with the constant null space the
// coarse b is projected (src/solver_mg.cpp:1412-1454).
__device__ __forceinline__ void tail_restrict(const TailGeo& F,
                                              const TailGeo& g,
                                              const TailImage& im,
                                              int null_space,
                                              double* scratch) {
  const int mx = F.coarsen_mask & 1, my = (F.coarsen_mask >> 1) & 1,
            mz = (F.coarsen_mask >> 2) & 1;
  const int fr = F.work + 2 * F.cells;
  double v = 0.0;
#pragma unroll 1
  for (int s = threadIdx.x; s < g.cells; s += kTailThreads) {
    const int c = im.table(kTailCell, s);
    const int xb = im.table(kTailIjk, s) << mx,
              yb = im.table(kTailIjk + 1, s) << my,
              zb = im.table(kTailIjk + 2, s) << mz;
    const bool x1 = mx && xb + 1 < F.nx, y1 = my && yb + 1 < F.ny,
               z1 = mz && zb + 1 < F.nz;
    const int p = fr + cell_index(F.nx, F.ny, xb, yb, zb);
    // a child that does not exist reads an existing one and adds +0
    const int ox = x1 ? 1 : 0, oy = y1 ? F.nx : 0, oz = z1 ? F.nx * F.ny : 0;
    double r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r[e] = tail_lds[p + (e & 1 ? ox : 0) + (e & 2 ? oy : 0) +
                      (e & 4 ? oz : 0)];
    double sum = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      sum += (!(e & 1) || x1) && (!(e & 2) || y1) && (!(e & 4) || z1) ? r[e]
                                                                      : 0.0;
    tail_lds[g.work + c] = 0.0;
    tail_lds[g.work + g.cells + c] = sum;
    if (null_space) v += im.coef(kTailVol, s) * sum;
  }
  if (!null_space) return;
  v = block_sum(v, scratch);
  if (threadIdx.x == 0) scratch[0] = v / g.volume;
  __syncthreads();
  const double mean = scratch[0];
#pragma unroll 1
  for (int s = threadIdx.x; s < g.cells; s += kTailThreads) {
    const int at = g.work + g.cells + im.table(kTailCell, s);
    tail_lds[at] = im.coef(kTailVol, s) > 0.0 ? tail_lds[at] - mean : 0.0;
  }
}

// Prolongation (src/solver_mg.cpp:3893-3993): x_f += sum of ((wx*wy)*wz)*x_c
// over the (az, ay, ax) corners; fine solids := 0.  The nearer plane of a
// cell weighs 3/4: the second one of an even cell, the first of an odd one.
__device__ __forceinline__ void tail_prolong(const TailGeo& F,
                                             const TailImage& im,
                                             const TailGeo& g) {
#pragma unroll 1
  for (int s = threadIdx.x; s < F.cells; s += kTailThreads) {
    int low[3], high[3];
    double wl[3], wh[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      low[a] = im.table(kTailLow + a, s);
      high[a] = im.table(kTailHigh + a, s);
      const bool odd = (im.table(kTailIjk + a, s) & 1) != 0;
      const bool one = high[a] == kTailNone;
      wl[a] = one ? 1.0 : (odd ? 0.75 : 0.25);
      wh[a] = odd ? 0.25 : 0.75;
    }
    const int at = F.work + im.table(kTailCell, s);
    const bool fluid = im.coef(kTailVol, s) > 0.0;
    // (a corner that does not exist repeats the first one and is left out)
    double x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      int p = g.work;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        p += ((e >> a) & 1) && high[a] != kTailNone ? high[a] : low[a];
      x[e] = tail_lds[p];
    }
    double value = 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      bool there = true;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        there = there && (!((e >> a) & 1) || high[a] != kTailNone);
      const double w = (e & 1 ? wh[0] : wl[0]) * (e & 2 ? wh[1] : wl[1]) *
                       (e & 4 ? wh[2] : wl[2]);
      if (there) value += w * x[e];
    }
    tail_lds[at] = fluid ? tail_lds[at] + value : 0.0;
  }
}

__global__ void __launch_bounds__(kTailThreads) k_tail(TailRun a) {
  __shared__ double scratch[16];
  const int tid = threadIdx.x;
  // ---- the blob's head and the first level's x and b into LDS, every load
  // independent of the others (a.work and a.head are even)
  const int work0 = kTailSlots;
  const double mean = mean_value<kTailThreads>(a.mean, scratch);
  struct alignas(16) Pair {
    double v[2];
  };
#pragma unroll 4
  for (int i = 2 * tid; i < a.head; i += 2 * kTailThreads)
    *reinterpret_cast<Pair*>(tail_lds + a.work + i) =
        *reinterpret_cast<const Pair*>(a.blob + i);
  const int ops_at = a.work + a.head;
  for (int i = tid; i < a.nops; i += kTailThreads)
    tail_lds[ops_at + i] = reinterpret_cast<const double*>(a.ops)[i];
  for (int c = tid; c < a.cells0; c += kTailThreads) {
    const double x = a.zero_x ? 0.0 : a.x0[c];
    double b = a.b0[c];
    if (a.mean.at != nullptr) b = a.act0[c] ? b - mean : 0.0;
    tail_lds[work0 + c] = x;
    tail_lds[work0 + a.cells0 + c] = b;
  }
  if (tid == 0) tail_lds[0] = 0.0;
  __syncthreads();
  for (int o = 0; o < a.nops; ++o) {
    TailOp op;
    {
      const uint32_t* w = reinterpret_cast<const uint32_t*>(
          tail_lds + ops_at + o);
      const uint32_t lo = __builtin_amdgcn_readfirstlane(w[0]);
      const uint32_t hi = __builtin_amdgcn_readfirstlane(w[1]);
      op.kind = static_cast<uint8_t>(lo);
      op.level = static_cast<uint8_t>(lo >> 8);
      op.reverse = static_cast<uint8_t>(lo >> 16);
      op.retain = static_cast<uint8_t>(lo >> 24);
      op.sweeps = static_cast<uint16_t>(hi);
    }
    const TailGeo g = tail_geo(a, op.level);
    const TailImage im = tail_image(a, op.level, g);
    if (op.kind == T_SMOOTH) {
      if (g.cells <= kWave) {
        if (tid < kWave) tail_smooth_mode<1, true>(g, im, op, a.cheb);
      } else if (g.cells <= kTailThreads) {
        tail_smooth_mode<1, false>(g, im, op, a.cheb);
      } else {
        tail_smooth_mode<kTailMaxCells / kTailThreads, false>(g, im, op,
                                                              a.cheb);
      }
    } else {
      const TailGeo cg = tail_geo(a, op.level + 1);
      if (op.kind == T_RESTRICT)
        tail_restrict(g, cg, tail_image(a, op.level + 1, cg), a.null_space,
                      scratch);
      else
        tail_prolong(g, im, cg);
    }
    __syncthreads();
  }
  for (int c = tid; c < a.cells0; c += kTailThreads)
    a.x0[c] = tail_lds[work0 + c];
}

}  // namespace hf
