// Legs of the multigrid cycle on small levels (gfx950): everything a level
// does on the way down (smoothing, retained defect, restriction) or on the way
// up (prolongation, smoothing) in one launch.
#pragma once

#include <type_traits>

#include "hf_cycle.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// A block owns a box of cells of the level and works on the box grown by a
// halo of `h` cells: x of the whole region sits in LDS, the coefficients of a
// thread's two cells (a pair along z) in registers, and every pass of the
// smoothing runs over the region, the part of it that is right shrinking by
// one cell per pass that reads neighbours.  What remains after the last pass
// (and the defect, on the way down) is the block's own box.  The values are
// those of the separate launches bit for bit: each update reads the same
// operands in the same order, x is rounded to the storage type after every
// pass as a store and a load would, and cells that several blocks compute
// come out the same in each.
//
// What bounds it: launches.  A 32^3 level took six on the way down and five
// on the way up, 3.5 to 5 us each however little they did (two colours per
// sweep, the defect, the restriction).  One launch per leg computes a region
// many times its box, on CUs that are idle otherwise; a 12^3 region is small
// enough that a thread has two cells and the code stays short, which counts
// where every instruction is fetched cold.
//
// Boundaries: a position outside the domain holds 0 (Dirichlet; it is never
// updated) or is the wrapped cell (periodic, any number of periods); a
// Neumann face reads the cell itself, by an offset of 0 in place of the
// neighbour's.
// ---------------------------------------------------------------------------
constexpr int kLegE = 12;  // region extent
constexpr int kLegPlane = kLegE * kLegE;
// one pair per thread, in whole wavefronts: the last threads own none (three
// planes of LDS beyond the region keep their accesses inside)
constexpr int kLegThreads = (kLegPlane * kLegE / 2 + kWave - 1) / kWave * kWave;
constexpr int kLegHalo = 5;  // the widest halo a leg takes

// What a pass updates: one colour; one colour from the values before the pass
// (the separated route of src/solver_mg.cpp:3262-3307 on a level with an odd
// periodic extent, where two cells of one colour meet); every cell, from the
// values before the stage (Chebyshev-Jacobi, src/solver_mg.cpp:2916-3090),
// without or with an odd periodic extent.
enum LegMode : int {
  kLegRb = 0,
  kLegSeparated = 1,
  kLegCheb = 2,
  kLegChebOdd = 3
};

template <class T, class Tc>
struct LegArgs {
  Lv<T> F;
  Lv<Tc> Cl;
  Bc bc;
  T* xout;             // not F.x when F.x is read
  MeanRef mean;        // pending constant projection of b (at: null, none)
  int passes;          // colour passes, or Chebyshev stages
  int first;           // colour of the first pass
  int from_zero;       // way down: x starts from zero
  int h;               // halo
  int zero_x;          // way down: also store x = 0 on the coarse level
  int o;               // box extent (even)
  int gx, gy;          // boxes along x and y
  double* partials;    // way down: vol * b of the coarse cells; up: vol * x
  typename Compute<T>::type rf[kLegHalo];  // stage factors
  typename Compute<T>::type pf[kLegHalo];
};

// A region coordinate on an axis of n cells: the cell it is (wrapped on a
// periodic axis), or false outside the domain.
__device__ __forceinline__ bool leg_cell(int g, int n, bool periodic, int& w) {
  w = g;
  if (g >= 0 && g < n) return true;
  w = 0;
  if (!periodic) return false;
  w = g % n;
  if (w < 0) w += n;
  return true;
}

template <class T, class Tc, bool kDown, int kMode>
__global__ void __launch_bounds__(kLegThreads) k_leg(LegArgs<T, Tc> a) {
  using C = typename Compute<T>::type;
  using Cc = typename Compute<Tc>::type;
  __shared__ C xs[kLegPlane * (kLegE + 3)];
  __shared__ double scratch[16];
  const Lv<T>& L = a.F;
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int gxy = a.gx * a.gy;
  const int bz = lb / gxy;
  const int by = (lb - bz * gxy) / a.gx;
  const int bx = lb - bz * gxy - by * a.gx;
  const int tid = threadIdx.x;
  const int lx = tid % kLegE, ly = tid / kLegE % kLegE;
  const int lz = 2 * (tid / kLegPlane);
  const int gi = bx * a.o - a.h + lx, gj = by * a.o - a.h + ly,
            gk = bz * a.o - a.h + lz;
  const bool perx = a.bc.m[0] == 2, pery = a.bc.m[2] == 2,
             perz = a.bc.m[4] == 2;
  int wi, wj, wk[2];
  const bool in_x = leg_cell(gi, nx, perx, wi);
  const bool in_y = leg_cell(gj, ny, pery, wj);
  // LDS offsets of the neighbours (0: the cell itself, at a Neumann face or
  // past the region, where the value is not used)
  auto off = [](bool edge, bool wall, int step) -> int {
    return edge || wall ? 0 : step;
  };
  const int oxl = off(lx == 0, !perx && gi == 0 && a.bc.m[0] == 1, -1);
  const int oxh =
      off(lx == kLegE - 1, !perx && gi == nx - 1 && a.bc.m[1] == 1, 1);
  const int oyl = off(ly == 0, !pery && gj == 0 && a.bc.m[2] == 1, -kLegE);
  const int oyh = off(ly == kLegE - 1,
                      !pery && gj == ny - 1 && a.bc.m[3] == 1, kLegE);
  // Red-black: the pair is held colour 0 first (region coordinates have the
  // cells' parity: periodic extents are even), so that a pass works on one
  // slot; else slot q is cell q.
  const int flip = kMode == kLegRb ? (gi + gj + gk) & 1 : 0;

  // Way up: the column's corners in a coarse plane and their x, y weights.
  // The coarse cells that the region interpolates from (at most 8 along an
  // axis from `origin`, wrapped, or repeated past a wall) are read through
  // LDS; only where an odd periodic extent breaks the pairing of region
  // coordinates with coarse ones do the cells read them from memory.
  constexpr bool kStaged =
      !kDown && (kMode == kLegRb || kMode == kLegCheb);
  __shared__ C cs[kStaged ? 512 : 1];
  int corner[4] = {0, 0, 0, 0};
  bool there[4] = {true, true, true, true};
  C wxy[4];
  const int cplane = a.Cl.nx * a.Cl.ny;
  const int oz = ((bz * a.o - a.h) >> 1) - 1;
  // the lower coarse neighbour of region coordinate g, less the origin
  auto staged = [&](int g, int g0) -> int {
    return (g >> 1) - 1 + (g & 1) - ((g0 >> 1) - 1);
  };
  if constexpr (!kDown) {
    if constexpr (kStaged) {
      if (tid < 512) {
        auto wrap = [](int g, int n, bool periodic) -> int {
          int w;
          return leg_cell(g, n, periodic, w) ? w : (g < 0 ? 0 : n - 1);
        };
        const int cx = wrap(((bx * a.o - a.h) >> 1) - 1 + (tid & 7), a.Cl.nx,
                            perx);
        const int cy = wrap(((by * a.o - a.h) >> 1) - 1 + ((tid >> 3) & 7),
                            a.Cl.ny, pery);
        const int cz = wrap(oz + (tid >> 6), a.Cl.nz, perz);
        cs[tid] = C(ld(a.Cl.x[cell_index(a.Cl.nx, a.Cl.ny, cx, cy, cz)]));
      }
    }
    int xl, xr, xw, yl, yr, yw;
    interp(wi, 1, a.Cl.nx, perx, &xl, &xr, &xw);
    interp(wj, 1, a.Cl.ny, pery, &yl, &yr, &yw);
    const C wx = C(xw) * C(0.25), wy = C(yw) * C(0.25);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      corner[e] = kStaged ? staged(gi, bx * a.o - a.h) + (e & 1) +
                                8 * (staged(gj, by * a.o - a.h) + (e >> 1))
                          : wrapi(e & 2 ? yr : yl, a.Cl.ny) * a.Cl.nx +
                                wrapi(e & 1 ? xr : xl, a.Cl.nx);
      there[e] = (!(e & 1) || xl != xr) && (!(e & 2) || yl != yr);
      wxy[e] = (e & 1 ? wx : C(1) - wx) * (e & 2 ? wy : C(1) - wy);
    }
    if constexpr (kStaged) __syncthreads();
  }

  // ---- load the pair's coefficients, b and x
  C d[2], b[2], f[2][6];
  T braw[2];
  int at[2], ozl[2], ozh[2], colour[2];
  bool valid[2], fluid_b[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int z = q ^ flip;
    const bool in = leg_cell(gk + z, nz, perz, wk[q]) && in_x && in_y &&
                    lz < kLegE;
    valid[q] = in;
    colour[q] = (wi + wj + wk[q]) & 1;
    at[q] = lx + kLegE * ly + kLegPlane * (lz + z);
    ozl[q] = off(lz + z == 0, !perz && gk + z == 0 && a.bc.m[4] == 1,
                 -kLegPlane);
    ozh[q] = off(lz + z == kLegE - 1,
                 !perz && gk + z == nz - 1 && a.bc.m[5] == 1, kLegPlane);
    // (positions outside read cell 0: their values are not used)
    const int j = in ? wj : 0, k = in ? wk[q] : 0;
    const int c = in ? cell_index(nx, ny, wi, wj, wk[q]) : 0;
    const StencilCoef<C> s = stencil_coef<C>(L, j, k, c);
    d[q] = s.d;
    f[q][0] = s.xl;
    f[q][1] = s.xh;
    f[q][2] = s.yl;
    f[q][3] = s.yh;
    f[q][4] = s.zl;
    f[q][5] = s.zh;
    braw[q] = L.b[c];
    fluid_b[q] = a.mean.at != nullptr && L.act[c] != 0;
    C x = C(0);
    if (!kDown || !a.from_zero) x = C(ld(L.x[c]));
    if constexpr (!kDown) {
      // plus the interpolated correction, 0 on solid cells (k_prolong_z)
      const bool fluid = L.act[c] != 0;
      int zl, zr, zw;
      interp(k, 1, a.Cl.nz, perz, &zl, &zr, &zw);
      C low[4], high[4];
      if constexpr (kStaged) {
        // (a thread without a pair reads the first cells)
        const C* p = cs + (lz < kLegE ? 64 * staged(gk + z, bz * a.o - a.h)
                                      : 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          low[e] = p[corner[e]];
          high[e] = p[64 + corner[e]];
        }
      } else {
        const int pl = wrapi(zl, a.Cl.nz) * cplane,
                  pr = wrapi(zr, a.Cl.nz) * cplane;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          low[e] = C(ld(a.Cl.x[pl + corner[e]]));
          high[e] = C(ld(a.Cl.x[pr + corner[e]]));
        }
      }
      const C wh = C(zw) * C(0.25), wl = C(1) - wh;
      C value = C(0);
      // (a corner that does not exist repeats another one)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (there[e]) value += wxy[e] * wl * low[e];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (there[e] && zl != zr) value += wxy[e] * wh * high[e];
      x = fluid ? sw_round<T>(x + value) : C(0);
    }
    xs[at[q]] = in ? x : C(0);
  }
  const double mean = mean_value<kLegThreads>(a.mean, scratch);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    if (a.mean.at != nullptr) {
      const T projected = st<T>(static_cast<double>(ld(braw[q])) - mean);
      b[q] = fluid_b[q] ? C(ld(projected)) : C(0);
    } else {
      b[q] = C(ld(braw[q]));
    }
  }
  __syncthreads();

  // A x of slot q, in the reference order
  auto action = [&](int q, C xc) -> C {
    const C* p = xs + at[q];
    C v = d[q] * xc;
    v -= f[q][0] * p[oxl];
    v -= f[q][1] * p[oxh];
    v -= f[q][2] * p[oyl];
    v -= f[q][3] * p[oyh];
    v -= f[q][4] * p[ozl[q]];
    v -= f[q][5] * p[ozh[q]];
    return v;
  };
  const C omega = C(0.72);
  if constexpr (kMode == kLegRb) {
    auto colour_pass = [&](auto slot) {
      constexpr int q = decltype(slot)::value;
      const C xc = xs[at[q]];
      const C n = sw_round<T>(xc + omega * (b[q] - action(q, xc)) / d[q]);
      if (valid[q]) xs[at[q]] = n;
      __syncthreads();
    };
#pragma unroll 1
    for (int sweep = 0; 2 * sweep < a.passes; ++sweep) {
      // colours first, 1 - first
      if (a.first == 0) colour_pass(std::integral_constant<int, 0>{});
      colour_pass(std::integral_constant<int, 1>{});
      if (a.first != 0) colour_pass(std::integral_constant<int, 0>{});
    }
  } else {
    C dir[2] = {C(0), C(0)};
#pragma unroll 1
    for (int pass = 0; pass < a.passes; ++pass) {
      C xn[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const C xc = xs[at[q]];
        // (the separated route keeps A x at storage precision)
        const C v = action(q, xc);
        const C r = b[q] - (kMode == kLegSeparated ? sw_round<T>(v) : v);
        if constexpr (kMode == kLegCheb || kMode == kLegChebOdd) {
          const C scaled = a.rf[pass] * r / d[q];
          const C t = pass == 0 ? scaled : a.pf[pass] * dir[q] + scaled;
          dir[q] = sw_round<T>(t);
          xn[q] = sw_round<T>(xc + t);
        } else {
          xn[q] = colour[q] == ((a.first + pass) & 1)
                      ? sw_round<T>(xc + omega * r / d[q])
                      : xc;
        }
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (valid[q]) xs[at[q]] = xn[q];
      __syncthreads();
    }
  }

  // ---- the block's own box: x out, and the defect or the mean's terms
  double sum = 0.0;
  C defect[2];
  bool own[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int z = q ^ flip;
    own[q] = lx >= a.h && lx < a.h + a.o && ly >= a.h && ly < a.h + a.o &&
             lz + z >= a.h && lz + z < a.h + a.o && gi < nx && gj < ny &&
             gk + z < nz;
    const C xc = xs[at[q]];
    if constexpr (kDown) defect[q] = sw_round<T>(b[q] - action(q, xc));
    if (!own[q]) continue;
    const int c = cell_index(nx, ny, gi, gj, gk + z);
    const T stored = st<T>(xc);
    a.xout[c] = stored;
    if (!kDown && a.partials != nullptr && L.act[c])
      sum += L.vol[c] * static_cast<double>(ld(stored));
  }
  if constexpr (kDown) {
    // children summed in dz, dy, dx order, those outside the domain left out
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (own[q]) xs[at[q]] = defect[q];
    __syncthreads();
    const int o2 = a.o / 2;
    if (tid < o2 * o2 * o2) {
      const int ck = tid / (o2 * o2);
      const int cj = (tid - ck * o2 * o2) / o2;
      const int ci = tid - (ck * o2 + cj) * o2;
      const int fi = bx * a.o + 2 * ci, fj = by * a.o + 2 * cj,
                fk = bz * a.o + 2 * ck;
      if (fi < nx && fj < ny && fk < nz) {
        const C* p = xs + a.h + 2 * ci + kLegE * (a.h + 2 * cj) +
                     kLegPlane * (a.h + 2 * ck);
        Cc total = Cc(0);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int dx = e & 1, dy = (e >> 1) & 1, dz = e >> 2;
          if (fi + dx < nx && fj + dy < ny && fk + dz < nz)
            total += Cc(p[dx + kLegE * dy + kLegPlane * dz]);
        }
        const int cc =
            cell_index(a.Cl.nx, a.Cl.ny, fi >> 1, fj >> 1, fk >> 1);
        const Tc stored = st<Tc>(total);
        a.Cl.b[cc] = stored;
        if (a.zero_x) a.Cl.x[cc] = st<Tc>(0.0);
        if (a.partials != nullptr)
          sum = a.Cl.vol[cc] * static_cast<double>(ld(stored));
      }
    }
  }
  if (a.partials != nullptr) {
    sum = block_sum(sum, scratch);
    if (tid == 0) a.partials[lb] = sum;
  }
}

}  // namespace hf
