// Stencil passes over rows of any length (gfx950).
#pragma once

#include "hf_cycle.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// One pass over a level with the operator of every cell, or of every cell of
// a colour: A x with x . A x (kRowsOperator), b - A x (kRowsDefect), the true
// residual r = b - A x with r . r and, on request, the preconditioner's entry
// made from it (kRowsResidual; axpby(r, 1, b, -1, Ax),
// src/solver_krylov.cpp:1082-1091, and k_mg_entry: fluid ? r : 0 at level 0's
// storage precision, which the restart after an unconverged check reads), or the
// separated colour update of levels with an odd periodic extent, x_out =
// x + 0.72 (b - A x) / D on the colour's cells and x elsewhere
// (kRowsColour; src/solver_mg.cpp:3262-3307: every cell of the pass reads
// the x before it, also a neighbour of its own colour across a periodic
// seam, so x_out is another array).
//
// A lane owns the pair of cells (2m, 2m + 1) of a row on kPer planes; the
// pairs of a plane are numbered row after row and dealt to the wavefronts
// without regard to the rows, so no lane idles on a row that no tile width
// divides (201 cells leave a fifth of 64-wide tiles empty).  The last pair of
// an odd row is its last cell: such a lane reads the pair before and takes
// the high element (kLine, nx = 1: there is none, the elements are read one
// by one), so every access stays inside the row, and no access needs more
// than the alignment of one element.  All loads of the planes are issued
// before the first use.  Planes of at most half a block of pairs lie several
// to a block (kRowsPacked), one to a lane.
//
// What bounds it: the streams themselves.  A x, FP64, against one cell per
// lane in 64-wide tiles: 201x149x97 22.3 us against 29.5, 143x101x75 10.6
// against 14.4, 300x180x140 73.8 against 91; pairs in tiles of whole rows
// (k_fg_stencil2) take 80 there, 166 against 176 at 256^3.  A colour pass at
// 143x101x75 in FP32: 7.1 us against 14.2 for A x of every cell and the
// update as launches of their own; the true residual and its entry at
// 512x256x256 442 us against 466.
// ---------------------------------------------------------------------------
constexpr int kRowsOperator = 0, kRowsDefect = 1, kRowsColour = 2,
              kRowsResidual = 3;

// The pair at p, aligned as one element.
template <class T>
struct RowsPair {
  T v[2];
};
template <class T>
__device__ __forceinline__ RowsPair<T> rows_load(const T* p) {
  if constexpr (sizeof(T) == 2) {
    return {p[0], p[1]};
  } else {
    typedef T Two __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const Two t = *reinterpret_cast<const Two*>(p);
    return {t[0], t[1]};
  }
}
template <class T>
__device__ __forceinline__ void rows_store(T* p, T lo, T hi) {
  if constexpr (sizeof(T) == 2) {
    p[0] = lo;
    p[1] = hi;
  } else {
    typedef T Two __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    *reinterpret_cast<Two*>(p) = Two{lo, hi};
  }
}

template <class T, class Te>
struct RowsArgs {
  Lv<T> L;
  Bc bc;
  const T* x;
  T* out;
  // block sums: of x . A x (kRowsOperator; may be null); of r . r, then, each
  // `stride` further, vol * entry over the fluid cells (proj) and b . b
  // (with_bb; kRowsResidual)
  double* partials;
  int stride, proj, with_bb;
  const uint8_t* act;  // with entry
  Widths w;
  Te* entry;           // null: not made
  int colour;        // kRowsColour
  int pairs;         // of a row: (nx + 1) / 2
  int per_plane;     // blocks of a plane
  int packed;        // planes side by side in a block (then per_plane = 1)
};

// Planes of many pairs; planes of few, side by side in a block; rows of one
// cell (either).
constexpr int kRowsWide = 0, kRowsPacked = 1, kRowsLine = 2;

template <class T, int kMode, int kPer, int kPlane, class Te = T>
__global__ void __launch_bounds__(kBlock) k_rows(RowsArgs<T, Te> a) {
  using C = typename Compute<T>::type;
  constexpr bool kLine = kPlane == kRowsLine;
  __shared__ double scratch[16];
  const Lv<T>& L = a.L;
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  int zb, q;
  if (kPlane != kRowsWide && a.packed > 1) {
    const int lanes = a.pairs * ny;
    const int side = static_cast<int>(threadIdx.x) / lanes;
    zb = lb * a.packed + side;
    q = side < a.packed && static_cast<uint32_t>(zb) <=
                                static_cast<uint32_t>((nz - 1) / kPer)
            ? static_cast<int>(threadIdx.x) - side * lanes
            : lanes;  // (no pair)
  } else {
    zb = lb / a.per_plane;
    q = (lb - zb * a.per_plane) * kBlock + static_cast<int>(threadIdx.x);
  }
  double dot = 0.0, mean = 0.0, bb = 0.0;
  if (q < a.pairs * ny) {
    const int j = q / a.pairs;
    const int i0 = 2 * (q - j * a.pairs);
    const int plane = nx * ny;
    const int k0 = zb * kPer;
    const bool single = i0 + 1 == nx;
    const int at = j * nx + i0;
    const int lo = single ? at - 1 : at;  // the pair that the lane reads
    const bool low_x = i0 == 0, high_x = i0 + 2 >= nx;
    const bool low_y = j == 0, high_y = j + 1 == ny;
    // neighbours along the row and the rows beside it; across a boundary the
    // wrapped cell, used where the boundary is periodic
    const int xl_at = low_x ? at + nx - 1 : at - 1;
    const int xh_at = high_x ? j * nx : at + 2;
    const int yl_at = low_y ? lo + (ny - 1) * nx : lo - nx;
    const int yh_at = high_y ? lo - (ny - 1) * nx : lo + nx;
    const int mxl = low_x ? a.bc.m[0] : 2, mxh = high_x ? a.bc.m[1] : 2;
    const int myl = low_y ? a.bc.m[2] : 2, myh = high_y ? a.bc.m[3] : 2;
    auto nb = [](int mode, C self, C v) -> C {
      return mode == 2 ? v : (mode == 1 ? self : C(0));
    };
    auto pair = [&](const T* p) -> RowsPair<C> {
      if constexpr (kLine) return {C(ld(p[1])), C(ld(p[1]))};
      const RowsPair<T> r = rows_load(p);
      const C hi = C(ld(r.v[1]));
      return {single ? hi : C(ld(r.v[0])), hi};
    };
    // a plane of the level: wrapped below and above (plane 0 or nz - 1 where
    // a last block has no such plane)
    auto plane_at = [&](int k) -> int {
      const int w = k < 0 ? nz - 1 : (k >= nz ? k - nz : k);
      return min(w, nz - 1);
    };
    RowsPair<C> xp[kPer + 2], fz[kPer + 1], yl[kPer], yh[kPer], fyl[kPer],
        fyh[kPer], d[kPer], b[kPer], fx[kPer];
    C fx2[kPer], xl[kPer], xh[kPer];
    bool fluid[kPer][2];
    double wxy[2] = {0.0, 0.0};
    if (kMode == kRowsResidual && a.entry != nullptr) {
      wxy[0] = a.w.x[i0] * a.w.y[j];
      wxy[1] = a.w.x[single ? i0 : i0 + 1] * a.w.y[j];
    }
#pragma unroll
    for (int u = 0; u < kPer + 2; ++u)
      xp[u] = pair(a.x + (plane_at(k0 - 1 + u) * plane + lo));
#pragma unroll
    for (int u = 0; u < kPer + 1; ++u)
      fz[u] = pair(L.fz + (min(k0 + u, nz) * plane + lo));
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = min(k0 + u, nz - 1);
      const int c = k * plane;
      d[u] = pair(L.D + (c + lo));
      if constexpr (kMode != kRowsOperator) b[u] = pair(L.b + (c + lo));
      fyl[u] = pair(L.fy + (c + k * nx + lo));
      fyh[u] = pair(L.fy + (c + k * nx + nx + lo));
      const T* const face = L.fx + (c + k * ny + j + at);
      const RowsPair<T> f = rows_load(face);
      fx[u] = {C(ld(f.v[0])), C(ld(f.v[1]))};
      fx2[u] = C(ld(face[single ? 1 : 2]));
      yl[u] = pair(a.x + (c + yl_at));
      yh[u] = pair(a.x + (c + yh_at));
      xl[u] = C(ld(a.x[c + xl_at]));
      xh[u] = C(ld(a.x[c + xh_at]));
      if (kMode == kRowsResidual && a.entry != nullptr) {
        fluid[u][0] = a.act[c + at] != 0;
        fluid[u][1] = a.act[c + at + (single ? 0 : 1)] != 0;
      }
    }
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const int k = k0 + u;
      if (k >= nz) break;
      const int mzl = k == 0 ? a.bc.m[4] : 2, mzh = k + 1 == nz ? a.bc.m[5] : 2;
      const C x0 = xp[u + 1].v[0], x1 = xp[u + 1].v[1];
      // beside the pair: of an odd row's last cell, the high neighbour
      const C low = nb(mxl, x0, xl[u]);
      const C high = nb(mxh, single ? x0 : x1, xh[u]);
      // the operator of one cell: its element of every pair through `of`
      auto apply = [&](C xc, C nl, C nh, C fl, C fh, auto of) -> C {
        C v = of(d[u]) * xc;
        v -= fl * nl;
        v -= fh * nh;
        v -= of(fyl[u]) * nb(myl, xc, of(yl[u]));
        v -= of(fyh[u]) * nb(myh, xc, of(yh[u]));
        v -= of(fz[u]) * nb(mzl, xc, of(xp[u]));
        v -= of(fz[u + 1]) * nb(mzh, xc, of(xp[u + 2]));
        return v;
      };
      T o[2];
      if constexpr (kMode == kRowsColour) {
        // one cell of the pair has the colour
        const bool second = ((a.colour + j + k) & 1) != 0;
        const int second_ = second ? 1 : 0;
        auto pick = [second_](const RowsPair<C>& p) -> C {
          const C lo = p.v[0], hi = p.v[1];  // (values: registers)
          return second_ ? hi : lo;
        };
        const C xc = pick(xp[u + 1]);
        const C v = apply(xc, second_ ? x0 : low,
                          second_ || single ? high : x1, pick(fx[u]),
                          pick({fx[u].v[1], fx2[u]}), pick);
        // (A x is rounded to the storage type, as where it is stored)
        const C omega = C(0.72);
        const T n = st<T>(xc + omega * (pick(b[u]) - C(ld(st<T>(v)))) /
                               pick(d[u]));
        o[0] = second ? st<T>(x0) : n;
        o[1] = second ? n : st<T>(x1);
      } else {
        const C v0 = apply(x0, low, single ? high : x1, fx[u].v[0],
                           fx[u].v[1],
                           [](const RowsPair<C>& p) { return p.v[0]; });
        const C v1 = apply(x1, x0, high, fx[u].v[1], fx2[u],
                           [](const RowsPair<C>& p) { return p.v[1]; });
        if constexpr (kMode == kRowsOperator) {
          dot += static_cast<double>(x0) * static_cast<double>(v0);
          if (!single) dot += static_cast<double>(x1) * static_cast<double>(v1);
          o[0] = st<T>(v0);
          o[1] = st<T>(v1);
        } else {
          o[0] = st<T>(b[u].v[0] - v0);
          o[1] = st<T>(b[u].v[1] - v1);
        }
        if constexpr (kMode == kRowsResidual) {
          Te made[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            if (e == 1 && single) break;
            dot += o[e] * o[e];
            bb += b[u].v[e] * b[u].v[e];
            if (a.entry == nullptr) continue;
            made[e] = fluid[u][e] ? st<Te>(o[e]) : st<Te>(0.0);
            if (fluid[u][e])
              mean += wxy[e] * a.w.z[k] * static_cast<double>(ld(made[e]));
          }
          if (a.entry != nullptr) {
            Te* const entry = a.entry + (k * plane + at);
            if (single)
              *entry = made[0];
            else
              rows_store(entry, made[0], made[1]);
          }
        }
      }
      T* const out = a.out + (k * plane + at);
      if (single)
        *out = o[0];
      else
        rows_store(out, o[0], o[1]);
    }
  }
  if constexpr (kMode == kRowsOperator || kMode == kRowsResidual) {
    if (a.partials == nullptr) return;
    dot = block_sum(dot, scratch);
    if (threadIdx.x == 0) a.partials[lb] = dot;
  }
  if constexpr (kMode == kRowsResidual) {
    if (a.proj) {
      mean = block_sum(mean, scratch);
      if (threadIdx.x == 0) a.partials[lb + a.stride] = mean;
    }
    if (a.with_bb) {
      bb = block_sum(bb, scratch);
      if (threadIdx.x == 0) a.partials[lb + 2 * a.stride] = bb;
    }
  }
}

}  // namespace hf
