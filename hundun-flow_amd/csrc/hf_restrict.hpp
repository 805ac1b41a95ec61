// Retained defect and restriction of a level in one pass (gfx950).
#pragma once

#include "hf_rows.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// The retained defect fused with the restriction that consumes it
// (src/solver_mg.cpp:3633-3720), on a level with even extents coarsened along
// every axis.  A lane owns a coarse cell: the pairs of two rows on two
// planes, whose defects, rounded to the fine storage type, it adds in the
// order of k_restrict (dz, dy, dx); the fine r is not stored.  Lanes take the
// cells of a coarse plane row after row and go through its two fine planes,
// carrying x and the z faces.  zero_x and partials as in k_restrict.
//
// kFirstStage: the level was to be smoothed by one Chebyshev-Jacobi stage
// from x = 0 (the pre-smoothing of a from-zero visit), which is not run:
// every x this kernel reads is formed from that cell's b and D as the stage
// stores it, st(0 + rf0 b / D), and the kernel also stores x of its own
// cells into xs (the stage's direction is dead: the next stage on the level
// starts a new recurrence).  A lane forms twelve of them for its four cells
// of a plane.
//
// What bounds it: the streams.  Against one fine cell per lane with the
// children's defects passed through LDS: 256^3 FP32 95 us against 107, 128^3
// 10.4 against 13.0, 512x256x256 186 against 204, 128^3 FP64 18.8 against
// 19.5, 64^3 FP64 4.9 against 5.4; with the first stage, which paid on FP32
// levels only below 2^20 cells (five divisions a cell), 256^3 FP32 112 against
// 139 for stage and defect apart, 512x256x256 216 against 265, FP64 403
// against 430; 64^3 FP64 6.2 against 7.5.
// ---------------------------------------------------------------------------
template <class Tf, class Tc>
struct DefectArgs {
  Lv<Tf> L;
  Bc bc;
  Lv<Tc> Cl;
  int zero_x;
  double* partials;
  typename Compute<Tf>::type rf0;
  Tf* xs;
  int per_plane;  // blocks of a coarse plane
};

// Wavefronts per SIMD that the registers are to leave room for.  Left to
// itself the compiler fits six FP64 ones, with few loads of each in flight;
// four with more are faster (64^3 4.9 us against 6.6, 128^3 18.8 against 22.3,
// 512x256x256 333 against 352).  In FP32 its own seven are as good.
template <class Tf>
constexpr int kDefectWavesLow = sizeof(Tf) == 8 ? 4 : 1;
template <class Tf>
constexpr int kDefectWavesHigh = sizeof(Tf) == 8 ? 4 : 8;

template <class Tf, class Tc, bool kFirstStage>
__global__ void __launch_bounds__(kBlock) __attribute__((
    amdgpu_waves_per_eu(kDefectWavesLow<Tf>, kDefectWavesHigh<Tf>)))
k_defect_restrict(DefectArgs<Tf, Tc> a) {
  using C = typename Compute<Tf>::type;
  using Cc = typename Compute<Tc>::type;
  struct alignas(2 * sizeof(Tf)) Stored {
    Tf v[2];
  };
  struct Two {
    C v[2];
  };
  __shared__ double scratch[16];
  const Lv<Tf>& L = a.L;
  const Lv<Tc>& Cl = a.Cl;
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int zb = lb / a.per_plane;
  const int q = (lb - zb * a.per_plane) * static_cast<int>(blockDim.x) +
                static_cast<int>(threadIdx.x);
  double pv = 0.0;
  if (q < Cl.nx * Cl.ny) {
    const int cj = q / Cl.nx;
    const int ci = q - cj * Cl.nx;
    const int i0 = 2 * ci, j0 = 2 * cj;
    const int plane = nx * ny;
    const int at = j0 * nx + i0;  // the first row's pair; the other at + nx
    const bool low_x = i0 == 0, high_x = i0 + 2 == nx;
    const bool low_y = j0 == 0, high_y = j0 + 2 == ny;
    const int xl_at = low_x ? at + nx - 1 : at - 1;
    const int xh_at = high_x ? at + 2 - nx : at + 2;
    const int yl_at = low_y ? at + (ny - 1) * nx : at - nx;
    const int yh_at = high_y ? i0 : at + 2 * nx;
    const int mxl = low_x ? a.bc.m[0] : 2, mxh = high_x ? a.bc.m[1] : 2;
    const int myl = low_y ? a.bc.m[2] : 2, myh = high_y ? a.bc.m[3] : 2;
    auto nb = [](int mode, C self, C v) -> C {
      return mode == 2 ? v : (mode == 1 ? self : C(0));
    };
    auto load = [](const Tf* p) -> Two {
      const Stored s = *reinterpret_cast<const Stored*>(p);
      return {{C(ld(s.v[0])), C(ld(s.v[1]))}};
    };
    auto first = [&](C b, C d) -> C {
      return C(ld(st<Tf>(C(0) + a.rf0 * b / d)));
    };
    // x of a pair, of a cell
    auto x2 = [&](int c) -> Two {
      if constexpr (kFirstStage) {
        const Two b = load(L.b + c), d = load(L.D + c);
        return {{first(b.v[0], d.v[0]), first(b.v[1], d.v[1])}};
      } else {
        return load(L.x + c);
      }
    };
    auto x1 = [&](int c) -> C {
      if constexpr (kFirstStage)
        return first(C(ld(L.b[c])), C(ld(L.D[c])));
      else
        return C(ld(L.x[c]));
    };
    const int k0 = 2 * zb;
    int c = k0 * plane + at;
    const int low_z = k0 > 0 ? c - plane : c + (nz - 1) * plane;
    Two xc[2], zl[2], fzl[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      xc[r] = x2(c + r * nx);
      zl[r] = x2(low_z + r * nx);
      fzl[r] = load(L.fz + c + r * nx);
      if (k0 == 0) {
        zl[r].v[0] = nb(a.bc.m[4], xc[r].v[0], zl[r].v[0]);
        zl[r].v[1] = nb(a.bc.m[4], xc[r].v[1], zl[r].v[1]);
      }
    }
    Cc sum = Cc(0);
#pragma unroll
    for (int dz = 0; dz < 2; ++dz) {
      const int kk = k0 + dz;
      const bool top = kk + 1 == nz;
      const int up = top ? at : c + plane;
      const Two below = x2(yl_at + kk * plane), beyond = x2(yh_at + kk * plane);
      Two zh[2], fzh[2], d[2], b[2], fy[3], fx[2];
      C fx2[2], xl[2], xh[2];
#pragma unroll
      for (int r = 0; r < 3; ++r)
        fy[r] = load(L.fy + (c + kk * nx + r * nx));
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        zh[r] = x2(up + r * nx);
        fzh[r] = load(L.fz + (c + plane + r * nx));
        d[r] = load(L.D + (c + r * nx));
        b[r] = load(L.b + (c + r * nx));
        const Tf* const face = L.fx + (c + kk * ny + j0 + r * (nx + 1));
        const RowsPair<Tf> f = rows_load(face);
        fx[r] = {{C(ld(f.v[0])), C(ld(f.v[1]))}};
        fx2[r] = C(ld(face[2]));
        xl[r] = x1(xl_at + kk * plane + r * nx);
        xh[r] = x1(xh_at + kk * plane + r * nx);
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        if constexpr (kFirstStage)
          *reinterpret_cast<Stored*>(a.xs + (c + r * nx)) = {
              {st<Tf>(xc[r].v[0]), st<Tf>(xc[r].v[1])}};
        if (top) {
          zh[r].v[0] = nb(a.bc.m[5], xc[r].v[0], zh[r].v[0]);
          zh[r].v[1] = nb(a.bc.m[5], xc[r].v[1], zh[r].v[1]);
        }
        const C nl[2] = {nb(mxl, xc[r].v[0], xl[r]), xc[r].v[0]};
        const C nh[2] = {xc[r].v[1], nb(mxh, xc[r].v[1], xh[r])};
        const C fl[2] = {fx[r].v[0], fx[r].v[1]};
        const C fh[2] = {fx[r].v[1], fx2[r]};
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const C self = xc[r].v[e];
          const C yl = r == 0 ? nb(myl, self, below.v[e]) : xc[0].v[e];
          const C yh = r == 0 ? xc[1].v[e] : nb(myh, self, beyond.v[e]);
          C v = d[r].v[e] * self;
          v -= fl[e] * nl[e];
          v -= fh[e] * nh[e];
          v -= fy[r].v[e] * yl;
          v -= fy[r + 1].v[e] * yh;
          v -= fzl[r].v[e] * zl[r].v[e];
          v -= fzh[r].v[e] * zh[r].v[e];
          sum += Cc(ld(st<Tf>(b[r].v[e] - v)));
        }
      }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        zl[r] = xc[r];
        xc[r] = zh[r];
        fzl[r] = fzh[r];
      }
      c += plane;
    }
    const int cc = zb * Cl.nx * Cl.ny + q;
    const Tc stored = st<Tc>(sum);
    Cl.b[cc] = stored;
    if (a.zero_x) Cl.x[cc] = st<Tc>(0.0);
    if (a.partials != nullptr)
      pv = Cl.vol[cc] * static_cast<double>(ld(stored));
  }
  if (a.partials != nullptr) {
    pv = block_sum(pv, scratch);
    if (threadIdx.x == 0) a.partials[lb] = pv;
  }
}

}  // namespace hf
