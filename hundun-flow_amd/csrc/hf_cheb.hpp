// Two Chebyshev-Jacobi stages of a large level in one pass (gfx950).
#pragma once

#include <limits.h>

#include <type_traits>

#include "hf_cycle.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// A block owns a tile of columns and marches through the planes of a z-chunk;
// at step k the first stage is made on plane k and the second on plane k - 1,
// so every array of the level is read once and x written once, where a launch
// per stage (k_cheb_stage2) reads them twice and carries the direction
// through memory.  The region is the tile and a halo of two cells; a cell
// that several blocks compute comes out the same in each, and the result
// equals two launches bit for bit (the direction between the stages is
// rounded to the storage type, as where it is stored).
//
// A lane owns a pair of cells of a row; the planes above and below are its
// own registers, and the lateral neighbours of x on plane k and of the first
// stage's x on plane k - 1 lie in LDS, written a step ahead: one barrier per
// step.  The loads of a step are issued a step before.
//
// What bounds it: the streams with their halos (a block is 1024 threads, one
// per CU, and a step about 2.5 us).  Two stages, against two k_cheb_stage2
// launches: 256^3 FP32 137 us against 234, FP64 251 against 443; 160^3 31
// against 52 and 51 against 114; 512x256x256 276 against 451 and 498 against
// 854; 128^3 22.8 against 22.7 and 30.7 against 44.6.
//
// Boundaries: a position outside the domain holds 0 (Dirichlet; never
// updated) or is the wrapped cell (periodic); on a Neumann face the neighbour
// is the cell itself.
// ---------------------------------------------------------------------------
constexpr int kChCols = 64;  // region columns: 32 pairs
constexpr int kChHalo = 2;
constexpr int kChOutX = kChCols - 2 * kChHalo;
// rows of the region, one per 32 lanes
template <class T>
constexpr int kChRows = std::is_same<T, double>::value ? 16 : 32;
template <class T>
constexpr int kChThreads = kChRows<T> * 32;
template <class T>
constexpr int kChOutY = kChRows<T> - 2 * kChHalo;

template <class T>
struct ChebMarchArgs {
  Lv<T> L;
  Bc bc;
  T* xout;
  // the stages' factors: x += pf d + rf (b - A x) / D (pf = 0 in the first)
  typename Compute<T>::type rf1, rf2, pf2;
  int zc;      // planes per chunk
  int gx, gy;  // tiles along x and y
};

template <class T>
__global__ void __launch_bounds__(kChThreads<T>)
k_cheb_march(ChebMarchArgs<T> a) {
  using C = typename Compute<T>::type;
  struct Two {
    C v[2];
  };
  constexpr int kRows = kChRows<T>;
  constexpr int kPlane = kRows * kChCols;
  // x of plane k and x of the first stage on plane k - 1, two buffers each
  __shared__ C xs[2][kPlane];
  __shared__ C ys[2][kPlane];
  const Lv<T>& L = a.L;
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  int blk = xcd_block32(blockIdx.x, gridDim.x);
  const int tx = __builtin_amdgcn_readfirstlane(blk % a.gx);
  blk /= a.gx;
  const int ty = __builtin_amdgcn_readfirstlane(blk % a.gy);
  const int tz = __builtin_amdgcn_readfirstlane(blk / a.gy);
  const int x0 = tx * kChOutX - kChHalo, y0 = ty * kChOutY<T> - kChHalo;
  const int z0 = tz * a.zc, z1 = min(nz, z0 + a.zc);
  const bool perx = a.bc.m[0] == 2, pery = a.bc.m[2] == 2,
             perz = a.bc.m[4] == 2;
  const int m = threadIdx.x & 31;  // pair of the row
  const int row = threadIdx.x >> 5;
  const int gi = x0 + 2 * m, gj = y0 + row;
  int wi = gi, wj = gj;
  bool ok = true;
  if (gi < 0 || gi >= nx) {
    ok = perx;
    wi = perx ? ((gi % nx) + nx) % nx : 0;
  }
  if (gj < 0 || gj >= ny) {
    ok = ok && pery;
    wj = pery ? ((gj % ny) + ny) % ny : 0;
  }
  if (!ok) wi = wj = 0;
  const int pos = row * kChCols + 2 * m;
  // lateral neighbours, as offsets from the cell (0: itself, at a Neumann
  // face; the region's rim, whose values are not used)
  const int xl = m == 0 || (!perx && gi == 0 && a.bc.m[0] == 1) ? 0 : -1;
  const int xh =
      m == 31 || (!perx && gi + 2 == nx && a.bc.m[1] == 1) ? 0 : 1;
  const int yl =
      row == 0 || (!pery && gj == 0 && a.bc.m[2] == 1) ? 0 : -kChCols;
  const int yh = row == kRows - 1 || (!pery && gj + 1 == ny && a.bc.m[3] == 1)
                     ? 0
                     : kChCols;
  const uint32_t nxy = static_cast<uint32_t>(nx) * ny;
  constexpr uint32_t kS = sizeof(T);
  const uint64_t cells = static_cast<uint64_t>(nxy) * nz;
  const SwRsrc rx = sw_rsrc(L.x, cells);
  const SwRsrc rd = sw_rsrc(L.D, cells);
  const SwRsrc rfx = sw_rsrc(L.fx, cells + static_cast<uint64_t>(ny) * nz);
  const SwRsrc rfy = sw_rsrc(L.fy, cells + static_cast<uint64_t>(nx) * nz);
  const SwRsrc rfz = sw_rsrc(L.fz, cells + nxy);
  const SwRsrc rb = sw_rsrc(L.b, cells);
  const SwRsrc rout = sw_rsrc(a.xout, cells);
  const uint32_t oc = static_cast<uint32_t>(wj * nx + wi) * kS;
  const uint32_t ofx = static_cast<uint32_t>(wj * (nx + 1) + wi) * kS;
  const bool mine = ok && m >= 1 && m < 31 && row >= kChHalo &&
                    row < kRows - kChHalo && gi < nx && gj < ny;

  // the plane in memory of plane k: wrapped, or (not used then) the nearest
  auto plane_of = [&](int k) -> uint32_t {
    if (!perz) return static_cast<uint32_t>(min(max(k, 0), nz - 1));
    const int w = k % nz;
    return static_cast<uint32_t>(w < 0 ? w + nz : w);
  };
  auto inside = [&](int k) -> bool {
    return perz || (k >= 0 && k < nz);
  };
  auto pair = [](SwPair<T> p) -> Two { return {{C(ld(p.lo)), C(ld(p.hi))}}; };
  auto load_x = [&](int k) -> SwPair<T> {
    return sw_load2<T>(rx, oc, plane_of(k) * nxy * kS);
  };
  auto x_of = [&](SwPair<T> raw, int k) -> Two {
    const Two x = pair(raw);
    const bool have = ok && inside(k);
    return {{have ? x.v[0] : C(0), have ? x.v[1] : C(0)}};
  };

  // coefficients of one plane (the low z faces are the high ones of the
  // plane below, but for the first plane of a periodic axis)
  struct Raw {
    SwPair<T> d, b, fyl, fyh, fzh, x;
    T f0, f1, f2;
  };
  struct Coef {
    Two d, b, fyl, fyh, fzl, fzh;
    C f0, f1, f2;
  };
  auto issue = [&](int k) -> Raw {  // coefficients of plane k, x of k + 1
    const uint32_t w = plane_of(k);
    const uint32_t sc = w * nxy * kS;
    const uint32_t sx = w * (nxy + ny) * kS;
    const uint32_t sy = w * (nxy + nx) * kS;
    Raw r;
    r.d = sw_load2<T>(rd, oc, sc);
    r.b = sw_load2<T>(rb, oc, sc);
    r.fyl = sw_load2<T>(rfy, oc, sy);
    r.fyh = sw_load2<T>(rfy, oc, sy + nx * kS);
    r.fzh = sw_load2<T>(rfz, oc, sc + nxy * kS);
    r.f0 = sw_load<T>(rfx, ofx, sx);
    r.f1 = sw_load<T>(rfx, ofx, sx + kS);
    r.f2 = sw_load<T>(rfx, ofx, sx + 2 * kS);
    r.x = load_x(k + 1);
    return r;
  };
  const Two first_fz = pair(sw_load2<T>(rfz, oc, 0));
  const int seam0 = 0, seam1 = perz ? nz : INT_MIN;
  const int wall0 = !perz && a.bc.m[4] == 1 ? 0 : INT_MIN;
  const int wall1 = !perz && a.bc.m[5] == 1 ? nz - 1 : INT_MIN;

  // A x of the pair: own x, planes below and above, lateral neighbours at p
  auto apply = [&](const Coef& c, const Two& xc, const Two& lo, const Two& hi,
                   const C* p, int k, C* out) {
    const C left = p[xl], right = p[1 + xh];
    const C nl[2] = {left, xc.v[0]}, nh[2] = {xc.v[1], right};
    const C fl[2] = {c.f0, c.f1}, fh[2] = {c.f1, c.f2};
    const C below[2] = {p[yl], p[1 + yl]}, beyond[2] = {p[yh], p[1 + yh]};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      C v = c.d.v[e] * xc.v[e];
      v -= fl[e] * nl[e];
      v -= fh[e] * nh[e];
      v -= c.fyl.v[e] * below[e];
      v -= c.fyh.v[e] * beyond[e];
      v -= c.fzl.v[e] * (k == wall0 ? xc.v[e] : lo.v[e]);
      v -= c.fzh.v[e] * (k == wall1 ? xc.v[e] : hi.v[e]);
      out[e] = v;
    }
  };

  // x: planes k - 1, k, k + 1; y (after the first stage): planes k - 2, k - 1
  Two xm, xc, y2 = {{C(0), C(0)}}, y1 = {{C(0), C(0)}}, dir = {{C(0), C(0)}};
  Coef cp{};  // coefficients of plane k - 1
  cp.d = {{C(1), C(1)}};
  cp.fzh = pair(sw_load2<T>(rfz, oc, plane_of(z0 - 1) * nxy * kS));

  auto step = [&](int k, Raw& raw, auto v_) {
    constexpr int V = decltype(v_)::value;
    Coef c;
    c.d = pair(raw.d);
    c.b = pair(raw.b);
    c.fyl = pair(raw.fyl);
    c.fyh = pair(raw.fyh);
    c.fzh = pair(raw.fzh);
    const bool seam = k == seam0 || k == seam1;
    c.fzl.v[0] = seam ? first_fz.v[0] : cp.fzh.v[0];
    c.fzl.v[1] = seam ? first_fz.v[1] : cp.fzh.v[1];
    c.f0 = C(ld(raw.f0));
    c.f1 = C(ld(raw.f1));
    c.f2 = C(ld(raw.f2));
    const Two xp = x_of(raw.x, k + 1);
    raw = issue(k + 1);
    // ---- first stage on plane k
    C v[2];
    Two y, n;
    apply(c, xc, xm, xp, xs[V] + pos, k, v);
    const bool have = ok && inside(k);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const C d = a.rf1 * (c.b.v[e] - v[e]) / c.d.v[e];
      n.v[e] = sw_round<T>(d);
      const C x1 = sw_round<T>(xc.v[e] + d);
      y.v[e] = have ? x1 : C(0);
    }
    // ---- second stage on plane k - 1
    apply(cp, y1, y2, y, ys[V] + pos, k - 1, v);
    if (k - 1 >= z0 && mine) {
      C out[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const C scaled = a.rf2 * (cp.b.v[e] - v[e]) / cp.d.v[e];
        out[e] = y1.v[e] + (a.pf2 * dir.v[e] + scaled);
      }
      sw_store2(rout, oc, static_cast<uint32_t>(k - 1) * nxy * kS,
                st<T>(out[0]), st<T>(out[1]));
    }
    // ---- the next step's lateral neighbours, in the other buffers
    xs[1 - V][pos] = xp.v[0];
    xs[1 - V][pos + 1] = xp.v[1];
    ys[1 - V][pos] = y.v[0];
    ys[1 - V][pos + 1] = y.v[1];
    __syncthreads();
    xm = xc;
    xc = xp;
    y2 = y1;
    y1 = y;
    dir = n;
    cp = c;
  };

  // from plane z0 - 1 (whose first stage the second one on z0 reads) to z1
  const int kstart = z0 - 1, kend = z1 + 1;
  xm = x_of(load_x(kstart - 1), kstart - 1);
  xc = x_of(load_x(kstart), kstart);
  xs[0][pos] = xc.v[0];
  xs[0][pos + 1] = xc.v[1];
  ys[0][pos] = C(0);
  ys[0][pos + 1] = C(0);
  Raw raw = issue(kstart);
  __syncthreads();
  for (int k = kstart; k < kend; k += 2) {
    step(k, raw, std::integral_constant<int, 0>{});
    if (k + 1 >= kend) break;
    step(k + 1, raw, std::integral_constant<int, 1>{});
  }
}

}  // namespace hf
