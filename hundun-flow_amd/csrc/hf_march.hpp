// Two red-black sweeps of a large level in one pass over its arrays (gfx950).
#pragma once

#include <limits.h>

#include <type_traits>

#include "hf_cycle.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// A block owns a tile of columns and marches through the planes of a z-chunk;
// at step k the four colour passes of the two sweeps are made on planes k,
// k-1, k-2 and k-3 (each pass on a plane needs the pass before it on that
// plane and its two neighbours).  Every array of the level is read once and
// x written once for the two sweeps, where a launch per sweep
// (k_rb_sweep) moves everything twice.  The region is the tile and a halo of
// four cells, which shrinks by one per pass that reads neighbours; cells
// that several blocks compute come out the same in each, so the result
// equals four colour passes bit for bit.
//
// A lane owns a pair of cells of a row (2m, 2m + 1), one of each colour in
// every plane.  At step k exactly one column of the pair is active: its cell
// on plane k has the first colour, on k-1 the second, and so on, so that
// column takes all four passes of the step, and the lateral neighbours it
// reads, columns of the other parity, are not written in the step: one
// barrier per step, and no order among the wavefronts within it.  A
// wavefront owns rows r and r + 2, whose active columns agree, so the active
// column is uniform and every register index static (the loop is unrolled
// over the four planes a coefficient lives; a wavefront runs the instance of
// its parity).
//
// The loads of a step are issued a step ahead (coefficients of plane k + 1,
// x of plane k + 2), and a barrier does not wait for them.
//
// What bounds it: the chain of the four passes and the barrier at one block
// per CU, about 1.4 us a step from L2 and 2 us with HBM behind it (the
// coefficients of four planes take the registers of more wavefronts than
// sixteen, and without b in LDS they spill: 384 us in place of 298 below).
// Counters at 512x256x256 FP32: wavefronts issue for 21% of their time, wait
// for memory, LDS or the barrier for 45 and for a turn to issue for the rest;
// the vector units work for 44% of the time (256x256x128 FP64: 34%).  Two
// sweeps, one launch against two k_rb_sweep launches, from x and from zero:
// 512x256x256 FP32 298 and 267 us against 478 and 445, 256x256x128 FP64 163
// and 149 against 277 and 254, 192x192x128 BF16 44 and 41 against 83 and 77.
// HBM traffic at 512x256x256 FP32 is 1.2 GB for 0.94 GB of operands.  Within
// a solve, with the projection's mean: 345 us from zero and 330 with the mean
// of the output (351 while that read the fluid flags).
//
// Boundaries: a position outside the domain holds 0 (Dirichlet; never
// updated) or is the wrapped cell (periodic); on a Neumann face the neighbour
// offset is 0, the cell itself at the time of its update.
// ---------------------------------------------------------------------------
constexpr int kMaCols = 64;   // region columns: 32 pairs
constexpr int kMaHalo = 4;
constexpr int kMaOutX = kMaCols - 2 * kMaHalo;
constexpr int kMaRing = 8;    // planes of x in LDS
// rows of the region: two per wavefront, and as many wavefronts as the
// coefficients of four planes leave registers for
template <class T>
constexpr int kMaRows = std::is_same<T, double>::value ? 16 : 32;
template <class T>
constexpr int kMaThreads = kMaRows<T> * 32;
template <class T>
constexpr int kMaOutY = kMaRows<T> - 2 * kMaHalo;

template <class T>
struct MarchArgs {
  Lv<T> L;
  Bc bc;
  T* xout;
  T* bout;             // projected b (kZero with mean), else null
  MeanRef mean;        // pending projection mean (kZero; at: null, none)
  int first;           // colour updated first: 0 forward, 1 reverse
  int zc;              // planes per chunk
  int gx, gy;          // tiles along x and y
  // kMean: per-block partial sums of w_x w_y w_z x of the output (the
  // constant projection's mean), cell widths per axis.  Solid cells add 0:
  // the prolongation before this smoothing left x = 0 there, b is 0, and a
  // refresh refuses a solid row with an open face (row_invalid).
  double* partials;
  const double* wx;
  const double* wy;
  const double* wz;
};

// Two floats, doubles or bf16 of one row.
template <class C>
struct MaPair {
  C v[2];
};

template <class T, bool kZero, bool kMean>
__global__ void __launch_bounds__(kMaThreads<T>) k_rb_march(MarchArgs<T> a) {
  using C = typename Compute<T>::type;
  constexpr int kRows = kMaRows<T>;
  constexpr int kPlane = kRows * kMaCols;
  __shared__ C xs[kMaRing * kPlane];
  __shared__ C bs[4 * kPlane];  // b of planes k .. k - 3, the lane's own
  __shared__ double red[16];
  const Lv<T>& L = a.L;
  const int nx = L.nx, ny = L.ny, nz = L.nz;
  int blk = xcd_block32(blockIdx.x, gridDim.x);
  const int tx = __builtin_amdgcn_readfirstlane(blk % a.gx);
  blk /= a.gx;
  const int ty = __builtin_amdgcn_readfirstlane(blk % a.gy);
  const int tz = __builtin_amdgcn_readfirstlane(blk / a.gy);
  const int x0 = tx * kMaOutX - kMaHalo, y0 = ty * kMaOutY<T> - kMaHalo;
  const int z0 = tz * a.zc, z1 = min(nz, z0 + a.zc);
  const bool perx = a.bc.m[0] == 2, pery = a.bc.m[2] == 2,
             perz = a.bc.m[4] == 2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int m = lane & 31;                           // pair of the row
  const int row = 4 * (wave >> 1) + (wave & 1) + 2 * (lane >> 5);
  // cell coordinates: unwrapped (gi even) and the cell they are
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
  // LDS: a row's even columns, then its odd ones
  const int pos = row * kMaCols + m;  // column 0; column 1 at pos + 32
  // lateral neighbours of column c (0 / 1), as offsets from pos
  const int xl0 = m == 0 || (!perx && gi == 0 && a.bc.m[0] == 1) ? 0 : 31;
  const int xh1 =
      m == 31 || (!perx && gi + 2 == nx && a.bc.m[1] == 1) ? 32 : 1;
  const int yl =
      row == 0 || (!pery && gj == 0 && a.bc.m[2] == 1) ? 0 : -kMaCols;
  const int yh = row == kRows - 1 || (!pery && gj + 1 == ny && a.bc.m[3] == 1)
                     ? 0
                     : kMaCols;
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
  const SwRsrc rbout = sw_rsrc(kZero ? a.bout : a.xout, cells);
  const uint32_t oc = static_cast<uint32_t>(wj * nx + wi) * kS;
  const uint32_t ofx = static_cast<uint32_t>(wj * (nx + 1) + wi) * kS;
  const bool mine = ok && m >= 2 && m < 30 && row >= kMaHalo &&
                    row < kRows - kMaHalo && gi < nx && gj < ny;
  const double mean = kZero ? mean_value<kMaThreads<T>>(a.mean, red) : 0.0;
  const C omega = C(0.72);

  // the plane in memory of plane k: wrapped, or (not used then) the nearest
  auto plane_of = [&](int k) -> int {
    if (!perz) return min(max(k, 0), nz - 1);
    const int w = k % nz;
    return w < 0 ? w + nz : w;
  };
  // ... of the plane after the one that lies at w, unwrapped k
  auto next_of = [&](int w, int k) -> int {
    return perz ? (w + 1 == nz ? 0 : w + 1) : min(max(k + 1, 0), nz - 1);
  };
  // (planes outside a wall: every k is inside a periodic axis)
  const uint32_t planes = perz ? 0xffffffffu : static_cast<uint32_t>(nz);
  auto inside = [&](int k) -> bool {
    return static_cast<uint32_t>(k) < planes || perz;
  };
  auto pair = [](SwPair<T> p) -> MaPair<C> {
    return {C(ld(p.lo)), C(ld(p.hi))};
  };

  // coefficients of the pair on four planes (ring slot: step mod 4); the low
  // z faces are the high ones of the plane below, but for the first plane of
  // a periodic axis, whose low faces are an array plane of their own
  MaPair<C> d[4], fyl[4], fyh[4], fzh[4], fz0, fzb;
  C fx[4][3];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    d[u] = fyl[u] = fyh[u] = fzh[u] = {C(1), C(1)};
    fx[u][0] = fx[u][1] = fx[u][2] = C(0);
  }
  // raw operands in flight: coefficients of the next step's plane, x of the
  // plane above it
  SwPair<T> nd{}, nb{}, nyl{}, nyh{}, nzh{}, nx2{};
  T nf0{}, nf1{}, nf2{};
  uint32_t nact = 0;
  // loads of coefficient plane wc and x plane wx (planes in memory)
  auto issue = [&](int wc, int wx) {
    const uint32_t k = static_cast<uint32_t>(wc);
    const uint32_t sc = k * nxy * kS;
    const uint32_t sx = k * (nxy + ny) * kS;
    const uint32_t sy = k * (nxy + nx) * kS;
    nd = sw_load2<T>(rd, oc, sc);
    nb = sw_load2<T>(rb, oc, sc);
    nf0 = sw_load<T>(rfx, ofx, sx);
    nf1 = sw_load<T>(rfx, ofx, sx + kS);
    nf2 = sw_load<T>(rfx, ofx, sx + 2 * kS);
    nyl = sw_load2<T>(rfy, oc, sy);
    nyh = sw_load2<T>(rfy, oc, sy + nx * kS);
    nzh = sw_load2<T>(rfz, oc, sc + nxy * kS);
    if (kZero && a.mean.at != nullptr)
      nact = *reinterpret_cast<const uint16_t*>(L.act + (sc + oc) / kS);
    if constexpr (!kZero)
      nx2 = sw_load2<T>(rx, oc, static_cast<uint32_t>(wx) * nxy * kS);
  };
  // the planes that are the axis's first, and the low z faces there; those of
  // plane z0 - 3 too (the plane below it is not loaded)
  const int seam0 = 0, seam1 = perz ? nz : INT_MIN;
  fz0 = pair(sw_load2<T>(rfz, oc, 0));
  fzh[3] = pair(sw_load2<T>(
      rfz, oc, static_cast<uint32_t>(plane_of(z0 - 3)) * nxy * kS));
  double mlo = 0.0, mhi = 0.0;  // kMean: sums of wz x of the two columns

  // planes in memory whose loads are issued next: coefficients, x
  int wc = plane_of(z0 - 3), wx = plane_of(z0 - 2);

  // planes at which a Neumann wall reads the cell itself (INT_MIN: none)
  const int wall0 = !perz && a.bc.m[4] == 1 ? 0 : INT_MIN;
  const int wall1 = !perz && a.bc.m[5] == 1 ? nz - 1 : INT_MIN;

  // One step: plane k, active column S; V = (k - kstart) mod 8 gives the LDS
  // slot of plane k (V + 1: kstart - 1 lies in slot 0) and its register slot,
  // so that every LDS access has a constant offset.
  auto step = [&](int k, auto v_, auto s_) {
    constexpr int V = decltype(v_)::value, S = decltype(s_)::value;
    constexpr int U = V & 3;
    // ---- operands of plane k and x of plane k + 1, loaded a step ago
    fzb = fzh[U];  // of plane k - 4
    d[U] = pair(nd);
    fyl[U] = pair(nyl);
    fyh[U] = pair(nyh);
    fzh[U] = pair(nzh);
    fx[U][0] = C(ld(nf0));
    fx[U][1] = C(ld(nf1));
    fx[U][2] = C(ld(nf2));
    MaPair<C> bk;
    if (kZero && a.mean.at != nullptr) {
      const T lo = st<T>(static_cast<double>(ld(nb.lo)) - mean);
      const T hi = st<T>(static_cast<double>(ld(nb.hi)) - mean);
      bk.v[0] = (nact & 0xffu) ? C(ld(lo)) : C(0);
      bk.v[1] = (nact & 0xff00u) ? C(ld(hi)) : C(0);
    } else {
      bk = pair(nb);
    }
    bs[U * kPlane + pos] = bk.v[0];
    bs[U * kPlane + pos + 32] = bk.v[1];
    MaPair<C> above = {C(0), C(0)};
    if constexpr (!kZero) {
      const bool have = ok && inside(k + 1);
      const MaPair<C> x = pair(nx2);
      above.v[0] = have ? x.v[0] : C(0);
      above.v[1] = have ? x.v[1] : C(0);
    }
    // the lane's position on plane k + q
    auto slot = [&](int q) -> C* {
      return xs + ((V + 1 + q) & (kMaRing - 1)) * kPlane + pos;
    };
    {
      C* const p = slot(1);
      p[0] = above.v[0];
      p[32] = above.v[1];
    }
    wc = next_of(wc, k);
    wx = next_of(wx, k + 1);
    issue(wc, wx);
    // ---- the passes, two at a time: their lateral neighbours, of the other
    // parity, are not written in this step, so they are read together; each
    // pass reads the plane above as the pass before left it
    constexpr int own = 32 * S;
    C below = C(0), last = above.v[S], side = C(0);
#pragma unroll
    for (int h = 0; h < 4; h += 2) {
      C xc[3], nl[2], nh[2], nyl_[2], nyh_[2], bv[2], n[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const C* const p = slot(-h - q);
        xc[q] = h > 0 && q == 0 ? below : p[own];
        nl[q] = S == 0 ? p[xl0] : p[0];
        nh[q] = S == 0 ? p[32] : p[xh1];
        nyl_[q] = p[own + yl];
        nyh_[q] = p[own + yh];
        bv[q] = h + q == 0 ? bk.v[S] : bs[((U + 4 - h - q) & 3) * kPlane + pos + own];
      }
      xc[2] = below = slot(-h - 2)[own];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int kk = k - h - q;
        const int R = (U + 4 - h - q) & 3;
        C lowx = xc[q + 1], highx = q == 0 ? last : n[0];
        lowx = kk == wall0 ? xc[q] : lowx;
        highx = kk == wall1 ? xc[q] : highx;
        C v = d[R].v[S] * xc[q];
        v -= fx[R][S] * nl[q];
        v -= fx[R][S + 1] * nh[q];
        v -= fyl[R].v[S] * nyl_[q];
        v -= fyh[R].v[S] * nyh_[q];
        const C zl = h + q == 3 ? fzb.v[S] : fzh[(R + 3) & 3].v[S];
        v -= (kk == seam0 || kk == seam1 ? fz0.v[S] : zl) * lowx;
        v -= fzh[R].v[S] * highx;
        const C xn =
            sw_round<T>(xc[q] + omega * (bv[q] - v) / d[R].v[S]);
        n[q] = ok && inside(kk) ? xn : xc[q];
      }
      slot(-h)[own] = n[0];
      slot(-h - 1)[own] = n[1];
      // (keeps the second half's reads out of the first half's registers)
      __builtin_amdgcn_sched_barrier(0);
      last = n[1];
      side = S == 0 ? nh[1] : nl[1];  // the pair's other cell
    }
    // ---- plane k - 3 is done: out
    const int kk = k - 3;
    if (kk >= z0 && kk < z1 && mine) {
      const T lo = st<T>(S == 0 ? last : side);
      const T hi = st<T>(S == 0 ? side : last);
      const uint32_t sc = static_cast<uint32_t>(kk) * nxy * kS;
      sw_store2(rout, oc, sc, lo, hi);
      if constexpr (kMean) {
        const double wz = a.wz[kk];
        mlo += wz * static_cast<double>(ld(lo));
        mhi += wz * static_cast<double>(ld(hi));
      }
    }
    if (kZero && a.bout != nullptr && k >= z0 && k < z1 && mine)
      sw_store2(rbout, oc, static_cast<uint32_t>(k) * nxy * kS,
                st<T>(bk.v[0]), st<T>(bk.v[1]));
    __syncthreads();
  };

  // march from plane z0 - 3 (the lowest whose first pass is needed) to
  // z1 + 2, four steps at a time
  const int kstart = z0 - 3, kend = z1 + 3;
  auto march = [&](auto s_) {
    constexpr int S = decltype(s_)::value;
    using I0 = std::integral_constant<int, S>;
    using I1 = std::integral_constant<int, 1 - S>;
    // (eight steps at a time, leaving after any even one)
    for (int k = kstart; k < kend; k += 8) {
      step(k, std::integral_constant<int, 0>{}, I0{});
      step(k + 1, std::integral_constant<int, 1>{}, I1{});
      if (k + 2 >= kend) break;
      step(k + 2, std::integral_constant<int, 2>{}, I0{});
      step(k + 3, std::integral_constant<int, 3>{}, I1{});
      if (k + 4 >= kend) break;
      step(k + 4, std::integral_constant<int, 4>{}, I0{});
      step(k + 5, std::integral_constant<int, 5>{}, I1{});
      if (k + 6 >= kend) break;
      step(k + 6, std::integral_constant<int, 6>{}, I0{});
      step(k + 7, std::integral_constant<int, 7>{}, I1{});
    }
  };
  // x of planes z0 - 4 and z0 - 3 before the first step
  {
    MaPair<C> lo = {C(0), C(0)}, hi = {C(0), C(0)};
    if constexpr (!kZero) {
      auto load = [&](int k) -> MaPair<C> {
        const MaPair<C> x = pair(sw_load2<T>(
            rx, oc, static_cast<uint32_t>(plane_of(k)) * nxy * kS));
        const bool have = ok && inside(k);
        return {have ? x.v[0] : C(0), have ? x.v[1] : C(0)};
      };
      lo = load(kstart - 1);
      hi = load(kstart);
    }
    C* p = xs + pos;
    p[0] = lo.v[0];
    p[32] = lo.v[1];
    p = xs + kPlane + pos;
    p[0] = hi.v[0];
    p[32] = hi.v[1];
  }
  issue(wc, wx);
  __syncthreads();
  // the active column of plane kstart: its cell has the first colour there
  const int s0 = (a.first + x0 + y0 + 4 * (wave >> 1) + (wave & 1) + kstart) & 1;
  if (s0)
    march(std::integral_constant<int, 1>{});
  else
    march(std::integral_constant<int, 0>{});
  if constexpr (kMean) {
    double msum = 0.0;
    if (mine)
      msum = a.wx[gi] * a.wy[gj] * mlo + a.wx[gi + 1] * a.wy[gj] * mhi;
    msum = block_sum(msum, red);
    if (threadIdx.x == 0)
      a.partials[xcd_block32(blockIdx.x, gridDim.x)] = msum;
  }
}

}  // namespace hf
