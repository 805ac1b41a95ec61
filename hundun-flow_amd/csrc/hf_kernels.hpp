// gfx950 kernels of the pressure solver.  Every kernel is HBM-stream bound
// (the 7-point operator is ~0.27 flop/byte in FP64), so the design goals are
// coalesced x-fastest streams, one pass per array where the algorithm allows
// it, and an XCD-aware block order so neighbour rows/planes hit the same L2.
#pragma once

#include "hf_device.hpp"

namespace hf {

// ---------------------------------------------------------------------------
// Setup: face coefficient rule (src/solver_piso.cpp:1060-1118), mobility
// m = 1/rho, beta = A_f / (d_L/m_L + d_R/m_R); Neumann physical faces are 0;
// periodic physical faces use half widths of the wrapped cells.
// ---------------------------------------------------------------------------
struct AxisGeom {
  const double* faces[3];  // n+1 coordinates per axis
  int n[3];
  int8_t kind[6];          // hf_boundary_kind per physical face
};

__device__ __forceinline__ double face_rule(const double* f, int count,
                                            int normal, int kind, double area,
                                            double ml, double mr) {
  if ((normal == 0 || normal == count) && kind == 1) return 0.0;
  if ((normal == 0 || normal == count) && kind == 0) {
    const double owner = normal == 0 ? mr : ml;
    double distance;
    if (normal == 0) {
      const double w0 = f[1] - f[0];
      distance = (f[0] + 0.5 * w0) - f[0];
    } else {
      const double wl = f[count] - f[count - 1];
      distance = f[count] - (f[count - 1] + 0.5 * wl);
    }
    return 2.0 * area / (distance / owner + distance / owner);
  }
  double dl, dr;
  if (normal == 0 || normal == count) {
    dl = 0.5 * (f[count] - f[count - 1]);
    dr = 0.5 * (f[1] - f[0]);
  } else {
    const double loc = f[normal];
    const double wl = f[normal] - f[normal - 1];
    const double wr = f[normal + 1] - f[normal];
    dl = loc - (f[normal - 1] + 0.5 * wl);
    dr = (f[normal] + 0.5 * wr) - loc;
  }
  return area / (dl / ml + dr / mr);
}

// d beta / d m_L and d beta / d m_R for the same rule (adjoint).
__device__ __forceinline__ void face_rule_grad(const double* f, int count,
                                               int normal, int kind,
                                               double area, double ml,
                                               double mr, double* gl,
                                               double* gr) {
  *gl = 0.0;
  *gr = 0.0;
  if ((normal == 0 || normal == count) && kind == 1) return;
  if ((normal == 0 || normal == count) && kind == 0) {
    // beta = area*m_o/d: linear in the owner mobility
    const double owner = normal == 0 ? mr : ml;
    const double beta = face_rule(f, count, normal, kind, area, ml, mr);
    if (normal == 0)
      *gr = beta / owner;
    else
      *gl = beta / owner;
    return;
  }
  double dl, dr;
  if (normal == 0 || normal == count) {
    dl = 0.5 * (f[count] - f[count - 1]);
    dr = 0.5 * (f[1] - f[0]);
  } else {
    const double loc = f[normal];
    const double wl = f[normal] - f[normal - 1];
    const double wr = f[normal + 1] - f[normal];
    dl = loc - (f[normal - 1] + 0.5 * wl);
    dr = (f[normal] + 0.5 * wr) - loc;
  }
  const double s = dl / ml + dr / mr;
  const double beta = area / s;
  // d beta/d m = beta^2/area * d/m^2
  *gl = beta * beta / area * (dl / (ml * ml));
  *gr = beta * beta / area * (dr / (mr * mr));
}

// All face coefficients: a thread owns the low face of its cell along each
// axis, and the high one at the end of the axis.  32 bytes a cell and nine
// FP64 divisions, which bound it: 220 us at 256^3.  A launch per axis, with
// 64-bit divisions for the indices, read m three times over: 345 us.
__global__ void k_assemble_faces(AxisGeom g, const double* m, double* bx,
                                 double* by, double* bz) {
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const int plane = nx * ny;
  const int c = xcd_block32(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  if (c < 0 || c >= plane * nz) return;
  const int k = c / plane;
  const int r = c - k * plane;
  const int j = r / nx;
  const int ijk[3] = {r - j * nx, j, k};
  const int step[3] = {1, nx, plane};
  double w[3];
#pragma unroll
  for (int a = 0; a < 3; ++a)
    w[a] = g.faces[a][ijk[a] + 1] - g.faces[a][ijk[a]];
  const double mc = m[c];
  double* out[3] = {bx, by, bz};
  const int at[3] = {c + j + ny * k, c + nx * k, c};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double area = a == 0 ? w[1] * w[2]
                               : (a == 1 ? w[0] * w[2] : w[0] * w[1]);
    const int n = g.n[a], i = ijk[a];
    const double low = m[i > 0 ? c - step[a] : c + (n - 1) * step[a]];
    out[a][at[a]] =
        face_rule(g.faces[a], n, i, g.kind[2 * a], area, low, mc);
    if (i + 1 == n)
      out[a][at[a] + step[a]] =
          face_rule(g.faces[a], n, n, g.kind[2 * a + 1], area, mc,
                    m[c - (n - 1) * step[a]]);
  }
}

__global__ void k_face_sum_diag(int nx, int ny, int nz, const double* bx,
                                const double* by, const double* bz,
                                double* diag) {
  const int64_t cells = (int64_t)nx * ny * nz;
  const int64_t c = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (c >= cells) return;
  const int j = static_cast<int>((c / nx) % ny);
  const int k = static_cast<int>(c / ((int64_t)nx * ny));
  const int64_t row = j + (int64_t)ny * k;
  const int64_t fyo = c + (int64_t)nx * k;
  diag[c] = bx[c + row] + bx[c + row + 1] + by[fyo] + by[fyo + nx] + bz[c] +
            bz[c + (int64_t)nx * ny];
}

// Storage-precision copies of one level's operator (null: the level is FP64).
template <class T>
struct StoredCoeffs {
  T* D;
  T* fx;
  T* fy;
  T* fz;
};

// What a refresh kernel leaves for k_refresh_finish: the block sums of fluid
// volume and, on level 0, the block maxima of the row ratio; failed checks
// set bits of *bad.
struct RefreshOut {
  double* volume;
  double* ratio;  // null: not taken
  int* bad;
};

// Certified SDD M-matrix check of one row (src/solver_mg.cpp:1965-2019).
__device__ __forceinline__ bool row_invalid(double d, double faces,
                                            double vol) {
  const bool fail =
      !isfinite(d) || !(d > 0.0) || !isfinite(faces) || faces < 0.0;
  return fail || (vol == 0.0 ? d != 1.0 || faces != 0.0 : faces > d);
}

// Largest value of the block (fixed order); valid in thread 0.
__device__ __forceinline__ double block_max(double v, double* scratch) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
#pragma unroll
  for (int offset = kWave / 2; offset > 0; offset >>= 1)
    v = fmax(v, __shfl_down(v, offset, kWave));
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  double m = 0.0;
  if (threadIdx.x == 0) {
    const int waves = (blockDim.x + kWave - 1) / kWave;
    for (int w = 0; w < waves; ++w) m = fmax(m, scratch[w]);
  }
  __syncthreads();
  return m;
}

// Level-0 masking (src/solver_mg.cpp:1469-1570): faces times activity,
// solid diagonal 1, fluid diagonal D - original faces + active faces, fluid
// volume w_x*w_y*w_z (0 on solids); with it the checks of the masked row, its
// ratio (sum of the six faces, physical boundaries included) / D for the
// diagonal shortcut (src/solver_mg.cpp:1573-1611), the storage-precision
// copies and a copy of the face masks for the adjoint.  A thread owns its
// cell and the cell's low faces, and the high ones at the end of an axis.
// One pass, 96 bytes a cell for an FP32 cycle, near the copy rate: 362 us at
// 256^3.  Masking, the checks, the ratio, the copies and the volume sum as
// launches of their own took 1020 us.
struct Finest {
  int nx, ny, nz;
  const double* D;
  const double* b[3];
  const uint8_t* ca;      // null: every cell and face active
  const uint8_t* fa[3];
  const double* w[3];
  double* oD;
  double* of[3];
  double* vol;
  uint8_t* act;
  uint8_t* ofa[3];
};

template <class T>
__global__ void k_mask_level(Finest f, StoredCoeffs<T> s, RefreshOut out) {
  __shared__ double scratch[16];
  const int nx = f.nx, ny = f.ny, plane = nx * ny;
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int c = lb * kBlock + static_cast<int>(threadIdx.x);
  double vol = 0.0, ratio = 0.0;
  if (c >= 0 && c < plane * f.nz) {
    const int k = c / plane;
    const int r = c - k * plane;
    const int j = r / nx;
    const int ijk[3] = {r - j * nx, j, k};
    const int n[3] = {nx, ny, f.nz};
    const int step[3] = {1, nx, plane};
    const int at[3] = {c + j + ny * k, c + nx * k, c};
    const bool solid = f.ca != nullptr && f.ca[c] == 0;
    vol = f.w[0][ijk[0]] * f.w[1][j] * f.w[2][k];
    if (solid) vol = 0.0;
    T* copies[3] = {s.fx, s.fy, s.fz};
    double original = 0.0, active = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        const int face = at[a] + side * step[a];
        const double raw = f.b[a][face];
        const uint8_t open = f.ca == nullptr ? 1 : f.fa[a][face];
        const double masked =
            raw * (f.ca == nullptr ? 1.0 : static_cast<double>(open));
        original = a == 0 && side == 0 ? raw : original + raw;
        active = a == 0 && side == 0 ? masked : active + masked;
        if (side == 0 || ijk[a] + 1 == n[a]) {
          f.of[a][face] = masked;
          if (copies[a] != nullptr) copies[a][face] = st<T>(masked);
          if (f.ca != nullptr) f.ofa[a][face] = open;
        }
      }
    }
    double d = f.D[c];
    if (f.ca != nullptr) d = solid ? 1.0 : d - original + active;
    f.oD[c] = d;
    if (s.D != nullptr) s.D[c] = st<T>(d);
    f.vol[c] = vol;
    f.act[c] = solid ? 0 : 1;
    if (row_invalid(d, active, vol)) atomicOr(out.bad, 2);
    ratio = active / d;
    if (!(ratio >= 0.0)) ratio = 0.0;  // max(0, NaN) keeps 0 (std::max)
  }
  vol = block_sum(vol, scratch);
  if (threadIdx.x == 0) out.volume[lb] = vol;
  if (out.ratio != nullptr) {
    ratio = block_max(ratio, scratch);
    if (threadIdx.x == 0) out.ratio[lb] = ratio;
  }
}

// Coarse aggregation (src/solver_mg.cpp:1706-1962) evaluated per coarse
// entry in the reference's association order: the x pass sums (or, for a
// normal face, selects) first, then y, then z.
struct Agg {
  int fn[3];  // fine shape
  int cn[3];  // coarse shape
  int mask;   // coarsened axes
};

__device__ __forceinline__ int64_t fidx(const int e[3], int i, int j, int k) {
  return i + (int64_t)e[0] * (j + (int64_t)e[1] * k);
}

// Value of one fine channel entry (cell channel: face_axis < 0).
template <class Loader>
__device__ __forceinline__ double aggregate_entry(const Agg& a, int face_axis,
                                                  int ci, int cj, int ck,
                                                  Loader&& load) {
  // Per axis: list of up to 2 fine indices (selection or pair).
  int idx[3][2];
  int cnt[3];
  const int co[3] = {ci, cj, ck};
  for (int ax = 0; ax < 3; ++ax) {
    if ((a.mask & (1 << ax)) == 0) {
      idx[ax][0] = co[ax];
      cnt[ax] = 1;
    } else if (face_axis == ax) {
      const int g = 2 * co[ax];
      idx[ax][0] = g < a.fn[ax] ? g : a.fn[ax];
      cnt[ax] = 1;
    } else {
      idx[ax][0] = 2 * co[ax];
      idx[ax][1] = 2 * co[ax] + 1;
      cnt[ax] = idx[ax][1] < a.fn[ax] ? 2 : 1;
    }
  }
  // x pass innermost, z pass outermost: z(y(x)).
  double vz = 0.0;
  for (int dz = 0; dz < cnt[2]; ++dz) {
    double vy = 0.0;
    for (int dy = 0; dy < cnt[1]; ++dy) {
      double vx = 0.0;
      for (int dx = 0; dx < cnt[0]; ++dx)
        vx = (dx == 0 && cnt[0] == 1 && ((a.mask & 1) == 0 || face_axis == 0))
                 ? load(idx[0][dx], idx[1][dy], idx[2][dz])
                 : vx + load(idx[0][dx], idx[1][dy], idx[2][dz]);
      vy = (cnt[1] == 1 && ((a.mask & 2) == 0 || face_axis == 1)) ? vx : vy + vx;
    }
    vz = (cnt[2] == 1 && ((a.mask & 4) == 0 || face_axis == 2)) ? vy : vz + vy;
  }
  return vz;
}

struct Fine64 {
  const double* D;
  const double* fx;
  const double* fy;
  const double* fz;
  const double* vol;
};
struct Coarse64 {
  double* D;
  double* fx;
  double* fy;
  double* fz;
  double* vol;
  uint8_t* act;
};

// One coarse level: a thread forms its cell's volume and reaction, its six
// faces (each from the fine faces below it), the diagonal from them, the
// checks and the storage-precision copies; it stores the low faces, and the
// high ones at the end of an axis.  scale: the distance correction per axis.
// ratio: the diagonal shortcut's maximum; at or below `limit` the level is
// not built.
template <class T>
__global__ void k_coarse_level(Agg a, Fine64 f, Coarse64 c, StoredCoeffs<T> s,
                               RefreshOut out, double scale_x, double scale_y,
                               double scale_z, const double* ratio,
                               double limit) {
  __shared__ double scratch[16];
  if (ratio != nullptr && *ratio <= limit) return;
  const int nx = a.cn[0], ny = a.cn[1], nz = a.cn[2], plane = nx * ny;
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int t = lb * kBlock + static_cast<int>(threadIdx.x);
  double vol = 0.0;
  if (t >= 0 && t < plane * nz) {
    const int ck = t / plane;
    const int r = t - ck * plane;
    const int cj = r / nx;
    const int ci = r - cj * nx;
    const int* fn = a.fn;
    const int fe[3][3] = {{fn[0] + 1, fn[1], fn[2]},
                          {fn[0], fn[1] + 1, fn[2]},
                          {fn[0], fn[1], fn[2] + 1}};
    const double* fine[3] = {f.fx, f.fy, f.fz};
    vol = aggregate_entry(a, -1, ci, cj, ck, [&](int i, int j, int k) {
      return f.vol[fidx(fn, i, j, k)];
    });
    double d = aggregate_entry(a, -1, ci, cj, ck, [&](int i, int j, int k) {
      const int64_t cc = fidx(fn, i, j, k);
      if (f.vol[cc] == 0.0) return 0.0;
      const double faces =
          f.fx[fidx(fe[0], i, j, k)] + f.fx[fidx(fe[0], i + 1, j, k)] +
          f.fy[fidx(fe[1], i, j, k)] + f.fy[fidx(fe[1], i, j + 1, k)] +
          f.fz[fidx(fe[2], i, j, k)] + f.fz[fidx(fe[2], i, j, k + 1)];
      const double reaction = f.D[cc] - faces;
      return reaction > 0.0 ? reaction : 0.0;
    });
    const int co[3] = {ci, cj, ck};
    const int at[3] = {t + cj + ny * ck, t + nx * ck, t};
    const int step[3] = {1, nx, plane};
    const double scale[3] = {scale_x, scale_y, scale_z};
    double* coarse[3] = {c.fx, c.fy, c.fz};
    T* copies[3] = {s.fx, s.fy, s.fz};
    double faces = 0.0;
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        int e[3] = {ci, cj, ck};
        e[ax] += side;
        double v = aggregate_entry(a, ax, e[0], e[1], e[2],
                                   [&](int i, int j, int k) {
                                     return fine[ax][fidx(fe[ax], i, j, k)];
                                   });
        v = scale[ax] == 1.0 ? v : v * scale[ax];
        faces = ax == 0 && side == 0 ? v : faces + v;
        if (side == 0 || co[ax] + 1 == a.cn[ax]) {
          const int face = at[ax] + side * step[ax];
          coarse[ax][face] = v;
          if (copies[ax] != nullptr) copies[ax][face] = st<T>(v);
        }
      }
    }
    d += faces;
    if (vol == 0.0) d = 1.0;
    c.D[t] = d;
    if (s.D != nullptr) s.D[t] = st<T>(d);
    c.vol[t] = vol;
    c.act[t] = vol > 0.0 ? 1 : 0;
    if (vol < 0.0 || !isfinite(vol) || !(d > 0.0) || !isfinite(d))
      atomicOr(out.bad, 1);
    if (row_invalid(d, faces, vol)) atomicOr(out.bad, 2);
  }
  vol = block_sum(vol, scratch);
  if (threadIdx.x == 0) out.volume[lb] = vol;
}

// *out = the largest of `count` block maxima (one block).
__global__ void __launch_bounds__(1024)
k_refresh_ratio(const double* ratio, int count, double* out) {
  __shared__ double scratch[16];
  double m = 0.0;
  for (int b = threadIdx.x; b < count; b += blockDim.x) m = fmax(m, ratio[b]);
  m = block_max(m, scratch);
  if (threadIdx.x == 0) *out = m;
}

// Block l: the fluid volume of level l from its block sums, which lie one
// level after the other; block 0 also turns the check flags into a scalar.
struct RefreshLevels {
  int first[33];  // first block sum of a level; the last entry ends them
};

__global__ void __launch_bounds__(1024)
k_refresh_finish(const double* volume, RefreshLevels levels, const int* bad,
                 double* volumes, double* flag) {
  __shared__ double scratch[16];
  const int l = blockIdx.x;
  double v = 0.0;
  for (int b = levels.first[l] + static_cast<int>(threadIdx.x);
       b < levels.first[l + 1]; b += blockDim.x)
    v += volume[b];
  v = block_sum(v, scratch);
  if (threadIdx.x != 0) return;
  volumes[l] = v;
  if (l == 0) *flag = static_cast<double>(*bad);
}

// ---------------------------------------------------------------------------
// Reductions: per-block partials (deterministic shuffle tree) and a single
// block finaliser that also performs the scalar Krylov algebra on device so
// the host only reads back what it must test.
// ---------------------------------------------------------------------------
enum FinalOp : int {
  F_STORE = 0,     // scalars[a] = sum0
  F_ALPHA = 1,     // pap = sum0, alpha = rho / pap (rho: scalars[slot])
  F_RHO = 2,       // rho = sum0
  F_BETA_FR = 3,   // beta = sum0/rho, the other rho = sum0
  F_BETA_PR = 4,   // zq = sum1, beta = -alpha*zq/rho, the other rho = sum0
  F_MEAN = 5,      // scalars[a] = sum0 / volume
  F_MGALPHA = 6,   // three sums -> residual-minimising alpha
  F_STORE2 = 7,    // scalars[a] = sum0, scalars[a+1] = sum1
  F_STORE_MEAN = 8 // scalars[a] = sum0, scalars[S_MEAN0] = sum1 / volume
};

// First fold of many block partials: block (s, a) sums span s of
// accumulator a in index order.
__global__ void k_fold_partials(const double* partials, int64_t blocks,
                                int64_t stride, double* out,
                                int64_t out_stride, int64_t span) {
  __shared__ double scratch[16];
  const int64_t a = blockIdx.y;
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * span;
  const int64_t hi = lo + span < blocks ? lo + span : blocks;
  double v = 0.0;
  for (int64_t b = lo + threadIdx.x; b < hi; b += blockDim.x)
    v += partials[a * stride + b];
  v = block_sum(v, scratch);
  if (threadIdx.x == 0) out[a * out_stride + blockIdx.x] = v;
}

__global__ void __launch_bounds__(1024)
k_finalize(const double* partials, int64_t blocks, int64_t stride, int nacc,
           double* scalars, int op, int slot, double volume, int unit_linear) {
  __shared__ double scratch[16];
  double sums[3] = {0.0, 0.0, 0.0};
  for (int a = 0; a < nacc; ++a) {
    // eight loads in flight: one block takes 16384 partials in 7 us, where a
    // fold by several blocks before it took 9
    double v = 0.0;
    for (int64_t base = threadIdx.x; base < blocks;
         base += 8 * static_cast<int64_t>(blockDim.x)) {
      double q[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t b = base + u * static_cast<int64_t>(blockDim.x);
        q[u] = b < blocks ? partials[a * stride + b] : 0.0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) v += q[u];
    }
    sums[a] = block_sum(v, scratch);
  }
  if (threadIdx.x != 0) return;
  switch (op) {
    case F_STORE:
      scalars[slot] = sums[0];
      break;
    case F_STORE2:
      scalars[slot] = sums[0];
      scalars[slot + 1] = sums[1];
      break;
    case F_ALPHA:
      scalars[S_PAP] = sums[0];
      scalars[S_ALPHA] = scalars[slot] / sums[0];
      break;
    case F_RHO:
      scalars[slot] = sums[0];
      break;
    case F_BETA_FR:
      scalars[other_rho(slot)] = sums[0];
      scalars[S_BETA] = sums[0] / scalars[slot];
      break;
    case F_BETA_PR:
      scalars[other_rho(slot)] = sums[0];
      scalars[S_ZQ] = sums[1];
      scalars[S_BETA] = -scalars[S_ALPHA] * sums[1] / scalars[slot];
      break;
    case F_STORE_MEAN:
      scalars[slot] = sums[0];
      scalars[S_MEAN0] = sums[1] / volume;
      break;
    case F_MEAN:
      scalars[slot] = sums[0] / volume;
      break;
    case F_MGALPHA: {
      scalars[S_PROJ0] = sums[0];
      scalars[S_PROJ1] = sums[1];
      scalars[S_PROJ2] = sums[2];
      const double tiny = 2.220446049250313080847e-16 * sums[0];
      scalars[S_MGALPHA] =
          unit_linear ? 1.0 : (sums[2] > tiny ? sums[1] / sums[2] : 0.0);
      break;
    }
    default:
      break;
  }
}

}  // namespace hf

#include "hf_cycle.hpp"

namespace hf {

// Scaled 2-norm (global_norm, src/solver_krylov.cpp:650-711): the largest
// magnitude, then the compensated sum of squares of the elements divided by
// it.  The solvers take it where a plain sum of squares overflowed, so a
// norm overflows only where the reference's does.  A non-finite element
// makes its block's maximum +inf.
__global__ void k_absmax(Chunk ch, const double* v, double* partials) {
  __shared__ double scratch[16];
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int lo = lb * ch.chunk;
  const int hi = min(ch.n, lo + ch.chunk);
  double m = 0.0;
  for (int c = lo + threadIdx.x; c < hi; c += blockDim.x) {
    const double a = v[c];
    m = isfinite(a) ? fmax(m, fabs(a)) : INFINITY;
  }
  m = block_max(m, scratch);
  if (threadIdx.x == 0) partials[lb] = m;
}

__global__ void __launch_bounds__(1024)
k_max_fold(const double* partials, int64_t count, double* scalars, int slot) {
  __shared__ double scratch[16];
  double m = 0.0;
  for (int64_t b = threadIdx.x; b < count; b += blockDim.x)
    m = fmax(m, partials[b]);
  m = block_max(m, scratch);
  if (threadIdx.x == 0) scalars[slot] = m;
}

// Per block: the Neumaier-compensated sum of (v / scale)^2 of each thread's
// elements, then the block's sum of those.
__global__ void k_scaled_squares(Chunk ch, const double* v,
                                 const double* scale, double* partials) {
  __shared__ double scratch[16];
  const int lb = xcd_block32(blockIdx.x, gridDim.x);
  const int lo = lb * ch.chunk;
  const int hi = min(ch.n, lo + ch.chunk);
  const double s = *scale;
  double sum = 0.0, correction = 0.0;
  for (int c = lo + threadIdx.x; c < hi; c += blockDim.x) {
    const double q = v[c] / s;
    const double square = q * q;
    const double next = sum + square;
    correction += fabs(sum) >= fabs(square) ? (sum - next) + square
                                            : (square - next) + sum;
    sum = next;
  }
  sum = block_sum(sum + correction, scratch);
  if (threadIdx.x == 0) partials[lb] = sum;
}

// Adjoint: grad_logrho(c) = -sum over the six faces f of c of
//   (lam_L - lam_R)(p_L - p_R) * d beta_f / d m_c * d m_c / d log rho_c
// with m = 1/rho, d m / d log rho = -m.  Masked faces carry no gradient.
__global__ void k_grad_logrho(AxisGeom g, const double* m, const double* p,
                              const double* lam, const uint8_t* fxa,
                              const uint8_t* fya, const uint8_t* fza,
                              double* out) {
  const int64_t nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const int64_t cells = nx * ny * nz;
  const int64_t c = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (c >= cells) return;
  const int ijk[3] = {static_cast<int>(c % nx), static_cast<int>((c / nx) % ny),
                      static_cast<int>(c / (nx * ny))};
  const uint8_t* fa[3] = {fxa, fya, fza};
  double grad = 0.0;
  for (int axis = 0; axis < 3; ++axis) {
    const int a1 = axis == 0 ? 1 : 0;
    const int a2 = axis == 2 ? 1 : 2;
    const double area =
        (g.faces[a1][ijk[a1] + 1] - g.faces[a1][ijk[a1]]) *
        (g.faces[a2][ijk[a2] + 1] - g.faces[a2][ijk[a2]]);
    int e[3] = {g.n[0], g.n[1], g.n[2]};
    e[axis] += 1;
    for (int side = 0; side < 2; ++side) {
      const int normal = ijk[axis] + side;  // face index along axis
      int fc[3] = {ijk[0], ijk[1], ijk[2]};
      fc[axis] = normal;
      const int64_t fi = fc[0] + (int64_t)e[0] * (fc[1] + (int64_t)e[1] * fc[2]);
      if (fa[axis] != nullptr && fa[axis][fi] == 0) continue;
      int cl[3] = {fc[0], fc[1], fc[2]};
      int cr[3] = {fc[0], fc[1], fc[2]};
      cl[axis] = normal == 0 ? g.n[axis] - 1 : normal - 1;
      cr[axis] = normal == g.n[axis] ? 0 : normal;
      const int kind = normal == 0 ? g.kind[2 * axis]
                                   : (normal == g.n[axis] ? g.kind[2 * axis + 1]
                                                          : 2);
      const bool physical = normal == 0 || normal == g.n[axis];
      if (physical && kind == 1) continue;
      const int64_t il = cl[0] + nx * (cl[1] + ny * cl[2]);
      const int64_t ir = cr[0] + nx * (cr[1] + ny * cr[2]);
      double gl, gr;
      face_rule_grad(g.faces[axis], g.n[axis], normal, kind, area, m[il], m[ir],
                     &gl, &gr);
      double jump;
      if (physical && kind == 0) {
        const int64_t owner = normal == 0 ? ir : il;
        jump = lam[owner] * p[owner];  // ghost value 0
      } else {
        jump = (lam[il] - lam[ir]) * (p[il] - p[ir]);
      }
      // this cell is the left cell of its high face and the right cell of
      // its low face (a periodic self-face counts both)
      double dbeta = 0.0;
      if (il == c) dbeta += gl;
      if (ir == c) dbeta += gr;
      grad -= jump * dbeta * (-m[c]);
    }
  }
  out[c] = grad;
}

}  // namespace hf
