// Device side of the tabulated LTE gas: the six-plane Helmholtz table, the
// bicubic Hermite interpolant of H(rho, T) and its exact divided
// differences, thermodynamics from H, temperature recovery (inverse-table
// guess + Newton, always FP64), the Itoh-Abe discrete gradients behind the
// entropy-conserving means, and the LTEEC flux with Lax-Friedrichs
// dissipation.  The interpolant and the flux arithmetic take the type R:
// double, or float for the mixed-precision form (the planes then come from
// an FP32 copy of the table, and the discrete gradients switch to the
// derivative form below FP32's resolution instead of FP64's).
//
// Restates include/LTEHelmholtzTable.hpp:84-105, LTEHelmholtzInterpolation.hpp:26-211,
// LTEHelmholtzEOS.hpp:14-397, LTEECFlux.hpp:11-85, DissipationOperator.hpp:15-28.
// A query outside the table (or a recovery that does not converge) yields
// NaN instead of trapping; the grid searches never read outside the grids.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

// No multiply-add contraction in the table arithmetic: the Hermite sums and
// the thermodynamic combinations built on them (c^2, the divided differences)
// cancel strongly, and fusing changes their rounding enough to move the
// right-hand side of a smooth state by ~2e-12 relative (an uncontracted CPU
// build and a contracted one of the same code differ by that much).  Restored
// to the default at the end of this header.
#pragma clang fp contract(off)

namespace thx {
namespace lte {

// Cell search in an increasing grid: cell[key(x)] is the cell of the lower
// edge of x's bucket, from which the cell of x is at most a few steps away.
// The key of a positive grid is linear in the high word of x's
// bit pattern, piecewise linear in log x; of another grid, linear in x.
struct Buckets {
  const unsigned short *cell = nullptr;
  int count = 0, shift = 0, positive = 0;
  unsigned base = 0;
  double x0 = 0, scale = 0;
};

struct View {
  int nx = 0, ny = 0;
  const double *rho = nullptr, *T = nullptr, *e = nullptr;  // grids
  const double *planes = nullptr;                           // 6 * nx * ny: H, H_rho, H_T, H_rhoT, mu, lambda
  const float *planes32 = nullptr;                          // the planes rounded to FP32 (mixed precision)
  const double *inv = nullptr;                              // nx * ny temperature guesses
  // bucket tables of the grids (Buckets), for cell searches by a lookup
  // instead of a bisection; an empty one means bisect
  Buckets brho, bT, be;
  // per node of the state being evaluated (written by k_lte_nodes): the
  // recovered temperature and the table cell i | j << 16 (-1 outside)
  double *node_T = nullptr;
  int *node_cell = nullptr;
  // and what the flux pair takes at it, where set: pressure, sound speed and
  // (Pirozzoli) gamma = cp/cv in FP64; for LTEEC the sound speed, H, H_rho,
  // H_rhorho, H_T and H_rhoT ([5][Ntot] of the pair fluxes' type) and, in the
  // mixed form, the pressure
  double *node_p = nullptr, *node_c = nullptr, *node_g = nullptr;
  void *node_rec = nullptr;
  // the scaled Hermite coefficients of every cell (kCellStride values per
  // cell, k_lte_cells), in FP64 and, for the mixed form of LTEEC, in FP32
  const double *cells64 = nullptr;
  const float *cells32 = nullptr;
  // viscosity of the Navier-Stokes form: the mu plane, or Sutherland's law
  // mu0 (T0 + Ts) (T/T0)^1.5 / (T + Ts) when sutherland is set
  int sutherland = 0;
  double mu0 = 0, T0 = 0, Ts = 0;
};

// LTETransport.hpp:22-29 (viscosity_from_temperature)
__device__ __forceinline__ double sutherland_viscosity(const View &v, double T) {
  const double rel = T / v.T0;
  return v.mu0 * (v.T0 + v.Ts) * rel * sqrt(rel) / (T + v.Ts);
}

// bisection: largest i with grid[i] <= value (count-2 at the top end); -1 outside
__device__ __forceinline__ int find_cell(const double *grid, int count, double value) {
  if (!(value >= grid[0]) || !(value <= grid[count - 1])) return -1;
  int lo = 0, hi = count - 1;
  while (hi - lo > 1) {
    const int mid = lo + (hi - lo) / 2;
    if (value < grid[mid]) hi = mid;
    else lo = mid;
  }
  return lo;
}

// find_cell by the grid's buckets (two dependent loads instead of
// log2(count)), with the cell's ends
__device__ __forceinline__ int find_cell(const double *grid, int count, const Buckets &b, double value, double &lo,
                                         double &hi) {
  if (!(value >= grid[0]) || !(value <= grid[count - 1])) return -1;
  int i;
  if (b.cell) {
    const int k = b.positive ? (int)(((unsigned)(__double_as_longlong(value) >> 32) - b.base) >> b.shift)
                             : (int)((value - b.x0) * b.scale);
    i = b.cell[min(max(k, 0), b.count - 1)];
  } else {
    i = find_cell(grid, count, value);
  }
  lo = grid[i];
  hi = grid[i + 1];
  while (i < count - 2 && value >= hi) {
    lo = hi;
    hi = grid[++i + 1];
  }
  while (i > 0 && value < lo) {  // rounding of the linear key
    hi = lo;
    lo = grid[--i];
  }
  return i;
}

template <int D, typename R>
__device__ __forceinline__ R pbasis(int side, R x) {
  const R x2 = x * x;
  if constexpr (D == 0) return side == 0 ? 2 * x2 * x - 3 * x2 + 1 : -2 * x2 * x + 3 * x2;
  else if constexpr (D == 1) return side == 0 ? 6 * x2 - 6 * x : -6 * x2 + 6 * x;
  else return side == 0 ? 12 * x - 6 : -12 * x + 6;
}
template <int D, typename R>
__device__ __forceinline__ R sbasis(int side, R x) {
  const R x2 = x * x;
  if constexpr (D == 0) return side == 0 ? x2 * x - 2 * x2 + x : x2 * x - x2;
  else if constexpr (D == 1) return side == 0 ? 3 * x2 - 4 * x + 1 : 3 * x2 - 2 * x;
  else return side == 0 ? 6 * x - 4 : 6 * x - 2;
}
template <int D, typename R>
__device__ __forceinline__ R dpbasis(int side, R x, R y) {
  R v;
  if constexpr (D == 0) v = 2 * (x * x + x * y + y * y) - 3 * (x + y);
  else if constexpr (D == 1) v = 6 * (x + y) - 6;
  else v = 12;
  return side == 0 ? v : -v;
}
template <int D, typename R>
__device__ __forceinline__ R dsbasis(int side, R x, R y) {
  if constexpr (D == 0) return x * x + x * y + y * y - (side == 0 ? 2 : 1) * (x + y) + (side == 0 ? 1 : 0);
  else if constexpr (D == 1) return 3 * (x + y) - (side == 0 ? 4 : 2);
  else return 6;
}
template <int D, typename R>
__device__ __forceinline__ R cscale(R w) {
  return D == 0 ? R(1) : (D == 1 ? w : w * w);
}

// The four planes at the lower corner of one cell
template <typename R = double>
struct Cell {
  const R *H = nullptr;  // plane 0 at the corner; plane k at H + k*plane
  int stride = 0, plane = 0;
  R wr = 0, wt = 0;
};

// the table's planes in the arithmetic type
template <typename R>
__device__ __forceinline__ const R *planes_of(const View &v) {
  if constexpr (sizeof(R) == sizeof(double)) return v.planes;
  else return v.planes32;
}

template <int DR, int DT, typename R>
__device__ __forceinline__ R evaluate(const Cell<R> &c, R xi, R eta) {
  R r = 0;
#pragma unroll
  for (int ds = 0; ds < 2; ++ds) {
    const R dv = pbasis<DR>(ds, xi), dsl = sbasis<DR>(ds, xi);
#pragma unroll
    for (int ts = 0; ts < 2; ++ts) {
      const int o = ds + ts * c.stride;
      const R tv = pbasis<DT>(ts, eta), tsl = sbasis<DT>(ts, eta);
      r += c.H[o] * dv * tv;
      r += (c.H[c.plane + o] * c.wr) * dsl * tv;
      r += (c.H[2 * c.plane + o] * c.wt) * dv * tsl;
      r += (c.H[3 * c.plane + o] * c.wr * c.wt) * dsl * tsl;
    }
  }
  return r / (cscale<DR>(c.wr) * cscale<DT>(c.wt));
}

template <typename R = double>
struct Eval {
  Cell<R> cell;
  R xi = 0, eta = 0, rho = 0, T = 0;
  int ci = 0, cj = 0;  // the cell's grid indices
  bool valid = false;
  template <int DR = 0, int DT = 0>
  __device__ R H() const { return evaluate<DR, DT>(cell, xi, eta); }
  __device__ R pressure() const { return rho * rho * H<1, 0>(); }
  __device__ R energy() const { return H() - T * H<0, 1>(); }
  __device__ R gibbs() const { return H() + rho * H<1, 0>(); }
  __device__ R p_rho() const { return 2 * rho * H<1, 0>() + rho * rho * H<2, 0>(); }
  __device__ R cv() const { return -T * H<0, 2>(); }
  __device__ R cp() const {  // LTEHelmholtzEOS.hpp:76-80
    const R m = H<1, 1>();
    return cv() + T * rho * rho * m * m / p_rho();
  }
  // LTEHelmholtzEOS.hpp:99-110: viscosity (plane 4) or thermal conductivity
  // (plane 5), bilinear in the cell's coordinates
  template <int PROP>
  __device__ R transport() const {
    const R *p = cell.H + PROP * cell.plane;
    return p[0] * (1 - xi) * (1 - eta) + p[1] * xi * (1 - eta) + p[cell.stride] * (1 - xi) * eta +
           p[cell.stride + 1] * xi * eta;
  }
  __device__ R c2() const {
    const R m = H<1, 1>();
    return p_rho() - rho * rho * m * m / H<0, 2>();
  }
};

// Evaluation at (rho, T) in a known cell (i, j)
template <typename R = double>
__device__ __forceinline__ Eval<R> at_cell(const View &v, R rho, R T, int i, int j) {
  Eval<R> r;
  const int off = j * v.nx + i;
  const R dr = R(v.rho[i + 1] - v.rho[i]), dt = R(v.T[j + 1] - v.T[j]);
  r.cell.H = planes_of<R>(v) + off;
  r.cell.stride = v.nx;
  r.cell.plane = v.nx * v.ny;
  r.cell.wr = dr;
  r.cell.wt = dt;
  r.xi = (rho - R(v.rho[i])) / dr;
  r.eta = (T - R(v.T[j])) / dt;
  r.rho = rho;
  r.T = T;
  r.ci = i;
  r.cj = j;
  r.valid = true;
  return r;
}

// Evaluation at (rho, T) whose cell is known (i | j << 16, from
// find_cell of the two grids), or a flagged NaN evaluation for -1, as at()
// gives for a query outside the table.
template <typename R = double>
__device__ __forceinline__ Eval<R> at_packed(const View &v, R rho, R T, int cell) {
  Eval<R> r = at_cell<R>(v, rho, T, cell < 0 ? 0 : (cell & 0xFFFF), cell < 0 ? 0 : (cell >> 16));
  if (cell < 0) {
    r.valid = false;
    r.xi = r.eta = R(__builtin_nan(""));
  }
  return r;
}

// LTEHelmholtzEOS.hpp:106-130; an invalid query reads cell (0,0) and is flagged
template <typename R = double>
__device__ __forceinline__ Eval<R> at(const View &v, R rho, R T) {
  const int i = find_cell(v.rho, v.nx, double(rho));
  const int j = find_cell(v.T, v.ny, double(T));
  Eval<R> r = at_cell<R>(v, rho, T, i < 0 ? 0 : i, j < 0 ? 0 : j);
  r.valid = i >= 0 && j >= 0;
  if (!r.valid) r.xi = r.eta = R(__builtin_nan(""));  // every derived quantity is NaN
  return r;
}

// LTEHelmholtzEOS.hpp:151-223; NaN unless converged
__device__ __forceinline__ double temperature_from_energy(const View &v, double rho, double e) {
  const int i = find_cell(v.rho, v.nx, rho);
  const int j = find_cell(v.e, v.ny, e);
  if (i < 0 || j < 0) return __builtin_nan("");
  const double x = (rho - v.rho[i]) / (v.rho[i + 1] - v.rho[i]);
  const double y = (e - v.e[j]) / (v.e[j + 1] - v.e[j]);
  const double *p = v.inv + j * v.nx + i;
  const double lower = p[0] + x * (p[1] - p[0]);
  const double upper = p[v.nx] + x * (p[v.nx + 1] - p[v.nx]);
  double T = lower + y * (upper - lower);
  const double Tlo = v.T[0], Thi = v.T[v.ny - 1];
  for (int it = 0; it < 100; ++it) {
    const Eval<double> s = at<double>(v, rho, T);
    if (!s.valid) return __builtin_nan("");
    const double cv = s.cv(), guess = s.energy();
    if (!(cv > 0) || !isfinite(guess)) return __builtin_nan("");
    const double step = (e - guess) / cv;
    const double next = T + step;
    const bool inside = isfinite(next) && next >= Tlo && next <= Thi;
    if (fabs(step) <= 1e-9 + 1e-12 * T) return next < Tlo ? Tlo : (next > Thi ? Thi : next);
    T = next;
    if (!inside) return __builtin_nan("");
  }
  return __builtin_nan("");
}

// ---- LTEEC: entropy-conserving means from per-node values and cell records

// One cell's record (index j*nx + i): the 16 Hermite coefficients in
// evaluate()'s order -- per corner (rho side, then T side) H, H_rho wr,
// H_T wt, (H_rhoT wr) wt -- then wr, wt and the reciprocals of wr, wt, wr wr,
// wr wt and wt wt; one value of padding keeps FP64 records on 64-byte lines.  A pair
// reads one or two records of consecutive values instead of 32 values strided
// over four planes and four grid points, with the scalings already applied.
constexpr int kCellStride = 24;

template <typename R>
__global__ void __launch_bounds__(256) k_lte_cells(View v, R *out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = t % v.nx, j = t / v.nx;
  if (i >= v.nx - 1 || j >= v.ny - 1) return;
  const Eval<R> ev = at_cell<R>(v, R(v.rho[i]), R(v.T[j]), i, j);
  const Cell<R> &c = ev.cell;
  R *o = out + (size_t)t * kCellStride;
#pragma unroll
  for (int ds = 0; ds < 2; ++ds)
#pragma unroll
    for (int ts = 0; ts < 2; ++ts) {
      const int k = ds + ts * c.stride, m = 4 * (2 * ds + ts);
      o[m] = c.H[k];
      o[m + 1] = c.H[c.plane + k] * c.wr;
      o[m + 2] = c.H[2 * c.plane + k] * c.wt;
      o[m + 3] = c.H[3 * c.plane + k] * c.wr * c.wt;
    }
  o[16] = c.wr;
  o[17] = c.wt;
  o[18] = R(1) / c.wr;
  o[19] = R(1) / c.wt;
  o[20] = R(1) / (c.wr * c.wr);
  o[21] = R(1) / (c.wr * c.wt);
  o[22] = R(1) / (c.wt * c.wt);
}
template <typename R>
__device__ __forceinline__ const R *cells_of(const View &v) {
  if constexpr (sizeof(R) == sizeof(double)) return v.cells64;
  else return v.cells32;
}

// n / d with y the correctly rounded 1 / d (Markstein's division by a known
// reciprocal): in FP64 the quotient estimate n y corrected by its remainder,
// which rounds as the IEEE quotient in three instructions instead of a
// division's eleven; FP32 divides.
template <typename R>
__device__ __forceinline__ R div_by(R n, R d, R y) {
  if constexpr (sizeof(R) == sizeof(double)) {
    const R q = n * y;
    return fma(fma(-d, q, n), y, q);
  } else {
    return n / d;
  }
}

// One node as an endpoint of a pair: H and H_rho at (rho, T), the cell (i | j
// << 16) and the coordinates in it, beta = 1/T
template <typename R>
struct PairNode {
  R rho, T, beta, xi, eta, H, Hr;
  int cell;
};

// A node's endpoint from its state, recovered temperature and cell (-1:
// outside the table, which makes every result NaN) and stored H, H_rho
template <typename R>
__device__ __forceinline__ PairNode<R> pair_node(const View &v, R rho, R T, int cell, R H, R Hr) {
  const Eval<R> ev = at_packed<R>(v, rho, T, cell);
  return PairNode<R>{rho, T, 1 / T, ev.xi, ev.eta, H, Hr, ev.ci | (ev.cj << 16)};
}

// Eval::pressure() of an endpoint
template <typename R>
__device__ __forceinline__ R pair_pressure(const PairNode<R> &s) {
  return s.rho * s.rho * s.Hr;
}

// Products of a cell's coefficients with one rho basis (value side 0, 1,
// slope side 0, 1), and their sum with one T basis: evaluate()'s operations in
// their order, the products shared by the T bases.  With the divided
// differences of one direction's bases between two points (dbasis4) in place
// of its bases, and divided by that direction's width once more, the sum is
// the divided difference of the interpolant along it.
template <typename R>
struct Basis4 {
  R v0, v1, s0, s1;
};
template <typename R>
__device__ __forceinline__ void cell_row(const R *c, const Basis4<R> &b, R *P) {
#pragma unroll
  for (int m = 0; m < 16; ++m) P[m] = c[m] * (m < 8 ? ((m & 1) ? b.s0 : b.v0) : ((m & 1) ? b.s1 : b.v1));
}
template <typename R>
__device__ __forceinline__ R cell_dot(const R *P, const Basis4<R> &t) {
  R r = 0;
#pragma unroll
  for (int m = 0; m < 16; ++m) r += P[m] * ((m & 4) ? ((m & 2) ? t.s1 : t.v1) : ((m & 2) ? t.s0 : t.v0));
  return r;
}
// Keeps a value's computation where it is written: sunk into the branch that
// uses it, a sum would drag its 16 products' registers along.
template <typename R>
__device__ __forceinline__ void pin(R &x) {
  asm volatile("" : "+v"(x));
}
template <int D, typename R>
__device__ __forceinline__ Basis4<R> basis4(R x) {
  return Basis4<R>{pbasis<D>(0, x), pbasis<D>(1, x), sbasis<D>(0, x), sbasis<D>(1, x)};
}
template <int D, typename R>
__device__ __forceinline__ Basis4<R> dbasis4(R x, R y) {
  return Basis4<R>{dpbasis<D>(0, x, y), dpbasis<D>(1, x, y), dsbasis<D>(0, x, y), dsbasis<D>(1, x, y)};
}

// Below these differences the discrete gradient takes the derivative form
// (LTEHelmholtzEOS.hpp:246-300): the reference's 2.22e-15 + 1.49e-8 x (about
// 10 eps and sqrt(eps) of FP64), and the same multiples of FP32's epsilon
// for the mixed-precision form.
template <typename R>
struct SecantTol {
  static constexpr double abs = 2.22e-15, rel = 1.49e-8;
};
template <>
struct SecantTol<float> {
  static constexpr float abs = 1.19e-6f, rel = 3.45e-4f;
};

// The order in which a pair enters the discrete gradients
// (LTEHelmholtzEOS.hpp:231-244): by density, then temperature
template <typename R>
__device__ __forceinline__ bool pair_reversed(R rho1, R T1, R rho2, R T2) {
  return rho1 > rho2 || (rho1 == rho2 && T1 > T2);
}

// The entropy-conserving density and energy means (LTEHelmholtzEOS.hpp:
// 225-397) of an ordered pair: the Itoh-Abe discrete gradients of p/T and g/T
// in (rho, 1/T).  `fall(side, k)` gives H_rhorho (2), H_T (3) or H_rhoT (4)
// of endpoint a (0) or b (1) for the derivative form, rarely needed.
//
// Every evaluation at an endpoint itself comes with the nodes (evaluated
// once per node and stage instead of in each of its pairs).  What is left is
// H and H_rho at the two cross corners (rho_a, T_b) and (rho_b, T_a), needed
// in both cases -- by the secants when the endpoints share a cell, by the
// corner differences when not, the searches of at() then finding exactly the
// cells (i_a, j_b) and (i_b, j_a) -- and, in a shared cell, eight divided
// differences: 12 sums of 16 products from 6 rho bases, where taking each
// gradient by itself evaluated 24 sums and 4 to 12 more per divergent branch.
template <typename R, typename F>
__device__ __forceinline__ void thermodynamic_means(const View &v, const PairNode<R> &a, const PairNode<R> &b, F fall,
                                                    R &rho_mean, R &e_mean) {
  const R b1 = a.beta, b2 = b.beta;
  const R dr = b.rho - a.rho, db = b2 - b1;
  const R rmax = a.rho > b.rho ? a.rho : b.rho;
  const R bmax = b1 > b2 ? b1 : b2;
  const bool dd = fabs(dr) >= R(SecantTol<R>::abs) + R(SecantTol<R>::rel) * rmax;
  const bool bd = fabs(db) >= R(SecantTol<R>::abs) + R(SecantTol<R>::rel) * bmax;
  const R p11 = pair_pressure(a), p22 = pair_pressure(b);
  const R g11 = a.H + a.rho * a.Hr, g22 = b.H + b.rho * b.Hr;
  R pd = 0, gd = 0, pb = 0, gb = 0;  // the density and beta components of the two gradients
  if (dd || bd) {
    const int ia = a.cell & 0xFFFF, ja = a.cell >> 16, ib = b.cell & 0xFFFF, jb = b.cell >> 16;
    const bool same = a.cell == b.cell;
    const R *ca = cells_of<R>(v) + (size_t)(jb * v.nx + ia) * kCellStride;
    const R *cb = cells_of<R>(v) + (size_t)(ja * v.nx + ib) * kCellStride;
    const Basis4<R> dt = dbasis4<0, R>(a.eta, b.eta);
    R c[16], P[16];
    R hx, gx, hdt_a, gdt_a, hy, gy, hdt_b, gdt_b;
    {
      const Basis4<R> tb = basis4<0, R>(b.eta);
#pragma unroll
      for (int m = 0; m < 16; ++m) c[m] = ca[m];
      cell_row(c, basis4<1, R>(a.xi), P);
      hx = div_by(cell_dot(P, tb), ca[16], ca[18]);  // H_rho(rho_a, T_b)
      hdt_a = cell_dot(P, dt);
      pin(hdt_a);
      __builtin_amdgcn_sched_barrier(0);
      cell_row(c, basis4<0, R>(a.xi), P);
      gx = cell_dot(P, tb);  // H(rho_a, T_b)
      gdt_a = cell_dot(P, dt);
      pin(gdt_a);
    }
    {
      __builtin_amdgcn_sched_barrier(0);
      const Basis4<R> ta = basis4<0, R>(a.eta);
#pragma unroll
      for (int m = 0; m < 16; ++m) c[m] = cb[m];
      cell_row(c, basis4<1, R>(b.xi), P);
      hy = div_by(cell_dot(P, ta), cb[16], cb[18]);  // H_rho(rho_b, T_a)
      hdt_b = cell_dot(P, dt);
      pin(hdt_b);
      __builtin_amdgcn_sched_barrier(0);
      cell_row(c, basis4<0, R>(b.xi), P);
      gy = cell_dot(P, ta);  // H(rho_b, T_a)
      gdt_b = cell_dot(P, dt);
      pin(gdt_b);
    }
    if (same) {
      const R wr = cb[16], wt = cb[17], iwr = cb[18], iwt = cb[19], iwrr = cb[20], iwrt = cb[21];
      if (dd) {
        const Basis4<R> ta = basis4<0, R>(a.eta), tb = basis4<0, R>(b.eta);
        cell_row(c, dbasis4<1, R>(a.xi, b.xi), P);
        R dhr1 = div_by(cell_dot(P, ta), wr * wr, iwrr), dhr2 = div_by(cell_dot(P, tb), wr * wr, iwrr);
        pin(dhr1);
        pin(dhr2);
        __builtin_amdgcn_sched_barrier(0);
        cell_row(c, dbasis4<0, R>(a.xi, b.xi), P);
        const R dh1 = div_by(cell_dot(P, ta), wr, iwr), dh2 = div_by(cell_dot(P, tb), wr, iwr);
        const R m1 = R(0.5) * (a.Hr + hy), m2 = R(0.5) * (hx + b.Hr);
        const R r2m = R(0.5) * (a.rho * a.rho + b.rho * b.rho), rs = a.rho + b.rho;
        const R p1 = r2m * dhr1 + rs * m1, p2 = r2m * dhr2 + rs * m2;
        pd = R(0.5) * (p1 * b1 + p2 * b2);
        const R g1 = dh1 + R(0.5) * rs * dhr1 + m1, g2 = dh2 + R(0.5) * rs * dhr2 + m2;
        gd = R(0.5) * (g1 * b1 + g2 * b2);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (bd) {
        const R mean_t = R(0.5) * (a.T + b.T);
        const R hb1 = R(0.5) * (a.Hr + hx) - mean_t * div_by(hdt_a, wr * wt, iwrt);
        const R hb2 = R(0.5) * (hy + b.Hr) - mean_t * div_by(hdt_b, wr * wt, iwrt);
        pb = R(0.5) * (a.rho * a.rho * hb1 + b.rho * b.rho * hb2);
        const R g1 = R(0.5) * (a.H + gx) - mean_t * div_by(gdt_a, wt, iwt) + a.rho * hb1;
        const R g2 = R(0.5) * (gy + b.H) - mean_t * div_by(gdt_b, wt, iwt) + b.rho * hb2;
        gb = R(0.5) * (g1 + g2);
      }
    } else {
      const R p12 = a.rho * a.rho * hx, p21 = b.rho * b.rho * hy;
      const R g12 = gx + a.rho * hx, g21 = gy + b.rho * hy;
      if (dd) {
        const R y = 1 / dr;
        pd = div_by(R(0.5) * ((p21 * b1 - p11 * b1) + (p22 * b2 - p12 * b2)), dr, y);
        gd = div_by(R(0.5) * ((g21 * b1 - g11 * b1) + (g22 * b2 - g12 * b2)), dr, y);
      }
      if (bd) {
        const R y = 1 / db;
        pb = div_by(R(0.5) * ((p12 * b2 - p11 * b1) + (p22 * b2 - p21 * b1)), db, y);
        gb = div_by(R(0.5) * ((g12 * b2 - g11 * b1) + (g22 * b2 - g21 * b1)), db, y);
      }
    }
  }
  if (!dd) {
    const R h1 = fall(0, 2), h2 = fall(1, 2);  // H_rhorho
    pd = R(0.5) * ((2 * a.rho * a.Hr + a.rho * a.rho * h1) * b1 + (2 * b.rho * b.Hr + b.rho * b.rho * h2) * b2);
    gd = R(0.5) * ((2 * a.Hr + a.rho * h1) * b1 + (2 * b.Hr + b.rho * h2) * b2);
  }
  if (!bd) {
    const R t1 = fall(0, 3), t2 = fall(1, 3), rt1 = fall(0, 4), rt2 = fall(1, 4);  // H_T, H_rhoT
    pb = R(0.5) * ((p11 - a.T * (a.rho * a.rho * rt1)) + (p22 - b.T * (b.rho * b.rho * rt2)));
    gb = R(0.5) * ((g11 - a.T * (t1 + a.rho * rt1)) + (g22 - b.T * (t2 + b.rho * rt2)));
  }
  rho_mean = pd / gd;
  e_mean = gb - pb / rho_mean;
}

// LTEECFlux.hpp:11-85 from the entropy-conserving means, the endpoints'
// states and pressures and, for faces, sound speeds; pd1, pd2: the pressures
// of the momentum flux's pressure term (p less a constant background in the
// mixed-precision form, which the divergence does not see; p itself in FP64)
template <int DIM, bool FACE, typename R>
__device__ __forceinline__ void lteec_flux(R rho_m, R e_m, const R *q1, const R *q2, R p1, R p2, R c1, R c2,
                                           const R *dir, R *F, R pd1, R pd2) {
  const R pm = R(0.5) * (pd1 + pd2);
  const R ir1 = R(1.0) / q1[0], ir2 = R(1.0) / q2[0];
  R vn = 0, ck = 0, pw = 0, v1n = 0, v2n = 0, n2 = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const R u1 = q1[1 + d] * ir1, u2 = q2[1 + d] * ir2;
    vn += R(0.5) * (u1 + u2) * dir[d];
    ck += R(0.5) * u1 * u2;
    pw += R(0.5) * (p1 * u2 + p2 * u1) * dir[d];
    if (FACE) {
      v1n += u1 * dir[d];
      v2n += u2 * dir[d];
      n2 += dir[d] * dir[d];
    }
  }
  R diss = 0;
  if (FACE) {
    const R nm = sqrt(n2);
    const R sp1 = fabs(v1n) + c1 * nm, sp2 = fabs(v2n) + c2 * nm;
    diss = R(0.5) * (sp1 > sp2 ? sp1 : sp2);
  }
  const R mass = rho_m * vn;
  F[0] = mass - diss * (q2[0] - q1[0]);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const R vel = R(0.5) * (q1[1 + d] * ir1 + q2[1 + d] * ir2);
    F[1 + d] = mass * vel + pm * dir[d] - diss * (q2[1 + d] - q1[1 + d]);
  }
  F[DIM + 1] = mass * (e_m + ck) + pw - diss * (q2[DIM + 1] - q1[DIM + 1]);
}
// What k_lte_nodes leaves per node: the temperature and cell alone (the
// stability estimate), with what LTEEC takes at a node, or with what the
// other pairs take (View::node_*).
enum NodeOut { NODE_T = 0, NODE_LTEEC = 1, NODE_PC = 2 };

// Temperature and table cell of every node of a state and the flux pair's
// node values there, one lane per node, once per node and stage for the RHS
// kernel's staged nodes and its neighbours' face points.  The recovery is
// temperature_from_energy (LTEHelmholtzEOS.hpp:151-223) with its searches and
// sums arranged for the loop: the density cell is found once, a temperature
// cell only when the iterate leaves the last one, and the 16 products of the
// cell's coefficients with the density basis are kept until then, so that an
// iteration is three sums of 16 products; the operations that round are its
// own, in its order.  The node values follow in the same kernel, where the
// cell's record is at hand.  Latency of the dependent lookups (state, bucket,
// inverse table, bucket, record) at 4 to 5 waves per SIMD bounds it.  At 24^3
// elements, p = 3 (884,736 nodes): 41 us with LTEEC's values, 42 us with the
// other pairs', against 72 us for the recovery alone with both cells bisected
// in every iteration and 39 (22) us for the values in a pass of their own.
template <int DIM, int OUT, typename R = double>
__global__ void __launch_bounds__(256) k_lte_nodes(const double *U, long long Ntot, View v) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= Ntot) return;
  double q[DIM + 2];
#pragma unroll
  for (int c = 0; c < DIM + 2; ++c) q[c] = U[c * Ntot + t];
  double m2 = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) m2 += q[1 + d] * q[1 + d];
  const double rho = q[0];
  const double e = (q[DIM + 1] - 0.5 * m2 / rho) / rho;
  double rlo = 0, rhi = 1, elo = 0, ehi = 1;
  const int i = find_cell(v.rho, v.nx, v.brho, rho, rlo, rhi);
  const int ie = find_cell(v.e, v.ny, v.be, e, elo, ehi);
  double T = __builtin_nan(""), xi = T;
  int j = -1;         // cell of the last evaluated temperature, [Tlo, Thi) (closed at the grid's end)
  double Tlo = 0, Thi = 0, wt = 1, iwt = 1, iwtt = 1;
  const double *rec = v.cells64;
  double P[16];       // its coefficients times the density basis
  const double Tmin = v.T[0], Tmax = v.T[v.ny - 1];
  // makes j, Tlo, Thi and rec those of the temperature x; false outside the grid
  auto locate = [&](double x) {
    if (j >= 0 && x >= Tlo && x < Thi) return true;
    const int n = find_cell(v.T, v.ny, v.bT, x, Tlo, Thi);
    if (n < 0) return false;
    j = n;
    rec = v.cells64 + (size_t)(j * v.nx + i) * kCellStride;
    wt = rec[17];
    iwt = rec[19];
    iwtt = rec[22];
    return true;
  };
  auto rho_rows = [&](auto D) {
    constexpr int K = decltype(D)::value;
    cell_row(rec, basis4<K, double>(xi), P);
  };
  if (i >= 0 && ie >= 0) {
    xi = (rho - rlo) / (rhi - rlo);
    const double y = (e - elo) / (ehi - elo);
    const double *p = v.inv + ie * v.nx + i;
    const double lower = p[0] + xi * (p[1] - p[0]);
    const double upper = p[v.nx] + xi * (p[v.nx + 1] - p[v.nx]);
    double x = lower + y * (upper - lower);
    int last = -1;
    for (int it = 0; it < 100; ++it) {
      if (!locate(x)) break;
      if (j != last) {
        rho_rows(std::integral_constant<int, 0>{});
        last = j;
      }
      const double eta = div_by(x - Tlo, wt, iwt);
      const double h = cell_dot(P, basis4<0, double>(eta));
      const double hT = div_by(cell_dot(P, basis4<1, double>(eta)), wt, iwt);
      const double hTT = div_by(cell_dot(P, basis4<2, double>(eta)), wt * wt, iwtt);
      const double cv = -x * hTT, guess = h - x * hT;
      if (!(cv > 0) || !isfinite(guess)) break;
      const double step = (e - guess) / cv;
      const double next = x + step;
      const bool inside = isfinite(next) && next >= Tmin && next <= Tmax;
      if (fabs(step) <= 1e-9 + 1e-12 * x) {
        T = next < Tmin ? Tmin : (next > Tmax ? Tmax : next);
        break;
      }
      x = next;
      if (!inside) break;
    }
  }
  const bool ok = i >= 0 && locate(T);
  v.node_T[t] = T;
  v.node_cell[t] = ok ? (i | (j << 16)) : -1;
  if constexpr (OUT != NODE_T) {
    // a node outside the table reads cell (0, 0) at NaN coordinates
    double eta = __builtin_nan("");
    if (ok) {
      eta = div_by(T - Tlo, wt, iwt);
    } else {
      xi = eta;
      rec = v.cells64;
    }
    const double wr = rec[16];
    const Basis4<double> t0 = basis4<0, double>(eta), t1 = basis4<1, double>(eta);
    rho_rows(std::integral_constant<int, 0>{});
    const double hTT = div_by(cell_dot(P, basis4<2, double>(eta)), wt * wt, iwtt);
    double h = 0, hT = 0;
    if constexpr (OUT == NODE_LTEEC && sizeof(R) == sizeof(double)) {
      h = cell_dot(P, t0);
      hT = div_by(cell_dot(P, t1), wt, iwt);
    }
    rho_rows(std::integral_constant<int, 1>{});
    const double hr = div_by(cell_dot(P, t0), wr, rec[18]);
    const double m = div_by(cell_dot(P, t1), wr * wt, rec[21]);
    rho_rows(std::integral_constant<int, 2>{});
    const double hrr = div_by(cell_dot(P, t0), wr * wr, rec[20]);
    const double p_rho = 2 * rho * hr + rho * rho * hrr;
    v.node_c[t] = sqrt(p_rho - rho * rho * m * m / hTT);
    if constexpr (OUT == NODE_PC) {
      v.node_p[t] = rho * rho * hr;
      if (v.node_g) {
        const double cv = -T * hTT;
        v.node_g[t] = (cv + T * rho * rho * m * m / p_rho) / cv;
      }
    } else {
      R *o = static_cast<R *>(v.node_rec) + t;
      if constexpr (sizeof(R) == sizeof(double)) {
        o[0] = h;
        o[Ntot] = hr;
        o[2 * Ntot] = hrr;
        o[3 * Ntot] = hT;
        o[4 * Ntot] = m;
      } else {
        v.node_p[t] = rho * rho * hr;
        const Eval<R> er = at_packed<R>(v, R(rho), R(T), ok ? (i | (j << 16)) : -1);
        o[0] = er.H();
        o[Ntot] = er.template H<1, 0>();
        o[2 * Ntot] = er.template H<2, 0>();
        o[3 * Ntot] = er.template H<0, 1>();
        o[4 * Ntot] = er.template H<1, 1>();
      }
    }
  }
}

// ---- the viscous path (LTEGasModel<LTEHelmholtzGasEOS, LTETransport>,
//      LTEGasModel.hpp:339; LTETransport.hpp:32-65 without SUTHERLAND)

// A node's quantities for the viscous flux: velocity, recovered temperature,
// tabulated viscosity and conductivity
template <int DIM, typename R = double>
struct ViscNode {
  R u[DIM];
  R T, mu, kappa;
};

// The entropy variables the viscous flux depends on, (u/T, -1/T), of a node
// whose temperature was recovered (LTEHelmholtzGasEOS.hpp:144-157; the first,
// (g - |u|^2/2)/T, does not enter the conversion to grad u and grad T,
// :159-171, so g is not evaluated)
template <int DIM, typename R>
__device__ __forceinline__ void viscous_variables(const R *q, R T, R *S) {
  const R beta = 1 / T;
#pragma unroll
  for (int d = 0; d < DIM; ++d) S[d] = beta * (q[1 + d] / q[0]);
  S[DIM] = -beta;
}

template <int DIM, typename R>
__device__ __forceinline__ ViscNode<DIM, R> visc_node(const View &v, const R *q, R T, int cell) {
  const Eval<R> s = at_packed<R>(v, q[0], T, cell);
  ViscNode<DIM, R> n;
#pragma unroll
  for (int d = 0; d < DIM; ++d) n.u[d] = q[1 + d] / q[0];
  n.T = T;
  n.mu = v.sutherland ? R(sutherland_viscosity(v, double(T))) : s.template transport<4>();
  n.kappa = s.template transport<5>();
  return n;
}

// The mixed-precision form's background pressure: the pressure of node 0 of
// a state (one lane writes it), as the ideal gas's k_pref takes it
template <int DIM>
__global__ void __launch_bounds__(64) k_pref_lte(const double *U, long long Ntot, View v, double *pref);

// A point's evaluated state from its conservative vector (LTEHelmholtzGasEOS.hpp:60-77)
template <int DIM>
__device__ __forceinline__ Eval<double> state_eval(const View &v, const double *q) {
  double m2 = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) m2 += q[1 + d] * q[1 + d];
  const double rho = q[0];
  const double e = (q[DIM + 1] - 0.5 * m2 / rho) / rho;
  const double T = temperature_from_energy(v, rho, e);
  return at<double>(v, rho, T);
}

template <int DIM>
__global__ void __launch_bounds__(64) k_pref_lte(const double *U, long long Ntot, View v, double *pref) {
  if (threadIdx.x != 0) return;
  double q[DIM + 2];
#pragma unroll
  for (int c = 0; c < DIM + 2; ++c) q[c] = U[c * Ntot];
  pref[0] = state_eval<DIM>(v, q).pressure();
}

}  // namespace lte
}  // namespace thx

#pragma clang fp contract(fast)
