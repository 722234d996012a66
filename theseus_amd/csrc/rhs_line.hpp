// The fused FP64 volume + face kernel of the ideal gas in line form: one lane per
// GLL line instead of one per node.
//
// A wave of 64 lanes holds the Np^(DIM-1) lines of as many elements as fit
// (3-D p = 3: 16 lines of 4 elements).  For each direction in turn a lane
// takes the nodes of its line into registers, evaluates the line's
// Np (Np - 1) / 2 two-point fluxes and the Riemann fluxes at both of its ends
// (the line's end nodes are the face points of that direction), and adds them
// to its nodes' running sums.  Between directions the sums move to the lanes
// of the next direction's lines through LDS, one field at a time.  So no
// flux rows, pair lists, face lists or per-node index arithmetic exist, every
// element-wise quantity (normals, Jacobian) is loaded by the lanes that use
// it, and a workgroup is one wave without barriers.
//
// Memory bounds it: HBM (on 32^3 elements, p = 3, with viscous terms 506 MB a
// launch, 98 us at the rate of a copy) and the vector memory path to it (TD
// busy 80 % of the time), not the FP64 issue (35 %).  So own data moves in
// memory order, 512 consecutive bytes a wave instruction, and changes to lines
// in LDS, neighbours along x come from the wave's own LDS, and per-element
// values are loaded by consecutive lanes once.  With a lane loading and storing
// its x-line's nodes (32 bytes apart) and each element's values in all its
// lanes, an SSP-RK3 step on 48^3 elements, p = 3, Ranocha/LLF with viscous terms
// took 1761 us, now 1540 (k_ns_grad_line's share included); an Euler evaluation
// on 17 x 15 x 13 elements at p = 4 24.5 us, now 22.3.  On 32^3 elements the
// kernel takes 96 to 107 us, on different cards, for the node form's 145 to 173,
// with 21 M vector instructions for 53 M, at 240 registers: two waves a SIMD
// (three spill and are slower).
#pragma once

#include "rhs_kernels.hpp"

namespace thx {

template <int DIM, int P>
struct LineShape {
  static constexpr int Np = P + 1;
  static constexpr int NL = DIM == 2 ? Np : Np * Np;  // lines of an element per direction
  static constexpr int ND = NL * Np;
  static constexpr int NQ = DIM + 2;
  static constexpr int EPW = 64 / NL;                 // elements of a wave
  // staged nodes leave one slot free after every x-line (StagedIndex), so
  // that the lanes of a wave read the nodes of x, y and z lines from
  // distinct LDS banks
  static constexpr int NDS = ND + NL;
  static_assert(EPW >= 1, "an element's lines fit one wave");
};

// Index of a wave's line t in direction d within an element's staged nodes:
// its first node and the stride between its nodes.
template <int Np>
__device__ __forceinline__ int line_base(int d, int t) {
  const int lo = t % Np, hi = t / Np;
  return d == 0 ? (Np + 1) * t : (d == 1 ? lo + (Np * Np + Np) * hi : lo + (Np + 1) * hi);
}
template <int Np>
__device__ __forceinline__ int line_stride(int d) {
  return d == 0 ? 1 : (d == 1 ? Np + 1 : Np * Np + Np);
}

// The branch of log_mean_pair that all logarithmic means of a line's pairs
// (of the densities and of the rho_1 p_2, rho_2 p_1) can take: 0 its first
// series, 1 its second, 2 neither.  Tested on the products of the
// extremes, whose ratio bounds every pair's; the second series holds below the
// first one's bound too, where the two agree to rounding.
template <int DIM, int Np>
__device__ __forceinline__ int line_series(const Pt<double, DIM> *s) {
  double r0 = s[0].q[0], r1 = r0, p0 = s[0].p, p1 = p0;
#pragma unroll
  for (int m = 1; m < Np; ++m) {
    r0 = dmin(r0, s[m].q[0]);
    r1 = dmax(r1, s[m].q[0]);
    p0 = dmin(p0, s[m].p);
    p1 = dmax(p1, s[m].p);
  }
  const double x = r0 * p0, y = r1 * p1, d = y - x, sum = x + y;
  if (!(r0 > 0.0 && p0 > 0.0)) return 2;
  const double dd = d * d, ss = sum * sum;
  if (dd < 0.98 * LogMeanEps<double>::value * ss) return 0;
  return dd < 0.98 * 0.0294 * ss ? 1 : 2;
}

#pragma clang fp contract(off)
// 2 sum_{k <= 11} u^k/(2k+1): log_mean_pair's second series, doubled
__device__ __forceinline__ double atanh_series2(double u) {
  double p = 2.0 / 23.0;
  p = fma(p, u, 2.0 / 21.0);
  p = fma(p, u, 2.0 / 19.0);
  p = fma(p, u, 2.0 / 17.0);
  p = fma(p, u, 2.0 / 15.0);
  p = fma(p, u, 2.0 / 13.0);
  p = fma(p, u, 2.0 / 11.0);
  p = fma(p, u, 2.0 / 9.0);
  p = fma(p, u, 2.0 / 7.0);
  p = fma(p, u, 0.4);
  p = fma(p, u, 2.0 / 3.0);
  return fma(p, u, 2.0);
}

// One line's volume terms with Ranocha's flux (RanochaFlux.hpp:20-79) in
// FP64, all logarithmic means in one of their series (LONG: the second): what
// depends on one node only -- half its normal velocity, p/(gamma-1) -- is
// formed once per node instead of once per pair, and the factors of one half
// are folded into it and into the series' coefficients; 50 operations a pair
// (LONG: 72).
template <bool LONG, int DIM, int Np>
__device__ __forceinline__ void line_ranocha_f64(const GasC<double> &g, const Pt<double, DIM> *s, const double *met,
                                                 const double *D2, double (*rate)[DIM + 2]) {
  double hvn[Np], pg[Np], hm[DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d) hm[d] = 0.5 * met[d];
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    hvn[m] = s[m].v[0] * hm[0];
#pragma unroll
    for (int d = 1; d < DIM; ++d) hvn[m] = fma(s[m].v[d], hm[d], hvn[m]);
    pg[m] = s[m].p * g.gammaM1Inverse;
  }
#pragma unroll
  for (int a = 0; a < Np; ++a)
#pragma unroll
    for (int b = a + 1; b < Np; ++b) {
      const double ra = s[a].q[0], rb = s[b].q[0], pa = s[a].p, pb = s[b].p;
      const double sr = ra + rb, tr = (rb - ra) * recip_nr(sr), ur = tr * tr;
      const double x = ra * pb, y = rb * pa, sx = x + y, rs = recip_nr(sx), tx = (y - x) * rs, ux = tx * tx;
      double lm, inv;  // LM(ra, rb) and 1/LM(x, y)
      if constexpr (LONG) {
        lm = sr * recip_nr(atanh_series2(ur));
        inv = rs * atanh_series2(ux);
      } else {
        lm = sr * fma(-ur, fma(ur, fma(ur, 22.0 / 945.0, 2.0 / 45.0), 1.0 / 6.0), 0.5);
        inv = rs * fma(ux, fma(ux, fma(ux, 2.0 / 7.0, 0.4), 2.0 / 3.0), 2.0);
      }
      const double mass = lm * (hvn[a] + hvn[b]), h = 0.5 * mass, ps = pa + pb;
      double dot = s[a].v[0] * s[b].v[0];
#pragma unroll
      for (int d = 1; d < DIM; ++d) dot = fma(s[a].v[d], s[b].v[d], dot);
      double F[DIM + 2];
      F[0] = mass;
#pragma unroll
      for (int d = 0; d < DIM; ++d) F[1 + d] = fma(h, s[a].v[d] + s[b].v[d], ps * hm[d]);
      F[DIM + 1] = fma(mass, fma(0.5, dot, (pg[a] * pb) * inv), fma(pa, hvn[b], pb * hvn[a]));
#pragma unroll
      for (int q = 0; q < DIM + 2; ++q) {
        rate[a][q] = fma(D2[a * Np + b], F[q], rate[a][q]);
        rate[b][q] = fma(D2[b * Np + a], F[q], rate[b][q]);
      }
    }
}

// Square root of a normal x by Goldschmidt's iteration from the hardware
// estimate, with a final remainder correction (within an ulp); 0 and infinity
// themselves, NaN below.  10 instructions for the 20 of the correctly rounded
// form, which also scales for subnormal arguments.
__device__ __forceinline__ double sqrt_nr(double x) {
  constexpr int kZeroOrInfinity = 1 << 5 | 1 << 6 | 1 << 9;  // -0, +0, +infinity of v_cmp_class
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  g = fma(fma(-g, g, x), h, g);
  return __builtin_amdgcn_class(x, kZeroOrInfinity) ? x : g;
}

// A face point's Lax-Friedrichs flux (LaxFriedrichsFlux.hpp:188-211) in FP64,
// lifted onto rate: rate += lift F, F = (f(own) + f(oth))/2 - (sg lambda/2)
// (q_oth - q_own), the low side first when sg = 1 (face_llf_signed); sub is
// subtracted from f(own) + f(oth).  f takes v.n first (m = rho v.n, m_c v.n +
// p n_c, (E + p) v.n), every fused operation written out so that both
// elements of a face form the same flux.
template <int DIM>
__device__ __forceinline__ void lift_llf_f64(const GasC<double> &g, const Pt<double, DIM> &own,
                                             const Pt<double, DIM> &oth, const double *n, double sg, double lift,
                                             const double *sub, double *rate) {
  double nn = n[0] * n[0], v1 = own.v[0] * n[0], v2 = oth.v[0] * n[0];
#pragma unroll
  for (int d = 1; d < DIM; ++d) {
    nn = fma(n[d], n[d], nn);
    v1 = fma(own.v[d], n[d], v1);
    v2 = fma(oth.v[d], n[d], v2);
  }
  const double nrm = sqrt_nr(nn);
  const double c1 = sqrt_nr(g.gamma * own.p * own.ir), c2 = sqrt_nr(g.gamma * oth.p * oth.ir);
  const double lambda = dmax(fma(nrm, c1, fabs(v1)), fma(nrm, c2, fabs(v2)));
  const double hl = 0.5 * lift, dl = -(sg * hl) * lambda;
  const double ps = own.p + oth.p;
  auto add = [&](int q, double f) { rate[q] = fma(dl, oth.q[q] - own.q[q], fma(hl, f, rate[q])); };
  double f1, f2;
  f1 = own.q[0] * v1;
  f2 = oth.q[0] * v2;
  add(0, f1 + f2);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    f1 = own.q[1 + d] * v1;
    f2 = oth.q[1 + d] * v2;
    add(1 + d, fma(ps, n[d], f1 + f2) - sub[d]);
  }
  f1 = (own.q[DIM + 1] + own.p) * v1;
  f2 = (oth.q[DIM + 1] + oth.p) * v2;
  add(DIM + 1, (f1 + f2) - sub[DIM]);
}

#pragma clang fp contract(fast)

// One line's volume terms: rate[m] += sum_{l != m} Dhat2(m, l) F#(m, l)
template <int VOL, bool SERIES, int DIM, int Np>
__device__ __forceinline__ void line_volume(const GasC<double> &g, const Pt<double, DIM> *s, const double *met, const double *D2,
                                            double (*rate)[DIM + 2]) {
#pragma unroll
  for (int a = 0; a < Np; ++a)
#pragma unroll
    for (int b = a + 1; b < Np; ++b) {
      double F[DIM + 2];
      volume_flux<VOL, double, DIM, SERIES>(g, s[a], s[b], met, F);
#pragma unroll
      for (int q = 0; q < DIM + 2; ++q) {
        rate[a][q] += D2[a * Np + b] * F[q];
        rate[b][q] += D2[b * Np + a] * F[q];
      }
    }
}

// What the lanes of a wave share of its elements e0, ..., e0 + nv - 1: loaded
// by consecutive lanes (a load per lane of the one value its element's lanes
// all need would occupy the vector memory path as much as a node's), read
// from LDS.  Elements past the last hold the last one's.
template <int DIM, int P>
struct LineMeta {
  static constexpr int EPW = LineShape<DIM, P>::EPW;
  double adj[EPW][DIM * DIM];
  double J[EPW];
  int nbr[EPW][2 * DIM];

  // one lane's loads, issued before they are stored
  struct Regs {
    static constexpr int NA = (EPW * DIM * DIM + 63) / 64, NN = (EPW * 2 * DIM + 63) / 64;
    double adj[NA], J;
    int nbr[NN];
  };
  __device__ static __forceinline__ Regs load(const RHSCore &a, int e0, int nv, int lane) {
    Regs r;
#pragma unroll
    for (int k = 0; k < Regs::NN; ++k) r.nbr[k] = a.nbr[(size_t)e0 * 2 * DIM + min(lane + 64 * k, nv * 2 * DIM - 1)];
#pragma unroll
    for (int k = 0; k < Regs::NA; ++k) r.adj[k] = a.adj[(size_t)e0 * DIM * DIM + min(lane + 64 * k, nv * DIM * DIM - 1)];
    r.J = a.J[e0 + min(lane, nv - 1)];
    return r;
  }
  __device__ __forceinline__ void store(const Regs &r, int lane) {
#pragma unroll
    for (int k = 0; k < Regs::NN; ++k)
      if (lane + 64 * k < EPW * 2 * DIM) (&nbr[0][0])[lane + 64 * k] = r.nbr[k];
#pragma unroll
    for (int k = 0; k < Regs::NA; ++k)
      if (lane + 64 * k < EPW * DIM * DIM) (&adj[0][0])[lane + 64 * k] = r.adj[k];
    if (lane < EPW) J[lane] = r.J;
  }
};

template <int DIM, int P>
struct LineLds {
  using S = LineShape<DIM, P>;
  double q[S::NQ][S::EPW * S::NDS];
  double x[S::EPW * S::NDS];  // one field on its way between directions
  LineMeta<DIM, P> m;
  double nl[S::EPW][DIM * DIM];  // the adjugate rows of the low-side neighbours
};

// Moves one value per node from the lines of one direction to those of
// another: LDS operations of a wave execute in order, so neither a barrier
// nor a second buffer is needed between fields.
template <int Np>
__device__ __forceinline__ void line_move(double *buf, int from, int fstride, int to, int tstride, double *v) {
#pragma unroll
  for (int m = 0; m < Np; ++m) buf[from + m * fstride] = v[m];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int m = 0; m < Np; ++m) v[m] = buf[to + m * tstride];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// The running sums' move, one field at a time
template <int DIM, int P>
__device__ __forceinline__ void line_move_sums(LineLds<DIM, P> &L, int from, int fstride, int to, int tstride,
                                               double (*rate)[DIM + 2]) {
  constexpr int Np = P + 1;
#pragma unroll
  for (int c = 0; c < DIM + 2; ++c) {
    double v[Np];
#pragma unroll
    for (int m = 0; m < Np; ++m) v[m] = rate[m][c];
    line_move<Np>(L.x, from, fstride, to, tstride, v);
#pragma unroll
    for (int m = 0; m < Np; ++m) rate[m][c] = v[m];
  }
}

// v of the lane N further in its row of 16 (cyclic)
template <int N>
__device__ __forceinline__ double row_rotate(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + N, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + N, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// blending_alpha in line form: f holds pressure * density (FP64) at the lane's
// x-line nodes.  The sums over an element's modes pair the operands as
// blending_alpha's tree does where its lines fill a power of two of lanes.
template <int DIM, int P>
__device__ __forceinline__ double line_alpha(const RHSCore &a, ConstBasis &B, double *buf, int el, int t, double *f) {
  using S = LineShape<DIM, P>;
  constexpr int Np = S::Np, NL = S::NL, NDS = S::NDS;
  auto sweep = [&] {
    double o[Np];
#pragma unroll
    for (int k = 0; k < Np; ++k) {
      o[k] = 0.0;
#pragma unroll
      for (int l = 0; l < Np; ++l) o[k] += B.Vinv[k * Np + l] * f[l];
    }
#pragma unroll
    for (int k = 0; k < Np; ++k) f[k] = o[k];
  };
  double *b = buf + el * NDS;
  sweep();
#pragma unroll
  for (int d = 1; d < DIM; ++d) {
    line_move<Np>(b, line_base<Np>(d - 1, t), line_stride<Np>(d - 1), line_base<Np>(d, t), line_stride<Np>(d), f);
    sweep();
  }
  // modes (t % Np, t / Np, m) of the last direction's line (2-D: (t, m))
  const int i = t % Np, j = t / Np;
  double s[3] = {0.0, 0.0, 0.0};
  const bool k1 = DIM == 2 ? t <= P - 1 : (i <= P - 1 && j <= P - 1);
  const bool k2 = DIM == 2 ? t <= P - 2 : (i <= P - 2 && j <= P - 2);
  double m2[Np];
#pragma unroll
  for (int m = 0; m < Np; ++m) m2[m] = f[m] * f[m];
  auto sum = [&](int upto) {
    if constexpr (Np == 4) return upto >= 3 ? (m2[0] + m2[2]) + (m2[1] + m2[3]) : (upto == 2 ? (m2[0] + m2[2]) + m2[1] : m2[0] + m2[1]);
    double r = 0.0;
#pragma unroll
    for (int m = 0; m < Np; ++m)
      if (m <= upto) r += m2[m];
    return r;
  };
  s[0] = sum(P);
  s[1] = k1 ? sum(P - 1) : 0.0;
  s[2] = k2 && P >= 2 ? sum(P - 2) : 0.0;
  if constexpr ((NL & (NL - 1)) == 0) {
    // a row of 16 lanes holds 16 / NL elements; rotations within the row pair
    // the lanes as exclusive-or does once the larger offsets are summed
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (NL == 16) {
        s[c] += row_rotate<8>(s[c]);
        s[c] += row_rotate<4>(s[c]);
        s[c] += row_rotate<2>(s[c]);
        s[c] += row_rotate<1>(s[c]);
      } else {
#pragma unroll
        for (int off = NL / 2; off > 0; off >>= 1) s[c] += __shfl_xor(s[c], off, 64);
      }
    }
  } else {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < 3; ++c) b[c * NL + t] = s[c];  // 3 NL <= NDS
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double r = 0.0;
      for (int l = 0; l < NL; ++l) r += b[c * NL + l];
      s[c] = r;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  return alpha_of_modes(a, s[0], s[1], s[2]);
}

// A load or store at a wave-uniform base plus a 32-bit byte offset, which
// needs no 64-bit address arithmetic per lane.
template <typename T>
__device__ __forceinline__ T ld(const T *base, unsigned byte) {
  return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte);
}
template <typename T>
__device__ __forceinline__ void st(T *base, unsigned byte, T v) {
  *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + byte) = v;
}

// Meshes whose fields and n.Fv rows can be addressed with 32-bit byte offsets;
// BND: with boundary faces (Euler).
template <int DIM, int P, int VOL, int SURF, bool VISC, bool BND = false>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_rhs_line(RHSArgs a) {
  static_assert(!(VISC && BND), "boundary faces: Euler");
  using S = LineShape<DIM, P>;
  constexpr int Np = S::Np, NL = S::NL, ND = S::ND, NQ = S::NQ, EPW = S::EPW, NDS = S::NDS;
  constexpr int NVD = DIM + 1;
  constexpr int NFACE = 2 * DIM * NL;
  __shared__ LineLds<DIM, P> L;

  // variable-step clock: a stage of a step of length 0 (the end time was reached) does nothing
  const double dt = a.case_dt ? a.case_dt[0] : a.dt;
  if (a.mode != 0 && a.case_dt && dt == 0.0) return;
  const GasC<double> &g = a.gas;
  ConstBasis &B = const_basis(a.basis);
  const int lane = threadIdx.x;
  const int el = min(lane / NL, EPW - 1);
  const int t = lane < EPW * NL ? lane % NL : 0;
  const int e0 = logical_block(a.xcd_remap) * EPW;  // the wave's elements e0, ..., e0 + nv - 1
  const int nv = min(EPW, a.ne - e0);
  const int e = e0 + min(el, nv - 1);
  const bool valid = lane < EPW * NL && el < nv;
  const long long Ntot = a.Ntot;
  const long long Gtot = (long long)a.ne * NFACE;
  const double *Vd = static_cast<const double *>(a.Vd);
  const double *Gf = static_cast<const double *>(a.Gf);
  // nodes in memory order: lane + 64 m of the wave's contiguous EPW ND nodes
  unsigned fn[Np];
  int fx[Np];  // staged
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    const int k = lane + 64 * m, node = k % ND;
    fn[m] = (unsigned)(e0 * ND + min(k, nv * ND - 1)) * 8u;
    fx[m] = k / ND * NDS + node + node / Np;
  }
  const int le = min(el, nv - 1);  // e - e0
  const auto mr = LineMeta<DIM, P>::load(a, e0, nv, lane);

  // ---- state to LDS, indicator
  constexpr int NA = LineMeta<DIM, P>::Regs::NA;
  {
    double nlr[NA];
    double q[NQ][Np];
#pragma unroll
    for (int c = 0; c < NQ; ++c)
#pragma unroll
      for (int m = 0; m < Np; ++m) q[c][m] = ld(a.U + c * Ntot, fn[m]);
    L.m.store(mr, lane);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < NA; ++k) {
      const int i = min(lane + 64 * k, nv * DIM * DIM - 1), r = i % (DIM * DIM);
      const int nb = L.m.nbr[i / (DIM * DIM)][r / DIM * 2];
      nlr[k] = a.adj[(size_t)(BND && nb < 0 ? e0 + i / (DIM * DIM) : nb) * DIM * DIM + r];
    }
#pragma unroll
    for (int c = 0; c < NQ; ++c)
#pragma unroll
      for (int m = 0; m < Np; ++m)
        if (64 * (m + 1) <= EPW * ND || lane + 64 * m < EPW * ND) L.q[c][fx[m]] = q[c][m];
#pragma unroll
    for (int k = 0; k < NA; ++k)
      if (lane + 64 * k < EPW * DIM * DIM) (&L.nl[0][0])[lane + 64 * k] = nlr[k];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  double alpha = 0.0;
  if (a.blending) {
    // pressure * density = (gamma - 1) (rhoE rho - |m|^2/2)
    double f[Np];
    const int xs = el * NDS + (Np + 1) * t;
#pragma unroll
    for (int m = 0; m < Np; ++m) {
      double m2 = L.q[1][xs + m] * L.q[1][xs + m];
#pragma unroll
      for (int d = 1; d < DIM; ++d) m2 = fma(L.q[1 + d][xs + m], L.q[1 + d][xs + m], m2);
      f[m] = g.gammaM1 * fma(L.q[DIM + 1][xs + m], L.q[0][xs + m], -0.5 * m2);
    }
    alpha = line_alpha<DIM, P>(a, B, L.x, el, t, f);
    if (valid && t == 0) a.alpha[e] = alpha;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  const bool blend = a.blending && alpha > 1e-16;
  const double adg = blend ? 1.0 - alpha : 1.0;

  // running sums of the volume terms and the faces' lifted fluxes: -1/J times them is du/dt
  double rate[Np][NQ];
#pragma unroll
  for (int m = 0; m < Np; ++m)
#pragma unroll
    for (int c = 0; c < NQ; ++c) rate[m][c] = 0.0;
  double D2[Np * Np];
#pragma unroll
  for (int k = 0; k < Np * Np; ++k) D2[k] = B.D2line[k];

  double xb[Np][NQ], vd[Np][VISC ? DIM + 1 : 1];
  // unrolled: in a rolled loop the constants of the branches rarely taken
  // (22 registers) stay live throughout
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int lb = el * NDS + line_base<Np>(d, t), ls = line_stride<Np>(d);
    const int nlo = L.m.nbr[le][2 * d], nhi = L.m.nbr[le][2 * d + 1];
    double met[DIM];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) met[dd] = L.m.adj[le][d * DIM + dd];
    // the two-point fluxes are linear in the metric: (1 - alpha) times the
    // volume terms of a blended element
    double metv[DIM];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) metv[dd] = adg * met[dd];
    constexpr int gs[3] = {1, Np, Np * Np};
    const int gb = d == 0 ? Np * t : (d == 1 ? (t % Np) + Np * Np * (t / Np) : t);
    double qn[2][NQ];
    double gn[2][NVD];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int nbe = side ? nhi : nlo;
      // a neighbour along x is mostly in the same wave; a boundary point
      // takes the element's own trace
      if (BND && nbe < 0) {
#pragma unroll
        for (int c = 0; c < NQ; ++c) qn[side][c] = L.q[c][lb + (side ? Np - 1 : 0) * ls];
      } else if (d == 0 && (unsigned)(nbe - e0) < (unsigned)nv) {
        const int ns = (nbe - e0) * NDS + (Np + 1) * t + (side ? 0 : Np - 1);
#pragma unroll
        for (int c = 0; c < NQ; ++c) qn[side][c] = L.q[c][ns];
      } else {
        const unsigned nb = (unsigned)(nbe * ND + gb + (side ? 0 : (Np - 1) * gs[d]));
#pragma unroll
        for (int c = 0; c < NQ; ++c) qn[side][c] = ld(a.U + c * Ntot, nb * 8u);
      }
      const unsigned fb = (unsigned)((side ? nhi : nlo) * NFACE + (2 * d + 1 - side) * NL + t);
#pragma unroll
      for (int c = 0; c < NVD; ++c) gn[side][c] = VISC ? ld(Gf + c * Gtot, fb * 8u) : 0.0;
    }
    Pt<double, DIM> end[2];  // the line's end nodes
    // ---- volume: every pair of the line once (DGSEMIntegrator.hpp:124-218)
    {
      Pt<double, DIM> s[Np];
#pragma unroll
      for (int m = 0; m < Np; ++m) {
#pragma unroll
        for (int c = 0; c < NQ; ++c) s[m].q[c] = L.q[c][lb + m * ls];
        derive(g, s[m]);
      }
      const int series = VOL == 1 || VOL == 2 ? line_series<DIM, Np>(s) : 2;
      if (series == 0) {
        if constexpr (VOL == 2) line_ranocha_f64<false, DIM, Np>(g, s, metv, D2, rate);
        else line_volume<VOL, true, DIM, Np>(g, s, metv, D2, rate);
      } else if (VOL == 2 && series == 1) {
        if constexpr (VOL == 2) line_ranocha_f64<true, DIM, Np>(g, s, metv, D2, rate);
      } else {
        // momentum and energy again from LDS, so that the branches above need not hold them
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int m = 0; m < Np; ++m)
#pragma unroll
          for (int c = 1; c < NQ; ++c) s[m].q[c] = L.q[c][lb + m * ls];
        line_volume<VOL, false, DIM, Np>(g, s, metv, D2, rate);
      }
      end[0] = s[0];
      end[1] = s[Np - 1];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_sched_barrier(0);
    // ---- faces: Riemann flux at the line's two ends, the low-side element's
    //      state first (EulerOperator_impl.hpp:211-392; NSOperator_impl.hpp:579-713):
    //      the neighbours' traces, n.Fv there and the normals (the low-side
    //      element's adjugate row)
    double nl[DIM];
    if (d == DIM - 1) {
      // the RK base state (mode 2; in the other modes the stage state itself,
      // a line already in cache) and the viscous divergence
      const double *Xp = a.mode == 2 ? a.X : a.U;
#pragma unroll
      for (int c = 0; c < NQ; ++c)
#pragma unroll
        for (int m = 0; m < Np; ++m) xb[m][c] = ld(Xp + c * Ntot, fn[m]);
#pragma unroll
      for (int c = 0; c < (VISC ? NVD : 0); ++c)
#pragma unroll
        for (int m = 0; m < Np; ++m) vd[m][c] = ld(Vd + c * Ntot, fn[m]);
    }
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) nl[dd] = L.nl[le][d * DIM + dd];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int m = side ? Np - 1 : 0;
      // a boundary point evaluates F*(q, q_ext, n_out) with the interior trace
      // first, or the wall flux (0, p* n_out, 0) (bc_kernels.hpp:138-287)
      const int nbe = side ? nhi : nlo;
      const bool bdr = BND && nbe < 0;
      const bool out = side || bdr;  // n points out of the element
      const double lift = B.lift;
      double n[DIM];
#pragma unroll
      for (int dd = 0; dd < DIM; ++dd) n[dd] = side ? met[dd] : (bdr ? -met[dd] : nl[dd]);
      if constexpr (BND) {
        if (bdr) {
          const int b = -(nbe + 1), type = a.bc_type[b];
          if (bc_wall_pressure(type, VISC) || bc_zero_flux(type, VISC)) {
            const double pw = bc_zero_flux(type, VISC) ? 0.0 : slipwall_pstar<DIM>(g, qn[side], n);
#pragma unroll
            for (int dd = 0; dd < DIM; ++dd) rate[m][1 + dd] += lift * (pw * n[dd]);
            continue;
          }
          bc_exterior<DIM>(type, a.bc_data + (size_t)b * BC_STRIDE, n, qn[side]);
        }
      }
      Pt<double, DIM> own = end[side], oth;
      // momentum and energy again from LDS rather than held through the volume terms
#pragma unroll
      for (int c = 1; c < NQ; ++c) own.q[c] = L.q[c][lb + m * ls];
#pragma unroll
      for (int c = 0; c < NQ; ++c) oth.q[c] = qn[side][c];
      derive(g, oth);
      if constexpr (SURF == 5) {
        // with VISC F* - 0.5 n.(Fv_L + Fv_R) (DGSEMIntegrator.hpp:261-316); the
        // own side's -0.5 n.Fv was folded into Vd by the gradient kernel
        lift_llf_f64<DIM>(g, own, oth, n, out ? 1.0 : -1.0, out ? lift : -lift, gn[side], rate[m]);
      } else {
        double F[NQ];
        if constexpr (BND) {
          Pt<double, DIM> pl, pr;
          pt_select(out, own, oth, pl);
          pt_select(out, oth, own, pr);
          surface_flux<SURF, double, DIM>(g, pl, pr, n, F);
        } else {
          surface_flux<SURF, double, DIM>(g, side ? own : oth, side ? oth : own, n, F);
        }
        if constexpr (VISC) {
#pragma unroll
          for (int c = 0; c < NVD; ++c) F[1 + c] -= 0.5 * gn[side][c];
        }
#pragma unroll
        for (int c = 0; c < NQ; ++c) rate[m][c] += (out ? lift : -lift) * F[c];
      }
    }
    // ---- the sums move to the next direction's lines
    if (d + 1 < DIM) line_move_sums<DIM, P>(L, lb, ls, el * NDS + line_base<Np>(d + 1, t), line_stride<Np>(d + 1), rate);
  }

  // ---- subcell FV residual of the wave's blended elements (DGSEMIntegrator.hpp:
  //      338-483), direction by direction as above: alpha times the interface
  //      fluxes (homogeneous in the normal) on top of the sums
  if (a.blending && __any(blend)) {
#pragma unroll 1
    for (int k = 0; k < DIM; ++k) {
      const int d = k == 0 ? DIM - 1 : k - 1, dn = k;  // ends on the lines of the last direction, as it began
      const int lb = el * NDS + line_base<Np>(d, t), ls = line_stride<Np>(d);
      double n[DIM];
#pragma unroll
      for (int dd = 0; dd < DIM; ++dd)
        n[dd] = (blend ? alpha : 0.0) * L.m.adj[le][d * DIM + dd];
      Pt<double, DIM> s[2];
      double F[2][NQ];
#pragma unroll
      for (int m = 0; m < Np; ++m) {
        Pt<double, DIM> &p = s[m & 1];
#pragma unroll
        for (int c = 0; c < NQ; ++c) p.q[c] = L.q[c][lb + m * ls];
        derive(g, p);
        if (m > 0) {
          double (&Fm)[NQ] = F[m & 1];
          if (blend) surface_flux<SURF, double, DIM>(g, s[(m - 1) & 1], p, n, Fm);
          else
#pragma unroll
            for (int c = 0; c < NQ; ++c) Fm[c] = 0.0;
        }
        // node m - 1 now has its two interface fluxes, the last node its one
#pragma unroll
        for (int k = m - 1; k <= (m == Np - 1 ? m : m - 1); ++k) {
          if (k < 0) continue;
#pragma unroll
          for (int c = 0; c < NQ; ++c) {
            const double lo = k > 0 ? F[k & 1][c] : 0.0, hi = k < Np - 1 ? F[(k + 1) & 1][c] : 0.0;
            rate[k][c] += (hi - lo) * B.iw[k];
          }
        }
      }
      line_move_sums<DIM, P>(L, lb, ls, el * NDS + line_base<Np>(dn, t), line_stride<Np>(dn), rate);
    }
  }

  // ---- epilogue, in memory order: dU, or the fused SSP-RK3 stage combination
  const double scale = -1.0 / L.m.J[le];
  const int lb = el * NDS + line_base<Np>(DIM - 1, t), ls = line_stride<Np>(DIM - 1);
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    if (lane < EPW * NL) {
#pragma unroll
      for (int m = 0; m < Np; ++m) L.x[lb + m * ls] = scale * rate[m][c];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int m = 0; m < Np; ++m) {
      if (lane + 64 * m < nv * ND) {
        double r = L.x[fx[m]];
        if (VISC && c > 0) r += vd[m][VISC ? c - 1 : 0];
        st(a.out + c * Ntot, fn[m], stage_value(a, dt, xb[m][c], L.q[c][fx[m]], r));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

}  // namespace thx
