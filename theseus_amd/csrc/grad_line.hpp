// Navier-Stokes pass 1 (k_ns_grad) of the ideal gas in FP64 in line form: as
// k_rhs_line, a wave holds the GLL lines of as many elements as fit, one lane
// a line.  A lane forms the viscous variables of its home line's nodes, takes the
// derivative along its line of each direction in turn (the face lift is part
// of the line's operator: own half in its corner entries, the neighbour's half
// from its trace), and with all of them on its home line forms the viscous
// flux of its nodes; the contravariant fluxes then go to the lines of their
// direction for the divergence, whose ends are n.Fv at the face points.
//
// On 32^3 elements, p = 3, in FP64 it takes 70 us for the node form's 90, with
// 11.4 M vector instructions for 28.9 M; its 300 MB of HBM traffic (133 read, 168
// written) at the rate of a copy are 58 us.  The vector memory path is the bound
// (TD busy 75 % of the time), with two waves a SIMD (220 registers; three spill).  Before k_rhs_line
// moved in memory order a step on 48^3 elements took 1636 us with it and 1840 with
// the node form.  The mixed mode keeps the node form: in FP32 this one took 47 us
// for 58, but folding the face lift into the line's operator moved the outputs
// by up to 2.5e-8 of the energy in two steps, and whether that is nearer to or
// further from 64 bits was not measured.
#pragma once

#include "rhs_line.hpp"

namespace thx {

template <int DIM, int P>
struct GradLineLds {
  using S = LineShape<DIM, P>;
  double S_[DIM + 1][S::EPW * S::NDS];  // viscous variables
  double x[S::EPW * S::NDS];            // one field on its way between directions
};

// Meshes without boundary faces where the face normals of an element and its
// neighbours agree (to rounding), whose fields and n.Fv rows can be addressed
// with 32-bit byte offsets.
template <int DIM, int P>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_ns_grad_line(RHSArgs a) {
  using S = LineShape<DIM, P>;
  constexpr int Np = S::Np, NL = S::NL, ND = S::ND, NQ = S::NQ, EPW = S::EPW, NDS = S::NDS;
  constexpr int NG = DIM + 1;
  constexpr int NFACE = 2 * DIM * NL;
  __shared__ GradLineLds<DIM, P> L;

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
  double *Vd = static_cast<double *>(a.Vd_out);
  double *Gf = static_cast<double *>(a.Gf_out);
  // the lane's home line, on which the nodes are loaded, their fluxes formed and
  // the divergence stored: of the last direction, whose lanes' nodes are
  // consecutive in memory (in 2-D too few; there the x-line, consecutive in the lane)
  constexpr int H = DIM == 3 ? 2 : 0;
  constexpr int HG = H == 0 ? 1 : NL;                                    // distance of its nodes in memory
  const unsigned hn = (unsigned)(e * ND + (H == 0 ? Np * t : t));        // its first node
  const int hs = el * NDS + line_base<Np>(H, t), hl = line_stride<Np>(H);  // the same, staged
  const double invJ = 1.0 / a.J[e];
  const double hw = 0.5 * B.iw[0];

  // every load at once: the fences between the directions' steps below would
  // put a memory latency into each of them
  int nbr[2 * DIM];
#pragma unroll
  for (int f = 0; f < 2 * DIM; ++f) nbr[f] = a.nbr[e * 2 * DIM + f];
  double adj[DIM][DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) adj[d][dd] = a.adj[(size_t)e * DIM * DIM + d * DIM + dd];
  double q[NQ][Np], qn[2 * DIM][NQ];
  bool inside[2 * DIM];  // a neighbour along x is mostly in the same wave
#pragma unroll
  for (int c = 0; c < NQ; ++c)
#pragma unroll
    for (int m = 0; m < Np; ++m) q[c][m] = ld(a.U + c * Ntot, (hn + m * HG) * 8u);
#pragma unroll
  for (int f = 0; f < 2 * DIM; ++f) {
    const int d = f / 2;
    constexpr int gs[3] = {1, Np, Np * Np};
    const int gb = d == 0 ? Np * t : (d == 1 ? (t % Np) + Np * Np * (t / Np) : t);
    const unsigned nb = (unsigned)(nbr[f] * ND + gb + (f % 2 ? 0 : (Np - 1) * gs[d]));
    inside[f] = d == 0 && (unsigned)(nbr[f] - e0) < (unsigned)nv;
    if (!inside[f]) {
#pragma unroll
      for (int c = 0; c < NQ; ++c) qn[f][c] = ld(a.U + c * Ntot, nb * 8u);
    }
  }

  // viscous variables of the home line's nodes and of the neighbours' traces
  double u[Np][DIM], por[Np];  // velocity, p/rho
  double Sn[2 * DIM][NG];
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    double s[NQ];
#pragma unroll
    for (int c = 0; c < NQ; ++c) s[c] = q[c][m];
    const NodeThermo<double, DIM> th = node_thermo<double, DIM>(g, s);
#pragma unroll
    for (int d = 0; d < DIM; ++d) u[m][d] = th.u[d];
    por[m] = th.p * th.ir;
    if (lane < EPW * NL) {
#pragma unroll
      for (int d = 0; d < DIM; ++d) L.S_[d][hs + m * hl] = th.beta * th.u[d];
      L.S_[DIM][hs + m * hl] = -th.beta;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int f = 0; f < 2 * DIM; ++f) {
    if (inside[f]) {
      const int ns = (nbr[f] - e0) * NDS + (Np + 1) * t + (f ? 0 : Np - 1);
#pragma unroll
      for (int c = 0; c < NG; ++c) Sn[f][c] = L.S_[c][ns];
    } else {
      double s[NQ];
#pragma unroll
      for (int c = 0; c < NQ; ++c) s[c] = qn[f][c];
      viscous_variables<double, DIM>(g, s, Sn[f]);
    }
  }

  // derivative along the lines of each direction, with the face lift
  // 0.5 (S_R - S_L)/w at the line's ends, brought back to the home lines
  double G[DIM][NG][Np];
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int lb = el * NDS + line_base<Np>(d, t), ls = line_stride<Np>(d);
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      double s[Np], v[Np];
#pragma unroll
      for (int m = 0; m < Np; ++m) s[m] = L.S_[c][lb + m * ls];
#pragma unroll
      for (int m = 0; m < Np; ++m) {
        v[m] = 0.0;
#pragma unroll
        for (int l = 0; l < Np; ++l) v[m] += B.D[m * Np + l] * s[l];
      }
      v[0] += hw * (s[0] - Sn[2 * d][c]);
      v[Np - 1] += hw * (Sn[2 * d + 1][c] - s[Np - 1]);
      if (d != H) line_move<Np>(L.x, lb, ls, hs, hl, v);
#pragma unroll
      for (int m = 0; m < Np; ++m) G[d][c][m] = v[m];
    }
  }

  // physical gradients, viscous flux, and its contravariant components, node by node
#pragma unroll
  for (int m = 0; m < Np; ++m) {
    NodeThermo<double, DIM> th;
#pragma unroll
    for (int d = 0; d < DIM; ++d) th.u[d] = u[m][d];
    th.p = por[m];
    th.ir = 1.0;
    double dV[DIM][DIM], dT[DIM];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) {
      double dS[NG];
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        double v = G[0][c][m] * adj[0][dd];
#pragma unroll
        for (int d = 1; d < DIM; ++d) v += G[d][c][m] * adj[d][dd];
        dS[c] = v * invJ;
      }
      viscous_gradients<double, DIM>(g, th, dS, dV[dd], dT[dd]);
    }
    double vf[VisComp<DIM>::N];
    viscous_flux<double, DIM>(g.mu, g.kappa, g.mu_bulk, th.u, dV, dT, vf);
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
      for (int c = 0; c < NG; ++c) {
        double v = adj[d][0] * vf[vis_index<DIM>(1 + c, 0)];
#pragma unroll
        for (int dd = 1; dd < DIM; ++dd) v += adj[d][dd] * vf[vis_index<DIM>(1 + c, dd)];
        G[d][c][m] = v;
      }
  }

  // divergence with the own half of the central viscous face flux,
  // -0.5 n.Fv lifted with the face weight; n.Fv for the neighbours' halves
  double dv[NG][Np];
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int lb = el * NDS + line_base<Np>(d, t), ls = line_stride<Np>(d);
    const unsigned fb = (unsigned)(e * NFACE + 2 * d * NL + t);
#pragma unroll
    for (int c = 0; c < NG; ++c) {
      double f[Np], v[Np];
#pragma unroll
      for (int m = 0; m < Np; ++m) f[m] = G[d][c][m];
      if (d != H) line_move<Np>(L.x, hs, hl, lb, ls, f);
      if (valid) {
        st(Gf + c * Gtot, fb * 8u, f[0]);
        st(Gf + c * Gtot, (fb + NL) * 8u, f[Np - 1]);
      }
#pragma unroll
      for (int m = 0; m < Np; ++m) {
        v[m] = 0.0;
#pragma unroll
        for (int l = 0; l < Np; ++l) v[m] += B.Dhat[m * Np + l] * f[l];
      }
      v[0] -= hw * f[0];
      v[Np - 1] += hw * f[Np - 1];
      if (d != H) line_move<Np>(L.x, lb, ls, hs, hl, v);
#pragma unroll
      for (int m = 0; m < Np; ++m) dv[c][m] = d == 0 ? v[m] : dv[c][m] + v[m];
    }
  }
  if (!valid) return;
#pragma unroll
  for (int c = 0; c < NG; ++c)
#pragma unroll
    for (int m = 0; m < Np; ++m) st(Vd + c * Ntot, (hn + m * HG) * 8u, invJ * dv[c][m]);
}

}  // namespace thx
