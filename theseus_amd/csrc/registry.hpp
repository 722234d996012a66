// Kernel registry: every compiled (dim, order, volume flux, surface flux)
// combination registers its launchers at load time; theseus_rhs_create
// looks the combination up and fails with THESEUS_ERR_UNSUPPORTED when it
// was not compiled.
#pragma once

#include <hip/hip_runtime.h>

#include "rhs_kernels.hpp"
#include "grad_line.hpp"
#include "rhs_line.hpp"
#include "rhs_lte.hpp"

namespace thx {

using RHSLaunch = void (*)(const RHSArgs &, int nblocks, hipStream_t);
using StabLaunch = void (*)(const StabArgs &, int nblocks, hipStream_t);
using MeasLaunch = void (*)(const MeasArgs &, int nblocks, hipStream_t);

// [precision][bnd]: precision 0 = FP64 arithmetic, 1 = FP32 flux
// arithmetic (mixed precision); bnd 1 = the variant with the boundary
// conditions (meshes with boundary faces), 0 = periodic meshes
struct FluxKernels {
  RHSLaunch euler[2][2] = {};  // fused volume + face
  RHSLaunch ns[2][2] = {};     // Navier-Stokes pass 2
  // the FP64 line form (k_rhs_line) on meshes without ([0]) and with boundary faces (Euler), and the
  // fewest workgroups (waves of line_epw elements) it is used from, by [boundary][blending]; null where it is not built
  RHSLaunch euler_line[2] = {}, ns_line = nullptr;
  int euler_line_min[2][2] = {}, ns_line_min[2] = {};
  int line_epw = 0;
};

struct ShapeKernels {
  RHSLaunch ns_grad[2][2] = {};  // Navier-Stokes pass 1
  // its FP64 line form (k_ns_grad_line) on meshes without boundary faces, and the fewest
  // workgroups (waves of line_epw elements) it is used from; null where it is not built
  RHSLaunch ns_grad_line = nullptr;
  int ns_grad_line_min = 0;
  int line_epw = 0;
  StabLaunch stability = nullptr;
  MeasLaunch measures = nullptr;
  int tpb = 0, epb = 0;
};

// Tile shapes of the Euler kernel the serving pool's autotuner chooses from:
// [tile][precision][bnd], tile 0 = the default elements per workgroup, tile 1 = twice that.
struct TileKernels {
  RHSLaunch euler[2][2][2] = {};
  int epb[2] = {0, 0};
  int tpb[2] = {0, 0};
};

// 3-D Euler over orders 2, 3 and 4 in one launch (k_rhs_orders):
// [precision][bnd]; a[i] are the arguments of order i + 2 (its basis is
// basis[i], device memory).
using OrdersLaunch = void (*)(const RHSArgs a[3], const BasisArgs *basis, const int off[2], const int nb[3],
                              hipStream_t);
struct OrdersKernels {
  OrdersLaunch euler[2][2] = {};
};

// The tabulated LTE gas.  [flux]: the pairing (LteFlux, rhs_lte.hpp);
// [precision]: 0 FP64, 1 the mixed-precision form (FP32 flux arithmetic).
// Each instantiation file registers the fields it sets (the rest null).
struct LteKernels {
  RHSLaunch rhs[4][2] = {};        // Euler
  RHSLaunch nodes = nullptr;       // temperature recovery and node values (k_lte_nodes, FP64), before rhs
  RHSLaunch ns_grad[2] = {};       // Navier-Stokes pass 1 of the tabulated gas (after nodes)
  RHSLaunch ns[4][2] = {};         // Navier-Stokes pass 2 (after ns_grad)
  RHSLaunch pref = nullptr;        // mixed precision: the background pressure of a state
  int tpb = 0, epb = 0;
};

void register_flux(int dim, int p, int vol, int surf, FluxKernels k);
void register_lte(int dim, int p, LteKernels k);
const LteKernels *find_lte(int dim, int p);
void register_tiles(int dim, int p, int vol, int surf, TileKernels k);
void register_orders(int vol, int surf, OrdersKernels k);
const OrdersKernels *find_orders(int vol, int surf);
const TileKernels *find_tiles(int dim, int p, int vol, int surf);
void register_shape(int dim, int p, ShapeKernels k);
const FluxKernels *find_flux(int dim, int p, int vol, int surf);
const ShapeKernels *find_shape(int dim, int p);

template <typename R, int DIM, int P, int VOL, int SURF, bool VISC, int EPBX = 0, bool BND = false>
void launch_rhs(const RHSArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_rhs<R, DIM, P, VOL, SURF, VISC, EPBX, BND>), dim3(nb), dim3(Shape<DIM, P, EPBX>::TPB), 0, s,
                     a);
}
template <typename R, int DIM, int P, bool BND = false>
void launch_ns_grad(const RHSArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_ns_grad<R, DIM, P, 0, BND>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
}
template <int DIM, int P>
void launch_ns_grad_line(const RHSArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_ns_grad_line<DIM, P>), dim3(nb), dim3(64), 0, s, a);
}
template <int DIM, int P>
void launch_stability(const StabArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_stability<DIM, P>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
}

template <int DIM, int P>
void launch_measures(const MeasArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_measures<DIM, P>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
}

// From how many waves on the line form (k_rhs_line) is not the slower one, 0 where
// it is not built.  It issues 0.4 to 0.6 of the node form's instructions but
// runs Np nodes in each lane's chain, so it needs waves to hide latency, and a
// wave that holds one blended element makes the subcell pass for all of its
// elements (2-D p = 3: 16).  At two waves a SIMD its time is a staircase of 1024
// (up to 1024 waves one each) and 2048 waves: the ratios dip just above them.
// Ratio of the times, node / line form, of a whole evaluation (with NS the
// gradient pass by its own rule), smooth state / state with shocks (blended
// elements along two lines or three planes, 1 to 2 % and 10 to 25 % of all):
//   waves              768        1024        1152        1536        2304        4096
//   2-D p = 3, periodic
//     Ranocha/LLF   1.18/0.91  1.28/1.14  1.28/0.90  1.38/1.00  1.44/1.29  1.38/1.13
//     central/HLL   1.12/1.01  1.23/1.25  1.16/1.07  1.35/1.09  1.24/1.09  1.42/1.12
//     Ch'kar/Roe    1.10/0.85  1.23/1.12  1.09/0.79  1.17/0.92  1.15/0.94  1.38/0.98
//     Ranocha       1.06/0.82  1.18/1.06  1.08/0.79  1.17/0.89  1.14/0.92  1.33/0.97, at 6144 1.39/1.02
//   2-D p = 4  Ranocha  1.43/0.91  1.51/0.93  1.31/0.95  1.53/0.85  1.47/0.98  1.78/1.18, at 3072 1.69/1.07
//     central/HLL, outflow boundary 1.26/1.10  1.40/1.21  1.23/1.08  1.35/1.08  1.35/1.17  1.61/1.30
//   3-D p = 2  Ranocha/LLF  1.22/1.19  1.37/1.35  1.12/1.10  1.44/1.26  1.29/1.31  1.55/1.30, at 512 0.91/0.91
//     Ch'kar/Roe    1.04/1.17  1.27/1.31  0.95/1.05  1.25/1.15  1.18/1.22  1.48/1.25
//   3-D p = 3
//     Ranocha/LLF   1.20/1.01  1.25/1.08  1.10/1.02  1.33/1.10  1.34/1.10  1.65/1.35, at 512 0.99/0.78
//       boundary    1.19/1.01  1.16/1.08  1.06/1.03  1.32/1.09  1.28/1.05  1.62/1.32, at 512 0.94/0.78
//       NS          1.12/1.01  1.12/1.01  1.04/0.99  1.15/1.07  1.15/1.09  1.30/1.21, at 512 0.95/0.80
//     central/HLL   1.28/1.21  1.31/1.30  1.23/1.13  1.47/1.33  1.34/1.19  1.54/1.40, at 512 1.05/0.96
//       boundary    1.13/1.11  1.14/1.17  1.09/1.04  1.27/1.22  1.18/1.09  1.36/1.30, at 512 0.91/0.90
//       NS          0.94/0.97  0.93/0.99  0.93/0.95  1.01/1.02  0.94/0.97  1.06/1.11, at 8192 0.87/0.93: not built
//     Ch'kar/Roe    0.85/0.87  1.16/1.18  0.89/0.94  1.05/1.04  1.09/1.04  1.47/1.29
//       NS          0.71/0.77  0.87/0.98  0.79/0.87  0.86/0.93  0.86/0.90  1.06/1.07, at 8192 1.03/1.07
//     Ranocha       0.99/0.85  1.39/1.17  1.02/0.95  1.25/1.06  1.26/1.02  1.61/1.29
//       boundary    0.94/0.84  1.30/1.13  0.98/0.93  1.20/1.02  1.21/0.98  1.54/1.23
//     central/Roe   1.25/1.19  1.29/1.28  1.13/1.06  1.35/1.24  1.31/1.14  1.49/1.35, at 512 1.01/0.95
//     central/LLF   1.44/1.35  1.48/1.42  1.39/1.29  1.65/1.45  1.57/1.37  1.78/1.57, at 512 1.21/1.10
//       NS          1.23/1.21  1.22/1.24  1.19/1.13  1.27/1.22  1.20/1.18  1.30/1.31, at 512 1.08/1.04
//   3-D p = 4 (two elements in 50 of 64 lanes, five nodes a lane)
//     Ranocha/LLF   1.06/0.88  1.08/0.90  0.93/0.93  1.10/1.03  1.14/1.10  1.37/1.15
//       NS          0.76/0.75  0.95/0.87  0.90/0.91  1.00/0.96  1.00/0.95  1.15/1.05
//     central/HLL   0.96/0.93  0.93/0.93  0.88/0.91  1.01/0.99  0.96/0.96  1.11/1.05, at 2048 1.18/1.19
//     Ranocha NS    0.62/0.60  0.95/0.89  0.82/0.83  0.88/0.90  0.90/0.89  1.09/0.97
//     central/LLF NS 0.81/0.79 0.90/0.93  0.91/0.91  0.99/0.95  0.86/0.87  1.00/1.01, at 8192 0.88/0.93: not built
// (every pair was measured so, also at 2048, 3072 and 6144 to 27648 waves).
// The minimum is where both stay above 0.95, the runs' own spread, from there on;
// without blending the first alone, which in 2-D is lower.  Left out as well, from
// ratios at 512, 1024, 2048 and 4096 waves without shocks: 3-D p = 4 central/HLL NS
// (0.61 0.75 0.93 0.88) and Chandrashekar (Euler 0.62 0.78 1.02 0.96), 2-D p = 4
// Chandrashekar NS (0.68 0.91 0.97 1.22), Pirozzoli (3-D p = 3 Euler 0.83 0.96 1.06 1.02,
// NS 0.60 0.76 0.89 0.84); with boundary faces at 1024, 2048 and 4096, 2-D
// Chandrashekar p = 3 (1.01 1.06 0.99) and p = 4 (0.98 0.96 1.13); and 3-D p = 4
// central/LLF and central/Roe with boundary faces (332 and 424 B of scratch).
// Mixed mode: not built.  Measured only with lanes that load their own line (before
// the state moved in memory order), p = 3, waves as above: Euler 1.03 1.06 1.33
// 1.14, NS 0.96 0.98 1.14 1.02; p = 4 0.81 0.89 1.15 1.09 and 0.82 0.96 1.10 1.04.
template <int DIM, int P, int VOL, int SURF>
constexpr int line_min_waves(bool visc, bool boundary, bool blending) {
  if (P < 2 || P > 4 || VOL == 3) return 0;
  const bool costly = VOL == 1 || SURF == 1;  // two-point fluxes with logarithms at the faces or divisions in the volume
  if (DIM == 2) {
    if (VOL == 1 && ((P == 4 && visc) || (P >= 3 && boundary))) return 0;
    if (blending && P == 3) return costly ? 6144 : (VOL == 0 && SURF != 3 ? 1024 : 1536);
    return blending && P == 4 && costly ? 3072 : 1024;
  }
  if (P == 2) return costly ? 1536 : (SURF == 5 ? 768 : 1024);
  if (P == 3) {
    if (visc) return VOL == 1 ? 4096 : SURF == 1 ? 1536 : SURF == 4 ? 0 : SURF == 3 ? 1024 : VOL == 2 ? 768 : 512;
    if (VOL == 1 || (SURF == 1 && boundary)) return 1536;
    return SURF == 1 ? 1024 : (boundary || VOL == 2 ? 768 : 512);
  }
  if (VOL == 1 || (VOL == 0 && (visc || (boundary && SURF != 4)))) return 0;
  return VOL == 2 && SURF == 5 ? 1536 : (visc ? 4096 : 2048);
}

template <int DIM, int P, int VOL, int SURF, bool VISC, bool BND = false>
void launch_rhs_line(const RHSArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_rhs_line<DIM, P, VOL, SURF, VISC, BND>), dim3(nb), dim3(64), 0, s, a);
}

template <int DIM, int VOL, int SURF, int P>
struct FluxRegistrar {
  FluxRegistrar() {
    FluxKernels k;
    constexpr auto min_waves = &line_min_waves<DIM, P, VOL, SURF>;
    if constexpr (min_waves(false, false, false) > 0) k.euler_line[0] = &launch_rhs_line<DIM, P, VOL, SURF, false>;
    if constexpr (min_waves(false, true, false) > 0) k.euler_line[1] = &launch_rhs_line<DIM, P, VOL, SURF, false, true>;
    if constexpr (min_waves(true, false, false) > 0) k.ns_line = &launch_rhs_line<DIM, P, VOL, SURF, true>;
    for (int blending = 0; blending < 2; ++blending) {
      for (int boundary = 0; boundary < 2; ++boundary) k.euler_line_min[boundary][blending] = min_waves(false, boundary, blending);
      k.ns_line_min[blending] = min_waves(true, false, blending);
    }
    if constexpr (P >= 2 && P <= 4) k.line_epw = LineShape<DIM, P>::EPW;
    k.euler[0][0] = &launch_rhs<double, DIM, P, VOL, SURF, false>;
    k.ns[0][0] = &launch_rhs<double, DIM, P, VOL, SURF, true>;
    k.euler[1][0] = &launch_rhs<float, DIM, P, VOL, SURF, false>;
    k.ns[1][0] = &launch_rhs<float, DIM, P, VOL, SURF, true>;
    k.euler[0][1] = &launch_rhs<double, DIM, P, VOL, SURF, false, 0, true>;
    k.ns[0][1] = &launch_rhs<double, DIM, P, VOL, SURF, true, 0, true>;
    k.euler[1][1] = &launch_rhs<float, DIM, P, VOL, SURF, false, 0, true>;
    k.ns[1][1] = &launch_rhs<float, DIM, P, VOL, SURF, true, 0, true>;
    register_flux(DIM, P, VOL, SURF, k);
  }
};

template <int DIM, int VOL, int SURF, int P>
struct TileRegistrar {
  TileRegistrar() {
    constexpr int E0 = Shape<DIM, P>::EPB, E1 = 2 * Shape<DIM, P>::EPB;
    TileKernels k;
    k.euler[0][0][0] = &launch_rhs<double, DIM, P, VOL, SURF, false>;
    k.euler[0][1][0] = &launch_rhs<float, DIM, P, VOL, SURF, false>;
    k.euler[1][0][0] = &launch_rhs<double, DIM, P, VOL, SURF, false, E1>;
    k.euler[1][1][0] = &launch_rhs<float, DIM, P, VOL, SURF, false, E1>;
    k.euler[0][0][1] = &launch_rhs<double, DIM, P, VOL, SURF, false, 0, true>;
    k.euler[0][1][1] = &launch_rhs<float, DIM, P, VOL, SURF, false, 0, true>;
    k.euler[1][0][1] = &launch_rhs<double, DIM, P, VOL, SURF, false, E1, true>;
    k.euler[1][1][1] = &launch_rhs<float, DIM, P, VOL, SURF, false, E1, true>;
    k.epb[0] = E0;
    k.epb[1] = E1;
    k.tpb[0] = Shape<DIM, P>::TPB;
    k.tpb[1] = Shape<DIM, P, E1>::TPB;
    register_tiles(DIM, P, VOL, SURF, k);
  }
};

template <typename R, int VOL, int SURF, bool BND>
void launch_rhs_orders(const RHSArgs a[3], const BasisArgs *basis, const int off[2], const int nb[3], hipStream_t s) {
  const RHSCore a2 = a[0], a3 = a[1], a4 = a[2];
  hipLaunchKernelGGL((k_rhs_orders<R, VOL, SURF, BND>), dim3(off[1] + nb[2]), dim3(128), 0, s, a2, a3, a4, basis,
                     off[0], off[1], nb[0], nb[1], nb[2]);
}

template <int VOL, int SURF>
struct OrdersRegistrar {
  OrdersRegistrar() {
    OrdersKernels k;
    k.euler[0][0] = &launch_rhs_orders<double, VOL, SURF, false>;
    k.euler[1][0] = &launch_rhs_orders<float, VOL, SURF, false>;
    k.euler[0][1] = &launch_rhs_orders<double, VOL, SURF, true>;
    k.euler[1][1] = &launch_rhs_orders<float, VOL, SURF, true>;
    register_orders(VOL, SURF, k);
  }
};

template <typename R, int DIM, int P, bool VISC = false, int FX = LTE_FLUX_LTEEC>
void launch_rhs_lte(const RHSArgs &a, int nb, hipStream_t s) {
  if constexpr (FX == LTE_FLUX_LTEEC)
    hipLaunchKernelGGL((k_rhs_lteec<R, DIM, P, VISC>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
  else
    hipLaunchKernelGGL((k_rhs_lte<R, DIM, P, VISC, FX>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
}
template <typename R, int DIM, int P>
void launch_ns_grad_lte(const RHSArgs &a, int nb, hipStream_t s) {
  hipLaunchKernelGGL((k_ns_grad<R, DIM, P, 0, false, true>), dim3(nb), dim3(Shape<DIM, P>::TPB), 0, s, a);
}
template <int DIM>
void launch_pref_lte(const RHSArgs &a, int, hipStream_t s) {
  hipLaunchKernelGGL((lte::k_pref_lte<DIM>), dim3(1), dim3(64), 0, s, a.U, a.Ntot, a.lte, const_cast<double *>(a.pref));
}

template <int DIM>
void launch_lte_nodes(const RHSArgs &a, int, hipStream_t s) {
  const dim3 grid((unsigned)((a.Ntot + 255) / 256));
  if (a.lte.node_rec && a.lte.cells32)
    hipLaunchKernelGGL((lte::k_lte_nodes<DIM, lte::NODE_LTEEC, float>), grid, dim3(256), 0, s, a.U, a.Ntot, a.lte);
  else if (a.lte.node_rec)
    hipLaunchKernelGGL((lte::k_lte_nodes<DIM, lte::NODE_LTEEC>), grid, dim3(256), 0, s, a.U, a.Ntot, a.lte);
  else if (a.lte.node_p)
    hipLaunchKernelGGL((lte::k_lte_nodes<DIM, lte::NODE_PC>), grid, dim3(256), 0, s, a.U, a.Ntot, a.lte);
  else
    hipLaunchKernelGGL((lte::k_lte_nodes<DIM, lte::NODE_T>), grid, dim3(256), 0, s, a.U, a.Ntot, a.lte);
}

template <int DIM, int P>
struct LteRegistrar {
  LteRegistrar() {
    LteKernels k;
    k.rhs[LTE_FLUX_LTEEC][0] = &launch_rhs_lte<double, DIM, P>;
    k.rhs[LTE_FLUX_LTEEC][1] = &launch_rhs_lte<float, DIM, P>;
    k.nodes = &launch_lte_nodes<DIM>;
    k.ns_grad[0] = &launch_ns_grad_lte<double, DIM, P>;
    k.ns_grad[1] = &launch_ns_grad_lte<float, DIM, P>;
    k.ns[LTE_FLUX_LTEEC][0] = &launch_rhs_lte<double, DIM, P, true>;
    k.ns[LTE_FLUX_LTEEC][1] = &launch_rhs_lte<float, DIM, P, true>;
    k.pref = &launch_pref_lte<DIM>;
    k.tpb = Shape<DIM, P>::TPB;
    k.epb = Shape<DIM, P>::EPB;
    register_lte(DIM, P, k);
  }
};

// The Pirozzoli, HLL and LLF pairings of the tabulated gas
template <int DIM, int P, int FX>
struct LteFluxRegistrar {
  LteFluxRegistrar() {
    LteKernels k;
    k.rhs[FX][0] = &launch_rhs_lte<double, DIM, P, false, FX>;
    k.rhs[FX][1] = &launch_rhs_lte<float, DIM, P, false, FX>;
    k.ns[FX][0] = &launch_rhs_lte<double, DIM, P, true, FX>;
    k.ns[FX][1] = &launch_rhs_lte<float, DIM, P, true, FX>;
    register_lte(DIM, P, k);
  }
};

// From how many waves on the gradient pass's line form (k_ns_grad_line) is the
// faster one, 0 where it is not built.  Ratio of the times, node / line form, of
// a whole Navier-Stokes evaluation (Ranocha/LLF) at 256, 512, 1024, 2048 and
// 4096 waves:
//   3-D  p = 2 1.01 1.06 1.10 1.10 1.07, p = 3 1.03 1.06 1.17 1.16 1.11,
//        p = 4 0.96 0.99 1.02 1.09 1.16
//   2-D  p = 2 1.04 1.03 1.07 1.03 1.07, p = 3 1.06 1.03 1.07 1.09 1.08,
//        p = 4 0.97 0.98 1.04 1.05 1.13
constexpr int grad_line_min_waves(int p) { return p < 2 || p > 4 ? 0 : (p == 4 ? 1024 : 512); }

template <int DIM, int P>
struct ShapeRegistrar {
  ShapeRegistrar() {
    ShapeKernels k;
    k.ns_grad[0][0] = &launch_ns_grad<double, DIM, P>;
    k.ns_grad[1][0] = &launch_ns_grad<float, DIM, P>;
    k.ns_grad[0][1] = &launch_ns_grad<double, DIM, P, true>;
    k.ns_grad[1][1] = &launch_ns_grad<float, DIM, P, true>;
    if constexpr (grad_line_min_waves(P) > 0) {
      k.ns_grad_line = &launch_ns_grad_line<DIM, P>;
      k.ns_grad_line_min = grad_line_min_waves(P);
      k.line_epw = LineShape<DIM, P>::EPW;
    }
    k.stability = &launch_stability<DIM, P>;
    k.measures = &launch_measures<DIM, P>;
    k.tpb = Shape<DIM, P>::TPB;
    k.epb = Shape<DIM, P>::EPB;
    register_shape(DIM, P, k);
  }
};

}  // namespace thx
