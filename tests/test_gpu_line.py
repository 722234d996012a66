"""The line forms of the fused kernel and the gradient pass (FP64, enough
elements to fill the chip) against the CPU oracle, at the element counts from
which they are used (odd counts: the last wave is partly filled), on states
that take each branch of the logarithmic means, with and without blended
elements.  The bound is that of the other FP64 RHS tests, relative L2 <= 1e-12."""
import numpy as np
import pytest

from theseus_amd import _abi as A

from .gpu_helpers import gpu_rhs, make_case, oracle_case, rel_l2, smooth_state
from .test_gpu_bc import _case as _bc_case

pytestmark = pytest.mark.gpu

# nodewise factors exp(+-a) on density and pressure: the nodes of a line differ
# by ratios within the first series (a = 0.004), the second (0.03) and beyond (0.5)
NOISE = {"short": 0.004, "long": 0.03, "far": 0.5}


def _state(mesh, order, gamma, noise):
    rng = np.random.default_rng(order)
    U = smooth_state(mesh, order, gamma, amp=0.1, seed=3).reshape(mesh.dim + 2, -1)
    rho, m, E = U[0], U[1:-1], U[-1]
    p = (gamma - 1) * (E - 0.5 * (m * m).sum(0) / rho)
    fr, fp = np.exp(NOISE[noise] * rng.uniform(-1, 1, (2, rho.size)))
    m = m * fr
    rho, p = rho * fr, p * fp
    return np.concatenate([rho[None], m, (p / (gamma - 1) + 0.5 * (m * m).sum(0) / rho)[None]]).reshape(-1)


@pytest.mark.parametrize("noise", list(NOISE))
@pytest.mark.parametrize("blending", [False, True])
@pytest.mark.parametrize("dim,n,order,pairing,visc", [
    (3, (20, 19, 19), 2, "chandrashekar", False), (3, (20, 19, 19), 2, "ranocha_llf", True),  # 1032 waves of 7
    (3, (13, 13, 13), 3, "ranocha_llf", False), (3, (13, 13, 13), 3, "hll", False),           # 550 waves of 4
    (3, (17, 15, 17), 3, "ranocha_llf", True), (3, (17, 15, 17), 3, "chandrashekar_roe", True),
    (3, (13, 13, 13), 4, "ranocha_llf", False), (3, (17, 15, 17), 4, "ranocha_llf", True),    # waves of 2
    (3, (13, 13, 13), 3, "hll", True), (2, (107, 107), 2, "hll", True), (2, (91, 91), 3, "llf", True),  # the gradient pass alone
    (2, (147, 147), 2, "llf", False), (2, (129, 128), 3, "ranocha_llf", False),
    (2, (111, 111), 4, "ranocha", True),
])
def test_line_form_fp64(oracle, dim, n, order, pairing, visc, blending, noise):
    flow = A.FLOW_NAVIER_STOKES if visc else A.FLOW_EULER
    rt, mesh = make_case(dim, order, n, pairing, flow=flow, blending=blending)
    U = _state(mesh, order, rt.gamma, noise)
    ref = oracle_case(oracle, rt, mesh).rhs(U)
    got, _ = gpu_rhs(rt, mesh, U)
    assert rel_l2(got, ref) <= 1e-12, rel_l2(got, ref)


@pytest.mark.parametrize("noise", ["short", "far"])
@pytest.mark.parametrize("blending", [False, True])
@pytest.mark.parametrize("kind", ["euler", "no_slip"])
@pytest.mark.parametrize("dim,n,order,pairing,periodic", [
    (2, (147, 147), 2, "roe", False), (2, (129, 128), 3, "ranocha_llf", (True, False)), (2, (111, 111), 4, "hll", False),
    (3, (20, 19, 19), 2, "chandrashekar", False), (3, (13, 13, 13), 3, "ranocha_llf", (False, True, False)),
    (3, (17, 16, 16), 4, "llf", False),
])
def test_line_form_boundaries(oracle, dim, n, order, pairing, periodic, kind, blending, noise):
    """Every boundary type of the Euler equations on the sides of a box"""
    rt, mesh = _bc_case(dim, order, n, pairing, A.FLOW_EULER, kind, blending=blending, periodic=periodic)
    U = _state(mesh, order, rt.gamma, noise)
    ref = oracle_case(oracle, rt, mesh).rhs(U)
    got, _ = gpu_rhs(rt, mesh, U)
    assert rel_l2(got, ref) <= 1e-12, rel_l2(got, ref)


@pytest.mark.parametrize("pairing,visc", [("ranocha_llf", False), ("ranocha_llf", True), ("hll", False), ("hll", True)])
@pytest.mark.parametrize("dim,n,order", [(2, (147, 147), 2), (2, (129, 128), 3), (2, (147, 147), 4), (3, (27, 27, 27), 2),
                                         (3, (21, 21, 21), 3), (3, (17, 16, 17), 4)])
def test_line_ends_at_rest(dim, n, order, pairing, visc):
    """Gas at rest: every flux is the pressure times the area vector, and the
    momentum rate at a line's end node is what the row of two-point fluxes and
    the face's lift leave of their sum, 0.  In units of eps p/(w0 h), eps =
    2^-53: a face weight off by its own rounding leaves 0.5 for every pressure;
    the roundings of the up to order partial sums (each at most 0.8 where the
    largest is 1.4/w0, of either sign: 0.46 on average) differ from pressure to
    pressure, so the mean over 64 pressures holds 0.46 sqrt(4/64) of them."""
    import torch

    from theseus_amd.mesh import gll_nodes
    from theseus_amd.operator import MakeRHSOperator

    if dim == 3 and order > 2 and pairing == "hll" and visc:
        pytest.skip("this pair's viscous form is not built in line form above order 2 in 3-D")
    flow = A.FLOW_NAVIER_STOKES if visc else A.FLOW_EULER
    rt, mesh = make_case(dim, order, n, pairing, flow=flow, blending=False)
    nd, Np = (order + 1) ** dim, order + 1
    w0, i = gll_nodes(order)[1][0], np.arange(nd)
    op = MakeRHSOperator(rt, mesh)
    assert op.kernel_form(0) == "line"
    u = torch.zeros(dim + 2, mesh.num_elements * nd, dtype=torch.float64, device="cuda")
    u[0] = 1.0
    du = torch.empty_like(u)
    mean = 0.0
    for p in 50.0 * 2.0 ** ((np.arange(64) + 0.5) / 64):
        u[-1] = p / (rt.gamma - 1)
        op.Mult(u.reshape(-1), du.reshape(-1))
        mean = mean + du[1:-1].cpu().numpy().reshape(dim, mesh.num_elements, nd) * (2.0 ** 53 * w0 / p / 64)
    op.close()
    for d in range(dim):
        for end in (0, order):
            worst = np.abs(mean[d][:, i // Np ** d % Np == end]).max() / n[d]
            assert worst <= 0.5 + 4 * 0.46 * (4 / 64) ** 0.5, (d, end, worst)
