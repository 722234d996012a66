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
