"""Non-physical and non-finite states: an evaluation says so with values that
are not finite where the equations have none, on every path that takes them."""
import dataclasses

import numpy as np
import pytest

from theseus_amd import _abi as A

from .gpu_helpers import gpu_rhs, make_case, smooth_state

pytestmark = pytest.mark.gpu


def _node(mesh, order, element, ijk):
    return element * (order + 1) ** mesh.dim + sum(i * (order + 1) ** d for d, i in enumerate(ijk))


@pytest.mark.parametrize("kind", ["pressure", "density"])
@pytest.mark.parametrize("pairing", ["hll", "llf", "roe", "ranocha_llf"])
@pytest.mark.parametrize("dim,order,n", [(2, 2, (4, 3)), (2, 3, (4, 3)), (3, 2, (3, 3, 3)), (3, 3, (3, 3, 3)),
                                         (3, 4, (3, 3, 3))])
def test_mixed_navier_stokes_interior_node(dim, order, n, pairing, kind):
    """p < 0 or rho < 0 at one interior node of one element, whose entropy
    variables do not exist: its energy rate is NaN, and elements that do not
    touch its element keep theirs."""
    rt, mesh = make_case(dim, order, n, pairing, flow=A.FLOW_NAVIER_STOKES, blending=False, mu=0.05)
    rt = dataclasses.replace(rt, precision=A.PRECISION_MIXED)
    U = smooth_state(mesh, order, rt.gamma, seed=order).reshape(dim + 2, -1)
    el = mesh.num_elements // 2
    bad = _node(mesh, order, el, (1,) * dim)
    if kind == "pressure":
        U[-1, bad] = 0.5 * (U[1:-1, bad] ** 2).sum() / U[0, bad] - 0.1
    else:
        U[0, bad] = -0.5
    got = gpu_rhs(rt, mesh, U.reshape(-1))[0].reshape(dim + 2, -1)
    assert np.isnan(got[-1, bad]), got[:, bad]
    nd = (order + 1) ** dim
    far = set(range(mesh.num_elements)) - {el} - {int(e) for e in mesh.face_neighbor.reshape(-1, 2 * dim)[el]}
    assert far and all(np.isfinite(got[:, e * nd:(e + 1) * nd]).all() for e in far)


@pytest.mark.parametrize("dim,order,n", [(2, 3, (4, 4)), (2, 3, (129, 128)), (3, 2, (3, 3, 3)), (3, 2, (20, 19, 19)),
                                         (3, 3, (3, 3, 3)), (3, 3, (16, 16, 13)), (3, 4, (3, 3, 3)), (3, 4, (17, 16, 13))])
def test_infinite_pressure_reaches_the_face_flux(dim, order, n):
    """Infinite energy at a face node: the sound speed there, the face's
    dissipation and with it the density rates of both sides are not finite
    (the node form on the small meshes, the line form on the others)."""
    rt, mesh = make_case(dim, order, n, "ranocha_llf", blending=False)
    U = smooth_state(mesh, order, rt.gamma, seed=order).reshape(dim + 2, -1)
    el = mesh.num_elements // 2
    low = int(mesh.face_neighbor.reshape(-1, 2 * dim)[el, 0])
    own, other = _node(mesh, order, el, (0,) + (1,) * (dim - 1)), _node(mesh, order, low, (order,) + (1,) * (dim - 1))
    U[-1, own] = np.inf
    got = gpu_rhs(rt, mesh, U.reshape(-1))[0].reshape(dim + 2, -1)
    assert not np.isfinite(got[0, [own, other]]).any(), got[:, [own, other]]
