"""The LTEEC pair fluxes on states that take each branch of the discrete
gradients -- the derivative form (equal endpoints), the divided differences
(endpoints in one table cell), the corner differences (endpoints in different
cells) and their mixtures -- at the edges of the workgroup's element packing,
against the CPU oracle.  The kernel keeps the oracle's operations and their
order (no contraction), so the bound is the one of every smooth tabulated
state, relative L2 <= 1e-12."""
import numpy as np
import pytest

from .gpu_helpers import per_field_rel, rel_l2
from .test_gpu_lte import _oracle

pytestmark = pytest.mark.gpu

# relative amplitude of density and temperature variations, table size
BRANCHES = {
    "derivative": (0.0, 0.0, 256),
    "temperature_only": (0.0, 0.1, 256),
    "density_only": (0.2, 0.0, 256),
    "one_cell": (0.05, 0.03, 12),
    "corners": (0.5, 0.3, 256),
    "mixed": (0.04, 0.02, 256),
}


def _setup(dim, n, order, rho_amp, T_amp, size):
    from theseus_amd import _abi as A
    from theseus_amd.config import RunTime
    from theseus_amd.lte import synthetic_table
    from theseus_amd.mesh import box_mesh, gll_nodes

    table = synthetic_table(nx=size, ny=size)
    mesh = box_mesh(dim, n, 0.0, 1.0, periodic=True)
    rt = RunTime(dim=dim, order=order, flow_model=A.FLOW_EULER, volume_flux=A.VOLUME_LTEEC,
                 surface_flux=A.SURFACE_LTEEC, blending=False, lte=True)
    X = 2 * np.pi * mesh.node_coordinates(gll_nodes(order)[0])
    w = [sum(np.sin((1 + (k + d) % 2) * X[d] + k + 0.3 * d) for d in range(dim)) / dim for k in range(5)]
    rho, T = 0.1 * (1 + rho_amp * w[0]), 3500.0 * (1 + T_amp * w[1])
    vel = [300.0 * (0.2 + w[2 + d]) for d in range(dim)]
    return rt, mesh, table, rho, T, vel


def _state(ora, rho, T, vel):
    e = np.array([ora._table.eval(r, t)["energy"] for r, t in zip(rho, T)])
    return np.concatenate([rho, *[rho * v for v in vel], rho * e + 0.5 * rho * sum(v * v for v in vel)])


def _mult(rt, mesh, table, U):
    import torch

    from theseus_amd.operator import MakeRHSOperator

    op = MakeRHSOperator(rt, mesh, lte_table=table)
    u = torch.from_numpy(U).cuda()
    du = torch.empty_like(u)
    op.Mult(u, du)
    torch.cuda.synchronize()
    op.close()
    return du.cpu().numpy()


# (2, 5, 2): 25 elements of 9 nodes, 7 a workgroup; (3, 3, 3): 27 of 64, the last workgroup half filled;
# (3, 3, 2): 27 of 27, 2 a workgroup; (3, 2, 4): one element of 125 on 128 lanes
@pytest.mark.parametrize("dim,n,order", [(2, 5, 2), (3, 3, 3), (3, 3, 2), (3, 2, 4)])
@pytest.mark.parametrize("branch", list(BRANCHES))
def test_lteec_branches(oracle, dim, n, order, branch):
    rt, mesh, table, rho, T, vel = _setup(dim, n, order, *BRANCHES[branch])
    ora = _oracle(oracle, rt, mesh, table)
    U = _state(ora, rho, T, vel)
    ref = ora.rhs(U)
    got = _mult(rt, mesh, table, U)
    assert np.isfinite(got).all()
    assert rel_l2(got, ref) <= 1e-12, per_field_rel(got, ref, dim + 2)


def test_lteec_outside_the_table_is_nan(oracle):
    """A node outside the table makes its lines NaN and leaves elements
    that do not touch its element as they are."""
    rt, mesh, table, rho, T, vel = _setup(3, 4, 3, 0.04, 0.02, 256)
    ora = _oracle(oracle, rt, mesh, table)
    U = _state(ora, rho, T, vel)
    ref = _mult(rt, mesh, table, U).reshape(5, 64, 64)
    bad = U.reshape(5, 64, 64).copy()
    bad[0, 21, 10] = 50.0  # density above the grid
    got = _mult(rt, mesh, table, bad.reshape(-1)).reshape(5, 64, 64)
    assert np.isnan(got[:, 21, 10]).all()
    touched = {21} | {int(v) for v in mesh.face_neighbor.reshape(64, 6)[21]}
    rest = [e for e in range(64) if e not in touched]
    assert np.array_equal(got[:, rest], ref[:, rest])


# The recovery's cell searches on grids of each kind: logarithmic (the
# workload's), uniform, two cells in a direction, and one whose cells crowd
# into few buckets (the searches then bisect).
GRIDS = {
    "log": dict(nx=40, ny=300),
    "uniform": dict(nx=50, ny=70, rho=(0.01, 1.0), rho_dist="uniform", T_dist="uniform"),
    "tiny": dict(nx=3, ny=3, rho=(0.05, 0.3), T=(2000.0, 6000.0)),
    "crowded": dict(nx=600, ny=64, rho=(1e-30, 1.0), rho_dist="uniform"),
}


@pytest.mark.parametrize("flux", ["lteec", "hll"])
@pytest.mark.parametrize("grid", list(GRIDS))
def test_recovery_on_grids(oracle, grid, flux):
    import dataclasses

    from theseus_amd import _abi as A
    from theseus_amd.lte import synthetic_table

    rt, mesh, _, rho, T, vel = _setup(3, 3, 3, 0.3, 0.2, 12)
    if flux == "hll":
        rt = dataclasses.replace(rt, volume_flux=A.VOLUME_CENTRAL, surface_flux=A.SURFACE_HLL)
    table = synthetic_table(**GRIDS[grid])
    ora = _oracle(oracle, rt, mesh, table)
    U = _state(ora, rho, T, vel)
    got = _mult(rt, mesh, table, U)
    assert np.isfinite(got).all()
    assert rel_l2(got, ora.rhs(U)) <= 1e-12
