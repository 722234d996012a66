"""Which form the fused kernel and the gradient pass run on a handle, and their
line forms where a uniform box would hide a mistake: sheared and graded
elements, a metric of its own in every element, elements numbered at random
(neighbours outside the wave), stored frames, device-chosen time steps and
recorded graphs.  Bounds as of the other FP64 right-hand sides: relative
L2 <= 1e-12 against the CPU oracle, bitwise where the same kernels run."""
from types import SimpleNamespace

import numpy as np
import pytest

from theseus_amd import _abi as A

from .gpu_helpers import make_case, oracle_case, rel_l2, smooth_state
from .test_gpu_bc import _case as _bc_case
from .test_gpu_line import _state

pytestmark = pytest.mark.gpu


def _flow(visc):
    return A.FLOW_NAVIER_STOKES if visc else A.FLOW_EULER


def _operator(rt, mesh, **kw):
    from theseus_amd.operator import MakeRHSOperator

    op = MakeRHSOperator(rt, mesh, **kw)
    return op, (op.kernel_form(0), op.kernel_form(1))


def _mult(op, U):
    import torch

    u = torch.from_numpy(U).cuda()
    du = torch.empty_like(u)
    op.Mult(u, du)
    return du.cpu().numpy()


def _remade(box, kind, seed=0):
    """The box's elements with another geometry, numbered at random: the mesh
    and the new place of each element."""
    from theseus_amd.mesh import tensor_mesh

    rng = np.random.default_rng(seed)
    dim, ne = box.dim, box.num_elements
    J, adj = box.elem_jac.copy(), box.elem_adj.reshape(ne, dim, dim).copy()
    if kind == "sheared":  # x -> M x: the area vectors by det M inv M
        M = np.eye(dim) + 0.3 * rng.uniform(-1, 1, (dim, dim))
        J, adj = J * np.linalg.det(M), np.linalg.det(M) * adj @ np.linalg.inv(M)
    elif kind == "graded":
        t = tensor_mesh([np.cumsum(np.r_[0.0, rng.uniform(0.6, 1.4, n) / n]) for n in box.n], periodic=box.periodic)
        J, adj = t.elem_jac.copy(), t.elem_adj.reshape(ne, dim, dim).copy()
    else:  # "own": every element its own, the faces' normals the low side's
        J *= rng.uniform(0.8, 1.25, ne)
        adj += 0.1 * np.abs(adj).max() * rng.uniform(-1, 1, adj.shape)
    place = rng.permutation(ne)
    nbr = box.face_neighbor.reshape(ne, 2 * dim)
    new = np.empty_like(nbr)
    new[place] = np.where(nbr >= 0, place[np.maximum(nbr, 0)], nbr)
    back = np.argsort(place)
    mesh = SimpleNamespace(dim=dim, n=box.n, num_elements=ne, lower=box.lower, upper=box.upper, periodic=box.periodic,
                           elem_jac=J[back].copy(), elem_adj=adj[back].reshape(ne, dim * dim).copy(),
                           face_neighbor=new, bc_type=box.bc_type, bc_data=box.bc_data)
    return mesh, back


def _moved(U, mesh, back):
    return np.ascontiguousarray(U.reshape(mesh.dim + 2, mesh.num_elements, -1)[:, back]).reshape(-1)


@pytest.mark.parametrize("dim,n,order,pairing,visc,blending,forms", [
    (3, (16, 16, 12), 3, "ranocha_llf", False, True, ("line", "node")),   # 768 waves of 4 elements
    (3, (16, 16, 12), 3, "ranocha_llf", True, True, ("line", "line")),
    (3, (17, 15, 12), 3, "ranocha_llf", True, True, ("node", "line")),    # 765
    (3, (127, 4, 4), 3, "llf", True, True, ("node", "node")),             # 508
    (3, (16, 16, 8), 3, "llf", True, True, ("line", "line")),             # 512
    (3, (16, 16, 8), 3, "hll", False, True, ("line", "node")),
    (3, (16, 16, 32), 3, "hll", True, True, ("node", "line")),            # not built
    (3, (16, 15, 24), 3, "chandrashekar", False, False, ("node", "node")),  # 1440 of 1536
    (3, (16, 16, 24), 3, "chandrashekar", False, True, ("line", "node")),
    (3, (16, 32, 31), 3, "chandrashekar_roe", True, True, ("node", "line")),  # 3968 of 4096
    (3, (16, 32, 32), 3, "chandrashekar_roe", True, False, ("line", "line")),
    (3, (8, 8, 8), 4, "ranocha_llf", True, True, ("node", "node")),       # 256 of 2
    (3, (16, 16, 8), 4, "ranocha_llf", True, True, ("node", "line")),     # 1024
    (3, (16, 16, 12), 4, "ranocha_llf", True, True, ("line", "line")),    # 1536
    (3, (16, 16, 12), 4, "hll", False, True, ("node", "node")),           # from 2048
    (3, (16, 16, 16), 4, "hll", False, True, ("line", "node")),
    (3, (16, 16, 64), 4, "llf", True, True, ("node", "line")),            # not built
    (3, (24, 24, 24), 3, "pirozzoli", False, True, ("node", "node")),
    (2, (128, 128), 3, "chandrashekar_roe", False, False, ("line", "node")),  # 1024 of 16
    (2, (128, 128), 3, "chandrashekar_roe", False, True, ("node", "node")),   # with blending from 6144
    (2, (256, 384), 3, "chandrashekar_roe", False, True, ("line", "node")),
    (2, (128, 191), 3, "ranocha_llf", False, True, ("node", "node")),         # 1528 of 1536
    (2, (128, 192), 3, "ranocha_llf", False, True, ("line", "node")),
    (2, (128, 128), 3, "hll", True, True, ("line", "line")),
    (2, (64, 64), 1, "ranocha_llf", True, True, ("node", "node")),
])
def test_forms(dim, n, order, pairing, visc, blending, forms):
    rt, mesh = make_case(dim, order, n, pairing, flow=_flow(visc), blending=blending)
    op, got = _operator(rt, mesh)
    op.close()
    assert got == forms


@pytest.mark.parametrize("dim,n,order,pairing,form", [
    (3, (16, 16, 8), 3, "hll", "node"), (3, (16, 16, 12), 3, "hll", "line"),                    # from 768 waves, periodic 512
    (3, (16, 16, 16), 3, "ranocha", "node"), (3, (16, 16, 24), 3, "ranocha", "line"),           # from 1536, periodic 1024
    (3, (16, 16, 11), 3, "ranocha_llf", "node"), (3, (17, 16, 16), 4, "llf", "node"),           # not built
])
def test_forms_with_boundaries(dim, n, order, pairing, form):
    rt, mesh = _bc_case(dim, order, n, pairing, A.FLOW_EULER, "euler", blending=True)
    op, got = _operator(rt, mesh)
    op.close()
    assert got == (form, "node")


@pytest.mark.parametrize("kind", ["sheared", "graded", "own"])
@pytest.mark.parametrize("noise", ["short", "far"])
@pytest.mark.parametrize("dim,n,order,pairing,visc", [
    (2, (147, 147), 2, "chandrashekar_roe", True), (2, (160, 154), 3, "ranocha_llf", True), (2, (193, 192), 4, "ranocha", False),
    (3, (20, 19, 19), 2, "ranocha_llf", True), (3, (16, 16, 13), 3, "ranocha_llf", False), (3, (17, 15, 17), 3, "ranocha_llf", True),
    (3, (24, 23, 12), 3, "chandrashekar", False), (3, (32, 32, 17), 3, "chandrashekar_roe", True),
    (3, (17, 16, 17), 3, "roe", True), (3, (17, 15, 17), 4, "ranocha_llf", True), (3, (17, 16, 17), 4, "hll", False),
])
def test_metrics_and_numbering(oracle, dim, n, order, pairing, visc, noise, kind):
    rt, box = make_case(dim, order, n, pairing, flow=_flow(visc), blending=True)
    mesh, back = _remade(box, kind, seed=order)
    U = _moved(_state(box, order, rt.gamma, noise), mesh, back)
    op, forms = _operator(rt, mesh)
    got = _mult(op, U)
    op.close()
    # the gradient pass's line form takes an element's own area vectors at both ends
    assert forms == ("line", "line" if visc and kind != "own" else "node")
    err = rel_l2(got, oracle_case(oracle, rt, mesh).rhs(U))
    assert err <= 1e-12, err


@pytest.mark.parametrize("kind", ["sheared", "own"])
@pytest.mark.parametrize("sides", ["euler", "no_slip"])
@pytest.mark.parametrize("noise", ["short", "far"])
@pytest.mark.parametrize("dim,n,order,pairing", [
    (2, (160, 154), 3, "ranocha_llf"), (2, (147, 147), 2, "chandrashekar"), (3, (17, 17, 17), 3, "hll"),
    (3, (17, 16, 16), 4, "ranocha_llf"), (3, (17, 16, 16), 4, "ranocha"), (3, (17, 16, 17), 4, "hll"),
])
def test_metrics_and_boundaries(oracle, dim, n, order, pairing, noise, sides, kind):
    rt, box = _bc_case(dim, order, n, pairing, A.FLOW_EULER, sides, blending=True)
    mesh, back = _remade(box, kind, seed=order)
    U = _moved(_state(box, order, rt.gamma, noise), mesh, back)
    op, forms = _operator(rt, mesh)
    got = _mult(op, U)
    op.close()
    assert forms == ("line", "node")
    err = rel_l2(got, oracle_case(oracle, rt, mesh).rhs(U))
    assert err <= 1e-12, err


@pytest.mark.parametrize("visc", [False, True])
def test_stored_frames(visc):
    """Elements stored in random frames of the cube: the aligned handle's
    results, bit for bit."""
    from theseus_amd.meshio import to_aligned, to_storage

    rt, box = make_case(3, 3, (15, 15, 14), "ranocha_llf", flow=_flow(visc), blending=True)
    mesh = SimpleNamespace(**{k: getattr(box, k) for k in ("dim", "num_elements", "face_neighbor", "bc_type", "elem_jac",
                                                           "elem_adj", "lower", "upper")})
    mesh.elem_orient = np.random.default_rng(5).integers(0, 48, size=box.num_elements).astype(np.uint8)
    U = smooth_state(box, 3, seed=5)
    op, forms = _operator(rt, box)
    ref = _mult(op, U)
    op.close()
    op, stored = _operator(rt, mesh, elem_orient=mesh.elem_orient)
    got = to_aligned(_mult(op, to_storage(U, mesh, 3)), mesh, 3)
    op.close()
    assert forms == stored == ("line", "line" if visc else "node")
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("dim,n,order,visc", [(2, (160, 154), 3, True), (3, (15, 15, 14), 3, True), (3, (17, 15, 17), 4, False)])
def test_device_clock_and_graph(dim, n, order, visc):
    """Steps of the length the device chooses equal steps given that length, and
    recorded steps equal eager ones, bit for bit, on every replay with eager
    work between."""
    import torch

    from theseus_amd.operator import DeviceClock

    rt, mesh = make_case(dim, order, n, "ranocha_llf", flow=_flow(visc), blending=True)
    op, forms = _operator(rt, mesh)
    assert forms == ("line", "line" if visc else "node")
    u0 = torch.from_numpy(smooth_state(mesh, order, seed=7)).cuda()
    chosen, given, clock = u0.clone(), u0.clone(), DeviceClock(0.5)
    lengths = []
    for _ in range(2):
        op.StepCFL(chosen, clock)
        lengths.append(clock.read()["dt_real"])
        op.Step(given, 0.0, lengths[-1])
    assert lengths[0] > 0.0 and torch.equal(chosen, given)

    state, clock2 = u0.clone(), DeviceClock(0.5)
    start = clock2.buf.clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        for _ in range(2):
            op.StepCFL(state, clock2)
    torch.cuda.synchronize()
    other = torch.from_numpy(smooth_state(mesh, order, seed=8, amp=0.1)).cuda()
    for replay in range(3):
        state.copy_(u0)
        clock2.buf.copy_(start)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(state, chosen) and clock2.read()["dt_real"] == lengths[-1], replay
        op.Step(other, 0.0, lengths[0])
        op.EstimateStability(other)
    op.close()


@pytest.mark.parametrize("dim,n,order,visc", [(2, (147, 147), 2, False), (2, (160, 154), 3, True), (2, (111, 111), 4, True),
                                              (3, (20, 19, 19), 2, True), (3, (21, 20, 20), 3, False), (3, (17, 15, 17), 3, True),
                                              (3, (17, 15, 17), 4, False), (3, (17, 15, 17), 4, True)])
def test_conservation_at_low_mach(dim, n, order, visc):
    """On a periodic box the volume-weighted sum of every rate is 0: 1e-12 of
    the sum of its magnitudes, as the full-size Taylor-Green vortex is held to,
    on a state whose pressure (71) is that of Mach 0.1."""
    from theseus_amd.mesh import gll_nodes

    rt, mesh = make_case(dim, order, n, "ranocha_llf", flow=_flow(visc), blending=True, mu=1 / 1600)
    U = smooth_state(mesh, order, rt.gamma, amp=0.01, seed=9, mach=1.0).reshape(dim + 2, -1)
    U[-1] += (1.0 / (rt.gamma * 0.1 ** 2) - 1.0 / rt.gamma) / (rt.gamma - 1)
    op, forms = _operator(rt, mesh)
    r = _mult(op, U.reshape(-1)).reshape(dim + 2, -1)
    op.close()
    assert forms[0] == "line"
    w = gll_nodes(order)[1]
    W = w
    for _ in range(dim - 1):
        W = np.multiply.outer(w, W)
    W = (W.reshape(-1)[None, :] * mesh.elem_jac[:, None]).reshape(-1)
    for k in range(dim + 2):
        assert abs((r[k] * W).sum()) <= 1e-12 * (np.abs(r[k]) * W).sum(), (k, (r[k] * W).sum(), (np.abs(r[k]) * W).sum())
