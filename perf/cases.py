"""What the engine is measured on: the calls a solver or a serving program
makes, at the sizes of this repository's workloads and over the ranges around
them.

A case is one pass through the public operator or pool interface:

  mult      dudt = L(u)                                (RHSOperator.Mult)
  step      one SSP-RK3 step in place, fixed dt        (RHSOperator.Step)
  step_cfl  one SSP-RK3 step, dt chosen on the device  (RHSOperator.StepCFL)
  serve     admit several cases, step them together, read them, release them (Pool)

``exact`` evaluates the same scheme with plain torch in 64 bits on the box
meshes used here (axis-aligned elements), independently of the engine.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from theseus_amd import _abi as A
from theseus_amd.config import RunTime
from theseus_amd.lte import R_AIR, synthetic_table
from theseus_amd.mesh import box_mesh, gll_nodes
from theseus_amd.operator import DeviceClock, MakeRHSOperator
from theseus_amd.serving import Pool, euler_runtime

F64 = torch.float64
GAMMA, PR, RE, MACH = 1.4, 0.71, 1600.0, 0.1
R_GAS = 287.05
CFL = 0.5
SERVE_STEPS = 20

FLUXES = {
    "ranocha_llf": (A.VOLUME_RANOCHA, A.SURFACE_LLF),
    "chandrashekar": (A.VOLUME_CHANDRASHEKAR, A.SURFACE_CHANDRASHEKAR),
    "chandrashekar_roe": (A.VOLUME_CHANDRASHEKAR, A.SURFACE_ROE),
    "hll": (A.VOLUME_CENTRAL, A.SURFACE_HLL),
    "lteec": (A.VOLUME_LTEEC, A.SURFACE_LTEEC),
}


def _case(name, flow, call, n, p, flux, blending=False, viscous=False, mixed=False):
    n = tuple(n)
    c = {"flow": flow, "call": call, "dim": len(n), "nx": n[0], "ny": n[1], "nz": n[2] if len(n) > 2 else 1,
         "p": p, "flux": flux, "blending": blending, "viscous": viscous, "mixed": mixed}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest workload: a 2-D Euler vortex, variable-step time loop; 256 elements, so launches and latency
        _case("vortex2d_16_p3", "vortex", "step_cfl", (16, 16), 3, "chandrashekar_roe", blending=True),
        # the lid-driven cavity, refined: no-slip walls, Navier-Stokes, fixed dt (boundary-condition kernels)
        _case("cavity2d_48x40_p3", "cavity", "step", (48, 40), 3, "chandrashekar", blending=True, viscous=True),
        # shock-capturing workload: four-quadrant Riemann problem, subcell blending, transmissive boundaries
        _case("riemann2d_128_p4", "riemann", "mult", (128, 128), 4, "hll", blending=True),
        # a coarse Taylor-Green run: 3-D Navier-Stokes with few elements per compute unit
        _case("tgv_8_p3", "tgv", "step", (8, 8, 8), 3, "ranocha_llf", blending=True, viscous=True),
        # the headline workload: 3-D Navier-Stokes Taylor-Green vortex, 10.5 million unknowns
        _case("tgv_32_p3", "tgv", "step", (32, 32, 32), 3, "ranocha_llf", blending=True, viscous=True),
        # the same in the mixed-precision form
        _case("tgv_32_p3_mixed", "tgv", "step", (32, 32, 32), 3, "ranocha_llf", blending=True, viscous=True, mixed=True),
        # a production-size run: 35 million unknowns
        _case("tgv_48_p3", "tgv", "step", (48, 48, 48), 3, "ranocha_llf", blending=True, viscous=True),
        # 3-D Euler at order 4 on a ragged grid (odd counts in every direction)
        _case("euler_17x15x13_p4", "tgv", "mult", (17, 15, 13), 4, "ranocha_llf"),
        # tabulated real gas with the entropy-conserving flux: the gas's headline workload
        _case("lteec_24_p3", "lte", "mult", (24, 24, 24), 3, "lteec"),
        # the tabulated gas's Navier-Stokes form, order 2, small and ragged
        _case("lteec_ns_11x10x9_p2", "lte", "mult", (11, 10, 9), 2, "lteec", viscous=True),
        # the tabulated gas with an ordinary flux pair: recovery and node passes weigh as much as the fluxes
        _case("lte_hll_24_p3", "lte", "mult", (24, 24, 24), 3, "hll"),
        # the serving path: a handful of mixed-precision cases admitted, stepped together, read back, released
        _case("serve_p3", "serve", "serve", (8, 13, 20), 3, "ranocha_llf", mixed=True),
    ]


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi, dim, cap):
        n = [logint(lo, hi) for _ in range(dim)]
        while math.prod(n) > cap:
            n[n.index(max(n))] -= 1
        return n

    kind = rng.choice(("vortex", "cavity", "riemann", "tgv", "tgv", "euler", "lte", "lte", "serve"))
    if kind == "vortex":
        return _case(None, "vortex", "step_cfl", box(8, 160, 2, 20000), rng.choice((2, 3, 4)), "chandrashekar_roe", blending=True)
    if kind == "cavity":
        return _case(None, "cavity", "step", box(8, 120, 2, 12000), rng.choice((2, 3)), "chandrashekar", blending=True,
                     viscous=True)
    if kind == "riemann":
        return _case(None, "riemann", "mult", box(16, 300, 2, 60000), rng.choice((3, 4)), "hll", blending=True)
    if kind == "tgv":
        p = rng.choice((2, 3, 3, 4))
        return _case(None, "tgv", "step", box(5, 44, 3, 6_000_000 // (p + 1) ** 3), p, "ranocha_llf",
                     blending=rng.random() < 0.7, viscous=True, mixed=rng.random() < 0.25)
    if kind == "euler":
        p = rng.choice((2, 3, 4))
        return _case(None, "tgv", "mult", box(5, 40, 3, 4_000_000 // (p + 1) ** 3), p,
                     rng.choice(("ranocha_llf", "chandrashekar", "hll")), blending=rng.random() < 0.4)
    if kind == "lte":
        p = rng.choice((2, 3, 3))
        return _case(None, "lte", "mult", box(5, 24, 3, 880_000 // (p + 1) ** 3), p, rng.choice(("lteec", "lteec", "hll")),
                     viscous=rng.random() < 0.4)
    return _case(None, "serve", "serve", [logint(8, 20) for _ in range(3)], rng.choice((2, 3, 4)), "ranocha_llf", mixed=True)


def _grid(c):
    return (c["nx"], c["ny"], c["nz"])[: c["dim"]]


def _serve_grids(c):
    """The served cases' sizes: each of the three counts twice, cubes."""
    return [c["nx"], c["ny"], c["nz"], c["nz"], c["ny"], c["nx"]]


def _nodes(c):
    npn = (c["p"] + 1) ** c["dim"]
    return sum(n ** 3 for n in _serve_grids(c)) * npn if c["flow"] == "serve" else math.prod(_grid(c)) * npn


def _bounds(c):
    return {"vortex": (-5.0, 5.0), "cavity": (0.0, 1.0), "riemann": (0.0, 1.0)}.get(c["flow"], (0.0, 2 * math.pi))


# Fixed walls and a lid at unit speed: (velocity, heat flux), the sides in the order x-, x+, y-, y+
_CAVITY_WALLS = ((0.0, 0.0, 0.0), (0.0, 0.0, 0.0), (0.0, 0.0, 0.0), (1.0, 0.0, 0.0))


def _mesh(c):
    lo, hi = _bounds(c)
    if c["flow"] == "cavity":
        return box_mesh(2, _grid(c), lo, hi, periodic=False, side_bc=[(A.BC_NO_SLIP_ADIABATIC, w) for w in _CAVITY_WALLS])
    if c["flow"] == "riemann":
        return box_mesh(2, _grid(c), lo, hi, periodic=False, bc=A.BC_SUPERSONIC_OUTFLOW)
    return box_mesh(c["dim"], _grid(c), lo, hi, periodic=True)


def _runtime(c):
    vol, surf = FLUXES[c["flux"]]
    mu, pr = (0.02, 0.72) if c["flow"] == "cavity" else (1.0 / RE, PR)
    return RunTime(dim=c["dim"], order=c["p"], flow_model=A.FLOW_NAVIER_STOKES if c["viscous"] else A.FLOW_EULER,
                   volume_flux=vol, surface_flux=surf, gamma=GAMMA, Pr=pr, mu=mu, R_gas=R_GAS, blending=c["blending"],
                   precision=A.PRECISION_MIXED if c["mixed"] else A.PRECISION_FP64, lte=c["flow"] == "lte")


# --- inputs ---------------------------------------------------------------

@functools.lru_cache(maxsize=1)
def _table():
    return synthetic_table()


def _coords(n, p, lo, hi, device):
    """Node coordinates, one tensor per direction, element-major with x fastest."""
    dim, Np = len(n), p + 1
    x01 = torch.tensor(gll_nodes(p)[0], dtype=F64, device=device)
    e = torch.arange(math.prod(n), device=device)
    k = torch.arange(Np ** dim, device=device)
    out, se, sk = [], 1, 1
    for d in range(dim):
        h = (hi - lo) / n[d]
        out.append((lo + h * ((e // se) % n[d])[:, None] + h * x01[(k // sk) % Np][None, :]).reshape(-1))
        se, sk = se * n[d], sk * Np
    return out


def _waves(rng, X, lo, hi, modes=4):
    """A smooth random field of unit size: a few low Fourier modes of the box."""
    f = torch.zeros_like(X[0])
    for _ in range(modes):
        arg = float(rng.uniform(0, 2 * math.pi))
        for x in X:
            arg = arg + (2 * math.pi / (hi - lo)) * int(rng.integers(0, 3)) * (x - lo)
        f += float(rng.uniform(0.3, 1.0)) / modes * torch.cos(arg)
    return f


def _conservative(rho, vel, p):
    ke = sum(0.5 * rho * v * v for v in vel)
    return torch.cat([rho, *[rho * v for v in vel], p / (GAMMA - 1.0) + ke]).contiguous()


def _state(c, seed, device, n=None):
    """The flow's initial field with the seed's perturbation."""
    rng = np.random.default_rng([seed, 17])
    lo, hi = _bounds(c)
    n = _grid(c) if n is None else n
    X = _coords(n, c["p"], lo, hi, device)
    w = [_waves(rng, X, lo, hi) for _ in range(4)]
    if c["flow"] == "vortex":  # isentropic vortex in a unit stream (Mach 0.85)
        x0, y0 = (float(v) for v in rng.uniform(-1, 1, 2))
        r2 = (X[0] - x0) ** 2 + (X[1] - y0) ** 2
        T = 1.0 - (GAMMA - 1) * 25.0 / (8 * GAMMA * math.pi ** 2) * torch.exp(1 - r2)
        du = 5.0 / (2 * math.pi) * torch.exp(0.5 * (1 - r2))
        rho = T ** (1 / (GAMMA - 1))
        return _conservative(rho * (1 + 0.02 * w[0]), [1 - du * (X[1] - y0), 1 + du * (X[0] - x0)], rho ** GAMMA * (1 + 0.02 * w[1]))
    if c["flow"] == "cavity":  # nearly at rest, Mach 0.1 with the lid
        p0 = 1.0 / (GAMMA * MACH ** 2)
        return _conservative(1 + 0.002 * w[0], [0.05 * w[1], 0.05 * w[2]], p0 * (1 + 0.002 * w[3]))
    if c["flow"] == "riemann":
        east, north = X[0] >= float(rng.uniform(0.4, 0.6)), X[1] >= float(rng.uniform(0.4, 0.6))
        pick = lambda ne, nw, sw, se: torch.where(north, torch.where(east, ne, nw), torch.where(east, se, sw))  # noqa: E731
        t = lambda *v: [torch.tensor(x, dtype=F64, device=device) for x in v]  # noqa: E731
        rho, u = pick(*t(1.5, 0.5323, 0.138, 0.5323)), pick(*t(0.0, 1.206, 1.206, 0.0))
        v, p = pick(*t(0.0, 0.0, 1.206, 1.206)), pick(*t(1.5, 0.3, 0.029, 0.3))
        return _conservative(rho * (1 + 0.05 * w[0]), [u + 0.02 * w[1], v + 0.02 * w[2]], p * (1 + 0.05 * w[3]))
    a = [float(v) for v in rng.uniform(0, 2 * math.pi, 3)]
    s = [X[d] + a[d] for d in range(3)]
    tu = torch.sin(s[0]) * torch.cos(s[1]) * torch.cos(s[2])
    tv = -torch.cos(s[0]) * torch.sin(s[1]) * torch.cos(s[2])
    tp = (torch.cos(2 * s[0]) + torch.cos(2 * s[1])) * (torch.cos(2 * s[2]) + 2) / 16.0
    if c["flow"] == "lte":  # dissociating gas around 0.1 kg/m^3, 3500 K, Mach 0.3
        rho = 0.1 * (1 + 0.03 * w[0])
        U = 0.3 * math.sqrt(1.3 * R_AIR * 3500.0)
        T = 3500.0 * (1 + 0.02 * w[1]) + U * U * tp / R_AIR
        vel = [U * tu, U * tv, 0.1 * U * w[2]]
        e = _Gas(_table(), device).at(rho, T).energy()
        return torch.cat([rho, *[rho * v for v in vel], rho * e + sum(0.5 * rho * v * v for v in vel)]).contiguous()
    amp = float(rng.uniform(0.5, 3.0)) if c["flow"] == "serve" else 1.0
    p0 = 100.0 / GAMMA if c["flow"] == "serve" else 1.0 / (GAMMA * MACH ** 2)
    return _conservative(1 + 0.02 * w[0], [amp * tu, amp * tv, 0.1 * w[2]], p0 + amp ** 2 * tp + 0.1 * w[3])


# Largest stable rates of the one-dimensional operators by order (RHS of the linear problems on a unit element)
_ADVECTION = (0.0, 2.19706891727, 5.41995189335, 9.64849524786, 14.7297419321, 20.5984751391)
_DIFFUSION = (0.0, 4.0, 25.5969429388, 82.9000427145, 203.470468982, 426.230394541)


def _rate(c, u, n):
    """Advective plus diffusive rate of an ideal-gas state on a box: dt = CFL / rate."""
    lo, hi = _bounds(c)
    rt = _runtime(c)
    q = u.reshape(c["dim"] + 2, -1)
    v = q[1:-1] / q[0]
    p = (GAMMA - 1) * (q[-1] - 0.5 * (q[1:-1] * v).sum(0))
    cs = torch.sqrt(GAMMA * p / q[0])
    ih = [n[d] / (hi - lo) for d in range(c["dim"])]
    rate = 1.05 * _ADVECTION[c["p"]] * float(sum((v[d].abs() + cs) * ih[d] for d in range(c["dim"])).max())
    if c["viscous"]:
        nu = rt.mu * max(1.0, 2.0 - rt.mu_bulk, GAMMA / rt.Pr) / float(q[0].min())
        rate += 1.25 * _DIFFUSION[c["p"]] * nu * sum(x * x for x in ih)
    return rate


def prepare(case, seed):
    c = case
    if c["flow"] == "serve":
        sizes = _serve_grids(c)
        meshes = {n: box_mesh(3, n, 0.0, 2 * math.pi, periodic=True) for n in set(sizes)}
        states = [_state(c, seed * 31 + i, "cuda", (n, n, n)) for i, n in enumerate(sizes)]
        pool = Pool(euler_runtime(c["p"]), hbm_budget_bytes=1 << 30, max_cases=16)
        return {"call": "serve", "pool": pool, "cases": [(meshes[n], u) for n, u in zip(sizes, states)],
                "out": [torch.empty_like(u) for u in states]}
    mesh = _mesh(c)
    u = _state(c, seed, "cuda")
    op = MakeRHSOperator(_runtime(c), mesh, lte_table=_table() if c["flow"] == "lte" else None)
    s = {"call": c["call"], "op": op, "u": u}
    if c["call"] == "mult":
        s["dudt"] = torch.empty_like(u)
    elif c["call"] == "step":
        s["dt"], s["t"] = CFL / _rate(c, u, _grid(c)), 0.0
    else:
        s["clock"] = DeviceClock(CFL)
    return s


def run(state):
    s = state
    if s["call"] == "mult":
        s["op"].Mult(s["u"], s["dudt"])
        return s["dudt"]
    if s["call"] == "step":
        s["t"] = s["op"].Step(s["u"], s["t"], s["dt"])
        return s["u"]
    if s["call"] == "step_cfl":
        s["op"].StepCFL(s["u"], s["clock"])
        return s["u"]
    pool, stream = s["pool"], torch.cuda.current_stream()
    ids = [pool.admit(mesh, u, CFL, stream, want_dt=False)[0] for mesh, u in s["cases"]]
    for _ in range(SERVE_STEPS):
        pool.step(stream)
    for i, out in zip(ids, s["out"]):
        pool.read(i, out, stream)
        pool.release(i, stream)
    return s["out"]


def work(case):
    """The state read and the result written once; the two-point fluxes, face fluxes and contractions of
    every evaluation in floating point operations."""
    c = case
    nodes, dim, Np = _nodes(c), c["dim"], c["p"] + 1
    evals = {"mult": 1, "serve": 3 * SERVE_STEPS}.get(c["call"], 3)
    per_pair = 650 if c["flux"] == "lteec" else {"ranocha_llf": 75, "chandrashekar": 85, "chandrashekar_roe": 85, "hll": 60}[c["flux"]]
    flops = dim * (Np - 1) / 2 * per_pair + dim * (Np - 1) * 2 * (dim + 2) + dim / Np * (150 if c["flux"] != "lteec" else 750)
    if c["viscous"]:
        flops += 4 * dim * Np * (dim + 2) + 150
    if c["flow"] == "lte":
        flops += 400
    return {"bytes": 2 * 8.0 * (dim + 2) * nodes, "flops": float(evals * nodes * flops)}


# --- the scheme in plain 64-bit torch ----------------------------------------

class _Gas:
    """The tabulated gas: bicubic Hermite H(rho, T) on the table's cells."""

    def __init__(self, t, device):
        as_t = lambda x: torch.tensor(np.asarray(x), dtype=F64, device=device)  # noqa: E731
        self.rho, self.T, self.P, self.nx, self.ny = as_t(t.rho), as_t(t.T), as_t(t.planes).reshape(6, -1), t.nx, t.ny

    def cell(self, grid, v):
        return (torch.searchsorted(grid, v.contiguous(), right=True) - 1).clamp(0, grid.numel() - 2)

    def at(self, rho, T, ij=None):
        i, j = (self.cell(self.rho, rho), self.cell(self.T, T)) if ij is None else ij
        return _Point(self, rho, T, i, j)

    def recover(self, rho, e):
        """T with e(rho, T) = e by Newton from the middle of the range of interest."""
        T = torch.full_like(rho, 3500.0)
        for _ in range(60):
            s = self.at(rho, T)
            step = (e - s.energy()) / (-T * s.H(0, 2))
            T = (T + step).clamp(float(self.T[0]), float(self.T[-1]))
            if float(step.abs().max()) < 1e-10:
                break
        return T


def _basis(der, x):
    """Hermite bases (value 0, value 1, slope 0, slope 1) on [0, 1], derivative `der`."""
    if der == 0:
        return 2 * x ** 3 - 3 * x ** 2 + 1, -2 * x ** 3 + 3 * x ** 2, x ** 3 - 2 * x ** 2 + x, x ** 3 - x ** 2
    if der == 1:
        return 6 * x ** 2 - 6 * x, -6 * x ** 2 + 6 * x, 3 * x ** 2 - 4 * x + 1, 3 * x ** 2 - 2 * x
    return 12 * x - 6, -12 * x + 6, 6 * x - 4, 6 * x - 2


def _divided(der, x, y):
    """Divided differences of those bases between x and y."""
    if der == 0:
        a, b = x * x + x * y + y * y, x + y
        return 2 * a - 3 * b, -2 * a + 3 * b, a - 2 * b + 1, a - b
    b = x + y
    return 6 * b - 6, -6 * b + 6, 3 * b - 4, 3 * b - 2


class _Point:
    def __init__(self, gas, rho, T, i, j):
        self.gas, self.rho, self.T, self.i, self.j = gas, rho, T, i, j
        self.wr, self.wt = gas.rho[i + 1] - gas.rho[i], gas.T[j + 1] - gas.T[j]
        self.xi, self.eta = (rho - gas.rho[i]) / self.wr, (T - gas.T[j]) / self.wt

    def tensor(self, br, bt):
        """Sum of the cell's 16 coefficients with the rho bases `br` and the T bases `bt`."""
        P, o = self.gas.P, self.j * self.gas.nx + self.i
        r = 0.0
        for a in range(2):
            for b in range(2):
                k = o + a + b * self.gas.nx
                r = r + P[0][k] * br[a] * bt[b] + P[1][k] * self.wr * br[2 + a] * bt[b]
                r = r + P[2][k] * self.wt * br[a] * bt[2 + b] + P[3][k] * self.wr * self.wt * br[2 + a] * bt[2 + b]
        return r

    def H(self, dr=0, dt=0):
        return self.tensor(_basis(dr, self.xi), _basis(dt, self.eta)) / (self.wr ** dr * self.wt ** dt)

    def energy(self):
        return self.H() - self.T * self.H(0, 1)

    def pressure(self):
        return self.rho ** 2 * self.H(1, 0)

    def gibbs(self):
        return self.H() + self.rho * self.H(1, 0)

    def cv(self):
        return -self.T * self.H(0, 2)

    def c2(self):
        return 2 * self.rho * self.H(1, 0) + self.rho ** 2 * self.H(2, 0) - self.rho ** 2 * self.H(1, 1) ** 2 / self.H(0, 2)

    def transport(self, plane):
        P, o, x, y = self.gas.P[plane], self.j * self.gas.nx + self.i, self.xi, self.eta
        return P[o] * (1 - x) * (1 - y) + P[o + 1] * x * (1 - y) + P[o + self.gas.nx] * (1 - x) * y + P[o + self.gas.nx + 1] * x * y


def _lte_means(a, b):
    """Entropy-conserving density and energy means from the discrete gradients of p/T and g/T in (rho, 1/T)."""
    gas = a.gas
    b1, b2, dr, db = 1 / a.T, 1 / b.T, b.rho - a.rho, 1 / b.T - 1 / a.T
    far_r = dr.abs() >= 2.22e-15 + 1.49e-8 * torch.maximum(a.rho, b.rho)
    far_b = db.abs() >= 2.22e-15 + 1.49e-8 * torch.maximum(b1, b2)
    same = (a.i == b.i) & (a.j == b.j)
    ab, ba = gas.at(a.rho, b.T, (a.i, b.j)), gas.at(b.rho, a.T, (b.i, a.j))
    xb = (b.rho - gas.rho[a.i]) / a.wr  # b's coordinates in a's cell (used where the cells agree)
    yb = (b.T - gas.T[a.j]) / a.wt
    rs = lambda der: tuple(v / a.wr ** (der + 1) for v in _divided(der, a.xi, xb))  # noqa: E731
    ts = lambda der: tuple(v / a.wt ** (der + 1) for v in _divided(der, a.eta, yb))  # noqa: E731
    r0, r1 = (lambda x: _basis(0, x)), (lambda x: tuple(v / a.wr for v in _basis(1, x)))
    t0 = lambda y: _basis(0, y)  # noqa: E731

    def gradient(value, rho_secant, beta_secant, d_rho, d_T):
        f11, f22, f12, f21 = value(a), value(b), value(ab), value(ba)
        safe = lambda x, ok: torch.where(ok, x, torch.ones_like(x))  # noqa: E731
        g_same = 0.5 * (rho_secant(a.eta) * b1 + rho_secant(yb) * b2)
        g_diff = 0.5 * ((f21 * b1 - f11 * b1) + (f22 * b2 - f12 * b2)) / safe(dr, far_r)
        g_near = 0.5 * (d_rho(a) * b1 + d_rho(b) * b2)
        h_same = 0.5 * (beta_secant(a.xi, a.rho) + beta_secant(xb, b.rho))
        h_diff = 0.5 * ((f12 * b2 - f11 * b1) + (f22 * b2 - f21 * b1)) / safe(db, far_b)
        h_near = 0.5 * ((f11 - a.T * d_T(a)) + (f22 - b.T * d_T(b)))
        return (torch.where(far_r, torch.where(same, g_same, g_diff), g_near),
                torch.where(far_b, torch.where(same, h_same, h_diff), h_near))

    def p_rho_secant(y):
        mean = 0.5 * (a.tensor(r1(a.xi), t0(y)) + a.tensor(r1(xb), t0(y)))
        return 0.5 * (a.rho ** 2 + b.rho ** 2) * a.tensor(rs(1), t0(y)) + (a.rho + b.rho) * mean

    def g_rho_secant(y):
        mean = 0.5 * (a.tensor(r1(a.xi), t0(y)) + a.tensor(r1(xb), t0(y)))
        return a.tensor(rs(0), t0(y)) + 0.5 * (a.rho + b.rho) * a.tensor(rs(1), t0(y)) + mean

    tm = 0.5 * (a.T + b.T)

    def hr_beta(x):
        return 0.5 * (a.tensor(r1(x), t0(a.eta)) + a.tensor(r1(x), t0(yb))) - tm * a.tensor(r1(x), ts(0))

    def p_beta_secant(x, rho):
        return rho ** 2 * hr_beta(x)

    def g_beta_secant(x, rho):
        return 0.5 * (a.tensor(r0(x), t0(a.eta)) + a.tensor(r0(x), t0(yb))) - tm * a.tensor(r0(x), ts(0)) + rho * hr_beta(x)

    pr, pb = gradient(_Point.pressure, p_rho_secant, p_beta_secant,
                      lambda s: 2 * s.rho * s.H(1, 0) + s.rho ** 2 * s.H(2, 0), lambda s: s.rho ** 2 * s.H(1, 1))
    gr, gb = gradient(_Point.gibbs, g_rho_secant, g_beta_secant,
                      lambda s: 2 * s.H(1, 0) + s.rho * s.H(2, 0), lambda s: s.H(0, 1) + s.rho * s.H(1, 1))
    rho_m = pr / gr
    return rho_m, gb - pb / rho_m


def _log_mean(x, y):
    u = ((y - x) / (x + y)) ** 2
    series = 0.5 * (x + y) / (1 + u * (1 / 3 + u * (1 / 5 + u / 7)))
    return torch.where(u < 1e-4, series, (y - x) / torch.where(u < 1e-4, torch.ones_like(x), torch.log(y / x)))


class _Scheme:
    """The semi-discrete operator of a case on a box, states shaped (equations, elements z..x, nodes z..x)."""

    def __init__(self, c, n, device):
        self.c, self.n, self.dim, self.Np, self.rt = c, n, len(n), c["p"] + 1, _runtime(c)
        lo, hi = _bounds(c)
        self.h = [(hi - lo) / v for v in n]
        x, w = gll_nodes(c["p"])
        self.w = w
        bary = [1 / math.prod(x[i] - x[j] for j in range(self.Np) if j != i) for i in range(self.Np)]
        D = np.array([[0.0 if i == j else bary[j] / bary[i] / (x[i] - x[j]) for j in range(self.Np)] for i in range(self.Np)])
        self.D = D - np.diag(D.sum(1))
        self.shape = (self.dim + 2, *n[::-1], *(self.Np,) * self.dim)
        self.gas = _Gas(_table(), device) if c["flow"] == "lte" else None

    def e_axis(self, d):
        return self.dim - d

    def n_axis(self, d):
        return 2 * self.dim - d

    # point samples: dict of tensors without the equation axis ("v": one per direction)
    def derive(self, q):
        s = {"q": q, "rho": q[0], "v": q[1:-1] / q[0], "E": q[-1]}
        ke = 0.5 * (q[1:-1] ** 2).sum(0) / q[0]
        if self.gas is None:
            s["p"] = (GAMMA - 1) * (q[-1] - ke)
            s["c"] = torch.sqrt(GAMMA * s["p"] / s["rho"])
            s["i"] = s["j"] = None
        else:
            s["T"] = self.gas.recover(s["rho"], (q[-1] - ke) / q[0])
            pt = self.gas.at(s["rho"], s["T"])
            s["p"], s["c"], s["i"], s["j"] = pt.pressure(), torch.sqrt(pt.c2()), pt.i, pt.j
        return s

    def pick(self, s, axis, k):
        """Node k along node axis `axis` (an axis of the equation-carrying arrays)."""
        one = lambda x, a: None if x is None else x.select(a, k)  # noqa: E731
        return {key: one(x, axis if key in ("q", "v") else axis - 1) for key, x in s.items()}

    def shift(self, s, axis, by):
        one = lambda x, a: None if x is None else torch.roll(x, by, a)  # noqa: E731
        return {key: one(x, axis if key in ("q", "v") else axis - 1) for key, x in s.items()}

    def physical(self, s, d):
        vn = s["v"][d]
        f = s["q"] * vn
        f[1 + d] += s["p"]
        f[-1] += s["p"] * vn
        return f

    def point(self, s):
        return self.gas.at(s["rho"], s["T"], (s["i"], s["j"]))

    def volume(self, a, b, d):
        flux = self.c["flux"]
        if flux == "hll":
            return 0.5 * (self.physical(a, d) + self.physical(b, d))
        vb = 0.5 * (a["v"] + b["v"])
        vn, pb = vb[d], 0.5 * (a["p"] + b["p"])
        f = torch.empty_like(a["q"])
        if flux == "lteec":
            rho_m, e_m = _lte_means(self.point(a), self.point(b))
            mass, pw = rho_m * vn, 0.5 * (a["p"] * b["v"][d] + b["p"] * a["v"][d])
            f[0], f[1:-1] = mass, mass * vb
            f[1 + d] += pb
            f[-1] = mass * (e_m + 0.5 * (a["v"] * b["v"]).sum(0)) + pw
            return f
        rho_l = _log_mean(a["rho"], b["rho"])
        f[0], f[1:-1] = rho_l * vn, rho_l * vn * vb
        if flux == "ranocha_llf":
            f[1 + d] += pb
            inv = 1 / ((GAMMA - 1) * _log_mean(a["rho"] / a["p"], b["rho"] / b["p"]))
            f[-1] = rho_l * vn * (inv + 0.5 * (a["v"] * b["v"]).sum(0)) + 0.5 * (a["p"] * b["v"][d] + b["p"] * a["v"][d])
        else:
            ba, bb = 0.5 * a["rho"] / a["p"], 0.5 * b["rho"] / b["p"]
            ph = 0.5 * (a["rho"] + b["rho"]) / (ba + bb)
            f[1 + d] += ph
            hh = 0.5 / ((GAMMA - 1) * _log_mean(ba, bb)) + ph / rho_l - 0.25 * (a["v"] ** 2 + b["v"] ** 2).sum(0) + (vb ** 2).sum(0)
            f[-1] = rho_l * vn * hh
        return f

    def surface(self, a, b, d):
        """Riemann flux along +d, a on the low side."""
        flux = self.c["flux"]
        jump = b["q"] - a["q"]
        lam = torch.maximum(a["v"][d].abs() + a["c"], b["v"][d].abs() + b["c"])
        if flux == "lteec":
            return self.volume(a, b, d) - 0.5 * lam * jump
        if flux == "ranocha_llf":
            return 0.5 * (self.physical(a, d) + self.physical(b, d)) - 0.5 * lam * jump
        fa, fb = self.physical(a, d), self.physical(b, d)
        if flux == "hll":
            sl = torch.minimum(a["v"][d] - a["c"], b["v"][d] - b["c"])
            sr = torch.maximum(a["v"][d] + a["c"], b["v"][d] + b["c"])
            mid = (sr * fa - sl * fb + sl * sr * jump) / (sr - sl)
            return torch.where(sl >= 0, fa, torch.where(sr <= 0, fb, mid))
        if flux == "chandrashekar":
            rm, dr = 0.5 * (a["rho"] + b["rho"]), b["rho"] - a["rho"]
            ba, bb = 0.5 * a["rho"] / a["p"], 0.5 * b["rho"] / b["p"]
            de = (0.5 * dr * a["v"] * b["v"] + rm * (b["v"] - a["v"]) * 0.5 * (a["v"] + b["v"])).sum(0)
            de = de + (0.5 * dr / _log_mean(ba, bb) + 0.5 * rm * (1 / bb - 1 / ba)) / (GAMMA - 1)
            diss = 0.5 * lam * jump
            diss[-1] = 0.5 * lam * de
            return self.volume(a, b, d) - diss
        ra, rb = torch.sqrt(a["rho"]), torch.sqrt(b["rho"])
        u = (ra * a["v"] + rb * b["v"]) / (ra + rb)
        H = (ra * (a["E"] + a["p"]) / a["rho"] + rb * (b["E"] + b["p"]) / b["rho"]) / (ra + rb)
        u2, un, rr = (u * u).sum(0), u[d], ra * rb
        a2 = (GAMMA - 1) * (H - 0.5 * u2)
        cs = torch.sqrt(a2)
        dv, dp = b["v"] - a["v"], b["p"] - a["p"]
        dun = dv[d]
        am, ap = 0.5 * (dp - rr * cs * dun) / a2, 0.5 * (dp + rr * cs * dun) / a2
        a0 = b["rho"] - a["rho"] - dp / a2
        lm, l0, lp = (un - cs).abs(), un.abs(), (un + cs).abs()
        nrm = torch.zeros_like(u)
        nrm[d] = 1.0
        dt = dv - dun * nrm
        diss = torch.empty_like(a["q"])
        diss[0] = lm * am + l0 * a0 + lp * ap
        diss[1:-1] = lm * am * (u - cs * nrm) + l0 * (a0 * u + rr * dt) + lp * ap * (u + cs * nrm)
        diss[-1] = lm * am * (H - cs * un) + l0 * (0.5 * a0 * u2 + rr * (u * dt).sum(0)) + lp * ap * (H + cs * un)
        return 0.5 * (fa + fb) - 0.5 * diss

    def wall_flux(self, s, d, sign):
        """(0, p* n, 0) of the wall Riemann problem, n = sign e_d."""
        v, p, rho = sign * s["v"][d], s["p"], s["rho"]
        gp, gm = GAMMA + 1, GAMMA - 1
        shock = p + 0.25 * v * gp * rho * (v + torch.sqrt(v * v + 8 / gp * p * (gm / gp + 1) / rho))
        fan = p * torch.clamp(1 + 0.5 * gm * v / s["c"], min=1e-4) ** (2 * GAMMA / gm)
        f = torch.zeros_like(s["q"])
        f[1 + d] = torch.where(v > 0, shock, fan)
        return f  # along +d: the outward flux is sign * f, lifted with sign

    def periodic(self):
        return self.c["flow"] not in ("cavity", "riemann")

    def indicator(self, s):
        """Persson-Peraire blending coefficient per element."""
        p, Np, dim = self.c["p"], self.Np, self.dim
        x = 2 * gll_nodes(p)[0] - 1
        V = torch.tensor(np.linalg.inv(np.polynomial.legendre.legvander(x, p)), dtype=F64, device=s["rho"].device)
        m = s["rho"] * s["p"]
        for d in range(dim):
            m = torch.tensordot(m, V, ([self.n_axis(d) - 1], [1])).movedim(-1, self.n_axis(d) - 1)
        m = m ** 2
        cut = lambda k: m[(..., *[slice(0, k)] * dim)].flatten(dim).sum(-1) if k > 0 else torch.zeros(m.shape[:dim], dtype=F64, device=m.device)  # noqa: E731
        mm, m1, m2 = cut(Np), cut(Np - 1), cut(Np - 2)
        eta = torch.where(m1 > 1e-30, torch.maximum(1 - m1 / mm, 1 - m2 / m1), torch.ones_like(mm))
        eta = torch.where(mm > 1e-30, eta, torch.zeros_like(mm)).clamp(0, 1)
        th = 0.5 * 10 ** (-1.8 * p ** 0.25)
        al = 1 / (1 + torch.exp(-9.21024 * (eta - th) / th))
        al = torch.where(al < 0.001, torch.zeros_like(al), torch.where(al > 0.999, torch.ones_like(al), al))
        return al.clamp(max=0.5)

    def viscous(self, s, du):
        """Adds the BR1 viscous terms."""
        q, rho, v, w0, dim = s["q"], s["rho"], s["v"], self.w[0], self.dim
        rt = self.rt
        if self.gas is None:
            beta = rho / s["p"]
            S = torch.cat([((GAMMA - torch.log(s["p"]) + GAMMA * torch.log(rho)) / (GAMMA - 1) - 0.5 * beta * (v * v).sum(0))[None],
                           beta * v, -beta[None]])
            mu = rt.mu * torch.ones_like(rho)
            kappa_t = rt.mu * GAMMA / ((GAMMA - 1) * rt.Pr) / beta ** 2
        else:
            pt = self.point(s)
            beta = 1 / s["T"]
            S = torch.cat([(beta * (pt.gibbs() - 0.5 * (v * v).sum(0)))[None], beta * v, -beta[None]])
            mu, kappa_t = pt.transport(4), pt.transport(5) / beta ** 2
        D = torch.tensor(self.D, dtype=F64, device=q.device)
        grad = []
        for d in range(dim):
            ea, na, ih = self.e_axis(d), self.n_axis(d), 1 / self.h[d]
            g = torch.tensordot(S, D, ([na], [1])).movedim(-1, na) * ih
            lo, hi = S.select(na, 0), S.select(na, self.Np - 1)
            jump = 0.5 * (torch.roll(lo, -1, ea) - hi)  # at the high face of each element
            jlow = torch.roll(jump, 1, ea)
            if not self.periodic():
                for side, tr, target, k, sg in ((0, lo, jlow, 0, -1.0), (1, hi, jump, self.n[d] - 1, 1.0)):
                    wall = _CAVITY_WALLS[2 * d + side]
                    t = tr.select(ea, k)
                    j = torch.zeros_like(t)
                    for m in range(dim):
                        j[1 + m] = wall[m] * -t[-1] - t[1 + m]
                    target.select(ea, k).copy_(sg * j)
            g.select(na, 0).add_(jlow * (ih / w0))
            g.select(na, self.Np - 1).add_(jump * (ih / w0))
            grad.append(g)
        gv = [[(grad[d][1 + m] + v[m] * grad[d][-1]) / beta for m in range(dim)] for d in range(dim)]
        div = sum(gv[d][d] for d in range(dim))
        Dh = self.D.copy()
        Dh[0, 0] += 1 / w0
        Dh[-1, -1] -= 1 / w0
        Dh = torch.tensor(Dh, dtype=F64, device=q.device)
        for d in range(dim):
            ea, na, ih = self.e_axis(d), self.n_axis(d), 1 / self.h[d]
            tau = [mu * (gv[d][m] + gv[m][d]) - (mu * rt.mu_bulk * div if m == d else 0.0) for m in range(dim)]
            f = torch.stack([*tau, kappa_t * grad[d][-1] + sum(v[m] * tau[m] for m in range(dim))])
            out = torch.tensordot(f, Dh, ([na], [1])).movedim(-1, na) * ih
            lo, hi = f.select(na, 0), f.select(na, self.Np - 1)
            fs = 0.5 * (hi + torch.roll(lo, -1, ea))
            flow = torch.roll(fs, 1, ea)
            if not self.periodic():
                for side, tr, target, k in ((0, lo, flow, 0), (1, hi, fs, self.n[d] - 1)):
                    wall = _CAVITY_WALLS[2 * d + side]
                    t = tr.select(ea, k).clone()
                    t[-1] = sum(wall[m] * t[m] for m in range(dim))
                    target.select(ea, k).copy_(t)
            out.select(na, 0).sub_(flow * (ih / w0))
            out.select(na, self.Np - 1).add_(fs * (ih / w0))
            du[1:] += out

    def rhs(self, u):
        s = self.derive(u.reshape(self.shape))
        du = torch.zeros_like(s["q"])
        faces = torch.zeros_like(du)
        fv = torch.zeros_like(du)
        Np, w0 = self.Np, self.w[0]
        for d in range(self.dim):
            ea, na, ih = self.e_axis(d), self.n_axis(d), 1 / self.h[d]
            nodes = [self.pick(s, na, k) for k in range(Np)]
            for a in range(Np):
                for b in range(a + 1, Np):
                    f = self.volume(nodes[a], nodes[b], d)
                    du.select(na, a).sub_(f * (2 * self.D[a, b] * ih))
                    du.select(na, b).sub_(f * (2 * self.D[b, a] * ih))
            lo, hi = nodes[0], nodes[Np - 1]
            f = self.surface(hi, self.shift(lo, ea, -1), d)
            flow = torch.roll(f, 1, ea)
            if not self.periodic():
                one = lambda t, k: {key: None if x is None else x.select(ea if key in ("q", "v") else ea - 1, k) for key, x in t.items()}  # noqa: E731
                for side, tr, target, k in ((0, lo, flow, 0), (1, hi, f, self.n[d] - 1)):
                    t = one(tr, k)
                    wall = self.c["flow"] == "cavity"
                    target.select(ea, k).copy_(self.wall_flux(t, d, 2 * side - 1) if wall else self.physical(t, d))
            faces.select(na, 0).add_(flow * (ih / w0))
            faces.select(na, Np - 1).sub_(f * (ih / w0))
            if self.c["blending"]:
                for k in range(Np - 1):
                    g = self.surface(nodes[k], nodes[k + 1], d)
                    fv.select(na, k).sub_(g * (ih / self.w[k]))
                    fv.select(na, k + 1).add_(g * (ih / self.w[k + 1]))
        if self.c["blending"]:
            al = self.indicator(s).reshape(1, *self.n[::-1], *(1,) * self.dim)
            du = (1 - al) * du + al * fv
        du += faces
        if self.c["viscous"]:
            self.viscous(s, du)
        return du.reshape(-1)

    def step(self, u, dt):
        a = u + dt * self.rhs(u)
        b = 0.75 * u + 0.25 * (a + dt * self.rhs(a))
        return u / 3 + 2 / 3 * (b + dt * self.rhs(b))


def exact(case, seed, device="cuda"):
    c = case
    if c["flow"] == "serve":
        out = []
        for i, n in enumerate(_serve_grids(c)):
            u = _state(c, seed * 31 + i, device, (n, n, n))
            s, dt = _Scheme(c, (n, n, n), device), CFL / _rate(c, u, (n, n, n))
            for _ in range(SERVE_STEPS):
                u = s.step(u, dt)
            out.append(u)
        return out
    u = _state(c, seed, device)
    s = _Scheme(c, _grid(c), device)
    return s.rhs(u) if c["call"] == "mult" else s.step(u, CFL / _rate(c, u, _grid(c)))
