"""Host-side mirror of the reference's RHS operator interface.

The reference exposes ``RHSOperatorBase`` (an ``mfem::TimeDependentOperator``)
with ``Mult(u, dudt)``, ``EstimateStability(u)`` and the concrete
``EulerOperator`` / ``NSOperator`` built by ``MakeRHSOperator(runTime, ...)``
(include/RHSOperator.hpp:19-188, include/SimFactory.hpp:22-31).  These
classes keep those names and argument meanings; vectors are FP64 device
tensors in the reference's byNODES L-vector layout, and every call goes
through the C-ABI of libtheseus_rhs.so.  There is no CPU fallback: the
constructor raises when the library is missing or the tensors are not on a
GPU.
"""
from __future__ import annotations

import ctypes as C
from dataclasses import dataclass

import numpy as np

from . import _abi as A
from .config import RunTime
from .mesh import BoxMesh


@dataclass
class StabilityEstimate:
    """StabilityEstimate.hpp:40-55"""

    advective_rate: float = 0.0
    surface_rate: float = 0.0
    diffusive_rate: float = 0.0

    def TotalRate(self) -> float:
        return max(self.advective_rate, self.surface_rate) + self.diffusive_rate

    def CFL(self, step: float) -> float:
        return step * self.TotalRate()


@dataclass
class IntegralMeasures:
    """Theseus::IntegralMeasures (dgsem_cache.hpp:16-26)."""

    mass: float = 0.0
    ke: float = 0.0
    en: float = 0.0
    max_press: float = 0.0
    min_press: float = 0.0
    max_temp: float = 0.0
    min_temp: float = 0.0
    max_dens: float = 0.0
    min_dens: float = 0.0

    @classmethod
    def from_c(cls, m: "A.IntegralMeasures") -> "IntegralMeasures":
        return cls(**m.as_dict())


class DeviceClock:
    """A theseus_clock in device memory: the state of a variable-step run
    (time, nominal and actual step, end time, CFL target, growth limit, last
    rate, steps taken) that StepCFL advances without a host round trip."""

    FIELDS = ("t", "dt", "dt_real", "t_final", "cfl", "max_dt_growth", "rate", "steps")

    def __init__(self, cfl: float, max_dt_growth: float = 1.2, t_final: float = float("inf"), t: float = 0.0,
                 device="cuda"):
        import torch

        c = A.Clock(t=float(t), dt=0.0, dt_real=0.0, t_final=float(t_final), cfl=float(cfl),
                    max_dt_growth=float(max_dt_growth), rate=0.0, steps=0)
        raw = np.frombuffer(bytes(c), dtype=np.uint8).copy()
        self.buf = torch.from_numpy(raw).to(device)

    @property
    def ptr(self) -> int:
        return self.buf.data_ptr()

    def read(self) -> dict:
        """Synchronous copy of the clock to the host."""
        raw = self.buf.cpu().numpy().tobytes()
        c = A.Clock.from_buffer_copy(raw)
        return {f: getattr(c, f) for f in self.FIELDS}


def _stream_ptr(stream):
    import torch

    if stream is None:
        stream = torch.cuda.current_stream()
    return C.c_void_p(stream.cuda_stream)


def build_descriptor(rt: RunTime, mesh: BoxMesh, elem_orient=None):
    """Fill a theseus_case_desc; returns (desc, keepalive arrays).
    elem_orient: per-element symmetry codes of the storage frames (None:
    every element stored aligned)."""
    if rt.dim != mesh.dim:
        raise ValueError(f"runTime dim {rt.dim} does not match mesh dim {mesh.dim}")
    jac = np.ascontiguousarray(mesh.elem_jac, dtype=np.float64)
    adj = np.ascontiguousarray(mesh.elem_adj, dtype=np.float64)
    nbr = np.ascontiguousarray(mesh.face_neighbor, dtype=np.int32)
    bct = np.ascontiguousarray(mesh.bc_type, dtype=np.int32)
    bcd = np.zeros((bct.size, A.BC_DATA_STRIDE))
    src = getattr(mesh, "bc_data", None)
    if src is not None and bct.size:
        src = np.asarray(src, dtype=np.float64).reshape(bct.size, -1)
        bcd[:, : src.shape[1]] = src
    bcd = np.ascontiguousarray(bcd.reshape(-1))
    d = A.CaseDesc()
    d.dim = rt.dim
    d.order = rt.order
    d.num_elements = mesh.num_elements
    d.flow_model = rt.flow_model
    d.volume_flux = rt.volume_flux
    d.surface_flux = rt.surface_flux
    d.precision = rt.precision
    d.blending = 1 if rt.blending else 0
    d.gamma = rt.gamma
    d.Pr = rt.Pr
    d.R_gas = rt.R_gas
    d.mu = rt.mu
    d.mu_bulk = rt.mu_bulk
    d.alpha_max = rt.alpha_max
    d.alpha_min = rt.alpha_min
    d.elem_jac = jac.ctypes.data_as(C.POINTER(C.c_double))
    d.elem_adj = adj.ctypes.data_as(C.POINTER(C.c_double))
    d.face_neighbor = nbr.ctypes.data_as(C.POINTER(C.c_int))
    d.num_bc = int(bct.size)
    d.bc_type = bct.ctypes.data_as(C.POINTER(C.c_int)) if bct.size else C.POINTER(C.c_int)()
    d.bc_data = bcd.ctypes.data_as(C.POINTER(C.c_double)) if bct.size else C.POINTER(C.c_double)()
    ori = None
    if elem_orient is not None:
        ori = np.ascontiguousarray(elem_orient, dtype=np.uint8)
        if ori.shape != (mesh.num_elements,):
            raise ValueError("elem_orient needs one code per element")
        d.elem_orient = ori.ctypes.data_as(C.POINTER(C.c_ubyte))
    return d, (jac, adj, nbr, bct, bcd, ori)


class RHSOperator:
    """RHSOperator<PhysicsT> (include/RHSOperator.hpp:119-188) over the GPU engine."""

    def __init__(self, runtime: RunTime, mesh: BoxMesh, lte_table=None, elem_orient=None):
        self._lib = A.load()
        self.runtime = runtime
        self.mesh = mesh
        desc, keep = build_descriptor(runtime, mesh, elem_orient)
        h = C.c_void_p()
        if lte_table is None:
            A.check(self._lib, self._lib.theseus_rhs_create(C.byref(desc), C.byref(h)))
        else:
            lt, lkeep = lte_descriptor(lte_table)
            A.check(self._lib, self._lib.theseus_rhs_create_lte(C.byref(desc), C.byref(lt), C.byref(h)))
            del lkeep
        self._h = h
        n = C.c_longlong()
        q = C.c_int()
        A.check(self._lib, self._lib.theseus_rhs_sizes(h, C.byref(n), C.byref(q)))
        self.ndof_total = int(n.value)
        self.num_equations = int(q.value)
        self.num_elements = mesh.num_elements
        self.dim = runtime.dim
        self.order = runtime.order

    # -- reference interface -------------------------------------------------
    @property
    def Height(self) -> int:
        return self.ndof_total * self.num_equations

    def _check(self, t, name):
        import torch

        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise TypeError(f"{name} must be a CUDA/HIP torch tensor (the engine has no CPU path)")
        if t.dtype != torch.float64:
            raise TypeError(f"{name} must be float64")
        if not t.is_contiguous():
            raise ValueError(f"{name} must be contiguous")
        if t.numel() != self.Height:
            raise ValueError(f"{name} has {t.numel()} entries, expected {self.Height}")

    def Mult(self, u, dudt, stream=None) -> None:
        """dudt = L(u) (RHSOperator_impl.hpp:719-793)."""
        self._check(u, "u")
        self._check(dudt, "dudt")
        A.check(self._lib, self._lib.theseus_rhs_eval(self._h, C.c_void_p(u.data_ptr()),
                                                      C.c_void_p(dudt.data_ptr()), _stream_ptr(stream)))

    def EstimateStability(self, u, stream=None) -> StabilityEstimate:
        """RHSOperator_impl.hpp:10-270 with the max-reduction on the device."""
        self._check(u, "u")
        s = A.Stability()
        A.check(self._lib, self._lib.theseus_rhs_estimate_stability(self._h, C.c_void_p(u.data_ptr()),
                                                                    C.byref(s), _stream_ptr(stream)))
        return StabilityEstimate(s.advective_rate, s.surface_rate, s.diffusive_rate)

    def Step(self, u, t: float, dt: float, stream=None) -> float:
        """One SSP-RK3 step in place (mfem::RK3SSPSolver::Step); returns t + dt."""
        self._check(u, "u")
        A.check(self._lib, self._lib.theseus_rhs_step_ssprk3(self._h, C.c_void_p(u.data_ptr()), float(t),
                                                             float(dt), _stream_ptr(stream)))
        return t + dt

    def StepCFL(self, u, clock: DeviceClock, stream=None) -> None:
        """One SSP-RK3 step with the step length chosen on the device from the
        stability estimate of u (the reference's variable-dt loop,
        src/Simulation.cpp:1136-1158,1240-1301); asynchronous, no host copy."""
        self._check(u, "u")
        A.check(self._lib, self._lib.theseus_rhs_step_ssprk3_cfl(self._h, C.c_void_p(u.data_ptr()),
                                                                 C.c_void_p(clock.ptr), _stream_ptr(stream)))

    def ComputeIntegralMeasures(self, u, stream=None) -> IntegralMeasures:
        """RHSOperator::ComputeIntegralMeasures (RHSOperator_impl.hpp:530-717)."""
        self._check(u, "u")
        m = A.IntegralMeasures()
        A.check(self._lib, self._lib.theseus_rhs_integral_measures(self._h, C.c_void_p(u.data_ptr()), C.byref(m),
                                                                   _stream_ptr(stream)))
        return IntegralMeasures.from_c(m)

    def ComputeIntegralMeasuresNoAlloc(self, u, out, stream=None) -> None:
        """The same measures written to the device tensor `out` (9 float64, in
        IntegralMeasures field order) without allocating and without a host
        synchronisation (theseus_rhs_integral_measures_noalloc); the baseline
        is not updated."""
        self._check(u, "u")
        if out.dtype != u.dtype or not out.is_cuda or out.numel() < 9 or not out.is_contiguous():
            raise ValueError("out must be a contiguous float64 device tensor of at least 9 values")
        A.check(self._lib, self._lib.theseus_rhs_integral_measures_noalloc(
            self._h, C.c_void_p(u.data_ptr()), C.c_void_p(out.data_ptr()), _stream_ptr(stream)))

    def EntropyProduction(self, u, dudt, stream=None) -> tuple[float, float]:
        """FP64 entropy production of the right-hand side dudt at u:
        (sum w J S(u).dudt, sum w J |S(u).dudt|), S the gas's entropy
        variables (EOS.hpp:206-234; LTEHelmholtzGasEOS.hpp:144-157 for the
        tabulated gas); <= 0 for an entropy-stable scheme on a periodic mesh,
        whatever precision computed dudt (theseus_rhs_entropy_production)."""
        self._check(u, "u")
        self._check(dudt, "dudt")
        r = A.EntropyProduction()
        A.check(self._lib, self._lib.theseus_rhs_entropy_production(self._h, C.c_void_p(u.data_ptr()),
                                                                    C.c_void_p(dudt.data_ptr()), C.byref(r),
                                                                    _stream_ptr(stream)))
        return r.production, r.magnitude

    def GetIntegralMeasuresBaseline(self) -> IntegralMeasures:
        """RHSOperator::GetIntegralMeasuresBaseline (RHSOperator.hpp:92)."""
        m = A.IntegralMeasures()
        A.check(self._lib, self._lib.theseus_rhs_integral_measures_baseline(self._h, C.byref(m)))
        return IntegralMeasures.from_c(m)

    def Alpha(self, stream=None):
        """Per-element blending coefficient of the last evaluation (device tensor)."""
        import torch

        out = torch.empty(self.num_elements, dtype=torch.float64, device="cuda")
        A.check(self._lib, self._lib.theseus_rhs_get_alpha(self._h, C.c_void_p(out.data_ptr()),
                                                           _stream_ptr(stream)))
        return out

    # -- instrumentation -------------------------------------------------------
    def enable_kernel_timing(self, capacity: int) -> None:
        A.check(self._lib, self._lib.theseus_rhs_enable_kernel_timing(self._h, int(capacity)))

    def kernel_timing(self, kind: int):
        """(mean ms, count) of kernel kind 0 (volume+face / NS pass 2) or 1 (NS pass 1)."""
        ms = C.c_double()
        n = C.c_int()
        A.check(self._lib, self._lib.theseus_rhs_kernel_timing(self._h, int(kind), C.byref(ms), C.byref(n)))
        return float(ms.value), int(n.value)

    def kernel_form(self, kind: int) -> str:
        """"line" or "node": the form of kernel kind 0 or 1 the evaluations run."""
        line = C.c_int()
        A.check(self._lib, self._lib.theseus_rhs_kernel_form(self._h, int(kind), C.byref(line)))
        return "line" if line.value else "node"

    def close(self) -> None:
        if getattr(self, "_h", None):
            self._lib.theseus_rhs_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass


class EulerOperator(RHSOperator):
    """EulerOperator<PhysicsT> (include/EulerOperator.hpp:12-49)."""


class NSOperator(RHSOperator):
    """NSOperator<PhysicsT> (include/NSOperator.hpp:12-71), BR1 viscous terms."""


def lte_descriptor(table):
    """theseus_lte_table from a theseus_amd.lte.HelmholtzTable; returns (desc,
    keepalive).  A table whose `sutherland` attribute is (mu0, T0, Ts) takes
    its viscosity from Sutherland's law (the reference's SUTHERLAND build)."""
    arrays = [np.ascontiguousarray(x, dtype=np.float64).reshape(-1)
              for x in (table.rho, table.T, table.e, table.planes, table.inv)]
    d = A.LteTable()
    d.nx, d.ny = int(table.rho.size), int(table.T.size)
    d.rho_grid, d.T_grid, d.e_grid, d.planes, d.inverse = (a.ctypes.data_as(C.POINTER(C.c_double)) for a in arrays)
    suth = getattr(table, "sutherland", None)
    if suth is not None:
        d.viscosity_model = 1
        d.mu0, d.T0, d.Ts = (float(x) for x in suth)
    return d, arrays


def MakeRHSOperator(runtime: dict | RunTime, mesh: BoxMesh, lte_table=None, elem_orient=None) -> RHSOperator:
    """SimFactory_impl.hpp:63-488: pick the operator from the runTime strings;
    with `lte_table` (a theseus_amd.lte.HelmholtzTable) the gas is the
    tabulated LTE gas (LTEGasModel.hpp:339) with the runtime's LTEEC,
    Pirozzoli, HLL or LLF flux pair; `elem_orient` gives the elements'
    storage frames (theseus_case_desc)."""
    rt = runtime if isinstance(runtime, RunTime) else RunTime.from_json(runtime)
    if rt.lte and lte_table is None:
        raise ValueError("the tabulated LTE gas needs its table (lte_table)")
    cls = NSOperator if rt.flow_model == A.FLOW_NAVIER_STOKES else EulerOperator
    return cls(rt, mesh, lte_table, elem_orient)
