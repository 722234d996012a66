"""A stability estimate after one whose second launch failed starts from clear
rates: its values are those of a handle that saw no failure.  The failure is
the runtime's own: an interposed hipLaunchKernel asks for a workgroup of 4096
lanes at the chosen launch, which the runtime refuses on the host."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <link.h>
#include <stddef.h>
#include <string.h>
struct Dim3 { unsigned x, y, z; };
typedef int (*Launch)(const void *, struct Dim3, struct Dim3, void **, size_t, void *);
static int fail_at = -1;
static Launch real;
static int find(struct dl_phdr_info *i, size_t n, void *d) {
  void *l;
  (void)n; (void)d;
  if (!strstr(i->dlpi_name, "libamdhip64.so")) return 0;
  l = dlopen(i->dlpi_name, RTLD_LAZY | RTLD_NOLOAD);
  if (l) real = (Launch)dlsym(l, "hipLaunchKernel");
  return real != NULL;
}
void refuse_launch(int n) { fail_at = n; }
int hipLaunchKernel(const void *f, struct Dim3 g, struct Dim3 b, void **a, size_t m, void *s) {
  if (!real) dl_iterate_phdr(find, NULL);
  if (fail_at >= 0 && fail_at-- == 0) { b.x = 4096; b.y = b.z = 1; }
  return real(f, g, b, a, m, s);
}
"""

SCRIPT = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before anything that binds hipLaunchKernel
import numpy as np, torch
from tests.gpu_helpers import make_case, smooth_state
from theseus_amd import _abi as A
from theseus_amd.operator import DeviceClock, MakeRHSOperator
from theseus_amd.serving import Pool, euler_runtime

def refused(n, call):
    shim.refuse_launch(n)
    try:
        call()
    except A.TheseusError as e:
        print("refused:", e, flush=True)
        return
    raise SystemExit("the launch was not refused")

rt, mesh = make_case(2, 3, (5, 4), "ranocha_llf")
slow, fast = (torch.from_numpy(smooth_state(mesh, 3, seed=3, mach=m)).cuda() for m in (0.3, 5.0))
est = lambda op, u: op.EstimateStability(u)
op, fresh = MakeRHSOperator(rt, mesh), MakeRHSOperator(rt, mesh)
ref = est(fresh, slow)
refused(1, lambda: est(op, fast))
assert est(op, slow) == ref, (est(op, slow), ref)
assert est(op, slow) == ref
clock, other = DeviceClock(0.5), DeviceClock(0.5)
refused(1, lambda: op.StepCFL(fast.clone(), clock))
op.StepCFL(slow.clone(), clock)
fresh.StepCFL(slow.clone(), other)
assert clock.read() == other.read(), (clock.read(), other.read())

rt, mesh = make_case(3, 3, (4, 4, 4), "ranocha_llf")
slow, fast = (torch.from_numpy(smooth_state(mesh, 3, seed=3, mach=m)).cuda() for m in (0.3, 5.0))
pools = [Pool(euler_runtime(3), hbm_budget_bytes=1 << 26, max_cases=4) for _ in range(2)]
stream = torch.cuda.current_stream()
# its launches: the mesh, the state, the estimate, the case's start
refused(3, lambda: pools[0].admit(mesh, fast, 0.5, stream, want_dt=False))
dt = [p.admit(mesh, slow, 0.5, stream, want_dt=True)[1] for p in pools]
assert dt[0] == dt[1] > 0, dt
print("ok", flush=True)
"""


def test_estimate_after_a_refused_launch(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", "shim.so", "shim.c", "-ldl"], cwd=tmp_path, check=True)
    (tmp_path / "run.py").write_text(SCRIPT)
    r = subprocess.run([sys.executable, str(tmp_path / "run.py"), str(tmp_path / "shim.so")], cwd=ROOT,
                       env={**os.environ, "PYTHONPATH": str(ROOT)}, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
