"""Host-pointer calls where pinned memory is refused: the same results by way
of pageable memory, as with larger calls.  The refusal comes from a library
that a child process loads before the product's (tests/cpp/hip_shim.cpp)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
pytest.importorskip("tdvmc_amd")

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = os.path.join(ROOT, "tests", "cpp", "build", "libhip_shim.so")

CHILD = """
import ctypes as C
shim = C.CDLL(%r, mode=C.RTLD_GLOBAL)
import numpy as np
import tdvmc_amd as tdvmc
from tests.helpers import make_cfg
refuse, refused = C.c_int.in_dll(shim, "shim_refuse_pinned"), C.c_int.in_dll(shim, "shim_refused")
cfg = make_cfg(N=7, D=2, L=4.0, P_s=8, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=12, hbar2_2m=0.5, GR_BIN_COUNT=30)
rng = np.random.default_rng(3)
R, u = rng.uniform(-2, 2, (5, 7, 2)), rng.normal(0, 0.1, 20)
A, O = rng.normal(size=(20, 20)), rng.normal(size=(40, 20))
got = []
for no in (0, 1):
    refuse.value = no
    with tdvmc.Context(cfg) as ctx:
        ctx.set_params(u, 0.3 * u)
        e = ctx.eval_configs(R, per_particle=True)
        gr, sk = ctx.observables_configs(R)
        m = ctx.moments(O, np.arange(40.0), np.ones(40))
        s = ctx.solve(u, np.array([1.0, 0.2]), A @ A.T + np.eye(20), u, 2 * u)
        a = ctx.adjoint(R, np.ones(5))
    got.append([x for d in (e, m, s) for _, x in sorted(d.items()) if x is not None] + [gr, sk, *a])
assert refused.value > 0
for x, y in zip(*got):
    # (the measurement adds in LDS in no fixed order: its last bits differ from call to call)
    assert np.allclose(x, y, rtol=1e-12, atol=1e-13 * max(1.0, np.max(np.abs(x))))
print("ok", refused.value)
"""


def test_calls_without_pinned_memory():
    print("host memory", flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD % SHIM], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr
