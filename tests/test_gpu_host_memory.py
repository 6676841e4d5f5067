"""Pinned memory of the host-pointer calls.  Where it is refused: the same
results by way of pageable memory, as with larger calls.  A context's first
larger call asks for none (it costs more than the call), the second does.  Both
are seen by a library that a child process loads before the product's
(tests/cpp/hip_shim.cpp)."""
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


ONCE = """
import ctypes as C
shim = C.CDLL(%r, mode=C.RTLD_GLOBAL)
import numpy as np
import tdvmc_amd as tdvmc
from tests.helpers import make_cfg
pinned = C.c_size_t.in_dll(shim, "shim_pinned")
cfg = make_cfg(N=64, D=3, L=5.0, P_s=8, pot="GAUSSIAN", sysparams=(0.5, 1.0), hbar2_2m=0.5)
R = np.random.default_rng(3).uniform(-2, 2, (300, 64, 3))
with tdvmc.Context(cfg) as ctx:
    ctx.set_params(np.linspace(0.2, 0.0, 8))
    asked, got = [], []
    for n in (300, 300, 300, 8, 300):
        pinned.value = 0
        got.append(ctx.eval_configs(R[:n]))
        asked.append(pinned.value)
for g in got[1:]:
    assert np.allclose(g["ER"], got[0]["ER"][:len(g["ER"])], rtol=1e-12)
with tdvmc.Context(cfg) as ctx:
    pinned.value = 0
    ctx.eval_configs(R[:4])
    asked.append(pinned.value)
print(*asked)
"""


def test_a_single_larger_call_asks_for_no_pinned_memory():
    print("one larger call", flush=True)
    r = subprocess.run([sys.executable, "-c", ONCE % SHIM], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    first, second, third, small, again, other = map(int, r.stdout.split())
    assert first == 0 and 300 * 64 * 3 * 8 < second <= 1 << 20
    assert third == small == again == 0
    assert 0 < other <= 1 << 16
