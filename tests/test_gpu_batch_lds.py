"""LDS of a batch's sweep with k-space terms: what the launched precision needs
(the FP64 form's coordinates and phase tables would halve the mixed form's
workgroups per CU).  The launch is seen by a library that a child process loads
before the product's (tests/cpp/hip_shim.cpp)."""
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
import tdvmc_amd as tdvmc
from tests.helpers import make_cfg
most = C.c_size_t.in_dll(shim, "shim_most_lds")
D, L, P_s, sizes = %d, 4.0, 24, (40, 33, 17)
cfgs = [make_cfg(N=n, D=D, L=L, P_s=P_s, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=%d, hbar2_2m=0.5, W=70) for n in sizes]
with tdvmc.Batch(cfgs) as b:
    out = []
    for precision in (tdvmc.MIXED, tdvmc.FP64):
        b.sweep(5, seed=1, precision=precision)
        most.value = 0
        b.sweep(5, seed=2, precision=precision)
        out.append(most.value)
print(*out)
"""


@pytest.mark.parametrize("D,K", [(2, 60), (2, 128), (3, 60)])
def test_mixed_sweep_takes_its_own_lds(D, K):
    print("batch lds", D, K, flush=True)
    r = subprocess.run([sys.executable, "-c", CHILD % (SHIM, D, K)], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    mixed, fp64 = map(int, r.stdout.split())
    # 16 walkers of 40 particles, 32-bit coordinates; spline rows (4 FP32 each) out to the largest distance
    rows = int(D ** 0.5 * 23) + 2
    assert mixed == 16 * 40 * D * 4 + 16 * rows
    assert fp64 > 2 * mixed
