"""FP64 moments where their two forms meet and at the edges of the chunks: up
to 64 computed columns and 32768 samples in two launches (chunks of 64
samples combined by the parallel-variance formula), beyond that packed."""
import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")


@pytest.mark.parametrize("W,P", [(1, 1), (2, 14), (63, 15), (64, 30), (65, 62), (130, 63), (4097, 62), (4097, 63), (32768, 5), (32769, 5)])
def test_fp64_moments_forms(W, P):
    rng = np.random.default_rng(W + P)
    O = 50.0 + 3.0 * rng.normal(size=(W, P))
    O[:, 0] = 1e4 + O[:, 0]
    ER = O @ rng.normal(size=P) * 0.1 + rng.normal(size=W)
    EI = 0.2 * rng.normal(size=W) + 0.05 * O[:, 0]
    print("moments forms", W, P, flush=True)
    with tdvmc.Context(make_cfg(N=4, D=3, L=4.0, P_s=8)) as ctx:
        m = ctx.moments(O, ER, EI, precision=tdvmc.FP64)
    ref = o.moments(O, ER, EI)
    # a covariance's rounding: eps times the spread of both columns, the means' (up to 1e4, so 2e-12) times the spread
    tol = 1e-12 * max(np.max(np.abs(ref["S"])), 1.0) + 4e-12 * np.sqrt(max(np.max(np.abs(ref["S"])), 1.0))
    for key in ("S", "FR", "FI"):
        assert np.max(np.abs(m[key] - ref[key])) <= tol, key
    assert np.max(np.abs(m["mO"] - ref["mO"]) / np.abs(ref["mO"])) < 1e-13
    assert np.max(np.abs(m["mE"] - ref["mE"]) / np.abs(ref["mE"])) < 1e-12
    assert np.array_equal(m["S"], m["S"].T)
