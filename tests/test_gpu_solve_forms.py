"""The Cholesky solve at the sizes where its kernels change over or a block is
partial: one block, a block and a row, the smallest panel buffers, the last
size of the kernel that factors ahead (P = 340) and of the 32-column blocks
(P = 581), and both sides of them.
Against the oracle's restatement, with the tolerance of the solver's other
tests; a repeated call gives the same bits (no race between the steps that run
side by side)."""
import numpy as np
import pytest

from oracle import oracle as o

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")

from tests.helpers import make_cfg  # noqa: E402


def _ctx():
    return tdvmc.Context(make_cfg(N=4, D=3, L=4.0, P_s=8, K=0))


def _moments(P, bad=()):
    rng = np.random.default_rng(P)
    A = rng.normal(size=(P, P))
    S = A @ A.T / P + 0.01 * np.eye(P)
    for i in bad:
        S[i, :] = 0.0
        S[:, i] = 0.0
        S[i, i] = -0.5
    return dict(mO=rng.normal(size=P), mE=np.array([1.3, -0.4]), S=S, FR=rng.normal(size=P), FI=rng.normal(size=P))


def _check(m, bad, pre):
    with _ctx() as ctx:
        r, again = (ctx.solve(m["mO"], m["mE"], m["S"], m["FR"], m["FI"], imag_time=1, precondition=pre, eps=1e-3, check=False)
                    for _ in range(2))
    ref = o.solve_param_dot(m, imag_time=1, precondition=pre, eps=1e-3)
    assert r["bad"] == ref["bad"] == bad
    for k in ("xR", "xI"):
        assert np.linalg.norm(r[k] - ref[k]) < 1e-10 * np.linalg.norm(ref[k])
        assert np.array_equal(r[k], again[k])
    for k in ("phiDotR", "phiDotI"):
        assert abs(r[k] - ref[k]) < 1e-10 * max(1, abs(ref[k]))


@pytest.mark.parametrize("pre", [0, 1])
@pytest.mark.parametrize("P", [1, 2, 15, 16, 17, 31, 32, 47, 48, 49, 64, 65, 336, 337, 340, 341, 561, 576, 577, 581, 582, 609])
def test_solve_edges(P, pre):
    print("solve", P, pre, flush=True)
    _check(_moments(P), 0, pre)


# non-positive pivots in the first block, on both sides of a block's edge, in a
# block factored ahead and in a partial last one
@pytest.mark.parametrize("P,bad", [(16, (0,)), (33, (15, 16, 32)), (50, (3, 31, 49)), (340, (0, 177, 339)), (577, (0, 300, 576))])
def test_solve_pivots(P, bad):
    print("solve", P, bad, flush=True)
    _check(_moments(P, bad), len(bad), 0)
