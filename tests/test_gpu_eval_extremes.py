"""FP64 pair distances at the ends of the range of their squares, against the
oracle: particles so far apart that the square overflows, and so close that it
is next to the smallest doubles, beside ordinary ones."""
import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import energy_scale, make_cfg, oracle_system, rel

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")


def _compare(cfg, R, R_ref, tol):
    s = oracle_system(cfg)
    rng = np.random.default_rng(5)
    uR, uI = rng.normal(0, 0.2, s.P), rng.normal(0, 0.2, s.P)
    ref = o.eval_configs(s, R_ref, uR, uI)
    assert all(np.all(np.isfinite(ref[k])) for k in ("expo", "ER", "EI", "O", "grad", "lap"))
    with tdvmc.Context(cfg) as ctx:
        ctx.set_params(uR, uI)
        for per_particle in (False, True):
            out = ctx.eval_configs(R, precision=tdvmc.FP64, per_particle=per_particle)
            assert rel(out["O"], ref["O"]) < tol and rel(out["expo"], ref["expo"]) < tol
            esc = energy_scale(ref)
            assert np.max(np.abs(out["ER"] - ref["ER"]) / esc) < tol
            assert np.max(np.abs(out["EI"] - ref["EI"]) / esc) < tol
            if per_particle:
                assert rel(out["grad"], ref["grad"]) < tol


@pytest.mark.parametrize("pot", ["LJ", "GAUSSIAN", "SQUARE_WELL"])
@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("far", [1e153, 1.2e154, 1e160, 1e200])
def test_far_particles_in_open_space(D, pot, far):
    cfg = make_cfg(N=6, D=D, L=0.0, P_s=8, pot=pot, sysparams=(0.5, 1.0), rc=4.0, hbar2_2m=0.5)
    R = np.random.default_rng(D).normal(0, 1.5, (3, 6, D))
    R[0, 2, D - 1] = far
    R[1, 0, 0] = -far
    R[1, 5, 0] = far
    print("far particles", D, pot, far, flush=True)
    _compare(cfg, R, R, 1e-10)


@pytest.mark.parametrize("L", [0.0, 7.0])
@pytest.mark.parametrize("D", [1, 2, 3])
@pytest.mark.parametrize("near", [1e-140, 1e-148, 2e-150, 1e-151, 1e-153])
def test_particles_next_to_each_other(D, L, near):
    cfg = make_cfg(N=6, D=D, L=L, P_s=8, pot="GAUSSIAN", sysparams=(0.5, 1.0), rc=0.0 if L else 3.0, hbar2_2m=0.5)
    R = np.random.default_rng(D).normal(0, 1.2, (2, 6, D))
    R[0, 1] = 0.0
    R[0, 4] = 0.0
    R[0, 4, D - 1] = near
    # u'(r) / r of the innermost pieces needs r / h beside 1 in the oracle's basis functions, which is lost below 1e-16:
    # its values at 1e-6, from where everything changes by a few times 1e-6 of its scale at most
    R_ref = R.copy()
    R_ref[0, 4, D - 1] = 1e-6
    print("near particles", D, L, near, flush=True)
    _compare(cfg, R, R_ref, 2e-5)
