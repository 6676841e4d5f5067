"""k-space part of the FP64 measurement against the oracle where its forms
meet: runs of terms and the direct form (8 terms per wavefront), rho_k from
the LDS table, from it with fewer threads per term, and without it (1-D, few
knots), cut shells (unpaired k), one and several rounds of particles."""
import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import energy_scale, make_cfg, oracle_system, rel

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("D,N,K,P_s", [(1, 5, 63, 6), (1, 9, 301, 6), (2, 3, 62, 8), (2, 2, 512, 4), (2, 70, 129, 12), (2, 33, 509, 8),
                                       (3, 2, 40, 8), (3, 3, 511, 4), (3, 65, 131, 10), (3, 130, 66, 10), (3, 20, 256, 24)])
def test_fp64_measurement_with_k_space_terms(D, N, K, P_s, real):
    L = 1.2 * N ** (1.0 / D)
    cfg = make_cfg(N=N, D=D, L=L, P_s=P_s, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=K, hbar2_2m=0.5)
    s = oracle_system(cfg)
    rng = np.random.default_rng(100 * D + N + K)
    R = rng.uniform(-L / 2, L / 2, (2, N, D))
    scale = np.concatenate([np.full(P_s, 0.2), np.full(K, 0.5 / K)])
    uR = rng.normal(0, 1, s.P) * scale
    uI = np.zeros(s.P) if real else rng.normal(0, 1, s.P) * scale
    ref = o.eval_configs(s, R, uR, uI)
    print("eval k-space", D, N, K, P_s, real, flush=True)
    with tdvmc.Context(cfg) as ctx:
        ctx.set_params(uR, uI)
        for per_particle in (False, True):
            out = ctx.eval_configs(R, precision=tdvmc.FP64, per_particle=per_particle)
            assert rel(out["O"], ref["O"]) < 1e-10 and rel(out["expo"], ref["expo"]) < 1e-10
            esc = energy_scale(ref)
            assert np.max(np.abs(out["ER"] - ref["ER"]) / esc) < 1e-10
            assert np.max(np.abs(out["EI"] - ref["EI"]) / esc) < 1e-10
            if per_particle:
                assert rel(out["grad"], ref["grad"]) < 1e-10 and rel(out["lap"], ref["lap"]) < 1e-10
