"""The FP64 measurement with one and two wavefronts per walker against the
oracle: last workgroups with idle slots, k-space terms on both sides of the
run form's rule and of the rho_k table's, per-particle output, real and complex
parameters.  A few configurations are repeated up to a walker count that takes
the form (tests/cpp/eval_rules_check.cpp says which one that is)."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import energy_scale, make_cfg, oracle_system

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "build", "eval_rules_check")


# wavefronts per walker (without and with per-particle output), D, N, K, knots, configurations (odd counts: idle slots in
# the last workgroup)
CASES = [(1, 1, 1, 5, 20, 6, 2049), (1, 1, 1, 16, 127, 8, 2050), (1, 1, 2, 2, 10, 4, 2051), (1, 2, 2, 25, 30, 12, 4099), (1, 1, 2, 16, 126, 16, 2049),
         (1, 1, 3, 7, 0, 24, 2050), (1, 2, 3, 32, 60, 10, 2051), (1, 1, 3, 13, 122, 8, 2049), (1, 2, 2, 31, 126, 8, 2049), (2, 2, 1, 30, 300, 6, 1025),
         (2, 2, 2, 9, 64, 8, 1025), (2, 2, 2, 33, 374, 8, 2049), (2, 2, 3, 16, 200, 8, 1027), (2, 2, 3, 36, 26, 24, 1025), (2, 4, 3, 48, 256, 10, 1025),
         (2, 4, 2, 64, 100, 24, 1025), (2, 4, 3, 63, 131, 10, 1025), (2, 4, 3, 50, 66, 16, 1025), (2, 4, 3, 80, 66, 10, 1025), (4, 4, 3, 81, 66, 10, 1025)]


@pytest.mark.parametrize("real", [True, False])
@pytest.mark.parametrize("waves,waves_pp,D,N,K,P_s,W", CASES)
def test_one_and_two_wavefronts_per_walker(waves, waves_pp, D, N, K, P_s, W, real):
    L = 1.2 * N ** (1.0 / D)
    cfg = make_cfg(N=N, D=D, L=L, P_s=P_s, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=K, hbar2_2m=0.5)
    s = oracle_system(cfg)
    rng = np.random.default_rng(100 * D + N + K)
    few = rng.uniform(-L / 2, L / 2, (3, N, D))
    row = np.arange(W) % 3
    scale = np.concatenate([np.full(P_s, 0.2), np.full(K, 0.5 / max(K, 1))])
    uR = rng.normal(0, 1, s.P) * scale
    uI = np.zeros(s.P) if real else rng.normal(0, 1, s.P) * scale
    ref = o.eval_configs(s, few, uR, uI)
    print("eval waves", waves, D, N, K, P_s, W, real, flush=True)
    with tdvmc.Context(cfg) as ctx:
        Kh = ctx.info.K_terms
        ctx.set_params(uR, uI)
        for per_particle in (False, True):
            used = subprocess.run([CHECK], input="%d %d %d %d %d %d 1 1" % (D, N, P_s, Kh, W, per_particle), capture_output=True, text=True,
                                  check=True).stdout.split()[0]
            assert int(used) == (waves_pp if per_particle else waves)
            out = ctx.eval_configs(few[row], precision=tdvmc.FP64, per_particle=per_particle)
            for key in ("O", "expo") + (("grad", "lap") if per_particle else ()):
                want = ref[key].reshape((3,) + out[key].shape[1:])
                assert np.max(np.abs(out[key] - want[row])) < 1e-10 * np.max(np.abs(want)), key
            esc = energy_scale(ref)[row]
            for key in ("ER", "EI"):
                assert np.max(np.abs(out[key] - ref[key][row]) / esc) < 1e-10, key
