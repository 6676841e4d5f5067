"""rho_k of the sweep: every count of k-space terms per lane it is compiled
for, with the phase tables of the FP64 form (2-D, 3-D) and without them (1-D,
mixed form).  A sampling stage measures with the rho_k that its sweep updated
move by move; tdvmc_measure recomputes them from the walkers."""
import numpy as np
import pytest

from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")


# (DIM, N, K, lanes, terms per lane): odd and even N, K that cut a shell (unpaired k), tables of one and of several
# factors per lane
CASES = [(1, 9, 40, 16, 2), (1, 8, 250, 32, 4), (2, 9, 30, 16, 1), (2, 5, 188, 16, 6), (2, 7, 370, 32, 6), (2, 12, 512, 64, 5),
         (3, 27, 18, 16, 1), (3, 26, 100, 16, 4), (3, 5, 207, 16, 7), (3, 5, 222, 16, 8), (3, 13, 147, 32, 3), (3, 11, 301, 32, 5), (3, 2, 256, 64, 2)]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("D,N,K,lanes,terms", CASES)
def test_swept_rho_k_matches_the_recomputed_one(D, N, K, lanes, terms, precision):
    L = 1.3 * N ** (1.0 / D)
    moves = 3 * N + 1
    cfg = make_cfg(N=N, D=D, L=L, P_s=6, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=K, hbar2_2m=0.5, W=67, step=0.4, therm=moves)
    rng = np.random.default_rng(K + N)
    R = rng.uniform(-L / 2, L / 2, (67, N, D))
    print("sweep k-space", D, N, K, lanes, precision, flush=True)
    with tdvmc.Context(cfg) as ctx:
        kh = ctx.info.K_terms
        assert -(-kh // lanes) == terms, kh
        uR = np.concatenate([rng.normal(0, 0.1, 6), rng.normal(0, 0.3 / K, K)])
        ctx.set_params(uR)
        ctx.set_sweep_lanes(lanes)
        ctx.set_walkers(R)
        a = ctx.sample(seed=5, precision=precision)
        acc, trials = ctx.acceptance()
        assert trials == 67 * moves and 0.05 * trials < acc < trials
        b = ctx.measure(precision=precision)
        walkers = ctx.get_walkers()
        # a term of rho_k is off by a few rounding units after each move and |rho_k| <= N, so |rho_k|^2 by 2 N moves
        # eps of its scale and its covariance by twice that
        tol = max(1e-11, 4.0 * N * moves * (6e-8 if precision else 1.2e-16))
        for key in ("localOperators", "S"):
            assert np.max(np.abs(a[key] - b[key])) <= tol * np.max(np.abs(b[key])), key
        if precision == 0:
            # the sums of another lane count differ in their last bits only: the same decisions
            ctx.set_sweep_lanes(64)
            ctx.set_walkers(R)
            ctx.set_rng_state(1, 0)
            ctx.sample(seed=5, precision=precision)
            assert np.array_equal(ctx.get_walkers(), walkers)
