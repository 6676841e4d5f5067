"""The mixed sweep's wide spline table (a single periodic system whose
workgroup needs at most 32 KB of LDS with it) against the plain one, which
batches keep: the same walkers to the bit, on both sides of the rule, for 1 to
3 dimensions, lane counts, few and many rows, with and without k-space terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")

from tests.helpers import make_cfg  # noqa: E402


# D, N, k-space terms, knots, lanes
@pytest.mark.parametrize("D,N,K,P_s,lanes", [(1, 2, 0, 4, 16), (1, 33, 10, 110, 32), (2, 7, 0, 24, 16), (2, 100, 60, 40, 64), (2, 31, 0, 80, 32),
                                             (3, 20, 20, 16, 16), (3, 64, 0, 40, 32), (3, 65, 30, 63, 32), (3, 64, 0, 100, 32),
                                             (3, 150, 0, 40, 32), (3, 161, 0, 40, 32), (3, 343, 0, 40, 64)])
def test_wide_table_matches_plain_table(D, N, K, P_s, lanes):
    L = 1.2 * N ** (1.0 / D)
    cfg = make_cfg(N=N, D=D, L=L, P_s=P_s, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=K, hbar2_2m=0.5, W=37)
    rng = np.random.default_rng(10 * N + D)
    print("sweep table", D, N, K, P_s, lanes, flush=True)
    with tdvmc.Batch([cfg]) as b:
        c = b.systems[0]
        u = np.concatenate([rng.normal(0, 0.3, P_s), rng.normal(0, 0.01, c.P - P_s)])
        c.set_params(u, np.zeros(c.P))
        R = c.get_walkers()
        b.set_sweep_lanes(lanes)
        b.sweep(3 * N, seed=5, precision=tdvmc.MIXED)
        want, acc = c.get_walkers(), c.acceptance()
    assert 0 < acc[0] and not np.array_equal(want, R)
    with tdvmc.Context(cfg) as ctx:
        ctx.set_params(u, np.zeros(ctx.P))
        ctx.set_walkers(R)
        ctx.set_sweep_lanes(lanes)
        ctx.sweep(3 * N, seed=tdvmc.batch_system_seed(5, 0), precision=tdvmc.MIXED)
        assert np.array_equal(ctx.get_walkers(), want)
        assert ctx.acceptance() == acc
