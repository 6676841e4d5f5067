"""FP64 g(r) and S(k) where their forms meet, against the oracle: the matrix
product (2-D, 3-D) and the direct sums (1-D), bins from thresholds with pairs
exactly half a box apart, one and several chunks of particles, small walkers
that share a workgroup, a box too large for the FP32 guess."""
import numpy as np
import pytest

from oracle import oracle as o
from tests.helpers import make_cfg

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")


@pytest.mark.parametrize("D,N,L,bins", [(1, 9, 9.0, 40), (2, 2, 3.0, 10), (2, 17, 4.0, 33), (2, 64, 8.0, 200), (2, 130, 11.0, 3000),
                                        (3, 2, 3.0, 7), (3, 15, 3.0, 50), (3, 65, 4.1, 200), (3, 129, 5.0, 400), (3, 20, 3e13, 50)])
@pytest.mark.parametrize("lattice", [False, True])
def test_fp64_observables_vs_oracle(D, N, L, bins, lattice):
    rng = np.random.default_rng(D * 1000 + N)
    W, P = 3, 10
    R = rng.uniform(-L, L, (W, N, D))
    if lattice:
        R = np.rint(R * (4.0 / L)) * (L / 4.0) + rng.integers(0, 2, R.shape) * (L / 512)   # exact halves and ties among them
    print("observables", D, N, bins, lattice, flush=True)
    cfg = make_cfg(N, D, L, P, W=W, GR_BIN_COUNT=bins, MC_NADDITIONALTHERMSTEPS=0, MC_NADDITIONALINITIALIZATIONSTEPS=0)
    with tdvmc.Context(cfg) as ctx:
        gr, sk = ctx.observables_configs(R, precision=tdvmc.FP64)
        ctx.set_walkers(R)
        gm, sm = ctx.additional_properties(seed=1, n_samples=1, precision=tdvmc.FP64)
    ogr, osk = o.observables(R, L, P, L / 2, bins)
    np.testing.assert_allclose(sk, osk, rtol=1e-10, atol=1e-11 * np.max(osk))
    if lattice:
        # a fused multiply-add in the minimum image moves an exact tie by a rounding unit: the same pairs, at most
        # in the neighbouring bin
        _, _, _, scl = o.gr_grid(D, P, L / 2, bins)
        c, co = (np.rint(g * scl * (N - 1) / D) for g in (gr, ogr))
        assert np.max(np.abs(np.cumsum(c - co, axis=1))) <= np.max(co)
    else:
        np.testing.assert_allclose(gr, ogr, rtol=1e-12, atol=0)
    np.testing.assert_allclose(gm, gr.mean(0), rtol=1e-12, atol=0)
    np.testing.assert_allclose(sm, sk.mean(0), rtol=1e-12, atol=1e-14 * np.max(sk))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("D,N", [(1, 6), (2, 9), (3, 14)])
def test_walkers_that_share_a_workgroup(D, N, precision):
    L, W = 1.5 * N ** (1.0 / D), 2500
    rng = np.random.default_rng(N)
    R = rng.uniform(-L / 2, L / 2, (W, N, D))
    cfg = make_cfg(N, D, L, 8, W=W, GR_BIN_COUNT=60, MC_NADDITIONALTHERMSTEPS=0, MC_NADDITIONALINITIALIZATIONSTEPS=0)
    print("shared workgroups", D, N, precision, flush=True)
    with tdvmc.Context(cfg) as ctx:
        gr, sk = ctx.observables_configs(R, precision=precision)
        ctx.set_walkers(R)
        gm, sm = ctx.additional_properties(seed=1, n_samples=2, precision=precision)
    np.testing.assert_allclose(gm, gr.mean(0), rtol=1e-12, atol=0)
    np.testing.assert_allclose(sm, sk.mean(0), rtol=1e-12, atol=0)
