"""What a TDVP step leaves on the device, for every solver of the ODE and with
and without a post-step update: the epoch of the random streams (stepped by
the measurement that follows a sweep, or by a launch of its own) and the
parameters in force (written by the last update, or unpacked after it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
tdvmc = pytest.importorskip("tdvmc_amd")

from tests.helpers import make_cfg  # noqa: E402

FRESH_STAGES = {0: 1, 1: 2, 2: 4, 3: 1, 5: 1}


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("spw,init,norm", [(1, 0, 0), (2, 7, 1)])
@pytest.mark.parametrize("ode", [0, 1, 2, 3, 5])
def test_epoch_and_parameters_after_steps(ode, spw, init, norm, graph):
    cfg = make_cfg(N=5, D=2, L=4.0, P_s=6, pot="GAUSSIAN", sysparams=(0.5, 1.0), K=6, W=64, therm=20, init=init,
                   SAMPLES_PER_WALKER=spw, ODE_SOLVER_TYPE=ode, USE_NORMALIZE_WF=norm, IMAGINARY_TIME=1)
    rng = np.random.default_rng(3)
    R = rng.uniform(-2, 2, (64, 5, 2))
    print("step", ode, spw, init, norm, graph, flush=True)
    with tdvmc.Context(cfg) as ctx:
        u0 = rng.normal(0, 0.1, ctx.P)
        ctx.set_walkers(R)
        ctx.set_params(u0, np.zeros(ctx.P))
        e0 = ctx.get_rng_state()[1]
        for _ in range(3):
            ctx.tdvp_step(1e-4, ode, use_graph=graph)
        assert ctx.get_rng_state()[1] - e0 == 3 * FRESH_STAGES[ode] * (spw + (init > 0))
        ctx.sample(1)
        ctx.sweep(10, 1)
        assert ctx.get_rng_state()[1] - e0 == 3 * FRESH_STAGES[ode] * (spw + (init > 0)) + spw + (init > 0) + 1
        assert ctx.step_status() == 0
        p = ctx.get_params()
        out = ctx.eval_configs(R[:3])
    with tdvmc.Context(cfg) as ref:
        ref.set_params(*p)
        want = ref.eval_configs(R[:3])
    # the measurement adds in LDS in no fixed order, so its last bits differ from
    # call to call; a step that had not taken hold would be off by 1e-4
    for k in ("expo", "ER", "other"):
        assert np.max(np.abs(out[k] - want[k])) <= 1e-12 * np.max(np.abs(want[k]))
