"""Performance cases: the calls a user of the library makes, over the sizes it is used at.

Every case names one operation (`op`) on one system:

    step     one TDVP step from the captured graph, then the new parameters (Context.tdvp_step, get_params)
    batch    one TDVP step of a batch of trapped drops, then every system's parameters (Batch.tdvp_step)
    stage    one sampling stage left in device memory: a sweep, the measurement, S and F (tdvmc_sample_dev)
    measure  new walkers on the device, their measurement, S and F (tdvmc_set_walkers_dev, tdvmc_measure_dev)
    eval     ln psi, O and E_L of configurations in host memory (Context.eval_configs)
    grad     the same on device tensors, with every particle's gradient and Laplacian (tdvmc_eval_configs_dev)
    observe  g(r) and S(k) of the walkers (Context.additional_properties)
    adjoint  ln psi and its backward through torch.autograd (autograd.LogPsi)
    solve    the regularised TDVP system (Context.solve)

A case's `n` is the particle count (`batch`: the number of systems), `ps` and `k` the pair-spline and k-space
parameters, `w` the walkers or configurations, `ode` the step's ODE type.

Systems: `box` "periodic" (density 0.365 sigma^-3 Lennard-Jones helium in 3-D, density 1 with a Gaussian pair
potential in 1-D and 2-D) or "trap" (2-D harmonic trap, one-body factor, Gaussian repulsion).  `real_time` cases
carry imaginary parameters.  Every sweep is N moves per walker.
"""
import ctypes
import itertools
import math

import numpy as np
import torch

import tdvmc_amd as tdvmc
from tdvmc_amd import workloads

SIGMA, EPS, HBAR2_2M = workloads.SIGMA_HE, workloads.EPS_HE, workloads.HBAR2_2M_HE4
TRAP_CUTOFF = 6.0
SHELLS, BINS = 50, 200
MIXED, FP64 = "mixed", "fp64"


def _case(op, dim, n, ps, k, w, precision, box="periodic", real_time=False, ode=0):
    return {"op": op, "dim": dim, "n": n, "ps": ps, "k": k, "w": w, "precision": precision, "box": box,
            "real_time": real_time, "ode": ode}


def _named(name, case):
    return dict(case, name=name)


def listed():
    return [
        # the smallest system of the workloads: an Euler step is a dozen short kernels
        _named("step_1d_n20", _case("step", 1, 20, 16, 0, 1024, FP64)),
        # helium at a size that fits one pair tile, in the default precision
        _named("step_3d_n64", _case("step", 3, 64, 32, 0, 16384, FP64)),
        # the benchmark's RK4 step
        _named("step_3d_n343_k256", _case("step", 3, 343, 40, 256, 65536, MIXED, ode=2)),
        # the real-time quench, Euler: imaginary parameters, the largest parameter set and walker count
        _named("step_2d_n400_k512", _case("step", 2, 400, 48, 512, 131072, MIXED, real_time=True)),
        # the benchmark's sampling stage in the plain form, a quarter of its walkers
        _named("stage_3d_n343_k256", _case("stage", 3, 343, 40, 256, 16384, FP64)),
        # a small 2-D system with sizes that divide nothing
        _named("stage_2d_n25_k30", _case("stage", 2, 25, 12, 30, 4099, FP64, real_time=True)),
        # 64 trapped drops of 3 to 100 particles in one batch, RK4
        _named("batch_2d_trap64", _case("batch", 2, 64, 24, 0, 4096, MIXED, box="trap", ode=2)),
        # measurement of walkers that another program moved, with their S and F
        _named("measure_3d_n343_k256", _case("measure", 3, 343, 40, 256, 8192, MIXED)),
        # a handful of configurations in host memory, as a driver asks for them one at a time
        _named("eval_3d_n64", _case("eval", 3, 64, 32, 0, 16, FP64)),
        # every particle's drift and Laplacian, on the device
        _named("grad_3d_n125_k60", _case("grad", 3, 125, 24, 60, 4096, FP64)),
        # g(r) and S(k) of the walkers at the end of a run
        _named("observe_3d_n343", _case("observe", 3, 343, 40, 0, 16384, FP64)),
        # the linear system of the benchmark's step, from host memory
        _named("solve_p296", _case("solve", 3, 343, 40, 256, 4096, FP64)),
    ]


def draw(rng):
    """A case of the same ranges: sizes over their logarithm, at most about a twentieth of the largest listed case's
    work."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["step", "stage", "measure", "eval", "grad", "observe", "adjoint", "solve", "batch"])
    precision = rng.choice([FP64, FP64, MIXED])
    if op == "solve":
        return _case(op, 3, 343, log(8, 64), 2 * log(2, 250), 4096, FP64, real_time=rng.random() < 0.5)
    if op == "batch":
        return _case(op, 2, log(4, 64), log(8, 32), 0, log(64, 2048), precision, box="trap", ode=rng.choice([0, 2, 3]))
    box = "trap" if op in ("step", "stage", "measure", "eval") and rng.random() < 0.2 else "periodic"
    dim = 2 if box == "trap" else rng.choice([1, 2, 3, 3])
    n = log(3, 110) if box == "trap" else log(8, 400)
    k = 0 if box == "trap" or op == "observe" or rng.random() < 0.3 else log(4, 512)
    c = _case(op, dim, n, log(8, 48), k, 1, precision, box, real_time=rng.random() < 0.3 and op not in ("adjoint", "observe"),
              ode=rng.choice([0, 2]) if op == "step" else 0)
    most = {"eval": 2048, "adjoint": 512, "grad": 8192}.get(op, 65536)
    c["w"] = log(1 if op in ("eval", "adjoint") else 32, most)
    limit = work(listed()[3])["flops"] / 20
    while work(c)["flops"] * (4 if precision == FP64 else 1) > limit and c["w"] > 1:
        c["w"] //= 2
    return c


# ------------------------------------------------------------------ systems

def _length(case):
    if case["box"] == "trap":
        return 0.0
    if case["dim"] == 3:
        return (case["n"] / 0.365) ** (1.0 / 3.0) * SIGMA
    return float(case["n"]) ** (1.0 / case["dim"])


def _cutoff(case):
    return TRAP_CUTOFF if case["box"] == "trap" else _length(case) / 2.0


def _potential(case):
    """(type, first, second parameter): Lennard-Jones (sigma, eps), Gaussian (width, height)."""
    if case["box"] == "trap":
        return "GAUSSIAN", 0.5, 2.0
    return {1: ("GAUSSIAN", 1.0, 1.0), 2: ("GAUSSIAN", 0.2, 5.0), 3: ("LJ", SIGMA, EPS)}[case["dim"]]


def _hbar2_2m(case):
    return HBAR2_2M if case["dim"] == 3 and case["box"] == "periodic" else 0.5


def _parameters(case, seed):
    """Real and imaginary parameters: [one-body][pair spline][k-space]."""
    g = np.random.default_rng([int(seed), 7])
    ps, k, one = case["ps"], case["k"], int(case["box"] == "trap")
    if case["dim"] == 3 and case["box"] == "periodic":
        pair = workloads.mcmillan_params(ps, _cutoff(case), 1.1 * SIGMA, 0.6 * SIGMA) * g.uniform(0.97, 1.03)
    else:
        pair = g.normal(0.0, 0.05, ps)
        pair[-1] = 0.0
    re = np.concatenate([[1.0 / (2.0 * g.uniform(0.8, 1.2) ** 2)] * one, pair, g.normal(0.0, 1e-3 / case["dim"], k)])
    im = np.zeros_like(re)
    if case["real_time"]:
        im = np.concatenate([g.normal(0.0, 0.01, one + ps), g.normal(0.0, 1e-4, k)])
    return re, im


def _config(case, seed):
    kind, a, b = _potential(case)
    re, im = _parameters(case, seed)
    cfg = {"CONFIG_VERSION": "0.24", "SYSTEM_TYPE": "BosonsBulk", "N": case["n"], "DIM": case["dim"], "LBOX": _length(case),
           "N_PARAM": case["ps"], "K_VECTORS": case["k"], "HBAR2_2M": _hbar2_2m(case), "PAIR_POTENTIAL": kind,
           "SYSTEM_PARAMS": [a, b], "PARAMS_REAL": re.tolist(), "PARAMS_IMAGINARY": im.tolist(),
           "MC_STEP": 0.3 * SIGMA if kind == "LJ" else (0.5 if case["dim"] < 2 or case["box"] == "trap" else 0.3),
           "MC_NTHERMSTEPS": case["n"], "SAMPLES_PER_WALKER": 1, "N_WALKERS": 1, "TIMESTEP": 1e-4, "SEED": 1 + seed % 1000003,
           "IMAGINARY_TIME": 0 if case["real_time"] else 1, "ODE_SOLVER_TYPE": case["ode"], "LINEAR_EQUATION_SOLVER_TYPE": 0,
           "GR_BIN_COUNT": BINS, "PRECISION": "MIXED" if case["precision"] == MIXED else "FP64"}
    if case["box"] == "trap":
        cfg.update(SYSTEM_TYPE="BosonsTrap", ONE_BODY=1, TRAP_OMEGA=1.0, SPLINE_CUTOFF=TRAP_CUTOFF)
    return cfg


def _walkers(case, seed, w=None, n=None):
    """[W][N][DIM] on the GPU: a lattice shaken by an eighth of its spacing in a box (hard cores: a sixteenth), a
    Gaussian cloud in a trap."""
    w, n, dim = w or case["w"], n or case["n"], case["dim"]
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 31 + 5)
    noise = torch.randn((w, n, dim), generator=g, dtype=torch.float64, device="cuda")
    if case["box"] == "trap":
        return noise * math.sqrt(0.5)
    length, side = _length(case), 1
    while side ** dim < n:
        side += 1
    spacing = length / side
    site = torch.arange(n, device="cuda") * side ** dim // n  # the n particles spread over all sites
    grid = torch.stack([site // side ** (dim - 1 - a) % side for a in range(dim)], dim=1).to(torch.float64)
    return (grid + 0.5) * spacing - length / 2.0 + noise.clamp_(-2.5, 2.5).mul_(spacing / (16.0 if dim == 3 else 8.0))


def _context(case, seed):
    ctx = tdvmc.Context(_config(case, seed))
    if case["op"] in ("step", "stage", "measure", "observe"):
        ctx.set_walker_count(case["w"])
    return ctx


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _ok(code):
    if code != tdvmc.OK:
        raise RuntimeError("tdvmc error %d" % code)


def _set_walkers(state):
    _ok(tdvmc.lib().tdvmc_set_walkers_dev(state["ctx"]._h, _ptr(state["R"]), state["R"].shape[0],
                                          ctypes.c_void_p(state["stream"].cuda_stream)))


def _samples(case, seed):
    """Moments as a stage leaves them: correlated operators of different scales, an energy correlated with them."""
    g = np.random.default_rng([int(seed), 11])
    p = case["ps"] + case["k"]
    x = g.normal(size=(case["w"], p))
    for i in range(1, p):
        x[:, i] = 0.7 * x[:, i - 1] + 0.714 * x[:, i]
    x = x * g.uniform(1.0, 20.0, p) + g.uniform(0.0, 200.0, p)
    er = -5.0 * case["n"] + x @ g.normal(0.0, 0.05, p) + g.normal(0.0, 10.0, case["w"])
    ei = x @ g.normal(0.0, 0.01, p) + g.normal(0.0, 1.0, case["w"])
    xc = x - x.mean(0)
    n = float(case["w"])
    return {"mO": x.mean(0), "mE": np.array([er.mean(), ei.mean()]), "S": xc.T @ xc / n,
            "FR": xc.T @ (er - er.mean()) / n, "FI": xc.T @ (ei - ei.mean()) / n}


def prepare(case, seed):
    op, state = case["op"], {"case": case}
    if op == "batch":
        return _prepare_batch(case, seed, state)
    state["ctx"] = ctx = _context(case, seed)
    state["stream"] = torch.cuda.Stream()
    if op == "solve":
        state["moments"] = _samples(case, seed)
        return state
    R = _walkers(case, seed)
    p, w, n, dim = ctx.P, case["w"], case["n"], case["dim"]
    if op in ("step", "stage", "measure", "observe"):
        state["R"] = R
        torch.cuda.synchronize()
        _set_walkers(state)
        torch.cuda.synchronize()
    dev = {"dtype": torch.float64, "device": "cuda"}
    if op in ("stage", "measure"):
        state["out"] = {"mean": torch.empty(p + 2, **dev), "S": torch.empty((p, p), **dev), "F": torch.empty((2, p), **dev)}
        state["seed"] = 1 + int(seed) % 1000003
    elif op == "grad":
        state["R"] = R
        state["out"] = {"expo": torch.empty(w, **dev), "ER": torch.empty(w, **dev), "EI": torch.empty(w, **dev),
                        "O": torch.empty((w, p), **dev), "grad": torch.empty((w, n, dim, 2), **dev), "lap": torch.empty((w, n, 2), **dev)}
    elif op == "eval":
        state["R"] = R.cpu().numpy()
    elif op == "adjoint":
        from tdvmc_amd.autograd import LogPsi
        state["fn"] = LogPsi
        state["R"] = R.cpu().requires_grad_(True)
        state["u"] = torch.tensor(_parameters(case, seed)[0], requires_grad=True)
        state["gbar"] = _gbar(case, seed)
    return state


def _gbar(case, seed):
    return torch.from_numpy(np.random.default_rng([int(seed), 13]).normal(0.0, 1.0 / case["w"], case["w"]))


def _prepare_batch(case, seed, state):
    cfgs = workloads.trap2d_batch64(W=1, n_systems=case["n"], seed_w=6 + int(seed) % 1000003)
    for c in cfgs:
        knots = np.linspace(0.0, 1.0, case["ps"])
        pair = np.interp(knots, np.linspace(0.0, 1.0, c["N_PARAM"]), c["PARAMS_REAL"][1:])
        c.update(N_PARAM=case["ps"], PARAMS_REAL=[c["PARAMS_REAL"][0], *pair.tolist()], ODE_SOLVER_TYPE=case["ode"], TIMESTEP=1e-4,
                 PRECISION="MIXED" if case["precision"] == MIXED else "FP64")
    state["batch"] = batch = tdvmc.Batch(cfgs)
    state["stream"] = torch.cuda.Stream()
    for i, ctx in enumerate(batch.systems):
        ctx.set_walker_count(case["w"])
        R = _walkers(case, seed + 1000 * i, n=ctx.N)
        torch.cuda.synchronize()
        _set_walkers({"ctx": ctx, "R": R, "stream": state["stream"]})
        torch.cuda.synchronize()
    return state


def run(state):
    case = state["case"]
    op, prec = case["op"], tdvmc.MIXED if case["precision"] == MIXED else tdvmc.FP64
    if op == "batch":
        state["batch"].tdvp_step(1e-4, case["ode"], prec, use_graph=True)
        params = [c.get_params() for c in state["batch"].systems]
        return [np.concatenate([p[i] for p in params]) for i in (0, 1)] + [np.array([p[2:] for p in params])]
    ctx, L = state["ctx"], tdvmc.lib()
    stream = ctypes.c_void_p(state["stream"].cuda_stream)
    if op == "step":
        ctx.tdvp_step(1e-4, case["ode"], prec, use_graph=True)
        return ctx.get_params()
    if op == "stage":
        o = state["out"]
        _ok(L.tdvmc_sample_dev(ctx._h, state["seed"], prec, _ptr(o["mean"]), _ptr(o["S"]), _ptr(o["F"]), stream))
        _ok(L.tdvmc_get_walkers_dev(ctx._h, _ptr(state["R"]), case["w"], stream))
        return dict(o, R=state["R"])
    if op == "measure":
        o = state["out"]
        _set_walkers(state)
        _ok(L.tdvmc_measure_dev(ctx._h, prec, _ptr(o["mean"]), _ptr(o["S"]), _ptr(o["F"]), stream))
        return o
    if op == "eval":
        return ctx.eval_configs(state["R"], precision=prec)
    if op == "grad":
        o = state["out"]
        _ok(L.tdvmc_eval_configs_dev(ctx._h, _ptr(state["R"]), case["w"], prec, _ptr(o["expo"]), _ptr(o["ER"]), _ptr(o["EI"]),
                                     _ptr(o["O"]), _ptr(o["grad"]), _ptr(o["lap"]), stream))
        return o
    if op == "observe":
        gr, sk = ctx.additional_properties(seed=1, n_samples=1, precision=prec)
        return {"gr": gr, "sk": sk}
    if op == "adjoint":
        R, u = state["R"], state["u"]
        R.grad = u.grad = None
        value = state["fn"].apply(ctx, R, u, prec)
        value.backward(state["gbar"])
        return {"value": value.detach(), "dR": R.grad, "du": u.grad}
    m = state["moments"]
    return ctx.solve(m["mO"], m["mE"], m["S"], m["FR"], m["FI"], imag_time=0 if case["real_time"] else 1, eps=1e-3)


# ------------------------------------------------------------------ the least work of one pass

def _pairs(n):
    return n * (n - 1) / 2.0


def _move_flops(n, dim, k):
    return 2.0 * (n - 1) * (4 * dim + 9) + 2.0 * k * (2 * dim + 8) + 10


def _measure_flops(n, dim, k):
    return _pairs(n) * (8 * dim + 29) + n * k * (2.0 * dim + 12) + n * (4 * dim + 2)


def _solve_flops(p):
    return p ** 3 / 3.0 + 4.0 * p * p


def work(case):
    op, dim, n, w = case["op"], case["dim"], case["n"], case["w"]
    p = case["ps"] + case["k"] + int(case["box"] == "trap")
    stages = 4 if case["ode"] == 2 else 1
    if op == "batch":
        flops = by = 0.0
        for c in workloads.trap2d_batch64(W=1, n_systems=case["n"]):
            m = c["N"]
            sweeps = 4 if case["ode"] == 2 else 1
            flops += w * (sweeps * m * _move_flops(m, 2, 0) + (4 if case["ode"] in (2, 3) else 1) * (_measure_flops(m, 2, 0) + p * (p + 1.0)))
            by += w * m * 2 * 8.0 * 2
        return {"flops": flops, "bytes": by}
    if op == "solve":
        return {"flops": _solve_flops(p), "bytes": 8.0 * (p * p + 6.0 * p)}
    flops, by = w * _measure_flops(n, dim, case["k"]), 8.0 * w * n * dim
    if op in ("step", "stage"):
        flops = stages * (flops + w * (n * _move_flops(n, dim, case["k"]) + p * (p + 1.0) + 6.0 * p))
        by = 2 * by + 8.0 * (p * p + 3.0 * p)
        if op == "step":
            flops += stages * _solve_flops(p)
    elif op == "measure":
        flops += w * (p * (p + 1.0) + 6.0 * p)
        by += 8.0 * (p * p + 3.0 * p)
    elif op in ("eval", "grad"):
        by += 8.0 * w * (p + (12 if op == "eval" else 3 + n * (2 * dim + 2)))
    elif op == "observe":
        vectors = _shells(dim)[0].shape[0]
        flops = w * (_pairs(n) * (5 * dim + 2) + n * vectors * (2.0 * dim + 3))
        by += 8.0 * (BINS + SHELLS)
    elif op == "adjoint":
        flops, by = 2 * flops, 2 * by + 8.0 * w * (n * dim + 2) + 16.0 * p
    return {"flops": flops, "bytes": by}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch

def _lattice(dim, k):
    """The k shortest non-zero integer vectors, by length, then component by component."""
    m = 1
    while k:
        v = sorted((v for v in itertools.product(range(-m, m + 1), repeat=dim) if any(v)), key=lambda v: (sum(x * x for x in v), v))
        if len(v) >= k and sum(x * x for x in v[k - 1]) < (m + 1) ** 2:
            return np.array(v[:k], dtype=np.float64)
        m += 1
    return np.zeros((0, dim))


def _shells(dim):
    """Vectors with non-negative components in the first SHELLS shells, and each one's shell."""
    top = 60 if dim > 1 else SHELLS ** 2
    limit = math.isqrt(top) + 2
    every = {}
    for v in itertools.product(range(limit), repeat=dim):
        every.setdefault(sum(x * x for x in v), []).append(v)
    every.pop(0)
    while True:
        keys = sorted(q for q in every if q < limit * limit)
        if len(keys) >= SHELLS:
            break
        limit *= 2
        every = {}
        for v in itertools.product(range(limit), repeat=dim):
            every.setdefault(sum(x * x for x in v), []).append(v)
        every.pop(0)
    vectors = [v for q in keys[:SHELLS] for v in every[q]]
    shell = [i for i, q in enumerate(keys[:SHELLS]) for _ in every[q]]
    return np.array(vectors, dtype=np.float64), np.array(shell)


_PIECES = ((1 / 6, -3 / 6, 3 / 6, -1 / 6), (4 / 6, 0.0, -6 / 6, 3 / 6), (1 / 6, 3 / 6, 3 / 6, -3 / 6), (0.0, 0.0, 0.0, 1 / 6))


def _fold(B, ps):
    """Basis sums B_0 .. B_{ps+1} to the operators of a spline with zero slope at both ends."""
    o = B[:, 1:ps + 1].clone()
    o[:, 0] = B[:, 1]
    o[:, 1] = B[:, 0] + B[:, 2]
    o[:, ps - 2] = o[:, ps - 2] + B[:, ps + 1]
    return o


def _coefficients(u, ps):
    return torch.stack([u[1], u[0], *u[1:ps], u[ps - 2]])


def _evaluate(case, R, re, im):
    """expo, ER, EI, O, other, gradient and Laplacian of the configurations R."""
    w, n, dim = R.shape
    length, rc, ps, one = _length(case), _cutoff(case), case["ps"], int(case["box"] == "trap")
    hinv = (ps - 1) / rc
    kind, pa, pb = _potential(case)
    re, im = (torch.as_tensor(x, device=R.device) for x in (re, im))
    d = R[:, :, None, :] - R[:, None, :, :]
    if length:
        d = d - length * torch.round(d / length)
    r = d.square().sum(-1).sqrt()
    upper = torch.ones((n, n), dtype=torch.bool, device=R.device).triu(1)
    off = ~torch.eye(n, dtype=torch.bool, device=R.device)
    inside = (r <= rc) & off
    safe = torch.where(off, r, 1.0)
    x = (safe * hinv).clamp(max=ps - 1.0)
    j = x.floor().clamp(max=ps - 2).long()
    t = x - j
    grad, lap = [], []
    for u in (re[one:one + ps], im[one:one + ps]):
        c = _coefficients(u, ps)
        du = d2u = 0.0
        for m, (_, b, e, f) in enumerate(_PIECES):
            cm = c[j + m]
            du = du + cm * (b + t * (2 * e + t * 3 * f)) * hinv
            d2u = d2u + cm * (2 * e + t * 6 * f) * hinv * hinv
        du = torch.where(inside, du / safe, 0.0)
        grad.append(torch.einsum("wij,wija->wia", du, d))
        lap.append(torch.where(inside, d2u, 0.0).sum(-1) + (dim - 1) * du.sum(-1))
    B = torch.zeros((w, ps + 2), dtype=R.dtype, device=R.device)
    pair = inside & upper
    for m, (a, b, e, f) in enumerate(_PIECES):
        v = torch.where(pair, a + t * (b + t * (e + t * f)), 0.0)
        B.scatter_add_(1, (j + m).reshape(w, -1), v.reshape(w, -1))
    outer = (upper & ~inside).sum((1, 2)).to(R.dtype)
    O = [_fold(B, ps)]
    expo = O[0] @ re[one:one + ps] + re[one + ps - 1] * outer
    if kind == "LJ":
        q = (pa / safe) ** 6
        v = 4.0 * pb * (q * q - q)
    else:
        v = pb * torch.exp(-0.5 * (safe / pa) ** 2)
    pot = torch.where(pair if length else upper, v, 0.0).sum((1, 2))
    if one:
        r2 = R.square().sum((1, 2))
        O.insert(0, -r2[:, None])
        expo = expo - re[0] * r2
        for i, u in enumerate((re[0], im[0])):
            grad[i] = grad[i] - 2.0 * u * R
            lap[i] = lap[i] - 2.0 * dim * u
    vext = 0.5 * R.square().sum((1, 2)) if one else 0.0
    if case["k"]:
        kv = torch.as_tensor(_lattice(dim, case["k"]) * (2.0 * math.pi / length), device=R.device)
        e = torch.polar(torch.ones((), dtype=R.dtype, device=R.device), R @ kv.T)
        rho = e.sum(1)
        ok = rho.real.square() + rho.imag.square()
        O.append(ok)
        expo = expo + ok @ re[one + ps:]
        z = e * rho.conj()[:, None, :]
        k2 = kv.square().sum(1)
        for i, u in enumerate((re[one + ps:], im[one + ps:])):
            grad[i] = grad[i] - 2.0 * (z.imag * u) @ kv
            lap[i] = lap[i] + 2.0 * ((1.0 - z.real) * (u * k2)).sum(-1)
    sums = [grad[0].square().sum((1, 2)), grad[1].square().sum((1, 2)), lap[0].sum(1), lap[1].sum(1), 2.0 * (grad[0] * grad[1]).sum((1, 2))]
    hb = _hbar2_2m(case)
    kin, ei = -hb * (sums[0] - sums[1] + sums[2]), -hb * (sums[4] + sums[3])
    other = torch.stack([kin, pot, torch.exp(expo), expo, *sums], dim=1)
    return {"expo": expo, "ER": kin + pot + vext, "EI": ei, "O": torch.cat(O, dim=1), "other": other, "grad": torch.stack(grad, dim=-1),
            "lap": torch.stack(lap, dim=-1), "outer": outer}


def _evaluate_all(case, R, re, im, keep):
    per = case["n"] * (case["n"] * (case["dim"] + 8) + 4 * case["k"])
    chunk = max(1, 200_000_000 // (8 * per) * 4)
    got = [{k: v for k, v in _evaluate(case, R[i:i + chunk], re, im).items() if k in keep} for i in range(0, R.shape[0], chunk)]
    return {k: torch.cat([g[k] for g in got]) for k in keep}


def exact(case, seed):
    op, w, n, dim = case["op"], case["w"], case["n"], case["dim"]
    if op in ("step", "stage", "batch"):
        return None  # Metropolis moves: what they return depends on every accept decision
    if op == "solve":
        m = _samples(case, seed)
        if case["real_time"]:
            b = np.stack([m["FI"], -m["FR"]], 1)
        else:
            b = np.stack([-m["FR"], -(m["FI"] + m["mO"] * m["mE"][1])], 1)
        x = np.linalg.solve(m["S"] + 1e-3 * np.eye(len(b)), b)
        phi = -(m["mO"] @ x)
        phi[1 if case["real_time"] else 0] -= m["mE"][0]
        return {"xR": x[:, 0].copy(), "xI": x[:, 1].copy(), "phiDotR": phi[0], "phiDotI": phi[1], "bad": 0}
    R = _walkers(case, seed)
    re, im = _parameters(case, seed)
    if op == "observe":
        return _observe(case, R)
    if op == "measure":
        e = _evaluate_all(case, R, re, im, ("O", "ER", "EI"))
        x = torch.cat([e["O"], e["ER"][:, None], e["EI"][:, None]], 1)
        mean = x.mean(0)
        x = x - mean
        p = e["O"].shape[1]
        cov = x.T @ x / w
        return {"mean": mean, "S": cov[:p, :p].contiguous(), "F": cov[p:, :p].contiguous()}
    if op == "eval":
        return _evaluate_all(case, R, re, im, ("expo", "ER", "EI", "O", "other"))
    if op == "grad":
        return _evaluate_all(case, R, re, im, ("expo", "ER", "EI", "O", "grad", "lap"))
    e = _evaluate_all(case, R, re, im, ("expo", "O", "grad", "outer"))
    gbar = _gbar(case, seed).cuda()
    du = gbar @ e["O"]
    du[case["ps"] - 1] += gbar @ e["outer"]
    return {"value": e["expo"], "dR": gbar[:, None, None] * e["grad"][..., 0], "du": du}


def _observe(case, R):
    w, n, dim = R.shape
    length, rc = _length(case), _cutoff(case)
    spacing = rc / BINS
    counts = torch.zeros(BINS, dtype=torch.float64, device=R.device)
    vectors, shell = _shells(dim)
    kv = torch.as_tensor(vectors * (2.0 * math.pi / length), device=R.device)
    shell = torch.as_tensor(shell, device=R.device)
    size = torch.bincount(shell, minlength=SHELLS).to(R.dtype)
    sk = torch.zeros(SHELLS, dtype=torch.float64, device=R.device)
    i, j = torch.triu_indices(n, n, 1, device=R.device)
    chunk = max(1, 25_000_000 // (n * n + n * len(vectors)))
    for a in range(0, w, chunk):
        x = R[a:a + chunk]
        d = x[:, i] - x[:, j]
        d = d - length * torch.round(d / length)
        r = d.square().sum(-1).sqrt()
        counts += torch.bincount((r[r < rc] / spacing).floor().long(), minlength=BINS)[:BINS]
        ph = x @ kv.T
        s = torch.zeros((2, x.shape[0], SHELLS), dtype=x.dtype, device=x.device)
        s[0].index_add_(1, shell, torch.cos(ph).sum(1))
        s[1].index_add_(1, shell, torch.sin(ph).sum(1))
        sk += ((s[0] ** 2 + s[1] ** 2) / (n * size)).sum(0)
    edge = torch.arange(BINS + 1, dtype=torch.float64, device=R.device) * spacing
    volume = {1: edge, 2: math.pi * edge ** 2, 3: 4.0 * math.pi / 3.0 * edge ** 3}[dim].diff()
    return {"gr": counts * (dim / (n - 1.0)) / volume / w, "sk": sk / w}
