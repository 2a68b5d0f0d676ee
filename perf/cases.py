"""The work that users of the engine have it do, as cases to be timed.

Three kinds of case, each through the public entry points of the `emtf` package:

* "engine": a batch of continuous tasks is advanced by some generations (`Engine.run`) and
  its individuals are read back ranked (`Engine.elites`) -- the whole population where every
  task has the same size, the elites that tasks hand to each other otherwise.
* "objective": the differentiable objective operator on a batch of points, forward or
  forward and backward.
* "cvrp": a batch of vehicle-routing instances is advanced by some generations and every
  instance's best tour is read.

The listed sizes are those of bench.py's workloads and of the tests' configurations.
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sg-emtf_amd"))

import emtf  # noqa: E402
from emtf import cvrp, objective, tasks  # noqa: E402

ALGOS = {"rand1": emtf.DE_RAND_1_BIN, "current1": emtf.DE_CURRENT_1_BIN, "ga": emtf.GA_SBX_PM}
FORMULAS = {"textbook": emtf.FORMULAS_TEXTBOOK, "reference_de": emtf.FORMULAS_REFERENCE_DE,
            "reference_ga": emtf.FORMULAS_REFERENCE_GA}
OPERATORS = ["sphere", "rosenbrock", "ackley", "rastrigin", "griewank", "weierstrass", "schwefel", "elliptic"]


def _engine(name, n, dim, pop, gens, **more):
    """An engine case: `n` tasks of dimension dim[0] .. dim[1] and population pop[0] .. pop[1]."""
    c = dict(kind="engine", tasks=n, dim_min=dim[0], dim_max=dim[1], pop_min=pop[0], pop_max=pop[1], gens=gens,
             algo="rand1", formulas="textbook", form="rotate", islands=1, exchange=0, migrate=0, interval=20,
             elites=4, polish=0)
    c.update(more)
    return dict(c, name=name) if name else c


def _objective(name, func, n, dim, grad, rotate=True):
    c = dict(kind="objective", func=func, n=n, dim=dim, grad=grad, rotate=rotate)
    return dict(c, name=name) if name else c


def _cvrp(name, n, nmin, nmax, pop, islands, gens):
    c = dict(kind="cvrp", instances=n, nmin=nmin, nmax=nmax, pop=pop, islands=islands, gens=gens)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a handful of tasks advanced by one transfer interval at a time: the CPU
        # configuration (8 unrotated tasks, 2 elites every 10 generations), where launches count
        _engine("de_8_tasks", 8, (50, 50), (64, 64), 10, form="shift", interval=10, elites=2),
        # the plain configuration, bench.py's default: one whole run of 2000 generations
        _engine("de_1024_tasks", 1024, (50, 50), (128, 128), 2000),
        # the reference's DE profile: its task generator, formulas and current/1 operator, with
        # islands that exchange and migrate, at an odd dimension and a ragged population
        _engine("de_islands_512_tasks", 512, (37, 37), (100, 100), 200, algo="current1", formulas="reference_de",
                form="diag", islands=4, exchange=10, migrate=5),
        # the reference's GA profile on the plain sizes
        _engine("ga_islands_1024_tasks", 1024, (50, 50), (128, 128), 400, algo="ga", formulas="reference_ga",
                form="diag", islands=4, exchange=10, migrate=5),
        # the batched uneven configuration: every kernel geometry at once
        _engine("de_uneven_4096_tasks", 4096, (10, 200), (32, 256), 100),
        # elites polished by the objectives' gradients at D = 100
        _engine("de_polish_1024_tasks", 1024, (100, 100), (128, 128), 200, polish=50),
        # a few points through the operator, forward and backward: an optimiser's inner step
        _objective("objective_grad_100x30", "rastrigin", 100, 30, True),
        # populations and samples scored in bulk
        _objective("objective_1Mx50", "ackley", 1 << 20, 50, False),
        _objective("objective_99991x200", "schwefel", 99991, 200, False),
        # a large batch of starts descended together
        _objective("objective_grad_250000x100", "griewank", 250000, 100, True),
        # a few routing instances, latency again, and bench.py's batch of 512
        _cvrp("cvrp_16_instances", 16, 50, 100, 64, 1, 10),
        _cvrp("cvrp_512_instances", 512, 50, 200, 128, 4, 100),
    ]


def _log_int(rng, lo, hi):
    return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))


# scalar operations of one individual's generation beside the rotation, per gene (for the
# size of a drawn case and work())
GENE_OPS = {"rand1": 40, "current1": 40, "ga": 150}


def _generation_flops(c):
    d = 0.5 * (c["dim_min"] + c["dim_max"])
    d2 = (c["dim_min"] ** 2 + c["dim_min"] * c["dim_max"] + c["dim_max"] ** 2) / 3.0
    p = 0.5 * (c["pop_min"] + c["pop_max"])
    return c["tasks"] * p * (2.0 * d2 + GENE_OPS[c["algo"]] * d)


def draw(rng):
    u = rng.random()
    if u < 0.5:
        algo = rng.choice(["rand1", "rand1", "current1", "ga"])
        form = rng.choice(["rotate", "rotate", "shift", "diag"])
        formulas = {"ga": "reference_ga"}.get(algo, "reference_de") if form == "diag" else "textbook"
        islands = rng.choice([1, 1, 2, 4])
        uneven = rng.random() < 0.3
        if uneven:
            d0 = rng.randint(2, 100)
            dim = (d0, rng.randint(d0, 256))
            pop = (32, 32 * rng.randint(2, 8))
        else:
            d0 = _log_int(rng, 2, 200)
            dim = (d0, d0)
            p0 = 2 * islands * max(2, _log_int(rng, 16, 512) // (2 * islands))
            pop = (p0, p0)
        polish = 0
        if not uneven and form != "diag" and dim[0] <= 100 and pop[0] <= 128 and rng.random() < 0.3:
            polish = rng.choice([10, 25])
        interval = rng.choice([0, 10, 20])
        c = _engine(None, _log_int(rng, 4, 2048), dim, pop, 1, algo=algo, formulas=formulas, form=form,
                    islands=islands, exchange=rng.choice([0, 10]) if islands > 1 else 0,
                    migrate=5 if islands > 1 else 0, interval=interval, elites=rng.randint(1, 4) if interval else 0,
                    polish=polish)
        top = max(1, min(1000, int(5.0e11 / _generation_flops(c))))
        c["gens"] = _log_int(rng, min(10, top), top)
        return c
    if u < 0.8:
        grad = rng.random() < 0.5
        dim = _log_int(rng, 2, 128 if grad else 256)
        top = min(1 << 20, int(4.0e7 / dim))
        return _objective(None, rng.choice(OPERATORS), _log_int(rng, 16, top), dim, grad, rng.random() < 0.8)
    nmin = rng.randint(10, 100)
    islands = rng.choice([1, 2, 4])
    return _cvrp(None, _log_int(rng, 4, 512), nmin, rng.randint(nmin, 200), 2 * islands * rng.randint(8, 16), islands,
                 _log_int(rng, 5, 100))


def _rotation(dim, gen):
    """A dense orthogonal matrix: four random reflections."""
    q = np.eye(dim)
    for v in gen.standard_normal((4, dim)):
        v /= np.linalg.norm(v)
        q -= np.outer(2.0 * (q @ v), v)
    return q.astype(np.float32)


def _tasks(c, seed):
    gen = np.random.Generator(np.random.PCG64(seed))
    if c["form"] == "diag":  # the reference's generator and boxes
        return [t for d, p in zip(*_sizes(c, gen))
                for t in tasks.reference_tasks(1, d, p, seed=int(gen.integers(1 << 30)))]
    out = []
    for t, (d, p) in enumerate(zip(*_sizes(c, gen))):
        task = dict(func=emtf.FUNC_IDS[tasks.CYCLE[t % 8]], dim=d, pop=p, lo=-100.0, hi=100.0, xform=emtf.SHIFT,
                    shift=gen.uniform(-80.0, 80.0, d).astype(np.float32))
        if c["form"] == "rotate":
            task.update(rot=_rotation(d, gen), xform=emtf.ROTATE)
        out.append(task)
    return out


def _sizes(c, gen):
    dims = gen.integers(c["dim_min"], c["dim_max"] + 1, c["tasks"])
    if c["pop_min"] == c["pop_max"]:
        pops = np.full(c["tasks"], c["pop_min"])
    else:
        pops = 32 * gen.integers(c["pop_min"] // 32, c["pop_max"] // 32 + 1, c["tasks"])
    return [int(d) for d in dims], [int(p) for p in pops]


def _points(case, seed):
    """The operator's inputs: points of the search box, an orthogonal matrix, a shift, an upstream gradient."""
    gen = torch.Generator("cuda").manual_seed(seed)
    n, dim = case["n"], case["dim"]
    x = torch.rand(n, dim, generator=gen, device="cuda") * 200.0 - 100.0
    shift = torch.rand(dim, generator=gen, device="cuda") * 160.0 - 80.0
    up = torch.rand(n, generator=gen, device="cuda") + 0.5
    rot = None
    if case["rotate"]:
        rot = torch.from_numpy(_rotation(dim, np.random.Generator(np.random.PCG64(seed)))).cuda()
    return x, rot, shift, up


def prepare(case, seed):
    if case["kind"] == "engine":
        params = dict(algo=ALGOS[case["algo"]], formulas=FORMULAS[case["formulas"]], n_islands=case["islands"],
                      exchange_interval=case["exchange"], migrate_interval=case["migrate"],
                      migrate_count=2 if case["migrate"] else 0, transfer_interval=case["interval"],
                      transfer_count=case["elites"], seed=seed)
        if case["polish"]:
            params.update(polish_interval=case["polish"], polish_steps=5, polish_topk=4)
        uniform = case["pop_min"] == case["pop_max"]
        return dict(kind="engine", engine=emtf.Engine(_tasks(case, seed), **params), gens=case["gens"],
                    rows=case["pop_max"] if uniform else 4)
    if case["kind"] == "objective":
        x, rot, shift, up = _points(case, seed)
        return dict(kind="objective", func=emtf.FUNC_IDS[case["func"]], x=x.requires_grad_(case["grad"]), rot=rot,
                    shift=shift, up=up if case["grad"] else None)
    # one instance of the largest size, the others between the bounds
    inst = cvrp.random_instances(1, seed=seed, nmin=case["nmax"], nmax=case["nmax"], pop=case["pop"])
    inst += cvrp.random_instances(case["instances"] - 1, seed=seed + 1, nmin=case["nmin"], nmax=case["nmax"],
                                  pop=case["pop"])
    engine = cvrp.CvrpEngine(inst, n_islands=case["islands"], migrate_interval=25 if case["islands"] > 1 else 0,
                             migrate_count=2 if case["islands"] > 1 else 0, seed=seed)
    return dict(kind="cvrp", engine=engine, gens=case["gens"])


def run(state):
    if state["kind"] == "engine":
        state["engine"].run(state["gens"])
        fitness, x = state["engine"].elites(state["rows"])
        return dict(fitness=fitness, x=x)
    if state["kind"] == "objective":
        f = objective.objective(state["func"], state["x"], state["rot"], state["shift"])
        if state["up"] is None:
            return dict(f=f)
        (gx,) = torch.autograd.grad(f, state["x"], state["up"])
        return dict(f=f, gx=gx)
    state["engine"].run(state["gens"])
    cost, tour = state["engine"].best()
    return dict(cost=cost, tour=tour)


def work(case):
    if case["kind"] == "engine":
        d = 0.5 * (case["dim_min"] + case["dim_max"])
        d2 = (case["dim_min"] ** 2 + case["dim_min"] * case["dim_max"] + case["dim_max"] ** 2) / 3.0
        p = 0.5 * (case["pop_min"] + case["pop_max"])
        rot = d2 if case["form"] == "rotate" else d
        # populations in and out, the transform, shift and table once
        return {"bytes": case["tasks"] * 4.0 * (2 * p * (d + 1) + rot + 2 * d),
                "flops": case["gens"] * _generation_flops(case)}
    if case["kind"] == "objective":
        n, dim = case["n"], case["dim"]
        gemm = 2.0 * n * dim * (dim if case["rotate"] else 1)
        if case["grad"]:  # x twice, f, the upstream gradient, gx; z again, then Q^T dz
            return {"bytes": 4.0 * n * (3 * dim + 2), "flops": 3 * gemm + 60.0 * n * dim}
        return {"bytes": 4.0 * n * (dim + 1), "flops": gemm + 20.0 * n * dim}
    n = 0.5 * (case["nmin"] + case["nmax"])
    # tours in and out; per gene and generation the crossover, the distance and the split's window
    return {"bytes": 2.0 * case["instances"] * case["pop"] * (n + 4),
            "flops": 60.0 * case["instances"] * case["pop"] * n * case["gens"]}


def _f64(func, z):
    """The textbook objectives of rows z in binary64 (Weierstrass without its constant, 0 at the optimum)."""
    dim = z.shape[1]
    j = torch.arange(dim, device=z.device, dtype=torch.float64)
    if func == "sphere":
        return (z * z).sum(1)
    if func == "rosenbrock":
        a, b = z[:, :-1], z[:, 1:]
        return (100.0 * (a * a - b) ** 2 + (a - 1.0) ** 2).sum(1)
    if func == "ackley":
        return (-20.0 * torch.exp(-0.2 * ((z * z).sum(1) / dim).sqrt())
                - torch.exp(torch.cos(2 * np.pi * z).sum(1) / dim) + 20.0 + np.e)
    if func == "rastrigin":
        return (z * z - 10.0 * torch.cos(2 * np.pi * z) + 10.0).sum(1)
    if func == "griewank":
        return 1.0 + (z * z).sum(1) / 4000.0 - torch.cos(z / (j + 1.0).sqrt()).prod(1)
    if func == "weierstrass":
        f = torch.zeros(z.shape[0], device=z.device, dtype=torch.float64)
        for k in range(21):
            f = f + 2.0 ** (1 - k) * torch.sin(np.pi * torch.remainder(3.0 ** k * z, 1.0)).square().sum(1)
        return f
    if func == "schwefel":
        return 418.9828872724338 * dim - (z * torch.sin(z.abs().sqrt())).sum(1)
    w = torch.pow(torch.tensor(1.0e6, device=z.device, dtype=torch.float64), j / (dim - 1)) if dim > 1 else j + 1.0
    return (w * z * z).sum(1)


def exact(case, seed):
    if case["kind"] != "objective":
        return None  # a population search and an integer search: no value in 64 bits
    x, rot, shift, up = _points(case, seed)
    f, gx = [], []
    for i in range(0, x.shape[0], 1 << 16):
        xi = x[i:i + (1 << 16)].double().requires_grad_(case["grad"])
        z = xi - shift.double()
        if rot is not None:
            z = z @ rot.double().T.contiguous()
        fi = _f64(case["func"], z)
        if case["grad"]:
            gx.append(torch.autograd.grad(fi, xi, up[i:i + (1 << 16)].double())[0])
        f.append(fi.detach())
    f = torch.cat(f)
    if not case["grad"]:
        return dict(f=f)
    # the derivative of Weierstrass's 3^20 term is below binary32's resolution of z
    return dict(f=f, gx=None if case["func"] == "weierstrass" else torch.cat(gx))
