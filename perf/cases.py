"""The work a user of this library has it do, as cases that can be timed.

A case is one pass through the public entry points: a force evaluation at
positions that the caller brings (``set_state`` and ``forces``), a stretch of
leapfrog steps with the state read back at its end (``step`` and ``state``,
one system or an ensemble, launched or captured), the gradient of a
trajectory through the autograd function, the O(N^2) solver, and the FP64
direct sum at chosen particles that accuracy is checked with.

The inputs are Plummer spheres, uniform cubes, pairs of spheres and ensembles
of spheres, made from the seed; their sizes and options are those of the
benchmark's workloads (N = 4096 uniform, 16384 and 1,048,576 Plummer, the
theta = 0.4, p = 6 pair, the ensemble of 512-particle and larger systems) and
of the tests, with odd sizes beside them.
"""
import math

import numpy as np
import torch

import nbody_amd as nb
from nbody_amd.adjoint import trajectory_function


def _case(name, kind, n, **opt):
    c = dict(kind=kind, n=n, ic="plummer", order=4, theta=0.5, eps=1e-2, cap=16, chunk=0, dt=1e-3, steps=1,
             nsys=1, graph=0, targets=0)
    c.update(opt)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: the default leaf capacity, a field of a few
        # hundred particles evaluated for a program with its own integrator
        _case("forces_uniform777", "forces", 777, ic="uniform", cap=8),
        # the small benchmark workload: 4096 uniform, capacity 16
        _case("forces_uniform4096", "forces", 4096, ic="uniform"),
        # an odd middle size at a higher order
        _case("forces_plummer30011_p5", "forces", 30011, order=5, cap=24),
        # the headline's options at a size whose answer can be checked whole
        _case("forces_plummer262144", "forces", 262144, eps=1e-3, cap=32),
        # a small simulation stepped between two frames
        _case("steps_plummer5003", "steps", 5003, steps=5),
        # the same with captured steps, the option made for small systems
        _case("steps_plummer5003_graph", "steps", 5003, steps=5, graph=1),
        # the headline: Plummer, N = 1,048,576, ten steps and the state
        _case("steps_plummer1048576", "steps", 1048576, eps=1e-3, cap=32, chunk=128, steps=10),
        # two spheres about to meet, theta = 0.4 and order 6
        _case("steps_pair300002_p6", "steps", 300002, ic="pair", order=6, theta=0.4, eps=5e-4, cap=32, dt=5e-4,
              steps=2),
        # many uneven systems in one handle, with the capacity and tile the
        # autotuner picks for them
        _case("steps_ensemble64", "steps", 65536, nsys=64, cap=64, chunk=128, steps=5),
        # the gradient of a trajectory in a training loop
        _case("gradient_plummer16384", "gradient", 16384, steps=20),
        # the O(N^2) solver, the stand-in for the naive simulation
        _case("direct_plummer16384", "direct", 16384, steps=2),
        # the FP64 sums that a force error is measured against
        _case("check_fp64_262144", "check", 262144, eps=1e-3, cap=32, targets=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forces", "forces", "forces", "steps", "steps", "steps", "ensemble", "gradient", "direct",
                       "check"])
    cap = rng.choice([8, 16, 24, 32, 48, 64])
    chunk = rng.choice([0, 64, 128])
    eps = rng.choice([1e-2, 1e-3])
    if kind == "forces":
        return _case(None, kind, _log_int(rng, 500, 400000), ic=rng.choice(["plummer", "plummer", "uniform", "pair"]),
                     order=rng.choice([3, 4, 4, 5]), cap=cap, chunk=chunk, eps=eps)
    if kind == "steps":
        return _case(None, kind, _log_int(rng, 2000, 700000), ic=rng.choice(["plummer", "plummer", "pair"]),
                     order=rng.choice([3, 4, 4]), cap=cap, chunk=chunk, eps=eps, steps=rng.randint(1, 5),
                     graph=rng.choice([0, 0, 1]))
    if kind == "ensemble":
        # n: the largest system of the ensemble
        return _case(None, "steps", _log_int(rng, 2000, 32768), nsys=rng.randint(3, 96), cap=cap, chunk=chunk,
                     steps=rng.randint(1, 5))
    if kind == "gradient":
        return _case(None, kind, _log_int(rng, 1000, 20000), cap=rng.choice([16, 24, 32]), steps=rng.randint(4, 20))
    if kind == "direct":
        return _case(None, kind, _log_int(rng, 300, 30000), steps=rng.randint(1, 4), eps=eps)
    return _case(None, "check", _log_int(rng, 2000, 400000), eps=eps, cap=32, targets=_log_int(rng, 64, 8192))


# ---- inputs ------------------------------------------------------------------
def _plummer(rng, n):
    """Plummer sphere of scale and total mass 1 truncated at r = 20: radii from
    the cumulative mass, speeds by rejection from q^2 (1 - q^2)^(7/2)."""
    def directions(k):
        u = rng.standard_normal((k, 3))
        return u / np.linalg.norm(u, axis=1, keepdims=True)

    frac = rng.uniform(1e-10, (1.0 + 1.0 / 400.0) ** -1.5, n)
    r = 1.0 / np.sqrt(frac ** (-2.0 / 3.0) - 1.0)
    q = np.empty(0)
    while len(q) < n:
        a, b = rng.uniform(0.0, 1.0, 2 * n + 64), rng.uniform(0.0, 0.1, 2 * n + 64)
        q = np.concatenate([q, a[b < a * a * (1.0 - a * a) ** 3.5]])
    speed = q[:n] * math.sqrt(2.0) * (1.0 + r * r) ** -0.25
    return r[:, None] * directions(n), speed[:, None] * directions(n), np.full(n, 1.0 / n)


def _inputs(case, seed):
    """(positions, velocities, masses, system offsets or None), float64."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    if case["nsys"] > 1:
        # log-uniform sizes from 512 to n; the sizes belong to the case, so
        # that other inputs are the same amount of work
        sizes = np.random.default_rng(n + case["nsys"]).uniform(math.log(512), math.log(n), case["nsys"])
        sizes = np.exp(sizes).astype(np.int64)
        parts = [_plummer(rng, int(k)) for k in sizes]
        off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint32)
        return tuple(np.concatenate([p[i] for p in parts]) for i in range(3)) + (off,)
    if case["ic"] == "uniform":
        return rng.uniform(0.0, 1.0, (n, 3)), np.zeros((n, 3)), np.full(n, 1.0 / n), None
    if case["ic"] == "pair":
        (xa, va, ma), (xb, vb, mb) = _plummer(rng, n - n // 2), _plummer(rng, n // 2)
        shift, drift = np.array([5.0, 0.0, 0.0]), np.array([0.3, 0.0, 0.0])
        return np.concatenate([xa - shift, xb + shift]), np.concatenate([va + drift, vb - drift]), \
            np.concatenate([ma, mb]), None
    return _plummer(rng, n) + (None,)


def _targets(case, seed):
    k = min(case["targets"], case["n"])
    return np.sort(np.random.default_rng(seed + 1).choice(case["n"], size=k, replace=False))


def _config(case):
    return nb.default_config(
        G=1.0, eps=case["eps"], theta=case["theta"], dt=case["dt"], leaf_capacity=case["cap"], order=case["order"],
        m2l_order=case["order"] if case["order"] == 6 else 0, p2p_chunk=case["chunk"], graph=case["graph"],
        solver=nb.SOLVER_DIRECT if case["kind"] == "direct" else nb.SOLVER_FMM)


def _gradient_inputs(case, seed):
    """Initial state and masses as float32 parameters, and a target snapshot."""
    x, v, m, _ = _inputs(case, seed)
    noise = np.random.default_rng(seed + 1).standard_normal(x.shape)
    goal = x + case["steps"] * case["dt"] * (v + 1e-3 * noise)
    return [torch.tensor(a, dtype=torch.float32, device="cuda") for a in (x, v, m, goal)]


def prepare(case, seed):
    if case["kind"] == "gradient":
        x, v, m, goal = _gradient_inputs(case, seed)
        return {"case": case, "apply": trajectory_function().apply, "config": _config(case), "goal": goal,
                "leaves": [t.requires_grad_() for t in (x, v, m)]}
    x, v, m, off = _inputs(case, seed)
    sim = nb.HipSimulation.from_arrays(x, v, m, m, config=_config(case), sys_off=off)
    state = {"case": case, "sim": sim}
    if case["kind"] == "forces":
        state["x"], state["v"] = x, v
    if case["kind"] == "check":
        state["targets"] = _targets(case, seed)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "gradient":
        x, v, m = state["leaves"]
        xn, vn = state["apply"](x, v, m, case["steps"], 10, state["config"])
        loss = (xn - state["goal"]).square().mean() + 0.1 * vn.square().mean()
        return [xn, vn, *torch.autograd.grad(loss, (x, v, m))]
    sim = state["sim"]
    if case["kind"] == "forces":
        sim.set_state(state["x"], state["v"])
        return list(sim.forces())
    if case["kind"] == "check":
        return list(sim.direct_fp64(state["targets"]))
    sim.step(case["steps"])
    return list(sim.state())


# ---- what a pass cannot do without ---------------------------------------------
def _evaluation_flops(case, n):
    """Near and far field of n particles in trees of leaf capacity cap: about
    70 cap neighbours a particle, 4 / cap cells a particle and 1000 accepted
    cells a cell at theta = 0.5, each a product over the kept terms."""
    p = case["order"]
    near = (0.5 / case["theta"]) ** 3
    sources = min(n, 70.0 * case["cap"] * near)
    cells = 4.0 * n / case["cap"]
    count = [(d + 1) * (d + 2) // 2 for d in range(p + 1)]
    q = p if p == 6 else p + 1
    terms = sum(count[a] * count[b] for a in range(p + 1) for b in range(p + 1) if a + b <= q)
    return n * sources * 20.0 + cells * min(cells, 1000.0 * near) * 2.0 * terms


def work(case):
    n, k = case["n"], case["kind"]
    if case["nsys"] > 1:
        mean = (case["n"] - 512.0) / math.log(case["n"] / 512.0)
        return {"bytes": case["nsys"] * mean * (128.0 + 96.0 * case["steps"]),
                "flops": case["nsys"] * case["steps"] * _evaluation_flops(case, mean)}
    if k == "check":
        return {"bytes": n * 32.0 + case["targets"] * 40.0, "flops": n * case["targets"] * 20.0}
    if k == "direct":
        return {"bytes": n * (128.0 + 96.0 * case["steps"]), "flops": case["steps"] * 20.0 * n * n}
    if k == "forces":
        return {"bytes": n * (56.0 + 16.0), "flops": _evaluation_flops(case, n)}
    if k == "gradient":
        # a step forward, a step recomputed and its transpose
        return {"bytes": n * (128.0 + 96.0 * 3 * case["steps"]),
                "flops": 3.0 * case["steps"] * _evaluation_flops(case, n)}
    return {"bytes": n * (128.0 + 96.0 * case["steps"]), "flops": case["steps"] * _evaluation_flops(case, n)}


# ---- the direct sums in 64 bits --------------------------------------------------
def _field(x, m, eps, targets=None):
    """Accelerations and potentials at the targets (default: every particle)."""
    t = x if targets is None else x[targets]
    acc, pot = torch.empty_like(t), torch.empty_like(t[:, 0])
    own = torch.arange(len(x), device=x.device) if targets is None else targets
    rows = max(1, (1 << 26) // len(x))
    for b in range(0, len(t), rows):
        d = x[None] - t[b:b + rows, None]
        w = d.square().sum(-1).add_(eps * eps).rsqrt_()
        mw = m * w
        pot[b:b + rows] = m[own[b:b + rows]] / eps - mw.sum(1)
        acc[b:b + rows] = (mw.mul_(w).mul_(w)[..., None] * d).sum(1)
    return acc, pot


def _systems(case, seed):
    x, v, m, off = _inputs(case, seed)
    off = [0, len(m)] if off is None else off
    for a, b in zip(off[:-1], off[1:]):
        yield [torch.tensor(t[int(a):int(b)], dtype=torch.float64, device="cuda") for t in (x, v, m)]


def _leapfrog(x, v, m, case):
    dt, path = case["dt"], [x]
    a = _field(x, m, case["eps"])[0]
    for _ in range(case["steps"]):
        v = v + 0.5 * dt * a
        x = x + dt * v
        a = _field(x, m, case["eps"])[0]
        v = v + 0.5 * dt * a
        path.append(x)
    return x, v, path


def _field_vjp(x, m, eps, w):
    """(da/dx)^T w and (da/dm)^T w: per pair with d = x_j - x_i, s = 1 / sqrt(d^2 + eps^2)
    and u = m_j w_i - m_i w_j, dx_i -= s^3 u - 3 s^5 (u . d) d."""
    gx, gm = torch.empty_like(x), torch.empty_like(m)
    rows = max(1, (1 << 25) // len(x))
    for b in range(0, len(x), rows):
        xi, wi, mi = x[b:b + rows, None], w[b:b + rows, None], m[b:b + rows, None, None]
        d = x[None] - xi
        s = d.square().sum(-1, keepdim=True).add_(eps * eps).rsqrt_()
        s3 = s ** 3
        u = m[None, :, None] * wi - mi * w[None]
        gx[b:b + rows] = -(s3 * u - 3.0 * s3 * s * s * (u * d).sum(-1, keepdim=True) * d).sum(1)
        gm[b:b + rows] = -(s3 * w[None] * d).sum((1, 2))
    return gx, gm


def _exact_gradient(case, seed):
    x, v, m, goal = [t.double() for t in _gradient_inputs(case, seed)]
    dt, eps = case["dt"], case["eps"]
    xn, vn, path = _leapfrog(x, v, m, case)
    xb, vb = 2.0 * (xn - goal) / xn.numel(), 0.2 * vn / vn.numel()
    gx, mb = _field_vjp(path[-1], m, eps, 0.5 * dt * vb)
    xb = xb + gx
    for j in range(case["steps"] - 1, -1, -1):
        vb = vb + dt * xb
        gx, gm = _field_vjp(path[j], m, eps, (0.5 if j == 0 else 1.0) * dt * vb)
        xb, mb = xb + gx, mb + gm
    return [xn, vn, xb, vb, mb]


def exact(case, seed):
    """What run() returns for these inputs by direct sums, where they take no
    longer than some seconds."""
    evaluations = {"forces": 1, "check": case["targets"] / case["n"], "gradient": 4 * case["steps"]}
    if case["n"] ** 2 * max(1, case["nsys"] / 8) * evaluations.get(case["kind"], case["steps"] + 1) > 2e11:
        return None
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    if case["kind"] in ("forces", "check"):
        x, _, m = next(_systems(case, seed))
        at = torch.tensor(_targets(case, seed), device="cuda") if case["kind"] == "check" else None
        acc, pot = _field(x, m, case["eps"], at)
        return [acc, pot]
    ends = [_leapfrog(x, v, m, case)[:2] + (m,) for x, v, m in _systems(case, seed)]
    x, v, m = (torch.cat([e[i] for e in ends]) for i in range(3))
    t = 0.0
    for _ in range(case["steps"]):
        t += case["dt"]
    return [x, v, m, m, t]
