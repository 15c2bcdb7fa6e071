"""The direct sums (FP32 solver, FP64 check) against numpy in 64 bits, at the
edges of their 64-target workgroups, source slices and targets per workgroup."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


def _sum64(x, m, eps, targets):
    acc, pot = np.zeros((len(targets), 3)), np.zeros(len(targets))
    for k, i in enumerate(targets):
        d = x - x[i]
        r2 = (d * d).sum(1) + eps * eps
        r2[i] = 1.0
        w = m / np.sqrt(r2)
        w[i] = 0.0
        acc[k] = ((w / r2)[:, None] * d).sum(0)
        pot[k] = -w.sum()
    return acc, pot


def _packed(x):
    """The positions that the FP32 solver sums over: FP32 offsets from the
    centre of the system's bounding cube."""
    lo = x.min(0)
    size = (x.max(0) - lo).max()
    return (x - (lo + 0.5 * (size if size > 0 else 1.0))).astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("n", [1, 2, 15, 63, 64, 65, 129, 1000, 4097])
@pytest.mark.parametrize("eps", [1e-2, 0.0])
def test_direct_solver(n, eps):
    x, v, m = nb.ics.plummer(n, 3)
    cfg = nb.default_config(solver=nb.SOLVER_DIRECT, eps=eps)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
        acc, pot = sim.forces()
    t = np.arange(0, n, max(1, n // 97))
    ar, pr = _sum64(_packed(x), m, eps, t)
    # FP32 terms and sums of up to n of them
    tol = 2e-5
    scale = np.sqrt((ar * ar).sum(1).mean()) + 1e-30
    assert np.max(np.abs(acc[t] - ar)) <= tol * max(scale, np.abs(ar).max()) + 1e-30
    assert np.max(np.abs(pot[t] - pr)) <= tol * np.abs(pr).max() + 1e-30


def test_direct_solver_ensemble():
    x, v, m, off = nb.ics.ensemble(5, nmin=30, nmax=700)
    cfg = nb.default_config(solver=nb.SOLVER_DIRECT, eps=1e-2)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg, sys_off=off) as sim:
        acc, _ = sim.forces()
    for a, b in zip(off[:-1], off[1:]):
        t = np.arange(a, b, 11)
        ar, _ = _sum64(_packed(x[a:b]), m[a:b], 1e-2, t - a)
        assert np.max(np.abs(acc[t] - ar)) <= 2e-5 * np.abs(ar).max()


@pytest.mark.parametrize("n,nt", [(1, 1), (2, 2), (500, 3), (511, 511), (1500, 1031), (5003, 4096), (5003, 4099)])
@pytest.mark.parametrize("eps", [1e-3, 0.0])
def test_fp64_sums(n, nt, eps):
    x, v, m = nb.ics.plummer(n, 5)
    t = np.random.default_rng(n).permutation(n)[:nt]
    with nb.HipSimulation.from_arrays(x, v, m, m, config=nb.default_config(eps=eps)) as sim:
        sim.step(1)
        x = sim.positions()
        acc, pot = sim.direct_fp64(t)
        acc2, pot2 = sim.direct_fp64_noalloc(t)
    assert np.array_equal(acc, acc2) and np.array_equal(pot, pot2)
    s = np.arange(0, nt, max(1, nt // 97))
    ar, pr = _sum64(x, m, eps, t[s])
    # 64-bit sums of up to n terms, each to a few ulps
    assert np.max(np.abs(acc[s] - ar)) <= 1e-13 * np.abs(ar).max() + 1e-300
    assert np.max(np.abs(pot[s] - pr)) <= 1e-13 * np.abs(pr).max() + 1e-300


def test_fp64_sums_of_coincident_particles():
    # distinct particles at one point, unsoftened: no finite potential; far away ones: no force
    x = np.array([[0.0, 0, 0], [0, 0, 0], [1, 0, 0], [1e160, 0, 0]])
    m = np.ones(4)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=nb.default_config(eps=0.0)) as sim:
        acc, pot = sim.direct_fp64([0, 2, 3])
    assert pot[0] == -np.inf and np.isnan(acc[0]).any()
    assert acc[1][0] == -2.0 and pot[1] == -2.0
    assert np.all(acc[2] == 0.0) and pot[2] == 0.0


# (particles, systems) either side of the rules that choose the kernel: systems
# of 192 particles, and total targets against 24,576 + 24 size, at most 98,304
@pytest.mark.parametrize("size,systems", [(191, 1), (192, 1), (191, 7), (192, 151), (192, 152), (257, 3), (8, 1031),
                                          (1, 65), (40000, 1), (98304, 1), (98305, 1)])
@pytest.mark.parametrize("eps", [1e-2, 0.0])
def test_direct_solver_forms(size, systems, eps):
    rng = np.random.default_rng(size)
    n = size * systems
    x, m = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n) / size
    off = (np.arange(systems + 1) * size).astype(np.uint32)
    cfg = nb.default_config(solver=nb.SOLVER_DIRECT, eps=eps)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg,
                                      sys_off=off if systems > 1 else None) as sim:
        acc, pot = sim.forces()
        sim.step(1)
        moved = sim.state()[1]
    for s in {0, systems // 2, systems - 1}:
        a, b = size * s, size * (s + 1)
        t = np.arange(a, b, max(1, size // 61))
        ar, pr = _sum64(_packed(x[a:b]), m[a:b], eps, t - a)
        # FP32 terms and sums of n of them in order: n half ulps of the largest partial sum
        tol = 2e-5 if size < 5000 else 1e-4
        assert np.max(np.abs(acc[t] - ar)) <= tol * np.abs(ar).max() + 1e-30
        assert np.max(np.abs(pot[t] - pr)) <= tol * np.abs(pr).max() + 1e-30
    # v after a step of dt from rest, to first order (the closing kick reaches every system)
    assert np.all(np.isfinite(moved)) and (size == 1 or np.all(np.any(moved != 0.0, axis=1)))


@pytest.mark.parametrize("what", ["charge", "position"])
@pytest.mark.parametrize("size", [192, 200, 208, 311])
def test_direct_solver_keeps_systems_apart(size, what):
    """A system beside one whose values overflow FP32 has the forces that it has alone."""
    rng = np.random.default_rng(size)
    x, m = rng.standard_normal((2 * size, 3)), rng.uniform(0.5, 1.5, 2 * size)
    cfg = nb.default_config(solver=nb.SOLVER_DIRECT, eps=1e-2)
    with nb.HipSimulation.from_arrays(x[:size], 0 * x[:size], m[:size], m[:size], config=cfg) as sim:
        alone = sim.forces()
    if what == "charge":
        m[size:] = 1e39
    else:
        x[size:] *= 1e39
    with nb.HipSimulation.from_arrays(x, 0 * x, m, m, config=cfg, sys_off=np.array([0, size, 2 * size])) as sim:
        acc, pot = sim.forces()
    assert np.array_equal(acc[:size], alone[0]) and np.array_equal(pot[:size], alone[1])


@pytest.mark.parametrize("small", [510, 511, 512])
def test_direct_solver_many_small_systems(small):
    """A system among many of two particles, 511 to 513 in all."""
    rng = np.random.default_rng(small)
    size = np.array([2] * (small // 2) + [333] + [2] * (small - small // 2))
    off = np.concatenate([[0], np.cumsum(size)])
    n, a = int(off[-1]), int(off[small // 2])
    x, m = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n)
    cfg = nb.default_config(solver=nb.SOLVER_DIRECT, eps=1e-2)
    with nb.HipSimulation.from_arrays(x[a:a + 333], 0 * x[a:a + 333], m[a:a + 333], m[a:a + 333], config=cfg) as sim:
        alone = sim.forces()[0]
    with nb.HipSimulation.from_arrays(x, 0 * x, m, m, config=cfg, sys_off=off) as sim:
        acc = sim.forces()[0]
    assert np.array_equal(acc[a:a + 333], alone)
    for i in range(20):
        j = i ^ 1
        ar, _ = _sum64(_packed(x[[i, j]]), m[[i, j]], 1e-2, [0])
        assert np.max(np.abs(acc[i] - ar[0])) <= 2e-5 * np.abs(ar).max()


# systems x size and targets either side of the rule for ensembles: 1024 and
# 2048 targets, mean sizes 1024 and 4096, and a last workgroup that is not full
@pytest.mark.parametrize("systems,size,nt", [(3, 500, 1023), (3, 500, 1024), (2, 1024, 1027), (2, 1025, 2047),
                                             (2, 1025, 2048), (2, 4096, 4099), (2, 4097, 4099), (700, 3, 2100),
                                             (65, 64, 1)])
def test_fp64_sums_of_ensembles(systems, size, nt):
    rng = np.random.default_rng(systems * size)
    n = systems * size
    x, m = rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n) / size
    off = np.arange(systems + 1) * size
    t = rng.permutation(n)[:nt]
    cfg = nb.default_config(eps=1e-3)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg, sys_off=off) as sim:
        acc, pot = sim.direct_fp64(t)
        acc2, pot2 = sim.direct_fp64_noalloc(t)
    assert np.array_equal(acc, acc2) and np.array_equal(pot, pot2)
    for k in range(0, nt, max(1, nt // 97)):
        s = t[k] // size
        ar, pr = _sum64(x[size * s:size * (s + 1)], m[size * s:size * (s + 1)], 1e-3, [t[k] - size * s])
        # 64-bit sums of up to 4097 terms, each to a few ulps; a sum that cancels has the terms' errors
        assert np.max(np.abs(acc[k] - ar[0])) <= 1e-12 * max(np.abs(ar).max(), np.abs(pr[0]))
        assert abs(pot[k] - pr[0]) <= 1e-13 * abs(pr[0])
