"""Opening ratios above 1, at which cells of level 1 are well separated: the
tabled M2L takes their pairs too, as the plain one does."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


def _rms(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return np.sqrt(np.mean((a - b) ** 2) / np.mean(b**2))


def _system(n, systems):
    rng = np.random.default_rng(n + systems)
    x, m = rng.uniform(-1, 1, (n, 3)), rng.uniform(0.5, 1.5, n) / n
    off = np.linspace(0, n, systems + 1).astype(np.uint32) if systems > 1 else None
    return x, 0.1 * rng.standard_normal((n, 3)), m, off


@pytest.mark.parametrize("theta", [1.0, 1.25, 1.5, 1.75, 2.0, 6.0, 64.0])
@pytest.mark.parametrize("n,systems,order", [(3000, 1, 4), (3000, 1, 5), (1000, 1, 6), (2500, 3, 4)])
def test_grouped_equals_plain(theta, n, systems, order):
    x, v, m, off = _system(n, systems)
    w = np.random.default_rng(1).standard_normal((n, 3))
    got = []
    for m2l in (nb.M2L_PLAIN, nb.M2L_GROUPED):
        cfg = nb.default_config(theta=theta, leaf_capacity=8, order=order, eps=1e-2, m2l=m2l)
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg, sys_off=off) as sim:
            acc, pot = sim.forces()
            gx, gm = sim.force_vjp(w)
            level = np.array(sim.debug_tree()["level"])
            got.append((acc, pot, gx, gm))
    assert level.max() >= 2
    # one operator and lists, FP32 in two orders
    for a, b in zip(got[1], got[0]):
        assert _rms(a, b) < 2e-5


@pytest.mark.parametrize("theta", [1.25, 2.0])
@pytest.mark.parametrize("m2l", [nb.M2L_BF16X3, nb.M2L_MFMA_F32])
def test_matrix_core_forms(theta, m2l):
    """They take level 1 as the grouped form does, so their error is of the same
    size."""
    x, v, m, _ = _system(4000, 1)
    err = []
    for form in (nb.M2L_GROUPED, m2l):
        cfg = nb.default_config(theta=theta, leaf_capacity=16, eps=1e-2, m2l=form)
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
            acc, _ = sim.forces()
            exact, _ = sim.direct_fp64(np.arange(len(m)))
        err.append(_rms(acc, exact))
    assert err[1] < 1.1 * err[0] and err[0] < (0.05 if theta < 1.5 else 0.25)


@pytest.mark.parametrize("theta", [1.25, 2.0])
def test_captured_steps(theta):
    x, v, m, _ = _system(4000, 1)
    end = []
    for graph in (0, 1):
        cfg = nb.default_config(theta=theta, leaf_capacity=16, eps=1e-2, graph=graph)
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
            sim.step(5)
            end.append(sim.state())
            assert not graph or sim.stats()["graph_replays"] >= 3
    assert np.max(np.abs(end[0][0] - end[1][0])) < 1e-9 and np.max(np.abs(end[0][1] - end[1][1])) < 1e-6
