"""M2M: the monopole of every root against the sum of its charges, at numbers of
cells a level around the eight that a wavefront takes."""
import numpy as np
import pytest

import nbody_amd as nb
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 4, 6])
@pytest.mark.parametrize("systems", [1, 7, 8, 9, 65])
def test_root_monopoles(systems, order):
    rng = np.random.default_rng(systems)
    size = rng.integers(40, 700, systems)
    off = np.concatenate([[0], np.cumsum(size)])
    n = int(off[-1])
    x = rng.standard_normal((n, 3))
    m = rng.uniform(0.5, 1.5, n)
    cfg = nb.default_config(leaf_capacity=4, order=order, theta=0.5, eps=1e-2)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg, sys_off=off) as sim:
        sim.forces()
        M = np.asarray(sim.debug_expansions()[0], dtype=np.float64).reshape(sim.stats()["num_nodes"], -1)
    want = np.add.reduceat(m, off[:-1])
    # 32-bit sums of at most 700 positive terms
    assert np.abs(M[:systems, 0] - want).max() <= 700 * 2.0**-24 * want.max()


@pytest.mark.parametrize("order", [2, 4, 6])
@pytest.mark.parametrize("systems", [1, 7, 8, 9, 65])
def test_root_moments(systems, order):
    """Every moment of every root (a wrong shift leaves the monopole as it is)
    against the sums over its particles."""
    rng = np.random.default_rng(systems + 100)
    size = rng.integers(40, 700, systems)
    off = np.concatenate([[0], np.cumsum(size)])
    n = int(off[-1])
    x = rng.standard_normal((n, 3))
    m = rng.uniform(0.5, 1.5, n)
    cfg = nb.default_config(leaf_capacity=4, order=order, theta=0.5, eps=1e-2)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg, sys_off=off) as sim:
        sim.forces()
        M = np.asarray(sim.debug_expansions()[0], dtype=np.float64)
        box = sim.debug_keys()[2]
    for s in range(systems):
        a, b = off[s], off[s + 1]
        half = 0.5 * box[s, 3]
        want = po.p2m(order, box[s, :3] + half, x[a:b], m[a:b])
        # 32-bit sums of at most 700 terms over a dozen shifts, each no larger
        # than if every particle sat in the cube's corner
        most = po.p2m(order, np.zeros(3), np.full((b - a, 3), half), m[a:b])
        assert np.all(np.abs(M[s] - want) <= 700 * 2.0**-24 * np.abs(most))
