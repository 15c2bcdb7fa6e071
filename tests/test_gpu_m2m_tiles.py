"""M2M: the monopole of every root against the sum of its charges, at numbers of
cells a level around the eight that a wavefront takes."""
import numpy as np
import pytest

import nbody_amd as nb

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
