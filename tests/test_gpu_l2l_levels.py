"""L2L: the levels that take one launch, and those below them that take one
each, against copies of one system on its own (whose levels all take one)."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


def _run(x, m, off, order):
    cfg = nb.default_config(leaf_capacity=1, order=order, theta=0.5, eps=1e-2)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg, sys_off=off) as sim:
        acc, pot = sim.forces()
        nodes = sim.stats()["num_nodes"]
        return np.asarray(acc), np.asarray(pot), nodes


@pytest.mark.parametrize("order", [1, 4, 6])
@pytest.mark.parametrize("copies", [2, 11, 24])
def test_copies_equal_one(copies, order):
    n = 5000
    rng = np.random.default_rng(3)
    x = rng.standard_normal((n, 3)) * rng.uniform(0.05, 1.0, (n, 1))
    m = np.full(n, 1.0 / n)
    a1, p1, nodes1 = _run(x, m, np.array([0, n]), order)
    a, p, nodes = _run(np.tile(x, (copies, 1)), np.tile(m, copies), n * np.arange(copies + 1), order)
    assert nodes == copies * nodes1
    if copies == 2:
        assert nodes < 65536  # one launch
    else:
        assert nodes > 65536  # several
    # 32-bit sums of up to some thousand terms, added in another order
    assert np.abs(a.reshape(copies, n, 3) - a1).max() <= 2e-5 * np.abs(a1).max()
    assert np.abs(p.reshape(copies, n) - p1).max() <= 2e-5 * np.abs(p1).max()
