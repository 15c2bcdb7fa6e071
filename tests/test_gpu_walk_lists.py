"""The walk's lists against the oracle's where its integer criterion changes
form: opening ratios of every kind, level gaps beyond ten (64-bit offsets), and
split lists longer than the workgroup's cache (taken in sections)."""
import numpy as np
import pytest

import nbody_amd as nb
import pyoracle as po

pytestmark = pytest.mark.gpu


def _cluster_and_halo(n, scale, seed):
    """A cluster of the given radius among a few particles filling the cube: its
    cells are many levels below the leaves that they meet."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, 3))
    k = n - 40
    x[:k] = 0.3 + scale * rng.standard_normal((k, 3))
    return x


CASES = [
    # particles, cluster radius, leaf capacity, theta
    (3000, 1e-5, 2, (1, 2)),       # gaps up to 19
    (3000, 1e-3, 4, (1, 2)),       # gaps about ten: both forms in one walk
    (6000, 0.05, 1, (1, 2)),       # a halo leaf's split list of thousands
    (2000, 0.2, 3, (1, 1)),
    (2000, 0.2, 3, (3, 4)),
    (2000, 0.2, 5, (2, 5)),
    (1200, 0.1, 4, (3, 10)),
    (1000, 0.3, 4, (17, 31)),
    (1500, 1e-4, 3, (63, 64)),
]


@pytest.mark.parametrize("n,scale,cap,th", CASES)
def test_lists_equal_oracle(n, scale, cap, th):
    x = _cluster_and_halo(n, scale, 11)
    m = np.full(n, 1.0 / n)
    cfg = nb.default_config(leaf_capacity=cap, order=2, theta=th[0] / th[1], eps=1e-2)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg) as sim:
        sim.forces()
        keys = sim.debug_keys()[0]
        mo, ms, po_, ps = sim.debug_lists()
    tree = po.build_tree(keys, cap=cap)
    lists = po.walk(tree, *th)
    assert np.array_equal(mo, lists.m2l_off) and np.array_equal(ms, lists.m2l_src)
    assert np.array_equal(po_, lists.p2p_off) and np.array_equal(ps, lists.p2p_src)
