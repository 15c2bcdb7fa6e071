"""The walk's lists against the oracle's on both sides of the number of groups
where a depth changes from eight wavefronts a workgroup to four."""
import numpy as np
import pytest

import nbody_amd as nb
import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dropped", [0, 15, 16, 17, 480])
def test_lists_equal_oracle(dropped):
    # one particle in each of 16^3 cells, less some whole cells of the level
    # above: its 512 - dropped groups take 16 more workgroups
    rng = np.random.default_rng(5)
    ijk = np.stack(np.meshgrid(*[np.arange(16)] * 3, indexing="ij"), -1).reshape(-1, 3)
    parent = (ijk[:, 0] >> 1) * 64 + (ijk[:, 1] >> 1) * 8 + (ijk[:, 2] >> 1)
    gone = 1 + rng.choice(510, dropped, replace=False)  # the corners stay: the cube's bounds
    x = (ijk + rng.uniform(0.25, 0.75, ijk.shape))[~np.isin(parent, gone)] / 16
    x[0], x[-1] = 0.0, 1.0
    n = len(x)
    m = np.full(n, 1.0 / n)
    cfg = nb.default_config(leaf_capacity=1, order=2, theta=0.5, eps=1e-2)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg) as sim:
        sim.forces()
        keys = sim.debug_keys()[0]
        mo, ms, po_, ps = sim.debug_lists()
    tree = po.build_tree(keys, cap=1)
    lists = po.walk(tree, 1, 2)
    assert np.array_equal(mo, lists.m2l_off) and np.array_equal(ms, lists.m2l_src)
    assert np.array_equal(po_, lists.p2p_off) and np.array_equal(ps, lists.p2p_src)
