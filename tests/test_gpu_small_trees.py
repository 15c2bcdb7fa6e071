"""Sorted order, tree and links of small systems against the oracle at the edges
of the one-launch sort (64 particles a workgroup, RANK_MAX = 40,960), of the
one-workgroup scan and of the bounding cube's tiles; equal keys keep their
order."""
import numpy as np
import pytest

import nbody_amd as nb
import pyoracle as po

pytestmark = pytest.mark.gpu

FIELDS = ["level", "sys", "ix", "iy", "iz", "begin", "count", "first_child", "nchild", "parent"]


def _positions(n, kind):
    rng = np.random.default_rng(n)
    if kind == "plummer":
        return nb.ics.plummer(n, n + 1)[0]
    x = rng.uniform(0, 1, (n, 3))
    # many particles at few points: long runs of equal keys
    x[: n // 2] = x[rng.integers(n // 2, n, n // 2)]
    return x


@pytest.mark.parametrize("kind", ["plummer", "coincident"])
@pytest.mark.parametrize("n", [2, 63, 64, 65, 1024, 1025, 4097, 40960, 40961, 65536, 65537, 91000])
def test_order_and_tree_match_oracle(n, kind):
    x = _positions(n, kind)
    m = np.full(n, 1.0 / n)
    cfg = nb.default_config(leaf_capacity=32, order=1, max_depth=12)
    with nb.HipSimulation.from_arrays(x, np.zeros_like(x), m, m, config=cfg) as sim:
        for turn in range(2):  # the second build starts from the sorted state
            sim.forces()
            keys, ids, box = sim.debug_keys()
            t = sim.debug_tree()
    keys_o, box_o = po.morton(x)
    order = np.argsort(keys_o, kind="stable")
    assert np.array_equal(box, box_o) and np.array_equal(keys, keys_o[order])
    assert np.array_equal(ids, order.astype(np.uint32))
    tree = po.build_tree(keys, cap=32, max_depth=12)
    for f in FIELDS:
        assert np.array_equal(t[f], getattr(tree, f)), f


def test_small_ensemble_matches_oracle():
    x, v, m, off = nb.ics.ensemble(9, nmin=1, nmax=3000)
    cfg = nb.default_config(leaf_capacity=8, order=1)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg, sys_off=off) as sim:
        sim.forces()
        keys, ids, box = sim.debug_keys()
        t = sim.debug_tree()
        bits = min(21, (64 - 4) // 3)
    keys_o, box_o = po.morton(x, sys_off=off, bits=bits)
    order = np.argsort(keys_o, kind="stable")
    assert np.array_equal(box, box_o) and np.array_equal(keys, keys_o[order])
    assert np.array_equal(ids, order.astype(np.uint32))
    tree = po.build_tree(keys, sys_off=off, bits=bits, cap=8, max_depth=bits)
    for f in FIELDS:
        assert np.array_equal(t[f], getattr(tree, f)), f
