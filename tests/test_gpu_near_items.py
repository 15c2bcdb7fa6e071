"""The near field cut into items (P2P lists longer than an item, target leaves
of more than one wavefront) against the plain kernel that takes a leaf's whole
list at once, on the same tree and lists."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


def _sphere(n, seed):
    return nb.ics.plummer(n, seed)


def _halo(n, seed):
    """A dense ball and a few particles far out: their large leaves meet every
    leaf of the ball."""
    x, v, m = nb.ics.plummer(n, seed)
    x[: n // 2] *= 0.02
    return x, v, m


def _coincident(n, seed):
    """Cells at the depth limit that hold far more than the leaf capacity."""
    x, v, m = nb.ics.uniform(n, seed)
    x[:: 3] = 0.5 + 1e-9 * (x[:: 3] - 0.5)
    return x, v, m


CASES = [
    ("one", _sphere, 1, dict(leaf_capacity=8)),
    ("two", _sphere, 2, dict(leaf_capacity=1)),
    ("one_leaf_63", _sphere, 63, dict(leaf_capacity=63)),
    ("one_leaf_65", _sphere, 65, dict(leaf_capacity=65)),
    ("leaves_of_129", _sphere, 4099, dict(leaf_capacity=129)),
    ("capacity_1", _sphere, 1537, dict(leaf_capacity=1)),
    ("halo", _halo, 20011, dict(leaf_capacity=8)),
    ("unsoftened", _halo, 5003, dict(leaf_capacity=16, eps=0.0)),
    ("depth_limit", _coincident, 3001, dict(leaf_capacity=16, max_depth=9)),
]


@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("name,ic,n,opt", CASES, ids=[c[0] for c in CASES])
def test_items_match_whole_lists(name, ic, n, opt, chunk):
    x, v, m = ic(n, 7)
    got = []
    for p2p in (nb.P2P_LANE, nb.P2P_LEAF):
        cfg = nb.default_config(**{**dict(eps=1e-2, p2p=p2p, p2p_chunk=chunk), **opt})
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
            got.append((*sim.forces(), sim.stats()["p2p_interactions"], sim.debug_lists()[3]))
    (a, p, pairs, src), (ar, pr, pairs_r, src_r) = got
    assert pairs == pairs_r and np.array_equal(src, src_r)
    # FP32 sums of up to n terms in two orders: error of each at most about
    # sqrt(n) half-ulps of the largest partial sum
    tol = 2e-5
    scale = np.sqrt(np.mean(np.sum(ar.astype(np.float64) ** 2, axis=1))) + 1e-30
    d = np.linalg.norm(a.astype(np.float64) - ar, axis=1)
    assert np.max(d / np.maximum(scale, np.linalg.norm(ar, axis=1))) < tol
    assert np.max(np.abs(p.astype(np.float64) - pr)) <= tol * np.max(np.abs(pr)) + 1e-30


@pytest.mark.parametrize("n,cap,slots", [(300000, 1024, 32768), (600000, 2048, 65536)])
def test_more_items_than_slots(n, cap, slots):
    """512 leaves of ten (19) target chunks that all meet each other in eight
    batches: cut to single batches they would take 40,960 (77,824) slots, of
    65,536.  No far-field pairs, so that every evaluation is the same sum to the
    bit."""
    x, v, m = nb.ics.uniform(n, 5)
    got = []
    for p2p in (nb.P2P_LANE, nb.P2P_LANE, nb.P2P_LEAF):
        cfg = nb.default_config(eps=1e-2, theta=0.125, leaf_capacity=cap, order=2, p2p=p2p)
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
            got += [sim.forces() for _ in range(3 if p2p == nb.P2P_LANE else 1)]
            s, off = sim.debug_sizes(), sim.debug_lists()[2]
            count = np.array(sim.debug_tree()["count"])
    assert s["m2l"] == 0 and s["leaves"] == 512
    leaf = np.diff(off) > 0
    assert np.sum(np.ceil(np.diff(off)[leaf] / 64) * np.ceil(count[leaf] / 64)) > slots
    for a, p in got[1:6]:
        assert np.array_equal(a, got[0][0]) and np.array_equal(p, got[0][1])
    # sums of a part of the sources added up are no further from the 64-bit sum
    # than single ones of all n
    t = np.arange(0, n, 149)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
        exact = sim.direct_fp64(t)
    err = [[np.sqrt(np.mean((f[t] - e) ** 2)) for f, e in zip(g, exact)] for g in (got[0], got[6])]
    assert err[0][0] <= err[1][0] and err[0][1] <= err[1][1]
