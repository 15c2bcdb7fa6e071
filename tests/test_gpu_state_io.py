"""State and forces between the sorted device arrays and the caller's: exact
round trips at the sizes where the copies change form (one pinned copy up to 4
MiB, chunks of 2 MiB through a ring of eight above)."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 777, 65536, 65537, 87382, 349526, 700001])
def test_state_round_trip(n):
    rng = np.random.default_rng(n)
    x, v, m, q = rng.uniform(-1, 1, (n, 3)), rng.standard_normal((n, 3)), rng.uniform(1, 2, n), rng.uniform(-1, 1, n)
    cfg = nb.default_config(eps=1e-2, leaf_capacity=64, order=2)
    with nb.HipSimulation.from_arrays(x, v, m, q, config=cfg) as sim:
        for turn in range(2):
            a0, p0 = sim.forces()          # leaves the state sorted
            got = sim.state()
            assert all(np.array_equal(a, b) for a, b in zip(got[:4], (x, v, m, q)))
            assert np.array_equal(sim.positions(), x)
            x, v = x[::-1].copy(), v + 1.0
            sim.set_state(x, v, 2.5)
            got = sim.state()
            assert all(np.array_equal(a, b) for a, b in zip(got, (x, v, m, q, 2.5)))
        x = x[::-1].copy()
        with nb.HipSimulation.from_arrays(x, v, m, q, config=cfg) as other:
            sim.set_state(x, v)
            a, p = sim.forces()
            b, r = other.forces()
        # one input order, one tree: equal up to the order of the far pairs' atomics
        assert np.allclose(a, b, rtol=1e-5, atol=1e-5 * np.abs(b).max()) and np.allclose(p, r, rtol=1e-5)


def test_set_state_refuses_and_keeps():
    x, v, m = nb.ics.plummer(3001, 2)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=nb.default_config()) as sim:
        t = sim.step(2)
        before = sim.state()
        for bad in (np.nan, np.inf, -np.inf):
            for k in (0, 1):
                y, w = x.copy(), v.copy()
                (y, w)[k][2999, 2] = bad
                with pytest.raises(RuntimeError, match="non-finite state"):
                    sim.set_state(y, w)
        after = sim.state()
        assert after[4] == t and all(np.array_equal(a, b) for a, b in zip(before, after))
        sim.set_state(x, v)
        assert np.array_equal(sim.positions(), x)


def test_ring_grows_behind_an_upload():
    """A transfer that needs a larger ring than the upload before it, which may
    still be on its way: targets (8 bytes each) up, their sums (32) down."""
    x, v, m = nb.ics.plummer(9001, 4)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=nb.default_config()) as sim:
        t = np.arange(9001)
        whole = sim.direct_fp64(t)
    for nt in (1, 2049, 8191):
        with nb.HipSimulation.from_arrays(x[:100], v[:100], m[:100], m[:100], config=nb.default_config()) as small:
            few = small.direct_fp64(np.arange(nt) % 100)
            assert np.array_equal(few[0], few[0][np.arange(nt) % 100])
        with nb.HipSimulation.from_arrays(x, v, m, m, config=nb.default_config()) as sim:
            acc, pot = sim.direct_fp64(t[:nt])
        assert np.allclose(acc, whole[0][:nt], rtol=1e-12, atol=0) and np.allclose(pot, whole[1][:nt], rtol=1e-12)
