"""A handle's first evaluation, in memory that other handles have used and
freed, equals its second: nothing is read before it is written."""
import numpy as np
import pytest

import nbody_amd as nb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cap", [(777, 8), (5003, 16), (4096, 16), (16384, 16), (30011, 24)])
def test_first_evaluation_equals_second(n, cap):
    x, v, m = nb.ics.plummer(n, 3)
    cfg = nb.default_config(leaf_capacity=cap, eps=1e-2)
    for _ in range(3):
        # leaves its pools, rows and tables, full of another tree's data, to the allocator
        y, w, q = nb.ics.uniform(2 * n + 4096, 1)
        with nb.HipSimulation.from_arrays(y, w, q, q, config=nb.default_config(leaf_capacity=4)) as other:
            other.step(1)
        with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg) as sim:
            a, p = sim.forces()
            b, r = sim.forces()
        # equal up to the order of the far pairs' atomics
        assert np.allclose(a, b, rtol=1e-5, atol=1e-5 * np.abs(b).max()) and np.allclose(p, r, rtol=1e-5)


def test_tree_outgrows_its_arrays():
    """A handle whose tree grows many times over (all particles close together
    in pairs, so that cells go down to the pairs) has a new handle's forces,
    and again after it shrinks."""
    n = 6001
    x, v, m = nb.ics.uniform(n, 2)
    tight = x.copy()
    tight[1::2] = tight[:-1:2] + 1e-5 * (x[1::2] - 0.5)
    cfg = nb.default_config(leaf_capacity=1, eps=1e-2)
    big = nb.default_config(leaf_capacity=512, eps=1e-2)
    for c in (cfg, big):
        with nb.HipSimulation.from_arrays(x, v, m, m, config=c) as sim:
            for pos in (x, tight, x, tight):
                sim.set_state(pos, v)
                a, p = sim.forces()
                g = sim.force_vjp(v + 1.0)[0]
                with nb.HipSimulation.from_arrays(pos, v, m, m, config=c) as new:
                    b, r = new.forces()
                    gn = new.force_vjp(v + 1.0)[0]
                assert np.allclose(a, b, rtol=1e-5, atol=1e-5 * np.abs(b).max()) and np.allclose(p, r, rtol=1e-5)
                assert np.allclose(g, gn, rtol=1e-4, atol=1e-4 * np.abs(gn).max())
