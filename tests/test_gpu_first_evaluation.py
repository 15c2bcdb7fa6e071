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
