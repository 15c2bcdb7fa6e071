"""Trees of one cell (no more particles than the leaf capacity, alone or in an
ensemble), at opening ratios up to the largest that is accepted: no M2L list,
no workgroup in the walk, the forces those of the direct sum."""
import numpy as np
import pytest

import nbody_amd as nb
from helpers import max_rel_floor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("theta", [0.5, 6.0, 64.0])
@pytest.mark.parametrize("size", [[1], [8], [2, 1], [8, 3, 1, 5, 8, 2, 7, 4, 6, 8]])
def test_forces_and_steps(theta, size):
    rng = np.random.default_rng(sum(size))
    off = np.concatenate([[0], np.cumsum(size)]).astype(np.uint32)
    n = int(off[-1])
    x, v, m = rng.standard_normal((n, 3)), rng.standard_normal((n, 3)), rng.uniform(0.5, 1.5, n)
    cfg = nb.default_config(theta=theta, eps=1e-2, leaf_capacity=8)
    with nb.HipSimulation.from_arrays(x, v, m, m, config=cfg, sys_off=off if len(size) > 1 else None) as sim:
        acc, pot = sim.forces()
        s = sim.debug_sizes()
        want, want_pot = sim.direct_fp64(np.arange(n))
        sim.step(2)
        assert np.all(np.isfinite(sim.positions()))
    assert s["depth"] == 0 and s["nodes"] == len(size) and s["m2l"] == 0 and s["p2p"] == len(size)
    alone = np.repeat(np.array(size) == 1, size)
    assert np.all(acc[alone] == 0.0)
    # FP32 sums of at most 7 pairs whose offsets carry half an ulp of the cell's size
    if not alone.all():
        assert max_rel_floor(acc[~alone], want[~alone]) < 2e-5
        assert np.max(np.abs(pot[~alone] - want_pot[~alone]) / np.abs(want_pot[~alone])) < 2e-5
