"""The walk's opening criterion in units of half the finer cell with a threshold
per level gap (csrc/walk.hip: walk_thresholds) is the criterion in units of half
the finest cell, 3 den^2 (d_A + d_B)^2 < 4 num^2 |c_B - c_A|^2, in exact integers."""
import random

import pytest

BITS = 21


def _threshold(num, den, gap):
    side = 2 + (2 << gap)
    return 3 * den * den * side * side // (4 * num * num)


@pytest.mark.parametrize("num,den", [(1, 2), (2, 5), (1, 1), (3, 4), (63, 64), (1, 64), (64, 1), (17, 31)])
def test_threshold_rule_is_the_criterion(num, den):
    rng = random.Random(num * 100 + den)
    for _ in range(4000):
        la, lb = rng.randint(0, BITS), rng.randint(0, BITS)
        lf = max(la, lb)
        # offsets near the threshold as well as anywhere
        t = _threshold(num, den, abs(la - lb))
        d = [rng.randint(-40, 40) for _ in range(3)]
        if rng.random() < 0.5:
            d[0] = int(t ** 0.5) + rng.randint(-2, 2)
        d = [2 * v + (0 if la == lb else 1) for v in d]
        # the pair as it stands in units of half the finest cell
        scale = 1 << (BITS - lf)
        dsq = sum(v * v for v in d)
        sides = (2 << (BITS - la)) + (2 << (BITS - lb))
        general = 3 * den * den * sides * sides < 4 * num * num * dsq * scale * scale
        assert (dsq > t) == general
