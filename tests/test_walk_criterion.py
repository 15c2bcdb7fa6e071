"""The walk's opening criterion as its kernel evaluates it: the library's
threshold per level gap (walk_thresholds, the host function that fills the
kernel's table), the bound on the offsets that are squared in 24 bits, and the
candidate offsets of a cell's eight children, against the criterion in exact
integers."""
import ctypes
import random

import pytest

import nbody_amd as nb
from test_rules_cpu import rules  # noqa: F401

BITS, LEVELS = 21, 22
RATIOS = [(1, 2), (2, 5), (1, 1), (3, 4), (63, 64), (64, 63), (1, 64), (64, 1), (1, 5), (17, 31), (64, 64), (2, 1)]


def _thresholds(num, den):
    thr = (ctypes.c_uint32 * LEVELS)()
    # nbh::walk_thresholds(uint32_t, uint32_t, uint32_t*)
    nb.lib()._ZN3nbh15walk_thresholdsEjjPj(ctypes.c_uint32(4 * num * num), ctypes.c_uint32(3 * den * den), thr)
    return list(thr)


@pytest.mark.parametrize("num,den", RATIOS)
def test_thresholds_of_every_gap(num, den):
    thr = _thresholds(num, den)
    for gap, t in enumerate(thr):
        sides = 2 + (2 << gap)
        lhs = 3 * den * den * sides * sides
        if t == 2**32 - 1:
            assert 4 * num * num * (2**32 - 1) <= lhs  # clamped: nothing below is accepted
        else:
            # the largest squared offset that is not accepted
            assert not lhs < 4 * num * num * t and lhs < 4 * num * num * (t + 1)
    assert (2**32 - 1 in thr) == (3 * den * den * (2 + (2 << 21)) ** 2 // (4 * num * num) >= 2**32 - 1)


def test_small_offsets_are_squared_exactly(rules):  # noqa: F811
    rules.small_offset.argtypes, rules.small_offset.restype = [ctypes.c_int], ctypes.c_int
    small = [d for d in (-2**22, -40000, -32001, -32000, -31999, 0, 31999, 32000, 32001, 40000, 2**22)
             if rules.small_offset(d)]
    assert small == [-32000, -31999, 0, 31999, 32000]
    worst = max(abs(d - o) for d in small for o in (0, 2))
    assert worst < 2**23 and 3 * worst * worst < 2**32


@pytest.mark.parametrize("num,den", RATIOS)
def test_offsets_of_octants_and_carried_leaves(num, den):
    """A candidate of the targets' level or above against the children of a
    cell, by octant (octant 0's offset less 0 or 2 half cells), and a candidate
    below a carried leaf: the kernel's offsets in half cells of the finer level
    and the threshold, and the criterion in half cells of the finest."""
    rng, thr = random.Random(64 * num + den), _thresholds(num, den)
    for _ in range(3000):
        la, lb = rng.randint(1, BITS), rng.randint(0, BITS)
        carried = lb > la
        cell = [rng.randrange(1 << la) for _ in range(3)]  # the leaf, or octant 0 of a cell's children
        if not carried:
            cell = [c & ~1 for c in cell]
        if rng.random() < 0.7:  # near the targets, where the answers differ
            reach = rng.choice([2, 6, 20])
            at = [((2 * c + 1) << lb) >> (la + 1) for c in cell]
            gb = [min(max(a + rng.randint(-reach, reach), 0), (1 << lb) - 1) for a in at]
        else:
            gb = [rng.randrange(1 << lb) for _ in range(3)]
        sa, sb = max(lb - la, 0), max(la - lb, 0)
        d0 = [((2 * g + 1) << sb) - ((2 * c + 1) << sa) for g, c in zip(gb, cell)]
        for octant in range(1 if carried else 8):
            bit = [octant >> 2, octant >> 1 & 1, octant & 1]
            d = [v - 2 * b for v, b in zip(d0, bit)]
            c = [((2 * g + 1) << (BITS - lb)) - ((2 * (a + b) + 1) << (BITS - la)) for g, a, b in zip(gb, cell, bit)]
            sides = (2 << (BITS - la)) + (2 << (BITS - lb))
            want = 3 * den * den * sides * sides < 4 * num * num * sum(v * v for v in c)
            t = thr[sa + sb]
            if t < 2**32 - 1:
                assert (sum(v * v for v in d) > t) == want
            elif want:
                assert sum(v * v for v in d) >= t
