"""The host's sizing rules (csrc/rules.h), compiled on the CPU."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")

SHIM = r"""
#include "rules.h"
using namespace nbh;
extern "C" {
void pool_sizes(uint32_t nodes, uint32_t max_sys_n, uint64_t n, int num, int den, unsigned long long blocks, int small,
                unsigned long long* out) {
    const PoolSizes s = pool_guess(nodes, max_sys_n, n, num, den, blocks, small != 0);
    out[0] = s.m2l;
    out[1] = s.p2p;
}
uint32_t item_batches(uint64_t entries, uint64_t work, uint32_t slots) { return near_item_batches(entries, work, slots); }
int small_offset(int d) { return walk_small(d); }
uint64_t slots_bound(uint64_t entries, uint64_t work, uint32_t slots) { return near_slots_bound(entries, work, slots); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "librules.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "nbody_amd", "csrc"), str(d / "shim.cpp"), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))
    lib.item_batches.argtypes = lib.slots_bound.argtypes = [ctypes.c_uint64, ctypes.c_uint64, ctypes.c_uint32]
    lib.item_batches.restype, lib.slots_bound.restype = ctypes.c_uint32, ctypes.c_uint64
    return lib


CHUNK_M, CHUNK_P, POOL_MAX = 2048, 512, 0xFFFF0000


def _pools(rules, nodes, num, den, blocks, max_sys_n=None, n=None, small=False):
    """(M2L, P2P) entries; without max_sys_n: one system of as many particles as cells."""
    n = n or max_sys_n or nodes
    out = (ctypes.c_ulonglong * 2)()
    rules.pool_sizes(ctypes.c_uint32(nodes), ctypes.c_uint32(max_sys_n or n), ctypes.c_uint64(n), num, den,
                     ctypes.c_ulonglong(blocks), int(small), out)
    return out[0], out[1]


@pytest.mark.parametrize("num,den", [(1, 64), (1, 2), (2, 5), (1, 1), (4, 1), (5, 1), (51, 10), (6, 1), (8, 1),
                                     (63, 1), (64, 1)])
def test_pools_hold_a_chunk(rules, num, den):
    """A pool is never empty, whatever theta and the number of cells, with no
    workgroup in the walk (trees of one cell) and with many."""
    for nodes in list(range(1, 66)) + [131072, 1 << 20, 100_000_000, 0x7FFFFFFF]:
        for blocks in (0, 64, 22 * 2048):
            for size in (dict(), dict(max_sys_n=1, n=nodes), dict(max_sys_n=8, n=8 * nodes)):
                for small in (False, True):
                    m, p = _pools(rules, nodes, num, den, blocks, small=small, **size)
                    assert CHUNK_M <= m <= POOL_MAX and CHUNK_P <= p <= POOL_MAX
                    assert m >= blocks * CHUNK_M and p >= blocks * CHUNK_P


@pytest.mark.parametrize("systems,particles,cells", [(131072, 8, 1), (1 << 20, 1, 1), (2048, 512, 231), (64, 4096, 700)])
def test_pools_count_one_system_s_cells(rules, systems, particles, cells):
    """A list never crosses systems: no more entries a cell than its own system
    has cells (particles, where cells form chains)."""
    m, p = _pools(rules, systems * cells, 1, 2, 0, max_sys_n=particles, n=systems * particles)
    most = systems * cells * min(cells, particles)
    assert m <= max(most, CHUNK_M) and p <= max(most, CHUNK_P)


def test_pools_at_small_theta(rules):
    """What theta < 1/2 adds stays within 2^29 entries, and a device without
    room gets 256 and 64 entries a cell at any theta."""
    for nodes in (3000, 100_000, 1_000_000):
        half = _pools(rules, nodes, 1, 2, 0, max_sys_n=10 * nodes)
        assert half == (nodes * 1024, nodes * 256)
        for den in (3, 5, 10, 64):
            got = _pools(rules, nodes, 1, den, 0, max_sys_n=10 * nodes)
            for g, h, usual in zip(got, half, (1024, 256)):
                assert h <= g <= max(h, 1 << 29)
                assert g == max(h, min(1 << 29, nodes * min(nodes, usual * den**3 // 8))) or den % 2
            assert _pools(rules, nodes, 1, den, 0, max_sys_n=10 * nodes, small=True) == (nodes * 256, nodes * 64)


def _slots(nb, tc, g):
    """Slots of leaves of nb batches and tc chunks of targets, cut at g."""
    return int(np.where(nb > g, tc * -(-nb // g), 0).sum())


@pytest.mark.parametrize("slots", [1024, 6148, 32768])
def test_near_field_slots_suffice(rules, slots):
    """No lists ask for more slots than there are, nor than the bound that they
    are allocated by; lists short of it are cut to single batches."""
    rng = np.random.default_rng(slots)
    for trial in range(400):
        leaves = int(10 ** rng.uniform(0, 5))
        rows = rng.integers(1, 6, leaves)
        entries = np.ceil(10 ** rng.uniform(0, rng.uniform(0.5, 4.5), leaves)).astype(np.int64)
        nb = rows - 1 + -(-entries // 64)  # rows of a list are rounded up on their own
        tc = np.ceil(2 ** rng.uniform(0, rng.choice([0.01, 1, 5, 15]), leaves)).astype(np.int64)
        work = int((tc * nb).sum())
        g = rules.item_batches(int(entries.sum()), work, slots)
        used = _slots(nb, tc, g)
        assert used <= rules.slots_bound(int(entries.sum()), work, slots) <= max(slots, 0)
        if work <= slots and entries.sum() <= 64 * 16384:
            assert g == 1
    # a leaf at the depth limit that holds a million particles, and the largest work
    for tc, nb in ((1 << 14, 1 << 14), (1 << 25, 1 << 25)):
        work = tc * nb
        g = rules.item_batches(64 * nb, work, slots)
        assert (tc * -(-nb // g) if nb > g else 0) <= rules.slots_bound(64 * nb, work, slots) <= slots


def test_large_leaves_asked_for_more_slots_than_there_are(rules):
    """512 leaves of 10 chunks with 8 batches: 40,960 slots when the cut looked
    at the entries alone."""
    nb, tc = np.full(512, 8), np.full(512, 10)
    assert _slots(nb, tc, 1) > 32768
    assert _slots(nb, tc, rules.item_batches(64 * 8 * 512, int((nb * tc).sum()), 32768)) <= 32768
