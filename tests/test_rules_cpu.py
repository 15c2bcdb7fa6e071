"""The host's sizing rules (csrc/rules.h), compiled on the CPU."""
import ctypes
import os
import shutil
import subprocess

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
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "librules.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC",
                    "-I" + os.path.join(ROOT, "nbody_amd", "csrc"), str(d / "shim.cpp"), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


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
