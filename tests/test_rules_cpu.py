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
void pool_sizes(uint32_t nodes, int num, int den, unsigned long long blocks, unsigned long long* out) {
    const PoolSizes s = pool_guess(nodes, num, den, blocks);
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


def _pools(rules, nodes, num, den, blocks):
    out = (ctypes.c_ulonglong * 2)()
    rules.pool_sizes(ctypes.c_uint32(nodes), num, den, ctypes.c_ulonglong(blocks), out)
    return out[0], out[1]


@pytest.mark.parametrize("num,den", [(1, 64), (1, 2), (2, 5), (1, 1), (4, 1), (5, 1), (51, 10), (6, 1), (8, 1),
                                     (63, 1), (64, 1)])
def test_pools_hold_a_chunk(rules, num, den):
    """A pool is never empty, whatever theta and the number of cells, with no
    workgroup in the walk (trees of one cell) and with many."""
    for nodes in list(range(1, 66)) + [131072, 1 << 20, 100_000_000, 0x7FFFFFFF]:
        for blocks in (0, 64, 22 * 2048):
            m, p = _pools(rules, nodes, num, den, blocks)
            assert CHUNK_M <= m <= POOL_MAX and CHUNK_P <= p <= POOL_MAX
            assert m >= blocks * CHUNK_M and p >= blocks * CHUNK_P
