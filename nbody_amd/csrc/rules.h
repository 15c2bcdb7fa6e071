// rules.h -- the host's sizing rules, in plain C++ (no HIP) so that they can be
// compiled and checked on the CPU.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>

namespace nbh {

// Chunk sizes of the walk's segment pools (entries).  A workgroup starts with
// a chunk of its own, reserves more with one atomic each and carves row
// segments from them; the host sizes the pools for one unused tail per
// workgroup and depth.
constexpr uint32_t POOL_CHUNK_M = 2048, POOL_CHUNK_P = 512, POOL_CHUNK_S = 512;
// the most entries of a pool (its counter has 32 bits)
constexpr unsigned long long POOL_MAX = 0xffff0000ull;

// First sizes (entries) of the M2L and P2P pools for `nodes` cells walked by
// `blocks` workgroups at theta = num / den: a cell keeps about 1000 M2L and
// 230 P2P sources at theta = 1/2, in proportion to 1/theta^3, and no more than
// there are cells.  One chunk at least, whatever the tree and theta: the
// walk's first kernel stores entry 0 of the M2L pool, also of a tree without
// a list (one cell, no workgroup of the walk), where the product below is less
// than one entry from theta = 5.1 on.
struct PoolSizes {
    unsigned long long m2l, p2p;
};
inline PoolSizes pool_guess(uint32_t nodes, int num, int den, unsigned long long blocks) {
    const double near = std::pow(0.5 * den / num, 3.0);
    auto pool = [&](double per_cell, uint32_t chunk) {
        const double entries = nodes * std::min((double)nodes, per_cell * near);
        const unsigned long long want =
            (unsigned long long)std::min(entries, (double)POOL_MAX) + blocks * chunk;
        return std::min(std::max<unsigned long long>(want, chunk), POOL_MAX);
    };
    return {pool(1024.0, POOL_CHUNK_M), pool(256.0, POOL_CHUNK_P)};
}

}  // namespace nbh
