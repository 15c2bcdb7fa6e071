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

// The walk's criterion 3 den^2 (d_A + d_B)^2 < 4 num^2 |c_B - c_A|^2 in units of
// half the finer cell of the pair, `gap` levels apart: the largest squared
// centre offset that it does not accept, 3 den^2 (2 + 2 2^gap)^2 / 4 num^2
// rounded down (2^32 - 1: not below 2^32 - 1).
constexpr uint32_t walk_threshold(uint32_t num4, uint32_t den3, int gap) {
    const uint64_t side = 2ull + (2ull << gap);
    return (uint32_t)std::min<uint64_t>((uint64_t)den3 * side * side / num4, 0xffffffffu);
}
// Offsets of octant 0's centre whose squares, and those of the other octants'
// (2 less), are products of 24 bits with a sum of three in 32 bits.
constexpr int WALK_SMALL = 32000;
constexpr bool walk_small(int d) { return (uint32_t)(d + WALK_SMALL) <= 2u * WALK_SMALL; }
static_assert(WALK_SMALL + 2 < 1 << 23 && 3ull * (WALK_SMALL + 2) * (WALK_SMALL + 2) < 1ull << 32, "squares fit");

// First sizes (entries) of the M2L and P2P pools for `nodes` cells of a handle
// whose largest system holds max_sys_n of its n particles, walked by `blocks`
// workgroups at theta = num / den.  A cell keeps about 1000 M2L and 230 P2P
// sources at theta = 1/2, in proportion to 1/theta^3, and no more than its own
// system has cells or, since a cell's sources are disjoint, particles.  What
// theta < 1/2 adds stays within POOL_GUESS_MAX: a pool that is too small is
// grown after the walk, which is then repeated.  `small`: 256 and 64 sources a
// cell, for a device without room for more.  One chunk at least, whatever the
// tree and theta: the walk's first kernel stores entry 0 of the M2L pool, also
// of a tree without a list (one cell, no workgroup of the walk), where the
// product below is less than one entry from theta = 5.1 on.
constexpr double POOL_GUESS_MAX = 1u << 29;  // entries, 2 GiB
struct PoolSizes {
    unsigned long long m2l, p2p;
};
inline PoolSizes pool_guess(uint32_t nodes, uint32_t max_sys_n, uint64_t n, int num, int den,
                            unsigned long long blocks, bool small) {
    const double near = std::pow(0.5 * den / num, 3.0);
    const double cells = std::min(std::ceil((double)nodes * max_sys_n / n), (double)max_sys_n);
    auto pool = [&](double usual, double few, uint32_t chunk) {
        const double at_half = nodes * std::min(cells, usual * std::min(near, 1.0));
        const double at_theta = nodes * std::min(cells, usual * near);
        const double entries =
            small ? nodes * std::min(cells, few) : std::max(at_half, std::min(at_theta, POOL_GUESS_MAX));
        const unsigned long long want =
            (unsigned long long)std::min(entries, (double)POOL_MAX) + blocks * chunk;
        return std::min(std::max<unsigned long long>(want, chunk), POOL_MAX);
    };
    return {pool(1024.0, 256.0, POOL_CHUNK_M), pool(256.0, 64.0, POOL_CHUNK_P)};
}

// Near field: batches (of up to 64 entries of a row of a P2P list) that a list
// is cut towards, and the most partial-sum slots.  A leaf of nb batches and tc
// chunks of 64 targets is cut if nb > G, into k = ceil(nb / G) items a chunk,
// and takes tc k slots.  G keeps an item near 1 / NEAR_BATCHES of all batches
// (entries / 64), and the slots of every leaf within `slots` whatever the
// lists: with work = the sum of tc nb over the leaves, G = 1 takes at most work
// slots, and G > 1 at most 2 work / (G + 1), since k <= 2 nb / (G + 1) for nb >
// G.  So which lists are cut depends on the tree and the lists alone.  (Half as
// many slots cut large leaves less: a step of N = 300,000 at capacity 512 7.9 ms
// instead of 7.2, of 400,000 9.6 instead of 9.0.)
constexpr uint32_t NEAR_BATCHES = 16384, NEAR_SLOTS = 4 * NEAR_BATCHES;
constexpr uint32_t NEAR_WHOLE = 0x7fffffffu;  // more batches than any list has
constexpr uint32_t near_item_batches(uint64_t entries, uint64_t work, uint32_t slots) {
    const uint64_t by_size = (entries / 64 + NEAR_BATCHES - 1) / NEAR_BATCHES;
    const uint64_t by_slots = (2 * work + slots - 1) / slots;  // G + 1
    const uint64_t g = by_slots > by_size + 1 ? by_slots - 1 : by_size;
    return (uint32_t)(g < 1 ? 1 : g > NEAR_WHOLE ? NEAR_WHOLE : g);
}
// at least the slots that are then taken
constexpr uint64_t near_slots_bound(uint64_t entries, uint64_t work, uint32_t slots) {
    const uint64_t g = near_item_batches(entries, work, slots);
    return g == 1 ? work : g == NEAR_WHOLE ? 0 : 2 * work / (g + 1);
}

}  // namespace nbh
