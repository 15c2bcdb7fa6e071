// near.h -- near-field work items (launch.h: NearItem) as the near-field
// kernels and the kernels that join their sums see them.
#pragma once

#include "common.h"
#include "launch.h"

namespace nbh {

// The items of an evaluation: those of the leaves that were cut first (they
// stand at their slots), then the others'.  None if a captured step's tree or
// walk outgrew its buffers.  An item with b1 = 0 is empty.
struct NearCount {
    uint32_t cut, uncut;
};
__device__ __forceinline__ NearCount near_count(const FmmParams& F) {
    if (F.C->overflow & OVF_WALK) return NearCount{0, 0};
    const unsigned long long u = F.C->near_used;
    return NearCount{(uint32_t)(u >> 32), (uint32_t)u};
}
__device__ __forceinline__ NearItem near_item(const FmmParams& F, const NearCount& c, uint32_t w) {
    return F.near_items[w < c.cut ? w : F.near_slot_cap + (w - c.cut)];
}

// f(first, end) for batches [b0, b1) of node A's P2P list: a batch is the (up
// to 64) entries from `first` on, below `end`, the end of its row.
template <typename F>
__device__ __forceinline__ void near_batches(const ListView& lists, int A, uint32_t b0, uint32_t b1, F&& f) {
    uint32_t b = 0;  // batches before row r
    for (uint32_t r = lists.first[A]; r != NO_ROW && b < b1; r = lists.next[r]) {
        const uint32_t st = lists.p_start[r], cnt = lists.p_cnt[r];
        const uint32_t nb = (cnt + WAVE - 1) / WAVE;
        const uint32_t lo = b0 > b ? b0 - b : 0u, hi = min(nb, b1 - b);
        for (uint32_t k = lo; k < hi; ++k) f(st + k * WAVE, st + cnt);
        b += nb;
    }
}

// The near field of particle i of leaf A where the leaf's list was cut: the
// sum of its items' partial sums, in item order.  False: it was not cut (or
// the evaluation was stood down before the lists were).
__device__ __forceinline__ bool near_partial_sum(const FmmParams& F, uint32_t A, uint32_t i, float4& sum) {
    if (!F.near_items || (F.C->overflow & OVF_WALK)) return false;
    const uint32_t k = F.near_k[A];
    if (k <= 1) return false;
    const uint32_t o = i - (uint32_t)F.nodes.link[A].x;
    const float4* p = F.near_part + ((size_t)F.near_first[A] + (size_t)(o / WAVE) * k) * WAVE + o % WAVE;
    sum = p[0];
    // (a leaf may be cut into hundreds of items: eight loads in flight)
#pragma unroll 8
    for (uint32_t j = 1; j < k; ++j) {
        const float4 v = p[(size_t)j * WAVE];
        sum.x += v.x;
        sum.y += v.y;
        sum.z += v.z;
        sum.w += v.w;
    }
    return true;
}

}  // namespace nbh
