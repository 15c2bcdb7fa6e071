// walk.hip -- on-device dual-tree walk emitting compact M2L and P2P lists.
//
// Replaces the host-driven level loop of OpenClSimulation::step
// (open_cl_simulation.cpp:81-98): find_interactions (interaction.cl:10-100),
// the host classification (open_cl_simulation.cpp:242-267), the per-node
// interaction counters (interaction.cl:104-154) and the host prefix sums
// (open_cl_simulation.cpp:371-484).
//
// The reference splits unordered pairs (A,B) from (root, root): a side with
// children is replaced by its children, a childless side by itself
// (interaction.cl:42-49, 58-59); pairs are approximated when
//   A != B  and  0.75 (d_A + d_B)^2 / |c_B - c_A|^2 < theta^2   (:63-79)
// and split further when not approximated and either side has children
// (:80-82).  Unsplit, unapproximated pairs are near-field (P2P).  Read as
// directed pairs (target <- source), the set of pairs is the same, and the
// candidates for target A at recursion depth s are
//   - A at level s:       expand(SL(parent(A)))
//   - leaf A above s:     expand(SL(A))        (A stays, the source splits)
// where SL(X) are the sources that X's pairs were split against and
// expand(B) = children(B) if B has children, else {B}.
//
// Rows and groups.  The walk runs one depth at a time.  A row is one target at
// one depth: rows of depth s are the level-s cells (in id order) followed by
// the leaves carried from depth s-1.  Every row of depth s-1 is a group: its
// candidate set expand(SL(row)) is shared by all of its targets at depth s --
// the cell's children, or the carried leaf itself.  One workgroup takes one
// group, each of its wavefronts a slice of the split list: a candidate is
// loaded once and classified against every target (up to 8); then count,
// reserve, write.  Each row's M2L, P2P and split entries land as contiguous
// segments carved from per-workgroup chunks of three pools; a node's rows are
// chained in depth order (first row = its level row, next = its carried row one
// depth deeper), and the force kernels follow the chain, so no compaction pass
// is needed.
//
// Each target's entries come out in ascending source id, chain order included:
// split lists are ascending, kept leaves (coarser levels) precede children,
// and deeper depths only add deeper (larger-id) sources.
//
// The MAC is evaluated exactly in integers (units of half the finest cell):
//   3 den^2 (d_A + d_B)^2 < 4 num^2 |c_B - c_A|^2,  theta = num/den.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace nbh {

__device__ __forceinline__ uint32_t depth_base(const Counters* C, int s) {
    uint32_t b = 0;
    for (int q = 0; q < s; ++q) b += C->level_count[q] + C->carried[q];
    return b;
}

// A workgroup's LDS cache of one split list (SL_CACHE entries at a time): the
// entry's node id, geometry and first child.  Loading it once, coalesced,
// leaves one global round trip (the children's geometry) per candidate chunk.
constexpr int SL_CACHE = 512;
constexpr int SL_FLY = 4;
struct SLCache {
    int4* geo;
    int* node;
    int* fc;
};

// Enumerate expand(SL) for the cached entries [lo, hi) of a split list (one
// wavefront's slice of a workgroup-shared cache); f(phase, valid, B, geo) is
// called once per chunk of 64 lanes (uniformly), in ascending candidate order:
// phase 0 the entries without children (kept as themselves), then phase 1 the
// children of the others, entry by entry.
template <typename F>
__device__ __forceinline__ void enumerate_slice(const WalkParams& W, const SLCache& cache, uint32_t lo, uint32_t hi,
                                                F&& f) {
    const int lane = lane_id();
    for (uint32_t e0 = lo; e0 < hi; e0 += WAVE) {
        const uint32_t e = e0 + lane;
        int B = -1;
        int4 gb = make_int4(0, 0, 0, 0);
        if (e < hi) {
            B = cache.node[e];
            gb = cache.geo[e];
        }
        const bool valid = B >= 0 && (gb.w >> 8) == 0;
        if (__ballot(valid) == 0) continue;
        f(0, valid, B, gb);
    }
    // children: 8 entries x 8 slots per chunk, SL_FLY chunks' cells loaded
    // before the first is classified (every lane loads, a lane without a child
    // node 0: a load under a branch is waited for at the branch's end, and each
    // chunk then pays a memory round trip of its own)
    const int c = lane & 7;
    for (uint32_t e0 = lo; e0 < hi; e0 += 8 * SL_FLY) {
        int C[SL_FLY];
        int4 g[SL_FLY];
#pragma unroll
        for (int k = 0; k < SL_FLY; ++k) {
            const uint32_t e = e0 + 8 * k + (lane >> 3);
            C[k] = -1;
            if (e < hi && c < (cache.geo[e].w >> 8)) C[k] = cache.fc[e] + c;
        }
#pragma unroll
        for (int k = 0; k < SL_FLY; ++k) g[k] = W.nodes.geo[max(C[k], 0)];
#pragma unroll
        for (int k = 0; k < SL_FLY; ++k)
            if (__ballot(C[k] >= 0)) f(1, C[k] >= 0, C[k], g[k]);
    }
}

// The call sequence of enumerate_slice, with the candidate ids only (no
// geometry loads): f(phase, valid, B).  The validity tests read the cache
// alone, so the calls match enumerate_slice's one for one.
template <typename F>
__device__ __forceinline__ void enumerate_slice_ids(const SLCache& cache, uint32_t lo, uint32_t hi, F&& f) {
    const int lane = lane_id();
    for (uint32_t e0 = lo; e0 < hi; e0 += WAVE) {
        const uint32_t e = e0 + lane;
        int B = -1;
        bool valid = false;
        if (e < hi) {
            B = cache.node[e];
            valid = B >= 0 && (cache.geo[e].w >> 8) == 0;
        }
        if (__ballot(valid) == 0) continue;
        f(0, valid, B);
    }
    const int c = lane & 7;
    for (uint32_t e0 = lo; e0 < hi; e0 += 8) {
        const uint32_t e = e0 + (lane >> 3);
        int C = -1;
        if (e < hi && c < (cache.geo[e].w >> 8)) C = cache.fc[e] + c;
        if (__ballot(C >= 0)) f(1, C >= 0, C);
    }
}

// Take n entries from a wave's chunk {next, end}, reserving a new chunk of
// max(n, chunk) entries from the pool when the current one is exhausted.
// Returns the first index, or 0xffffffff when the pool is full.
__device__ __forceinline__ uint32_t pool_take(uint2& ch, uint32_t n, uint32_t chunk, uint32_t* used,
                                              unsigned long long cap) {
    if (ch.x + n > ch.y || ch.y == 0) {
        const uint32_t want = n > chunk ? n : chunk;
        const uint32_t s0 = atomicAdd(used, want);
        if ((unsigned long long)s0 + want > cap) {
            ch = make_uint2(0, 0);
            return 0xffffffffu;
        }
        ch = make_uint2(s0, s0 + want);
    }
    const uint32_t r = ch.x;
    ch.x += n;
    return r;
}

// 64-target chunks of a leaf
__device__ __forceinline__ uint32_t target_chunks(int4 link) { return ((uint32_t)link.y + WAVE - 1) / WAVE; }

// Depth 0: one row per root (one per system), the candidate being the root
// itself: a childless root is its own P2P source, otherwise (root, root) is
// split.  One thread per root.
__global__ __launch_bounds__(64) void walk_root_kernel(WalkParams W) {
    Counters* C = W.C;
    if (C->overflow & OVF_NODES) return;  // a captured step's tree outgrew its node arrays
    const uint32_t n_roots = C->level_count[0];
    // (one workgroup) the pools start behind every workgroup's first chunks
    if (threadIdx.x == 0) {
        C->m2l_pool_used.v = W.blocks * POOL_CHUNK_M;
        C->p2p_pool_used.v = W.blocks * POOL_CHUNK_P;
        C->sl_used.v = W.blocks * POOL_CHUNK_S;
        // the same-level M2L kernel's lanes past their lists load entry 0 and
        // the node it names: it lies in a chunk that may stay empty
        if (W.m2l_pool_cap > 0) W.m2l_pool[0] = (int)C->level_off[0];
    }
    __syncthreads();
    // this thread's totals, added once at the end: an atomic a root on one line
    // is ~12 ns, 0.8 ms of 65,536 systems' each time
    unsigned long long p2p = 0, split = 0, near = 0;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n_roots; r += gridDim.x * blockDim.x) {
        if (r >= W.row_cap) {
            atomicOr(&C->overflow, (uint32_t)OVF_ROWS);
            continue;
        }
        const int A = (int)(C->level_off[0] + r);
        const bool leaf = (W.nodes.geo[A].w >> 8) == 0;
        W.row_first[A] = r;
        W.row_next[r] = NO_ROW;
        W.row_node[r] = A;
        W.row_m_start[r] = 0;
        W.row_m_cnt[r] = 0;
        W.row_mx_cnt[r] = 0;
        uint32_t pc = 0, ps = 0, sc = 0, ss = 0;
        if (leaf) {
            ps = atomicAdd(&C->p2p_pool_used.v, 1u);
            if (ps < W.p2p_pool_cap) {
                W.p2p_pool[ps] = A;
                pc = 1;
                ++p2p;
                near += target_chunks(W.nodes.link[A]);
            } else {
                atomicOr(&C->overflow, (uint32_t)OVF_P2P);
                ps = 0;
            }
        } else {
            ss = atomicAdd(&C->sl_used.v, 1u);
            if (ss < W.sl_cap) {
                W.sl[ss] = A;
                sc = 1;
                ++split;
            } else {
                atomicOr(&C->overflow, (uint32_t)OVF_SL);
                ss = 0;
            }
        }
        W.row_p_start[r] = ps;
        W.row_p_cnt[r] = pc;
        W.row_sl_start[r] = ss;
        W.row_sl_cnt[r] = sc;
    }
    p2p = wave_sum(p2p);
    split = wave_sum(split);
    near = wave_sum(near);
    if (threadIdx.x == 0) {
        LineTotals& tot = C->tot[0];
        atomicAdd(&tot.p2p, p2p);
        atomicAdd(&tot.split, split);
        atomicAdd(&tot.near_work, near);
    }
}

constexpr int MAXT = 8;  // targets per group: the children of one cell, by octant
// Calls of enumerate_slice per wavefront and group: a slice of at most
// SL_CACHE / NW entries (128 for four wavefronts) gives chunks of 64 kept
// entries (two) and chunks of the children of 8 (sixteen).
template <int NW>
constexpr int cat_calls() { return (SL_CACHE / NW + WAVE - 1) / WAVE + SL_CACHE / NW / 8; }

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int l) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}

// Per lane o < 8 (an octant): running entry counts of one phase by category.
struct CatCount {
    uint32_t m, x, p, s;  // M2L same level, M2L other level, P2P, split
};
// adds a chunk's entries: a the candidates that the lane's target accepts, of
// the valid ones v, with lb those that are leaves and sl those of the
// target's level
__device__ __forceinline__ void cat_add(CatCount& c, uint64_t a, uint64_t v, uint64_t lb, uint64_t sl, bool leaf) {
    const uint64_t near = v & ~a;
    const uint32_t m = __popcll(a & sl), pp = leaf ? __popcll(near & lb) : 0;
    c.m += m;
    c.x += __popcll(a) - m;
    c.p += pp;
    c.s += __popcll(near) - pp;
}

// Depth s >= 1: one workgroup of NW (4 or 8) wavefronts per group (row of
// depth s-1).  The group's split list is cached once for the workgroup and
// each wavefront classifies the candidates of a contiguous slice of it
// against all targets.  Pass 1 counts per (wavefront, phase, target,
// category); one reservation per pool is made for the group; every
// wavefront then writes its entries at offsets ordered phase-major,
// wavefront-minor, which is the order of one wavefront walking the whole
// list.  Lists longer than the cache (a coarse leaf beside a dense region
// keeps thousands of entries) are taken a cache at a time: pass 1 counts,
// pass 2 classifies each section again, the wavefronts' counts of the section
// giving their offsets.  Rows are taken with a fixed stride over the
// workgroups; their headers are read 64 at a time so rows without work (leaves
// with nothing left to split) cost one batched read.
//
// The criterion for the 8 targets of a cell: in units of half the finer cell
// of the pair the centre offset is (dx, dy, dz) for octant 0 and one or more
// of them less 2 for the others, so a candidate takes six squares, eight sums
// and eight compares with a threshold that depends on the level gap alone
// (floor of 3 den^2 (d_A + d_B)^2 / 4 num^2, exact).  Squares are 24-bit
// products in 32 bits where every offset of the chunk is small (rules.h; all but
// level gaps of ten and more, which take the 64-bit form).  A chunk's
// accepted candidates are one 64-bit mask per target; the categories follow
// from it and three masks of the candidates (valid, leaf, target's level) by
// scalar logic, and pass 2 replays the masks from LDS.
//
// Measured, a depth's kernel on average, against 64-bit offsets and a category
// per lane, candidate and target, 256 cached entries with longer lists walked
// by one wavefront, and every reservation an atomic: pair of 150,001 (theta =
// 0.4) 281 -> 129 us, Plummer 1,048,576 151 -> 120 us (beside the M2L), 5003
// 30 -> 20 us.  What is left of a heavy group (200 entries, 8 targets) at N =
// 30,011 is 2 us of loads, 5 of counts, 12 of writes alone on its CU, and up
// to 60 us where the CU's other groups are heavy too: the 4-byte list stores
// bound it (one store per target with the list chosen per lane took the same).
template <int NW>
__global__ __launch_bounds__(WAVE * NW) void walk_group_kernel(WalkParams W, int s) {
    __shared__ int4 cgeo[SL_CACHE];
    __shared__ int cnode[SL_CACHE];
    __shared__ int cfc[SL_CACHE];
    __shared__ CatCount cnt_s[NW][2][MAXT];       // [wave][phase][octant]
    __shared__ uint32_t bcast[8];                         // pool starts, carried row, failure
    __shared__ uint64_t mask_s[NW][cat_calls<NW>()][MAXT + 3];  // accepted by octant; valid, leaf, level
    __shared__ uint32_t thr_s[MAX_LEVELS];
    Counters* C = W.C;
    if (C->overflow & OVF_NODES) return;  // a captured step's tree outgrew its node arrays
    const uint32_t n_prev_level = C->level_count[s - 1];
    const uint32_t n_groups = n_prev_level + C->carried[s - 1];
    const uint32_t base_prev = depth_base(C, s - 1);
    const uint32_t base = base_prev + n_groups;
    const uint32_t n_level = C->level_count[s];
    const uint32_t loff = C->level_off[s], loff_prev = C->level_off[s - 1];
    const int lane = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const SLCache cache{cgeo, cnode, cfc};
    const uint32_t nblk = gridDim.x;
    if (threadIdx.x < MAX_LEVELS) thr_s[threadIdx.x] = W.thr[threadIdx.x];
    // lanes 0..2 of the first wavefront: the M2L, P2P and split pools
    const uint32_t pool_chunk = lane == 0 ? POOL_CHUNK_M : lane == 1 ? POOL_CHUNK_P : POOL_CHUNK_S;
    uint32_t* const pool_used = lane == 0   ? &C->m2l_pool_used.v
                                : lane == 1 ? &C->p2p_pool_used.v
                                            : &C->sl_used.v;
    const unsigned long long pool_cap = lane == 0 ? W.m2l_pool_cap : lane == 1 ? W.p2p_pool_cap : W.sl_cap;
    // the workgroup's first chunk of each pool is its own without asking: the
    // pools begin with one for every workgroup of every depth, and the
    // counters start behind them (walk_root_kernel).  At small sizes a
    // workgroup has one group, and a thousand of them reserving at once
    // waited up to 40 us for the counters.
    uint2 chunk;
    chunk.x = (W.first_block + blockIdx.x) * pool_chunk;
    chunk.y = chunk.x + pool_chunk;
    if (chunk.y > pool_cap) chunk = make_uint2(0, 0);
    // totals, lanes 0..4 of the first wavefront: M2L, P2P, split, M2L of other levels, near-field work
    unsigned long long acc = 0;
    for (uint64_t j0 = 0; (uint64_t)blockIdx.x + j0 * nblk < n_groups; j0 += WAVE) {
        // headers of the next 64 rows of this workgroup (identical in every wavefront)
        const uint64_t gl = (uint64_t)blockIdx.x + (j0 + lane) * nblk;
        int P_l = 0;
        int4 gp_l = make_int4(0, 0, 0, 0);
        uint32_t st_l = 0, sn_l = 0;
        bool live = false;
        if (gl < n_groups && base_prev + gl < W.row_cap) {  // rows past the cap were flagged when made
            const uint32_t g = (uint32_t)gl, rg = base_prev + g;
            P_l = g < n_prev_level ? (int)(loff_prev + g) : W.row_node[rg];
            gp_l = W.nodes.geo[P_l];
            st_l = W.row_sl_start[rg];
            sn_l = W.row_sl_cnt[rg];
            if ((unsigned long long)st_l + sn_l > W.sl_cap) sn_l = 0;  // only after an overflow
            live = (gp_l.w >> 8) > 0 || sn_l > 0;
        }
        for (uint64_t todo = __ballot(live); todo; todo &= todo - 1) {  // uniform over the workgroup
            const int jl = __ffsll((unsigned long long)todo) - 1;
            const uint32_t g = (uint32_t)(blockIdx.x + (j0 + jl) * nblk);
            const uint32_t rg = base_prev + g;
            const int P = __builtin_amdgcn_readlane(P_l, jl);
            const int gpx = __builtin_amdgcn_readlane(gp_l.x, jl), gpy = __builtin_amdgcn_readlane(gp_l.y, jl);
            const int gpz = __builtin_amdgcn_readlane(gp_l.z, jl), gpw = __builtin_amdgcn_readlane(gp_l.w, jl);
            const uint32_t sl_st = __builtin_amdgcn_readlane(st_l, jl);
            const uint32_t sl_n = __builtin_amdgcn_readlane(sn_l, jl);
            const int nch = gpw >> 8;
            int nt, A0;
            uint32_t row0 = 0;
            const int4 lp = W.nodes.link[P];
            if (nch > 0) {  // the cell's children: level-s rows in id order
                nt = nch;
                A0 = lp.z;
                row0 = base + (uint32_t)(A0 - (int)loff);
            } else {  // a leaf with sources left to split: carried to depth s (its row is taken below)
                nt = 1;
                A0 = P;
            }
            __syncthreads();  // the previous group is done with the cache, counts and broadcasts
            if ((unsigned long long)row0 + nt > W.row_cap) {
                // the host retries with more rows; rows that fit are left empty so
                // that the next depth reads only rows of this evaluation
                if (threadIdx.x == 0) atomicOr(&C->overflow, (uint32_t)OVF_ROWS);
                const uint32_t r = row0 + lane;
                if (wv == 0 && lane < nt && r < W.row_cap) {
                    W.row_node[r] = A0 + lane;
                    W.row_next[r] = NO_ROW;
                    W.row_m_start[r] = W.row_m_cnt[r] = W.row_mx_cnt[r] = 0;
                    W.row_p_start[r] = W.row_p_cnt[r] = 0;
                    W.row_sl_start[r] = W.row_sl_cnt[r] = 0;
                }
                continue;
            }
            // the split list, cached for the workgroup (a section of it at a
            // time if it is longer than the cache) and sliced over the wavefronts
            auto section = [&](uint32_t p0) -> uint32_t {  // entries cached
                const uint32_t pn = min((uint32_t)SL_CACHE, sl_n - p0);
                for (uint32_t k = threadIdx.x; k < pn; k += blockDim.x) {
                    const int B = W.sl[sl_st + p0 + k];
                    cache.node[k] = B;
                    cache.geo[k] = W.nodes.geo[B];
                    cache.fc[k] = W.nodes.link[B].z;
                }
                return pn;
            };
            // targets: lane o < 8 holds the child of octant o (of a carried leaf,
            // lane 0 the leaf): its index among the children, which are in
            // octant order, whether it is a leaf, and its 64-target chunks
            int tgt = 0;  // index | leaf << 3 | present << 4 | chunks << 5
            if (nch > 0) {
                int4 gt = make_int4(0, 0, 0, 0), lk = make_int4(0, 0, 0, 0);
                if (lane < nt) {
                    gt = W.nodes.geo[A0 + lane];
                    lk = W.nodes.link[A0 + lane];
                }
                const int oct = (gt.x & 1) << 2 | (gt.y & 1) << 1 | (gt.z & 1);
                // (lanes without a child push past the octants)
                tgt = __builtin_amdgcn_ds_permute((lane < nt ? oct : 8 + (lane & 31)) << 2,
                                                  lane | ((gt.w >> 8) == 0) << 3 | 1 << 4 | target_chunks(lk) << 5);
            } else {
                tgt = 1 << 3 | 1 << 4 | target_chunks(lp) << 5;
            }
            const bool pres_l = lane < (nch > 0 ? MAXT : 1) && (tgt >> 4 & 1);
            const bool leaf_l = tgt >> 3 & 1;
            const int t_l = tgt & 7;
            const uint32_t omask = __builtin_amdgcn_readfirstlane((uint32_t)__ballot(pres_l));
            const uint32_t leaves = omask & __builtin_amdgcn_readfirstlane((uint32_t)__ballot(leaf_l));
            const int lt_level = (gpw & 0xff) + (nch > 0 ? 1 : 0);
            // octant 0's centre, in half cells of the targets' level
            const int tx = nch > 0 ? 4 * gpx + 1 : 2 * gpx + 1, ty = nch > 0 ? 4 * gpy + 1 : 2 * gpy + 1;
            const int tz = nch > 0 ? 4 * gpz + 1 : 2 * gpz + 1;
            // the candidates that each octant's target accepts (lane o: octant o)
            auto accept = [&](uint64_t v, int4 gb) -> uint64_t {
                const int lb = gb.w & 0xff;
                const int sa = max(lb - lt_level, 0), sb = max(lt_level - lb, 0);
                const int dx = ((2 * gb.x + 1) << sb) - (tx << sa), dy = ((2 * gb.y + 1) << sb) - (ty << sa);
                const int dz = ((2 * gb.z + 1) << sb) - (tz << sa);
                const uint32_t thr = thr_s[sa + sb];
                const bool big = !walk_small(dx) || !walk_small(dy) || !walk_small(dz) || thr == 0xffffffffu;
                uint64_t a = 0;
                if (!(__ballot(big) & v)) {
                    const uint32_t x[2] = {(uint32_t)__mul24(dx, dx), (uint32_t)__mul24(dx - 2, dx - 2)};
                    const uint32_t y[2] = {(uint32_t)__mul24(dy, dy), (uint32_t)__mul24(dy - 2, dy - 2)};
                    const uint32_t z[2] = {(uint32_t)__mul24(dz, dz), (uint32_t)__mul24(dz - 2, dz - 2)};
#pragma unroll
                    for (int o = 0; o < MAXT; ++o) {
                        const uint64_t k = __ballot(x[o >> 2] + y[o >> 1 & 1] + z[o & 1] > thr) & v;
                        a = lane == o ? k : a;
                    }
                } else {
                    const uint64_t side = 2ull + (2ull << (sa + sb));
                    const uint64_t lhs = (uint64_t)W.den3 * side * side;
#pragma nounroll
                    for (int o = 0; o < MAXT; ++o) {
                        const int64_t ex = dx - (o >> 2) * 2, ey = dy - (o >> 1 & 1) * 2, ez = dz - (o & 1) * 2;
                        const uint64_t k = __ballot(lhs < (uint64_t)W.num4 * (uint64_t)(ex * ex + ey * ey + ez * ez)) & v;
                        a = lane == o ? k : a;
                    }
                }
                return a;
            };
            uint32_t pn = 0, lo = 0, hi = 0;
            auto slice = [&] {
                lo = (pn * wv) / NW;
                hi = (pn * (wv + 1)) / NW;
            };
            // counts of this wavefront's slice per phase (lane o: octant o), and
            // every call's masks, kept for the writes
            CatCount k0, k1;
            auto count_slice = [&] {
                int ncall = 0;  // uniform
                if (lo < hi)
                    enumerate_slice(W, cache, lo, hi, [&](int ph, bool valid, int B, int4 gb) {
                        const uint64_t v = __ballot(valid), lb = __ballot((gb.w >> 8) == 0);
                        const uint64_t sl = __ballot((gb.w & 0xff) == lt_level);
                        const uint64_t a = accept(v, gb);
                        if (ph == 0) cat_add(k0, a, v, lb, sl, leaf_l);
                        else cat_add(k1, a, v, lb, sl, leaf_l);
                        if (lane < MAXT + 3)
                            mask_s[wv][ncall][lane] = lane < MAXT ? a : lane == MAXT ? v : lane == MAXT + 1 ? lb : sl;
                        ++ncall;
                    });
            };
            auto write_slice = [&](CatCount& c0, CatCount& c1) {
                int k = 0;
                if (lo < hi)
                    enumerate_slice_ids(cache, lo, hi, [&](int ph, bool, int B) {
                        const uint64_t w = mask_s[wv][k][min(lane, MAXT + 2)];
                        ++k;
                        const uint64_t v = readlane64(w, MAXT), lb = readlane64(w, MAXT + 1), sl = readlane64(w, MAXT + 2);
                        CatCount c = ph == 0 ? c0 : c1;
#pragma nounroll
                        for (uint32_t om = omask; om; om &= om - 1) {
                            const int o = __ffs((int)om) - 1;  // uniform
                            const uint64_t a = readlane64(w, o), near = v & ~a;
                            const uint64_t bm = a & sl, bx = a & ~sl;
                            const uint64_t bp = (leaves >> o & 1) ? near & lb : 0ull, bs = near & ~bp;
                            auto put = [&](int* pool, uint32_t first, uint64_t b) {
                                if (__builtin_amdgcn_inverse_ballot_w64(b))
                                    pool[first + __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32),
                                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u))] = B;
                            };
                            if (bm) put(W.m2l_pool, __builtin_amdgcn_readlane(c.m, o), bm);
                            if (bx) put(W.m2l_pool, __builtin_amdgcn_readlane(c.x, o), bx);
                            if (bp) put(W.p2p_pool, __builtin_amdgcn_readlane(c.p, o), bp);
                            if (bs) put(W.sl, __builtin_amdgcn_readlane(c.s, o), bs);
                        }
                        cat_add(c, w, v, lb, sl, leaf_l);
                        (ph == 0 ? c0 : c1) = c;
                    });
            };
            // one section: counted, reserved for, written.  More: all of them
            // counted (their sums in k0, k1), reserved for, then each counted
            // again and written.  b0, b1: where the section's entries of each
            // phase start in lane o's segments (phase 1 after all of phase 0)
            const uint32_t ns = max(1u, (sl_n + SL_CACHE - 1) / SL_CACHE), steps = ns == 1 ? 1 : 2 * ns;
            CatCount b0{0, 0, 0, 0}, b1{0, 0, 0, 0};
            k0 = k1 = CatCount{0, 0, 0, 0};
            for (uint32_t step = 0; step < steps; ++step) {
                if (step) __syncthreads();  // the cache and the counts are free
                pn = section((step < ns ? step : step - ns) * SL_CACHE);
                __syncthreads();
                slice();
                if (step >= ns) k0 = k1 = CatCount{0, 0, 0, 0};
                count_slice();
                if (step + 1 < ns) continue;
                if (lane < MAXT) {
                    cnt_s[wv][0][lane] = k0;
                    cnt_s[wv][1][lane] = k1;
                }
                __syncthreads();
                if (step + 1 == ns) {
                    // per octant (lane o): totals, of phase 0 and of both
                    CatCount T{0, 0, 0, 0}, Z{0, 0, 0, 0};
                    if (pres_l) {
#pragma unroll
                        for (int ph = 0; ph < 2; ++ph) {
#pragma unroll
                            for (int w = 0; w < (int)NW; ++w) {
                                const CatCount k = cnt_s[w][ph][lane];
                                T.m += k.m; T.x += k.x; T.p += k.p; T.s += k.s;
                            }
                            if (ph == 0) Z = T;
                        }
                    }
                    // totals of the group and segment starts of lane o's target:
                    // inclusive prefixes over lanes 0..7; a row's M2L segment holds
                    // its same-level sources, then the others
                    uint32_t em = T.m + T.x, ep = T.p, es = T.s, ex = T.x;
#pragma unroll
                    for (int o = 1; o < MAXT; o <<= 1) {
                        const uint32_t ym = __shfl_up(em, o, WAVE), yp = __shfl_up(ep, o, WAVE);
                        const uint32_t ys = __shfl_up(es, o, WAVE), yx = __shfl_up(ex, o, WAVE);
                        if (lane >= o) { em += ym; ep += yp; es += ys; ex += yx; }
                    }
                    const uint32_t tm = __builtin_amdgcn_readlane(em, MAXT - 1);
                    const uint32_t tp = __builtin_amdgcn_readlane(ep, MAXT - 1);
                    const uint32_t ts = __builtin_amdgcn_readlane(es, MAXT - 1);
                    // (here, with every lane active: under a condition on the lane the
                    // last sums of lane 7 may be left out)
                    const uint32_t tx = __builtin_amdgcn_readlane(ex, MAXT - 1);
                    // reserve one block per pool for all targets of the group (lanes
                    // 0..2 of the first wavefront, a pool each) and a carried leaf's
                    // row (lane 3): the atomics go out together
                    if (wv == 0) {
                        // (only leaves have P2P entries)
                        unsigned long long near = (unsigned long long)((uint32_t)tgt >> 5) * ((T.p + WAVE - 1) / WAVE);
#pragma unroll
                        for (int o = 1; o < MAXT; o <<= 1) near += __shfl_xor(near, o, WAVE);
                        const uint32_t need = lane == 0 ? tm : lane == 1 ? tp : lane == 2 ? ts : 0u;
                        const uint32_t ovf = lane == 0 ? OVF_M2L : lane == 1 ? OVF_P2P : OVF_SL;
                        uint32_t at = 0;
                        if (need) {
                            at = pool_take(chunk, need, pool_chunk, pool_used, pool_cap);
                            if (at == 0xffffffffu) atomicOr(&C->overflow, ovf);
                        }
                        if (lane == 3 && nch == 0) {
                            at = base + n_level + atomicAdd(&C->carried[s], 1u);
                            if (at >= W.row_cap) {  // (no row to leave empty)
                                atomicOr(&C->overflow, (uint32_t)OVF_ROWS);
                                at = 0xffffffffu;
                            }
                        }
                        const bool fail = __ballot(lane < 4 && at == 0xffffffffu) != 0;
                        if (!fail) acc += lane == 3 ? tx : lane == 4 ? near : need;
                        if (lane < 4) bcast[lane] = at;
                        if (lane == 4) bcast[4] = fail;
                    }
                    __syncthreads();
                    if (nch == 0) row0 = bcast[3];
                    if (row0 == 0xffffffffu) break;  // uniform: no row left for the carried leaf
                    const bool fail = bcast[4] != 0;
                    const uint32_t m0 = bcast[0] + em - (T.m + T.x), p0 = bcast[1] + ep - T.p, s0 = bcast[2] + es - T.s;
                    if (wv == 0 && pres_l) {
                        const uint32_t r = row0 + t_l;
                        W.row_node[r] = A0 + t_l;
                        W.row_next[r] = NO_ROW;
                        W.row_m_start[r] = fail ? 0u : m0;
                        W.row_m_cnt[r] = fail ? 0u : T.m + T.x;
                        W.row_mx_cnt[r] = fail ? 0u : T.x;
                        W.row_p_start[r] = fail ? 0u : p0;
                        W.row_p_cnt[r] = fail ? 0u : T.p;
                        W.row_sl_start[r] = fail ? 0u : s0;
                        W.row_sl_cnt[r] = fail ? 0u : T.s;
                        if (nch > 0) W.row_first[A0 + t_l] = r;
                    }
                    if (nch == 0 && threadIdx.x == 0) W.row_next[rg] = row0;
                    if (fail || !(tm | tp | ts)) break;  // uniform; the host retries after a failure
                    b0 = CatCount{m0, m0 + T.m, p0, s0};
                    b1 = CatCount{m0 + Z.m, m0 + T.m + Z.x, p0 + Z.p, s0 + Z.s};
                    if (ns > 1) continue;
                }
                CatCount c0{0, 0, 0, 0}, c1{0, 0, 0, 0};  // this wavefront's next positions
                if (pres_l) {
#pragma unroll
                    for (int w = 0; w < (int)NW; ++w) {
                        if (w == wv) { c0 = b0; c1 = b1; }
                        const CatCount u0 = cnt_s[w][0][lane], u1 = cnt_s[w][1][lane];
                        b0.m += u0.m; b0.x += u0.x; b0.p += u0.p; b0.s += u0.s;
                        b1.m += u1.m; b1.x += u1.x; b1.p += u1.p; b1.s += u1.s;
                    }
                }
                write_slice(c0, c1);
            }
        }
    }
    if (threadIdx.x < 5 && acc) {
        LineTotals& tot = C->tot[blockIdx.x % CNT_COPIES];
        atomicAdd(lane == 0   ? &tot.m2l
                  : lane == 1 ? &tot.p2p
                  : lane == 2 ? &tot.split
                  : lane == 3 ? &tot.m2lx
                              : &tot.near_work,
                  acc);
    }
}

void walk_thresholds(uint32_t num4, uint32_t den3, uint32_t* thr) {
    for (int g = 0; g < MAX_LEVELS; ++g) thr[g] = walk_threshold(num4, den3, g);
}

void launch_walk_root(const WalkParams& W, hipStream_t st) {
    hipLaunchKernelGGL(walk_root_kernel, dim3(1), dim3(64), 0, st, W);
}
uint32_t walk_group_resident_blocks(int num_cu) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(&walk_group_kernel<4>),
                                                     WAVE * 4, 0) != hipSuccess ||
        per_cu < 1)
        per_cu = 1;
    return (uint32_t)per_cu * (uint32_t)(num_cu > 0 ? num_cu : 1);
}
// A depth with at most two groups a compute unit lasts as long as its heaviest
// group, which eight wavefronts finish sooner than four (N = 5003, a depth's
// kernel on average 19.1 -> 17.5 us, the two longest 34 -> 26 us).  With more
// groups they only hold each other up: N = 30,011, all depths with four
// wavefronts 26.4 us, with eight 29.8, by this rule 25.9.
void launch_walk_group(const WalkParams& W, int s, uint32_t grid, hipStream_t st) {
    if (grid <= WALK_WIDE) hipLaunchKernelGGL(walk_group_kernel<8>, dim3(grid), dim3(WAVE * 8), 0, st, W, s);
    else hipLaunchKernelGGL(walk_group_kernel<4>, dim3(grid), dim3(WAVE * 4), 0, st, W, s);
}

}  // namespace nbh
