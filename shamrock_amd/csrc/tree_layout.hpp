// SPDX-License-Identifier: CeCILL-2.1
//
// tree_layout.hpp -- 64-byte node records of the compressed-leaf BVH (one record per cell,
// internal cells first, then leaves, as in the reference's total cell numbering
// KarrasTreeTraverser.hpp:55-66).
//   [0..2] aabb min  [3..5] aabb max  [6] rint = max h * htol
//   [7] internal: (left total id, right total id) ; leaf: (first, end) in sorted order
#pragma once

#include "common.hpp"

namespace shamx {

    constexpr int NODE_F64 = 8;

    __host__ __device__ inline void node_pack(f64 *nodes, u32 node, u32 a, u32 b) {
        u32 *w = (u32 *) (nodes + (u64) node * NODE_F64 + 7);
        w[0]   = a;
        w[1]   = b;
    }
    __host__ __device__ inline void node_set_children(f64 *nodes, u32 node, u32 l, u32 r) {
        node_pack(nodes, node, l, r);
    }
    __host__ __device__ inline void node_set_range(f64 *nodes, u32 node, u32 s0, u32 s1) {
        node_pack(nodes, node, s0, s1);
    }
    __host__ __device__ inline void node_children(const f64 *nodes, u32 node, u32 &l, u32 &r) {
        const u32 *w = (const u32 *) (nodes + (u64) node * NODE_F64 + 7);
        l            = w[0];
        r            = w[1];
    }

    // Tiers over the leaves: tier 0 are the leaves (in Morton order), cell j of tier t holds the
    // cells [8 j, 8 j + 8) of tier t - 1 (box and largest rint; the records above), up to a tier
    // of at most 64 cells.  Eight leaves of a run are about one octant, the children of a cell
    // are one contiguous read, and a leaf range is a handful of cells per tier.
    constexpr u32 TIER_MAX = 10; // 64 * 8^10 leaves
    struct Tiers {
        u32 top = 0;               // index of the top tier
        u32 n[TIER_MAX + 1] = {};   // cells per tier; n[0] leaves
        u32 off[TIER_MAX + 1] = {}; // first record of a tier (tier 0: the tree's leaves)
    };
    struct Cell {
        f64 lo[3], hi[3], r;
    };
    __device__ inline Cell cell_load(const f64 *__restrict rec) {
        return Cell{{rec[0], rec[1], rec[2]}, {rec[3], rec[4], rec[5]}, rec[6]};
    }
    constexpr f64 F64_BIG = 1.7976931348623157e308;
    __device__ inline Cell cell_none() {
        // (a reach of -inf: a leaf whose lengths are all NaN has it, and keeps it in its cells)
        return Cell{{F64_BIG, F64_BIG, F64_BIG}, {-F64_BIG, -F64_BIG, -F64_BIG},
                    -__builtin_inf()};
    }
    __device__ inline void cell_merge(Cell &c, const Cell &o) {
        for (int k = 0; k < 3; k++) {
            c.lo[k] = fmin(c.lo[k], o.lo[k]);
            c.hi[k] = fmax(c.hi[k], o.hi[k]);
        }
        c.r = fmax(c.r, o.r);
    }
    // union over the lanes whose index differs in the bits o
    __device__ inline void cell_merge_xor(Cell &c, int o) {
        Cell t;
        for (int k = 0; k < 3; k++) {
            t.lo[k] = __shfl_xor(c.lo[k], o, WAVE);
            t.hi[k] = __shfl_xor(c.hi[k], o, WAVE);
        }
        t.r = __shfl_xor(c.r, o, WAVE);
        cell_merge(c, t);
    }

} // namespace shamx
