// SPDX-License-Identifier: CeCILL-2.1
//
// neigh.hip -- two-stage neighbour cache (NeighbourCache::start_neighbors_cache_2stages,
// shammodels/sph/src/modules/NeighbourCache.cpp:222-604).
//   stage 1: per leaf, the list of interacting leaves (:276-404), by a search over the tiers of the
//            leaves
//   owner  : per local particle, the LAST leaf in depth-first order whose box contains it
//            (inclusive max, :406-451)
//   stage 2: per local particle, candidates of the owner's neighbour leaves kept when
//            r_ab^2 <= max(rint_a, rint_b)^2 R^2 with rint = h * htol (:465-590)
// The solver's lists are written in one pass into rows of fixed capacity, longer ones again into
// an overflow region; the phase entry's (and rows that u32 indices cannot address that way) in a
// count pass, a scan and a fill pass.  Either way a list holds its entries in the order of the
// reference's walk, left child first (KarrasTreeTraverser.hpp:69-118), which is that of the leaf
// index: lists and their order are deterministic and the reference's.
#include "compact.hpp"
#include "launch.hpp"
#include "tree_layout.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace shamx {

    namespace {
        // orders the LDS accesses of one wave's lanes around this point (LDS executes a wave's
        // operations in issue order; the fences keep the compiler from moving them across)
        __device__ inline void wave_lds_sync() {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }

        // ------------------------------------------------------------- stage 1
        // A leaf's list (:276-404) holds the leaves n whose box meets its box widened by its
        // reach, or whose widened box meets its box; the reference finds them by a depth-first
        // walk of the Karras tree with the same criterion on every cell.  A cell's box and reach
        // hold those of all leaves below it and the criterion is monotone in both (rounding
        // included), so a leaf is reached exactly when it passes itself, and left-first order is
        // the order of the leaf index.  Any search that tests every leaf that can pass, in index
        // order, therefore gives the reference's list.
        //
        // The search runs over the tiers of the tree (tree_layout.hpp): the number of dependent
        // steps is log8 of the leaf count.
        // boxes [alo, ahi] and [blo, bhi] meet (BBAA::cella_neigh_b, geometry_utils.hpp:125-135:
        // max of the lower bounds <= min of the upper ones; a NaN bound never separates, there
        // as here)
        __device__ inline bool boxes_meet(const f64 *alo, const f64 *ahi, const f64 *blo,
                                          const f64 *bhi) {
            return !((alo[0] > bhi[0]) | (blo[0] > ahi[0]) | (alo[1] > bhi[1]) |
                     (blo[1] > ahi[1]) | (alo[2] > bhi[2]) | (blo[2] > ahi[2]));
        }
        // a box that its reach r, below zero, shrinks past a point meets none
        __device__ inline void close_shrunk(f64 r, f64 *lo, f64 *hi) {
            if (r < 0 && ((lo[0] > hi[0]) | (lo[1] > hi[1]) | (lo[2] > hi[2])))
                lo[0] = __builtin_inf(), hi[0] = -__builtin_inf();
        }

        // One wave finds the lists of eight consecutive leaves (the targets).  Per tier it keeps a
        // first-in first-out queue in LDS of the cells that pass the criterion of the targets'
        // common box, and takes eight cells of one tier at a time, their 64 children in the
        // lanes; it takes from the lowest tier that has eight, else from the highest that has
        // any, so a queue never holds more than 8 + 64 entries (tier 0: 64 + 64) and every queue
        // stays in index order.  Leaves leave tier 0 64 at a time: a lane holds a leaf, the
        // targets are tested one after the other with the reference's criterion, and a target's
        // list grows by the lanes of its ballot, in order.
        //
        // Eight targets share the search while their common box is tight.  A run of leaves that
        // crosses a boundary of the Morton curve, or holds one leaf of large reach, has a common
        // box that meets far more leaves than its members do, so a group is halved while the
        // halves are cheaper: per leaf met the search costs about 80 lane instructions and each
        // target 30, so a group of T with box volume V against V1 and V2 of its halves splits
        // when (80 + 30 T) V > (80 + 15 T) (V1 + V2).
        //
        // Bound by instruction issue (first steps of Sedov 128^3: 3410 VALU and 2010 scalar
        // instructions per wave, 60 % of the VALU issue peak, 16 % of wave time waiting).  It
        // replaces a depth-first walk of the binary tree shared by 64 leaves per wave, a chain of
        // about 1000 dependent record loads.  Per build: Sedov 128^3 (391 k leaves) 1.54 -> 0.62 ms,
        // disc of 1 M particles 4.06 -> 0.78 ms, Plummer sphere of 4.2 M 1.54 -> 0.68 ms,
        // M8 box of 39 k 1.21 -> 0.09 ms, 1,728 particles 0.39 -> 0.04 ms; without the
        // halving of loose groups the first three take 1.87, 5.8 and 9.4 ms.
        //
        // COUNT: list lengths only.  ROWS: leaf g's list at ids[g * cap], at most cap entries
        // written, the count going on past it.  FILL: at ids[offset[g]].  LIST: the targets
        // are the leaves of `list`, one per wave.  lap[g] (COUNT and ROWS) says whether a later
        // leaf's box meets leaf g's box, which is what can make that leaf own one of its
        // particles.
        enum LeafOut { LEAF_COUNT, LEAF_ROWS, LEAF_FILL };
        constexpr int LW_WAVES = 4, LQ_CAP = 128;
        constexpr u32 LEAF_TGT = 8;
        template<int OUT, bool LIST>
        __global__ void __launch_bounds__(LW_WAVES *WAVE)
            k_leaf_lists(u32 L, u32 I, const f64 *__restrict nodes, const f64 *__restrict tiers,
                         Tiers tt, f64 Rkern, u32 *__restrict cnt, u32 *__restrict offset,
                         u32 *__restrict ids, u32 cap, u32 *__restrict lap,
                         const u32 *__restrict list, u32 n_list) {
            constexpr u32 T = LIST ? 1 : LEAF_TGT;
            __shared__ u32 queue[LW_WAVES][TIER_MAX + 1][LQ_CAP];
            __shared__ f64 tgt[LW_WAVES][T][12]; // box and widened box of every target
            const u32 lane = (u32) __lane_id();
            const u32 wid  = (u32) __builtin_amdgcn_readfirstlane((int) (threadIdx.x / WAVE));
            const u32 item = blockIdx.x * LW_WAVES + wid;
            if (item >= (LIST ? n_list : (L + T - 1) / T)) return;
            const u32 g0 =
                LIST ? (u32) __builtin_amdgcn_readfirstlane((int) list[item]) : item * T;
            const u32 nt = LIST ? 1u : min(T, L - g0);
            const u64 lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
            u32(*q)[LQ_CAP] = queue[wid];
            auto at = [](u32 v, u32 l) { return (u32) __builtin_amdgcn_readlane((int) v, (int) l); };
            // lane t (< nt): target t, its list's length and first entry, the size of the group
            // that it is searched in
            u32 len = 0, base = 0, laps = 0, size = T;
            {
                Cell wide = cell_none();
                if (lane < nt) {
                    const Cell c = cell_load(nodes + (u64) (I + g0 + lane) * NODE_F64);
                    const f64 r  = c.r * Rkern;
                    f64 *m       = tgt[wid][lane];
                    for (int k = 0; k < 3; k++) {
                        wide.lo[k] = c.lo[k] - r;
                        wide.hi[k] = c.hi[k] + r;
                    }
                    close_shrunk(r, wide.lo, wide.hi);
                    for (int k = 0; k < 3; k++) {
                        m[k]       = c.lo[k];
                        m[3 + k]   = c.hi[k];
                        m[6 + k]   = wide.lo[k];
                        m[9 + k]   = wide.hi[k];
                    }
                    if (OUT == LEAF_ROWS) base = (g0 + lane) * cap;
                    if (OUT == LEAF_FILL) base = offset[g0 + lane];
                }
                if (!LIST) {
                    auto vol = [](const Cell &c) {
                        f64 v = 1;
                        for (int k = 0; k < 3; k++) v *= fmax(c.hi[k] - c.lo[k], 0.);
                        return v;
                    };
                    f64 v = vol(wide);
                    bool split[3];
#pragma unroll
                    for (int b = 0; b < 3; b++) { // groups of 2, 4, 8
                        const f64 parts = v + __shfl_xor(v, 1 << b, WAVE);
                        cell_merge_xor(wide, 1 << b);
                        v           = vol(wide);
                        const f64 t = (f64) (2 << b);
                        split[b]    = (80. + 30. * t) * v > (80. + 15. * t) * parts;
                    }
                    for (int b = 2; b >= 0 && split[b]; b--) size = 1u << b;
                }
            }
            // queue state of tier t in lane t: entries and position of the first
            u32 qn = 0, qh = 0;
            f64 ulo[3], uhi[3], elo[3], ehi[3]; // the group's common box and widened box
            // the cells of tier t in the lanes (on: this lane has one) that pass for the group
            // go to the tier's queue
            auto sift = [&](u32 t, u32 cell, bool on) {
                bool pass = false;
                if (on) {
                    const f64 *rec = t ? tiers + (u64) (tt.off[t] + cell) * NODE_F64
                                       : nodes + (u64) (I + cell) * NODE_F64;
                    const Cell b   = cell_load(rec);
                    const f64 r    = b.r * Rkern;
                    const f64 xlo[3] = {b.lo[0] - r, b.lo[1] - r, b.lo[2] - r};
                    const f64 xhi[3] = {b.hi[0] + r, b.hi[1] + r, b.hi[2] + r};
                    pass = boxes_meet(ulo, uhi, xlo, xhi) | boxes_meet(elo, ehi, b.lo, b.hi);
                }
                const u64 m = __ballot(pass);
                const u32 p = at(qh + qn, t);
                if (pass) q[t][(p + (u32) __popcll(m & lt)) % LQ_CAP] = cell;
                if (lane == t) qn += (u32) __popcll(m);
                wave_lds_sync();
            };
            // up to 64 leaves of tier 0 against the targets [t0, t1)
            auto leaves = [&](u32 t0, u32 t1) {
                const u32 n   = min(at(qn, 0), (u32) WAVE);
                const u32 h0  = at(qh, 0);
                const bool on = lane < n;
                const u32 g   = on ? q[0][(h0 + lane) % LQ_CAP] : 0u;
                if (lane == 0) qh += n, qn -= n;
                const Cell b = cell_load(nodes + (u64) (I + g) * NODE_F64);
                const f64 r  = b.r * Rkern;
                f64 xlo[3] = {b.lo[0] - r, b.lo[1] - r, b.lo[2] - r};
                f64 xhi[3] = {b.hi[0] + r, b.hi[1] + r, b.hi[2] + r};
                close_shrunk(r, xlo, xhi);
                const bool later =
                    OUT != LEAF_FILL &&
                    __ballot(on & (g > g0 + t0) & boxes_meet(ulo, uhi, b.lo, b.hi)) != 0;
                for (u32 t = t0; t < t1; t++) {
                    const f64 *a = tgt[wid][t];
                    const bool pass =
                        on & (boxes_meet(a, a + 3, xlo, xhi) | boxes_meet(a + 6, a + 9, b.lo, b.hi));
                    const u64 m = __ballot(pass);
                    if (OUT != LEAF_COUNT && pass) {
                        const u32 p = at(len, t) + (u32) __popcll(m & lt);
                        if (OUT == LEAF_FILL || p < cap) ids[at(base, t) + p] = I + g;
                    }
                    if (lane == t) len += (u32) __popcll(m);
                    if (later && __ballot(on & (g > g0 + t) & boxes_meet(a, a + 3, b.lo, b.hi)))
                        laps |= 1u << t;
                }
            };
            wave_lds_sync();
            for (u32 t0 = 0, t1; t0 < nt; t0 = t1) {
                const u32 sz = at(size, t0);
                t1           = min(t0 + sz, nt);
                for (int k = 0; k < 3; k++) {
                    ulo[k] = elo[k] = F64_BIG;
                    uhi[k] = ehi[k] = -F64_BIG;
                }
                for (u32 t = t0; t < t1; t++) {
                    const f64 *m = tgt[wid][t];
                    for (int k = 0; k < 3; k++) {
                        ulo[k] = fmin(ulo[k], m[k]);
                        uhi[k] = fmax(uhi[k], m[3 + k]);
                        elo[k] = fmin(elo[k], m[6 + k]);
                        ehi[k] = fmax(ehi[k], m[9 + k]);
                    }
                }
                u32 t = tt.top, cell = lane;
                bool on = lane < tt.n[tt.top];
                for (;;) {
                    sift(t, cell, on);
                    u64 some;
                    for (;;) {
                        some = __ballot(qn > 0);
                        // 64 leaves, or the last ones
                        if (at(qn, 0) < (u32) WAVE && some != 1ull) break;
                        leaves(t0, t1);
                    }
                    if (!some) break;
                    const u64 eight = __ballot(qn >= 8) & ~1ull;
                    const u32 f     = eight ? (u32) __builtin_ctzll(eight)
                                            : 63u - (u32) __builtin_clzll(some);
                    const u32 k     = min(at(qn, f), 8u);
                    const u32 h0    = at(qh, f);
                    if (lane == f) qh += k, qn -= k;
                    const u32 slot = lane / 8;
                    cell           = q[f][(h0 + slot) % LQ_CAP] * 8 + lane % 8;
                    t              = f - 1;
                    on             = (slot < k) & (cell < tt.n[t]);
                }
            }
            if (OUT != LEAF_FILL && lane < nt) {
                cnt[g0 + lane] = len;
                lap[g0 + lane] = (laps >> lane) & 1u;
                if (OUT == LEAF_ROWS) offset[g0 + lane] = base;
            }
        }

        // rows (leaf lists or particle rows) longer than their fixed capacity: flag and count
        __global__ void k_over_mark(u32 n, const u32 *__restrict cnt, u32 cap,
                                    u32 *__restrict flag, u32 *__restrict ocnt) {
            u32 i = blockIdx.x * blockDim.x + threadIdx.x;
            if (i >= n) return;
            const bool o = cnt[i] > cap;
            flag[i]      = o ? 1u : 0u;
            ocnt[i]      = o ? cnt[i] : 0u;
        }
        // the flagged rows in order into list (as map[i] when map is given), their offsets in
        // the overflow region after the fixed-capacity rows
        __global__ void k_over_list(u32 n, const u32 *__restrict flag, const u32 *__restrict fpos,
                                    const u32 *__restrict opos, u32 base,
                                    const u32 *__restrict map, u32 *__restrict list,
                                    u32 *__restrict offset) {
            u32 i = blockIdx.x * blockDim.x + threadIdx.x;
            if (i >= n || !flag[i]) return;
            list[fpos[i]] = map ? map[i] : i;
            offset[i]     = base + opos[i];
        }

        // Member batches: a batch is 64 consecutive sorted positions of a leaf.  Item l < L is the
        // first batch of leaf l, the further ones of larger leaves follow after the L first ones,
        // those of a leaf together (xstart: its first), in the order the leaves come by
        __device__ inline u32 item_batch(u32 item, u32 l, u32 L, const u32 *__restrict xstart) {
            return item < L ? 0u : item - xstart[l] + 1;
        }
        __device__ inline u32 batch_item(u32 b, u32 l, const u32 *__restrict xstart) {
            return b == 0 ? l : xstart[l] + b - 1;
        }
        __global__ void k_items(u32 L, u32 I, const f64 *__restrict nodes,
                                u32 *__restrict item_leaf, u32 *__restrict xstart,
                                u32 *__restrict n_extra) {
            u32 l = blockIdx.x * blockDim.x + threadIdx.x;
            if (l >= L) return;
            u32 m0, m1;
            node_children(nodes, I + l, m0, m1);
            item_leaf[l]  = l;
            u32 x         = 0;
            const u32 ext = m1 - m0 > WAVE ? (m1 - m0 - 1) / WAVE : 0u;
            if (ext) {
                x = L + atomicAdd(n_extra, ext);
                for (u32 j = 0; j < ext; j++) item_leaf[x + j] = l;
            }
            xstart[l] = x;
        }

        // the last leaf whose box contains p (is_coord_in_range_incl_max, geometry_utils.hpp:74-81),
        // L when none does: the tiers right to left, entering the cells that contain p
        __device__ inline bool box_holds(const f64 *__restrict rec, const double4 &p) {
            return (rec[0] <= p.x) & (p.x <= rec[3]) & (rec[1] <= p.y) & (p.y <= rec[4]) &
                   (rec[2] <= p.z) & (p.z <= rec[5]);
        }
        __device__ inline u32 last_leaf_holding(u32 L, u32 I, const f64 *__restrict nodes,
                                                const f64 *__restrict tiers, const Tiers &tt,
                                                const double4 &p) {
            u32 t = tt.top, c = tt.n[tt.top] - 1;
            for (;;) {
                const f64 *rec = t ? tiers + (u64) (tt.off[t] + c) * NODE_F64
                                   : nodes + (u64) (I + c) * NODE_F64;
                if (box_holds(rec, p)) {
                    if (t == 0) return c;
                    t--;
                    c = min(c * 8 + 7, tt.n[t] - 1);
                    continue;
                }
                while (t < tt.top && c % 8 == 0) { // the first of its cell: on from that cell
                    t++;
                    c /= 8;
                }
                if (c == 0) return L;
                c--;
            }
        }

        // Owner leaf (:406-451) of every local particle, OWN_LANES lanes per member batch (64
        // sorted positions of a leaf): the last leaf whose box contains it.  When its own leaf does,
        // that is the last leaf of the own leaf's list whose box contains it (a leaf that contains
        // a particle of this one meets its box and is in its list, unless a reach below zero
        // shrinks the box); leaves whose box no later leaf meets (lap) own all their particles.  A
        // particle that its leaf's box does not contain (the caller moved it since the boxes were
        // made) is searched for in the tiers; in no box: err bit 2.  Particles owned by another leaf
        // go to mism, and lap is set for the leaf that keeps them.  leaf_cap: as in stage 2.
        // Bound by memory latency.  Lanes 8 / 16: 2.1M Sedov (6 particles per leaf) 31 / 49 us, 4M
        // Plummer 83 / 75 us, 1M disc 22 / 31 us.
        constexpr u32 OWN_LANES = 8;
        __global__ void __launch_bounds__(256)
            k_owner(u32 n, u32 L, u32 I, const f64 *__restrict nodes,
                    const f64 *__restrict tiers, Tiers tt,
                    const u32 *__restrict item_leaf, const u32 *__restrict xstart,
                    const u32 *__restrict n_extra,
                    const u32 *__restrict sort_index, const double4 *__restrict ps,
                    u32 *lap, const u32 *__restrict leaf_cnt,
                    const u32 *__restrict leaf_offset, const u32 *__restrict leaf_ids,
                    u32 leaf_cap, u32 *__restrict owner, u32 *__restrict mism,
                    u32 *__restrict mism_len, u32 *__restrict err) {
            const u32 item = (blockIdx.x * 256 + threadIdx.x) / OWN_LANES;
            if (item >= L + *n_extra) return;
            const u32 l = item < L ? item : item_leaf[item];
            u32 m0, m1;
            node_children(nodes, I + l, m0, m1);
            m0 += item_batch(item, l, L, xstart) * WAVE;
            m1 = min(m1, m0 + WAVE);
            // (another lane of this leaf may set lap meanwhile: the search then finds the same)
            const bool over = lap[l] != 0;
            const f64 *box  = nodes + (u64) (I + l) * NODE_F64;
            for (u32 s = m0 + threadIdx.x % OWN_LANES; s < m1; s += OWN_LANES) {
                const u32 a     = sort_index[s];
                const double4 p = ps[s];
                if (a >= n) continue;
                u32 own = l;
                if (!(box_holds(box, p) & (box[6] >= 0))) {
                    own = last_leaf_holding(L, I, nodes, tiers, tt, p);
                    if (own >= L) {
                        atomicOr(err, 2u);
                        own = l;
                    }
                } else if (over) {
                    const u32 k0 = leaf_offset[l];
                    u32 k = k0 + (leaf_cap ? min(leaf_cnt[l], leaf_cap) : leaf_cnt[l]);
                    while (k > k0) {
                        const u32 nd = leaf_ids[--k];
                        if (nd <= I + l) break;
                        if (box_holds(nodes + (u64) nd * NODE_F64, p)) {
                            own = nd - I;
                            break;
                        }
                    }
                }
                owner[a] = own;
                if (own != l) {
                    mism[atomicAdd(mism_len, 1u)] = a;
                    lap[l]                        = 1;
                }
            }
        }

        // stage 2 count / fill.  SORTED layout: the CSR is indexed by the sorted position of
        // the particle and holds sorted positions of its neighbours; otherwise both are
        // particle ids (the reference layout).
        template<bool FILL, bool SORTED, bool STRIDE>
        __global__ void k_part_neigh(u32 n, const u32 *__restrict list,
                                     const u32 *__restrict list_len, u32 I,
                                     const f64 *__restrict nodes,
                                     const u32 *__restrict sort_index,
                                     const u32 *__restrict owner,
                                     const u32 *__restrict leaf_cnt,
                                     const u32 *__restrict leaf_offset,
                                     const u32 *__restrict leaf_ids, const f64 *__restrict x,
                                     const f64 *__restrict y, const f64 *__restrict z,
                                     const f64 *__restrict h, const u32 *__restrict inv,
                                     f64 htol, f64 Rker2, u32 *__restrict cnt,
                                     u32 *__restrict offset, u32 *__restrict ids, u32 cap,
                                     u32 leaf_cap) {
            u32 t = blockIdx.x * blockDim.x + threadIdx.x;
            if (t >= (list ? *list_len : n)) return;
            u32 a      = list ? list[t] : t;
            u32 ia     = SORTED ? inv[a] : a;
            f64 rint_a = h[a] * htol;
            f64 xa = x[a], ya = y[a], za = z[a];
            f64 ca = rint_a * rint_a * Rker2;
            u32 lo = owner[a];
            u32 k0 = leaf_offset[lo],
                k1 = k0 + (leaf_cap ? min(leaf_cnt[lo], leaf_cap) : leaf_cnt[lo]);
            const u32 c0 = STRIDE ? ia * cap : (FILL ? offset[ia] : 0u);
            const u32 ce = c0 + cap;
            u32 c        = c0;
            for (u32 k = k0; k < k1; k++) {
                u32 s0, s1;
                node_children(nodes, leaf_ids[k], s0, s1); // leaf record: sorted range
                for (u32 s = s0; s < s1; s++) {
                    u32 b    = sort_index[s];
                    f64 dx   = xa - x[b], dy = ya - y[b], dz = za - z[b];
                    f64 rab2 = dx * dx + dy * dy + dz * dz;
                    f64 rb   = h[b] * htol;
                    bool no_interact = rab2 > ca && rab2 > rb * rb * Rker2;
                    if (!no_interact) {
                        if (FILL && (!STRIDE || c < ce)) ids[c] = SORTED ? s : b;
                        c++;
                    }
                }
            }
            if (!FILL || STRIDE) cnt[ia] = c - c0;
            if (STRIDE) offset[ia] = c0;
        }

        // sorted copy of positions and h (AoS, 32 B per object) + inverse permutation
        // (sorted layout: with the row counts set to zero, the rows of images stay empty)
        __global__ void k_sorted_copy(u32 nm, const u32 *__restrict sort_index,
                                      const f64 *__restrict x, const f64 *__restrict y,
                                      const f64 *__restrict z, const f64 *__restrict h,
                                      double4 *__restrict ps, u32 *__restrict inv,
                                      u32 *__restrict cnt) {
            u32 s = blockIdx.x * blockDim.x + threadIdx.x;
            if (s >= nm) return;
            u32 b  = sort_index[s];
            ps[s]  = make_double4(x[b], y[b], z[b], h[b]);
            inv[b] = s;
            if (cnt) cnt[s] = 0;
        }

        // Sorted layout: the sorted positions of the local particles in order (lpos; perm: the
        // particles there, moved: how many of them are not at their own index), compacted as in
        // compact.hpp; without images every position is local
        template<int ITEMS>
        __global__ void __launch_bounds__(CT_BLK)
            k_local_count(u32 nm, u32 n, const u32 *__restrict sort_index,
                          u32 *__restrict tile_cnt) {
            tile_count<ITEMS>(nm, tile_cnt, [&](u32 j) { return sort_index[j] < n; });
        }
        template<int ITEMS>
        __global__ void __launch_bounds__(CT_BLK)
            k_local_rows(u32 nm, u32 n, const u32 *__restrict sort_index,
                         const u32 *__restrict tile_cnt, u32 nt, u32 *__restrict lpos,
                         u32 *__restrict perm, u32 *__restrict moved) {
            __shared__ u32 part[CT_BLK / WAVE];
            u32 mv = 0;
            tile_compact<ITEMS>(
                nm, tile_cnt, nt, nm == n, [&](u32 j) { return sort_index[j] < n; },
                [&](u32 p, u32 j) {
                    lpos[p] = j;
                    if (perm) {
                        const u32 a = sort_index[j];
                        perm[p]     = a;
                        mv += a != p ? 1u : 0u;
                    }
                },
                [](u32) {});
            if (!perm) return; // the same for the whole grid
            mv = wave_reduce(mv, [](u32 a, u32 b) { return a + b; });
            if (__lane_id() == 0) part[threadIdx.x / WAVE] = mv;
            __syncthreads();
            if (threadIdx.x == 0) {
                for (int w = 1; w < CT_BLK / WAVE; w++) mv += part[w];
                if (mv) atomicAdd(moved, mv);
            }
        }

        constexpr int GRP_WAVES = 4;

        // stage 2, one wave per member batch: a batch is 64 consecutive sorted positions of a
        // leaf (item_leaf / xstart map the wave to its leaf and batch), its members the local
        // particles among them whose owner is this leaf; the candidates are the particles of
        // the neighbour leaves, in list order then sorted order.  Candidates are taken 64 at a
        // time; those farther from the members' bounding box than both the members' largest
        // cut radius and their own are dropped (they cannot pass the pair test: the box
        // distance bounds every member distance from below, kept with a 1e-12 margin so that
        // rounding cannot drop a pair), and the rest are queued in order.  64 queued ones at a time,
        // a lane each, are tested against the members one after the other; a member's row grows
        // by the lanes of its ballot.  A lane finds its candidate from a bit mask of the ranges'
        // first candidates.  The queue keeps the lanes of the pair tests full whatever the
        // members' number and the share of candidates dropped.  (With tests on candidate x member
        // lanes right after each 64 candidates, many lanes idled, and each lane searched its range
        // by bisection, six dependent LDS reads.)  It holds sorted positions alone: a queued
        // particle is read again, a cache hit.  With its position kept in LDS as well the kernel
        // had 4 waves per SIMD for 8 and spent 58 % of the time in waits.  Bound by these loads'
        // latency and by the issue of about 20 instructions per member and 64 candidates; the next
        // leaves and candidates are requested while the present ones are tested.
        // Before, with the positions in LDS, now: 2.1M Sedov 1.63, 1.61, 1.38 ms; 4M Plummer
        // 4.58, 4.42, 3.53 ms; 1M disc 0.89, 0.83, 0.68 ms.  (Two members per turn: no change.)
        // n_items: the batches beyond the leaves' first ones.
        // LIST: one wave per particle of list (item_leaf holds particle ids, n_items their
        // count): its whole row at offset[its sorted position], the path of rows longer than
        // their fixed capacity.
        template<bool FILL, bool SORTED, bool STRIDE, bool LIST = false, bool BCULL = false>
        __global__ void __launch_bounds__(GRP_WAVES * WAVE)
            k_group_neigh(u32 n, u32 L, u32 I, const f64 *__restrict nodes,
                          const u32 *__restrict sort_index, const double4 *__restrict ps,
                          const u32 *__restrict owner, const u32 *__restrict lap,
                          const u32 *__restrict leaf_cnt, const u32 *__restrict leaf_offset,
                          const u32 *__restrict leaf_ids, const u32 *__restrict item_leaf,
                          const u32 *__restrict xstart, const u32 *__restrict n_items, f64 htol,
                          f64 Rker2,
                          u32 *__restrict cnt, u32 *__restrict offset, u32 *__restrict ids,
                          u32 cap, u32 leaf_cap, const u32 *__restrict inv = nullptr,
                          const f64 *__restrict bbox = nullptr) {
            constexpr u32 QN = 2 * WAVE;
            __shared__ u32 queue[GRP_WAVES][QN];    // queued candidates: sorted positions
            __shared__ double4 mpos[GRP_WAVES][WAVE]; // member x, y, z, cut radius^2
            // the ranges of a pass: sorted position less index of the first candidate, that index
            __shared__ uint2 rng[GRP_WAVES][WAVE];
            __shared__ u32 first[GRP_WAVES][2]; // bit c: candidate c of a window starts a range
            // BCULL: the neighbour leaves of one pass (range, leaf, batches before it)
            __shared__ u32 lr0[GRP_WAVES][BCULL ? WAVE : 1], lr1[GRP_WAVES][BCULL ? WAVE : 1];
            __shared__ u32 lbs[GRP_WAVES][BCULL ? WAVE : 1], lbx[GRP_WAVES][BCULL ? WAVE : 1];
            const int lane = __lane_id();
            const u32 wid  = (u32) __builtin_amdgcn_readfirstlane((int) (threadIdx.x / WAVE));
            const u32 item = blockIdx.x * GRP_WAVES + wid;
            if (item >= (LIST ? 0u : L) + *n_items) return;
            u32 l, mb, m1;
            if constexpr (LIST) { // the batch is the listed particle alone (lane 0)
                const u32 a0 = item_leaf[item];
                l            = owner[a0];
                mb           = inv[a0];
                m1           = mb + 1;
            } else {
                l = item < L ? item : item_leaf[item];
                u32 m0;
                node_children(nodes, I + l, m0, m1);
                mb = m0 + item_batch(item, l, L, xstart) * WAVE;
            }
            const u64 lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
            // leaf_cap (fixed-capacity leaf rows): a row that overflowed holds only leaf_cap
            // entries; the build is repeated then, but nothing may be read past the row
            const u32 k0 = leaf_offset[l],
                      k1 = k0 + (leaf_cap ? min(leaf_cnt[l], leaf_cap) : leaf_cnt[l]);
            // the first neighbour leaves, requested before the members are looked at; in the loop
            // below the next ones are requested a pass ahead
            u32 nd_next     = k0 + lane < k1 ? leaf_ids[k0 + lane] : 0u;
            const bool all  = lap[l] == 0; // the leaf owns all its particles (k_owner)
            u32 sm   = mb + lane;
            bool mem = false;
            u32 a    = 0;
            double4 pa{0, 0, 0, 0};
            if (sm < m1) {
                a               = sort_index[sm];
                const double4 p = ps[sm];
                if (a < n && (all || owner[a] == l)) {
                    mem    = true;
                    f64 ra = p.w * htol;
                    pa        = make_double4(p.x, p.y, p.z, ra * ra * Rker2);
                }
            }
            const u64 members = __ballot(mem);
            if (!members) return;
            const u32 M    = (u32) __popcll(members);
            const u32 rank = (u32) __popcll(members & lt); // member index of this lane
            const u32 ia   = SORTED ? sm : a;
            const u32 row0 = STRIDE ? (mem ? ia * cap : 0u) : ((FILL && mem) ? offset[ia] : 0u);
            if (mem) mpos[wid][rank] = pa;
            // lane m (< M): row start and length so far of the member of rank m
            u32 mrow, mlen = 0;
            {
                // lane `rank` receives from the member lane of that rank
                mrow = (u32) __builtin_amdgcn_ds_permute((int) (mem ? rank : 63u) * 4, (int) row0);
            }
            // the members' bounding box and largest cut radius^2
            constexpr f64 BIG = 1.7976931348623157e308;
            auto fmn = [](f64 p, f64 q) { return fmin(p, q); };
            auto fmx = [](f64 p, f64 q) { return fmax(p, q); };
            const f64 blx = wave_reduce(mem ? pa.x : BIG, fmn), bhx = wave_reduce(mem ? pa.x : -BIG, fmx);
            const f64 bly = wave_reduce(mem ? pa.y : BIG, fmn), bhy = wave_reduce(mem ? pa.y : -BIG, fmx);
            const f64 blz = wave_reduce(mem ? pa.z : BIG, fmn), bhz = wave_reduce(mem ? pa.z : -BIG, fmx);
            const f64 br2 = wave_reduce(mem ? pa.w : 0.0, fmx);
            auto at = [](u32 v, u32 l) { return (u32) __builtin_amdgcn_readlane((int) v, (int) l); };
            // lanes of m below this one
            auto below = [](u64 m) {
                return (u32) __builtin_amdgcn_mbcnt_hi(
                    (u32) (m >> 32), (u32) __builtin_amdgcn_mbcnt_lo((u32) m, 0u));
            };
            u32 qh = 0, qn = 0; // first queued candidate and their number (wave-uniform)
            // the first nq (<= 64) queued candidates against the members
            auto test = [&](u32 nq) {
                const bool on = (u32) lane < nq;
                const u32 sl  = (qh + (on ? (u32) lane : 0u)) % QN;
                const u32 sb    = queue[wid][sl];
                double4 q       = ps[sb];
                const f64 rb    = q.w * htol;
                q.w             = rb * rb * Rker2;
                const u32 id    = FILL ? (SORTED ? sb : sort_index[sb]) : 0u;
                for (u32 m = 0; m < M; m++) {
                    const double4 me = mpos[wid][m];
                    const f64 dx = me.x - q.x, dy = me.y - q.y, dz = me.z - q.z;
                    const f64 rab2  = dx * dx + dy * dy + dz * dz;
                    const bool keep = on & !((rab2 > me.w) & (rab2 > q.w));
                    const u64 km    = __ballot(keep);
                    const u32 len   = at(mlen, m);
                    if (FILL && keep) {
                        const u32 p = len + below(km);
                        if (!STRIDE || p < cap) ids[at(mrow, m) + p] = id;
                    }
                    mlen = (u32) lane == m ? len + (u32) __popcll(km) : mlen;
                }
                qh += nq;
                qn -= nq;
            };
            // candidates of this lane's range [s0, s0 + sz) of sorted positions, the lanes' ranges
            // in order: the near ones into the queue, tested when there are 64
            auto candidates = [&](u32 s0, u32 sz) {
                u32 inc = sz;
                for (int o = 1; o < WAVE; o <<= 1) {
                    u32 t = __shfl_up(inc, o, WAVE);
                    if (lane >= o) inc += t;
                }
                const u32 total = at(inc, WAVE - 1);
                if (total == 0) return;
                const u64 some = __ballot(sz > 0);
                const u32 nr   = (u32) __popcll(some);
                wave_lds_sync();
                if (sz) rng[wid][below(some)] = make_uint2(s0 - (inc - sz), inc - sz);
                wave_lds_sync();
                const u32 start = (u32) lane < nr ? rng[wid][lane].y : 0xffffffffu;
                // the sorted position of candidate c0 + lane
                auto find = [&](u32 c0) -> u32 {
                    // ranges begun before this window, and those that begin in it
                    const u32 before = (u32) __popcll(__ballot(start < c0));
                    const u32 w      = start - c0;
                    if (lane < 2) first[wid][lane] = 0;
                    wave_lds_sync();
                    if (w < (u32) WAVE && start != 0xffffffffu)
                        atomicOr(&first[wid][w / 32], 1u << (w % 32));
                    wave_lds_sync();
                    const u64 fm = (u64) first[wid][0] | ((u64) first[wid][1] << 32);
                    const u32 c  = c0 + lane;
                    const u32 j  = before + below(fm) + (u32) ((fm >> lane) & 1ull) - 1;
                    return c < total ? rng[wid][j].x + c : 0u;
                };
                u32 sb_next    = find(0);
                double4 q_next = ps[sb_next];
                for (u32 c0 = 0; c0 < total; c0 += WAVE) {
                    const u32 sb     = sb_next;
                    const double4 q  = q_next;
                    const bool valid = c0 + lane < total;
                    if (c0 + WAVE < total) { // the next candidates load while these are tested
                        sb_next = find(c0 + WAVE);
                        q_next  = ps[sb_next];
                    }
                    f64 rb    = q.w * htol;
                    f64 rb2   = rb * rb * Rker2;
                    f64 ex = q.x < blx ? blx - q.x : (q.x > bhx ? q.x - bhx : 0.0);
                    f64 ey = q.y < bly ? bly - q.y : (q.y > bhy ? q.y - bhy : 0.0);
                    f64 ez = q.z < blz ? blz - q.z : (q.z > bhz ? q.z - bhz : 0.0);
                    f64 d2 = (ex * ex + ey * ey + ez * ez) * (1.0 - 1e-12);
                    const bool near = valid & !((d2 > br2) & (d2 > rb2));
                    const u64 nm    = __ballot(near);
                    if (near) queue[wid][(qh + qn + below(nm)) % QN] = sb;
                    qn += (u32) __popcll(nm);
                    wave_lds_sync();
                    if (qn >= (u32) WAVE) {
                        test(WAVE);
                        wave_lds_sync();
                    }
                }
            };
            for (u32 kb = k0; kb < k1; kb += WAVE) {
                // neighbour leaves in batches of up to 64: lane i loads the range of the i-th
                // leaf of the batch; candidates are the concatenated ranges in order
                u32 k  = kb + lane;
                u32 r0 = 0, r1 = 0;
                const u32 nd = nd_next;
                nd_next      = k + WAVE < k1 ? leaf_ids[k + WAVE] : 0u;
                if (k < k1) {
                    node_children(nodes, nd, r0, r1); // leaf: sorted range
                    // the whole range is dropped when none of its particles can reach a
                    // member: the leaf's box is farther from the members' box than both the
                    // members' largest cut radius and the leaf's (rint = max h * htol).  The
                    // box distance bounds each particle's from below, so this drops only
                    // candidates the per-particle test below would drop
                    const f64 *rec = nodes + (u64) nd * NODE_F64;
                    const f64 ex   = fmax(fmax(rec[0] - bhx, blx - rec[3]), 0.);
                    const f64 ey   = fmax(fmax(rec[1] - bhy, bly - rec[4]), 0.);
                    const f64 ez   = fmax(fmax(rec[2] - bhz, blz - rec[5]), 0.);
                    const f64 d2   = (ex * ex + ey * ey + ez * ez) * (1.0 - 1e-12);
                    const f64 rr2  = rec[6] * rec[6] * Rker2;
                    if (d2 > br2 && d2 > rr2) r1 = r0;
                }
                const u32 nr = min(k1 - kb, (u32) WAVE);
                if constexpr (!BCULL) {
                    candidates(r0, r1 - r0);
                } else {
                    // each range split into the member batches of its leaf (64 sorted
                    // positions from the leaf's start; bbox: their boxes and largest cut
                    // radius^2), every batch dropped whole by the test above
                    const bool okl = nd >= I && nd - I < L;
                    const u32 nbl  = okl ? (r1 - r0 + WAVE - 1) / WAVE : 0u;
                    u32 binc       = nbl;
                    for (int o = 1; o < WAVE; o <<= 1) {
                        u32 t = __shfl_up(binc, o, WAVE);
                        if (lane >= o) binc += t;
                    }
                    const u32 totb = __shfl(binc, WAVE - 1, WAVE);
                    wave_lds_sync();
                    lr0[wid][lane] = r0;
                    lr1[wid][lane] = r1;
                    lbs[wid][lane] = okl ? nd - I : 0u;
                    lbx[wid][lane] = binc - nbl;
                    wave_lds_sync();
                    for (u32 t0 = 0; t0 < totb; t0 += WAVE) {
                        const u32 tb = t0 + lane;
                        u32 s0 = 0, s1 = 0;
                        if (tb < totb) {
                            // the range holding batch tb: largest j with lbx[j] <= tb
                            u32 j = 0;
                            for (u32 st = WAVE / 2; st > 0; st >>= 1) {
                                u32 q = j + st;
                                if (q < nr && lbx[wid][q] <= tb) j = q;
                            }
                            const u32 bi = tb - lbx[wid][j];
                            s0           = lr0[wid][j] + bi * WAVE;
                            s1           = min(s0 + WAVE, lr1[wid][j]);
                            const f64 *bx = bbox + (u64) batch_item(bi, lbs[wid][j], xstart) * 8;
                            const f64 ex  = fmax(fmax(bx[0] - bhx, blx - bx[3]), 0.);
                            const f64 ey  = fmax(fmax(bx[1] - bhy, bly - bx[4]), 0.);
                            const f64 ez  = fmax(fmax(bx[2] - bhz, blz - bx[5]), 0.);
                            const f64 d2  = (ex * ex + ey * ey + ez * ez) * (1.0 - 1e-12);
                            if (d2 > br2 && d2 > bx[6]) s1 = s0;
                        }
                        candidates(s0, s1 - s0);
                    }
                }
            }
            if (qn) test(qn);
            const u32 cm = __shfl(mlen, (int) rank, WAVE);
            if (mem) {
                if (!FILL || STRIDE) cnt[ia] = cm;
                if (STRIDE) offset[ia] = row0;
            }
        }

        // box of every member batch (all its sorted positions, images included: they are
        // candidates too) and the largest cut radius^2 among them, 8 doubles per batch:
        // lo x, y, z, hi x, y, z, (h htol)^2 R^2, unused.  One wave per batch.
        __global__ void __launch_bounds__(GRP_WAVES * WAVE)
            k_batch_boxes(u32 L, u32 I, const f64 *__restrict nodes,
                          const u32 *__restrict item_leaf, const u32 *__restrict xstart,
                          const u32 *__restrict n_extra,
                          const double4 *__restrict ps, f64 htol, f64 Rker2,
                          f64 *__restrict bbox) {
            const int lane = __lane_id();
            const u32 item = blockIdx.x * GRP_WAVES + threadIdx.x / WAVE;
            if (item >= L + *n_extra) return;
            const u32 l = item_leaf[item];
            u32 m0, m1;
            node_children(nodes, I + l, m0, m1);
            const u32 sm = m0 + item_batch(item, l, L, xstart) * WAVE + lane;
            constexpr f64 BIG = 1.7976931348623157e308;
            f64 lx = BIG, ly = BIG, lz = BIG, hx = -BIG, hy = -BIG, hz = -BIG, r2 = 0;
            if (sm < m1) {
                const double4 q = ps[sm];
                const f64 rb    = q.w * htol;
                lx = hx = q.x, ly = hy = q.y, lz = hz = q.z;
                r2 = rb * rb * Rker2;
            }
            auto fmn = [](f64 p, f64 q) { return fmin(p, q); };
            auto fmx = [](f64 p, f64 q) { return fmax(p, q); };
            lx = wave_reduce(lx, fmn), ly = wave_reduce(ly, fmn), lz = wave_reduce(lz, fmn);
            hx = wave_reduce(hx, fmx), hy = wave_reduce(hy, fmx), hz = wave_reduce(hz, fmx);
            r2 = wave_reduce(r2, fmx);
            if (lane < 8) {
                const f64 v[8] = {lx, ly, lz, hx, hy, hz, r2, 0.};
                bbox[(u64) item * 8 + lane] = v[lane];
            }
        }
    } // namespace

    namespace {
        // max of n u32 values into *out (device; *out must start at 0)
        __global__ void __launch_bounds__(256)
            k_max_u32(u32 n, const u32 *__restrict v, u32 *__restrict out) {
            __shared__ u32 lds[256 / WAVE];
            u32 m = 0;
            for (u32 i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
                m = max(m, v[i]);
            m = wave_reduce(m, [](u32 p, u32 q) { return p > q ? p : q; });
            if (__lane_id() == 0) lds[threadIdx.x / WAVE] = m;
            __syncthreads();
            if (threadIdx.x == 0) {
                for (int w = 1; w < 256 / WAVE; w++) m = max(m, lds[w]);
                atomicMax(out, m);
            }
        }
        void max_u32(hipStream_t s, u32 n, const u32 *v, u32 *out) {
            if (n) k_max_u32<<<std::min<u32>(div_up(n, 256), 256), 256, 0, s>>>(n, v, out);
        }

        // out += {max of cnt[0, n), sum, number of rows longer than cap, their entries} (device;
        // the four words must start at 0)
        __global__ void __launch_bounds__(256)
            k_row_stats(u32 n, const u32 *__restrict cnt, u32 cap, u32 *__restrict mx,
                        u32 *__restrict tot, u32 *__restrict over) {
            __shared__ u32 lds[4][256 / WAVE];
            u32 v[4] = {0, 0, 0, 0};
            for (u32 i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
                const u32 c = cnt[i];
                const bool o = c > cap;
                v[0]         = max(v[0], c);
                v[1] += c;
                v[2] += o ? 1u : 0u;
                v[3] += o ? c : 0u;
            }
            v[0] = wave_reduce(v[0], [](u32 p, u32 q) { return p > q ? p : q; });
            for (int k = 1; k < 4; k++) v[k] = wave_reduce(v[k], [](u32 p, u32 q) { return p + q; });
            if (__lane_id() == 0)
                for (int k = 0; k < 4; k++) lds[k][threadIdx.x / WAVE] = v[k];
            __syncthreads();
            if (threadIdx.x == 0) {
                for (int w = 1; w < 256 / WAVE; w++) {
                    v[0] = max(v[0], lds[0][w]);
                    for (int k = 1; k < 4; k++) v[k] += lds[k][w];
                }
                atomicMax(mx, v[0]);
                if (v[1]) atomicAdd(tot, v[1]);
                if (v[2]) {
                    atomicAdd(over, v[2]);
                    atomicAdd(over + 1, v[3]);
                }
            }
        }
        void row_stats(hipStream_t s, u32 n, const u32 *cnt, u32 cap, u32 *mx, u32 *tot,
                       u32 *over) {
            if (n)
                k_row_stats<<<std::min<u32>(div_up(n, 1024), 512), 256, 0, s>>>(n, cnt, cap, mx,
                                                                                tot, over);
        }

        // lists of all leaves, eight per wave
        template<int OUT>
        void leaf_lists(hipStream_t s, NeighBuffers &nb, const TreeBuffers &t, f64 Rkern,
                        u32 cap) {
            k_leaf_lists<OUT, false>
                <<<div_up(div_up(t.L, LEAF_TGT), LW_WAVES), LW_WAVES * WAVE, 0, s>>>(
                    t.L, t.I, t.nodes.data(), t.tiers.data(), t.tt, Rkern, nb.leaf_cnt.data(),
                    nb.leaf_offset.data(), nb.leaf_ids.data(), cap, nb.lap.data(), nullptr, 0);
        }

        // the stage-2 wave items (one per 64 sorted positions of every leaf), those beyond the
        // leaves' first ones counted at counters[7]; returns the launch's block count, sized for
        // the bound L + nm / 64 (waves past the count return at once)
        u32 batch_items(hipStream_t s, NeighBuffers &nb, const TreeBuffers &t) {
            const u32 L = t.L, bound = L + div_up(t.n_obj, (u32) WAVE);
            nb.xstart.resize(L);
            nb.item_leaf.resize(bound);
            k_items<<<div_up(L, 256), 256, 0, s>>>(L, t.I, t.nodes.data(), nb.item_leaf.data(),
                                                    nb.xstart.data(), nb.counters.data() + 7);
            return div_up(bound, (u32) GRP_WAVES);
        }

        // error flags (counters[4]) into exceptions
        void check_flags(u32 f) {
            if (f & 2u)
                throw std::runtime_error("neighbour cache: a particle is outside every leaf box");
        }
        // owner leaves and mismatch list
        void owners(hipStream_t s, NeighBuffers &nb, const TreeBuffers &t, u32 n_local,
                    u32 gblocks, u32 leaf_cap) {
            k_owner<<<div_up((u64) gblocks * GRP_WAVES * OWN_LANES, 256), 256, 0, s>>>(
                n_local, t.L, t.I, t.nodes.data(), t.tiers.data(), t.tt, nb.item_leaf.data(),
                nb.xstart.data(), nb.counters.data() + 7, t.sort_index.data(), nb.ps.data(),
                nb.lap.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(),
                leaf_cap, nb.owner.data(), nb.mism.data(), nb.counters.data() + 5,
                nb.counters.data() + 4);
        }

        // boxes of the member batches for the batch-level cull of stage 2, on sets whose tree
        // sort took the spatial tie order (runs of equal codes: leaves of hundreds of
        // particles, where a leaf-level test keeps most candidates); SHAMX_BATCH_CULL=1 forces
        // it (tests).  nullptr: no batch cull.
        const f64 *batch_boxes(hipStream_t s, NeighBuffers &nb, const TreeBuffers &t,
                               u32 gblocks, f64 htol, f64 Rker2) {
            const char *e = std::getenv("SHAMX_BATCH_CULL");
            if (!t.fine_ties && !(e && std::atoi(e) == 1)) return nullptr;
            nb.bbox.resize((size_t) gblocks * GRP_WAVES * 8);
            k_batch_boxes<<<gblocks, GRP_WAVES * WAVE, 0, s>>>(
                t.L, t.I, t.nodes.data(), nb.item_leaf.data(), nb.xstart.data(),
                nb.counters.data() + 7, nb.ps.data(), htol, Rker2, nb.bbox.data());
            return nb.bbox.data();
        }
        // stage-2 launch, with the batch-level cull when bb holds the batch boxes
        template<bool FILL, bool SORTED, bool STRIDE, class... A>
        void launch_group(hipStream_t s, u32 gblocks, const f64 *bb, A... a) {
            if (bb)
                k_group_neigh<FILL, SORTED, STRIDE, false, true>
                    <<<gblocks, GRP_WAVES * WAVE, 0, s>>>(a..., nullptr, bb);
            else
                k_group_neigh<FILL, SORTED, STRIDE><<<gblocks, GRP_WAVES * WAVE, 0, s>>>(a...);
        }

        // packed rows, two passes (count, scan, fill); SORTED: rows by sorted position
        // (leaf_cap: capacity of fixed-capacity leaf lists, 0 for packed ones)
        template<bool SORTED>
        void stage2_packed(hipStream_t s, NeighBuffers &nb, const TreeBuffers &t, u32 n_local,
                           u32 gblocks, const f64 *x, const f64 *y, const f64 *z, const f64 *h,
                           f64 htol, f64 Rker2, u32 *hc, u32 leaf_cap = 0) {
            u32 L = t.L, I = t.I;
            u32 rows      = SORTED ? t.n_obj : n_local;
            u32 *mism_len      = nb.counters.data() + 5;
            const u32 *n_items = nb.counters.data() + 7;
            const f64 *bb = batch_boxes(s, nb, t, gblocks, htol, Rker2);
            launch_group<false, SORTED, false>(s, gblocks, bb,
                n_local, L, I, t.nodes.data(), t.sort_index.data(), nb.ps.data(),
                nb.owner.data(), nb.lap.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(),
                nb.item_leaf.data(), nb.xstart.data(), n_items, htol, Rker2, nb.cnt.data(),
                nullptr, nullptr, 0, leaf_cap);
            k_part_neigh<false, SORTED, false><<<div_up(n_local, 128), 128, 0, s>>>(
                n_local, nb.mism.data(), mism_len, I, t.nodes.data(), t.sort_index.data(),
                nb.owner.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(), x,
                y, z, h, nb.inv.data(), htol, Rker2, nb.cnt.data(), nullptr, nullptr, 0,
                leaf_cap);
            exclusive_scan_u32(s, nb.cnt.data(), nb.offset.data(), rows, nb.counters.data() + 1,
                               nb.scratch.data());
            // longest leaf list and row (counters[8], [9])
            fill_u32(s, nb.counters.data() + 8, 0, 2);
            max_u32(s, L, nb.leaf_cnt.data(), nb.counters.data() + 8);
            max_u32(s, rows, nb.cnt.data(), nb.counters.data() + 9);
            SHAMX_HIP(hipMemcpyAsync(hc, nb.counters.data(), 16 * sizeof(u32),
                                     hipMemcpyDeviceToHost, s));
            SHAMX_HIP(hipStreamSynchronize(s));
            check_flags(hc[4]);
            nb.n_pairs    = hc[1];
            nb.n_mismatch = hc[5];
            nb.ids.resize(std::max<u64>(nb.n_pairs, 1));
            launch_group<true, SORTED, false>(s, gblocks, bb,
                n_local, L, I, t.nodes.data(), t.sort_index.data(), nb.ps.data(),
                nb.owner.data(), nb.lap.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(),
                nb.item_leaf.data(), nb.xstart.data(), n_items, htol, Rker2, nullptr,
                nb.offset.data(), nb.ids.data(), 0, leaf_cap);
            k_part_neigh<true, SORTED, false><<<div_up(n_local, 128), 128, 0, s>>>(
                n_local, nb.mism.data(), mism_len, I, t.nodes.data(), t.sort_index.data(),
                nb.owner.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(), x,
                y, z, h, nb.inv.data(), htol, Rker2, nullptr, nb.offset.data(), nb.ids.data(), 0,
                leaf_cap);
        }

        // SHAMX_NEIGH_ROWS=packed (read at every build) takes packed particle rows even where
        // fixed-capacity rows fit, so that path can be tested at small sizes
        bool packed_rows_forced() {
            const char *e = std::getenv("SHAMX_NEIGH_ROWS");
            return e && std::strcmp(e, "packed") == 0;
        }

        // row capacity for a measured maximum: 1/8 headroom, rounded up to 16 entries so that
        // rows start on 64-byte boundaries
        u32 grow_cap(u32 need) { return (need + need / 8 + 16 + 15) & ~15u; }
    } // namespace

    void local_rows(hipStream_t s, u32 nm, u32 n, const u32 *sort_index, u32 *lpos, u32 *perm,
                    u32 *moved, DevArray<u32> &tile_cnt) {
        if (nm == 0) return;
        const u32 nt = compact_tiles(nm);
        tile_cnt.resize(nt);
        compact_dispatch(nm, [&](auto items) {
            constexpr int IT = decltype(items)::value;
            if (nt > 1 && nm != n)
                k_local_count<IT><<<nt, CT_BLK, 0, s>>>(nm, n, sort_index, tile_cnt.data());
            k_local_rows<IT><<<nt, CT_BLK, 0, s>>>(nm, n, sort_index, tile_cnt.data(), nt, lpos,
                                                   perm, moved);
        });
        SHAMX_HIP(hipGetLastError());
    }

    void neigh_build(hipStream_t s, NeighBuffers &nb, TreeBuffers &t, u32 n_local,
                     const f64 *x, const f64 *y, const f64 *z, const f64 *h, f64 htol,
                     f64 Rkern, bool sorted_layout) {
        u32 L = t.L, I = t.I, nm = t.n_obj;
        nb.n_local       = n_local;
        nb.sorted_layout = sorted_layout;
        u32 rows         = sorted_layout ? nm : n_local;
        nb.counters.resize(16);
        nb.scratch.resize(std::max({scan_scratch_bytes(L), scan_scratch_bytes(rows),
                                    scan_scratch_bytes(nm)}));
        nb.leaf_cnt.resize(L);
        nb.leaf_offset.resize(L);
        nb.lap.resize(L);
        nb.owner.resize(std::max<u32>(n_local, 1));
        nb.cnt.resize(std::max<u32>(rows, 1));
        nb.offset.resize(std::max<u32>(rows, 1));
        fill_u32(s, nb.counters.data(), 0, 16);
        f64 Rker2 = Rkern * Rkern;
        u32 *hc = nb.host.data(); // 16 pinned words: the reads queue on the stream

        // sorted copy and inverse permutation, member batches
        nb.ps.resize(nm);
        nb.inv.resize(nm);
        nb.mism.resize(std::max<u32>(n_local, 1));
        k_sorted_copy<<<div_up(nm, 256), 256, 0, s>>>(nm, t.sort_index.data(), x, y, z, h,
                                                      nb.ps.data(), nb.inv.data(),
                                                      sorted_layout ? nb.cnt.data() : nullptr);
        const u32 gblocks = batch_items(s, nb, t);

        // leaf lists in two passes (count, scan, fill); returns once their length is known
        auto packed_leaves = [&] {
            leaf_lists<LEAF_COUNT>(s, nb, t, Rkern, 0);
            exclusive_scan_u32(s, nb.leaf_cnt.data(), nb.leaf_offset.data(), L,
                               nb.counters.data(), nb.scratch.data());
            SHAMX_HIP(hipMemcpyAsync(hc, nb.counters.data(), 8 * sizeof(u32),
                                     hipMemcpyDeviceToHost, s));
            SHAMX_HIP(hipStreamSynchronize(s));
            nb.n_leaf_pairs = hc[0];
            nb.leaf_ids.resize(std::max<u64>(nb.n_leaf_pairs, 1));
            leaf_lists<LEAF_FILL>(s, nb, t, Rkern, 0);
        };

        if (!sorted_layout) {
            // reference layout
            packed_leaves();
            nb.leaf_stride = 0;
            if (n_local == 0) {
                nb.n_pairs = 0;
                return;
            }
            owners(s, nb, t, n_local, gblocks, 0);
            stage2_packed<false>(s, nb, t, n_local, gblocks, x, y, z, h, htol, Rker2, hc);
            nb.row_stride = 0;
            SHAMX_HIP(hipGetLastError());
            return;
        }

        // sorted layout: the local rows in sorted order
        nb.lpos.resize(std::max<u32>(n_local, 1));
        if (nb.want_perm) nb.perm.resize(std::max<u32>(n_local, 1));
        local_rows(s, nm, n_local, t.sort_index.data(), nb.lpos.data(),
                   nb.want_perm ? nb.perm.data() : nullptr, nb.counters.data() + 3, nb.tile_cnt);

        // Both stages in one pass each, rows of fixed capacity, chosen from the previous build
        // (about four times the mean length, at most the longest row plus headroom).  Rows
        // longer than their capacity (the counts run on past it) are listed and filled again,
        // whole, into an overflow region after the fixed-capacity rows, their offsets pointing
        // there: consumers read (offset, count) and see one layout.  Leaf lists that overflow
        // must be complete before stage 2 reads them: once a build has seen leaf overflow,
        // the next ones resolve it between the stages (one more host sync); the first time, the
        // build is repeated.
        // capacity for rows of measured longest `mx` and total `tot` over `rows_` rows, at most
        // what u32 entry indices address for rows_ rows (a multiple of 16: 64-byte rows)
        auto fit = [](u32 rows_, u32 cap) {
            u64 lim = 0xffffffffull / std::max<u32>(rows_, 1);
            return (u32) std::max<u64>(16, std::min<u64>(cap, lim) & ~15ull);
        };
        auto choose = [&](u32 mx, u64 tot, u32 used_rows, u32 rows_) {
            u64 mean4 = (4 * div_up(tot, (u64) std::max<u32>(used_rows, 1)) + 15) & ~15ull;
            return fit(rows_, (u32) std::min<u64>(grow_cap(mx), std::max<u64>(64, mean4)));
        };
        if (nb.cap_leaf == 0) nb.cap_leaf = fit(L, 128);
        if (nb.cap_part == 0) nb.cap_part = fit(nm, 256);
        if (const char *e = std::getenv("SHAMX_NEIGH_CAP")) { // tests: force overflow
            nb.cap_leaf = nb.cap_part = std::max(16, std::atoi(e)) & ~15;
        }
        u32 *mism_len = nb.counters.data() + 5;
        const u32 big = std::max(L, nm);
        for (auto *a_ : {&nb.oflag, &nb.ocnt, &nb.ofpos, &nb.opos, &nb.olist}) a_->resize(big);
        // list the rows of cnt[0, n) longer than cap (map: their labels) with their offsets
        // from `base` on, where the host knows that there are some
        auto list_over = [&](u32 n, const u32 *cnt, u32 cap, u64 base, const u32 *map,
                             u32 *offset) {
            k_over_mark<<<div_up(n, 256), 256, 0, s>>>(n, cnt, cap, nb.oflag.data(),
                                                        nb.ocnt.data());
            exclusive_scan_u32(s, nb.oflag.data(), nb.ofpos.data(), n, nullptr,
                               nb.scratch.data());
            exclusive_scan_u32(s, nb.ocnt.data(), nb.opos.data(), n, nullptr, nb.scratch.data());
            k_over_list<<<div_up(n, 256), 256, 0, s>>>(n, nb.oflag.data(), nb.ofpos.data(),
                                                        nb.opos.data(), (u32) base, map,
                                                        nb.olist.data(), offset);
        };
        // the n_over leaves whose lists (of `tot` entries in all) are longer than cl, one per
        // wave, into the overflow region of leaf_ids
        auto resolve_leaves = [&](u32 cl, u32 n_over, u32 tot) {
            const u64 base = (u64) L * cl;
            if (base + tot > 0xffffffffull)
                throw std::runtime_error("neighbour cache: leaf lists exceed u32 entry indices");
            nb.leaf_ids.resize_keep(std::max<u64>(base + tot, 1), s);
            list_over(L, nb.leaf_cnt.data(), cl, base, nullptr, nb.leaf_offset.data());
            k_leaf_lists<LEAF_FILL, true>
                <<<div_up(n_over, (u32) LW_WAVES), LW_WAVES * WAVE, 0, s>>>(
                    L, I, t.nodes.data(), t.tiers.data(), t.tt, Rkern, nb.leaf_cnt.data(),
                    nb.leaf_offset.data(), nb.leaf_ids.data(), 0, nb.lap.data(),
                    nb.olist.data(), n_over);
        };
        for (int attempt = 0;; attempt++) {
            if (attempt == 4) throw std::runtime_error("neighbour cache: capacities do not settle");
            u32 cl = nb.cap_leaf, cp = nb.cap_part;
            if (attempt) {
                fill_u32(s, mism_len, 0, 1);
                fill_u32(s, nb.counters.data() + 8, 0, 8);
            }
            if ((u64) L * cl > 0xffffffffull) {
                // u32 entry indices cannot address fixed-capacity leaf lists: two passes each
                packed_leaves();
                owners(s, nb, t, n_local, gblocks, 0);
                stage2_packed<true>(s, nb, t, n_local, gblocks, x, y, z, h, htol, Rker2, hc);
                nb.leaf_stride = 0;
                nb.row_stride  = 0;
                nb.cap_leaf    = choose(hc[8], nb.n_leaf_pairs, L, L);
                nb.cap_part    = choose(hc[9], nb.n_pairs, n_local, nm);
                break;
            }
            // stage 1: fixed-capacity leaf lists
            nb.leaf_ids.resize(std::max<u64>((u64) L * cl, 1));
            leaf_lists<LEAF_ROWS>(s, nb, t, Rkern, cl);
            row_stats(s, L, nb.leaf_cnt.data(), cl, nb.counters.data() + 8,
                      nb.counters.data() + 10, nb.counters.data() + 12);
            const bool packed        = (u64) nm * cp > 0xffffffffull || packed_rows_forced();
            const bool resolve_first = nb.leaf_overflowed || packed;
            if (resolve_first) {
                SHAMX_HIP(hipMemcpyAsync(hc, nb.counters.data(), 16 * sizeof(u32),
                                         hipMemcpyDeviceToHost, s));
                SHAMX_HIP(hipStreamSynchronize(s));
                if (hc[12]) resolve_leaves(cl, hc[12], hc[13]);
            }
            const u32 leaf_cap = resolve_first ? 0u : cl; // lists past cl are truncated
            owners(s, nb, t, n_local, gblocks, leaf_cap);
            if (packed) {
                // particle rows packed (count, scan, fill)
                const u32 n_leaf_pairs = hc[10];
                nb.leaf_overflowed     = hc[12] > 0;
                const u32 mxl          = hc[8];
                stage2_packed<true>(s, nb, t, n_local, gblocks, x, y, z, h, htol, Rker2, hc, 0);
                nb.n_leaf_pairs = n_leaf_pairs;
                nb.leaf_stride  = cl;
                nb.row_stride   = 0;
                nb.cap_leaf     = choose(mxl, n_leaf_pairs, L, L);
                nb.cap_part     = choose(hc[9], nb.n_pairs, n_local, nm);
                break;
            }
            // stage 2: fixed-capacity particle rows
            nb.ids.resize(std::max<u64>((u64) nm * cp, 1));
            launch_group<true, true, true>(s, gblocks, batch_boxes(s, nb, t, gblocks, htol, Rker2),
                n_local, L, I, t.nodes.data(), t.sort_index.data(), nb.ps.data(),
                nb.owner.data(), nb.lap.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(),
                nb.item_leaf.data(), nb.xstart.data(), nb.counters.data() + 7, htol, Rker2,
                nb.cnt.data(), nb.offset.data(), nb.ids.data(), cp, leaf_cap);
            k_part_neigh<true, true, true><<<div_up(n_local, 128), 128, 0, s>>>(
                n_local, nb.mism.data(), mism_len, I, t.nodes.data(), t.sort_index.data(),
                nb.owner.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(), nb.leaf_ids.data(), x,
                y, z, h, nb.inv.data(), htol, Rker2, nb.cnt.data(), nb.offset.data(),
                nb.ids.data(), cp, leaf_cap);
            row_stats(s, nm, nb.cnt.data(), cp, nb.counters.data() + 9, nb.counters.data() + 11,
                      nb.counters.data() + 14);
            SHAMX_HIP(hipMemcpyAsync(hc, nb.counters.data(), 16 * sizeof(u32),
                                     hipMemcpyDeviceToHost, s));
            SHAMX_HIP(hipStreamSynchronize(s));
            check_flags(hc[4]);
            if (!resolve_first && hc[12]) {
                // leaf lists overflowed for the first time: stage 2 read truncated lists
                nb.leaf_overflowed = true;
                continue;
            }
            nb.leaf_overflowed = hc[12] > 0;
            nb.n_leaf_pairs    = hc[10];
            nb.n_pairs         = hc[11];
            nb.n_mismatch      = hc[5];
            nb.leaf_stride     = cl;
            nb.row_stride      = cp;
            const u32 mxl = hc[8], mxp = hc[9];
            // particle rows past cp: list them (sorted positions -> particle ids) and fill each
            // again, one wave per row, into the overflow region of ids
            if (hc[14]) {
                const u64 base = (u64) nm * cp;
                if (base + hc[15] > 0xffffffffull)
                    throw std::runtime_error("neighbour cache: rows exceed u32 entry indices");
                nb.ids.resize_keep(base + hc[15], s);
                list_over(nm, nb.cnt.data(), cp, base, t.sort_index.data(), nb.offset.data());
                k_group_neigh<true, true, false, true>
                    <<<div_up(hc[14], (u32) GRP_WAVES), GRP_WAVES * WAVE, 0, s>>>(
                        n_local, L, I, t.nodes.data(), t.sort_index.data(), nb.ps.data(),
                        nb.owner.data(), nb.lap.data(), nb.leaf_cnt.data(), nb.leaf_offset.data(),
                        nb.leaf_ids.data(), nb.olist.data(), nullptr, nb.counters.data() + 14,
                        htol, Rker2, nullptr, nb.offset.data(), nb.ids.data(), 0, 0,
                        nb.inv.data());
            }
            nb.cap_leaf = choose(mxl, nb.n_leaf_pairs, L, L);
            nb.cap_part = choose(mxp, nb.n_pairs, n_local, nm);
            break;
        }
        nb.moved = hc[3];
        SHAMX_HIP(hipGetLastError());
    }

} // namespace shamx
