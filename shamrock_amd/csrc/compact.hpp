// SPDX-License-Identifier: CeCILL-2.1
//
// compact.hpp -- ordered compaction of a list in two launches over its tiles: tile_count writes
// the kept entries of every tile, tile_compact adds the counts of the tiles before its own (a few
// cached loads per thread), tests its entries again and emits the kept ones with their positions.
// Testing twice is cheaper than a pass over stored flags; flags, a two-launch scan and a
// compaction are four launches, each a few microseconds at any size below a few hundred thousand.
// A list of one tile needs tile_compact only.
//
// Tiles of 1024 entries up to 2^23 entries, where the chip is not full and a block's own time
// counts (the leaf reduction of 2.46 M positions: 67 us for its four iterations against 114 us
// with tiles of 4096, whose 600 blocks leave the chip half empty), 4096 beyond, where adding the
// counts of the earlier tiles, quadratic in their number, would weigh more.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace shamx {

    constexpr int CT_BLK       = 256;
    constexpr u32 CT_SMALL_MAX = 1u << 23;
    // entries per tile and tiles of a list of at most n entries
    inline u32 compact_items(u32 n) { return n <= CT_SMALL_MAX ? 4 : 16; }
    inline u32 compact_tiles(u32 n) { return div_up(n, CT_BLK * compact_items(n)); }
    // f(integral_constant of the entries per thread)
    template<class F>
    inline void compact_dispatch(u32 n, F &&f) {
        if (compact_items(n) == 4) f(std::integral_constant<int, 4>{});
        else f(std::integral_constant<int, 16>{});
    }

    // pred(j): entry j is kept; n: the list's length, same in every thread of the block
    template<int ITEMS, class Pred>
    __device__ inline void tile_count(u32 n, u32 *__restrict tile_cnt, Pred &&pred) {
        __shared__ u32 part[CT_BLK / WAVE];
        const u32 t0 = blockIdx.x * (CT_BLK * ITEMS);
        u32 c        = 0;
        if (t0 < n) {
#pragma unroll 4
            for (int k = 0; k < ITEMS; k++) {
                const u32 j = t0 + k * CT_BLK + threadIdx.x;
                c += (u32) __popcll(__ballot(j < n && pred(j)));
            }
        }
        if (__lane_id() == 0) part[threadIdx.x / WAVE] = c;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < CT_BLK / WAVE; w++) c += part[w];
            tile_cnt[blockIdx.x] = c;
        }
    }

    // emit(p, j) for the kept entries j, p their position in the compacted list; total(c) in one
    // thread of the grid with the number of kept entries.  all: every entry is kept (no counts
    // are read).
    template<int ITEMS, class Pred, class Emit, class Total>
    __device__ inline void tile_compact(u32 n, const u32 *__restrict tile_cnt, u32 nt, bool all,
                                        Pred &&pred, Emit &&emit, Total &&total) {
        constexpr int NW = CT_BLK / WAVE;
        static_assert(ITEMS * NW <= WAVE, "one wave scans the counts");
        __shared__ u32 part[NW];
        __shared__ u32 cnt[ITEMS * NW]; // kept entries per 64 of the tile, then before it
        const u32 t0   = blockIdx.x * (CT_BLK * ITEMS);
        const u32 lane = (u32) __lane_id(), wid = threadIdx.x / WAVE;
        // kept entries of the earlier tiles; block 0 adds all of them for the total
        u32 before = all ? t0 : 0u;
        if (all) {
            if (blockIdx.x == 0 && threadIdx.x == 0) total(n);
        } else if (nt > 1) {
            const u32 lim = blockIdx.x == 0 ? nt : blockIdx.x;
#pragma unroll 4
            for (u32 i = threadIdx.x; i < lim; i += CT_BLK) before += tile_cnt[i];
            before = wave_reduce(before, [](u32 p, u32 q) { return p + q; });
            if (lane == 0) part[wid] = before;
            __syncthreads();
            before = 0;
            for (int w = 0; w < NW; w++) before += part[w];
            if (blockIdx.x == 0) {
                if (threadIdx.x == 0) total(before);
                before = 0;
            }
        }
        if (t0 >= n) { // block-uniform
            if (!all && nt == 1 && threadIdx.x == 0) total(0);
            return;
        }
        u64 bal[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            const u32 j = t0 + k * CT_BLK + threadIdx.x;
            bal[k]      = __ballot(j < n && pred(j));
            if (lane == 0) cnt[k * NW + wid] = (u32) __popcll(bal[k]);
        }
        __syncthreads();
        if (wid == 0) {
            const u32 v = lane < ITEMS * NW ? cnt[lane] : 0u;
            u32 inc     = v;
            for (int o = 1; o < WAVE; o <<= 1) {
                u32 t = __shfl_up(inc, o, WAVE);
                if ((int) lane >= o) inc += t;
            }
            if (lane < ITEMS * NW) cnt[lane] = inc - v;
            if (!all && nt == 1 && lane == WAVE - 1) total(inc);
        }
        __syncthreads();
        const u64 lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
        for (int k = 0; k < ITEMS; k++) {
            if ((bal[k] >> lane) & 1ull)
                emit(before + cnt[k * NW + wid] + (u32) __popcll(bal[k] & lt),
                     t0 + k * CT_BLK + threadIdx.x);
        }
    }

} // namespace shamx
