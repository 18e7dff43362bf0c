// What a wave of k_lanes_gemv and k_lanes_gemv_few (ixh_lanes.hip) asks for ahead of knowing whether it needs it, where the workgroups of
// k_lanes_prompt (ixh_lanes_prompt.hip) leave their sums, and how the work of k_lanes_gemm (ixh_lanes_gemm.hip) is cut.  Plain C++, so that
// the ranges can be walked without a GPU.
#pragma once
#include <stdint.h>

#include <algorithm>

#ifdef __HIPCC__
#define LN_BOTH __host__ __device__ __forceinline__
#else
#define LN_BOTH inline
#endif

namespace ixh {

// The list's groups (64 quads each) of a share of cells whose listed quads are first_quad .. end_quad - 1, in a list of
// `groups` groups (at least one).  The first group is asked for whether the share lists anything or not, and behind the
// last listed quad of a full list there is none: `last` bounds every request, `n` is how many groups count.
struct LnGroups {
    uint32_t first, last, n;
};
LN_BOTH LnGroups ln_groups(uint32_t first_quad, uint32_t end_quad, uint32_t groups) {
    const uint32_t first = first_quad >> 6, end = (end_quad + 63u) >> 6;
    const uint32_t last = (end > first ? end : first + 1u) - 1u;
    return {first, last < groups ? last : groups - 1u, end_quad > first_quad ? last - first + 1u : 0u};
}

// k_lanes_gemv_few asks for 64 quads at a time from quad `from` (a multiple of four) on, four of them a lane: which four, of a cell
// whose listed quads end at `end`.  Behind the last ones these are asked for again, also by a cell without any at a full list's end.
LN_BOTH uint32_t ln_four_quads(uint32_t from, uint32_t lane, uint32_t end) {
    const uint32_t at = (from >> 2) + (lane >> 2), last = (end ? end - 1u : 0u) >> 2;
    return at < last ? at : last;
}

// Byte offset, in a row of `cells` cells of activations, of a listed element at position `pos` of segment `seg` (64 cells each), for rows
// of a whole segment and more: a position of another segment's quad may lie behind the row, and a place without an element (value
// 0) holds position 0: both go to the zeros behind the last cell.  `in_range`: the quad is of the row quad and segment in work.
LN_BOTH uint32_t ln_listed_at(uint32_t pos, uint32_t value, bool in_range, uint32_t seg, uint32_t cells) {
    return value && in_range ? seg * 65536u + pos : cells * 1024u;
}

// A workgroup's cells are dealt to its 2^log_waves waves in runs: wave w has the cells ln_share(n, w) .. ln_share(n, w + 1) - 1.  The
// first of sixteen waves has 1.47 times the mean, the last one 0.53 times: a SIMD serves the oldest of its waves first, so the last ones
// have their first cells 1.4 us after the first ones and in even shares end 1.6 to 2 us after them (us a layer, even shares /
// 1.12 .. 0.88 / 1.23 .. 0.77 / 1.47 .. 0.53 / 1.6 .. 0.4 of the mean: 17408 x 5120 at 5 bits 14.4 / 14.2 / 14.0 / 13.8 / 14.1, 5120 x
// 5120 7.3 / 7.2 / 7.3 / 7.0 / 7.1, 5120 x 17408 at 3 bits 10.4 / 10.5 / 10.2 / 10.5 / 10.8).  That lead does not grow with the layer: from
// 256 cells on the first wave has 7.5 more than the mean (8192 x 65536 at 3 bits with 0.53 to 1.47 of it 52.3, so 47.1).
LN_BOTH uint32_t ln_share(uint32_t n, uint32_t wave, uint32_t log_waves) {
    return (32u * n * wave + (n < 256u ? n : 256u) * wave * ((1u << log_waves) - wave)) >> (log_waves + 5u);
}

// Activations: 16-byte pieces of whole rows are asked for before anything else where every row starts 16-byte aligned and
// has a whole piece; of the pieces past a row's last whole one that one is asked for again.
LN_BOTH bool ln_whole_pieces(uint64_t x, uint32_t in_f, int m, int64_t ldx) {
    return (x & 15u) == 0 && in_f >= 8u && (m == 1 || ldx % 8 == 0);
}
LN_BOTH uint32_t ln_piece_column(uint32_t col, uint32_t in_f) {  // in_f >= 8
    const uint32_t last = (in_f & ~7u) - 8u;
    return col < last ? col : last;
}

// `groups` workgroups share `tiles` tiles of `cells` cells each in runs that differ by one cell at most: workgroup g has the
// cells lp_begin(g) .. lp_begin(g + 1) - 1, counted through the tiles.  tiles * cells * groups is below 2^32.
LN_BOTH uint32_t lp_begin(uint32_t g, uint32_t groups, uint32_t tiles, uint32_t cells) { return g * (tiles * cells) / groups; }
LN_BOTH uint32_t lp_group_of(uint32_t cell, uint32_t groups, uint32_t tiles, uint32_t cells) {
    return ((cell + 1u) * groups - 1u) / (tiles * cells);
}

// Of a tile that it has a part of only, a workgroup leaves its sums in memory; a whole tile it finishes by itself.  A run begins
// inside one tile at most and ends inside one other: part g is workgroup g's of the tile that its run begins in, and behind
// those come the parts of tiles that a run ends in, by tile (the first one is never among them) or by workgroup, whichever are
// fewer.  There are none of these where every tile has its own workgroups, and no parts at all where every workgroup has whole tiles.
LN_BOTH uint32_t lp_part(uint32_t g, uint32_t tile, bool begins, uint32_t groups, uint32_t tiles) {
    return begins ? g : groups + (tiles <= groups ? tile - 1u : g);
}
LN_BOTH uint32_t lp_parts(uint32_t groups, uint32_t tiles) {
    if (tiles % groups == 0) return 0;
    if (groups % tiles == 0) return groups;
    return groups + (tiles < groups ? tiles : groups) - 1u;
}

// k_lanes_gemm: blocks of 16 weight rows that a workgroup has in work at a time, and the most blocks of 16 activation rows.
constexpr uint32_t kLgBlocks = 16;
constexpr uint32_t kLgMost = 8;

// n things to k parts, floor(i n / k) in front of part i, without a division in the kernel: four of them in front of the first request took
// 0.5 us a launch (5 bits, 9 rows of 512 x 512 5.40 -> 4.78 us, 17 of 2048 x 2048 8.29 -> 7.83).  The first parts having one more
// instead takes up to 6 % more (9216 x 5120 at 5 bits, 9 to 32 rows).  (Plain arguments: a structure's members are not in registers when the kernel starts.)
struct LgSplit {
    uint32_t share, more;  // a part's whole share, and the rest of it in 2^-32, rounded up: exact for up to 2^16 parts
    LgSplit(uint32_t n, uint32_t k) : share(n / k), more((uint32_t)((((uint64_t)(n % k) << 32) + k - 1u) / k)) {}
};
LN_BOTH uint32_t lg_first(uint32_t i, uint32_t share, uint32_t more) { return i * share + (uint32_t)((uint64_t)i * more >> 32); }

// Rounds of a workgroup with `own` blocks, and the blocks of a round (the last one may have fewer).  `most_at_once`: those of the launch's
// largest workgroups, whose rounds are even.  A workgroup of one block less has as many rounds, in which that is enough, or one round less: its
// blocks are then whole rounds of kLgBlocks.
LN_BOTH uint32_t lg_rounds(uint32_t own) { return (own + kLgBlocks - 1u) / kLgBlocks; }
LN_BOTH uint32_t lg_at_once(uint32_t own, uint32_t most_at_once) {
    return own % kLgBlocks == 0u ? kLgBlocks : own < kLgBlocks ? own : most_at_once;
}
LN_BOTH uint32_t lg_most_at_once(uint32_t blocks, uint32_t groups) {
    const uint32_t most = (blocks + groups - 1u) / groups, rounds = lg_rounds(most);
    return (most + rounds - 1u) / rounds;
}

// How the work is cut: groups of 16 .. 128 activation rows, slices of the columns and groups of 16-row blocks, a workgroup
// per CU. Of all such cuts the one with the shortest estimate, in units of some half nanosecond: 250 for each block of weights that a SIMD has
// in a stage (its vector instructions), 125 for each 16 activation rows, 3 for each of these and block (operands read from LDS), and no
// less than the way of a stage's requests and activations takes with few blocks; the slices' sums cost a launch and their way through memory.
// Fitted to all cuts, timed, of 52 shapes from 256 x 4096 to 17408 x 5120 at 9 to 160 rows and 3, 5 and 8 bits: within 0.55 % of the shortest
// in the mean, 13 % at worst (1.2 and 33 without that least, which cut long rows so that a workgroup has few blocks and many cells: 2048 x 17408
// at 16 rows 18.4 us against 14.3, 8192 x 2048 (5 bits) at 64 rows 18.9 against 16.2).  Where it errs, a call takes up to 4 % more than by the
// estimate that it replaced: 9952 x 4160 (4 bits) at 113 rows 36.2 -> 37.8 us, 10560 x 2048 (5 bits) at 94 23.8 -> 24.6, 544 x 6272 (8 bits) at 160
// 12.6 -> 13.2, 7552 x 544 (5 bits) at 33 10.4 -> 10.8.
struct LgPlan { uint32_t m_groups, mb, slices, groups; };
inline LgPlan lg_plan(uint32_t n_tiles, uint32_t n_cells, int m, uint32_t all_cus) {
    const uint32_t blocks = (n_tiles + 3u) / 4u, m_blocks = ((uint32_t)m + 15u) / 16u;
    LgPlan best{};
    uint64_t best_cost = ~0ull;
    for (uint32_t m_groups = (m_blocks + kLgMost - 1u) / kLgMost; m_groups <= std::max((m_blocks + 1u) / 2u, 1u); ++m_groups) {
        const uint32_t mb = (m_blocks + m_groups - 1u) / m_groups, cus = std::max(all_cus / m_groups, 1u);
        for (uint32_t s = 1; s <= std::min(n_cells, cus); ++s) {
            const uint32_t groups = std::min(std::max(cus / s, 1u), blocks);
            const uint32_t share = (blocks + groups - 1u) / groups, rounds = lg_rounds(share);
            const uint32_t at_once = (share + rounds - 1u) / rounds, cells = (n_cells + s - 1u) / s;
            const uint64_t stage = std::max(250u * ((at_once + 3u) / 4u) + 125u * mb + 3u * mb * at_once, 400u + 115u * mb);
            const uint64_t sums = s > 1 ? 1600u + (uint64_t)s * (uint32_t)m * blocks * 16u / 670u : 0u;
            const uint64_t cost = 4u * stage * rounds * cells + sums;
            if (cost < best_cost) { best_cost = cost; best = {m_groups, mb, s, groups}; }
        }
        if (m_groups * 2u > all_cus) break;
    }
    return best;
}

}  // namespace ixh
