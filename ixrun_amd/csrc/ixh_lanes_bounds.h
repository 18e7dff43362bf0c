// What a wave of k_lanes_gemv and k_lanes_gemv_few (ixh_lanes.hip) asks for ahead of knowing whether it needs it, and where the workgroups of
// k_lanes_prompt (ixh_lanes_prompt.hip) leave their sums.  Plain C++, so that the ranges can be walked without a GPU.
#pragma once
#include <stdint.h>

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

}  // namespace ixh
