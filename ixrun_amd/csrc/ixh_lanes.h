// The lane layout: a second form of a packed tensor in which every code has a fixed place, made once when a layer is
// deployed and read by the products of up to four activation rows (ixh_lanes.hip), of up to 16 (ixh_lanes_rows.hip) and of
// more (ixh_lanes_gemm.hip, ixh_lanes_prompt.hip).
//
// The nested-bitmap streams locate a code by the number of codes before it, so a kernel that reads them spends most
// of its time on ranks: prefix sums over bitmap words, windows at bit offsets that depend on them, a splice or a
// gather per element (7 to 16 vector instructions a weight).  Here a weight is `bits` wide (3, 4, 5 or 8) and sits in
// the registers of the lane that multiplies it as soon as it is loaded; the few elements whose value does not fit go
// to a list.  The values are the same integers: nothing is rounded on the way.  (They are taken from the bf16 weights, so a tensor whose scale
// makes some of these infinite has no lane layout.)
//
//   cell      4 weight rows x 512 columns = 2048 weights, 64 lanes x `bits` dwords.  Cell (t, c) holds rows 4 t ..
//             4 t + 3 and columns 512 c ..; cells are stored row quads first: index t * n_cells + c.
//   lane l    row l % 4, slice s = l / 4 (q = s / 4, kg = s % 4) of the columns 128 q + 32 i + 8 kg + j, i < 4, j < 8:
//             32 weights, in pairs p = 4 i + j / 2.
//   dwords    the first min(bits, 4) of a lane are consecutive, lane after lane, so are the others behind them.
//   codes     value + 2^(bits-1) - 1; a listed element has the code of its sign, +1 or -1, which a kernel that adds the
//             list to the plane's products takes off again: with the code of 0 an infinite activation there would give NaN.
//             The padding of the last row quad and of the last cell of a row has the code of 0.
//   pairs     2 * bits wide, first element in the low half.  bits = 4: pair p in byte p % 4 of dword p / 4.
//             bits = 3: five pairs a dword from bit 2 on (p = 5 d + f at bit 2 + 6 f), the two low bits of the three
//             dwords are pair 15.  bits = 5: three a dword from bit 2 on (p = 3 d + f), the two low bits of the five
//             dwords are pair 15.  bits = 8: four bytes a dword, in element order.
//   listed    in quads, one element of each of a cell's four rows; row r's of quad n is at lane_listed(n, r), so that a
//             lane's four consecutive ones are of one row.  A cell has as many quads as its fullest row has listed elements
//             (the others end in value 0 at position lane_none()), from exc_off[cell] on (one more at the end).  exc_pos:
//             the byte offset of the element's column in activations kept in the order of lane_offset() below, from column
//             32768 * (column / 32768) on.
#pragma once
#include "ixh_dev.h"
#include "ixh_lanes_bounds.h"

namespace ixh {

constexpr uint32_t kLnCell = 2048;       // weights of a cell
constexpr uint32_t kLnCols = 512;        // columns of a cell
constexpr uint32_t kLnSegCells = 64;     // cells after which exc_pos starts over at column 0

// Byte offset of a column in activations kept for the lanes: the 64-byte blocks i = 0..3 of the columns of a slice
// group q at block i ^ q, so that the sixteen slices of a wave read from different banks.
__host__ __device__ inline uint32_t lane_offset(uint32_t col) {
    const uint32_t b = 2u * col;
    return b ^ ((b >> 2) & 0xC0u);
}

// Four quads are sixteen elements, four of each row in turn.
__host__ __device__ inline uint32_t lane_listed(uint32_t quad, uint32_t row) { return (quad >> 2) * 16u + row * 4u + (quad & 3u); }

// Where a quad's place without an element points: behind the row's last cell, where a kernel keeps an activation of 0 (value
// 0 times an infinite activation is NaN).  Rows of 64 and more cells have no offset left for that: 0, and the kernel looks at
// the value instead.
__host__ __device__ inline uint32_t lane_none(uint32_t n_cells) { return n_cells < kLnSegCells ? n_cells * 2u * kLnCols : 0u; }

struct LanesDev {
    const uint32_t *plane;
    const uint32_t *exc_off;
    const uint16_t *exc_pos;
    const int8_t *exc_val;
    const uint16_t *scale;
    uint32_t out_f, in_f, n_tiles, n_cells;
    uint32_t list_groups;  // whole groups of 64 quads that the list holds
    int bits;
};

// Scratch that a call was given; a launch that wants more sets `need`, starts nothing and returns IXH_EWORKSPACE.  How the work is
// cut decides what is needed, and finding the cut takes the host 0.3 to 3 us: it is found once, by the launch that uses it.
struct LnScratch {
    float *at;
    size_t bytes, need;
    bool holds(size_t n) {
        need = n;
        return !n || (at && bytes >= n);
    }
};

int launch_lanes_pack(const uint16_t *w, const LanesDev &L, uint32_t *plane, uint32_t *counts, hipStream_t s);
int launch_lanes_list(const uint16_t *w, const LanesDev &L, uint16_t *pos, int8_t *val, hipStream_t s);
// 1 to 16 rows; five and more, fewer too long for k_lanes_gemv (which takes no scratch), and two to four of very many row quads go on to
// launch_lanes_rows, and some of nine and more from there to launch_lanes_gemm
bool lanes_gemv_takes(const LanesDev &L, int m);
int launch_lanes_gemv(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                      int64_t ldy, LnScratch &ws, hipStream_t s);
size_t lanes_rows_workspace_bytes(const LanesDev &L, int m);  // in k_lanes_rows
size_t lanes_rows_workspace_most(const LanesDev &L);           // of any count from five to sixteen, whichever kernel takes it
int launch_lanes_rows(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y, int64_t ldy,
                      LnScratch &ws, hipStream_t s);
// 17 and more rows (ixh_lanes_gemm.hip), the bias added before the one rounding (once) or after one, then rounded again;
// IXH_EUNSUPPORTED unless lanes_gemm_aligned:
// x 16-byte aligned, in_f and ldx multiples of 8, x within 4 GB
bool lanes_gemm_aligned(const LanesDev &L, const uint16_t *x, int m, int64_t ldx);
size_t lanes_gemm_workspace_bytes(const LanesDev &L, int m);
int launch_lanes_gemm(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, bool once, uint16_t *y,
                      int64_t ldy, LnScratch &ws, hipStream_t s);
// of them, those of many rows and large layers (ixh_lanes_prompt.hip): x as above, the bias added once
bool lanes_prompt_wins(const LanesDev &L, int m);
size_t lanes_prompt_workspace_bytes(const LanesDev &L, int m);
int launch_lanes_prompt(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y, int64_t ldy,
                        LnScratch &ws, hipStream_t s);

}  // namespace ixh
