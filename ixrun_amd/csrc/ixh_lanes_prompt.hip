// Products of many activation rows with weights in the lane layout (ixh_lanes.h): decode and matrix products side by side.
#include <algorithm>

#include "ixh_lanes_dev.h"

namespace ixh {

constexpr uint32_t kLpWaves = 8, kLpThreads = kLpWaves * kWave;
constexpr uint32_t kLpRows = 16u * kLpWaves;         // weight rows of a workgroup
constexpr uint32_t kLpTile = kLpRows * 128u * 2u;    // bytes of a stage's weights: 128 rows x 128 columns
constexpr uint32_t kLpRounds = 3;                    // groups of 16 quads of a cell's list that a wave holds

__host__ __device__ constexpr uint32_t lp_tiles(uint32_t n_quads) { return (n_quads * 4u + kLpRows - 1u) / kLpRows; }

struct LpOut {
    const uint16_t *bias;
    uint16_t *y;
    int64_t ldy;
    uint32_t m, out_f, wide;  // wide: y and ldy allow stores of 8 bytes
    uint32_t parts;           // lp_parts: of tiles, for each group of activation rows
};
// four weight rows' sums of activation row r: the bias is added before the one rounding
__device__ __forceinline__ void lp_store(const LpOut &out, uint32_t r, uint32_t row, ln_f32x4 sum) {
    if (r >= out.m || row >= out.out_f) return;
    uint16_t *const to = out.y + (int64_t)r * out.ldy + row;
    uint16_t v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        v[k] = (uint16_t)f32_to_bf16_bits(sum[k] + (out.bias && row + k < out.out_f ? bf16_bits_to_f32(out.bias[row + k]) : 0.0f));
    if (out.wide && row + 4u <= out.out_f) {
        *reinterpret_cast<ln_u32x2 *>(to) = ln_u32x2{v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16};
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (row + k < out.out_f) to[k] = v[k];
    }
}

constexpr uint32_t kLpXBlocks = 2;  // row blocks of a workgroup of k_lanes_xtile

// Bound: memory (5120 x 17408 at 512 rows: 36 MB in 7.9 us under the profiler; 9.1 with a branch around each request, 8.0 to 9.4 with one,
// four or eight row blocks a workgroup, or with half or four times its column blocks).  X [m][in_f] row-major -> operand order: block (kb, mb), 32 columns x 16 rows, is 1 KB, lane l's 16 bytes are row l % 16, columns
// 8 (l / 16) .. + 7; zeros past the last row and column.  A workgroup writes four column blocks of two row blocks, so that
// whole lines are read; rows past the last are the last one's (no result has part in them).
__global__ void __launch_bounds__(256)
k_lanes_xtile(const uint16_t *__restrict__ x, int64_t ldx, uint32_t m, uint32_t in_f, uint32_t n_kb, uint32_t n_mblk,
              ln_u32x4 *__restrict__ xt) {
    const uint32_t lane = threadIdx.x & 63u, kb = blockIdx.x * 4u + (threadIdx.x >> 6), col = kb * 32u + (lane >> 4) * 8u;
    const uint16_t *const from = x + min(col, in_f - 8u);
    ln_u32x4 v[kLpXBlocks];
#pragma unroll
    for (uint32_t j = 0; j < kLpXBlocks; ++j)
        v[j] = *reinterpret_cast<const ln_u32x4 *>(from + (int64_t)min((blockIdx.y * kLpXBlocks + j) * 16u + (lane & 15u), m - 1u) * ldx);
    ln_u32x4 *const to = xt + ((size_t)kb * n_mblk + blockIdx.y * kLpXBlocks) * 64u + lane;
#pragma unroll
    for (uint32_t j = 0; j < kLpXBlocks; ++j)
        if (blockIdx.y * kLpXBlocks + j < n_mblk) to[j * 64u] = col < in_f ? v[j] : ln_u32x4{0u, 0u, 0u, 0u};
}

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_prompt<BITS, MI, NW>: 128 MI / NW activation rows by 128 weight rows a workgroup, over a run of the cells of a tile.
//
// Bound: the matrix unit and what stands between two stages.  5120 x 17408 at 512 rows (3 bits): 97 us a call; one after the other
// under the profiler 86 to 96 for this kernel, 8 for the activations' reordering and 11 for adding the sums (63 MB read).  (Which blocks share
// an XCD's L2 matters little: all of an XCD on the same columns 2 to 4 % slower, on neighbouring runs up to 3 %.  Operands straight from
// row-major activations: 126 instead of 88.)  The
// products would take 58 at the rate of a large library product; decode into memory and that library's product took 126.  Clocks a stage
// of a wave, 7500 in all, of which its products are 2048 (and its neighbour's on the SIMD as many): first operand with the decode
// 1750, the others 700 to 1050 each, listed elements 700, a stage's share of a cell's list 700, barrier 1150.  A cell's list is worked
// out in the rounds that have elements, and stored in the stages that a round has any in: 3 bits at 192 / 256 / 384 / 512 rows 53.9 / 61.0 /
// 77.6 / 98.5 -> 51.6 / 58.8 / 76.0 / 95.6, 9120 x 9216 at 5 bits 57.5 / 65.0 / 79.4 / 98.9 -> 55.0 / 62.8 / 77.4 / 96.8.  Operands of
// weights two or three blocks ahead change nothing.
//
// Eight waves decode 128 rows x 128 columns a stage to LDS in operand order, 16 rows each, while they multiply the stage before: the
// pairs of a wave's next stage are looked up between the products of its first four operands (a decode of its own before the products
// left the matrix unit idle meanwhile: 84 -> 81 us at 384 rows, 72 -> 65 at 256).  Each weight is decoded once for up to 512 rows; the
// activations come from the L2 straight to registers as operands (k_lanes_xtile), two or four steps ahead: they are shared by no other
// wave of the workgroup, and through LDS they would take its time from the lookups and the weights.  MI x 16 rows by 128 / NW weight
// rows of sums a wave: 128 registers at 512 rows, so the rest is kept small: operands of weights read one block ahead, listed elements
// worked out once a cell and kept in LDS, places recomputed.  All the same <BITS, 4, 1>, 385 to 512 rows, has all 256 registers in
// use and 11 / 14 / 16 / 18 more (at 3 / 4 / 5 / 8 bits; 48 to 76 bytes a lane) in memory; the other forms spill none.  Requests are never
// inside a branch or past a way out, else they are all waited for at the join (with the last stage peeled by conditions the same loop
// took 110 us at 512 rows, and a form whose loop spilled its sums 287).
//
// Parts of a tile meet in the workspace and k_lanes_prompt_reduce adds them in the columns' order; a workgroup with the whole of a tile
// writes y itself (32768 x 4096, 512 rows: 160 -> 130 us).
// ---------------------------------------------------------------------------------------------------------------
template <int BITS, int MI, int NW>
__global__ void __launch_bounds__(kLpThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_lanes_prompt(const uint32_t *__restrict__ plane, const ln_u32x4 *__restrict__ xt, const uint32_t *__restrict__ exc_off,
               const uint16_t *__restrict__ scale_at, uint32_t n_cells, uint32_t n_tiles, uint32_t n_mblk,
               const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val, ln_f32x4 *__restrict__ ws, LpOut out) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lp_smem[];
    using P = LnPairs<BITS, true>;
    constexpr uint32_t NI = 8 / NW, MW = 8 / NW;  // weight blocks of a wave, waves along the activation rows
    constexpr uint32_t AHEAD = MI * NI >= 16 ? 2 : 4;  // steps of 32 columns that the activations' operands are asked for ahead
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)lp_smem;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 15u, kg = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t mg = blockIdx.y, mw = wave % MW, nw = wave / MW;
    const uint32_t mb0 = (mg * MW + mw) * MI;  // the wave's first block of activation rows
    const uint32_t scale_raw = *scale_at;
    const float scale = bf16_bits_to_f32(scale_raw);
    // The table of pairs behind the first tile's requests (0.4 us of 49 to 76); at 512 rows in front of them, where that leaves eight
    // registers fewer in memory (0.9 us of 96).
    constexpr bool LUT_FIRST = MI == 4 && NW == 1;
    constexpr bool FLOAT = !LUT_FIRST;  // (its spilled registers: 96.4 us with shifts, 97.3 so; 256 rows 56.8 and 56.1)
    if constexpr (LUT_FIRST) ln_build_lut<BITS, true>(smem, scale, tid, kLpThreads);
    const uint32_t u_end = lp_begin(blockIdx.x + 1u, gridDim.x, lp_tiles(n_tiles), n_cells);
    bool begins = true;  // the run, in this tile
#pragma unroll 1
    for (uint32_t u = lp_begin(blockIdx.x, gridDim.x, lp_tiles(n_tiles), n_cells); u < u_end; begins = false) {
        const uint32_t tile = u / n_cells, c0 = u - tile * n_cells, c1 = min(n_cells, c0 + u_end - u);
        u += c1 - c0;

        // ---- the wave's part of the decode: block `wave` of the workgroup's eight, lane (n, kg) the codes of row n ----
        const uint32_t quad0 = (tile * kLpWaves + wave) * 4u;  // the block's first row quad
        const uint32_t first = min(quad0, n_tiles - 1u), per_quad = n_cells * (256u * BITS);
        const __amdgpu_buffer_rsrc_t codes_rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(reinterpret_cast<const uint8_t *>(plane) + (size_t)first * per_quad), 0, (int)(min(n_tiles - first, 4u) * per_quad), 0x00020000);
        const uint32_t in_cell = 4u * kg + (n & 3u), codes_at = (min(quad0 + (n >> 2), n_tiles - 1u) - first) * per_quad + in_cell * (BITS == 3 ? 12u : 16u);
        constexpr uint32_t CODES = MI * NI >= 32 ? 1 : 2;  // stages that the codes are asked for ahead of their decode: long stages need one
        uint32_t w[CODES][BITS];
        auto codes = [&](uint32_t c, uint32_t q) {
            const uint32_t at = c * (256u * BITS) + q * (BITS == 3 ? 192u : 256u);
            uint32_t(&d)[BITS] = w[q % CODES];
            if constexpr (BITS == 3) {
                const ln_u32x3 v = __builtin_bit_cast(ln_u32x3, __builtin_amdgcn_raw_buffer_load_b96(codes_rs, (int)codes_at, (int)at, 0));
                d[0] = v[0]; d[1] = v[1]; d[2] = v[2];
            } else {
                const ln_u32x4 v = __builtin_bit_cast(ln_u32x4, __builtin_amdgcn_raw_buffer_load_b128(codes_rs, (int)codes_at, (int)at, 0));
                d[0] = v[0]; d[1] = v[1]; d[2] = v[2]; d[3] = v[3];
                if constexpr (BITS == 5)
                    d[4] = __builtin_amdgcn_raw_buffer_load_b32(codes_rs, (int)(codes_at - 12u * in_cell), (int)(at + 1024u - q * 192u), 0);
                if constexpr (BITS == 8) {
                    const ln_u32x4 u = __builtin_bit_cast(ln_u32x4, __builtin_amdgcn_raw_buffer_load_b128(codes_rs, (int)codes_at, (int)(at + 1024u), 0));
                    d[4] = u[0]; d[5] = u[1]; d[6] = u[2]; d[7] = u[3];
                }
            }
        };
        // (The list's steps are those of k_lanes_gemm, each kernel with a form of its own: as functions of ixh_lanes_dev.h they left this
        // one as it is, and k_lanes_gemm<5 | 8, 7 | 8, 2> with 10 to 21 registers in memory.)
        struct Extent { uint32_t first, end; };
        // the lane's place in a list, worked out where it is used: held over the loop it would cost registers that the sums need
        struct Place { uint32_t row, quad, kg; };
        auto place = [&] {
            uint32_t l = lane;
            asm volatile("" : "+v"(l));
            return Place{l & 3u, l & 12u, l >> 4};
        };
        auto extent = [&](uint32_t c) {
            const uint32_t t = quad0 + place().kg, cell = min(t, n_tiles - 1u) * n_cells + min(c, c1 - 1u);
            const uint32_t a = exc_off[cell], b = exc_off[cell + 1u];
            return Extent{a, t < n_tiles ? b : a};
        };
        struct Quads { ln_u32x2 pos[kLpRounds]; uint32_t val[kLpRounds]; };
        auto quads = [&](const Extent &e) {
            Quads l;
            const Place me = place();
#pragma unroll
            for (uint32_t r = 0; r < kLpRounds; ++r) {
                const uint32_t quad = (e.first & ~3u) + me.quad + 16u * r, at = quad < e.end ? lane_listed(quad, me.row) : 0u;
                l.pos[r] = *reinterpret_cast<const ln_u32x2 *>(exc_pos + at);
                l.val[r] = *reinterpret_cast<const uint32_t *>(exc_val + at);
            }
            return l;
        };
        codes(c0, 0);
        if (CODES == 2) codes(c0, 1);
        Extent e_now = extent(c0);
        Quads list = quads(e_now);

        const uint32_t x_step = n_mblk * 1024u;
        const __amdgpu_buffer_rsrc_t x_rs =
            __builtin_amdgcn_make_buffer_rsrc((void *)xt, 0, (int)(n_cells * 16u * x_step), 0x00020000);
        ln_u32x4 a[AHEAD][MI];
        auto x_load = [&](uint32_t c, uint32_t t) {  // step t of the cell's sixteen: place t % 4 of stage q holds columns 32 (t % 4 ^ q)
            const uint32_t at = (16u * c + (t ^ (t >> 2))) * x_step + mb0 * 1024u;
#pragma unroll
            for (uint32_t i = 0; i < MI; ++i)
                a[t % AHEAD][i] = __builtin_bit_cast(ln_u32x4, __builtin_amdgcn_raw_buffer_load_b128(x_rs, (int)(lane * 16u), (int)(at + i * 1024u), 0));
        };
#pragma unroll
        for (uint32_t t = 0; t < AHEAD; ++t) x_load(c0, t);
        if (!LUT_FIRST && begins) ln_build_lut<BITS, true>(smem, scale, tid, kLpThreads);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

        const uint32_t lut_lane = smem + ((lane & ((1u << P::kCopies) - 1u)) << 2);
        const uint32_t store_at = smem + P::kLutBytes + wave * 4096u;
        const LN_LDS(ln_u32x4) *const w_at = reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(smem + P::kLutBytes + nw * (NI * 4096u) + lane * 16u));
        LN_LDS(ln_u32x4) *const put_at = reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(smem + P::kLutBytes + 2u * kLpTile + tid * (16u * kLpRounds)));
        uint32_t in_stage[kLpRounds];  // bit q: the block has elements of the cell's stage q in the round
        bool any[kLpRounds], more;    // (8 bits list next to nothing: whether it has any, which takes fewer registers)
        uint32_t c_put;
        // listed elements of a cell: value (high half), where it goes in the wave's part of a stage's tile (bits 0 .. 11), the stage of
        // the cell (bits 12 .. 14; none of the four where there is no element)
        auto take_list = [&](uint32_t c) {
            c_put = c;
            const Place me = place();
#pragma unroll
            for (uint32_t r = 0; r < kLpRounds; ++r) {
                if constexpr (BITS != 8) {
                    in_stage[r] = 0;
                    if (!__any((e_now.first & ~3u) + 16u * r < e_now.end)) continue;
                }
                const uint32_t quad = (e_now.first & ~3u) + me.quad + 16u * r;
                ln_u32x4 put;
                uint32_t stages = 0;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const uint32_t p = (k & 1) ? list.pos[r][k >> 1] >> 16 : list.pos[r][k >> 1];
                    const int v = quad + k - e_now.first < e_now.end - e_now.first ? (int)(list.val[r] << (24 - 8 * k)) >> 24 : 0;
                    put[k] = (ln_pack(0.0f, (float)v * scale) & 0xFFFF0000u) | (v != 0 ? (p & 0x300u) << 4 : 0x4000u) |
                                     (((p & 0xF0u) << 4) + (p & 14u) + (me.kg << 6) + me.row * 16u);
                    if constexpr (BITS != 8) stages |= 1u << ((put[k] >> 12) & 7u);
                }
                put_at[r] = put;
                if constexpr (BITS == 8) any[r] = __any((e_now.first & ~3u) + 16u * r < e_now.end);
                else
#pragma unroll
                    for (uint32_t q = 0; q < 4; ++q) in_stage[r] |= (uint32_t)(__any(stages & (1u << q)) != 0) << q;
            }
            more = __any((e_now.first & ~3u) + 16u * kLpRounds < e_now.end);
            e_now = extent(c + 1u);
        };
        auto store = [&](uint32_t q) {  // stage q of the cell, to its half of the tile
            const uint32_t base = store_at + (q & 1u) * kLpTile;
            uint32_t o[16];
            ln_decode<BITS, true, FLOAT>(w[q % CODES], lut_lane, scale, o);
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(base + ((k ^ q) << 10) + lane * 16u)) =
                    ln_u32x4{o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]};
        };
        auto patch = [&](uint32_t q) {  // the listed elements of that stage over it
            const uint32_t base = store_at + (q & 1u) * kLpTile;
            ln_wave_order();
#pragma unroll
            for (uint32_t r = 0; r < kLpRounds; ++r)
                if (BITS == 8 ? any[r] : (in_stage[r] & (1u << q)) != 0) {
                    const ln_u32x4 put = put_at[r];
                    if constexpr (MI == 4) {
#pragma unroll
                        for (uint32_t e = 0; e < 4; ++e)
                            if ((put[e] & 0x7000u) == (q << 12))
                                *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(base + (put[e] & 0xFFFu))) = (uint16_t)(put[e] >> 16);
                    } else {  // (elements of other stages go aside, a dword a lane: where there are the registers, shorter than a branch each)
                        const Place me = place();
                        const uint32_t aside = smem + P::kLutBytes + 2u * kLpTile + kLpThreads * (16u * kLpRounds) + (me.kg * 16u + me.quad + me.row) * 4u;
#pragma unroll
                        for (uint32_t e = 0; e < 4; ++e) {
                            const uint32_t to = (put[e] ^ (q << 12)) & 0x7FFFu;
                            *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(to < 4096u ? base + to : aside)) = (uint16_t)(put[e] >> 16);
                        }
                    }
                }
            if (more) {  // rows with yet more listed elements in the cell
                const Extent e_put = extent(c_put);
                const Place me = place();
                for (uint32_t f = (e_put.first & ~3u) + 16u * kLpRounds + (me.quad >> 2); f < e_put.end; f += 4u) {
                    const uint32_t p = exc_pos[lane_listed(f, me.row)];
                    const int v = exc_val[lane_listed(f, me.row)];
                    if (v != 0 && (p & 0x300u) == (q << 8))
                        *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(base + (me.kg << 6) + me.row * 16u + ((p & 0xF0u) << 4) + (p & 14u))) =
                            (uint16_t)(ln_pack((float)v * scale, 0.0f) & 0xFFFFu);
                }
            }
        };

        take_list(c0);
        store(0);
        patch(0);
        codes(c0, CODES);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

        // A stage of products, and the next stage's decode (past the slice's end: the last cell's first stage again, which nobody
        // reads). Requests are never inside a branch: see k_lanes_gemv.
        if (mb0 >= n_mblk) {  // no activations: the decode only
#pragma unroll 1
            for (uint32_t c = c0; c < c1; ++c) {
                const uint32_t c_next = min(c + 1u, c1 - 1u);
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) {
                    if (q == (MI * NI >= 24 ? 2u : 1u)) list = quads(e_now);
                    if (q == 3) take_list(c + 1u);
                    store((q + 1u) & 3u);
                    patch((q + 1u) & 3u);
                    codes(q + 1u + CODES < 4u ? c : c_next, (q + 1u + CODES) & 3u);
                    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                }
            }
            continue;
        }
        ln_f32x4 acc[MI][NI];
#pragma unroll
        for (uint32_t i = 0; i < MI; ++i)
#pragma unroll
            for (uint32_t j = 0; j < NI; ++j) acc[i][j] = ln_f32x4{0, 0, 0, 0};
#pragma unroll 1
        for (uint32_t c = c0; c < c1; ++c) {
            const uint32_t c_next = min(c + 1u, c1 - 1u);
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                constexpr uint32_t PER = 16 / NI;  // pairs of weights decoded with each block's products
                const uint32_t p = (q + 1u) & 3u, base = store_at + (p & 1u) * kLpTile + lane * 16u;
                uint32_t o[16];
                auto piece = [&](uint32_t k) {
                    *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(base + ((k ^ p) << 10))) = ln_u32x4{o[4 * k], o[4 * k + 1], o[4 * k + 2], o[4 * k + 3]};
                };
                auto products = [&](uint32_t j) {
                    const uint32_t t = 4u * q + j;
                    ln_u32x4 v[2];
                    auto weights = [&](uint32_t b) {
                        v[b & 1u] = w_at[(q & 1u) * (kLpTile / 16u) + b * 256u + j * 64u];
                    };
                    weights(0);
#pragma unroll
                    for (uint32_t b = 0; b < NI; ++b) {
                        if (b + 1 < NI) weights(b + 1);
                        if (j == 0) {
                            if (b && b * PER % 4 == 0) piece(b * PER / 4 - 1);
                            uint32_t d[16];
                            ln_decode<BITS, true, FLOAT>(w[p % CODES], lut_lane, scale, d);
#pragma unroll
                            for (uint32_t k = b * PER; k < b * PER + PER; ++k) o[k] = d[k];
                            __builtin_amdgcn_sched_barrier(0);
                        }
#pragma unroll
                        for (uint32_t i = 0; i < MI; ++i)
                            acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_bf16x8, v[b & 1u]),
                                                                                __builtin_bit_cast(ln_bf16x8, a[t % AHEAD][i]), acc[i][b], 0, 0, 0);
                        // (at 512 rows left to the compiler, 98.5 -> 95.4 us; at 384 62.4 -> 63.3)
                        if ((NI == 8 && (MI != 4 || BITS == 8)) || j == 0) __builtin_amdgcn_sched_barrier(0);
                    }
                    if (j == 0) piece(3);
                    x_load(t + AHEAD < 16u ? c : c_next, (t + AHEAD) & 15u);
                    __builtin_amdgcn_sched_barrier(0);
                };
                if (q == (MI * NI >= 24 ? 2u : 1u)) list = quads(e_now);
                if (q == 3) {
                    take_list(c + 1u);
                    __builtin_amdgcn_sched_barrier(0);
                }
                products(0);
                products(1);
                patch(p);
                __builtin_amdgcn_sched_barrier(0);
                // Behind patch() at 257 rows and more, behind the stage's last products to 256: requests come back in order, and what comes
                // from HBM then stands in front of fewer operands that the same stage still waits for (17408 x 5120, 5 bits, 192 rows
                // 72.9 -> 70.5 us; 144 calls of 129 to 256 rows 0.988 in the mean, 3 bits 1.000; longer stages 0.97 to 1.03, mean 1.00).
                if (NW == 1) codes(q + 1u + CODES < 4u ? c : c_next, (q + 1u + CODES) & 3u);
                products(2);
                products(3);
                if (NW == 2) codes(q + 1u + CODES < 4u ? c : c_next, (q + 1u + CODES) & 3u);
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            }
        }

        // ---- the sums: lane (n, kg) of block (i, b) has weight rows 4 kg .. + 3 of activation row n.  A whole tile's go to y ----
        if (c0 == 0 && c1 == n_cells) {
#pragma unroll
            for (uint32_t i = 0; i < MI; ++i)
#pragma unroll
                for (uint32_t b = 0; b < NI; ++b)
                    lp_store(out, (mb0 + i) * 16u + n, tile * kLpRows + (nw * NI + b) * 16u + 4u * kg, acc[i][b]);
            continue;
        }
        const uint32_t part = mg * out.parts + lp_part(blockIdx.x, tile, begins, gridDim.x, lp_tiles(n_tiles));
        ln_f32x4 *const to = ws + ((size_t)part * kLpWaves + wave) * (MI * NI * 64u) + lane;
#pragma unroll
        for (uint32_t i = 0; i < MI; ++i)
#pragma unroll
            for (uint32_t b = 0; b < NI; ++b) to[(i * NI + b) * 64u] = acc[i][b];
    }
}

// y from the sums of a tile's parts, in the columns' order; `per`: workgroups of each tile, where it is a whole number, else 0.  Every wave is
// over after some requests, so what comes before them counts: forms by template and no division where all tiles are alike, 1 % of a call
// in the mean (5120 x 17408, 3 bits, 256 / 512 rows 66.9 / 99.5 -> 65.7 / 98.1 us; two or four runs of 256 sums a workgroup gain less).
template <int MI, int NW>
__global__ void __launch_bounds__(256)
k_lanes_prompt_reduce(const ln_f32x4 *__restrict__ ws, uint32_t groups, uint32_t per, uint32_t tiles, uint32_t n_cells, LpOut out) {
    constexpr uint32_t NI = 8 / NW, MW = 8 / NW, SIZE = kLpWaves * MI * NI * 64u;
    const uint32_t at = blockIdx.x * 256u + threadIdx.x, tile = blockIdx.y, mg = blockIdx.z;
    const uint32_t lane = at & 63u, block = at >> 6, b = block % NI, i = block / NI % MI, wave = block / (NI * MI);
    const uint32_t r = ((mg * MW + wave % MW) * MI + i) * 16u + (lane & 15u), row = tile * kLpRows + ((wave / MW) * NI + b) * 16u + 4u * (lane >> 4);
    uint32_t g0 = tile * per, g1 = g0 + per - 1u, head = g0;
    if (per == 0) {
        const uint32_t u0 = tile * n_cells;
        g0 = lp_group_of(u0, groups, tiles, n_cells), g1 = lp_group_of(u0 + n_cells - 1u, groups, tiles, n_cells);
        head = lp_part(g0, tile, lp_begin(g0, groups, tiles, n_cells) == u0, groups, tiles);
    }
    if (g0 == g1) return;  // its one workgroup wrote y
    if (r >= out.m || row >= out.out_f) return;
    const ln_f32x4 *const from = ws + (size_t)mg * out.parts * SIZE + at;
    ln_f32x4 sum = from[(size_t)head * SIZE];
#pragma unroll 4
    for (uint32_t g = g0 + 1u; g <= g1; ++g) sum += from[(size_t)g * SIZE];
    lp_store(out, r, row, sum);
}

struct LpPlan { uint32_t mi, nw, m_groups, groups, n_mblk; };
static LpPlan lp_plan(const LanesDev &L, int m) {
    LpPlan p{};
    p.n_mblk = ((uint32_t)m + 15u) / 16u;
    p.m_groups = (p.n_mblk + 31u) / 32u;  // of up to 512 rows: 128 sums a lane
    const uint32_t blocks = (p.n_mblk + p.m_groups - 1u) / p.m_groups;
    p.nw = blocks <= 16 ? 2u : 1u;
    p.mi = blocks <= 12 || (blocks > 16 && blocks <= 24) ? 3u : 4u;
    // One workgroup a CU (LDS).  Where a whole number of them to a tile leaves the longest at most about a cell more than an even
    // share, that: no workgroup then starts over in a second tile, which costs about a cell's time (5120 x 17408, 512 rows: 104 us
    // with six workgroups a tile, 114 with all 256 CUs at 5.3 cells each; 17408 x 5120 has 136 tiles: 169 us with one workgroup a
    // tile, 125 shared out evenly).
    const uint32_t cus = std::max(ln_cus() / p.m_groups, 1u), tiles = lp_tiles(L.n_tiles), per_tile = std::min(cus / tiles, L.n_cells);
    const uint32_t longest = per_tile ? (L.n_cells + per_tile - 1u) / per_tile : ~0u, share = (tiles * L.n_cells + cus - 1u) / cus;
    p.groups = share + 1u <= longest ? std::min(cus, tiles * L.n_cells) : per_tile * tiles;
    return p;
}

static size_t lp_x_bytes(const LanesDev &L, const LpPlan &p) { return (size_t)L.n_cells * 16u * p.n_mblk * 1024u; }
static uint32_t lp_part_size(const LpPlan &p) { return kLpWaves * p.mi * (8u / p.nw) * 64u; }  // 16-byte units

// Above 128 rows and 3 * 2^23 weights.  Fewer rows do not hide the decode behind their products, and fewer weights leave a workgroup a
// few cells, which the pipeline's start and the sums' way through memory outweigh.  us, k_lanes_gemm against this: 5120 x 17408
// (3 bits) 50 / 53 at 128 rows, 61 / 52 at 144, 138 / 97 at 512; 5120 x 5120 25 / 28, 27 / 29, 56 / 48; 5120 x 4096 25 / 28 at 144
// rows and 47 / 46 at 512; 4096 x 4096 (5 bits) 26 / 28 at 192 rows, 41 / 44 at 512; 2048 x 2048 23 / 35 at 512; at 129 / 256 / 512 rows:
// 5120 x 5120 (5) 31 / 29, 37 / 35, 60 / 52, 17408 x 5120 (5) 80 / 65, 101 / 83, 196 / 120, 5120 x 5120 (8) 26 / 26,
// 33 / 33, 55 / 51, 12288 x 6144 (8) 52 / 54, 68 / 69, 114 / 104.  (The line is that of a k_lanes_gemm that took 10 to 20 % longer; it is now up to
// 7 % the faster one on this side of it, up to some 192 rows of 2^25 weights and 256 at 8 bits.)  The bounds keep offsets within 32 bits.
bool lanes_prompt_wins(const LanesDev &L, int m) {
    return m > 128 && (uint64_t)L.out_f * L.in_f > 3u << 23 && (uint64_t)lp_tiles(L.n_tiles) * L.n_cells < 1u << 24 &&
           (uint64_t)L.n_cells * 16u * (((uint32_t)m + 15u) / 16u) * 1024u < 1ull << 31;
}

// (15: to the next whole 16 bytes of whatever address is given)
static size_t lp_bytes(const LanesDev &L, const LpPlan &p) {
    return 15u + lp_x_bytes(L, p) + (size_t)p.m_groups * lp_parts(p.groups, lp_tiles(L.n_tiles)) * lp_part_size(p) * 16u;
}
size_t lanes_prompt_workspace_bytes(const LanesDev &L, int m) { return lp_bytes(L, lp_plan(L, m)); }

template <int BITS, int MI, int NW>
static int prompt_launch(const LanesDev &L, const LpPlan &p, const ln_u32x4 *xt, ln_f32x4 *sums, const LpOut &out, hipStream_t s) {
    constexpr size_t lds = LnPairs<BITS, true>::kLutBytes + 2u * kLpTile + 16u * kLpRounds * kLpThreads + kWave * 4u;
    static_assert(lds <= kLnLds, "LDS of a CU");
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_prompt<BITS, MI, NW>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    const dim3 grid(p.groups, p.m_groups);
    hipLaunchKernelGGL((k_lanes_prompt<BITS, MI, NW>), grid, dim3(kLpThreads), lds, s, L.plane, xt, L.exc_off, L.scale, L.n_cells, L.n_tiles,
                       p.n_mblk, L.exc_pos, L.exc_val, sums, out);
    return IXH_OK;
}

template <int BITS>
static int prompt_rows(const LanesDev &L, const LpPlan &p, const ln_u32x4 *xt, ln_f32x4 *sums, const LpOut &out, hipStream_t s) {
    if (p.nw == 1) return p.mi == 3 ? prompt_launch<BITS, 3, 1>(L, p, xt, sums, out, s) : prompt_launch<BITS, 4, 1>(L, p, xt, sums, out, s);
    return p.mi == 3 ? prompt_launch<BITS, 3, 2>(L, p, xt, sums, out, s) : prompt_launch<BITS, 4, 2>(L, p, xt, sums, out, s);
}

int launch_lanes_prompt(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y, int64_t ldy,
                        LnScratch &ws, hipStream_t s) {
    const LpPlan p = lp_plan(L, m);
    if (!ws.holds(lp_bytes(L, p))) return IXH_EWORKSPACE;
    ln_u32x4 *const xt = reinterpret_cast<ln_u32x4 *>(((uintptr_t)ws.at + 15u) & ~(uintptr_t)15u);
    ln_f32x4 *const sums = reinterpret_cast<ln_f32x4 *>(reinterpret_cast<uint8_t *>(xt) + lp_x_bytes(L, p));
    const uint32_t n_kb = L.n_cells * 16u, tiles = lp_tiles(L.n_tiles);
    hipLaunchKernelGGL(k_lanes_xtile, dim3(n_kb / 4u, (p.n_mblk + kLpXBlocks - 1u) / kLpXBlocks), dim3(256), 0, s, x, ldx, (uint32_t)m, L.in_f, n_kb, p.n_mblk, xt);
    const LpOut out{bias, y, ldy, (uint32_t)m, L.out_f, ((uintptr_t)y & 7u) == 0 && ldy % 4 == 0, lp_parts(p.groups, tiles)};
    int rc;
    switch (L.bits) {
        case 3: rc = prompt_rows<3>(L, p, xt, sums, out, s); break;
        case 4: rc = prompt_rows<4>(L, p, xt, sums, out, s); break;
        case 5: rc = prompt_rows<5>(L, p, xt, sums, out, s); break;
        default: rc = prompt_rows<8>(L, p, xt, sums, out, s); break;
    }
    if (rc != IXH_OK) return rc;
    if (out.parts) {
        const auto reduce = p.nw == 1 ? p.mi == 3 ? k_lanes_prompt_reduce<3, 1> : k_lanes_prompt_reduce<4, 1>
                                      : p.mi == 3 ? k_lanes_prompt_reduce<3, 2> : k_lanes_prompt_reduce<4, 2>;
        hipLaunchKernelGGL(reduce, dim3(lp_part_size(p) / 256u, tiles, p.m_groups), dim3(256), 0, s, sums, p.groups,
                           p.groups % tiles == 0 ? p.groups / tiles : 0u, tiles, L.n_cells, out);
    }
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

}  // namespace ixh
