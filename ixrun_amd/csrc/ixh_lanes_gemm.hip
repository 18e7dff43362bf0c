// Products of 5 and more activation rows with weights in the lane layout (ixh_lanes.h).
#include "ixh_lanes_dev.h"

namespace ixh {

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_gemm<BITS, MB, DEPTH>: up to 16 * MB activation rows at a time, MB <= 8; DEPTH activation operands in flight.
//
// Bound: a stage's parts (decode, listed elements, products), which follow one another in a wave while all waves meet at its end; no unit is
// full.  10240 x 5120 at 55 / 40 / 5 %, 100 rows: vector instructions are in issue for 41 % of the time, LDS is busy for 42 (a fifth of
// that with collisions), the matrix unit for 18; waves wait for 56 % of theirs.  34.7 us with the slices' sums (37.7 with two blocks of 16
// weight rows a wave from 49 rows on, which halves the reads of activations, and half as many waves to fill in for one another: 64 rows
// 30.9 -> 27.3, 128 rows 40.6 -> 37.5; 74.3 for the decode to memory and the library's GEMM); without the products and the operands
// read for them 28.4, without the listed elements 30.1, without the decode 33.1, without the activations' copies 32.9.  Looking up the next
// stage's weights between the products of this one changes nothing, nor does the list half a cell earlier; waves of their own for decode
// and products (eight and four, a stage of 64 columns) take 44; activations straight
// from the L2 as operands twice as long.  A wave takes 16 weight rows x 128 columns a stage: it decodes them to its own 4 KB of LDS in
// operand order, stores the listed elements over their places and reads the operands back.  All waves of the workgroup are in the same
// 128 columns, whose activations one copy in LDS serves (in operand order, two stages of it: the next one is fetched during the
// multiply), so a weight is decoded once per 128 activation rows and never reaches memory.  One barrier a stage, which waits for LDS
// only: codes and list are asked for one cell ahead.
//
// A workgroup owns a slice of the columns (whole cells) of a run of 16-row blocks, sixteen at most at a time; the slices' sums
// meet in the workspace and launch_lanes_reduce adds them in slice order.
// ---------------------------------------------------------------------------------------------------------------
// Sixteen copies of the pair table at 4 bits, whose pairs are all looked up and whose 16 KB LDS holds beside 128 activation rows: two / sixteen, us from
// graphs, 10240 x 5120 at 17 / 64 / 100 / 128 rows 21.9 / 27.3 / 34.2 / 36.6 and 20.5 / 25.5 / 32.3 / 34.9, 17408 x 5120 at 80 46.5 / 43.4, 2048 x 2048 at 16 /
// 100 7.5 / 12.1 and 7.4 / 11.5, 320 x 2048 at 20 7.2 / 7.0, 30 such calls 0.957 in the mean and none more than before. At 5 bits, where two of three pairs are worked
// out, four copies gain nothing (10240 x 5120 at 17 / 64 / 100 rows 22.4 / 27.5 / 34.7 and 22.3 / 27.6 / 34.8), and 64 KB are not there.
template <int BITS> constexpr bool kLgWide = BITS == 4;
constexpr uint32_t kLgTile = 4096;
constexpr uint32_t kLgTileBytes = kLgTile + 256u;  // and a dword a lane behind it, for what is not to be stored
// where what the next stage could begin with between the products of this one takes more registers than there are
template <int BITS, int MB> constexpr bool kLgTight = (BITS <= 4 && MB == 6) || (BITS == 5 && MB == 5);

__device__ __forceinline__ void lg_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 5 bits: two of the three whole pairs of a dword by arithmetic, which evens out the LDS and the vector unit.  A code at bit P is, as the
// bits of a float, a multiple of the smallest one: times 2^127 it is code * 2^(P - 22), and that times scale * 2^(22 - P) less 15 scale is
// value * scale, all exact: an AND, a product and a multiply-add, each at the full rate, where a shift left, an AND-OR and a
// multiply-add took 12 clocks instead of 7.  (us, all looked up / one of three by arithmetic / two, 10240 x 5120 at 55 / 40 / 5 %: 17 rows
// 23.9 / 23.1 / 22.4, 32 rows 24.6 / 23.6 / 23.0, 64 rows 29.7 / 28.5 / 27.5, 100 rows 36.1 / 35.1 / 34.7, 128 rows 39.6 / 39.0 / 37.8; 4096 x 4096,
// 100 rows 21.1 / 20.7 / 20.5.)
struct LgScale { float at2, at7, at12, at17, off; };
__device__ __forceinline__ float lg_value(uint32_t field, float by, float off) { return __fmaf_rn(__uint_as_float(field) * 0x1p127f, by, off); }
__device__ __forceinline__ void lg_decode5(const uint32_t (&w)[5], uint32_t lut_lane, const LgScale &k, uint32_t (&o)[16]) {
    using P = LnPairs<5, false>;
    constexpr int TO = P::kCopies + 2;
    uint32_t last = ln_shift_add<TO>(w[0] & 3u, lut_lane);
    last = ln_shift_add<TO + 2>(w[1] & 3u, last), last = ln_shift_add<TO + 4>(w[2] & 3u, last);
    last = ln_shift_add<TO + 6>(w[3] & 3u, last), last = ln_shift_add<TO + 8>(w[4] & 3u, last);
    o[15] = *reinterpret_cast<const LN_LDS(uint32_t) *>((uintptr_t)last);
#pragma unroll
    for (int d = 0; d < 5; ++d) o[3 * d + 2] = *reinterpret_cast<const LN_LDS(uint32_t) *>((uintptr_t)(((w[d] >> (22 - TO)) & P::kMask) + lut_lane));
#pragma unroll
    for (int d = 0; d < 5; ++d) {
        o[3 * d] = ln_pack(lg_value(w[d] & 31u << 2, k.at2, k.off), lg_value(w[d] & 31u << 7, k.at7, k.off));
        o[3 * d + 1] = ln_pack(lg_value(w[d] & 31u << 12, k.at12, k.off), lg_value(w[d] & 31u << 17, k.at17, k.off));
    }
}

template <int BITS, int MB, int DEPTH>
__global__ void __launch_bounds__(kLgBlocks *kWave)
k_lanes_gemm(const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint16_t *__restrict__ scale_at, uint32_t c_share,
             uint32_t c_more, uint32_t b_share, uint32_t b_more, uint32_t in_f, uint32_t ldx, uint32_t m_all, uint32_t most_at_once, uint32_t n_cells, uint32_t n_tiles,
             const uint32_t *__restrict__ exc_off, const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val, uint32_t out_f,
             float *__restrict__ ws, bool ws_aligned, const uint16_t *__restrict__ bias, bool once, uint16_t *__restrict__ y, int64_t ldy) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lg_smem[];
    using P = LnPairs<BITS, kLgWide<BITS>>;
    constexpr uint32_t kTile = kLgTileBytes;
    constexpr uint32_t kThreads = kLgBlocks * kWave;
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)lg_smem;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 15u, kg = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t slice = blockIdx.x, group = blockIdx.y, row0 = blockIdx.z * (16u * MB);
    const uint32_t m_last = m_all - 1u;
    const uint32_t n_blocks = (n_tiles + 3u) / 4u;
    const uint32_t c0 = lg_first(slice, c_share, c_more), c1 = lg_first(slice + 1u, c_share, c_more), len = c1 - c0;
    const uint32_t b0 = lg_first(group, b_share, b_more), b1 = lg_first(group + 1u, b_share, b_more), own = b1 - b0;
    const uint32_t rounds = lg_rounds(own), at_once = lg_at_once(own, most_at_once);
    const uint32_t total = rounds * len;
    const uint32_t tile_at = smem + P::kLutBytes + wave * kTile;
    // (base registers that the compiler takes as they are, the rest in the accesses' offset fields)
    uint32_t tile_lane = tile_at + lane * 16u, x_lane = smem + P::kLutBytes + kLgBlocks * kTile + lane * 16u;
    uint32_t x_to = smem + P::kLutBytes + kLgBlocks * kTile + tid * 16u;
    asm("" : "+v"(tile_lane), "+v"(x_lane), "+v"(x_to));

    // ---- activations of the 128 columns from 128 g on: 16-byte pieces in operand order; of each 256 pieces, 16 rows, a thread has the
    // same columns ----
    constexpr uint32_t XP = (MB * 256u + kThreads - 1u) / (kThreads);
    struct Pieces { ln_u32x4 v[XP]; };
    uint32_t x_row[XP];
#pragma unroll
    for (uint32_t k = 0; k < XP; ++k)  // (the activations lie within 4 GB)
        x_row[k] = min(row0 + ((tid + k * kThreads) >> 8) * 16u + n, m_last) * ldx * 2u;
    const uint32_t x_in = (tid >> 4 & 15u) * 16u, x_bytes = in_f * 2u;
    auto x_load = [&](uint32_t g) {
        Pieces r;
        const uint32_t at = min(g * 256u + x_in, x_bytes - 16u);
#pragma unroll
        for (uint32_t k = 0; k < XP; ++k)
            r.v[k] = *reinterpret_cast<const ln_u32x4 *>(reinterpret_cast<const uint8_t *>(x) + (x_row[k] + at));
        return r;
    };
    auto x_store = [&](Pieces &r, uint32_t g, uint32_t buf) {
        if (g * 256u + 256u > x_bytes) {
            const bool in = g * 256u + x_in < x_bytes;
#pragma unroll
            for (uint32_t k = 0; k < XP; ++k) r.v[k] = in ? r.v[k] : ln_u32x4{0, 0, 0, 0};
        }
#pragma unroll
        for (uint32_t k = 0; k < XP; ++k)
            if (wave * kWave + k * kThreads < MB * 256u)
                *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_to + buf * (MB * 4096u) + k * (kThreads * 16u))) = r.v[k];
    };

    Pieces first = x_load(4u * c0);
    // (5 bits: scales of 2^100 and more are taken as 2^-32 of them, so that their multiples are no infinities.  The rounding is the same: a
    // layout's weights are finite at the scale itself.)
    const float scale_full = bf16_bits_to_f32(*scale_at);
    const bool big = BITS == 5 && fabsf(scale_full) >= 0x1p100f;
    const float scale = big ? scale_full * 0x1p-32f : scale_full;

    if (wave >= at_once) {  // no block: this wave's part of the copies only
        ln_build_lut<BITS, kLgWide<BITS>>(smem, scale, tid, kThreads);
        x_store(first, 4u * c0, 0);
        lg_barrier();
        uint32_t c = c0;
        for (uint32_t u = 0; u < total; ++u) {
            const uint32_t c_next = c + 1u == c1 ? c0 : c + 1u;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t g = q < 3 ? 4u * c + q + 1u : 4u * c_next;
                Pieces r = x_load(g);
                x_store(r, g, (q + 1u) & 1u);
                lg_barrier();
            }
            c = c_next;
        }
        return;
    }

    // Requests are made for blocks past the last too (the last one again), and never inside a branch: the compiler counts
    // what is in flight.
    struct Cell { uint32_t block, c; };
    uint32_t w[2][BITS];  // two quarters of a cell ahead
    // where a lane's codes of a block are in a cell of column 0, in bytes (below 2^31), less a quarter's offset
    constexpr uint32_t kLane = 4u * (BITS < 4 ? BITS : 4u), kCellBytes = 256u * BITS;
    auto row_quad = [&](const Cell &k) {
        return min(4u * (k.block) + (n >> 2), n_tiles - 1u) * n_cells * kCellBytes + (4u * kg + (n & 3u)) * kLane;
    };
    auto codes = [&](const uint32_t from, uint32_t c, uint32_t q) {
        const uint8_t *const cell = reinterpret_cast<const uint8_t *>(plane) + c * kCellBytes;
        uint32_t (&to)[BITS] = w[q & 1u];
        if constexpr (BITS == 3) {
            const ln_u32x3 v = *reinterpret_cast<const ln_u32x3 *>(cell + from + q * 192u);
            to[0] = v[0], to[1] = v[1], to[2] = v[2];
        } else {
            const ln_u32x4 v = *reinterpret_cast<const ln_u32x4 *>(cell + from + q * 256u);
            to[0] = v[0], to[1] = v[1], to[2] = v[2], to[3] = v[3];
            if constexpr (BITS == 5) to[4] = *reinterpret_cast<const uint32_t *>(cell + (from - (4u * kg + (n & 3u)) * 12u) + (1024u + q * 64u));
            if constexpr (BITS == 8) {
                const ln_u32x4 u = *reinterpret_cast<const ln_u32x4 *>(cell + from + (1024u + q * 256u));
                to[4] = u[0], to[5] = u[1], to[6] = u[2], to[7] = u[3];
            }
        }
    };
    // the list of row quad kg of the block in the cell: of its row n % 4 this lane has four of every sixteen quads, three times
    // (at 5 % listed elements the fullest of four rows has 31 in 512 columns, 45 are four standard deviations away)
    constexpr uint32_t ROUNDS = 3;
    struct Extent { uint32_t first, end; };
    auto extent = [&](const Cell &k) {
        const uint32_t t = 4u * (k.block) + kg, cell = min(t, n_tiles - 1u) * n_cells + k.c;
        const uint32_t a = exc_off[cell], b = exc_off[cell + 1u];
        return Extent{a, t < n_tiles ? b : a};
    };
    auto mine = [&](const Extent &e) { return (e.first & ~3u) + (n & ~3u); };
    struct Quads { ln_u32x2 pos[ROUNDS]; uint32_t val[ROUNDS]; };
    auto quads = [&](const Extent &e) {
        Quads l;
#pragma unroll
        for (uint32_t r = 0; r < ROUNDS; ++r) {
            const uint32_t quad = mine(e) + 16u * r, at = quad < e.end ? lane_listed(quad, n & 3u) : 0u;
            l.pos[r] = *reinterpret_cast<const ln_u32x2 *>(reinterpret_cast<const uint8_t *>(exc_pos) + at * 2u);
            l.val[r] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const uint8_t *>(exc_val) + at);
        }
        return l;
    };
    auto after = [&](const Cell &k) { return k.c + 1u < c1 ? Cell{k.block, k.c + 1u} : Cell{k.block + at_once, c0}; };

    const uint32_t in_row = (kg << 6) + (n & 3u) * 16u;
    const bool none_is_0 = lane_none(n_cells) == 0u;
    Cell now{b0 + wave, c0}, next = after(now);
    Extent e_now = extent(now);
    uint32_t from = row_quad(now), from_next = row_quad(next);
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) codes(from, c0, q);
    Quads list = quads(e_now);
    Extent e_next = extent(next);
    ln_build_lut<BITS, kLgWide<BITS>>(smem, scale, tid, kThreads);
    x_store(first, 4u * c0, 0);
    lg_barrier();
    const LgScale scales{scale * 0x1p20f, scale * 0x1p15f, scale * 0x1p10f, scale * 0x1p5f, -15.0f * scale};
    const uint32_t lut_lane = smem + ((lane & ((1u << P::kCopies) - 1u)) << 2);

    ln_f32x4 acc[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[b] = ln_f32x4{0, 0, 0, 0};
    for (uint32_t u = 0; u < total; ++u) {
        // ---- listed elements: value (high half), where it goes in the tile of its quarter (bits 0..11; the tile's block i
        // is at i ^ q, as the list has it), the quarter (bits 12..14; none of the four where there is no element) ----
        // Rounds that no row has elements for are passed over (us, taken / passed over: 3 bits, 0.3 % listed, 5120 x 17408 at 17 rows 28.1 /
        // 26.5; 5 bits, 5 % listed, 10240 x 5120 at 17 / 64 / 100 / 128 rows 22.1 / 27.3 / 35.6 / 39.7 and 22.4 / 27.5 / 34.7 / 37.8).
        uint32_t put[4 * ROUNDS];
        const uint32_t cell_bits = (now.c % kLnSegCells << 10) * 0x10001u;
        // A round's stores in each quarter that any lane has elements of, without branches around them: a lane's elements of other
        // quarters go behind the tile.  (A branch a store / so: 5 bits at 5 % listed, 10240 x 5120 at 17 / 64 / 100 / 128 rows 22.8 / 36.3 /
        // 36.7 / 41.3 and 22.4 / 27.5 / 34.7 / 37.8 us; 3 bits, 5120 x 17408 at 17 rows 29.5 and 26.5.)
        uint32_t in_q[ROUNDS];  // bit q: the lane has elements of quarter q in the round
#pragma unroll
        for (uint32_t r = 0; r < ROUNDS; ++r) {
            in_q[r] = 0;
            if (!__any((e_now.first & ~3u) + 16u * r < e_now.end)) continue;
            const uint32_t quad = mine(e_now) + 16u * r - e_now.first, n_quads = e_now.end - e_now.first, val = list.val[r];
            const uint32_t w01 = ln_pack((float)(int)(int8_t)val * scale, (float)(int)(int8_t)(val >> 8) * scale);
            const uint32_t w23 = ln_pack((float)(int)(int8_t)(val >> 16) * scale, (float)((int)val >> 24) * scale);
            ln_u32x2 pos = list.pos[r] ^ cell_bits;
            // a place without an element has a position of another cell, where rows are short enough for one
            if (none_is_0) {
                asm volatile("");
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) pos[k >> 1] |= (val >> (8 * k) & 255u) ? 0u : 0xFC00u << (16u * (k & 1));
            }
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t two = pos[k >> 1], p = k & 1 ? two >> 16 : two & 0xFFFFu, wk = k & 2 ? w23 : w01;
                uint32_t to = min(ln_shift_add<4>(p & 0xFFF0u, 0u), 0x4000u);
                to = quad + k < n_quads ? to : 0x4000u;
                in_q[r] |= 1u << (to >> 12);
                put[4 * r + k] = to | (p & 14u) | in_row | (k & 1 ? wk & 0xFFFF0000u : wk << 16);
            }
            if constexpr (BITS == 5 && MB == 8) {  // (in a scalar register: there is no other left)
                const uint32_t in = in_q[r];
                in_q[r] = 0;
#pragma unroll
                for (uint32_t q = 0; q < 4; ++q) in_q[r] |= __any(in & (1u << q)) ? 1u << q : 0u;
            }
        }
        const bool more = __any((e_now.first & ~3u) + 16u * ROUNDS < e_now.end);
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t g_next = q < 3 ? 4u * now.c + q + 1u : 4u * next.c;
            Pieces x_next = x_load(g_next);
            uint32_t o[16];
            if constexpr (BITS == 5) lg_decode5(w[q & 1u], lut_lane, scales, o);
            else ln_decode<BITS, kLgWide<BITS>>(w[q & 1u], lut_lane, scale, o);
            codes(q < 2 ? from : from_next, q < 2 ? now.c : next.c, q ^ 2u);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i)
                *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(tile_lane + ((i ^ q) << 10))) =
                    ln_u32x4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
            ln_wave_order();
#pragma unroll
            for (uint32_t r = 0; r < ROUNDS; ++r) {
                if (__any(in_q[r] & (1u << q))) {
#pragma unroll
                    for (uint32_t e = 4 * r; e < 4 * r + 4; ++e)
                        *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(tile_at + min((put[e] ^ (q << 12)) & 0x7FFFu, kLgTile + 4u * lane))) =
                            (uint16_t)(put[e] >> 16);
                }
            }
            if (more) {  // rows with yet more listed elements in the cell
                for (uint32_t f = (e_now.first & ~3u) + 16u * ROUNDS + (n >> 2); f < e_now.end; f += 4u) {
                    const uint32_t p = exc_pos[lane_listed(f, n & 3u)];
                    const int v = exc_val[lane_listed(f, n & 3u)];
                    if (v != 0 && (p & 0x300u) == (q << 8))
                        *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(tile_at + in_row + ((p & 0xF0u) << 4) + (p & 14u))) =
                            (uint16_t)(ln_pack((float)v * scale, 0.0f) & 0xFFFFu);
                }
            }
            if (q == 3) {  // the list of the next cell, over the multiply
                e_now = e_next;
                list = quads(e_now);
                e_next = extent(after(next));
            }
            x_store(x_next, g_next, (q + 1u) & 1u);  // (its other half is in use; no wave is behind the last barrier)
            ln_wave_order();
            const uint32_t x_at = x_lane + (q & 1u) * (MB * 4096u);
            // operands in the order of their products, DEPTH activation operands in flight: a read takes some 130 clocks, a product 16
            // (17 rows of 10240 x 5120 at 5 bits 23.1 -> 22.7 us with six, against all of 16 activation rows and then their products; two
            // from 65 rows on, for which there are registers: three gain up to 1 % where nothing is spilled for them)
            constexpr uint32_t READS = 4u * MB;
            ln_u32x4 a[2], v[DEPTH];
            auto a_read = [&](uint32_t i) { a[i & 1u] = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(tile_lane + ((i ^ q) << 10))); };
            auto x_read = [&](uint32_t k) { v[k % DEPTH] = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + k % MB * 4096u + k / MB * 1024u)); };
            a_read(0);
#pragma unroll
            for (uint32_t k = 0; k + 1u < DEPTH && k < READS; ++k) x_read(k);
#pragma unroll
            for (uint32_t k = 0; k < READS; ++k) {
                if (k + DEPTH - 1u < READS) x_read(k + DEPTH - 1u);
                if (k % MB == 0 && k / MB < 3u) a_read(k / MB + 1u);
                asm volatile("" ::: "memory");
                acc[k % MB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_bf16x8, a[k / MB & 1u]),
                                                                      __builtin_bit_cast(ln_bf16x8, v[k % DEPTH]), acc[k % MB], 0, 0, 0);
            }
            lg_barrier();
            if constexpr (kLgTight<BITS, MB>) __builtin_amdgcn_sched_barrier(0);
        }
        if (now.c + 1u == c1) {  // the slice's sums of the blocks: weight rows 4 kg .. of activation row n of each of the MB blocks
            const bool mine = now.block < b1;
            const uint32_t at = now.block * 16u + 4u * kg;
            uint32_t r = row0 + n;
            asm volatile("" : "+v"(r));  // addresses are worked out here and not kept in registers over the loop
#pragma unroll
            for (int b = 0; b < MB; ++b, r += 16u) {
                if (BITS == 5) acc[b] *= big ? 0x1p32f : 1.0f;
                if (mine && r < m_all) {
                    if (c_share < n_cells) {
                        float *const to = ws + ((size_t)slice * m_all + r) * (n_blocks * 16u) + at;
                        if (ws_aligned) *reinterpret_cast<ln_f32x4 *>(to) = acc[b];
                        else
#pragma unroll
                            for (uint32_t k = 0; k < 4; ++k) to[k] = acc[b][k];
                    } else {
#pragma unroll
                        for (uint32_t k = 0; k < 4; ++k) {
                            if (at + k >= out_f) continue;
                            uint32_t h = f32_to_bf16_bits(acc[b][k]);
                            if (bias) h = f32_to_bf16_bits((once ? acc[b][k] : bf16_bits_to_f32(h)) + bf16_bits_to_f32(bias[at + k]));
                            y[(int64_t)r * ldy + at + k] = (uint16_t)h;
                        }
                    }
                }
                acc[b] = ln_f32x4{0, 0, 0, 0};
            }
        }
        const bool same = next.block == now.block;
        now = next;
        next = after(now);
        from = from_next;
        if (!same || next.block != now.block) from_next = row_quad(next);
    }
}

static LgPlan lg_cut(const LanesDev &L, int m) { return lg_plan(L.n_tiles, L.n_cells, m, ln_cus()); }

static size_t lg_bytes(const LanesDev &L, const LgPlan &p, int m) {
    return p.slices > 1 ? (size_t)p.slices * (uint32_t)m * ((L.n_tiles + 3u) / 4u * 16u) * sizeof(float) : 0;
}

size_t lanes_gemm_workspace_bytes(const LanesDev &L, int m) {
    return lanes_prompt_wins(L, m) ? lanes_prompt_workspace_bytes(L, m) : lg_bytes(L, lg_cut(L, m), m);
}

template <int BITS, int MB, int DEPTH>
static int gemm_launch(const LanesDev &L, const LgPlan &p, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, bool once,
                       uint16_t *y, int64_t ldy, float *ws, hipStream_t s) {
    constexpr size_t lds = LnPairs<BITS, kLgWide<BITS>>::kLutBytes + kLgBlocks * kLgTileBytes + 2u * MB * 4096u;
    static_assert(lds <= kLnLds, "LDS of a CU");
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_gemm<BITS, MB, DEPTH>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    const uint32_t blocks = (L.n_tiles + 3u) / 4u;
    const LgSplit c(L.n_cells, p.slices), b(blocks, p.groups);
    IXH_LAUNCH((k_lanes_gemm<BITS, MB, DEPTH>), dim3(p.slices, p.groups, p.m_groups), dim3(kLgBlocks * kWave), lds, s, L.plane, x, L.scale,
                       c.share, c.more, b.share, b.more, L.in_f, (uint32_t)ldx, (uint32_t)m, lg_most_at_once(blocks, p.groups), L.n_cells,
                       L.n_tiles, L.exc_off, L.exc_pos, L.exc_val, L.out_f, ws, ((uintptr_t)ws & 15u) == 0, bias, once, y, ldy);
    if (p.slices > 1)
        return launch_lanes_reduce(ws, p.slices, m, L.out_f, (L.n_tiles + 3u) / 4u * 16u, bias, once, y, ldy, s);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

bool lanes_gemm_aligned(const LanesDev &L, const uint16_t *x, int m, int64_t ldx) {
    return ((uintptr_t)x & 15u) == 0 && L.in_f % 8u == 0 && (m == 1 || (ldx % 8 == 0 && ldx < (1ll << 31) / m));
}

template <int BITS, class... A>
static int gemm_rows(const LanesDev &L, const LgPlan &p, A... a) {
    switch (p.mb) {
        case 1: return gemm_launch<BITS, 1, 6>(L, p, a...);
        case 2: return gemm_launch<BITS, 2, 6>(L, p, a...);
        case 3: return gemm_launch<BITS, 3, 6>(L, p, a...);
        case 4: return gemm_launch<BITS, 4, 6>(L, p, a...);
        case 5: return gemm_launch<BITS, 5, 2>(L, p, a...);
        case 6: return gemm_launch<BITS, 6, 2>(L, p, a...);
        case 7: return gemm_launch<BITS, 7, 2>(L, p, a...);
        default: return gemm_launch<BITS, 8, 2>(L, p, a...);
    }
}

int launch_lanes_gemm(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, bool once, uint16_t *y,
                      int64_t ldy, LnScratch &ws, hipStream_t s) {
    if (!lanes_gemm_aligned(L, x, m, ldx)) return IXH_EUNSUPPORTED;
    if (lanes_prompt_wins(L, m)) return launch_lanes_prompt(L, x, m, ldx, bias, y, ldy, ws, s);
    const LgPlan p = lg_cut(L, m);
    if (!ws.holds(lg_bytes(L, p, m))) return IXH_EWORKSPACE;
    if (m == 1) ldx = L.in_f;
    switch (L.bits) {
        case 3: return gemm_rows<3>(L, p, x, m, ldx, bias, once, y, ldy, ws.at, s);
        case 4: return gemm_rows<4>(L, p, x, m, ldx, bias, once, y, ldy, ws.at, s);
        case 5: return gemm_rows<5>(L, p, x, m, ldx, bias, once, y, ldy, ws.at, s);
        default: return gemm_rows<8>(L, p, x, m, ldx, bias, once, y, ldy, ws.at, s);
    }
}

}  // namespace ixh
