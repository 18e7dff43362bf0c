// Products of 5 to 16 activation rows with weights in the lane layout (ixh_lanes.h).
#include <algorithm>

#include "ixh_lanes_dev.h"

namespace ixh {

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_rows<BITS, MT, WIDE>: up to MT activation rows, MT = 8 or 16.
//
// Bound: a launch's start-up (some 5 us to the first product: the activations of a slice are turned round on the way to LDS),
// then the decode's LDS look-ups and vector instructions; the busiest unit is busy for some 60 % of the rest. us a layer:
// 17408 x 5120 at 55 / 40 / 5 %, 8 rows 32.6 -> 19.1, 5120 x 17408 at 3 bits, 16 rows 25.1 -> 17.9, 1536 x 2048, 8 rows
// 9.7 -> 6.8, against k_lanes_gemm, which decodes to LDS, stores the listed elements over their places, reads the operands
// back and meets at a barrier every 128 columns.
//
// Here a lane's decoded weights are its operand of v_mfma_f32_16x16x32_bf16 as they are: lane (n, kg) takes the codes of row n
// of a block of 16 (four row quads) in the columns 32 i + 8 kg .. + 7, which one lane of the layout holds.  The activations of
// a slice of the columns stay in LDS for the whole launch, so nothing waits at a barrier in between, and they are there once,
// a column's rows together: ds_read_b64_tr_b16 turns four columns of sixteen lanes into the other operand, and a listed element's
// activations are one read of 16 or 32 bytes at its position.  Listed elements are multiplied in fp32 (as in k_lanes_gemv: weight
// less the plane's sign times the scale) by the lane of their row, 16 quads of each of four row quads at a time, between the
// steps of the plane.
//
// A workgroup owns a slice of the columns (whole cells, as many as LDS holds) of a run of blocks; its steps, 16 rows x 256
// columns, block after block, are dealt to its waves in contiguous shares.  What a wave has of a block goes to LDS, and the
// parts are added in wave order.  Slices (rows longer than LDS holds) meet in the workspace.
// One step in flight and a loop of one step: the loop twice as long with two in flight took 3 to 6 % more.
// ---------------------------------------------------------------------------------------------------------------
// rows' pairs of columns a lane has in registers on the way to LDS: as many as 512 columns x 16 or 768 x 8 take of 16 waves
template <int MT> constexpr uint32_t kLrXAhead = MT == 8 ? 3 : 2;

typedef __bf16 lr_bf16x4 __attribute__((ext_vector_type(4)));

// Where a column's activations are in LDS: rows of MT bf16, the columns of a cell in the order of the list's positions
// (lane_offset), so that a position times MT is a byte offset. At 16 rows the halves of a row of 32 bytes and of a run of eight
// rows change places with the column, so that both a random column's half and the sixteen pieces that a transposing read
// takes from four groups of eight columns lie on all banks.
template <int MT> __device__ __forceinline__ uint32_t lr_place(uint32_t bytes) {
    return MT == 16 ? bytes ^ ((bytes >> 1) & 0x90u) : bytes;
}

// A transposing read: sixteen lanes name sixteen pieces of 8 bytes, four columns of a place each, and lane n of them gets
// activation row n of the four columns.
__device__ __forceinline__ lr_bf16x4 lr_turned(uint32_t at) {
    return __builtin_bit_cast(lr_bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((LN_LDS(ln_s16x4) *)(uintptr_t)at));
}

// (the order of a cell's columns is worked out on the address bits of 128 rows)
template <int BITS, bool WIDE> constexpr uint32_t kLrXAt = (LnPairs<BITS, WIDE>::kLutBytes + 4095u) & ~4095u;

template <int BITS, int MT, bool WIDE>
__global__ void __launch_bounds__(1024)
k_lanes_rows(const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint32_t *__restrict__ exc_off,
             const uint16_t *__restrict__ scale_at, uint32_t n_cells, uint32_t n_tiles, uint32_t in_f, uint32_t shape,
             uint32_t cells_split, uint32_t blocks_split, const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val,
             int64_t ldx, uint32_t out_f, uint32_t x_rows, float *__restrict__ ws, const uint16_t *__restrict__ bias,
             uint16_t *__restrict__ y, int64_t ldy) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lr_smem[];
    using P = LnPairs<BITS, WIDE>;
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)lr_smem;
    const uint32_t m = shape & 31u, log_waves = (shape >> 5) & 7u;
    const bool x_pairs = (shape >> 8) & 1u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 15u, kg = lane >> 4;
    const uint32_t n_waves = 1u << log_waves, n_threads = kWave << log_waves;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    // slices of the columns in whole cells, groups of blocks of 16 rows: the first ones have one more than the others
    const uint32_t slice = blockIdx.x, group = blockIdx.y, c_share = cells_split >> 20, c_more = cells_split & 0xFFFFFu;
    const uint32_t C = c_share + (slice < c_more), c0 = slice * c_share + min(slice, c_more);
    const uint32_t b_share = blocks_split >> 24, b_more = blocks_split & 0xFFFFFFu;
    const uint32_t n_blocks = b_share + (group < b_more), t0 = 4u * (group * b_share + min(group, b_more));
    const uint32_t t1 = min(t0 + 4u * n_blocks, n_tiles);
    // a step: 16 rows x 256 columns, half a cell of four row quads
    const uint32_t H = 2u * C, total = n_blocks * H;
    const uint32_t s0 = (wave * total) >> log_waves, n_steps = (((wave + 1u) * total) >> log_waves) - s0;
    constexpr uint32_t ROW = 2u * MT;
    const uint32_t x_at = smem + kLrXAt<BITS, WIDE>;
    float *const parts = reinterpret_cast<float *>(lr_smem + kLrXAt<BITS, WIDE> + x_rows * ROW);  // [wave + block][16][MT]

    const uint32_t scale_raw = *scale_at;
    // ---- asked for first: this wave's activations, its first units, the list's extent, the scale ----
    // a pair of columns a lane, all rows; pairs past the last column are those of the last
    struct Pairs { uint32_t v[MT]; };
    // Rows' places in 32 bits (where pairs are asked for, they lie within 4 GB): with the rows' addresses in 64 a wave's first request was
    // behind 240 instructions at 16 rows, 105 now (5120 x 17408, 3 bits, 16 rows 20.3 -> 19.8 us; 1024 x 1024, 5 bits 6.6 -> 6.3, eight rows 5.6 -> 5.5).
    const uint32_t x_step = (uint32_t)ldx * 2u, x_last = (m - 1u) * x_step;
    auto x_load = [&](uint32_t task) {
        Pairs r;
        const uint32_t col = c0 * kLnCols + task * 128u + 2u * lane;
        if (x_pairs) {
            const uint32_t at = min(col, in_f - 2u) * 2u;
#pragma unroll
            for (uint32_t k = 0; k < MT; ++k)
                r.v[k] = *reinterpret_cast<const uint32_t *>(reinterpret_cast<const uint8_t *>(x) + (min(k * x_step, x_last) + at));
        } else {
            const uint32_t at = min(col, in_f - 1u), next = min(col + 1u, in_f - 1u);
            uint32_t hi[MT];
            int64_t step = ldx;
            asm volatile("" : "+s"(step));  // (rows' addresses are worked out here, not in front of the other way's requests)
#pragma unroll
            for (uint32_t k = 0; k < MT; ++k) {
                const uint16_t *const row = x + (int64_t)min(k, m - 1u) * step;
                r.v[k] = row[at], hi[k] = row[next];
            }
#pragma unroll
            for (uint32_t k = 0; k < MT; ++k) r.v[k] |= hi[k] << 16;
        }
        return r;
    };
    auto x_store = [&](const Pairs &in, uint32_t task) {
        const uint32_t col = c0 * kLnCols + task * 128u + 2u * lane;
        const uint32_t keep = (col < in_f ? 0xFFFFu : 0u) | (col + 1u < in_f ? 0xFFFF0000u : 0u);
        const uint32_t to = lane_offset(task * 128u + 2u * lane) * MT;
        uint32_t v[MT];
#pragma unroll
        for (uint32_t k = 0; k < MT; ++k) v[k] = k < m ? in.v[k] & keep : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
            for (uint32_t h = 0; h < MT / 8u; ++h) {
                ln_u32x4 o;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    o[k] = __builtin_amdgcn_perm(v[8 * h + 2 * k + 1], v[8 * h + 2 * k], j ? 0x07060302u : 0x05040100u);
                *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + (lr_place<MT>(to + j * ROW) ^ (h * 16u)))) = o;
            }
    };
    Pairs xv[kLrXAhead<MT>];
#pragma unroll
    for (uint32_t k = 0; k < kLrXAhead<MT>; ++k) {
        if (wave + k * n_waves >= 2u * H) break;
        xv[k] = x_load(wave + k * n_waves);
    }
    __builtin_amdgcn_sched_barrier(0);

    // the steps' cursors: `ahead` is two steps in front; past the wave's share it stays at its last step
    struct Cursor { uint32_t block, at; };
    const uint32_t first_block = min(s0 / H, n_blocks - 1u);  // (an empty share at the end)
    Cursor now{first_block, min(s0 - first_block * H, H - 1u)}, ahead = now;
    uint32_t w[2][BITS];
    auto load = [&](uint32_t (&to)[2][BITS]) {
        const uint32_t t = min(t0 + 4u * ahead.block + (n >> 2), n_tiles - 1u);
        const uint8_t *const cell = reinterpret_cast<const uint8_t *>(plane) + (t * n_cells + c0 + (ahead.at >> 1)) * (256u * BITS);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j)
            ln_load_lane<BITS>(reinterpret_cast<const uint32_t *>(cell), 32u * (ahead.at & 1u) + 16u * j + 4u * kg + (n & 3u), to[j]);
    };
    auto go_on = [&](bool more) {
        ahead.at += more;
        if (ahead.at == H) ahead = Cursor{ahead.block + 1u, 0u};
    };
    load(w);
    go_on(1u < n_steps);
    // The list of row quad kg of a run of steps (of one block): whole cells, and of a cell that the run has half of half the
    // list; which half does not matter.
    struct Extent { uint32_t a0, a1, b0, b1, qa, qb; };  // as asked for
    auto extent = [&](uint32_t block, uint32_t from, uint32_t to) {
        const uint32_t t = min(t0 + 4u * block + kg, n_tiles - 1u);
        const uint32_t *const p = exc_off + (t * n_cells + c0);
        Extent e;
        e.qa = from & 1u, e.qb = to & 1u;
        e.a0 = p[from >> 1], e.a1 = p[(from >> 1) + e.qa], e.b0 = p[to >> 1], e.b1 = p[(to >> 1) + e.qb];
        return e;
    };
    struct Range { uint32_t first, end; };
    auto range = [&](const Extent &e, uint32_t block) {
        Range r{e.a0 + (e.qa ? (e.a1 - e.a0) / 2u : 0u), e.b0 + (e.qb ? (e.b1 - e.b0) / 2u : 0u)};
        if (t0 + 4u * block + kg >= t1) r.end = r.first;
        return r;
    };
    uint32_t run_end = min(n_steps, H - now.at);  // steps after s0
    const Extent e_first = extent(now.block, now.at, now.at + run_end);
    auto run_after = [&] {  // the run that follows the one that ends at run_end, empty if there is none
        const uint32_t left = n_steps - run_end;
        return extent(left ? now.block + 1u : now.block, 0u, min(left, H));
    };
    Extent e_next = run_after();
    const float scale = bf16_bits_to_f32(scale_raw);
    __builtin_amdgcn_sched_barrier(0);

    ln_build_lut<BITS, WIDE>(smem, scale, tid, n_threads);
    // the column that places without an element point at, and what shares its run of eight rows
    if (tid < 16u) *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + H * 256u * ROW + tid * 16u)) = ln_u32x4{0, 0, 0, 0};
    auto groups_of = [&](const Range &r) {  // of the row quad that has most
        const int mine = (int)(r.end > r.first ? (r.end - (r.first & ~3u) + 15u) / 16u : 0u);
        return (uint32_t)max(max(__builtin_amdgcn_readlane(mine, 0), __builtin_amdgcn_readlane(mine, 16)),
                             max(__builtin_amdgcn_readlane(mine, 32), __builtin_amdgcn_readlane(mine, 48)));
    };
    struct Group { ln_u32x2 pos; uint32_t val; } list[2];
    Range r_now = range(e_first, now.block);
    auto quad_of = [&](const Range &r, uint32_t i) { return (r.first & ~3u) + 16u * i + (n & ~3u); };
    auto g_load = [&](const Range &r, uint32_t i) {
        const uint32_t quad = quad_of(r, i), at = quad < r.end ? lane_listed(quad, n & 3u) : 0u;
        return Group{*reinterpret_cast<const ln_u32x2 *>(exc_pos + at), *reinterpret_cast<const uint32_t *>(exc_val + at)};
    };
#pragma unroll
    for (uint32_t k = 0; k < kLrXAhead<MT>; ++k)
        if (wave + k * n_waves < 2u * H) x_store(xv[k], wave + k * n_waves);
    for (uint32_t task = wave + kLrXAhead<MT> * n_waves; task < 2u * H; task += n_waves) x_store(x_load(task), task);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t p = 0; p < 2; ++p) list[p] = g_load(r_now, p);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const uint32_t lut_lane = smem + ((lane & ((1u << P::kCopies) - 1u)) << 2);
    const uint32_t piece = MT == 16 ? n & 3u : n & 1u;
    const uint32_t x_mine = (x_at + lr_place<MT>((8u * kg + (n >> 2)) * ROW)) ^ (piece * 8u);
    const uint32_t c_seg = c0 * 1024u, x_none = H * 256u * ROW, scale_bits = __float_as_uint(scale) & 0x7FFFFFFFu;

    ln_f32x4 acc[2] = {};
    float ex[MT];
#pragma unroll
    for (int r = 0; r < MT; ++r) ex[r] = 0.0f;

    auto listed = [&](const Group &g, const Range &r, uint32_t i) {
        const uint32_t quad = quad_of(r, i);
        uint32_t at[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t p = ((g.pos[k >> 1] >> (16 * (k & 1))) - c_seg) & 0xFFFFu;
            at[k] = min(p * MT, x_none);
        }
        if (n_cells >= kLnSegCells)
#pragma unroll
            for (int k = 0; k < 4; ++k) at[k] = (g.val >> (8 * k)) & 255u ? at[k] : x_none;
        if (__any(quad < r.first || quad + 3u >= r.end))
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) at[k] = quad + k >= r.first && quad + k < r.end ? at[k] : x_none;
        const uint32_t w01 = ln_pack((float)(int)(int8_t)g.val * scale, (float)(int)(int8_t)(g.val >> 8) * scale);
        const uint32_t w23 = ln_pack((float)(int)(int8_t)(g.val >> 16) * scale, (float)((int)g.val >> 24) * scale);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t wk = k & 2 ? w23 : w01, wb = k & 1 ? wk & 0xFFFF0000u : wk << 16;
            const float wv = __uint_as_float(wb) - __uint_as_float((wb & 0x80000000u) | scale_bits);  // (no element: times 0)
#pragma unroll
            for (uint32_t h = 0; h < MT / 8u; ++h) {
                const ln_u32x4 v = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + (lr_place<MT>(at[k]) ^ (h * 16u))));
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    ex[8 * h + 2 * j] = __fmaf_rn(wv, __uint_as_float(v[j] << 16), ex[8 * h + 2 * j]);
                    ex[8 * h + 2 * j + 1] = __fmaf_rn(wv, __uint_as_float(v[j] & 0xFFFF0000u), ex[8 * h + 2 * j + 1]);
                }
            }
        }
    };

    uint32_t run_at = 0, l = 0, l_all = groups_of(r_now);  // where the run began, its groups taken and in all
#pragma unroll 1
    for (uint32_t s = 0; s < n_steps;) {
        // (a wave that has more to do takes precedence: see k_lanes_gemv)
        const uint32_t behind = (n_steps - s) * 4u / (n_steps + 1u);
        if (behind >= 3u) __builtin_amdgcn_s_setprio(3);
        else if (behind == 2u) __builtin_amdgcn_s_setprio(2);
        else if (behind == 1u) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
        uint32_t o[2][16];
        ln_decode<BITS, WIDE>(w[0], lut_lane, scale, o[0]);
        ln_decode<BITS, WIDE>(w[1], lut_lane, scale, o[1]);
        load(w);
        go_on(s + 2u < n_steps);
        // (columns 128 q + 32 i of a cell lie at 128 q + 32 (i ^ q))
        const uint32_t x_s = x_mine + now.at * (256u * ROW), q = 2u * (now.at & 1u);
#pragma unroll
        for (uint32_t j = 0; j < 2; ++j)
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t a = (x_s + j * (128u * ROW)) ^ (((q + j) ^ i) * (32u * ROW));
                const lr_bf16x4 lo = lr_turned(a), hi = lr_turned(MT == 16 ? a ^ (4u * ROW) : a + 4u * ROW);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(ln_bf16x8, ln_u32x4{o[j][4 * i], o[j][4 * i + 1], o[j][4 * i + 2], o[j][4 * i + 3]}),
                    __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), acc[j], 0, 0, 0);
            }
        ++now.at;
        ++s;
        // as large a part of the run's list as of its steps
#pragma unroll 1
        while (l * (run_end - run_at) < l_all * (s - run_at)) {
            listed(list[0], r_now, l);
            list[0] = list[1];
            list[1] = g_load(r_now, l + 2u);
            ++l;
        }
        if (s < run_end) continue;

        // the run's sums: of listed elements over the four lanes of a row, of the plane as they are
        float *const part = parts + (wave + now.block) * (16u * MT);
#pragma unroll
        for (int r = 0; r < MT; ++r) {
            ex[r] += ln_dpp<0x124>(ex[r]);
            ex[r] += ln_dpp<0x128>(ex[r]);
        }
        if (n < 4u)
#pragma unroll
            for (uint32_t r = 0; r < MT; r += 4)
                *reinterpret_cast<ln_f32x4 *>(part + (4u * kg + n) * MT + r) = ln_f32x4{ex[r], ex[r + 1], ex[r + 2], ex[r + 3]};
        ln_wave_order();
        if (n < MT)
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) part[(4u * kg + k) * MT + n] += acc[0][k] + acc[1][k];
        acc[0] = acc[1] = ln_f32x4{0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < MT; ++r) ex[r] = 0.0f;
        ++now.block;
        now.at = 0;
        if (run_end < n_steps) {
            run_at = run_end;
            r_now = range(e_next, now.block);
            l = 0, l_all = groups_of(r_now);
            run_end += min(n_steps - run_end, H);
            e_next = run_after();
#pragma unroll
            for (uint32_t k = 0; k < 2; ++k) list[k] = g_load(r_now, k);
        }
    }
    __syncthreads();

    // ---- the waves' parts of every block, in wave order; part `wave + block` is of the wave's steps of the block ----
    for (uint32_t block = wave; block < n_blocks; block += n_waves) {
        const uint32_t wa = ((block * H + 1u) * n_waves - 1u) / total, wb = ((block + 1u) * H * n_waves - 1u) / total;
        const uint32_t at = 4u * t0 + 16u * block + n;
        const float *const part = parts + block * (16u * MT) + n * MT + kg;
        float sum[MT / 4] = {};
        for (uint32_t k = wa; k <= wb; ++k)  // (waves without a step left no part)
            if ((k * total) >> log_waves != ((k + 1u) * total) >> log_waves)
#pragma unroll
                for (uint32_t j = 0; j < MT / 4; ++j) sum[j] += part[k * (16u * MT) + 4u * j];
        const float plus = bias && at < out_f ? bf16_bits_to_f32(bias[at]) : 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < MT / 4; ++j) {
            const uint32_t r = kg + 4u * j;
            if (r >= m) continue;
            if (gridDim.x > 1u) {
                if (at < 4u * n_tiles) ws[((size_t)slice * m + r) * (n_tiles * 4u) + at] = sum[j];
            } else if (at < out_f) {
                uint32_t h = f32_to_bf16_bits(sum[j]);
                if (bias) h = f32_to_bf16_bits(bf16_bits_to_f32(h) + plus);
                y[(int64_t)r * ldy + at] = (uint16_t)h;
            }
        }
    }
}

// How the work is cut: slices of the columns, workgroups of a slice, waves of a workgroup. Of a few cuts the one with the shortest
// estimate, in clocks: 4000 to the first product and 510 for each wave that has to be there, 22 or 29 (up to 8 or 16 rows) for 128
// columns of activations a wave turns round, 28 or 56 for each cell of them that an XCD fetches, then whichever is longer, 2700 for a step of
// 16 x 256 weights in a wave or 135 in the CU, and 16 for each block and cell where the longer slices are always the same XCDs'; the slices'
// sums cost a launch and their way through memory.  Fitted to all cuts, timed, of 54 shapes from 512 x 512 to 17408 x 5120 and 20480 x 4096
// at 8 and 16 rows and 3, 5 and 8 bits: within 1.0 % of the shortest in the mean, 9 % at worst (1.9 and 15 with 400 for a wave and without
// the XCDs' terms: eight rows of 2048 x 11008, 5 bits, in eleven slices instead of eight 12.6 us against 11.3, 2048 x 6144 by sixteen waves
// instead of eight 11.0 against 10.5; where this one errs: 1760 x 12320, 5 bits, at 16 rows 15.4 us against 14.3 by that, 5024 x 9472, 3 bits, at
// eight 13.2 against 12.4, 2880 x 13728, 8 bits, at eight 15.1 against 14.6).  (Without a cost of each wave, and the slices dearer, layers of few rows had one slice of sixteen waves
// where several of four fill the CUs: 960 x 3072 at 11 rows 11.0 us against 8.9, 256 x 4096 11.9 against 8.7.)
struct LrPlan { uint32_t slices, groups, waves, x_rows; size_t lds; };

template <int BITS, int MT, bool WIDE>
static LrPlan lr_plan(const LanesDev &L) {
    LrPlan best{};
    uint64_t best_cost = ~0ull;
    const uint32_t cus = ln_cus(), blocks = (L.n_tiles + 3u) / 4u;
    constexpr size_t kPart = 64u * MT;  // bytes of a wave's part of a block
    const uint32_t most = (uint32_t)((kLnLds - kLrXAt<BITS, WIDE> - 24u * kPart) / (kLnCols * 2u * MT));  // cells of a slice
    const uint32_t s_min = (L.n_cells + most - 1u) / most;
    for (uint32_t s = s_min; s <= min(L.n_cells, s_min + 15u); ++s) {
        // (16 rows more: the zeros that places without an element point at)
        const uint32_t cells = (L.n_cells + s - 1u) / s, x_rows = cells * kLnCols + 16u;
        // workgroups go round the eight XCDs: slices that one of them has; the longer ones are always the same one's
        const uint32_t xcd_slices = s / min(s & (0u - s), 8u);
        const bool uneven = xcd_slices == 1u && L.n_cells % s != 0u;
        for (uint32_t waves = 16; waves >= 4; waves /= 2) {
            const size_t fixed = kLrXAt<BITS, WIDE> + (size_t)x_rows * 2u * MT + waves * kPart;
            if (fixed + kPart > kLnLds) continue;
            // as many workgroups as CUs, or as it takes for the parts of a workgroup's blocks to fit
            const uint32_t fit = min((uint32_t)((kLnLds - fixed) / kPart), 255u);
            const uint32_t groups = max(min(max(cus / s, 1u), blocks), (blocks + fit - 1u) / fit);
            const uint32_t nb = (blocks + groups - 1u) / groups;
            if (waves > 4u && waves > 2u * (L.n_cells / s) * (blocks / groups)) continue;  // a step for every wave
            const size_t lds = fixed + nb * kPart;
            const uint32_t per_cu = min((uint32_t)(kLnLds / lds), 16u / waves), rounds = (groups * s + cus * per_cu - 1u) / (cus * per_cu);
            const uint32_t steps = nb * cells * 2u, mine = (steps + waves - 1u) / waves;
            const uint32_t resident = min(per_cu, (groups * s + cus - 1u) / cus);
            const uint64_t run = std::max<uint64_t>((uint64_t)mine * 2700u, (uint64_t)steps * resident * 135u);
            const uint64_t sums = s > 1 ? (MT == 8 ? 4800u : 3300u) + (uint64_t)s * L.n_tiles * 4u * MT * 8u / 3300u : 0u;
            const uint64_t turned = (uint64_t)cells * 64u / waves * (MT == 8 ? 22u : 29u) + (uint64_t)cells * xcd_slices * (MT == 8 ? 28u : 56u);
            const uint64_t cost = rounds * (4000u + 510u * waves + turned + run + (uneven ? 16u * cells * nb : 0u)) + sums;
            if (cost < best_cost) { best_cost = cost; best = {s, groups, waves, x_rows, lds}; }
        }
    }
    return best;
}

// The larger pair table up to eight rows (LDS has the room beside their activations) and from some cells a CU on: below, what it
// saves is less than its 64 KB take to write (5 bits, 8 rows, larger / smaller: 512 x 512 5.9 / 5.2 us, 2000 x 2048 with 8 cells a CU
// 6.9 / 6.6, 4000 x 3072 with 24 8.9 / 8.6, 2000 x 8192 with 32 11.1 / 11.8, 5000 x 5120 with 50 12.7 / 12.8).  At 4 bits,
// where it is 16 KB, up to sixteen rows (smaller / larger at 16, 1.5 % of the weights listed: 17408 x 5120 22.6 / 20.4, 5120 x 17408 22.6 / 19.8,
// 10240 x 5120 17.1 / 15.9, 5120 x 5120 with 50 cells a CU 13.9 / 13.1; 5 % listed 26.5 / 24.7, 26.7 / 24.1, 20.0 / 18.9, 15.5 / 14.8; 4096 x 4096 with
// 32 10.6 / 10.6, 8192 x 1024 with 16 7.3 / 7.3, 1024 x 1024 6.7 / 6.8.  lr_plan's costs were fitted without this form.)
template <int BITS> static bool lr_wide(const LanesDev &L, int m) {
    const uint64_t cells = (uint64_t)L.n_tiles * L.n_cells;
    return m <= 8 ? (BITS == 4 || BITS == 5) && cells > 24u * ln_cus() : BITS == 4 && cells > 32u * ln_cus();
}

template <int BITS> static LrPlan lr_plan_rows(const LanesDev &L, int m) {
    if (lr_wide<BITS>(L, m)) return m <= 8 ? lr_plan<BITS, 8, true>(L) : lr_plan<BITS, 16, true>(L);
    return m <= 8 ? lr_plan<BITS, 8, false>(L) : lr_plan<BITS, 16, false>(L);
}
static LrPlan lr_plan_of(const LanesDev &L, int m) {
    switch (L.bits) {
        case 3: return lr_plan_rows<3>(L, m);
        case 4: return lr_plan_rows<4>(L, m);
        case 5: return lr_plan_rows<5>(L, m);
        default: return lr_plan_rows<8>(L, m);
    }
}

// Nine to sixteen rows: turning the activations round for the whole of a long slice, or starting up for a single cell, takes longer than
// k_lanes_gemm's way, whose sixteen waves share a copy of 128 columns a stage, up to 20 * 2^20 weights, and of long rows from 25 * 2^20 to
// 46 at 5 bits and 38 at 8; not of tall layers, of which a workgroup here has one slice.  us, this / that at 16 rows (nine and twelve
// are within 4 % of that where nothing else is said):
//   5 bits   1024 x 1024 7.2 / 7.6, 2048 x 2048 8.8 / 8.7, 2560 x 2560 10.6 / 9.2, 2048 x 4096 10.4 / 9.7, 4096 x 2048 9.1 / 9.8, 1536 x 6144
//            12.6 / 10.2, 4096 x 4096 12.0 / 11.6, 4096 x 5120 13.9 / 12.9, 3072 x 8192 15.5 / 14.0, 4096 x 6144 14.2 / 14.8, 5120 x 5120 15.8 /
//            15.0, 4096 x 8192 15.9 / 16.0, 6144 x 6144 18.4 / 17.8, 6656 x 6656 20.9 / 19.0, 9216 x 5120 21.1 / 19.1, 4096 x 12288 20.1 / 20.8
//   8 bits   2048 x 2048 7.1 / 7.4, 2048 x 4096 9.0 / 8.3, 1536 x 6144 10.4 / 8.8, 4096 x 4096 9.7 / 10.0, 4096 x 5120 11.1 / 10.8, 4096 x 6144
//            11.7 / 11.9, 5120 x 5120 13.3 / 12.4, 2880 x 9536 13.4 / 13.1, 4096 x 8192 14.5 / 14.3, 6144 x 6144 15.5 / 15.6, 8192 x 5120 16.1 /
//            16.5, 6656 x 6656 18.4 / 16.5, 4096 x 11008 16.7 / 17.3, 2560 x 17408 16.2 / 17.2
//   4 bits   (1.5 % listed) 2048 x 2048 7.8 / 7.3, 2560 x 2560 9.2 / 8.0, 1536 x 6144 10.7 / 8.6, 4096 x 4096 10.4 / 9.4, 4096 x 5120 11.3 / 11.2,
//            3072 x 8192 12.4 / 11.8, 4096 x 6144 11.4 / 12.4, 5120 x 5120 12.7 / 12.6, 6144 x 6144 13.4 / 14.4, 4096 x 11008 14.3 / 16.1, 10240 x
//            5120 15.2 / 17.4; with 5 % listed 9 to 18 % more either way, the same side ahead; at nine rows 5120 x 5120 12.7 / 11.5, 3072 x 8192 12.2 /
//            10.8.  (Between 20 and 25 * 2^20 that way would be ahead where rows are long.)
//   3 bits   (whose pairs sit in LDS 32 times over here) 2048 x 2048 7.6 / 7.5, 2560 x 2560 8.5 / 8.4, 2048 x 4096 9.1 / 8.4, 4096 x 2048 7.7 / 8.5,
//            1536 x 6144 10.5 / 9.1, 2048 x 8192 10.1 / 9.9, 4096 x 4096 9.8 / 9.9, 4096 x 5120 10.9 / 11.3, 4096 x 6144 11.2 / 12.7
static bool lr_gemm_wins(const LanesDev &L, int m) {
    const uint64_t n = (uint64_t)L.out_f * L.in_f;
    if (m <= 8) return false;
    if (L.bits != 3 && L.in_f <= kLnCols) return n <= 20u << 20;
    if (L.out_f >= 2ull * L.in_f) return false;
    if (L.bits == 3) return L.in_f >= 2560u && n > 4u << 20 && n <= 20u << 20;
    if (n <= 20u << 20) return L.in_f >= 2048u;
    return L.bits != 4 && L.in_f >= 4608u && n >= 25u << 20 && n <= (L.bits == 5 ? 46u : 38u) << 20;
}

static size_t lr_bytes(const LanesDev &L, const LrPlan &p, int m) {
    return p.slices > 1 ? (size_t)p.slices * (uint32_t)m * L.n_tiles * 4u * sizeof(float) : 0;
}

size_t lanes_rows_workspace_bytes(const LanesDev &L, int m) { return lr_bytes(L, lr_plan_of(L, m), m); }

// (k_lanes_gemm cuts the columns finer for fewer rows, and then takes more)
size_t lanes_rows_workspace_most(const LanesDev &L) {
    size_t most = max(lanes_rows_workspace_bytes(L, 8), lanes_rows_workspace_bytes(L, 16));
    if (lr_gemm_wins(L, 16))
        for (int m = 9; m <= 16; ++m) most = max(most, lanes_gemm_workspace_bytes(L, m));
    return most;
}

template <int BITS, int MT, bool WIDE>
static int rows_launch(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y, int64_t ldy,
                       LnScratch &ws, hipStream_t s) {
    const LrPlan p = lr_plan<BITS, MT, WIDE>(L);
    if (!ws.holds(lr_bytes(L, p, m))) return IXH_EWORKSPACE;
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_rows<BITS, MT, WIDE>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLnLds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    const bool pairs = ((uintptr_t)x & 3u) == 0 && L.in_f % 2u == 0 && ldx % 2 == 0 && ldx < 1ll << 27;
    const uint32_t blocks = (L.n_tiles + 3u) / 4u, log_waves = 31u - (uint32_t)__builtin_clz(p.waves);
    const uint32_t shape = (uint32_t)m | log_waves << 5 | (uint32_t)pairs << 8;
    IXH_LAUNCH((k_lanes_rows<BITS, MT, WIDE>), dim3(p.slices, p.groups), dim3(kWave * p.waves), p.lds, s, L.plane, x, L.exc_off,
                       L.scale, L.n_cells, L.n_tiles, L.in_f, shape, (L.n_cells / p.slices) << 20 | L.n_cells % p.slices,
                       (blocks / p.groups) << 24 | blocks % p.groups, L.exc_pos, L.exc_val, ldx, L.out_f, p.x_rows, ws.at, bias, y, ldy);
    if (p.slices > 1) return launch_lanes_reduce(ws.at, p.slices, m, L.out_f, L.n_tiles * 4u, bias, false, y, ldy, s);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

int launch_lanes_rows(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y, int64_t ldy,
                      LnScratch &ws, hipStream_t s) {
    if (lr_gemm_wins(L, m) && lanes_gemm_aligned(L, x, m, ldx)) return launch_lanes_gemm(L, x, m, ldx, bias, false, y, ldy, ws, s);
#define LR_ROWS(B)                                                                                                              \
    (lr_wide<B>(L, m) ? m <= 8 ? rows_launch<B, 8, (B == 4 || B == 5)>(L, x, m, ldx, bias, y, ldy, ws, s)                        \
                               : rows_launch<B, 16, B == 4>(L, x, m, ldx, bias, y, ldy, ws, s)                                   \
     : m <= 8         ? rows_launch<B, 8, false>(L, x, m, ldx, bias, y, ldy, ws, s)                                              \
                      : rows_launch<B, 16, false>(L, x, m, ldx, bias, y, ldy, ws, s))
    switch (L.bits) {
        case 3: return LR_ROWS(3);
        case 4: return LR_ROWS(4);
        case 5: return LR_ROWS(5);
        default: return LR_ROWS(8);
    }
#undef LR_ROWS
}

}  // namespace ixh
