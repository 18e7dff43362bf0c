// Products of few activation rows with weights in the lane layout (ixh_lanes.h), and the kernels that write it.
#include "ixh_lanes_dev.h"

namespace ixh {

template <int BITS>
__device__ __forceinline__ void ln_load(const uint32_t *__restrict__ plane, uint32_t cell, uint32_t lane, uint32_t (&w)[BITS]) {
    ln_load_lane<BITS>(plane + (size_t)cell * (64u * BITS), lane, w);
}

// sums over the lanes l, l + 16, l + 32 and l + 48, in each of them; over the lanes of a weight row, l + 4 k
__device__ __forceinline__ float lv_sum_of_rows(float v) {
    const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
    const auto g = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(g[0]) + __uint_as_float(g[1]);
}
__device__ __forceinline__ float lv_row_sum(float v) {
    v += ln_dpp<0x124>(v);
    v += ln_dpp<0x128>(v);
    return lv_sum_of_rows(v);
}

// products of a lane's four listed elements (places: two words of two byte offsets; four values) with the activations of MT rows
template <int MT>
__device__ __forceinline__ void lv_listed(const uint32_t (&at)[4], uint32_t vals, float scale, uint32_t x_row, float (&p)[4][MT]) {
    const uint32_t scale_bits = __float_as_uint(scale) & 0x7FFFFFFFu;
    const uint32_t w01 = ln_pack((float)(int)(int8_t)vals * scale, (float)(int)(int8_t)(vals >> 8) * scale);
    const uint32_t w23 = ln_pack((float)(int)(int8_t)(vals >> 16) * scale, (float)((int)vals >> 24) * scale);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t wk = k & 2 ? w23 : w01;
        const uint32_t wb = k & 1 ? wk & 0xFFFF0000u : wk << 16;
        const float wv = __uint_as_float(wb) - __uint_as_float((wb & 0x80000000u) | scale_bits);  // (no element: times 0)
#pragma unroll
        for (int r = 0; r < MT; ++r) {
            const uint32_t h = *reinterpret_cast<const LN_LDS(uint16_t) *>((uintptr_t)(at[k] + (uint32_t)r * x_row));
            p[k][r] = wv * __uint_as_float(h << 16);
        }
    }
}

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_gemv<BITS, MT, WIDE>: up to MT activation rows, MT = 1, 2 or 4.
//
// Bound: a launch's start-up and tail (some 4 us), the memory, then LDS (look-ups, activations, the list's gathers). A workgroup owns
// whole row quads, so each output is made in one place (no workspace, no second launch).  Its cells are dealt to its waves in runs
// that go down the row quads column by column: addresses depend on nothing that is loaded, and a cell's activations, read from LDS,
// serve the cells of a column (in memory order, where each cell read them anew, 5120 x 17408 at 3 bits took 11.5 us for 11.0).  The
// activations are copied to LDS once per workgroup, 16-byte pieces of a 512-column cell at piece ^ (q << 2) so that the sixteen slices
// of a wave read from different banks.
//
// Products: v_mfma_f32_16x16x32_bf16 with the weights as they lie in the lanes: its column 4 kg + row is a weight row's 8 columns kg of
// each 32, and its row 4 r + kg is activation row r at the columns kg, so that a lane's sum of its own kg is one of its four results and
// the twelve others (columns of one kg, activations of another) are thrown away.  A cell's sums over the four kg go to LDS; the row
// quad's outputs add them up in column order.  Four matrix instructions a cell, up to four activation rows, and no sums in registers
// over the loop.  (k_lanes_gemv_by_wave: a wave adds the cells of a row quad up in LDS, in their order, where cells are too many for a place each.)
//
// A wave has two cells in flight, one of them before the activations are there, and the loop over its ten or so cells is short:
// what is asked for early keeps the activations of the workgroup's later waves waiting, and much of what a launch fetches is
// instructions (us, two / three ahead, one row: 17408 x 5120 5 bits 14.9 / 15.6, 4096 x 11008 9.4 / 9.9, 5120 x 5120 7.2 / 7.8,
// 5120 x 17408 3 bits 10.4 / 10.2; both cells in front of the activations 2 to 6 % more).
//
// Listed elements: a workgroup's are one run of quads, taken 64 at a time between the cells (two thirds of their 2 us hide there) and
// dealt to the waves by such groups, wherever the row quads begin in them: weight less what the plane has there (its sign times the
// scale; the difference is exact in fp32) times gathered activation, once a group, added to the lane's sum of the row quad that the
// element is of.  (Dealt as the list of the wave's cells, a share was a part of one or two groups on a tensor with few of them, and
// every wave had some: 5120 x 17408 3 bits 11.0 -> 10.4 us, 17408 x 5120 with four rows 14.4 -> 13.4.)  One group ahead: two
// ahead 17408 x 5120 5 bits 14.9 for 14.4.  Taking the sign off costs two instructions an element; a plane without it turns an infinite
// activation in a listed column into NaN.
//
// us a call where the last-level cache has the weights / from a graph over copies that it cannot hold, one row: 5120 x 17408 3 bits 9.9 / 12.7,
// 17408 x 5120 5 bits 13.6 / 16.2, 4096 x 11008 8.7 / 11.2, 5120 x 5120 - / 7.65; at 5 bits 17408 x 5120 with two rows - / 18.0, with four - / 19.2.
// ---------------------------------------------------------------------------------------------------------------
constexpr uint32_t kLnAhead = 2;      // cells in flight
constexpr uint32_t kLnFirst = 1;      // of these, asked for before the activations are there
constexpr uint32_t kLnListAhead = 1;  // groups of the list in flight
constexpr uint32_t kLnXAhead = 3;     // 16-byte pieces of the activations a thread asks for before anything else
constexpr uint32_t kLnXPad = 64;      // bytes behind a row of activations in LDS: zeros

#define LV_ARGUMENTS                                                                                                                     \
    const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint32_t *__restrict__ exc_off,                            \
        const uint16_t *__restrict__ scale_at, uint32_t shape, uint32_t all_tiles, uint32_t tiles_per_wg, uint32_t in_f,                 \
        uint32_t inv_tiles, uint32_t list_groups, const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val, int64_t ldx, \
        const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, int64_t ldy, uint32_t out_f
template <int BITS, int MT, bool WIDE, bool BY_WAVE> __device__ __forceinline__ void lv_gemv(LV_ARGUMENTS) {
    extern __shared__ __attribute__((aligned(16))) uint8_t ln_smem[];
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)ln_smem;
    // (what the first requests need lies in the arguments that the hardware loads into registers)
    const uint32_t C = shape & 0xFFFFFu, log_waves = (shape >> 20) & 7u, m = 1u + (shape >> 24);
    const bool x_aligned = (shape >> 23) & 1u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n_waves = 1u << log_waves, n_threads = kWave << log_waves;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t t0 = blockIdx.x * tiles_per_wg;
    const uint32_t n_tiles = min(tiles_per_wg, all_tiles - t0);
    const uint32_t n_seq = tiles_per_wg * C, cell0 = t0 * C;
    const uint32_t s0 = ln_share(n_seq, wave, log_waves), s1 = ln_share(n_seq, wave + 1u, log_waves);
    const uint32_t x_at = smem + LnPairs<BITS, WIDE>::kLutBytes, x_row = C * 1024u + kLnXPad, x_pieces = MT * C * 64u;
    float *const parts = reinterpret_cast<float *>(ln_smem + LnPairs<BITS, WIDE>::kLutBytes + MT * x_row);
    float *const list_parts = parts + (BY_WAVE ? tiles_per_wg << log_waves : n_seq) * (MT * 4u);  // of wave w and row quad t at t + w
    uint32_t *const list_waves = reinterpret_cast<uint32_t *>(list_parts + (tiles_per_wg + n_waves) * (MT * 4u));

    auto x_piece = [&](uint32_t e) {
        const uint32_t r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
        ln_u32x4 v = {0u, 0u, 0u, 0u};
        if (r < m && col < in_f) {
            const uint16_t *src = x + (int64_t)r * ldx + col;
            if (x_aligned && col + 8u <= in_f) {
                v = *reinterpret_cast<const ln_u32x4 *>(src);
            } else {
                uint32_t h[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) h[k] = col + k < in_f ? src[k] : 0u;
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = h[2 * k] | (h[2 * k + 1] << 16);
            }
        }
        return v;
    };
    auto x_store = [&](uint32_t e, ln_u32x4 v) {
        const uint32_t r = MT == 1 ? 0u : e / (C * 64u), piece = e - r * (C * 64u);
        *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + r * x_row + lane_offset(piece * 8u))) = v;
    };

    // ---- everything that depends on nothing is asked for: scale, activations, the first cells, the list's extent ----
    // (Past the end requests repeat the last group or piece.  The compiler counts requests in flight, and one that may or may not have been
    // made turns its counted waits into waits for all that is older.  Requests for cells run on past a wave's share, up to two of them, the next
    // wave's, and repeat only the workgroup's last column: row quad at most n_tiles - 1, column at most C - 1.  That is 7 to 10 % more
    // bytes; turns that leave a share's last two cells to the loop behind them, and with that no request too many for an even share, took
    // between 4.5 % less and 4.5 % more over 45 layers and rows, in the mean as long.)
    const uint32_t scale_raw = *scale_at;
    ln_u32x4 xv[kLnXAhead];
    if (x_aligned)
#pragma unroll
        for (uint32_t p = 0; p < kLnXAhead; ++p) {
            if (p * n_threads >= x_pieces) break;
            const uint32_t e = min(tid + p * n_threads, x_pieces - 1u), row = MT == 1 ? 0u : e / (C * 64u);
            // whole pieces of a row only; the others are read below
            const uint32_t at = MT == 1 ? 0u : min(row, m - 1u) * (uint32_t)ldx;
            xv[p] = *reinterpret_cast<const ln_u32x4 *>(x + (at + ln_piece_column((e - row * (C * 64u)) * 8u, in_f)));
        }
    uint32_t buf[kLnAhead][BITS];
    // the share's cells, column by column
    struct At { uint32_t c, t; };
    auto at_of = [&](uint32_t s) {
        const uint32_t c = tiles_per_wg == 1 ? s : __umulhi(s, inv_tiles);
        return At{c, s - c * tiles_per_wg};
    };
    At ask = at_of(s0), now = ask;
    auto load_next = [&](uint32_t (&w)[BITS]) {
        ln_load<BITS>(plane, cell0 + min(ask.t, n_tiles - 1u) * C + ask.c, lane, w);
        if (ask.t + 1u < tiles_per_wg) ++ask.t;
        else if (ask.c + 1u < C) ask = At{ask.c + 1u, 0u};
    };
#pragma unroll
    for (uint32_t p = 0; p < kLnFirst; ++p) load_next(buf[p]);
    // where the list's ranges begin: a range is what is listed of a row quad within one segment of exc_pos; lane 63 has the end of
    // the workgroup's last one.  (A vector load, which the barrier does not wait for.)
    const uint32_t segs = (C + kLnSegCells - 1u) / kLnSegCells, n_ranges = n_tiles * segs;
    auto ranges_from = [&](uint32_t first) {
        const uint32_t k = min(first + lane, n_ranges), row = segs == 1u ? k : k / segs;
        return exc_off[cell0 + (lane == 63u ? n_tiles * C : row * C + (k - row * segs) * kLnSegCells)];
    };
    uint32_t begins = ranges_from(0u);

    __builtin_amdgcn_sched_barrier(0);

    // ---- pair table, zeroed sums and activations to LDS ----
    const float scale = bf16_bits_to_f32(scale_raw);
    ln_build_lut<BITS, WIDE>(smem, scale, tid, n_threads);
    for (uint32_t e = tid; e < n_tiles; e += n_threads) list_waves[e] = 0u;
    if constexpr (BY_WAVE)
        for (uint32_t e = tid; e < (tiles_per_wg << log_waves) * (MT * 4u); e += n_threads) parts[e] = 0.0f;
    if (tid < MT * (kLnXPad / 16u))
        *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + tid / (kLnXPad / 16u) * x_row + C * 1024u + tid % (kLnXPad / 16u) * 16u)) =
            ln_u32x4{0, 0, 0, 0};
#pragma unroll
    for (uint32_t p = 0; p < kLnXAhead; ++p) {
        const uint32_t e = tid + p * n_threads, r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
        if (e < x_pieces && x_aligned && r < m && col + 8u <= in_f) x_store(e, xv[p]);
    }
    if (x_pieces > kLnXAhead * n_threads || !x_aligned || m < MT || in_f % kLnCols != 0)
        for (uint32_t e = tid; e < x_pieces; e += n_threads) {  // what is not stored yet
            const uint32_t r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
            if (e >= kLnXAhead * n_threads || !x_aligned || r >= m || col + 8u > in_f) x_store(e, x_piece(e));
        }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t p = kLnFirst; p < kLnAhead; ++p) load_next(buf[p]);
    // The list's groups, 64 quads each, whole ones dealt to the waves.  The first is asked for in front of the barrier, and nothing waits for
    // the cells' requests before it (us from a graph, behind the barrier and the search below / here: 1536 x 1536 4.62 / 4.53, 5120 x 5120 at 5 bits
    // 7.79 / 7.75, 8192 x 2048 6.98 / 6.90).
    struct Group { ln_u32x2 pos; uint32_t val; } list[kLnListAhead];
    auto begin_of = [&](uint32_t r) { return (uint32_t)__builtin_amdgcn_readlane((int)begins, (int)r); };
    const uint32_t quads_end = begin_of(63u);
    const LnGroups all = ln_groups(begin_of(0u), quads_end, list_groups);
    const uint32_t g_first = all.first + ((wave * all.n) >> log_waves), n_groups = all.first + (((wave + 1u) * all.n) >> log_waves) - g_first;
    auto g_load = [&](uint32_t i) {
        const uint32_t g = min(g_first + i, all.last);
        return Group{*reinterpret_cast<const ln_u32x2 *>(exc_pos + (size_t)g * 256u + lane * 4u),
                     *reinterpret_cast<const uint32_t *>(exc_val + (size_t)g * 256u + lane * 4u)};
    };
#pragma unroll
    for (uint32_t p = 0; p < kLnListAhead; ++p) list[p] = g_load(p);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // the range that the first group begins in, its row quad and segment
    const uint32_t quad_first = max(g_first << 6, begin_of(0u));
    uint32_t chunk = 0;
    if (n_ranges > 62u) {
        while (begin_of(62u) <= quad_first && chunk + 62u < n_ranges) {
            chunk += 62u;
            begins = ranges_from(chunk);
        }
        asm volatile("" : "+v"(begins));  // waited for here: none is in flight where the ways meet
    }
    uint32_t range = (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(begins <= quad_first) & 0x7FFFFFFFFFFFFFFEull);
    uint32_t l_tile = segs == 1u ? chunk + range : (chunk + range) / segs, l_seg = chunk + range - l_tile * segs;
    uint32_t r0 = begin_of(range), r1 = begin_of(range + 1u);

    const uint32_t lut_lane = smem + ((lane & ((1u << LnPairs<BITS, WIDE>::kCopies) - 1u)) << 2);
    const uint32_t q = lane >> 4, kg = lane & 3u, am = min((lane >> 2) & 3u, (uint32_t)MT - 1u);
    uint32_t xa[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) xa[i] = x_at + am * x_row + q * 256u + ((i ^ q) << 6) + kg * 16u;

    float ex[MT];  // of the lane's row
#pragma unroll
    for (int r = 0; r < MT; ++r) ex[r] = 0.0f;
    // one group of listed elements, range by range: the lane has four of its row, quads quad .. quad + 3
    auto list_group = [&](const Group &in, uint32_t i) {
        const uint32_t g0 = (g_first + i) << 6, quad = g0 + (lane & ~3u), vals = in.val;
        float p[4][MT];
        for (bool first = true;; first = false) {
            if (first || C >= kLnSegCells) {  // (positions start over in the next segment)
                uint32_t at[4] = {x_at + (in.pos[0] & 0xFFFFu), x_at + (in.pos[0] >> 16), x_at + (in.pos[1] & 0xFFFFu), x_at + (in.pos[1] >> 16)};
                if (C >= kLnSegCells)
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        at[k] = x_at + ln_listed_at(at[k] - x_at, (vals >> (8 * k)) & 255u, quad + k - r0 < r1 - r0, l_seg, C);
                lv_listed<MT>(at, vals, scale, x_row, p);
            }
            if (g0 < r0 || g0 + 64u > r1) {  // quads of other ranges among them
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
                    for (int r = 0; r < MT; ++r) ex[r] += quad + k - r0 < r1 - r0 ? p[k][r] : 0.0f;
            } else {
#pragma unroll
                for (int r = 0; r < MT; ++r) ex[r] += (p[0][r] + p[1][r]) + (p[2][r] + p[3][r]);
            }
            const bool goes_on = g0 + 64u < r1, row_ends = !goes_on && l_seg + 1u == segs;
            // all that the wave has of the row quad (nothing may be listed in its other segments)
            if (row_ends || (goes_on ? i + 1u == n_groups : r1 >= quads_end || (i + 1u == n_groups && r1 == g0 + 64u))) {
#pragma unroll
                for (int r = 0; r < MT; ++r) {
                    const float v = lv_row_sum(ex[r]);
                    if (lane < 4) list_parts[(l_tile + wave) * (MT * 4u) + (uint32_t)r * 4u + lane] = v;
                    ex[r] = 0.0f;
                }
                if (lane == 0) __hip_atomic_fetch_or(list_waves + l_tile, 1u << wave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (goes_on) break;
            l_tile += row_ends;
            l_seg = row_ends ? 0u : l_seg + 1u;
            r0 = r1;
            if (r0 >= quads_end) break;
            if (++range < 62u) {
                r1 = begin_of(range + 1u);
            } else {
                const uint32_t next = l_seg + 1u == segs ? (l_tile + 1u) * C : l_tile * C + (l_seg + 1u) * kLnSegCells;
                r1 = exc_off[cell0 + next];
                asm volatile("" : "+s"(r1));  // waited for here: none is in flight where the ways meet
            }
            if (r0 >= g0 + 64u) break;
        }
    };

    uint32_t s = s0, g = 0;
    auto list_next = [&] {
        list_group(list[0], g);
#pragma unroll
        for (uint32_t p = 1; p < kLnListAhead; ++p) list[p - 1] = list[p];
        list[kLnListAhead - 1] = g_load(g + kLnListAhead);
        ++g;
    };
    // an activation operand serves the cells of a column
    ln_u32x4 xc[4];
    auto x_read = [&] {
#pragma unroll
        for (int i = 0; i < 4; ++i) xc[i] = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(xa[i] + now.c * 1024u));
    };
    x_read();
    const bool kg0 = (lane & 4u) != 0, kg1 = (lane & 8u) != 0;
    uint32_t part_at = (uint32_t)(uintptr_t)(LN_LDS(float) *)parts + (BY_WAVE ? wave * tiles_per_wg : s0) * (MT * 16u) + (lane >> 4) * 16u + (lane & 3u) * 4u;
    auto cell = [&](uint32_t (&w)[BITS], bool more) {
        uint32_t o[16];
        float before = 0.0f;
        const uint32_t to = BY_WAVE ? part_at + now.t * (MT * 16u) : part_at;
        if constexpr (BY_WAVE) before = *reinterpret_cast<const LN_LDS(float) *>((uintptr_t)to);
        ln_decode<BITS, WIDE>(w, lut_lane, scale, o);
        if (more) load_next(w);
        ln_f32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_bf16x8, xc[i]),
                                                        __builtin_bit_cast(ln_bf16x8, ln_u32x4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]}), d, 0, 0, 0);
        ++s;
        if (++now.t == tiles_per_wg) {
            now = At{now.c + 1u < C ? now.c + 1u : now.c, 0u};
            x_read();
        }
        float v = kg1 ? (kg0 ? d[3] : d[2]) : (kg0 ? d[1] : d[0]);
        v += ln_dpp<0x124>(v);
        v += ln_dpp<0x128>(v);
        if ((lane & 12u) == 0 && lane < MT * 16u) *reinterpret_cast<LN_LDS(float) *>((uintptr_t)to) = BY_WAVE ? before + v : v;
        if constexpr (!BY_WAVE) part_at += MT * 16u;
    };
    // Whole turns of the buffers, without a way out in between: with one the compiler takes the last request made before it
    // for the first buffer's and waits for all that is in flight at the top of every turn.
    while (s + kLnAhead <= s1) {
        // Left alone, the waves of a SIMD are served oldest first; a wave that has more cells to go takes precedence (3 bits
        // 10.4 us, 10.9 without; the shares are uneven as well, see ln_share).
        const uint32_t behind = (s1 - s) * 4u / (s1 - s0 + 1u);
        if (behind >= 3u) __builtin_amdgcn_s_setprio(3);
        else if (behind == 2u) __builtin_amdgcn_s_setprio(2);
        else if (behind == 1u) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (uint32_t p = 0; p < kLnAhead; ++p) cell(buf[p], true);
        // as large a part of the list as of the cells
#pragma unroll 1
        while (g * (s1 - s0) < n_groups * (s - s0)) list_next();
    }
#pragma unroll 1
    while (s < s1) {
        cell(buf[0], false);
#pragma unroll
        for (uint32_t p = 1; p < kLnAhead; ++p)
#pragma unroll
            for (int d = 0; d < BITS; ++d) buf[p - 1][d] = buf[p][d];
    }
#pragma unroll 1
    while (g < n_groups) list_next();
    __syncthreads();

    // ---- outputs: a row quad's sums over the columns and the waves' parts of the list ----
    for (uint32_t t = wave; t < n_tiles; t += n_waves) {
        const uint32_t part = lane >> 2, at = (t0 + t) * 4u + (lane & 3u);
        const bool listed = (list_waves[t] >> part) & 1u;
#pragma unroll
        for (int r = 0; r < MT; ++r) {
            float sum = listed ? list_parts[(t + part) * (MT * 4u) + (uint32_t)r * 4u + (lane & 3u)] : 0.0f;
            for (uint32_t c = part; c < (BY_WAVE ? n_waves : C); c += 16u) sum += parts[(c * tiles_per_wg + t) * (MT * 4u) + (uint32_t)r * 4u + (lane & 3u)];
            sum = lv_row_sum(sum);
            if (lane < 4 && at < out_f && (uint32_t)r < m) {
                uint32_t b = f32_to_bf16_bits(sum);
                if (bias) b = f32_to_bf16_bits(bf16_bits_to_f32(b) + bf16_bits_to_f32(bias[at]));
                y[(int64_t)r * ldy + at] = (uint16_t)b;
            }
        }
    }
}

#define LV_PASSED plane, x, exc_off, scale_at, shape, all_tiles, tiles_per_wg, in_f, inv_tiles, list_groups, exc_pos, exc_val, ldx, bias, y, ldy, out_f
template <int BITS, int MT, bool WIDE> __global__ void __launch_bounds__(1024) k_lanes_gemv(LV_ARGUMENTS) {
    lv_gemv<BITS, MT, WIDE, false>(LV_PASSED);
}
template <int BITS, int MT, bool WIDE> __global__ void __launch_bounds__(1024) k_lanes_gemv_by_wave(LV_ARGUMENTS) {
    lv_gemv<BITS, MT, WIDE, true>(LV_PASSED);
}
#undef LV_ARGUMENTS
#undef LV_PASSED

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_gemv_few<BITS, MT, N>: the same where a wave has one cell, or two (N).
//
// Bound: a launch, its instructions' way from the caches (3 to 7 KB of them; k_lanes_gemv has 9 to 14, of which such a layer runs through
// all but its loop) and one chain of requests: scale, activations, cells and where their lists lie, then the lists.  All of them are made
// before anything is waited for.  A cell's part of the list is in one segment and one row quad, so nothing is dealt or searched, and
// its sums join the cell's.  The smaller pair table: the larger one takes longer to write than it saves.  us from a graph, k_lanes_gemv / this:
// one row 256 x 512 4.52 / 3.40, 1536 x 1536 (3 bits) 4.42 / 3.28, 4096 x 1024 (5) 4.43 / 3.52; four rows 1536 x 1536 (3) 5.84 / 3.92; two cells: 3000 x
// 3000 (5) 5.40 / 4.89, 8192 x 2048 (3) 5.94 / 5.42, (5) 6.85 / 6.65, 4096 x 4096 at 4 bits 6.40 / 6.49, four rows 8.70 / 8.35 (5).
// ---------------------------------------------------------------------------------------------------------------
template <int BITS, int MT, int N>
__global__ void __launch_bounds__(1024)
k_lanes_gemv_few(const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint32_t *__restrict__ exc_off,
                 const uint16_t *__restrict__ scale_at, const uint16_t *__restrict__ bias, uint32_t shape, uint32_t inv_cells,
                 uint32_t out_f, uint32_t in_f, const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val,
                 int64_t ldx, uint16_t *__restrict__ y, int64_t ldy) {
    extern __shared__ __attribute__((aligned(16))) uint8_t ln_smem[];
    using P = LnPairs<BITS, false>;
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)ln_smem;
    const uint32_t C = shape & 255u, tiles_per_wg = (shape >> 8) & 255u, n_waves = 1u << ((shape >> 16) & 7u), m = 1u + (shape >> 20);
    const bool x_aligned = (shape >> 19) & 1u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t t0 = blockIdx.x * tiles_per_wg, cell0 = t0 * C, n_here = min(tiles_per_wg, ((out_f + 3u) >> 2) - t0) * C;
    const uint32_t x_at = smem + P::kLutBytes, x_row = C * 1024u + kLnXPad;
    float *const parts = reinterpret_cast<float *>(ln_smem + P::kLutBytes + MT * x_row);

    // ---- all requests (for cells that a wave does not have, the last one's) ----
    uint32_t bias_raw[N];
#pragma unroll
    for (uint32_t n = 0; n < N; ++n) bias_raw[n] = *(bias ? bias + min((t0 + wave + n * n_waves) * 4u + (lane & 3u), out_f - 1u) : scale_at);
    const uint32_t scale_raw = *scale_at, col = tid * 8u;
    ln_u32x4 xv[MT];
    if (x_aligned)
#pragma unroll
        for (uint32_t r = 0; r < MT; ++r)
            xv[r] = *reinterpret_cast<const ln_u32x4 *>(x + (int64_t)min(r, m - 1u) * ldx + ln_piece_column(col, in_f));
    uint32_t w[N][BITS], e0[N], e1[N];
#pragma unroll
    for (uint32_t n = 0; n < N; ++n) {
        const uint32_t cell = cell0 + min(wave + n * n_waves, n_here - 1u);
        ln_load<BITS>(plane, cell, lane, w[n]);
        e0[n] = exc_off[cell], e1[n] = exc_off[cell + 1u];
    }
    asm volatile("" ::"s"(y), "s"(ldy));  // (arguments that are read from memory: with these, not at the end)
    // 64 quads of the list from a multiple of four on: the lane has four of its row
    struct Listed { ln_u32x2 pos; uint32_t val; };
    auto list_load = [&](uint32_t from, uint32_t end) {
        const uint32_t at = ln_four_quads(from, lane, end) * 16u + (lane & 3u) * 4u;
        return Listed{*reinterpret_cast<const ln_u32x2 *>(exc_pos + at), *reinterpret_cast<const uint32_t *>(exc_val + at)};
    };
    Listed in[N];
#pragma unroll
    for (uint32_t n = 0; n < N; ++n) in[n] = list_load(e0[n] & ~3u, e1[n]);
    __builtin_amdgcn_sched_barrier(0);

    // ---- pair table and activations to LDS: a thread has the same piece of each row ----
    const float scale = bf16_bits_to_f32(scale_raw);
    ln_build_lut<BITS, false>(smem, scale, tid, n_waves * kWave);
    if (tid < MT * (kLnXPad / 16u))
        *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + tid / (kLnXPad / 16u) * x_row + C * 1024u + tid % (kLnXPad / 16u) * 16u)) =
            ln_u32x4{0, 0, 0, 0};
    if (tid < C * 64u) {
#pragma unroll
        for (uint32_t r = 0; r < MT; ++r) {
            ln_u32x4 v = {0u, 0u, 0u, 0u};
            if (x_aligned && col + 8u <= in_f) {
                if (r < m) v = xv[r];
            } else if (r < m) {
                const uint16_t *const src = x + (int64_t)r * ldx;
                uint32_t h[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) h[k] = src[min(col + k, in_f - 1u)];
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    v[k] = (col + 2u * k < in_f ? h[2 * k] : 0u) | (col + 2u * k + 1u < in_f ? h[2 * k + 1] << 16 : 0u);
            }
            *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + r * x_row + lane_offset(col))) = v;
        }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    const uint32_t lut_lane = smem + ((lane & ((1u << P::kCopies) - 1u)) << 2);
    const uint32_t q = lane >> 4, kg = lane & 3u, am = min((lane >> 2) & 3u, (uint32_t)MT - 1u), x_lane = x_at + am * x_row + q * 256u + kg * 16u;
    const bool kg0 = (lane & 4u) != 0, kg1 = (lane & 8u) != 0;
#pragma unroll
    for (uint32_t n = 0; n < N; ++n) {
        // ---- the cell's products (see k_lanes_gemv) ----
        if (n && wave + n * n_waves >= n_here) break;
        const uint32_t cell = wave + n * n_waves, x_cell = x_lane + (cell - ((cell * inv_cells) >> 16) * C) * 1024u;
        uint32_t o[16];
        ln_decode<BITS, false>(w[n], lut_lane, scale, o);
        ln_f32x4 d = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const ln_u32x4 a = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(x_cell + ((i ^ q) << 6)));
            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_bf16x8, a),
                                                        __builtin_bit_cast(ln_bf16x8, ln_u32x4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]}), d, 0, 0, 0);
        }
        float v = kg1 ? (kg0 ? d[3] : d[2]) : (kg0 ? d[1] : d[0]);
        v += ln_dpp<0x124>(v);
        v += ln_dpp<0x128>(v);
        // ---- its listed elements (a first group also where there are none: behind a branch it would not be asked for before it) ----
        float ex[MT];
#pragma unroll
        for (int r = 0; r < MT; ++r) ex[r] = 0.0f;
        uint32_t from = e0[n] & ~3u;
#pragma unroll 1
        for (;;) {
            const uint32_t at[4] = {x_at + (in[n].pos[0] & 0xFFFFu), x_at + (in[n].pos[0] >> 16), x_at + (in[n].pos[1] & 0xFFFFu), x_at + (in[n].pos[1] >> 16)};
            float p[4][MT];
            lv_listed<MT>(at, in[n].val, scale, x_row, p);
            const uint32_t quad = from + (lane & ~3u) - e0[n];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < MT; ++r) ex[r] += quad + k < e1[n] - e0[n] ? p[k][r] : 0.0f;
            from += 64u;
            if (from >= e1[n]) break;
            in[n] = list_load(from, e1[n]);
        }
#pragma unroll
        for (uint32_t r = 0; r < MT; ++r) {
            const float sum = lv_row_sum(ex[r]);
            v += lane >> 4 == r ? sum : 0.0f;
        }
        if (cell < n_here && (lane & 12u) == 0 && lane < MT * 16u) parts[cell * (MT * 4u) + (lane >> 4) * 4u + (lane & 3u)] = v;
    }
    __syncthreads();

    // ---- outputs: a row quad's sums over the columns ----
#pragma unroll
    for (uint32_t n = 0; n < N; ++n) {
        const uint32_t t = wave + n * n_waves, at = lane & (MT * 4u - 1u), out_row = (t0 + t) * 4u + (lane & 3u), r = lane >> 2;
        if (t * C >= n_here) break;
        float sum = 0.0f;
        for (uint32_t k = lane / (MT * 4u); k < C; k += 64u / (MT * 4u)) sum += parts[(t * C + k) * (MT * 4u) + at];
        if (MT == 1) sum += ln_dpp<0x124>(sum);
        if (MT <= 2) sum += ln_dpp<0x128>(sum);
        sum = lv_sum_of_rows(sum);
        if (r < m && out_row < out_f) {
            uint32_t b = f32_to_bf16_bits(sum);
            if (bias) b = f32_to_bf16_bits(bf16_bits_to_f32(b) + bf16_bits_to_f32(bias_raw[n]));
            y[(int64_t)r * ldy + out_row] = (uint16_t)b;
        }
    }
}

// outputs from the slices' sums, in slice order
__global__ void __launch_bounds__(256)
k_lanes_reduce(const float *__restrict__ ws, uint32_t slices, int m, uint32_t out_f, uint32_t ws_ld,
               const uint16_t *__restrict__ bias, bool once, uint16_t *__restrict__ y, int64_t ldy) {
    const uint32_t row = blockIdx.x * 256u + threadIdx.x, r = blockIdx.y;
    if (row >= out_f) return;
    const float *p = ws + (size_t)r * ws_ld + row;
    const size_t stride = (size_t)m * ws_ld;
    float sum = 0.0f;
    for (uint32_t g = 0; g < slices; g += 8) {
        float v[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) v[k] = p[(size_t)min(g + k, slices - 1u) * stride];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
            if (g + k < slices) sum += v[k];
    }
    uint32_t h = f32_to_bf16_bits(sum);
    if (bias) h = f32_to_bf16_bits((once ? sum : bf16_bits_to_f32(h)) + bf16_bits_to_f32(bias[row]));
    y[(int64_t)r * ldy + row] = (uint16_t)h;
}

int launch_lanes_reduce(const float *ws, uint32_t slices, int m, uint32_t out_f, uint32_t ws_ld, const uint16_t *bias, bool once,
                        uint16_t *y, int64_t ldy, hipStream_t s) {
    IXH_LAUNCH(k_lanes_reduce, dim3((out_f + 255u) / 256u, m), dim3(256), 0, s, ws, slices, m, out_f, ws_ld, bias, once,
                       y, ldy);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

// ---------------------------------------------------------------------------------------------------------------
// Writing the layout from the decoded bf16 weights (deploy time): one wave per cell.  value = round(w / scale) gives
// back the integer exactly (w is value * scale rounded to 8 significant bits, |value| <= 128).
// ---------------------------------------------------------------------------------------------------------------
template <int BITS>
__device__ __forceinline__ void ln_cell_values(const uint16_t *__restrict__ w, const LanesDev &L, uint32_t cell,
                                               uint32_t lane, int (&v)[32]) {
    const uint32_t t = cell / L.n_cells, c = cell - t * L.n_cells;
    const uint32_t row = 4u * t + (lane & 3u), col0 = kLnCols * c + 128u * (lane >> 4) + 8u * ((lane >> 2) & 3u);
    const float scale = bf16_bits_to_f32(*L.scale);
#pragma unroll
    for (uint32_t e = 0; e < 32; ++e) {
        const uint32_t col = col0 + 32u * (e >> 3) + (e & 7u);
        v[e] = 0;
        if (row < L.out_f && col < L.in_f)
            v[e] = __float2int_rn(bf16_bits_to_f32(w[(size_t)row * L.in_f + col]) / scale);
    }
}

template <int BITS> __device__ __forceinline__ bool ln_listed(int v) {
    constexpr int T = (1 << (BITS - 1)) - 1;
    return v > T || v < -T;
}

template <int BITS>
__global__ void __launch_bounds__(256)
k_lanes_pack(const uint16_t *__restrict__ w, LanesDev L, uint32_t *__restrict__ plane, uint32_t *__restrict__ counts) {
    const uint32_t lane = threadIdx.x & 63u, cell = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (cell >= L.n_tiles * L.n_cells) return;
    int v[32];
    ln_cell_values<BITS>(w, L, cell, lane, v);
    constexpr int T = (1 << (BITS - 1)) - 1;
    uint32_t n = 0, code[32], d[BITS];
#pragma unroll
    for (int e = 0; e < 32; ++e) {
        const bool listed = ln_listed<BITS>(v[e]);
        n += listed;
        code[e] = (uint32_t)((listed ? (v[e] > 0 ? 1 : -1) : v[e]) + T);
    }
#pragma unroll
    for (int k = 0; k < BITS; ++k) d[k] = 0;
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const uint32_t pair = code[2 * p] | (code[2 * p + 1] << BITS);
        if constexpr (BITS == 8) d[p >> 1] |= pair << (16 * (p & 1));
        else if constexpr (BITS == 4) d[p >> 2] |= pair << (8 * (p & 3));
        else {
            constexpr int PER = BITS == 3 ? 5 : 3;
            if (p < 15) d[p / PER] |= pair << (2 + 2 * BITS * (p % PER));
            else
                for (int k = 0; k < BITS; ++k) d[k] |= (pair >> (2 * k)) & 3u;
        }
    }
    uint32_t *out = plane + (size_t)cell * (64u * BITS);
    constexpr int HEAD = BITS < 4 ? BITS : 4;
#pragma unroll
    for (int k = 0; k < BITS; ++k) {
        if (k < HEAD) out[lane * HEAD + k] = d[k];
        else out[64 * HEAD + lane * (BITS - HEAD) + (k - HEAD)] = d[k];
    }
    for (int o = 4; o < 64; o <<= 1) n += __shfl_xor(n, o);  // of the lane's row
    n = max(n, (uint32_t)__shfl_xor(n, 1));
    n = max(n, (uint32_t)__shfl_xor(n, 2));
    if (lane == 0) counts[cell] = n;
}

template <int BITS>
__global__ void __launch_bounds__(256)
k_lanes_list(const uint16_t *__restrict__ w, LanesDev L, uint16_t *__restrict__ pos, int8_t *__restrict__ val) {
    const uint32_t lane = threadIdx.x & 63u, cell = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (cell >= L.n_tiles * L.n_cells) return;
    int v[32];
    ln_cell_values<BITS>(w, L, cell, lane, v);
    uint32_t n = 0;
#pragma unroll
    for (int e = 0; e < 32; ++e) n += ln_listed<BITS>(v[e]);
    uint32_t before = n;  // listed elements of the row in the slices up to this one
    for (int o = 4; o < 64; o <<= 1) {
        const uint32_t u = __shfl_up(before, o);
        if (lane >= (uint32_t)o) before += u;
    }
    uint32_t at = L.exc_off[cell] + before - n;
    const uint32_t end = L.exc_off[cell + 1];
    const uint32_t col0 = (kLnCols * (cell % L.n_cells) + 128u * (lane >> 4) + 8u * ((lane >> 2) & 3u)) % (kLnSegCells * kLnCols);
#pragma unroll
    for (uint32_t e = 0; e < 32; ++e)
        if (ln_listed<BITS>(v[e]) && at < end) {
            pos[lane_listed(at, lane & 3u)] = (uint16_t)lane_offset(col0 + 32u * (e >> 3) + (e & 7u));
            val[lane_listed(at, lane & 3u)] = (int8_t)v[e];
            ++at;
        }
}

int launch_lanes_pack(const uint16_t *w, const LanesDev &L, uint32_t *plane, uint32_t *counts, hipStream_t s) {
    const dim3 grid((L.n_tiles * L.n_cells + 3u) / 4u), block(256);
    switch (L.bits) {
        case 3: hipLaunchKernelGGL(k_lanes_pack<3>, grid, block, 0, s, w, L, plane, counts); break;
        case 4: hipLaunchKernelGGL(k_lanes_pack<4>, grid, block, 0, s, w, L, plane, counts); break;
        case 5: hipLaunchKernelGGL(k_lanes_pack<5>, grid, block, 0, s, w, L, plane, counts); break;
        default: hipLaunchKernelGGL(k_lanes_pack<8>, grid, block, 0, s, w, L, plane, counts); break;
    }
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

int launch_lanes_list(const uint16_t *w, const LanesDev &L, uint16_t *pos, int8_t *val, hipStream_t s) {
    const dim3 grid((L.n_tiles * L.n_cells + 3u) / 4u), block(256);
    const int rc = launch_fill_u16(pos, L.list_groups * 256u, (uint16_t)lane_none(L.n_cells), s);
    if (rc != IXH_OK) return rc;
    switch (L.bits) {
        case 3: hipLaunchKernelGGL(k_lanes_list<3>, grid, block, 0, s, w, L, pos, val); break;
        case 4: hipLaunchKernelGGL(k_lanes_list<4>, grid, block, 0, s, w, L, pos, val); break;
        case 5: hipLaunchKernelGGL(k_lanes_list<5>, grid, block, 0, s, w, L, pos, val); break;
        default: hipLaunchKernelGGL(k_lanes_list<8>, grid, block, 0, s, w, L, pos, val); break;
    }
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

// Workgroups of 16, 8 or 4 waves, one, two or four to a CU: the split whose last round of row quads is fullest.  No waves where LDS
// holds none: its first pass, sixteen waves, decides that.
struct LvSplit { uint32_t waves, tiles; };
template <int BITS, int MT, bool WIDE, bool BY_WAVE> static size_t lv_lds(const LanesDev &L, uint32_t tiles, uint32_t waves) {
    return LnPairs<BITS, WIDE>::kLutBytes + (size_t)MT * (L.n_cells * 1024u + kLnXPad) + ((size_t)tiles * ((BY_WAVE ? waves : L.n_cells) + 1u) + waves) * (MT * 16u) + tiles * 4u;
}
// Several rows of layers of many row quads a CU and few cells to each: k_lanes_rows, which has 16 weight rows to a wave's sums, is faster (us from
// graphs, k_lanes_gemv / k_lanes_rows, at 3 / 4 / 5 bits: four rows 24576 x 5120 18.7 / 21.3 / 23.7 and 17.9 / 21.4 / 24.3, 32768 x 4096 19.9 / 22.1 / 24.9
// and 16.9 / 21.3 / 24.0, 131072 x 1024 28.8 / 29.3 / 32.5 and 18.3 / 22.3 / 25.4; two rows 32768 x 1024 10.9 / 11.5 / 12.0 and 10.4 / 11.2 / 12.3, 65536 x
// 2048 19.7 / 21.5 / 23.2 and 17.2 / 21.1 / 23.8, 248320 x 1024 36.7 / 45.1 / 51.3 and 28.8 / 43.4 / 50.9; 128256 x 4096 at 3 and 5 bits 51.7 / 84.3 and before
// k_lanes_gemv had the room 57.5 / 92.3).
template <int MT> static bool lv_rows_win(const LanesDev &L) {
    const uint32_t tiles = (L.n_tiles + ln_cus() - 1) / ln_cus();
    return MT == 4 ? tiles > 30u && tiles * L.n_cells > 32u : MT == 2 && tiles > 60u && L.n_cells <= 4u;
}
template <int BITS, int MT, bool WIDE, bool BY_WAVE = false> static LvSplit lv_split(const LanesDev &L) {
    LvSplit best{};
    if (lv_rows_win<MT>(L)) return best;
    uint64_t best_cost = ~0ull;
    for (uint32_t per_cu = 1; per_cu <= 4; per_cu *= 2) {
        const uint32_t waves = 16u / per_cu, slots = ln_cus() * per_cu;
        const uint32_t tiles = (L.n_tiles + slots - 1) / slots;
        if (lv_lds<BITS, MT, WIDE, BY_WAVE>(L, tiles, waves) * per_cu > kLnLds) break;
        const uint64_t cost = (uint64_t)tiles * per_cu;  // row quads a CU works through
        if (cost < best_cost) { best_cost = cost; best = {waves, tiles}; }
    }
    return best;
}

// row quads by `tiles` to a workgroup of `waves`, N cells a wave
template <int BITS, int MT, int N>
static int lanes_gemv_few_launch(const LanesDev &L, uint32_t tiles, uint32_t waves, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias,
                                 uint16_t *y, int64_t ldy, hipStream_t s) {
    const size_t lds = LnPairs<BITS, false>::kLutBytes + MT * (L.n_cells * 1024u + kLnXPad) + tiles * L.n_cells * (MT * 16u);
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_gemv_few<BITS, MT, N>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLnLds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    const bool aligned = ln_whole_pieces((uintptr_t)x, L.in_f, m, ldx);
    const uint32_t shape = L.n_cells | tiles << 8 | (uint32_t)__builtin_ctz(waves) << 16 | (uint32_t)aligned << 19 | (uint32_t)(m - 1) << 20;
    // (a cell / n_cells as a product with 2^16 / n_cells, rounded up: exact for the 32 cells that there are at most)
    IXH_LAUNCH((k_lanes_gemv_few<BITS, MT, N>), dim3((L.n_tiles + tiles - 1u) / tiles), dim3(kWave * waves), lds, s, L.plane, x, L.exc_off,
                       L.scale, bias, shape, 65536u / L.n_cells + 1u, L.out_f, L.in_f, L.exc_pos, L.exc_val, ldx, y, ldy);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

template <int BITS, int MT, bool WIDE, bool BY_WAVE = false>
static int lanes_gemv_launch(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                             int64_t ldy, hipStream_t s) {
    const auto [best_waves, best_tiles] = lv_split<BITS, MT, WIDE, BY_WAVE>(L);
    // A cell or two a wave: up to two cells a wave k_lanes_gemv is slower or even, see there.  (A thread takes one piece of a row of activations:
    // no more cells in a row than waves.)
    if (best_waves && L.n_cells <= best_waves && best_tiles * L.n_cells <= 2u * best_waves) {
        uint32_t waves = best_waves;
        while (waves / 2u >= best_tiles * L.n_cells) waves /= 2u;
        if (best_tiles * L.n_cells <= waves) return lanes_gemv_few_launch<BITS, MT, 1>(L, best_tiles, waves, x, m, ldx, bias, y, ldy, s);
        return lanes_gemv_few_launch<BITS, MT, 2>(L, best_tiles, waves, x, m, ldx, bias, y, ldy, s);
    }
    // Sums by wave where there is no room for sums by cell, which save an LDS read a cell (us from graphs, k_lanes_rows or the smaller
    // pair table in their place / so: two rows 65536 x 20480 at 5 bits 227 / 203, 20480 x 30720 108 / 100, 16384 x 32768 at 3 bits 54.4 / 51.8, 4096 x 36864
    // 20.4 / 21.5; one row 20480 x 40960 at 5 bits 129.6 / 125.8).
    if constexpr (!BY_WAVE && MT <= 2)
        if (!best_waves && L.n_cells > 16u) {
            const int rc = lanes_gemv_launch<BITS, MT, WIDE, true>(L, x, m, ldx, bias, y, ldy, s);
            if (rc != IXH_EUNSUPPORTED) return rc;
        }
    // the smaller pair table where rows are too long beside the larger one
    if constexpr (!BY_WAVE && WIDE && (BITS == 4 || BITS == 5) && MT <= 2)
        if (!best_waves) return lanes_gemv_launch<BITS, MT, false>(L, x, m, ldx, bias, y, ldy, s);
    if (!best_waves) return IXH_EUNSUPPORTED;
    uint32_t log_waves = 31u - (uint32_t)__builtin_clz(best_waves);
    while ((1u << log_waves) > best_tiles * L.n_cells) --log_waves;
    const auto kernel = [] {
        if constexpr (BY_WAVE) return k_lanes_gemv_by_wave<BITS, MT, WIDE>;
        else return k_lanes_gemv<BITS, MT, WIDE>;
    }();
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLnLds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    // (the kernel's offsets of 16-byte pieces are 32 bits of elements)
    const bool aligned = ln_whole_pieces((uintptr_t)x, L.in_f, m, ldx) && (m == 1 || ldx < (1ll << 30));
    const uint32_t shape = L.n_cells | log_waves << 20 | (uint32_t)aligned << 23 | (uint32_t)(m - 1) << 24;
    // quotients by best_tiles as products with 2^32 / best_tiles, rounded up: exact for the cells of a workgroup, n_cells * best_tiles,
    // while these times best_tiles are below 2^32; each has 16 bytes of LDS
    const uint32_t inv_tiles = best_tiles == 1 ? 0u : (uint32_t)(((1ull << 32) + best_tiles - 1u) / best_tiles);
    IXH_LAUNCH(kernel, dim3((L.n_tiles + best_tiles - 1) / best_tiles), dim3(kWave << log_waves),
                       (lv_lds<BITS, MT, WIDE, BY_WAVE>(L, best_tiles, 1u << log_waves)), s, L.plane, x, L.exc_off, L.scale, shape, L.n_tiles, best_tiles, L.in_f,
                       inv_tiles, L.list_groups, L.exc_pos, L.exc_val, ldx, bias, y, ldy, L.out_f);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

template <int BITS>
static int lanes_gemv_rows(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                           int64_t ldy, LnScratch &ws, hipStream_t s) {
    int rc = IXH_EUNSUPPORTED;
    if (m == 1) rc = lanes_gemv_launch<BITS, 1, true>(L, x, m, ldx, bias, y, ldy, s);
    else if (m == 2) rc = lanes_gemv_launch<BITS, 2, true>(L, x, m, ldx, bias, y, ldy, s);
    else if (m <= 4) rc = lanes_gemv_launch<BITS, 4, true>(L, x, m, ldx, bias, y, ldy, s);
    return rc == IXH_EUNSUPPORTED ? launch_lanes_rows(L, x, m, ldx, bias, y, ldy, ws, s) : rc;
}

// whether lanes_gemv_launch finds a split
template <int BITS> static bool lanes_gemv_fits(const LanesDev &L, int m) {
    constexpr bool SMALLER = BITS != 4 && BITS != 5;  // (a smaller table of pairs, up to two rows)
    if (m == 1) return lv_split<BITS, 1, SMALLER>(L).waves != 0 || (L.n_cells > 16u && lv_split<BITS, 1, SMALLER, true>(L).waves != 0);
    if (m == 2) return lv_split<BITS, 2, SMALLER>(L).waves != 0 || (L.n_cells > 16u && lv_split<BITS, 2, SMALLER, true>(L).waves != 0);
    return m <= 4 && lv_split<BITS, 4, true>(L).waves != 0;
}
bool lanes_gemv_takes(const LanesDev &L, int m) {
    switch (L.bits) {
        case 3: return lanes_gemv_fits<3>(L, m);
        case 4: return lanes_gemv_fits<4>(L, m);
        case 5: return lanes_gemv_fits<5>(L, m);
        default: return lanes_gemv_fits<8>(L, m);
    }
}

int launch_lanes_gemv(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                      int64_t ldy, LnScratch &ws, hipStream_t s) {
    switch (L.bits) {
        case 3: return lanes_gemv_rows<3>(L, x, m, ldx, bias, y, ldy, ws, s);
        case 4: return lanes_gemv_rows<4>(L, x, m, ldx, bias, y, ldy, ws, s);
        case 5: return lanes_gemv_rows<5>(L, x, m, ldx, bias, y, ldy, ws, s);
        default: return lanes_gemv_rows<8>(L, x, m, ldx, bias, y, ldy, ws, s);
    }
}

}  // namespace ixh
