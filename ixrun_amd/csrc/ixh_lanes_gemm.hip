// Products of 5 and more activation rows with weights in the lane layout (ixh_lanes.h).
#include "ixh_lanes_dev.h"

namespace ixh {

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_gemm<BITS, MB, NB>: up to 16 * MB activation rows at a time, MB <= 8; NB blocks of 16 weight rows a wave (two from
// MB = 4 on: an activation operand that is read serves both).
//
// Bound: a stage's parts (decode and its stores, listed elements, products), which follow one another in a wave, while all waves meet at its
// end, and LDS under them; no unit of the CU is busy for more than half of a stage, the matrix unit for 12 %.  10240 x 5120 at 55 / 40 / 5 %,
// 100 rows: 37.4 us with the slices' sums (44.2 when a lane held an element of each of four rows of the list, so that a store of listed elements
// went to a quarter of the banks, 39.0 with a branch around each such store); 74.3 for the decode to memory and the library's GEMM.  Looking up the next stage's
// weights between the products of this one changes nothing, nor do two workgroups of half the size on a CU; activations straight from
// the L2 as operands take twice as long.  A wave takes 16 weight rows x 128 columns a stage: it decodes them to its own 4 KB of LDS in
// operand order, stores the listed elements over their places and reads the operands back.  All waves of the workgroup are in the same
// 128 columns, whose activations one copy in LDS serves (in operand order, two stages of it: the next one is fetched during the
// multiply), so a weight is decoded once per 128 activation rows and never reaches memory.  One barrier a stage, which waits for LDS
// only: codes and list are asked for one cell ahead.
//
// A workgroup owns a slice of the columns (whole cells) of a run of 16-row blocks, sixteen at most at a time; the slices' sums
// meet in the workspace and launch_lanes_reduce adds them in slice order.
// ---------------------------------------------------------------------------------------------------------------
constexpr uint32_t kLgBlocks = 16;  // of 16 weight rows, in work at a time
constexpr uint32_t kLgTile = 4096;
// whether a store of a listed element has a branch around it; otherwise what is not to be stored goes to a dword a lane behind the tile
template <int BITS, int MB> constexpr bool kLgBranch = MB == (BITS <= 4 ? 6 : 5);
template <int BITS, int MB> constexpr uint32_t kLgTileBytes = kLgTile + (kLgBranch<BITS, MB> ? 0u : 256u);
constexpr uint32_t kLgMost = 8;  // blocks of 16 activation rows

__device__ __forceinline__ void lg_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int BITS, int MB, int NB>
__global__ void __launch_bounds__(kLgBlocks / NB *kWave)
k_lanes_gemm(const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint32_t *__restrict__ exc_off,
             const uint16_t *__restrict__ scale_at, uint32_t n_cells, uint32_t n_tiles, uint32_t slices, uint32_t groups,
             const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val, uint32_t in_f, uint32_t m_all, int64_t ldx,
             uint32_t out_f, float *__restrict__ ws, bool ws_aligned, const uint16_t *__restrict__ bias, bool once,
             uint16_t *__restrict__ y, int64_t ldy) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lg_smem[];
    using P = LnPairs<BITS, false>;
    constexpr bool BRANCH = kLgBranch<BITS, MB>;
    constexpr uint32_t kTile = kLgTileBytes<BITS, MB>;
    constexpr uint32_t kThreads = kLgBlocks / NB * kWave;
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)lg_smem;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 15u, kg = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t slice = blockIdx.x % slices, group = blockIdx.x / slices % groups, row0 = blockIdx.x / slices / groups * (16u * MB);
    const uint32_t m_last = m_all - 1u;
    const uint32_t n_blocks = (n_tiles + 3u) / 4u;
    const uint32_t c0 = slice * n_cells / slices, c1 = (slice + 1u) * n_cells / slices, len = c1 - c0;
    const uint32_t b0 = group * n_blocks / groups, b1 = (group + 1u) * n_blocks / groups;
    const uint32_t rounds = (b1 - b0 + kLgBlocks - 1u) / kLgBlocks;
    const uint32_t at_once = (b1 - b0 + rounds - 1u) / rounds;  // blocks of a round (the last one may have fewer)
    const uint32_t total = rounds * len;
    const uint32_t tile_at = smem + P::kLutBytes + wave * (NB * kTile);
    // (base registers that the compiler takes as they are, the rest in the accesses' offset fields)
    uint32_t tile_lane = tile_at + lane * 16u, x_lane = smem + P::kLutBytes + kLgBlocks * kTile + lane * 16u;
    uint32_t x_to = smem + P::kLutBytes + kLgBlocks * kTile + tid * 16u;
    asm("" : "+v"(tile_lane), "+v"(x_lane), "+v"(x_to));

    // ---- activations of the 128 columns from 128 g on: 16-byte pieces in operand order ----
    constexpr uint32_t XP = (MB * 256u + kThreads - 1u) / (kThreads);
    struct Pieces { ln_u32x4 v[XP]; };
    auto x_col = [&](uint32_t e, uint32_t g) { return g * 128u + ((e >> 6) & 3u) * 32u + ((e >> 4) & 3u) * 8u; };
    auto x_load = [&](uint32_t g) {
        Pieces r;
#pragma unroll
        for (uint32_t k = 0; k < XP; ++k) {
            const uint32_t e = min(tid + k * kThreads, MB * 256u - 1u), row = min(row0 + (e >> 8) * 16u + (e & 15u), m_last);
            const uint32_t at = row * (uint32_t)ldx + min(x_col(e, g), in_f - 8u);  // (the activations lie within 4 GB)
            r.v[k] = *reinterpret_cast<const ln_u32x4 *>(reinterpret_cast<const uint8_t *>(x) + 2u * at);
        }
        return r;
    };
    auto x_store = [&](const Pieces &r, uint32_t g, uint32_t buf) {
#pragma unroll
        for (uint32_t k = 0; k < XP; ++k) {
            const uint32_t e = tid + k * kThreads;
            const ln_u32x4 v = x_col(e, g) < in_f ? r.v[k] : ln_u32x4{0, 0, 0, 0};
            if (e < MB * 256u) *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_to + buf * (MB * 4096u) + k * (kThreads * 16u))) = v;
        }
    };

    Pieces first = x_load(4u * c0);
    const float scale = bf16_bits_to_f32(*scale_at);

    if (wave * NB >= at_once) {  // no block: this wave's part of the copies only
        ln_build_lut<BITS, false>(smem, scale, tid, kThreads);
        x_store(first, 4u * c0, 0);
        lg_barrier();
        uint32_t c = c0;
        for (uint32_t u = 0; u < total; ++u) {
            const uint32_t c_next = c + 1u == c1 ? c0 : c + 1u;
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t g = q < 3 ? 4u * c + q + 1u : 4u * c_next;
                const Pieces r = x_load(g);
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
    uint32_t w[NB][2][BITS];  // two quarters of a cell ahead
    auto codes = [&](const Cell &k, uint32_t j, uint32_t q) {
        const uint32_t t = min(4u * (k.block + j) + (n >> 2), n_tiles - 1u);
        const uint8_t *const cell = reinterpret_cast<const uint8_t *>(plane) + (t * n_cells + k.c) * (256u * BITS);  // (below 2^31)
        ln_load_lane<BITS>(reinterpret_cast<const uint32_t *>(cell), 16u * q + 4u * kg + (n & 3u), w[j][q & 1u]);
    };
    // the list of row quad kg of the block in the cell: of its row n % 4 this lane has four of every sixteen quads, three times
    // (at 5 % listed elements the fullest of four rows has 31 in 512 columns, 45 are four standard deviations away)
    constexpr uint32_t ROUNDS = 3;
    struct Extent { uint32_t first, end; };
    auto extent = [&](const Cell &k, uint32_t j) {
        const uint32_t t = 4u * (k.block + j) + kg, cell = min(t, n_tiles - 1u) * n_cells + k.c;
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

    Cell now{b0 + wave * NB, c0}, next = after(now);
    Extent e_now[NB], e_next[NB];
    Quads list[NB];
#pragma unroll
    for (uint32_t j = 0; j < NB; ++j) {
        e_now[j] = extent(now, j);
#pragma unroll
        for (uint32_t q = 0; q < 2; ++q) codes(now, j, q);
    }
#pragma unroll
    for (uint32_t j = 0; j < NB; ++j) {
        list[j] = quads(e_now[j]);
        e_next[j] = extent(next, j);
    }
    ln_build_lut<BITS, false>(smem, scale, tid, kThreads);
    x_store(first, 4u * c0, 0);
    lg_barrier();
    const uint32_t lut_lane = smem + ((lane & ((1u << P::kCopies) - 1u)) << 2);

    ln_f32x4 acc[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[j][b] = ln_f32x4{0, 0, 0, 0};
    for (uint32_t u = 0; u < total; ++u) {
        // ---- listed elements: value (high half), where it goes in the tile of its quarter (bits 0..11; the tile's block i
        // is at i ^ q, as the list has it), the quarter (bits 12..14; none of the four where there is no element) ----
        // Rounds that no row has elements for are passed over where lists are short (3 bits, 5120 x 17408 Student-t at 17 / 80 / 128
        // rows 28.8 / 43.7 / 49.5 -> 27.5 / 39.7 / 47.8 us) or a wave has one block (5 bits at 5 % listed, 10240 x 5120 at 40 rows 28.5
        // -> 27.7); with two blocks of 5 bits the branches cost more (100 rows 39.9 -> 40.6), and so they do at six blocks of activation
        // rows, which spill with them (3 bits, 96 rows: 10240 x 5120 32.9 -> 34.2, 17408 x 5120 51.2 -> 53.7; 4 bits the same).
        constexpr bool SKIP = (BITS <= 4 && MB != 6) || NB == 1;
        uint32_t put[NB][4 * ROUNDS];
        // A round's stores in each quarter that any lane has elements of, without branches around them: a lane's elements of other
        // quarters go behind the tile.  (5 bits at 5 % listed, 10240 x 5120 at 17 / 64 / 100 / 128 rows 24.5 / 32.2 / 39.0 / 41.5 -> 23.6 /
        // 30.5 / 37.6 / 40.2.)  Where that takes more registers than there are, each store has a branch of its own, in every quarter.
        uint32_t in_q[NB][ROUNDS];  // bit q: the lane has elements of quarter q in the round
        bool any[NB][ROUNDS];
        bool more[NB];
#pragma unroll
        for (uint32_t j = 0; j < NB; ++j) {
#pragma unroll
            for (uint32_t r = 0; r < ROUNDS; ++r) {
                in_q[j][r] = 0;
                any[j][r] = __any((e_now[j].first & ~3u) + 16u * r < e_now[j].end);
                if (SKIP && !any[j][r]) continue;
                const uint32_t quad = mine(e_now[j]) + 16u * r;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) {
                    const uint32_t p = (k & 1) ? list[j].pos[r][k >> 1] >> 16 : list[j].pos[r][k >> 1];
                    const int v = quad + k - e_now[j].first < e_now[j].end - e_now[j].first ? (int)(list[j].val[r] << (24 - 8 * k)) >> 24 : 0;
                    put[j][4 * r + k] = (ln_pack(0.0f, (float)v * scale) & 0xFFFF0000u) | (v != 0 ? (p & 0x300u) << 4 : 0x4000u) |
                                        (((p & 0xF0u) << 4) + (p & 14u) + (kg << 6) + (n & 3u) * 16u);
                    if constexpr (!BRANCH) in_q[j][r] |= 1u << ((put[j][4 * r + k] >> 12) & 7u);
                }
            }
            more[j] = __any((e_now[j].first & ~3u) + 16u * ROUNDS < e_now[j].end);
        }
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t g_next = q < 3 ? 4u * now.c + q + 1u : 4u * next.c;
            const Pieces x_next = x_load(g_next);
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                uint32_t o[16];
                ln_decode<BITS, false, NB == 1 ? 2 : 1>(w[j][q & 1u], lut_lane, scale, o);
                codes(q < 2 ? now : next, j, q ^ 2u);
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(tile_lane + j * kTile + ((i ^ q) << 10))) =
                        ln_u32x4{o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
            }
            ln_wave_order();
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
#pragma unroll
                for (uint32_t r = 0; r < ROUNDS; ++r) {
                    if constexpr (BRANCH) {
                        if (any[j][r])
#pragma unroll
                            for (uint32_t e = 4 * r; e < 4 * r + 4; ++e)
                                if ((put[j][e] & 0x7000u) == (q << 12))
                                    *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(tile_at + j * kTile + (put[j][e] & 0xFFFu))) =
                                        (uint16_t)(put[j][e] >> 16);
                    } else if (__any(in_q[j][r] & (1u << q))) {
#pragma unroll
                        for (uint32_t e = 4 * r; e < 4 * r + 4; ++e)
                            *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(tile_at + j * kTile + min((put[j][e] ^ (q << 12)) & 0x7FFFu, kLgTile + 4u * lane))) =
                                (uint16_t)(put[j][e] >> 16);
                    }
                }
                if (more[j]) {  // rows with yet more listed elements in the cell
                    for (uint32_t f = (e_now[j].first & ~3u) + 16u * ROUNDS + (n >> 2); f < e_now[j].end; f += 4u) {
                        const uint32_t p = exc_pos[lane_listed(f, n & 3u)];
                        const int v = exc_val[lane_listed(f, n & 3u)];
                        if (v != 0 && (p & 0x300u) == (q << 8))
                            *reinterpret_cast<LN_LDS(uint16_t) *>((uintptr_t)(tile_at + j * kTile + (kg << 6) + (n & 3u) * 16u +
                                                                             ((p & 0xF0u) << 4) + (p & 14u))) =
                                (uint16_t)(ln_pack((float)v * scale, 0.0f) & 0xFFFFu);
                    }
                }
            }
            if (q == 3) {  // the list of the next cell, over the multiply
#pragma unroll
                for (uint32_t j = 0; j < NB; ++j) {
                    e_now[j] = e_next[j];
                    list[j] = quads(e_now[j]);
                    e_next[j] = extent(after(next), j);
                }
            }
            x_store(x_next, g_next, (q + 1u) & 1u);  // (its other half is in use; no wave is behind the last barrier)
            ln_wave_order();
            ln_u32x4 a[NB][4];
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j)
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i)
                    a[j][i] = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(tile_lane + j * kTile + ((i ^ q) << 10)));
// activations one step ahead, and no further: all of them at once take more registers than there are
            constexpr bool AHEAD = NB == 2;
            constexpr uint32_t STEP = !AHEAD || BITS < 5 || MB == 4 ? 4u : 2u;  // pieces of 32 columns
            ln_u32x4 v[2][STEP];
            auto x_read = [&](uint32_t step) {
#pragma unroll
                for (uint32_t i = 0; i < STEP; ++i)
                    v[step & 1u][i] = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(x_lane + (q & 1u) * (MB * 4096u) + (step * STEP + i) * 1024u));
            };
            if (AHEAD) x_read(0);
#pragma unroll
            for (uint32_t step = 0; step < MB * 4u / STEP; ++step) {
                if (!AHEAD) x_read(step);
                else if (step + 1u < MB * 4u / STEP) x_read(step + 1u);
                asm volatile("" ::: "memory");
#pragma unroll
                for (uint32_t i = 0; i < STEP; ++i)
#pragma unroll
                    for (uint32_t j = 0; j < NB; ++j) {
                        ln_f32x4 &sum = acc[j][step * STEP / 4u];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ln_bf16x8, a[j][(step * STEP + i) & 3u]),
                                                                      __builtin_bit_cast(ln_bf16x8, v[step & 1u][i]), sum, 0, 0, 0);
                    }
            }
            lg_barrier();
        }
        if (now.c + 1u == c1) {  // the slice's sums of the blocks: weight rows 4 kg .. of activation row n of each of the MB blocks
#pragma unroll
            for (uint32_t j = 0; j < NB; ++j) {
                const bool mine = wave * NB + j < at_once && now.block + j < b1;
                const uint32_t at = (now.block + j) * 16u + 4u * kg;
                uint32_t r = row0 + n;
                asm volatile("" : "+v"(r));  // addresses are worked out here and not kept in registers over the loop
#pragma unroll
                for (int b = 0; b < MB; ++b, r += 16u) {
                    if (mine && r < m_all) {
                        if (slices > 1u) {
                            float *const to = ws + ((size_t)slice * m_all + r) * (n_blocks * 16u) + at;
                            if (ws_aligned) *reinterpret_cast<ln_f32x4 *>(to) = acc[j][b];
                            else
#pragma unroll
                                for (uint32_t k = 0; k < 4; ++k) to[k] = acc[j][b][k];
                        } else {
#pragma unroll
                            for (uint32_t k = 0; k < 4; ++k) {
                                if (at + k >= out_f) continue;
                                uint32_t h = f32_to_bf16_bits(acc[j][b][k]);
                                if (bias) h = f32_to_bf16_bits((once ? acc[j][b][k] : bf16_bits_to_f32(h)) + bf16_bits_to_f32(bias[at + k]));
                                y[(int64_t)r * ldy + at + k] = (uint16_t)h;
                            }
                        }
                    }
                    acc[j][b] = ln_f32x4{0, 0, 0, 0};
                }
            }
        }
        now = next;
        next = after(now);
    }
}

// How the work is cut: groups of 16 .. 128 activation rows, slices of the columns and groups of 16-row blocks, a workgroup
// per CU. Of all such cuts the one with the shortest estimate, in clocks, from all cuts, timed, of 19 shapes from 256 x 17408 to
// 17408 x 5120 at 24 to 256 rows.  Weights of few columns or few rows, and up to 64 activation rows of more than 2^23 weights: a
// stage takes 3500 from its first request to its last product, 200 for each 16 activation rows and 60 for each block of weights that
// shares it, and the slices' sums cost a launch and their way through memory.  Elsewhere 3000 and 400 for each 16 rows, whether 3 or
// 13 blocks share the stage, unless LDS, at 128 bytes a clock, is fuller than that, and a cheaper launch of the sums.  Those figures
// slice few columns that are better taken whole by more groups of activation rows (us, with them and with the first ones: 8192 x 1024 at
// 52 / 100 / 128 rows 13.7 / 20.2 / 21.5 and 12.5 / 16.5 / 16.7, 16384 x 512 at 80 rows 15.5 and 12.9, 256 x 17408 at 128 rows 18.7
// and 15.5, 4096 x 4096 (4 bits) at 40 rows 17.7 and 14.2); the first ones take too few groups elsewhere (3072 x 3072 at 128 rows
// 19.7 and 20.4, 2048 x 7168 (3 bits) at 80 rows 18.4 and 19.6, 2048 x 2048 at 40 rows 10.3 and 10.7).
struct LgPlan { uint32_t m_groups, mb, slices, groups; };
static LgPlan lg_plan(const LanesDev &L, int m) {
    const uint32_t blocks = (L.n_tiles + 3u) / 4u, m_blocks = ((uint32_t)m + 15u) / 16u;
    const bool shared = L.n_cells <= 2u || blocks <= 64u || (m <= 64 && (uint64_t)L.n_tiles * L.n_cells > 4096u);
    LgPlan best{};
    uint64_t best_cost = ~0ull;
    for (uint32_t m_groups = (m_blocks + kLgMost - 1u) / kLgMost; m_groups <= max((m_blocks + 1u) / 2u, 1u); ++m_groups) {
        const uint32_t mb = (m_blocks + m_groups - 1u) / m_groups, cus = max(ln_cus() / m_groups, 1u);
        for (uint32_t s = 1; s <= min(L.n_cells, cus); ++s) {
            const uint32_t groups = min(max(cus / s, 1u), blocks);
            const uint32_t share = (blocks + groups - 1u) / groups, rounds = (share + kLgBlocks - 1u) / kLgBlocks;
            const uint32_t at_once = (share + rounds - 1u) / rounds, cells = (L.n_cells + s - 1u) / s;
            const uint64_t stage = shared ? 3500u + 200u * mb + 60u * at_once : max(3000u + 400u * mb, at_once * (4u * mb + 24u) * 4u);
            const uint64_t sums = s > 1 ? (shared ? 14000u : 8000u) + (uint64_t)s * (uint32_t)m * blocks * 16u * 8u / 3400u : 0u;
            const uint64_t cost = 4u * stage * rounds * cells + sums;
            if (cost < best_cost) { best_cost = cost; best = {m_groups, mb, s, groups}; }
        }
        if (m_groups * 2u > ln_cus()) break;
    }
    return best;
}

static size_t lg_bytes(const LanesDev &L, const LgPlan &p, int m) {
    return p.slices > 1 ? (size_t)p.slices * (uint32_t)m * ((L.n_tiles + 3u) / 4u * 16u) * sizeof(float) : 0;
}

size_t lanes_gemm_workspace_bytes(const LanesDev &L, int m) {
    return lanes_prompt_wins(L, m) ? lanes_prompt_workspace_bytes(L, m) : lg_bytes(L, lg_plan(L, m), m);
}

template <int BITS, int MB, int NB>
static int gemm_launch(const LanesDev &L, const LgPlan &p, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, bool once,
                       uint16_t *y, int64_t ldy, float *ws, hipStream_t s) {
    constexpr size_t lds = LnPairs<BITS, false>::kLutBytes + kLgBlocks * kLgTileBytes<BITS, MB> + 2u * MB * 4096u;
    static_assert(lds <= kLnLds, "LDS of a CU");
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_gemm<BITS, MB, NB>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    hipLaunchKernelGGL((k_lanes_gemm<BITS, MB, NB>), dim3(p.slices * p.groups * p.m_groups), dim3(kLgBlocks / NB * kWave), lds, s, L.plane, x,
                       L.exc_off, L.scale, L.n_cells, L.n_tiles, p.slices, p.groups, L.exc_pos, L.exc_val, L.in_f, (uint32_t)m, ldx,
                       L.out_f, ws, ((uintptr_t)ws & 15u) == 0, bias, once, y, ldy);
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
        case 1: return gemm_launch<BITS, 1, 1>(L, p, a...);
        case 2: return gemm_launch<BITS, 2, 1>(L, p, a...);
        case 3: return gemm_launch<BITS, 3, 1>(L, p, a...);
        case 4: return gemm_launch<BITS, 4, 2>(L, p, a...);
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
    const LgPlan p = lg_plan(L, m);
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
