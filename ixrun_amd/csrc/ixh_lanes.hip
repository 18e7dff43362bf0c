// Products of few activation rows with weights in the lane layout (ixh_lanes.h), and the kernels that write it.
#include "ixh_lanes_dev.h"

namespace ixh {

template <int BITS>
__device__ __forceinline__ void ln_load(const uint32_t *__restrict__ plane, uint32_t cell, uint32_t lane, uint32_t (&w)[BITS]) {
    ln_load_lane<BITS>(plane + (size_t)cell * (64u * BITS), lane, w);
}

template <int CTRL> __device__ __forceinline__ float ln_dpp(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}

// ---------------------------------------------------------------------------------------------------------------
// k_lanes_gemv<BITS, MT>: up to MT activation rows, MT = 1, 2 or 4.
//
// Bound: HBM and a launch's start-up (5120 x 17408, one row, copies beyond the caches: 3 bits 14.6 us for 34.6 MB, 5 bits at
// 55 / 40 / 5 % 18.7 us for 72 MB, some 4 us before the first product; the packed streams' kernels take 16.8 and 48.7; 5120 x
// 5120 8.5 and 10.7 against 11.2 and 20.1).  A workgroup owns whole row quads, so each output is made in one place (no workspace, no second
// launch).  Its cells, in memory order, are dealt to its waves in contiguous shares; a wave keeps several cells of
// loads in flight, whose addresses depend on nothing that is loaded.  The activations are copied to LDS once per
// workgroup, 16-byte pieces of a 512-column cell at piece ^ (q << 2) so that the sixteen slices of a wave read from
// different banks.  Products: v_mfma_f32_4x4x4_16b_bf16, one of its sixteen 4 x 4 blocks per slice (weight row = lane
// % 4, activation row = lane % 4), so a weight costs no product instructions of its own.
//
// Listed elements lie in cell order, so those of a share are one run of quads.  They are taken 64 quads at a time, one
// such group with every cell from the share's first on, fetched as far ahead as the cells: weight less what the plane
// has there (its sign times the scale; the difference is exact in fp32) times gathered activation, added to the lane's sum of
// the row. Taking the sign off costs two instructions an element, 17408 x 5120 at 5 % listed 17.3 us against 17.0; a plane
// without it turns an infinite activation in a listed column into NaN.
// ---------------------------------------------------------------------------------------------------------------
constexpr uint32_t kLnAhead = 4;
constexpr uint32_t kLnXAhead = 3;  // 16-byte pieces of the activations a thread asks for before anything else
constexpr uint32_t kLnXPad = 256;  // bytes behind a row of activations in LDS: zeros (whole turns of the banks)

template <int BITS, int MT>
__global__ void __launch_bounds__(1024)
k_lanes_gemv(const uint32_t *__restrict__ plane, const uint16_t *__restrict__ x, const uint32_t *__restrict__ exc_off,
             const uint16_t *__restrict__ scale_at, uint32_t n_cells, uint32_t all_tiles, uint32_t tiles_per_wg, uint32_t in_f,
             const uint16_t *__restrict__ exc_pos, const int8_t *__restrict__ exc_val, int m, int64_t ldx,
             const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, int64_t ldy, uint32_t out_f, bool x_aligned,
             uint32_t list_groups) {
    extern __shared__ __attribute__((aligned(16))) uint8_t ln_smem[];
    const uint32_t smem = (uint32_t)(uintptr_t)(LN_LDS(uint8_t) *)ln_smem;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, n_threads = blockDim.x, n_waves = n_threads >> 6;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t t0 = blockIdx.x * tiles_per_wg, C = n_cells;
    const uint32_t n_tiles = min(tiles_per_wg, all_tiles - t0);
    const uint32_t n_seq = n_tiles * C, cell0 = t0 * C;
    const uint32_t s0 = wave * n_seq / n_waves, s1 = (wave + 1) * n_seq / n_waves;
    const uint32_t x_at = smem + LnPairs<BITS>::kLutBytes, x_row = C * 1024u + kLnXPad, x_pieces = MT * C * 64u;
    float *const parts = reinterpret_cast<float *>(ln_smem + LnPairs<BITS>::kLutBytes + MT * x_row);

    auto x_piece = [&](uint32_t e) {
        const uint32_t r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
        ln_u32x4 v = {0u, 0u, 0u, 0u};
        if (r < (uint32_t)m && col < in_f) {
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

    // ---- everything that depends on nothing is asked for: activations, the first cells, the list's extent ----
    // (Requests are never inside a branch: past the end they repeat the last cell, group or piece.  The compiler counts
    // requests in flight, and one that may or may not have been made turns its counted waits into waits for all.)
    ln_u32x4 xv[kLnXAhead];
#pragma unroll
    for (uint32_t p = 0; p < kLnXAhead; ++p) {
        const uint32_t e = min(tid + p * n_threads, x_pieces - 1u), r = MT == 1 ? 0u : min(e / (C * 64u), (uint32_t)m - 1u);
        // whole pieces of an aligned row only; the others are read below
        const uint32_t col = x_aligned ? ln_piece_column((e - e / (C * 64u) * (C * 64u)) * 8u, in_f) : 0u;
        xv[p] = x_aligned ? *reinterpret_cast<const ln_u32x4 *>(x + (int64_t)r * ldx + col) : ln_u32x4{0, 0, 0, 0};
    }
    uint32_t buf[kLnAhead][BITS];
    const uint32_t cell_last = max(cell0 + s1, cell0 + 1u) - 1u;
#pragma unroll
    for (uint32_t p = 0; p < kLnAhead; ++p) ln_load<BITS>(plane, min(cell0 + s0 + p, cell_last), lane, buf[p]);
    // the list's cursor: its range is the listed elements of one row quad within one segment of exc_pos
    uint32_t l_tile = s0 / C, l_cell = s0 % C;
    auto l_extent = [&](uint32_t at) { return min(min(s1 - at, C - l_cell), kLnSegCells - l_cell % kLnSegCells); };
    uint32_t l_seq = s0, l_cells = l_extent(s0);
    uint32_t r0 = exc_off[cell0 + s0], r1 = exc_off[cell0 + s0 + l_cells];
    const uint32_t e_end = exc_off[cell0 + s1];  // behind the share's last listed element

    // ---- pair table, activations and zeroed sums to LDS ----
    const float scale = bf16_bits_to_f32(*scale_at);
    ln_build_lut<BITS, true>(smem, scale, tid, n_threads);
    for (uint32_t e = tid; e < n_tiles * n_waves * (MT * 8u); e += n_threads) parts[e] = 0.0f;
    for (uint32_t e = tid; e < MT * (kLnXPad / 16u); e += n_threads)
        *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(x_at + e / (kLnXPad / 16u) * x_row + C * 1024u + e % (kLnXPad / 16u) * 16u)) =
            ln_u32x4{0, 0, 0, 0};
    // the list's groups, one per cell from the share's first cell on
    struct Group { ln_u32x2 pos; uint32_t val; } list[kLnAhead];
    const LnGroups groups = ln_groups(r0, e_end, list_groups);
    const uint32_t g_first = groups.first, n_groups = groups.n;
    auto g_load = [&](uint32_t i) {
        const uint32_t g = min(g_first + i, groups.last);
        return Group{*reinterpret_cast<const ln_u32x2 *>(exc_pos + (size_t)g * 256u + lane * 4u),
                     *reinterpret_cast<const uint32_t *>(exc_val + (size_t)g * 256u + lane * 4u)};
    };
#pragma unroll
    for (uint32_t p = 0; p < kLnAhead; ++p) list[p] = g_load(p);
#pragma unroll
    for (uint32_t p = 0; p < kLnXAhead; ++p) {
        const uint32_t e = tid + p * n_threads, r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
        if (e < x_pieces && x_aligned && r < (uint32_t)m && col + 8u <= in_f) x_store(e, xv[p]);
    }
    for (uint32_t e = tid; e < x_pieces; e += n_threads) {  // what is not stored yet
        const uint32_t r = MT == 1 ? 0u : e / (C * 64u), col = (e - r * (C * 64u)) * 8u;
        if (e >= kLnXAhead * n_threads || !x_aligned || r >= (uint32_t)m || col + 8u > in_f) x_store(e, x_piece(e));
    }
    __syncthreads();

    const uint32_t lut_lane = smem + ((lane & ((1u << LnPairs<BITS>::kCopies) - 1u)) << 2);
    const uint32_t q = lane >> 4, kg = (lane >> 2) & 3u, am = min(lane & 3u, (uint32_t)MT - 1u);
    uint32_t xa[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) xa[i] = x_at + am * x_row + q * 256u + ((i ^ q) << 6) + kg * 16u;

    ln_f32x4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};

    float ex[MT][4];
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
        for (int k = 0; k < 4; ++k) ex[r][k] = 0.0f;
    // sums over the lanes of a row's products, to `parts`: lane l has row l % 4
    auto put = [&](uint32_t tile, uint32_t half, int r, float v) {
        v += ln_dpp<0x124>(v);
        v += ln_dpp<0x128>(v);
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (lane < 4) parts[((tile * n_waves + wave) * 2u + half) * (MT * 4u) + (uint32_t)r * 4u + lane] = v;
    };
    const uint32_t none = lane_none(C) * 0x10001u, scale_bits = __float_as_uint(scale) & 0x7FFFFFFFu;
    // one group of listed elements, range by range
    auto list_group = [&](const Group &in, uint32_t i) {
        const uint32_t g0 = (g_first + i) << 6, quad = g0 + lane;
        for (;;) {
            uint32_t vals = in.val, p01 = in.pos[0], p23 = in.pos[1];
            if (g0 < r0 || g0 + 64u > r1) {  // quads outside the range count as if they held no element
                const bool in_range = quad >= r0 && quad < r1;
                vals = in_range ? vals : 0u;
                p01 = in_range ? p01 : none;
                p23 = in_range ? p23 : none;
            }
            const uint32_t x_seg = x_at + (l_cell / kLnSegCells) * (kLnSegCells * 1024u);
            uint32_t at[4] = {x_seg + (p01 & 0xFFFFu), x_seg + (p01 >> 16), x_seg + (p23 & 0xFFFFu), x_seg + (p23 >> 16)};
            if (C >= kLnSegCells)
#pragma unroll
                for (int k = 0; k < 4; ++k) at[k] = (vals >> (8 * k)) & 255u ? at[k] : x_at + C * 1024u;
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
                    ex[r][k] = __fmaf_rn(wv, __uint_as_float(h << 16), ex[r][k]);
                }
            }
            if (g0 + 64u < r1) break;  // the range goes on in the next group
            l_seq += l_cells;
            l_cell += l_cells;
            if (l_cell == C || l_seq == s1) {  // the row quad is complete
#pragma unroll
                for (int r = 0; r < MT; ++r) {
                    // every lane gets the sum of row lane % 4 over its quad of lanes
                    float own = 0.0f;
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) {
                        float v = ex[r][k];
                        v += ln_dpp<0xB1>(v);
                        v += ln_dpp<0x4E>(v);
                        own = (lane & 3u) == k ? v : own;
                        ex[r][k] = 0.0f;
                    }
                    put(l_tile, 1u, r, own);
                }
                l_cell = 0;
                ++l_tile;
            }
            if (l_seq == s1) break;
            l_cells = l_extent(l_seq);
            r0 = r1;
            r1 = exc_off[cell0 + l_seq + l_cells];
            if (r0 >= g0 + 64u) break;
        }
    };

    uint32_t c = s0 % C, tile = s0 / C;
    for (uint32_t s = s0; s < s1; s += kLnAhead) {
        // Left alone, the waves of a SIMD are served oldest first and the last one ends long after the first; a wave
        // that has more cells to go takes precedence.
        const uint32_t behind = (s1 - s) * 4u / (s1 - s0 + 1u);
        if (behind >= 3u) __builtin_amdgcn_s_setprio(3);
        else if (behind == 2u) __builtin_amdgcn_s_setprio(2);
        else if (behind == 1u) __builtin_amdgcn_s_setprio(1);
        else __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (uint32_t p = 0; p < kLnAhead; ++p) {
            if (s + p >= s1) break;
            uint32_t o[16];
            ln_decode<BITS, true>(buf[p], lut_lane, scale, o);
            ln_load<BITS>(plane, min(cell0 + s + p + kLnAhead, cell_last), lane, buf[p]);
            const uint32_t x_c = c * 1024u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const ln_u32x4 a = *reinterpret_cast<const LN_LDS(ln_u32x4) *>((uintptr_t)(xa[i] + x_c));
                acc0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(ln_s16x4, ln_u32x2{a[0], a[1]}),
                                                             __builtin_bit_cast(ln_s16x4, ln_u32x2{o[4 * i], o[4 * i + 1]}), acc0, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(ln_s16x4, ln_u32x2{a[2], a[3]}),
                                                             __builtin_bit_cast(ln_s16x4, ln_u32x2{o[4 * i + 2], o[4 * i + 3]}), acc1, 0, 0, 0);
            }
            if (s + p - s0 < n_groups) list_group(list[p], s + p - s0);
            list[p] = g_load(s + p - s0 + kLnAhead);
            ++c;
            if (c == C || s + p + 1 == s1) {
#pragma unroll
                for (int r = 0; r < MT; ++r) put(tile, 0u, r, acc0[r] + acc1[r]);
                acc0 = ln_f32x4{0, 0, 0, 0};
                acc1 = ln_f32x4{0, 0, 0, 0};
                c = 0;
                ++tile;
            }
        }
    }
    // a list of more groups than cells
    for (uint32_t i = s1 - s0; i < n_groups; ++i) list_group(g_load(i), i);
    __syncthreads();

    // ---- outputs: the waves' parts in wave order ----
    for (uint32_t e = tid; e < n_tiles * 4u * (uint32_t)m; e += n_threads) {
        const uint32_t r = e / (n_tiles * 4u), row = e - r * (n_tiles * 4u), at = t0 * 4u + row;
        if (at >= out_f) continue;
        float sum = 0.0f;
        for (uint32_t w = 0; w < 2u * n_waves; ++w) sum += parts[((row >> 2) * n_waves * 2u + w) * (MT * 4u) + r * 4u + (row & 3u)];
        uint32_t b = f32_to_bf16_bits(sum);
        if (bias) b = f32_to_bf16_bits(bf16_bits_to_f32(b) + bf16_bits_to_f32(bias[at]));
        y[(int64_t)r * ldy + at] = (uint16_t)b;
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
    hipLaunchKernelGGL(k_lanes_reduce, dim3((out_f + 255u) / 256u, m), dim3(256), 0, s, ws, slices, m, out_f, ws_ld, bias, once,
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
            pos[4u * at + (lane & 3u)] = (uint16_t)lane_offset(col0 + 32u * (e >> 3) + (e & 7u));
            val[4u * at + (lane & 3u)] = (int8_t)v[e];
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

// (fewer rows than five where those of whole rows do not fit k_lanes_gemv go to k_lanes_gemm as well)
template <int BITS, int MT>
static int lanes_gemv_launch(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                             int64_t ldy, hipStream_t s) {
    // Workgroups of 16, 8 or 4 waves, one, two or four to a CU: the split whose last round of row quads is fullest.
    const size_t fixed = LnPairs<BITS>::kLutBytes + (size_t)MT * (L.n_cells * 1024u + kLnXPad);
    auto lds_of = [&](uint32_t tiles, uint32_t waves) { return fixed + (size_t)tiles * waves * (MT * 32u); };
    uint32_t best_waves = 0, best_tiles = 0;
    uint64_t best_cost = ~0ull;
    for (uint32_t per_cu = 1; per_cu <= 4; per_cu *= 2) {
        const uint32_t waves = 16u / per_cu, slots = ln_cus() * per_cu;
        const uint32_t tiles = (L.n_tiles + slots - 1) / slots;
        if (lds_of(tiles, waves) * per_cu > kLnLds) break;
        const uint64_t cost = (uint64_t)tiles * per_cu;  // row quads a CU works through
        if (cost < best_cost) { best_cost = cost; best_waves = waves; best_tiles = tiles; }
    }
    if (!best_waves) return IXH_EUNSUPPORTED;
    const uint32_t waves = min(best_waves, best_tiles * L.n_cells);
    static const bool raised = hipFuncSetAttribute(reinterpret_cast<const void *>(k_lanes_gemv<BITS, MT>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLnLds) == hipSuccess;
    if (!raised) return IXH_ELAUNCH;
    const bool aligned = ln_whole_pieces((uintptr_t)x, L.in_f, m, ldx);
    hipLaunchKernelGGL((k_lanes_gemv<BITS, MT>), dim3((L.n_tiles + best_tiles - 1) / best_tiles), dim3(kWave * waves),
                       lds_of(best_tiles, waves), s, L.plane, x, L.exc_off, L.scale, L.n_cells, L.n_tiles, best_tiles, L.in_f,
                       L.exc_pos, L.exc_val, m, ldx, bias, y, ldy, L.out_f, aligned, L.list_groups);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

template <int BITS>
static int lanes_gemv_rows(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                           int64_t ldy, float *ws, hipStream_t s) {
    int rc = IXH_EUNSUPPORTED;
    if (m == 1) rc = lanes_gemv_launch<BITS, 1>(L, x, m, ldx, bias, y, ldy, s);
    else if (m == 2) rc = lanes_gemv_launch<BITS, 2>(L, x, m, ldx, bias, y, ldy, s);
    else if (m <= 4) rc = lanes_gemv_launch<BITS, 4>(L, x, m, ldx, bias, y, ldy, s);
    return rc == IXH_EUNSUPPORTED ? launch_lanes_gemm(L, x, m, ldx, bias, false, y, ldy, ws, s) : rc;
}

int launch_lanes_gemv(const LanesDev &L, const uint16_t *x, int m, int64_t ldx, const uint16_t *bias, uint16_t *y,
                      int64_t ldy, float *ws, hipStream_t s) {
    switch (L.bits) {
        case 3: return lanes_gemv_rows<3>(L, x, m, ldx, bias, y, ldy, ws, s);
        case 4: return lanes_gemv_rows<4>(L, x, m, ldx, bias, y, ldy, ws, s);
        case 5: return lanes_gemv_rows<5>(L, x, m, ldx, bias, y, ldy, ws, s);
        default: return lanes_gemv_rows<8>(L, x, m, ldx, bias, y, ldy, ws, s);
    }
}

}  // namespace ixh
