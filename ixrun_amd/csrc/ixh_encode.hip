// The INT8-X encoder on the device: bf16 weights -> scale, rank table, nested bitmaps and code streams,
// byte for byte what the reference's CPU writer produces (ixrun/quantize.py:41-122 with the bit packing of
// ixrun/bitpack.py:13-61, :87-89).  Three passes over the weights, all bound by HBM reads:
//   1. k_enc_absmax      largest magnitude, one partial result per workgroup (no atomics, nothing to clear)
//   2. k_enc_count<L>    the bf16 scale from the partial results, and the elements of every level per 512-element unit;
//                        k_enc_scan sums the counts into the rank table, which is the table the decoders take
//   3. k_enc_pack<L>     quantise again and pack; the table says at which bit of every stream a wave's elements
//                        start.  Only the words that two waves share are cleared (k_enc_borders) and OR-ed in
// Between passes 2 and 3 the caller reads the level totals (last table entries) and sizes the streams.
#include "ixh_dev.h"

namespace ixh {

constexpr uint32_t kEncUnit = 512;          // elements per wave and step: eight per lane
constexpr int kEncWaves = 4;                // waves per workgroup
constexpr uint32_t kEncParts = 256;         // partial maxima of pass 1 (one per workgroup of 1024 lanes)
constexpr uint32_t kScanTile = 4096;        // table entries per workgroup of the scan
constexpr int kEncAhead = 4;                // loads in flight per lane of pass 1

__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off));
    return v;
}

// scale = bf16( max(|w|max, bf16(1e-8)) / 127 ), the bf16 arithmetic of quantize.py:64 (the quotient is formed
// in fp32 and rounded once)
__device__ __forceinline__ uint32_t scale_bits_from_parts(const uint32_t *__restrict__ parts, uint32_t lane) {
    uint32_t m = 0;
    for (uint32_t i = lane; i < kEncParts; i += kWave) m = max(m, parts[i]);
    m = wave_max(m);
    const float floor_ = bf16_bits_to_f32(f32_to_bf16_bits(1e-8f));
    const float amax = fmaxf(bf16_bits_to_f32(m), floor_);
    return f32_to_bf16_bits(__fdiv_rn(amax, 127.0f));
}

// int8 of one weight: round-half-even of the fp32 quotient, clamped (quantize.py:65-70), without the division.
// Weight and scale are bf16 values (8-bit significands), so the exact quotient is either a tie k + 1/2 itself or at
// least 2^-9 away from every tie, and the fp32 rounding of the quotient cannot move it across one: the reference's
// round(fl(w / s)) equals round-half-even of the exact quotient.  w * (1/s) is within 2.5e-5 of that quotient (|q| <=
// 127.25); adding and subtracting 3072 snaps it to a multiple of 2^-12, which puts exact ties back on k + 1/2 and
// leaves everything else on its side.  Checked against the division for every bf16 weight and scale significand.
__device__ __forceinline__ float quantise(float w, float inv_scale) {
    const float snapped = __fmaf_rn(w, inv_scale, 3072.0f) - 3072.0f;
    return __builtin_amdgcn_fmed3f(rintf(snapped), -127.0f, 127.0f);
}

struct EncLevels {
    int n_levels;
    int bits[IXH_MAX_LEVELS];
};

// Elements p and p + 1, `fill` for one at or past n.  The loads are unconditional, so that they do not wait for one another.
__device__ __forceinline__ uint32_t pair_or(const uint16_t *__restrict__ w, uint64_t p, uint32_t n, uint32_t fill) {
    const uint32_t a = w[min(p, (uint64_t)n - 1)], b = w[min(p + 1, (uint64_t)n - 1)];
    return (p < n ? a : fill) | (p + 1 < n ? b : fill) << 16;
}

// Pairs of weights from element p on, eight in all; zero past n.  kWhole: all eight are there, at a multiple of 16 bytes.
template <bool kWhole>
__device__ __forceinline__ uint4 load8(const uint16_t *__restrict__ w, uint64_t p, uint32_t n) {
    if (kWhole) return *reinterpret_cast<const uint4 *>(w + p);
    return make_uint4(pair_or(w, p, n, 0u), pair_or(w, p + 2, n, 0u), pair_or(w, p + 4, n, 0u), pair_or(w, p + 6, n, 0u));
}

// The smallest magnitude, as bf16 bits, that quantises above the threshold of a level of `bits`: every wave finds it by quantising the
// 64 bf16 values around (threshold + 1/2) * scale.  (All of them above: a scale that is not a number, where every weight is.)
__device__ __forceinline__ uint32_t enc_cut(int bits, float scale, float inv_scale, uint32_t lane) {
    const float thr = (float)threshold_of(bits);
    const int around = (int)(__float_as_uint((thr + 0.5f) * scale) >> 16) - 32;
    const int mag = min(max(around + (int)lane, 0), 0x7fff);
    const uint64_t above = __ballot(fabsf(quantise(bf16_bits_to_f32((uint32_t)mag), inv_scale)) > thr);
    return above == ~0ull ? 0u : (uint32_t)min(max(around + (int)__builtin_ctzll(above | 1ull << 63), 0), 0x7fff);
}

// Bound by HBM (a read of 178 MB: 37 us, 4.8 TB/s; more loads in flight or more workgroups change nothing); what is left
// of a small weight's passes without loads in flight is 16 bytes a lane too (by single weights: 2^20 of them 4.3 -> 2.4 us).
__global__ void __launch_bounds__(1024) k_enc_absmax(const uint16_t *__restrict__ w, uint32_t n, uint32_t *parts) {
    const bool aligned = (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
    typedef uint16_t half2 __attribute__((ext_vector_type(2)));
    half2 m = {0, 0};
    auto take = [&](const uint4 &q) {
        const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) m = __builtin_elementwise_max(m, __builtin_bit_cast(half2, d[t] & 0x7fff7fffu));
    };
    const uint64_t stride = (uint64_t)gridDim.x * 1024u * 8u;
    uint64_t base = (uint64_t)blockIdx.x * 1024u * 8u;
    const uint32_t mine = threadIdx.x * 8u;
    for (; aligned && base + (kEncAhead - 1) * stride + 1024u * 8u <= n; base += kEncAhead * stride) {
        uint4 q[kEncAhead];
#pragma unroll
        for (int k = 0; k < kEncAhead; ++k) q[k] = load8<true>(w, base + k * stride + mine, n);
#pragma unroll
        for (int k = 0; k < kEncAhead; ++k) take(q[k]);
    }
    for (; aligned && base + 1024u * 8u <= n; base += stride) take(load8<true>(w, base + mine, n));
    for (; base < n; base += stride) take(load8<false>(w, base + mine, n));
    __shared__ uint32_t wave_m[16];
    uint32_t top = wave_max(max((uint32_t)m.x, (uint32_t)m.y));
    if ((threadIdx.x & 63) == 0) wave_m[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x < 16) {
        top = wave_m[threadIdx.x];
        for (int off = 8; off > 0; off >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, off));
        if (threadIdx.x == 0) parts[blockIdx.x] = top;
    }
}

// table[i * entries + u + 1] = number of level-i elements of unit u (raw counts; the scan turns them into ranks), and
// sums[i * groups + g] = that of a workgroup's kCountUnits units.
//
// Magnitudes order like their bf16 bits, so "|int8| above a level's threshold" is one comparison of 15-bit numbers, with a
// cutoff that every wave finds by quantising the 64 bf16 values around (threshold + 1/2) * scale: the very arithmetic of
// the pack.  (A level is "the thresholds below |v|", quantize.py:25-37: counting what is above each and taking
// differences gives the levels.)  Two weights to a subtraction; a row of 16 lanes takes a unit, so that four DPP steps sum
// four units.  Bound by its read, which the last-level cache serves in part: 5120 x 17408 in 28 us, 6.3 TB/s (35 when
// every weight was quantised in fp32).
constexpr uint32_t kCountUnits = 64;
// Weights of no more units than make two such workgroups a CU have workgroups of 16, a turn a wave, which are over in one trip to memory (a
// whole call, 64 / 16 units: 2048 x 2500 42.4 / 35.8 us, 3000 x 3000 47.2 / 40.8, 4096 x 4096 50.0 / 48.2, 4096 x 8192 68.7 / 73.2).
constexpr uint32_t kCountFewUnits = 16, kCountFew = 32768;

template <int L, bool kWhole, uint32_t UNITS>
__device__ __forceinline__ void
count_units(const uint16_t *__restrict__ w, uint32_t n, uint32_t n_units, const uint32_t *__restrict__ parts,
            const EncLevels &lv, int32_t *table, uint32_t *sums, uint16_t *scale_out) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t u_first = blockIdx.x * UNITS + wave * (UNITS / kEncWaves);
    constexpr int kTurns = UNITS / kEncWaves / 4;
    auto place = [&](int turn, int k) {
        return (uint64_t)(u_first + 4 * turn + (lane >> 4)) * kEncUnit + (lane & 15u) * 8u + 128u * k;
    };
    uint4 q[4];
    if (kWhole) {
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = load8<true>(w, place(0, k), n);
    }
    const uint32_t sbits = scale_bits_from_parts(parts, lane);
    if (blockIdx.x == 0 && threadIdx.x == 0) *scale_out = (uint16_t)sbits;
    const float scale = bf16_bits_to_f32(sbits), inv_scale = __fdiv_rn(1.0f, scale);
    uint32_t cut[L - 1];  // in both halves: the smallest magnitude above the level's threshold
#pragma unroll
    for (int i = 0; i < L - 1; ++i) {
        cut[i] = enc_cut(lv.bits[i], scale, inv_scale, lane) * 0x10001u;
    }
    const uint32_t entries = n_units + 1;
    uint32_t total[L - 1] = {};
#pragma unroll(kWhole ? kTurns : 1)
    for (int turn = 0; turn < kTurns; ++turn) {
        uint4 ahead[4];
        if (kWhole && turn + 1 < kTurns) {
#pragma unroll
            for (int k = 0; k < 4; ++k) ahead[k] = load8<true>(w, place(turn + 1, k), n);
        }
        uint32_t above[L - 1] = {};
#pragma unroll(kWhole ? 4 : 1)
        for (int k = 0; k < 4; ++k) {
            const uint4 c = kWhole ? q[k] : load8<false>(w, place(turn, k), n);
            const uint32_t d[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < L - 1; ++i) above[i] += __popc(((d[t] | 0x80008000u) - cut[i]) & 0x80008000u);
        }
        // sums over the row's lanes, 10-bit fields, three to a word: at most 512 of anything
        uint32_t acc[(L + 1) / 3] = {};
#pragma unroll
        for (int i = 0; i < L - 1; ++i) acc[i / 3] |= above[i] << (10 * (i % 3));
#pragma unroll
        for (int j = 0; j < (L + 1) / 3; ++j) acc[j] = row_scan_inclusive(acc[j]);
        const uint32_t u = u_first + 4 * turn + (lane >> 4);
        if ((lane & 15u) == 15u && u < n_units) {
            uint32_t prev = min(kEncUnit, n - u * kEncUnit);
#pragma unroll
            for (int i = 0; i < L - 1; ++i) {
                const uint32_t ab = min((acc[i / 3] >> (10 * (i % 3))) & 1023u, prev);
                table[(size_t)i * entries + u + 1] = (int32_t)(prev - ab);
                total[i] += prev - ab;
                prev = ab;
            }
        }
        if (kWhole) {
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = ahead[k];
        }
    }
    __shared__ uint32_t wave_t[kEncWaves][L - 1];
#pragma unroll
    for (int i = 0; i < L - 1; ++i) {
        const uint32_t t = wave_scan_inclusive(total[i]);
        if (lane == 63) wave_t[wave][i] = t;
    }
    __syncthreads();
    if (threadIdx.x < L - 1) {
        uint32_t t = 0;
#pragma unroll
        for (int k = 0; k < kEncWaves; ++k) t += wave_t[k][threadIdx.x];
        sums[threadIdx.x * gridDim.x + blockIdx.x] = t;
    }
}

template <int L, uint32_t UNITS>
__global__ void __launch_bounds__(kWave *kEncWaves)
k_enc_count(const uint16_t *__restrict__ w, uint32_t n, uint32_t n_units, const uint32_t *__restrict__ parts,
            EncLevels lv, int32_t *table, uint32_t *sums, uint16_t *scale_out) {
    const bool aligned = (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
    if (aligned && (uint64_t)(blockIdx.x + 1) * UNITS * kEncUnit <= n)
        count_units<L, true, UNITS>(w, n, n_units, parts, lv, table, sums, scale_out);
    else
        count_units<L, false, UNITS>(w, n, n_units, parts, lv, table, sums, scale_out);
}

// In place, per row: row[0] = 0, row[u + 1] = counts of units 0 .. u.  Each thread takes four consecutive entries; what
// the workgroups of k_enc_count in front of the tile counted comes first.  6 us, all of it latency (tiles twice as large,
// eight entries a thread, and sums from a kernel of their own: 14).
struct __attribute__((packed, aligned(4))) Int4 { int32_t v[4]; };
__global__ void __launch_bounds__(1024)
k_enc_scan(int32_t *table, uint32_t n_units, const uint32_t *__restrict__ sums, uint32_t groups, uint32_t group_units, int64_t *host_totals) {
    int32_t *row = table + (size_t)blockIdx.y * (n_units + 1);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ uint32_t wave_s[16], wave_c[16];
    const uint32_t first = blockIdx.x * kScanTile + tid * 4u;
    uint32_t v[4];
    if (first + 4 <= n_units) {
        const Int4 q = *reinterpret_cast<const Int4 *>(row + first + 1);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = (uint32_t)q.v[t];
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = first + t < n_units ? (uint32_t)row[first + t + 1] : 0u;
    }
    uint32_t c = 0;
    const uint32_t *row_sums = sums + (size_t)blockIdx.y * groups;
    for (uint32_t g = tid; g < blockIdx.x * (kScanTile / group_units); g += 1024) c += row_sums[g];
    c = wave_scan_inclusive(c);
    if (lane == 63) wave_c[wave] = c;
    const uint32_t mine = v[0] + v[1] + v[2] + v[3];
    const uint32_t incl = wave_scan_inclusive(mine);
    if (lane == 63) wave_s[wave] = incl;
    __syncthreads();
    uint32_t run = incl - mine;
    for (uint32_t k = 0; k < 16; ++k) run += wave_c[k] + (k < wave ? wave_s[k] : 0u);
    Int4 q;
#pragma unroll
    for (int t = 0; t < 4; ++t) q.v[t] = (int32_t)(run += v[t]);
    if (first + 4 <= n_units) {
        *reinterpret_cast<Int4 *>(row + first + 1) = q;
    } else {
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (first + t < n_units) row[first + t + 1] = q.v[t];
    }
    if (blockIdx.x == 0 && tid == 0) row[0] = 0;
    if (host_totals && blockIdx.x + 1 == gridDim.x && tid == 1023)
        __hip_atomic_store(host_totals + blockIdx.y, (int64_t)run, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Destination of the encoder: the same fields as Dev, writable.
struct EncOut {
    uint32_t *bm[IXH_MAX_LEVELS - 1];
    uint32_t bm_words[IXH_MAX_LEVELS - 1];
    uint32_t *st[IXH_MAX_LEVELS - 1];
    uint32_t st_words[IXH_MAX_LEVELS - 1];
    uint8_t *last;
    uint32_t last_bytes;
};

// LDS traffic of this wave so far is visible to all its lanes after this
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------------------------------------------
// k_enc_pack<L>: bound by vector issue; 5120 x 17408 at 55 / 40 / 5 % and levels 3, 5, 8: 789 vector instructions a wave and span, 71 us;
// 695 and 66 since a level's cutoff is compared with the weights as they are, codes are packed by dot products and a group leaves in one store;
// 62 since two elements at a time are put in their runs.  The launch, first loads and the write-back of the caches are some ten of it, and the
// 240 MB that it moves take 47.
//
// A wave takes spans of four units, 2048 elements, 32 consecutive ones a lane, so one prefix sum over the lanes serves them
// all and a lane's membership bits are a whole word of bitmap 0.  Every element goes to LDS as one byte, value + 128: those
// of the level to the dense run, the others to what waits for the next level, in order; that level splits its run the same
// way, 16 bytes a lane.  A dense run starts in LDS where its first code falls in the stream's groups of 32 codes, so a
// lane turns 32 bytes into `bits` whole words of the stream at once.  Only the groups (and bitmap words) that a wave
// shares with its neighbours are OR-ed into memory; k_enc_borders clears those beforehand.
// (Before, a wave packed 512 elements with an LDS atomic per code and a flush per stream: 279 us.)
// ---------------------------------------------------------------------------------------------------------------
constexpr uint32_t kEncSpan = 2048, kEncSpanUnits = kEncSpan / kEncUnit;
constexpr uint32_t kEncBuf = kEncSpan + 256;  // a dense run, and one behind it, with their margins
constexpr uint32_t kEncHeld = kEncSpan + 96;  // what waits for its level, with its margins
// A level's turn (a scan, comparisons, a store) takes as long for 100 elements as for 1024.  From four levels on what is not of the first waits in
// LDS for the second level, and so on to the last but one, a run a level, over the spans of a wave until what comes next would not fit: of levels 3,
// 4, 5, 6, 8 at 55 / 13 / 27 / 0.7 / 4 % a span leaves 920 elements to the second, 660 to the third, 96 to the fourth, so that these have their turns every other
// span, every third and once in twenty (5120 x 17408, whole calls: 196 -> 177 us, the launch 108 -> 86; Student-t weights, nearly all in the first, 165 -> 141;
// four levels 167 -> 161 and 150 -> 132, seven 269 -> 252 and 207 -> 163).  Three levels are bound by memory as much as by issue (139 -> 143
// and 133 -> 137): there the second has its turn each span.  Eight would leave two waves a SIMD room in LDS (315 -> 354).
template <int L> constexpr bool kEncHold = L > 3 && L < 8;
constexpr uint32_t dense_at = 32u;            // where a dense run's groups start in it

// Spans per wave: a wave that goes on hands its unfinished groups to its next span in registers, and only its first and last
// cost atomics (one span each: 107 .. 175 us instead of 70 .. 75).  The spans are dealt out evenly to as many waves as run at the
// same time (three levels, 89 registers: five on each of a CU's four SIMDs), so that no CU is left with a workgroup more than another: 5120 x 17408
// at 55 / 40 / 5 % 71.8 us, 76.7 with eight spans each (5.3 workgroups a CU), 74.4 with four waves a SIMD, 80.2 with six (a second
// round); at five levels (four waves a SIMD) 145.1 -> 130.2.
struct EncShare {
    uint32_t waves, spans, more;  // the first `more` waves have a span more than the others
    __device__ __forceinline__ uint32_t first_unit(uint32_t wave, uint32_t n_units) const {
        return min((wave * spans + min(wave, more)) * kEncSpanUnits, n_units);
    }
};

// level i's rank at unit `u`, and the index of the unit's first element in bitmap i
struct EncRanks {
    const int32_t *table;
    uint32_t entries, n;
    __device__ __forceinline__ uint32_t rank(int i, uint32_t u) const { return (uint32_t)table[(size_t)i * entries + u]; }
    __device__ __forceinline__ uint32_t space(int i, uint32_t u) const {
        uint32_t at = min(u * kEncUnit, n);
        for (int j = 0; j < i; ++j) at -= rank(j, u);
        return at;
    }
};

// clears what neighbouring waves share: of every stream the group of 32 codes that a wave's first code falls into,
// of every bitmap but the first the word of its first bit; and any words behind the last code
// (5.8 us with the ranks asked for level by level, 5.1 with all of them first, 5120 x 17408: a launch and their latency.)
template <int L>
__global__ void __launch_bounds__(256)
k_enc_borders(EncLevels lv, const int32_t *__restrict__ table, uint32_t n, uint32_t n_units, EncShare share, EncOut out) {
    const uint32_t s = blockIdx.x * 256u + threadIdx.x, u = share.first_unit(min(s, share.waves), n_units);
    const EncRanks r{table, n_units + 1, n};
    uint32_t all[L - 1], here[L - 1];
#pragma unroll
    for (int i = 0; i < L - 1; ++i) {
        all[i] = r.rank(i, n_units);
        here[i] = r.rank(i, u);
    }
    uint32_t bits = n, at = min(u * kEncUnit, n);  // of bitmap i in all, and those in front of the unit
#pragma unroll
    for (int i = 0; i < L - 1; ++i) {
        for (uint32_t k = (bits + 31u) / 32u + s; k < out.bm_words[i]; k += gridDim.x * 256u) out.bm[i][k] = 0u;
        const uint32_t b = (uint32_t)lv.bits[i];
        const uint64_t used = ((uint64_t)all[i] * b + 31u) / 32u;
        for (uint64_t k = used + s; k < out.st_words[i]; k += gridDim.x * 256u) out.st[i][k] = 0u;
        if (s <= share.waves) {
            const uint32_t word = (here[i] >> 5) * b;
            for (uint32_t k = 0; k < b; ++k)
                if (word + k < out.st_words[i]) out.st[i][word + k] = 0u;
            if (i > 0 && (at >> 5) < out.bm_words[i]) out.bm[i][at >> 5] = 0u;
        }
        bits -= all[i];
        at -= here[i];
    }
}

// Four codes (bytes, `bias` too high) to 4 B bits.  Dot products of the bytes with powers of two put as many codes side by side as a
// factor of a byte can move, and the bias comes off in what they start from (for three bits the last code is shifted there).
template <int B>
__device__ __forceinline__ uint32_t enc_four(uint32_t x, uint32_t bias) {
    constexpr uint32_t k1 = 1u << B, k2 = 1u << (2 * B), k3 = 1u << (3 * B);
    if constexpr (B <= 2) return __builtin_amdgcn_udot4(x, 1u | k1 << 8 | k2 << 16 | k3 << 24, 0u - bias * (1u + k1 + k2 + k3), false);
    if constexpr (B == 3) return __builtin_amdgcn_udot4(x, 1u | k1 << 8 | k2 << 16, ((x >> 24) << 9) - bias * (1u + k1 + k2 + k3), false);
    const uint32_t low = __builtin_amdgcn_udot4(x, 1u | k1 << 8, 0u - bias * (1u + k1), false);
    return (__builtin_amdgcn_udot4(x, (1u | k1 << 8) << 16, 0u - bias * (1u + k1), false) << (2 * B)) | low;
}
// 32 codes to B words
template <int B>
__device__ __forceinline__ void enc_words(const uint32_t (&x)[8], uint32_t bias, uint32_t (&w)[B]) {
#pragma unroll
    for (int k = 0; k < B; ++k) w[k] = 0u;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint32_t four = enc_four<B>(x[c], bias);
        const int bit = 4 * B * c, d = bit >> 5, sh = bit & 31;
        w[d] |= four << sh;
        if (sh + 4 * B > 32) w[d + 1] |= four >> (32 - sh);
    }
}

// `groups` groups of 32 codes (bytes in LDS at `run`) to the stream from group g0 on; `first` and `last` are the groups
// that the wave shares with its neighbours
template <int B>
__device__ __forceinline__ void enc_store_run(const uint8_t *run, uint32_t g0, uint32_t groups, uint32_t first, uint32_t last,
                                              uint32_t *dst, uint32_t dst_words, uint32_t lane) {
    constexpr uint32_t bias = 128u - ((1u << (B - 1)) - 1u);
    const bool inside = g0 > first && g0 + groups <= last && (g0 + groups) * B <= dst_words;
    for (uint32_t g = lane; g < groups; g += kWave) {
        const uint4 lo = *reinterpret_cast<const uint4 *>(run + g * 32u), hi = *reinterpret_cast<const uint4 *>(run + g * 32u + 16u);
        const uint32_t x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        uint32_t w[B];
        enc_words<B>(x, bias, w);
        const uint32_t at = (g0 + g) * B;
        if (inside) {
            struct __attribute__((packed, aligned(4))) Words { uint32_t v[B]; } all;
#pragma unroll
            for (int k = 0; k < B; ++k) all.v[k] = w[k];
            *reinterpret_cast<Words *>(dst + at) = all;
        } else if (g0 + g == first || g0 + g == last) {
#pragma unroll
            for (int k = 0; k < B; ++k)
                if (at + k < dst_words && w[k]) atomicOr(&dst[at + k], w[k]);
        } else {
#pragma unroll
            for (int k = 0; k < B; ++k)
                if (at + k < dst_words) dst[at + k] = w[k];
        }
    }
}
__device__ __forceinline__ void enc_store_run_of(uint32_t b, const uint8_t *run, uint32_t g0, uint32_t groups, uint32_t first,
                                                 uint32_t last, uint32_t *dst, uint32_t dst_words, uint32_t lane) {
    switch (b) {  // uniform
        case 1: enc_store_run<1>(run, g0, groups, first, last, dst, dst_words, lane); break;
        case 2: enc_store_run<2>(run, g0, groups, first, last, dst, dst_words, lane); break;
        case 3: enc_store_run<3>(run, g0, groups, first, last, dst, dst_words, lane); break;
        case 4: enc_store_run<4>(run, g0, groups, first, last, dst, dst_words, lane); break;
        case 5: enc_store_run<5>(run, g0, groups, first, last, dst, dst_words, lane); break;
        case 6: enc_store_run<6>(run, g0, groups, first, last, dst, dst_words, lane); break;
        default: enc_store_run<7>(run, g0, groups, first, last, dst, dst_words, lane); break;
    }
}

// bits = 2 * bits + in, one instruction (the compiler makes three of it)
__device__ __forceinline__ void enc_shift_in(uint32_t &bits, uint64_t in) {
    uint64_t carry;
    asm("s_nop 1\n\tv_addc_co_u32_e64 %0, %1, %0, %0, %2" : "+v"(bits), "=&s"(carry) : "s"(in));
}

// Elements' bytes to the next places of their runs, two elements at a time in the halves of a word: bit t and bit 16 + t of `not1` say which
// run each goes to, and each half of to1 and to0 holds the LDS address of its run's next byte, the second half's where the first half's
// elements will end.  The other run lies behind the dense one, so that no sum or difference leaves its half, and all but the selection are
// 32-bit operations, which take half the time of packed ones and of those that use or make a carry (an element at a time, by v_cndmask,
// v_addc and v_subb under masks in scalar registers, more of them than there are: 66.5 -> 62.0 us for the first level's, 5120 x 17408).
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef uint16_t enc_u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t lds_address(uint8_t *p) { return (uint32_t)(uintptr_t)(lds_u8 *)p; }
struct EncPut {
    uint32_t to1, to0, not1;
    __device__ __forceinline__ void two(int t, uint8_t first, uint8_t second) {
        auto halves = [](uint32_t x) { return __builtin_bit_cast(enc_u16x2, x); };
        const uint32_t out = (not1 >> t) & 0x00010001u;
        const uint32_t at = __builtin_bit_cast(uint32_t, halves(to1) + halves(to0 - to1) * halves(out));
        to1 += out ^ 0x00010001u;
        to0 += out;
        *(lds_u8 *)(uintptr_t)(at & 0xffffu) = first;
        *(lds_u8 *)(uintptr_t)(at >> 16) = second;
    }
};

// 32 weights from element p on, as pairs; infinite past n, which is in no level but the last.  `whole`: all of the wave's are there, at a multiple of 16 bytes.
__device__ __forceinline__ void load32(const uint16_t *__restrict__ w, uint32_t p, uint32_t n, bool whole, uint32_t (&d)[16]) {
    if (whole) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint4 q = *reinterpret_cast<const uint4 *>(w + p + 8 * k);
            d[4 * k] = q.x; d[4 * k + 1] = q.y; d[4 * k + 2] = q.z; d[4 * k + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; ++k) d[k] = pair_or(w, p + 2 * k, n, 0x7f80u);
    }
}

template <int L>
__global__ void __launch_bounds__(kWave *kEncWaves, L <= 3 ? 5 : 4)
k_enc_pack(const uint16_t *__restrict__ w, uint32_t n, uint32_t n_units, EncShare share,
           const uint16_t *__restrict__ scale_in, EncLevels lv, const int32_t *__restrict__ table, EncOut out) {
    constexpr int kBufs = kEncHold<L> || L < 4 ? L - 2 : 2;  // of elements on their way to the next level
    __shared__ __attribute__((aligned(32))) uint8_t bufs[kEncWaves][kEncBuf + kBufs * kEncHeld];
    static_assert(sizeof bufs <= 1u << 16, "EncPut holds LDS addresses in the halves of a word");
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t mine = blockIdx.x * kEncWaves + wave;
    if (mine >= share.waves) return;
    const uint32_t u_first = share.first_unit(mine, n_units), u_end = share.first_unit(mine + 1u, n_units);
    if (u_first >= u_end) return;
    const EncRanks ranks{table, n_units + 1, n};
    const bool aligned = (reinterpret_cast<uintptr_t>(w) & 15u) == 0;
    const float scale = bf16_bits_to_f32(*scale_in), inv_scale = __fdiv_rn(1.0f, scale);
    const float cut0 = bf16_bits_to_f32(enc_cut(lv.bits[0], scale, inv_scale, lane));
    uint8_t *const dense = bufs[wave];
    // elements that wait for level i, 1 .. L - 2
    auto held = [&](int i) { return dense + kEncBuf + (kEncHold<L> ? i - 1 : (i - 1) & 1) * kEncHeld; };
    // r0: codes of the level so far; space, count: what waits for it, index of the first in its bitmap and how many; r1[i][j]: codes of
    // level j up to where those of level i end (one row, where none waits); g_*, w_*: the groups and bitmap words shared with the
    // neighbouring waves; carry, bm_carry: what was left of an unfinished group and bitmap word
    uint32_t r0[L - 1], space[L - 1], count[L - 1], r1[L - 1][L - 1], g_first[L - 1], g_last[L - 1], carry[L - 1], w_first[L - 1], w_last[L - 1],
        bm_carry[L - 1];
    bool done[L - 1];  // the level has had all of the wave's elements
#pragma unroll
    for (int i = 0; i < L - 1; ++i) {
        r0[i] = ranks.rank(i, u_first);
        space[i] = ranks.space(i, u_first);
        count[i] = 0u;
        g_first[i] = r0[i] / 32u;
        g_last[i] = ranks.rank(i, u_end) / 32u;
        w_first[i] = space[i] / 32u;
        w_last[i] = ranks.space(i, u_end) / 32u;
        carry[i] = 128u - (uint32_t)threshold_of(lv.bits[i]);
        bm_carry[i] = 0u;
        done[i] = false;
#pragma unroll
        for (int j = 0; j < L - 1; ++j) r1[i][j] = 0u;
    }
    // a span's weights and the ranks at its end are asked for while the span before is packed
    uint32_t d[16], r1_next[L - 1], after;  // (after: the first level's at the end of the span behind that)
    auto ask = [&](uint32_t u) {
        const uint32_t e = u * kEncUnit, to = min(u + kEncSpanUnits, n_units);
        load32(w, e + lane * 32u, n, aligned && (uint64_t)e + kEncSpan <= n, d);
#pragma unroll
        for (int i = 0; i < L - 1; ++i) r1_next[i] = ranks.rank(i, to);
        after = kEncHold<L> ? ranks.rank(0, min(to + kEncSpanUnits, n_units)) : 0u;
    };
    ask(u_first);
    // In front of a dense run: the codes of its unfinished group; behind it code 0.  Around what waits for a level: value 0, a member of
    // every level.
    auto margins = [&](uint8_t *b, uint32_t first, uint32_t n_run, uint32_t front, uint32_t back) {
        const uint32_t off = first & 31u;
        if (lane < 32u) {
            if (lane < off) b[lane] = (uint8_t)front;
            b[off + n_run + lane] = (uint8_t)back;
        }
    };
    // a level's dense run of n_i codes to its stream, the unfinished group kept or, at the wave's end, stored
    auto store_level = [&](int i, uint32_t n_i, bool final) {
        const uint32_t to = r0[i] + n_i, whole = to / 32u - r0[i] / 32u;
        enc_store_run_of((uint32_t)lv.bits[i], dense + dense_at, r0[i] / 32u, final ? (to + 31u) / 32u - r0[i] / 32u : whole,
                         g_first[i], g_last[i], out.st[i], out.st_words[i], lane);
        carry[i] = dense[dense_at + whole * 32u + (lane & 31u)];
        r0[i] = to;
    };
    // the last level: one byte, value + 127, per element left over (quantize.py:84-86)
    auto store_last = [&](const uint8_t *run, uint32_t first, uint32_t n_run) {
        for (uint32_t k = lane; k < n_run; k += kWave)
            if (first + k < out.last_bytes) out.last[first + k] = (uint8_t)(max((int)run[k], 1) - 1);
    };
    uint32_t u0 = u_first;
    for (;;) {
        // ---- a span: quantise ----
        const uint32_t u1 = min(u0 + kEncSpanUnits, n_units);
        const bool final = u1 == u_end;
        const uint32_t e0 = u0 * kEncUnit, e1 = min(e0 + kEncSpan, n);
        const uint32_t p = e0 + lane * 32u;
        // (counts come from the caller's table: held to what there is)
        const uint32_t n_0 = min(r1_next[0] - r0[0], e1 - e0), left = e1 - e0 - n_0, then = after;
        uint32_t member = 0;
        float v[32];
#pragma unroll
        for (int t = 0; t < 32; ++t) {
            const float f = __uint_as_float(t & 1 ? d[t / 2] & 0xffff0000u : d[t / 2] << 16);
            v[t] = __fmaf_rn(f, inv_scale, 3072.0f);
            enc_shift_in(member, __builtin_amdgcn_ballot_w64(fabsf(f) < cut0));
        }
        member = __brev(member);  // bit t: element t is in the first level
        if (p < e1 && p / 32u < out.bm_words[0]) out.bm[0][p / 32u] = member;

        // ---- first level: codes to the dense run, the rest to what waits for the second or, in two levels, behind it (what lies past the
        // last element follows them and is overwritten by the margin) ----
        const uint32_t cnt = (uint32_t)__popc(member);
        const uint32_t before = wave_scan_inclusive(cnt) - cnt;
        const uint32_t next = e0 - r0[0];
        constexpr int k = L > 2 ? 1 : 0;
        if (!kEncHold<L> && k > 0) space[k] = next, count[k] = 0u;
        uint8_t *const rest = k > 0 ? held(k) + (space[k] & 31u) + count[k] : dense + ((dense_at + 31u + (r0[0] & 31u) + n_0) & ~31u) + 32u;
        {
            const uint32_t low = (uint32_t)__popc(member & 0xffffu);
            const uint32_t to1 = lds_address(dense) + dense_at + (r0[0] & 31u) + before;
            const uint32_t to0 = lds_address(rest) + lane * 32u - before;
            EncPut put{to1 | (to1 + low) << 16, to0 | (to0 + 16u - low) << 16, ~member};
            // 1.5 * 2^23 rounds half to even and leaves the integer in the low bits; the 3072 comes off with the same sum, which is
            // exact up to its rounding
            auto byte = [&](int t) { return (uint8_t)__float_as_uint(v[t] + (12582912.0f + 128.0f - 3072.0f)); };
#pragma unroll
            for (int t = 0; t < 16; ++t) put.two(t, byte(t), byte(16 + t));
        }
        if constexpr (L > 2) {
            // (by a true table there are no more than a span: so a level that has had its turn has room for any other's)
            count[1] = kEncHold<L> ? min(count[1] + left, kEncSpan) : left;
#pragma unroll
            for (int j = 1; j < L - 1; ++j) r1[1][j] = r1_next[j];
        }
        if (!final) ask(u1);
        margins(dense + dense_at, r0[0], n_0, carry[0], 128u - (uint32_t)threshold_of(lv.bits[0]));
        if (L > 2 && !kEncHold<L>) margins(held(1), space[k], count[k], 128u, 128u);
        wave_lds_sync();
        store_level(0, n_0, final);
        if constexpr (L == 2) store_last(rest, next, left);
        done[0] = final;
        wave_lds_sync();

        // ---- the levels behind the first: one has its turn where it has no room for what comes next, and at the wave's end; the next one
        // before it where that has none for what it will pass on ----
        for (bool again = true; again;) {
            again = false;
            bool now = false;
            if constexpr (kEncHold<L>) now = !final && count[1] > min(then - r0[0], kEncSpan);  // + (kEncSpan - those of the first level) > kEncSpan
            else if constexpr (L > 2) now = count[1] != 0u;
            if (!now && !final) break;  // (past all of it, which lies behind the span's code: an only span's wave runs straight on)
            // 16 elements a lane and turn; margin elements pass as members in front of the first and behind the last code, where the run's own
            // margins overwrite them
#pragma unroll
            for (int i = 1; i < L - 1; ++i) {
                const bool all = kEncHold<L> ? done[i - 1] : final, turn = kEncHold<L> ? now || (all && !done[i]) : all || count[i] != 0u;
                now = false;
                if (!turn) continue;
                const uint32_t n_i = min(r1[kEncHold<L> ? i : 1][i] - r0[i], count[i]), left = count[i] - n_i;
                if (kEncHold<L> && i < L - 2 && count[i < L - 2 ? i + 1 : i] + left > kEncSpan) {
                    now = again = true;
                    continue;
                }
                const uint32_t off = space[i] & 31u, end = off + count[i];
                const uint32_t thr = (uint32_t)threshold_of(lv.bits[i]);
                const uint32_t next = space[i] - r0[i];  // index of the first element that goes on
                const int k = i < L - 2 ? i + 1 : i;       // the level it goes to
                if (!kEncHold<L> && k > i) space[k] = next, count[k] = 0u;  // (as they are: but not kept in registers)
                uint8_t *const from = held(i);
                uint8_t *const rest = k > i ? held(k) + (space[k] & 31u) + count[k]
                                            : dense + ((dense_at + 31u + (r0[i] & 31u) + n_i) & ~31u) + 32u;
                if (kEncHold<L>) {
                    margins(from, space[i], count[i], 128u, 128u);
                    wave_lds_sync();
                }
                uint32_t base1 = dense_at + (r0[i] & 31u) - off, base0 = 0;
                uint32_t unfinished = 0;
                for (uint32_t s = 0; s < end; s += 1024u) {
                    const uint32_t at = s + 16u * lane;
                    uint32_t bits = 0, n_here = 0, x[4] = {0, 0, 0, 0}, m[4] = {0, 0, 0, 0};
                    if (at < end) {
                        const uint4 q = *reinterpret_cast<const uint4 *>(from + at);
                        x[0] = q.x; x[1] = q.y; x[2] = q.z; x[3] = q.w;
                        n_here = 16u;
                        // four bytes at a time: bit 7 of m set where 128 - threshold <= byte <= 128 + threshold
#pragma unroll
                        for (int k = 0; k < 4; ++k) {
                            const uint32_t low = x[k] & 0x7f7f7f7fu;
                            m[k] = ((low + thr * 0x01010101u) | x[k]) & ~((low + (127u - thr) * 0x01010101u) & x[k]) & 0x80808080u;
                        }
                        bits = (__builtin_amdgcn_udot4(m[1], 0x80402010u, __builtin_amdgcn_udot4(m[0], 0x08040201u, 0u, false), false) >> 7) |
                               (__builtin_amdgcn_udot4(m[3], 0x80402010u, __builtin_amdgcn_udot4(m[2], 0x08040201u, 0u, false), false) >> 7 << 8);
                    }
                    const uint32_t c1 = (uint32_t)__popc(bits), c0 = n_here - c1;
                    const uint32_t incl = wave_scan_inclusive(c1 | (c0 << 16));
                    if (at < end) {
                        const uint32_t low = (uint32_t)__popc(bits & 0xffu);
                        uint32_t to1 = lds_address(dense) + base1 + (incl & 0xffffu) - c1, to0 = lds_address(rest) + base0 + (incl >> 16) - c0;
                        EncPut put{to1 | (to1 + low) << 16, to0 | (to0 + 8u - low) << 16, ~((bits & 0xffu) | bits >> 8 << 16)};
#pragma unroll
                        for (int t = 0; t < 8; ++t)
                            put.two(t, (uint8_t)(x[t / 4] >> (8 * (t & 3))), (uint8_t)(x[2 + t / 4] >> (8 * (t & 3))));
                    }
                    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
                    base1 += total & 0xffffu;
                    base0 += total >> 16;
                    // bitmap i: the bits of this lane's elements that are the wave's, two lanes to a word
                    uint32_t mine = at < end ? bits : 0u;
                    if (at < off) mine &= off - at < 16u ? ~0u << (off - at) : 0u;
                    if (at + 16u > end) mine &= at < end ? (1u << (end - at)) - 1u : 0u;
                    uint32_t word = (mine & 0xffffu) | ((uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine, 0xB1, 0xf, 0xf, true) << 16);
                    if (at == 0) word |= bm_carry[i];
                    const uint32_t wi = space[i] / 32u + (at >> 5);
                    const bool last_word = at >= (end & ~31u);
                    if ((end & ~31u) - s < 1024u)
                        unfinished = (uint32_t)__builtin_amdgcn_readlane((int)word, (int)(((end & ~31u) - s) >> 4));
                    if ((lane & 1u) == 0 && at < end && wi < out.bm_words[i] && (all || !last_word)) {
                        if (wi == w_first[i] || wi == w_last[i]) {
                            if (word) atomicOr(&out.bm[i][wi], word);
                        } else {
                            out.bm[i][wi] = word;
                        }
                    }
                }
                bm_carry[i] = unfinished;
                if (k > i) {
                    count[k] += left;
#pragma unroll
                    for (int j = k; j < L - 1; ++j)
                        if (kEncHold<L>) r1[k][j] = r1[i][j];
                    if (!kEncHold<L>) margins(held(k), space[k], count[k], 128u, 128u);
                }
                margins(dense + dense_at, r0[i], n_i, carry[i], 128u - thr);
                wave_lds_sync();
                store_level(i, n_i, all);
                if (k == i) store_last(rest, next, left);
                space[i] += count[i];
                count[i] = 0u;
                if (kEncHold<L>) done[i] = all;
                wave_lds_sync();
            }
        }
        if (final) break;
        u0 = u1;
    }
}

// workspace: partial maxima (kEncParts), sums of k_enc_count's workgroups
static uint32_t count_groups(uint64_t n, uint32_t units) {
    const uint64_t group = (uint64_t)kEncUnit * units;
    return (uint32_t)((n + group - 1) / group);
}
static size_t workspace_bytes_by(uint64_t n, int n_levels, uint32_t units) {
    return 4u * (kEncParts + (size_t)(n_levels - 1) * count_groups(n, units));
}

size_t encode_workspace_bytes(uint64_t n, int n_levels) {
    return workspace_bytes_by(n, n_levels, (n + kEncUnit - 1) / kEncUnit <= kCountFew ? kCountFewUnits : kCountUnits);
}
// What a call does with: a small weight asks for more than a larger one may have (2^24 weights for 2048 sums a level, 2^25 for 1024), so
// a scratch that is shared by weights of several sizes takes the small ones by larger workgroups.
size_t encode_workspace_least(uint64_t n, int n_levels) { return workspace_bytes_by(n, n_levels, kCountUnits); }

template <int L>
static void scan_launch(const uint16_t *w, uint32_t n, uint32_t n_units, uint32_t group_units, const EncLevels &lv, const uint32_t *parts,
                        uint16_t *scale, int32_t *table, uint32_t *sums, hipStream_t s) {
    const dim3 grid(count_groups(n, group_units)), block(kWave * kEncWaves);
    if (group_units == kCountUnits)
        IXH_LAUNCH((k_enc_count<L, kCountUnits>), grid, block, 0, s, w, n, n_units, parts, lv, table, sums, scale);
    else
        IXH_LAUNCH((k_enc_count<L, kCountFewUnits>), grid, block, 0, s, w, n, n_units, parts, lv, table, sums, scale);
}

int launch_encode_scan(const uint16_t *w, uint32_t n, int n_levels, const int *bits, uint16_t *scale, int32_t *table,
                       void *workspace, size_t workspace_bytes, int64_t *host_totals, hipStream_t s) {
    const uint32_t n_units = (n + kEncUnit - 1) / kEncUnit;
    const uint32_t group_units = n_units <= kCountFew && workspace_bytes >= encode_workspace_bytes(n, n_levels) ? kCountFewUnits : kCountUnits;
    const uint32_t tiles = max(1u, (n_units + kScanTile - 1) / kScanTile);
    uint32_t *parts = static_cast<uint32_t *>(workspace);
    uint32_t *sums = parts + kEncParts;
    EncLevels lv;
    lv.n_levels = n_levels;
    for (int i = 0; i < IXH_MAX_LEVELS; ++i) lv.bits[i] = i < n_levels ? bits[i] : 0;
    IXH_LAUNCH(k_enc_absmax, dim3(kEncParts), dim3(1024), 0, s, w, n, parts);
    switch (n_levels) {
        case 2: scan_launch<2>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        case 3: scan_launch<3>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        case 4: scan_launch<4>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        case 5: scan_launch<5>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        case 6: scan_launch<6>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        case 7: scan_launch<7>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
        default: scan_launch<8>(w, n, n_units, group_units, lv, parts, scale, table, sums, s); break;
    }
    IXH_LAUNCH(k_enc_scan, dim3(tiles, n_levels - 1), dim3(1024), 0, s, table, n_units, sums,
                       count_groups(n, group_units), group_units, host_totals);
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

template <int L>
static void pack_launch(const uint16_t *w, uint32_t n, uint32_t n_units, const uint16_t *scale, const EncLevels &lv,
                        const int32_t *table, const EncOut &out, hipStream_t s) {
    static const uint32_t at_once = [] {
        int dev = 0, cus = 256, groups = 5;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&groups, k_enc_pack<L>, kWave * kEncWaves, 0);
        return (uint32_t)(max(cus, 1) * max(groups, 1)) * kEncWaves;
    }();
    const uint32_t spans = (n_units + kEncSpanUnits - 1) / kEncSpanUnits, waves = min(spans, at_once);
    const EncShare share{waves, waves ? spans / waves : 0u, waves ? spans % waves : 0u};
    IXH_LAUNCH(k_enc_borders<L>, dim3((share.waves + 256u) / 256u), dim3(256), 0, s, lv, table, n, n_units, share, out);
    if (n_units == 0) return;
    IXH_LAUNCH(k_enc_pack<L>, dim3((share.waves + kEncWaves - 1) / kEncWaves), dim3(kWave * kEncWaves), 0, s, w, n, n_units,
                       share, scale, lv, table, out);
}

int launch_encode_pack(const uint16_t *w, const Dev &P, const int32_t *table, hipStream_t s) {
    const uint32_t n = P.n;
    const uint32_t n_units = (n + kEncUnit - 1) / kEncUnit;
    EncLevels lv;
    lv.n_levels = P.n_levels;
    EncOut out;
    for (int i = 0; i < IXH_MAX_LEVELS; ++i) lv.bits[i] = i < P.n_levels ? P.bits[i] : 0;
    for (int i = 0; i < IXH_MAX_LEVELS - 1; ++i) {
        out.bm[i] = const_cast<uint32_t *>(P.bm[i]);
        out.bm_words[i] = P.bm_words[i];
        out.st[i] = const_cast<uint32_t *>(P.st[i]);
        out.st_words[i] = P.st_words[i];
    }
    out.last = const_cast<uint8_t *>(P.last);
    out.last_bytes = P.last_bytes;
    switch (P.n_levels) {
        case 2: pack_launch<2>(w, n, n_units, P.scale, lv, table, out, s); break;
        case 3: pack_launch<3>(w, n, n_units, P.scale, lv, table, out, s); break;
        case 4: pack_launch<4>(w, n, n_units, P.scale, lv, table, out, s); break;
        case 5: pack_launch<5>(w, n, n_units, P.scale, lv, table, out, s); break;
        case 6: pack_launch<6>(w, n, n_units, P.scale, lv, table, out, s); break;
        case 7: pack_launch<7>(w, n, n_units, P.scale, lv, table, out, s); break;
        default: pack_launch<8>(w, n, n_units, P.scale, lv, table, out, s); break;
    }
    return hipGetLastError() == hipSuccess ? IXH_OK : IXH_ELAUNCH;
}

}  // namespace ixh
