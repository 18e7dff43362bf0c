// What the kernels that read the lane layout (ixh_lanes.h) share: a lane's codes to dequantised pairs.
#pragma once
#include "ixh_fast358.h"
#include "ixh_lanes.h"

namespace ixh {

typedef uint32_t ln_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t ln_u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t ln_u32x2 __attribute__((ext_vector_type(2)));
typedef short ln_s16x4 __attribute__((ext_vector_type(4)));
typedef float ln_f32x4 __attribute__((ext_vector_type(4)));
typedef float ln_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 ln_bf16x2 __attribute__((ext_vector_type(2)));

typedef __bf16 ln_bf16x8 __attribute__((ext_vector_type(8)));

constexpr size_t kLnLds = 160 * 1024;

#define LN_LDS(T) __attribute__((address_space(3))) T

template <int CTRL> __device__ __forceinline__ float ln_dpp(float v) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ uint32_t ln_pack(float lo, float hi) {
    const ln_f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, ln_bf16x2));
}

// ---------------------------------------------------------------------------------------------------------------
// Pair tables.  A table of dequantised pairs (both weights as bf16) indexed by the 2 * BITS bits of a pair, in
// 2^kCopies copies side by side so that the lanes of a wave, which read unrelated entries, spread over the banks.
// A shift right, an AND, an add, a product and a multiply-add in fp32 take half the issue time of a shift left, a bit-field
// extract, a conversion or a packed operation (measured: 2.5 against 4.7 clocks a wave instruction), so a pair costs 5 clocks of issue
// and one LDS read where arithmetic (extract, convert, multiply, round) takes about 20.
// ---------------------------------------------------------------------------------------------------------------
template <int BITS, bool WIDE> struct LnPairs {
    // log2: 32 copies of 64 entries never collide, nor do 16 of 256 or 1024 much (a look-up 4.0 clocks of the LDS, against 6.1 with 8
    // copies of 1024 and 6.9 with one; 2.2 without collisions).  WIDE, where LDS has the room: 17408 x 5120, 5 bits, one row
    // 15.9 us with 8 copies and every third pair by arithmetic, 15.2 with 16.  k_lanes_gemm: see kLgWide.
    static constexpr int kCopies = BITS == 3 ? 5 : WIDE ? 4 : 1;
    static constexpr uint32_t kEntries = BITS == 8 ? 0u : 1u << (2 * BITS);
    static constexpr uint32_t kLutBytes = kEntries << (kCopies + 2);
    static constexpr uint32_t kMask = ((1u << (2 * BITS)) - 1u) << (kCopies + 2);
};

template <int BITS, bool WIDE>
__device__ __forceinline__ void ln_build_lut(uint32_t lut, float scale, uint32_t tid, uint32_t n_threads) {
    using P = LnPairs<BITS, WIDE>;
    if constexpr (P::kEntries != 0) {
        constexpr int T = (1 << (BITS - 1)) - 1;
        constexpr uint32_t RUN = P::kCopies >= 2 ? 4u : 2u;  // copies a thread stores at a time
        for (uint32_t e = tid * RUN; e < (P::kEntries << P::kCopies); e += n_threads * RUN) {
            const uint32_t idx = e >> P::kCopies;
            const uint32_t v = ln_pack((float)((int)(idx & ((1u << BITS) - 1u)) - T) * scale, (float)((int)(idx >> BITS) - T) * scale);
            if constexpr (RUN == 4) *reinterpret_cast<LN_LDS(ln_u32x4) *>((uintptr_t)(lut + e * 4u)) = ln_u32x4{v, v, v, v};
            else *reinterpret_cast<LN_LDS(ln_u32x2) *>((uintptr_t)(lut + e * 4u)) = ln_u32x2{v, v};
        }
    }
}

// at + v * 2^SH for whole numbers below 2^24, as the bits of floats of which they are multiples of the smallest: exact, and two clocks of
// issue where a shift left takes four and an add two more.  (Denormals are kept, build.sh.)
template <int SH> __device__ __forceinline__ uint32_t ln_shift_add(uint32_t v, uint32_t at) {
    constexpr float by = SH >= 0 ? (float)(1 << (SH >= 0 ? SH : 0)) : 1.0f / (float)(1 << (SH < 0 ? -SH : 0));
    return __float_as_uint(__fmaf_rn(__uint_as_float(v), by, __uint_as_float(at)));
}
template <int SH> __device__ __forceinline__ uint32_t ln_shift(uint32_t w) {
    if constexpr (SH >= 0) return w >> SH;
    else return w << -SH;
}
// Where copies of a table do not collide: 5120 x 17408 (3 bits), from graphs over copies beyond the last-level cache, at 1 / 8 / 16 / 64 rows
// 12.2 / 16.3 / 19.5 / 35.6 us with shifts, 11.8 / 15.8 / 18.8 / 34.9 so (one layer over and over, one row: 10.5 and 9.9), 10240 x 5120 (5 bits) at 1 / 8 rows 11.1 / 16.3 and 10.8 / 15.5.  With two copies the look-ups are what a wave waits
// for: 1536 x 3072 (4 bits) at 12 / 32 rows 8.0 / 8.6 with shifts, 8.2 / 8.8 so, 10240 x 5120 (4 bits) at 100 rows 33.2 either way.
template <class P> constexpr bool ln_float_shifts = P::kCopies > 1;
// the address of the pair whose code begins at bit OFF of a dword (without FLOAT less lut_lane)
template <class P, int BITS, int OFF, bool FLOAT> __device__ __forceinline__ uint32_t ln_pair_at(uint32_t w, uint32_t lut_lane) {
    constexpr int TO = P::kCopies + 2;
    constexpr uint32_t kField = (1u << (2 * BITS)) - 1u;
    if constexpr (!FLOAT) return ln_shift<OFF - TO>(w) & P::kMask;
    else if constexpr (OFF + 2 * BITS <= 24) return ln_shift_add<TO - OFF>(w & kField << OFF, lut_lane);
    else if constexpr (OFF + 2 * BITS == 32) return ln_shift_add<TO>(w >> OFF, lut_lane);
    else return ((w >> (OFF - TO)) & P::kMask) + lut_lane;
}

// the sixteen dequantised pairs of a lane's `BITS` dwords; at 5 bits in the smaller table one of the three whole pairs of a dword by
// arithmetic
template <int BITS, bool WIDE, bool FLOAT = ln_float_shifts<LnPairs<BITS, WIDE>>>
__device__ __forceinline__ void ln_decode(const uint32_t (&w)[BITS], uint32_t lut_lane, float scale, uint32_t (&o)[16]) {
    using P = LnPairs<BITS, WIDE>;
    if constexpr (BITS == 8) {
        // (c - 127) * scale as c * scale - 127 * scale: both products and the difference are exact in fp32
        const float off = -127.0f * scale;
#pragma unroll
        for (int p = 0; p < 16; ++p) {
            const uint32_t d = w[p >> 1] >> (16 * (p & 1));
            o[p] = ln_pack(__fmaf_rn((float)(d & 255u), scale, off), __fmaf_rn((float)((d >> 8) & 255u), scale, off));
        }
    } else {
        constexpr int PER = BITS == 4 ? 4 : BITS == 3 ? 5 : 3;  // whole pairs a dword
        constexpr int FIRST = BITS == 4 ? 0 : 2;
        uint32_t a[16];
#define LN_FIELD(d, f) ln_pair_at<P, BITS, FIRST + 2 * BITS * (f), FLOAT>(w[d], lut_lane)
#pragma unroll
        for (int d = 0; d < BITS; ++d) {
            a[PER * d] = LN_FIELD(d, 0);
            a[PER * d + 1] = LN_FIELD(d, 1);
            a[PER * d + 2] = LN_FIELD(d, 2);
            if constexpr (PER > 3) a[PER * d + 3] = LN_FIELD(d, 3);
            if constexpr (PER > 4) a[PER * d + 4] = LN_FIELD(d, 4);
        }
#undef LN_FIELD
        if constexpr (BITS == 3 || BITS == 5) {
            constexpr int TO = P::kCopies + 2;
            if constexpr (FLOAT) {
                a[15] = ln_shift_add<TO>(w[0] & 3u, lut_lane);
                a[15] = ln_shift_add<TO + 2>(w[1] & 3u, a[15]);
                a[15] = ln_shift_add<TO + 4>(w[2] & 3u, a[15]);
                if constexpr (BITS == 5) a[15] += ln_shift_add<TO + 8>(w[4] & 3u, ln_shift_add<TO + 6>(w[3] & 3u, 0u));
            } else {
                uint32_t last = 0;
#pragma unroll
                for (int d = 0; d < BITS; ++d) last |= (w[d] & 3u) << (TO + 2 * d);
                a[15] = last;
            }
        }
        if constexpr (BITS == 5 && !WIDE) {
            // Two copies collide: the last whole pairs of a dword by arithmetic, which evens out the LDS and the vector unit: the
            // code next to the exponent of 1.0 reads as 1 + code / 32, and (1 + code / 32) * 32 scale - 47 scale is value * scale,
            // every term exact in fp32.
            const float s32 = 32.0f * scale, off = -47.0f * scale;
#pragma unroll
            for (int d = 0; d < 5; ++d) {
                const float lo = __uint_as_float(((w[d] >> 4) & 0x7C0000u) | 0x3F800000u);
                const float hi = __uint_as_float(((w[d] >> 9) & 0x7C0000u) | 0x3F800000u);
                o[PER * d + 2] = ln_pack(__fmaf_rn(lo, s32, off), __fmaf_rn(hi, s32, off));
            }
        }
#pragma unroll
        for (int p = 0; p < 16; ++p)
            if (BITS != 5 || WIDE || p == 15 || p % 3 < 2)
                o[p] = *reinterpret_cast<const LN_LDS(uint32_t) *>((uintptr_t)(FLOAT ? a[p] : a[p] + lut_lane));
    }
}

template <int BITS>
__device__ __forceinline__ void ln_load_lane(const uint32_t *__restrict__ p, uint32_t lane, uint32_t (&w)[BITS]) {
    if constexpr (BITS == 3) {
        const ln_u32x3 v = *reinterpret_cast<const ln_u32x3 *>(p + lane * 3u);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2];
    } else {
        const ln_u32x4 v = *reinterpret_cast<const ln_u32x4 *>(p + lane * 4u);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
        if constexpr (BITS == 5) w[4] = p[256u + lane];
        if constexpr (BITS == 8) {
            const ln_u32x4 u = *reinterpret_cast<const ln_u32x4 *>(p + 256u + lane * 4u);
            w[4] = u[0]; w[5] = u[1]; w[6] = u[2]; w[7] = u[3];
        }
    }
}

__device__ __forceinline__ void ln_wave_order() {  // LDS accesses of the wave's lanes before this one come first
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

inline uint32_t ln_cus() {
    static const uint32_t n = [] {
        int dev = 0, v = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev);
        return (uint32_t)v;
    }();
    return n;
}

// outputs from `slices` sums each, [slice][activation row][ws_ld], added in slice order; the bias is added to the sum as it is
// (rounded once) or rounded to bf16
int launch_lanes_reduce(const float *ws, uint32_t slices, int m, uint32_t out_f, uint32_t ws_ld, const uint16_t *bias, bool once,
                        uint16_t *y, int64_t ldy, hipStream_t s);

}  // namespace ixh
