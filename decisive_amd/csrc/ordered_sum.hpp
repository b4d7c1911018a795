// The f32 sum of non-negative terms in index order, rounded after every
// addition as a serial loop rounds it, by one wave.
//
// A serial chain pays the latency of an addition for every term (about 10
// cycles: 12 us for 2560). But as long as the running sum s stays in one binade
// it is a whole number of that binade's ulps, and adding a term moves it by a
// whole number of ulps that depends on s only through the parity of s, where
// the term is an exact half (round to nearest even). So each lane adds its eight
// terms to the even and to the odd start of the binade, a scan over the lanes
// adds up the ulps, and where a lane's two answers differ the parity of the sum
// before it chooses. The lane in which s leaves the binade adds its terms to the
// exact s one by one, and the lanes after it start over in the new binade: one
// pass per 512 terms and one per binade crossed, about 14 for 2560 like-sized
// terms. Any terms give the serial sum, in at worst one pass per lane; an
// infinite or NaN term ends in the infinite or NaN sum of the loop.
#pragma once
#include "common.hpp"

namespace dz {

__device__ __forceinline__ uint32_t wave_scan_dpp(uint32_t v) {  // inclusive
    v += __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, false);  // lane 15 of rows 0, 2 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, false);  // lane 31 into rows 2, 3
    return v;
}

// All 64 lanes of one wave; terms in LDS, 16-byte aligned, n > 0.
__device__ __forceinline__ float ordered_sum(const float *terms, int n) {
    constexpr uint32_t BINADE = 1u << 23;  // ulps
    const int lane = threadIdx.x % 64;
    auto read = [&](int at, float (&t)[8]) __attribute__((always_inline)) {
        at += lane * 8;
        if (at + 8 <= n) {
            const float4_t a = *(const float4_t *)(terms + at), b = *(const float4_t *)(terms + at + 4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                t[e] = a[e];
                t[4 + e] = b[e];
            }
        } else {  // adding 0 changes nothing
#pragma unroll
            for (int e = 0; e < 8; e++) t[e] = at + e < n ? terms[at + e] : 0.0f;
        }
    };
    uint32_t sum = 0;  // the bits of s, uniform
    float t[8], ahead[8];
    read(0, t);
    for (int at = 0; at < n; at += 512) {
        read(at + 512, ahead);  // past the end: zeros
        int first = 0;          // the lanes before it are in s
        do {
            const uint32_t base = sum & 0xff800000u;
            float even = __builtin_bit_cast(float, base), odd = __builtin_bit_cast(float, base | 1u);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                even = __fadd_rn(even, t[e]);
                odd = __fadd_rn(odd, t[e]);
            }
            uint32_t up0 = min(__builtin_bit_cast(uint32_t, even) - base, BINADE);
            uint32_t up1 = min(__builtin_bit_cast(uint32_t, odd) - (base | 1u), BINADE);
            if (lane < first) up0 = up1 = 0;
            // the sum after each lane, in ulps of the binade; right up to the first
            // lane whose two answers differ, and below BINADE up to the first crossing
            uint32_t at_end = (sum - base) + wave_scan_dpp(up0);
            uint64_t ties = __ballot(up0 != up1);
            uint64_t crossed = __ballot(at_end >= BINADE);
            while (ties) {
                const int l = __builtin_ctzll(ties);
                if (crossed && __builtin_ctzll(crossed) < l) break;
                ties &= ties - 1;
                const uint32_t even_up = __builtin_amdgcn_readlane(up0, l);
                if ((__builtin_amdgcn_readlane(at_end, l) - even_up) & 1) {
                    const uint32_t more = __builtin_amdgcn_readlane(up1, l) - even_up;
                    if (lane >= l) at_end += more;
                    crossed = __ballot(at_end >= BINADE);
                }
            }
            if (!crossed) {
                sum = base + __builtin_amdgcn_readlane(at_end, 63);
                break;
            }
            const int l = __builtin_ctzll(crossed);
            if (l) sum = base + __builtin_amdgcn_readlane(at_end, l - 1);
            float s = __builtin_bit_cast(float, sum);
#pragma unroll
            for (int e = 0; e < 8; e++) s = __fadd_rn(s, t[e]);
            sum = __builtin_amdgcn_readlane(__builtin_bit_cast(uint32_t, s), l);
            first = l + 1;
        } while (first < 64);
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] = ahead[e];
    }
    return __builtin_bit_cast(float, sum);
}

// 1 / sqrt(ss / d + eps). v_sqrt_f32 is not correctly rounded; a float's square
// root taken in f64 and rounded to f32 is (the exact root is never near enough
// to a float midpoint for the f64 error to matter).
__device__ __forceinline__ float rms_row_scale(float ss, int d, float eps) {
    const float q = __fadd_rn(__fdiv_rn(ss, (float)d), eps);
    return __fdiv_rn(1.0f, __double2float_rn(__dsqrt_rn((double)q)));
}

}  // namespace dz
