// tiles.hpp -- what the tiled product kernels share: the block -> tile mapping,
// the W4A16 weight unpack and the W4A16 output store.
#pragma once

#include "common.hpp"

namespace dz {

namespace {

inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

// Tiles are assigned XCD-aware: consecutive block ids go to different XCDs,
// so tile ids are taken in XCD-major order and grouped GROUP_M tile-rows at a
// time, keeping the blocks that share an XCD's L2 on neighbouring tiles. A grid
// that is not whole rounds of the XCDs is taken in block order, where every L2
// reads all of the weight, or, with `any` and more than a block per compute unit,
// in XCD order too: the grouped Q8 products past four groups are bound by that (us,
// 16x64 tiles, N=4160, K=9216: 81 rows 37.9 in block order, 26.7 so; 97 rows 39.7 and
// 27.0; 1282 rows, N=7992, K=512 34.4 and 28.8, but K=256 21.7 and 22.6, K=64 18.8 and 19.8).
// The others, whose weights are half as large or whose stores weigh more, lose
// by it (grouped Q4, 503 rows, K=896, N=3869 15.3 and 16.1; W4A16, 596 rows,
// K=9360, N=6927 144 and 149; MLP, 264 rows, K=512, N=3520 13.2 and 13.7).
__device__ __forceinline__ void xcd_tile(int bid, int nblocks, int tiles_m, int tiles_n, int &tm, int &tn,
                                         bool any = false) {
    constexpr int XCDS = 8, GROUP_M = 4;
    int linear = bid;
    // XCD x has the blocks x, x + 8, ...: nblocks / 8 of them, and one more below the remainder
    if (any && nblocks > 32 * XCDS)
        linear = (bid % XCDS) * (nblocks / XCDS) + min(bid % XCDS, nblocks % XCDS) + bid / XCDS;
    else if (nblocks % XCDS == 0) linear = (bid % XCDS) * (nblocks / XCDS) + bid / XCDS;
    const int per_group = GROUP_M * tiles_n;
    const int group = linear / per_group;
    const int first_m = group * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int in_group = linear % per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// unpack_codes without asm: lo/hi masks come in SGPRs and the exponent in a
// VGPR, so each (w & mask) | magic is one v_and_or_b32
__device__ __forceinline__ uint4_t unpack_codes_c(uint32_t w, uint32_t mlo, uint32_t mhi, uint32_t magic) {
    const half2_t bias = {(half_t)-1032.0f, (half_t)-1032.0f};
    const half2_t sixteenth = {(half_t)0.0625f, (half_t)0.0625f};
    const half2_t bias16 = {(half_t)-72.0f, (half_t)-72.0f};
    const uint32_t w8 = w >> 8;
    uint4_t out;
    out[0] = half2_as_word(word_as_half2((w & mlo) | magic) + bias);
    out[1] = half2_as_word(__builtin_elementwise_fma(word_as_half2((w & mhi) | magic), sixteenth, bias16));
    out[2] = half2_as_word(word_as_half2((w8 & mlo) | magic) + bias);
    out[3] = half2_as_word(__builtin_elementwise_fma(word_as_half2((w8 & mhi) | magic), sixteenth, bias16));
    return out;
}

// Four consecutive outputs (columns c .. c + 3 at element `at`) of a W4A16
// GEMM: f32 (EPI 0), or rounded once to f16 plain (1), after the erf-GELU (2)
// or after the residual add (3). `vec`: n, ldo and the addresses allow whole
// vectors; otherwise columns past n are not touched.
template <int EPI>
__device__ __forceinline__ void w4a16_store(float4_t acc, void *__restrict__ out, const half_t *__restrict__ residual,
                                            size_t at, int c, int n, bool vec) {
    float v[4] = {acc[0], acc[1], acc[2], acc[3]};
    if (EPI == 0) {
        if (vec) {
            *(float4_t *)((float *)out + at) = float4_t{v[0], v[1], v[2], v[3]};
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < n) ((float *)out)[at + e] = v[e];
        }
        return;
    }
    half_t o[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (EPI == 1) o[e] = (half_t)v[e];
        else if (EPI == 2) o[e] = (half_t)f32_rounded(gelu_erf(v[e]));
        else o[e] = (half_t)0.0f;
    }
    if (EPI == 3) {
        if (vec) {
            const uint2_t rw = *(const uint2_t *)(residual + at);
            const half2_t r01 = word_as_half2(rw[0]), r23 = word_as_half2(rw[1]);
            o[0] = (half_t)f32_rounded(v[0] + (float)r01[0]);
            o[1] = (half_t)f32_rounded(v[1] + (float)r01[1]);
            o[2] = (half_t)f32_rounded(v[2] + (float)r23[0]);
            o[3] = (half_t)f32_rounded(v[3] + (float)r23[1]);
        } else {
            for (int e = 0; e < 4; e++)
                if (c + e < n) o[e] = (half_t)f32_rounded(v[e] + (float)residual[at + e]);
        }
    }
    if (vec) {
        const half2_t o01 = {o[0], o[1]}, o23 = {o[2], o[3]};
        *(uint2_t *)((half_t *)out + at) = uint2_t{half2_as_word(o01), half2_as_word(o23)};
    } else {
        for (int e = 0; e < 4; e++)
            if (c + e < n) ((half_t *)out)[at + e] = o[e];
    }
}

}  // namespace

}  // namespace dz
