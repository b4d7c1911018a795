// products_small.hip -- the products on small tiles, for grids that the tiles
// of products.hip leave mostly idle (tens to hundreds of rows).
#include <type_traits>

#include "kernels.hpp"
#include "tiles.hpp"

namespace dz {

namespace {

// ============================================================================
// W4A16 GEMM on small tiles
// ============================================================================
//
// The pipelined kernel's product on tiles of 16..64 rows, for grids that its
// 128- and 256-row tiles would leave mostly idle. There a compute unit holds
// about one wave per SIMD and every wave walks K alone, so the latency of a
// step bounds it: its LDS reads are issued a step ahead (two register sets),
// and the loads of NS - 1 further steps are in flight. A step is KS k-blocks of
// TILES column tiles with W = KS * TILES waves: wave w loads the codes and
// scales of (k-block w / TILES, tile w % TILES) and its share of the rows, so
// every wave has the same loads and waits by count (vmcnt). Same swizzle,
// unpack and k order as w4a16_pipe_kernel: the same bits. Any k (k % 8 == 0):
// what is past k reads as zero. 17 rows, K=N=4096: 36.4 us on 128x128 tiles,
// 12.0 on 32x32 here (13.9 with the LDS reads at the step's start, 13.4 with
// each wave unpacking a share into LDS for all: its LDS traffic bounds that).
// About 0.25 us per 128-k block: 93 instructions of one wave per SIMD.
template <int BM, int BN, int WGM, int WGN, int KS, bool G32, int EPI>
__global__ __launch_bounds__(WGM *WGN * 64) void w4a16_small_kernel(
    const uint8_t *__restrict__ codes, const uint8_t *__restrict__ scales, const half_t *__restrict__ x, int m,
    int k, int n, int kbs, void *__restrict__ out, const half_t *__restrict__ residual) {
    constexpr int W = WGM * WGN, TILES = BN / 16, NS = 4;
    constexpr int TM = BM / WGM, TN = BN / WGN, MB = TM / 16, NT = TN / 16;
    constexpr int XI = BM / 4, XL = XI * KS / W;  // 1 KiB loads of four rows: per k-block, and per wave and batch
    constexpr int PB = XL + 2;                    // loads per wave and batch
    constexpr int XST = KS * BM * 256, CST = W * 1152;
    static_assert(TM % 16 == 0 && TN % 16 == 0, "whole MFMA tiles");
    static_assert(W == KS * TILES && XL * W == XI * KS && XI % XL == 0, "every wave has a unit and whole loads");
    __shared__ __align__(16) uint8_t xs[NS * XST];
    __shared__ __align__(16) uint8_t cs[NS * CST];  // per unit 1 KiB of codes, then 128 bytes of scales

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int wm = wave / WGN, wn = wave % WGN;
    const int q = lane / 16, j = lane % 16;
    const int tiles_m = (m + BM - 1) / BM, tiles_n = (n + BN - 1) / BN;
    int tm, tn;
    xcd_tile(blockIdx.x, gridDim.x, tiles_m, tiles_n, tm, tn);
    const int row0 = tm * BM, col0 = tn * BN;
    const int tiles = (n + 15) / 16, tile0 = col0 / 16, tvalid = min(TILES, tiles - tile0);
    const int32x4_t rx = buffer_rsrc(x + (size_t)row0 * k, (uint32_t)(min(BM, m - row0) * k * 2));
    const int32x4_t rc = buffer_rsrc(codes + (size_t)tile0 * kbs * 1024, (uint32_t)(tvalid * kbs * 1024));
    const int32x4_t rs = buffer_rsrc(scales + (size_t)tile0 * kbs * 128, (uint32_t)(tvalid * kbs * 128));

    // this wave's activation loads: rows 4 i0 .. of k-block xu of a step; lane
    // (q, j) of load p fills slot j of row 4 (i0 + p) + q from chunk j ^ (row & 15)
    const int xu = wave / (XI / XL), i0 = wave % (XI / XL) * XL;
    const uint32_t xl0 = __builtin_amdgcn_readfirstlane(lds_address(xs) + (xu * XI + i0) * 1024);
    uint32_t xoff[XL];
    int cx[XL];
#pragma unroll
    for (int p = 0; p < XL; p++) {
        cx[p] = j ^ q ^ (4 * ((i0 + p) & 3));
        xoff[p] = (uint32_t)(((i0 + p) * 4 + q) * k * 2 + cx[p] * 16);
    }
    // its unit: k-block uu of the step, column tile ut
    const int uu = wave / TILES, ut = wave % TILES;
    const uint32_t cl0 = __builtin_amdgcn_readfirstlane(lds_address(cs) + wave * 1152);
    const uint32_t coff = (uint32_t)(ut * kbs * 1024 + lane * 16), soff = (uint32_t)(ut * kbs * 128 + lane * 16);
    constexpr uint32_t kOut = 0x80000000u;  // out of range of every resource

    auto load_batch = [&](int slot, int step) {
        if ((step + 1) * KS * 128 <= k) {
            const uint32_t at = (uint32_t)(step * KS + xu) * 256;
#pragma unroll
            for (int p = 0; p < XL; p++) dma16_at(xl0 + slot * XST + p * 1024, xoff[p], rx, at);
        } else {  // the last step may reach past k, and later ones load nothing
            const int kk = (step * KS + xu) * 128;
#pragma unroll
            for (int p = 0; p < XL; p++)
                dma16_at(xl0 + slot * XST + p * 1024, kk + cx[p] * 8 < k ? xoff[p] + (uint32_t)kk * 2 : kOut, rx, 0u);
        }
        const int kb = step * KS + uu;
        const bool live = kb < kbs;
        dma16_at(cl0 + slot * CST, live ? coff : kOut, rc, live ? (uint32_t)kb * 1024 : 0u);
        if (lane < 8) dma16_at(cl0 + slot * CST + 1024, live ? soff : kOut, rs, live ? (uint32_t)kb * 128 : 0u);
    };

    float4_t acc[MB][NT];
#pragma unroll
    for (int a = 0; a < MB; a++)
#pragma unroll
        for (int b = 0; b < NT; b++) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    uint32_t mlo = 0x000F000Fu, mhi = 0x00F000F0u, magic_v = 0x64006400u;
    asm volatile("" : "+s"(mlo), "+s"(mhi), "+v"(magic_v));

    struct Frags {
        half8_t x[KS][4][MB];
        uint4_t c[KS][NT];
        uint2_t s[KS][NT];
    };
    auto read = [&](int slot, Frags &f) {
        const uint8_t *xst = xs + slot * XST, *cst = cs + slot * CST;
#pragma unroll
        for (int u = 0; u < KS; u++) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint8_t *c = cst + (u * TILES + wn * NT + nt) * 1152;
                f.c[u][nt] = *(const uint4_t *)(c + lane * 16);
                f.s[u][nt] = *(const uint2_t *)(c + 1024 + j * 8);
            }
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int mb = 0; mb < MB; mb++)
                    f.x[u][s][mb] = *(const half8_t *)(xst + u * BM * 256 + (wm * TM + mb * 16 + j) * 256 +
                                                       (((4 * s + q) ^ j) * 16));
        }
    };
    auto compute = [&](const Frags &f, int live) {
#pragma unroll
        for (int u = 0; u < KS; u++) {
            if (u >= live) break;
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    half_t sh;
                    if (G32)
                        sh = __builtin_bit_cast(half_t,
                                                (unsigned short)((f.s[u][nt][s >> 1] >> (16 * (s & 1))) & 0xffffu));
                    else
                        sh = (half_t)word_as_float(f.s[u][nt][s >> 1]);
                    const half2_t s2 = {sh, sh};
                    uint4_t c8 = unpack_codes_c(f.c[u][nt][s], mlo, mhi, magic_v);
#pragma unroll
                    for (int e = 0; e < 4; e++) c8[e] = half2_as_word(word_as_half2(c8[e]) * s2);
#pragma unroll
                    for (int mb = 0; mb < MB; mb++) acc[mb][nt] = mfma_f16(as_half8(c8), f.x[u][s][mb], acc[mb][nt]);
                }
        }
    };

    const int steps = (kbs + KS - 1) / KS;
    Frags fr[2];
#pragma unroll
    for (int b = 0; b < NS; b++) load_batch(b, b);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NS - 1) * PB) : "memory");
    read(0, fr[0]);
    // step i in slot C, its operands already in registers: once batch i + 1 is
    // here and every wave has read slot C, the slot takes batch i + NS and the
    // next step's operands are read while this one computes
    auto run_step = [&](auto slot, int i) {
        constexpr int C = decltype(slot)::value;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * PB) : "memory");
        load_batch(C, i + NS);
        read((C + 1) % NS, fr[(C + 1) % 2]);
        compute(fr[C % 2], kbs - i * KS);
    };
    for (int i = 0; i < steps; i += NS) {
        run_step(std::integral_constant<int, 0>{}, i);
        if (i + 1 < steps) run_step(std::integral_constant<int, 1>{}, i + 1);
        if (i + 2 < steps) run_step(std::integral_constant<int, 2>{}, i + 2);
        if (i + 3 < steps) run_step(std::integral_constant<int, 3>{}, i + 3);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // no LDS write in flight once the block ends

    const bool vec = (n & 3) == 0 && ((uintptr_t)out & 15) == 0 && (EPI != 3 || ((uintptr_t)residual & 7) == 0);
#pragma unroll
    for (int mb = 0; mb < MB; mb++) {
        const int r = row0 + wm * TM + mb * 16 + j;
        if (r >= m) continue;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int c = col0 + wn * TN + nt * 16 + 4 * q;
            if (c < n) w4a16_store<EPI>(acc[mb][nt], out, residual, (size_t)r * n + c, c, n, vec);
        }
    }
}

// ============================================================================
// per-row int8 product of a few rows
// ============================================================================
//
// Up to 16 MB rows against all of the weight: HBM bound, so the weight is
// streamed as a GEMV does and not walked tile by tile. A block owns 16 weight
// rows; its 8 waves take the 64-byte chunks of k in turn (chunk c on wave c %
// 8), U of them in flight at once, and each chunk is MB v_mfma_i32_16x16x64_i8
// on operands that come straight from memory (the activations from the L2). The
// waves' int32 partials are exact, so they add in any order, in LDS. Rows and
// columns past the end read as zero (buffer range checks); RAGGED (k % 4 == 0)
// clears the weight's bytes past k.
template <int MB, int U, bool RAGGED>
__global__ __launch_bounds__(512) void i8_rows_kernel(const int8_t *__restrict__ a, const float *__restrict__ sa,
                                                       int m, const int8_t *__restrict__ b,
                                                       const float *__restrict__ sb, int n, int k,
                                                       void *__restrict__ y, int raw) {
    constexpr int WAVES = 8;
    __shared__ __align__(16) int32_t part[WAVES][MB * 256];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;
    const int q = lane / 16, j = lane % 16;
    const int col0 = blockIdx.x * 16, row0 = blockIdx.y * 16 * MB;
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)(b + (size_t)col0 * k), (short)0,
                                                                        min(16, n - col0) * k, 0x00020000);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(a + (size_t)row0 * k), (short)0,
                                                                        min(16 * MB, m - row0) * k, 0x00020000);
    const int chunks = (k + 63) / 64;
    const uint32_t off = (uint32_t)(j * k + 16 * q);
    int4_t acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; mb++) acc[mb] = int4_t{0, 0, 0, 0};
    for (int c0 = wave; c0 < chunks; c0 += WAVES * U) {
        int4_t bf[U], af[U][MB];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int kk = (c0 + u * WAVES) * 64;
            const uint32_t v = kk + 16 * q < k ? off + (uint32_t)kk : 0x80000000u;  // out of range of both
            bf[u] = __builtin_bit_cast(int4_t, __builtin_amdgcn_raw_buffer_load_b128(rb, v, 0, 0));
            if (RAGGED) {  // bytes past k are the next row's
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (kk + 16 * q + 4 * e >= k) bf[u][e] = 0;
            }
#pragma unroll
            for (int mb = 0; mb < MB; mb++)
                af[u][mb] = __builtin_bit_cast(int4_t, __builtin_amdgcn_raw_buffer_load_b128(ra, v + (uint32_t)(mb * 16 * k), 0, 0));
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int mb = 0; mb < MB; mb++) acc[mb] = mfma_i8(bf[u], af[u][mb], acc[mb]);
    }
    // acc[mb][v]: weight row 4 q + v, activation row 16 mb + j
#pragma unroll
    for (int mb = 0; mb < MB; mb++) *(int4_t *)&part[wave][(mb * 16 + j) * 16 + 4 * q] = acc[mb];
    __syncthreads();
    for (int i = threadIdx.x; i < MB * 256; i += WAVES * 64) {
        int dot = 0;
#pragma unroll
        for (int w = 0; w < WAVES; w++) dot += part[w][i];
        const int r = row0 + i / 16, c = col0 + i % 16;
        if (r >= m || c >= n) continue;
        if (raw) ((int32_t *)y)[(size_t)r * n + c] = dot;
        else ((float *)y)[(size_t)r * n + c] = __fmul_rn(__fmul_rn((float)dot, sa[r]), sb[c]);
    }
}

// False (nothing launched) where the 32-bit offsets of a block's panels do not reach.
template <int BM, int BN, int WGM, int WGN, int KS, int EPI>
bool w4a16_small_launch(const Weight &w, const half_t *x, int m, void *y, const half_t *res, hipStream_t s) {
    if ((size_t)BM * w.cols * 2 >= ((size_t)1 << 31) || (size_t)(BN / 16) * w.kblocks() * 1024 >= ((size_t)1 << 31))
        return false;
    const dim3 blocks(cdiv(m, BM) * cdiv(w.rows, BN));
    if (w.kind == WeightKind::Q4G32)
        hipLaunchKernelGGL((w4a16_small_kernel<BM, BN, WGM, WGN, KS, true, EPI>), blocks, dim3(WGM * WGN * 64), 0, s,
                           w.codes, w.scales, x, m, w.cols, w.rows, w.kblocks(), y, res);
    else
        hipLaunchKernelGGL((w4a16_small_kernel<BM, BN, WGM, WGN, KS, false, EPI>), blocks, dim3(WGM * WGN * 64), 0, s,
                           w.codes, w.scales, x, m, w.cols, w.rows, w.kblocks(), y, res);
    return true;
}

template <int EPI>
bool w4a16_small(const Weight &w, const half_t *x, int m, void *y, const half_t *res, int tile, hipStream_t s) {
    switch (tile) {
        case 0: return w4a16_small_launch<32, 32, 2, 2, 2, EPI>(w, x, m, y, res, s);
        case 1: return w4a16_small_launch<32, 64, 2, 4, 2, EPI>(w, x, m, y, res, s);
        case 2: return w4a16_small_launch<64, 64, 2, 2, 1, EPI>(w, x, m, y, res, s);
        case 3: return w4a16_small_launch<64, 128, 2, 4, 1, EPI>(w, x, m, y, res, s);
        default: return false;
    }
}

template <int MB, int U>
void i8_rows_launch(const int8_t *a, const float *sa, int m, const int8_t *b, const float *sb, int n, int k, void *y,
                    int raw, hipStream_t s) {
    const dim3 blocks(cdiv(n, 16), cdiv(m, 16 * MB));
    if (k % 16 != 0)
        hipLaunchKernelGGL((i8_rows_kernel<MB, U, true>), blocks, dim3(512), 0, s, a, sa, m, b, sb, n, k, y, raw);
    else
        hipLaunchKernelGGL((i8_rows_kernel<MB, U, false>), blocks, dim3(512), 0, s, a, sa, m, b, sb, n, k, y, raw);
}

}  // namespace

bool launch_i8_rows(const int8_t *a, const float *sa, int m, const int8_t *b, const float *sb, int n, int k, void *y,
                    int raw, hipStream_t s) {
    // loads of whole words; byte offsets of a panel stay below 2^31 (k <= 32768)
    if (k % 4 != 0 || k > 32768 || (((uintptr_t)a | (uintptr_t)b) & 3) != 0) return false;
    if (m <= 16) i8_rows_launch<1, 8>(a, sa, m, b, sb, n, k, y, raw, s);
    else i8_rows_launch<2, 4>(a, sa, m, b, sb, n, k, y, raw, s);
    return true;
}

// A smaller tile walks K faster and a larger one does more work per walk, so
// the first tile of this list whose grid gives no compute unit two blocks is
// taken, and none past the last (the pipelined 128- and 256-row tiles do more work per unit there).
// Measured (us, graph-timed; 32x32 / 32x64 / 64x64 / 64x128 / pipelined), one
// block per unit at most marked *: K=4096, N=4096: 17 rows 12.0* / 15.5* /
// 21.4* / 27.6* / 36.4; 128 rows 23.5 / 17.3* / 22.6* / 29.2* / 38.3; 200 rows
// 43.2 / 31.0 / 23.5* / 30.0* / 38.4; 512 rows 83.6 / 62.1 / 44.6 / 36.4* /
// 41.0; 1024 rows - / - / 84.7 / 65.4 / 49.8. K=1024, N=4096: 17 rows 5.4* /
// 6.3* / 7.8* / 9.5* / 11.2; 308 rows 22.5 / 17.7 / 15.8 / 11.3* / 13.4.
int w4a16_small_tile(int m, int n) {
    const unsigned cus = (unsigned)device_cus();
    constexpr int kRows[] = {32, 32, 64, 64}, kCols[] = {32, 64, 64, 128};
    for (int t = 0; t < 4; t++)
        if ((size_t)cdiv(m, kRows[t]) * cdiv(n, kCols[t]) <= cus) return t;
    return -1;
}

bool launch_w4a16_small(const Weight &w, const half_t *x, int m, void *y, int epi, const half_t *res, int tile,
                        hipStream_t s) {
    switch (epi) {
        case 0: return w4a16_small<0>(w, x, m, y, res, tile, s);
        case 1: return w4a16_small<1>(w, x, m, y, res, tile, s);
        case 2: return w4a16_small<2>(w, x, m, y, res, tile, s);
        default: return w4a16_small<3>(w, x, m, y, res, tile, s);
    }
}

}  // namespace dz
