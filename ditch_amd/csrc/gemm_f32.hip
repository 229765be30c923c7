// gemm_f32.hip — products on f32 and f16 weights for n > 16 tokens
// (tensor.matmulT, tensor.zig:1023-1045, with the reference's f32 fused
// multiply-adds: every product x * w exact, sums in f32).
//
// The products run on the fp32 MFMA (v_mfma_f32_16x16x4_f32), which forms
// every product exactly; it issues a 16 x 16 x 4 step in 32 cycles, so the
// product is MFMA-bound and what matters is keeping every SIMD busy. Eight
// rank-4 steps per 16 x 16 tile and 32-column unit pair register s of A with
// register s of B (k = 8 (l / 16) + s): the tile layout holds the lane's 8
// weights of a unit together, and an activation row's 8 columns are two
// 16-byte words.
//
//   - rows of whole units (K a multiple of 32, 16-byte aligned):
//     f32_tile_kernel, operands staged in LDS by DMA;
//   - other rows: f32_gemm_kernel, operands loaded to registers with bounds
//     on every column.
#include "gemm_f32.h"

namespace ditch {

namespace {

constexpr int FM = 4, FN = 2;  // token tiles x row groups per wave

template <int TF>
__device__ __forceinline__ void f32_weights(const uint8_t *unit, int lane, float (&b)[8]) {
    if constexpr (TF == TF_F32) {
        const float4 lo = *((const float4 *)unit + lane), hi = *((const float4 *)(unit + 1024) + lane);
        b[0] = lo.x; b[1] = lo.y; b[2] = lo.z; b[3] = lo.w;
        b[4] = hi.x; b[5] = hi.y; b[6] = hi.z; b[7] = hi.w;
    } else {
        const uint4 h = *((const uint4 *)unit + lane);
        const uint32_t wd[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            b[2 * j] = f16_to_f32((uint16_t)(wd[j] & 0xffffu));
            b[2 * j + 1] = f16_to_f32((uint16_t)(wd[j] >> 16));
        }
    }
}

// A wave owns 64 tokens x 32 rows (4 x 2 tiles) and takes its operands straight
// from memory into two alternating register sets; a workgroup is 4 / KS tiles,
// each over KS k slices whose sums are added in slice order through LDS.
template <int TF, int KS>
__global__ __launch_bounds__(256) void f32_gemm_kernel(GemmParams p, int tiles_m, int tiles) {
    constexpr int TW = 4 / KS;  // tiles per workgroup
    constexpr int UB = TF == TF_F32 ? 2048 : 1024;
    __shared__ floatx4 red[KS > 1 ? 4 * FM * FN * 64 : 1];  // [wave][tile][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ks = wave % KS, tw = wave / KS;
    int tile = (int)blockIdx.x * TW + tw;
    const bool live = tile < tiles;
    tile = live ? tile : tiles - 1;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const TileView &w = p.w;
    const int64_t U = w.units_k, K = w.cols;
    const int64_t groups = (w.rows + 15) / 16;
    const int64_t u0 = U * ks / KS, u1 = U * (ks + 1) / KS;
    const int q = lane >> 4;

    const uint8_t *wb[FN];
#pragma unroll
    for (int i = 0; i < FN; i++) {
        int64_t g = (int64_t)tn * FN + i;
        g = g < groups ? g : groups - 1;
        wb[i] = w.codes + g * U * UB;
    }
    // tokens past n read the last token's row: their outputs are not stored
    const float *xr[FM];
#pragma unroll
    for (int m = 0; m < FM; m++) {
        int64_t tok = (int64_t)tm * 64 + 16 * m + (lane & 15);
        tok = tok < p.n ? tok : p.n - 1;
        xr[m] = p.x + (p.row_index ? (int64_t)p.row_index[tok] : tok) * p.ldx;
    }

    auto load_a = [&](int64_t u, float (&a)[FM][8]) {
        const int64_t k0 = u * 32 + 8 * q;
#pragma unroll
        for (int m = 0; m < FM; m++) {
#pragma unroll
            for (int j = 0; j < 8; j++) a[m][j] = k0 + j < K ? xr[m][k0 + j] : 0.f;
        }
    };

    floatx4 acc[FM][FN];
#pragma unroll
    for (int m = 0; m < FM; m++)
#pragma unroll
        for (int i = 0; i < FN; i++) acc[m][i] = floatx4{0.f, 0.f, 0.f, 0.f};

    if (u0 < u1) {
        // two operand sets: the loads of one unit are issued before the
        // products of the other
        float a0[FM][8], b0[FN][8], a1[FM][8], b1[FN][8];
        auto load = [&](int64_t u, float (&a)[FM][8], float (&b)[FN][8]) {
            u = u < u1 ? u : u1 - 1;
            load_a(u, a);
#pragma unroll
            for (int i = 0; i < FN; i++) f32_weights<TF>(wb[i] + u * UB, lane, b[i]);
        };
        auto products = [&](const float (&a)[FM][8], const float (&b)[FN][8]) {
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int m = 0; m < FM; m++)
#pragma unroll
                    for (int i = 0; i < FN; i++) acc[m][i] = mfma_f32(a[m][s], b[i][s], acc[m][i]);
        };
        load(u0, a0, b0);
        int64_t u = u0;
        for (; u + 1 < u1; u += 2) {
            load(u + 1, a1, b1);
            products(a0, b0);
            load(u + 2, a0, b0);
            products(a1, b1);
        }
        if (u < u1) products(a0, b0);
    }

    if constexpr (KS > 1) {
#pragma unroll
        for (int m = 0; m < FM; m++)
#pragma unroll
            for (int i = 0; i < FN; i++) red[(wave * FM * FN + m * FN + i) * 64 + lane] = acc[m][i];
        __syncthreads();
        if (ks != 0) return;
#pragma unroll
        for (int k = 1; k < KS; k++)
#pragma unroll
            for (int m = 0; m < FM; m++)
#pragma unroll
                for (int i = 0; i < FN; i++) {
                    const floatx4 o = red[((wave + k) * FM * FN + m * FN + i) * 64 + lane];
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[m][i][r] = __fadd_rn(acc[m][i][r], o[r]);
                }
    }
    if (!live) return;
    int64_t tb[FM], rw[FN];
#pragma unroll
    for (int m = 0; m < FM; m++) tb[m] = (int64_t)tm * 64 + 16 * m + 4 * q;
#pragma unroll
    for (int i = 0; i < FN; i++) rw[i] = ((int64_t)tn * FN + i) * 16 + (lane & 15);
    store_block(p, tb, rw, acc);
}

// ---------------------------------------------------------------------------
// Rows of whole units: every operand travels global -> LDS by DMA, three
// stages of 32 columns ahead: weight units as the tile layout holds them,
// eight activation rows' 128 bytes a copy, so that its lanes read whole lines
// (the 16-byte words of row r permuted by xor r % 8, so that the reads of 8
// rows fall in distinct banks; 16-byte pieces of 16 rows a copy were 10 %
// slower). Loaded to registers instead, as above, a unit's operands are sunk
// by the compiler to a few MFMAs before their use.
//
// A workgroup is KS slices of K times WG x WG waves of 32 x 32 outputs each.
// While a unit is multiplied from registers (32 MFMAs, 1024 cycles), the next
// one's operands are read from LDS and the copies of the three after it run
// (one stage ahead, the first read of a weight from memory still showed: the
// f32 forward of 24 layers, 16 x 64 tokens, 9.48 ms against 8.70). WG = 1: a
// wave's pieces are its own and it waits for its copies alone. The slices'
// tiles are added in slice order through LDS.
//
// The four stage buffers leave two waves a SIMD (one at WG = 1), which is also
// the fastest: more finish their MFMAs together and then wait together (4096 x
// 4096 on 2048 tokens with two stage buffers: 505 us at two waves, 579 at
// three, 649 at four and five; the register-staged kernel 667).
// MFMA-bound: 4096 x 4096 on 2048 tokens 534 us = 129 TFLOP/s of the 157 of
// the fp32 matrix cores; 4864 x 896 on 1024 tokens 104 -> 79 us.
typedef __attribute__((address_space(3))) void lds_void;

template <int TF, int WG, int KS, int SPAN>
__global__ __launch_bounds__(64 * WG * WG * KS) void f32_tile_kernel(GemmParams p, int tiles_m, int tiles) {
    constexpr int NWS = WG * WG, NW = NWS * KS;       // waves of a slice, of the workgroup
    constexpr int AP = 4 * WG;                        // 1 KiB activation pieces of a slice's unit
    constexpr int BH = TF == TF_F32 ? 2 : 1;          // pieces of a weight unit of 16 rows
    constexpr int BP = 2 * WG * BH;
    constexpr int CA = AP / NWS, CB = BP / NWS;  // a wave's copies
    constexpr int ST = KS * (AP + BP) * 64;           // 16-byte words of a stage
    __shared__ u32x4 buf0[ST], buf1[ST], buf2[ST], buf3[ST];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ks = wave / NWS, ws = wave % NWS, wm = ws / WG, wn = ws % WG, q = lane >> 4;
    // each XCD a contiguous run of tiles, token blocks fastest: the run's
    // weights and the activations are read from its own L2
    const int per = tiles / 8, L = blockIdx.x, tile = L < per * 8 ? L % 8 * per + L / 8 : L;
    const int tm = tile % tiles_m, tn = tile / tiles_m;
    const TileView &w = p.w;
    const int U = (int)w.units_k, groups = (int)((w.rows + 15) / 16);
    // (slices of U / KS units or one more, in nu steps each)
    const int nu = (U + KS - 1) / KS, u0 = U * ks / KS, u1 = U * (ks + 1) / KS;

    // sources of this wave's copies at unit 0 (tokens and rows past the end
    // repeat the last one: their outputs are not stored)
    const char *asrc[CA];
#pragma unroll
    for (int j = 0; j < CA; j++) {
        int64_t tok = (int64_t)tm * (32 * WG) + (ws * CA + j) * 8 + (lane >> 3);
        tok = tok < p.n ? tok : p.n - 1;
        asrc[j] = (const char *)(p.x + (p.row_index ? (int64_t)p.row_index[tok] : tok) * p.ldx +
                                 4 * ((lane & 7) ^ (lane >> 3)));
    }
    const char *bsrc[CB];
#pragma unroll
    for (int j = 0; j < CB; j++) {
        int g = tn * (2 * WG) + (ws * CB + j) / BH;
        g = g < groups ? g : groups - 1;
        bsrc[j] = (const char *)w.codes + ((int64_t)g * U * BH + (ws * CB + j) % BH) * 1024 + lane * 16;
    }
    const int mine = ks * (AP + BP) * 64;  // the slice's part of a stage
    auto copy = [&](int u, u32x4 *stage) __attribute__((always_inline)) {
        const int64_t uu = u < U ? u : U - 1;
        u32x4 *dst = stage + mine;
#pragma unroll
        for (int j = 0; j < CA; j++)
            __builtin_amdgcn_global_load_lds((const void *)(asrc[j] + uu * 128),
                                             (lds_void *)&dst[(ws * CA + j) * 64], 16, 0, 0);
#pragma unroll
        for (int j = 0; j < CB; j++)
            __builtin_amdgcn_global_load_lds((const void *)(bsrc[j] + uu * BH * 1024),
                                             (lds_void *)&dst[(AP + ws * CB + j) * 64], 16, 0, 0);
    };
    // the copies of all stages but the newest have landed, and the reads of
    // the stages before are done (sharing the buffers, everyone's)
    static_assert(AP % NWS == 0 && BP % NWS == 0 && CA + CB < 16, "copies split evenly, counted by vmcnt");
    auto landed = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0x70 | (CA + CB));  // vmcnt(copies of a stage) lgkmcnt(0)
        if constexpr (WG > 1) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    floatx4 acc[2][2];
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 2; i++) acc[m][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    struct Ops {
        float a[2][8], b[2][8];
    };
    auto read = [&](Ops &o, const u32x4 *stage) __attribute__((always_inline)) {
        const u32x4 *src = stage + mine;
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const u32x4 v = src[(wm * 2 + m) * 128 + (lane & 15) * 8 + ((2 * q + h) ^ (lane & 7))];
#pragma unroll
                for (int j = 0; j < 4; j++) o.a[m][4 * h + j] = u2f(v[j]);
            }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const u32x4 *bp = src + (AP + (wn * 2 + i) * BH) * 64 + lane;
            if constexpr (TF == TF_F32) {
                const u32x4 lo = bp[0], hi = bp[64];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    o.b[i][j] = u2f(lo[j]);
                    o.b[i][4 + j] = u2f(hi[j]);
                }
            } else {
                const u32x4 v = bp[0];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    o.b[i][2 * j] = f16_to_f32_hw((uint16_t)(v[j] & 0xffffu));
                    o.b[i][2 * j + 1] = f16_to_f32_hw((uint16_t)(v[j] >> 16));
                }
            }
        }
    };
    auto products = [&](const Ops &o) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int m = 0; m < 2; m++)
#pragma unroll
                for (int i = 0; i < 2; i++) acc[m][i] = mfma_f32(o.a[m][s], o.b[i][s], acc[m][i]);
    };

    // every slice runs nu units (past its own: copied again, not multiplied;
    // past nu: copied and never read, so that the wait count stays the same)
    Ops even, odd;
    copy(u0, buf0);
    copy(u0 + 1, buf1);
    landed();
    read(even, buf0);
    copy(u0 + 2, buf2);
    auto step = [&](int s, const Ops &cur, Ops &next, u32x4 *nbuf, u32x4 *cbuf, bool own) __attribute__((always_inline)) {
        landed();                  // stage s + 1
        read(next, nbuf);
        copy(u0 + s + 3, cbuf);    // into the buffer of stage s - 1
        if (own || u0 + s < u1) products(cur);
    };
    const int common = U / KS;  // units that every slice has
    int s = 0;
    // sums of SPAN units are added to the total (launch_staged)
    floatx4 total[2][2];
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 2; i++) total[m][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    total[m][i][r] = __fadd_rn(total[m][i][r], acc[m][i][r]);
                    acc[m][i][r] = 0.f;
                }
    };
    auto four = [&](int s) __attribute__((always_inline)) {  // no branch inside: every wait is a count
        step(s, even, odd, buf1, buf3, true);
        step(s + 1, odd, even, buf2, buf0, true);
        if constexpr (SPAN == 2) fold();
        step(s + 2, even, odd, buf3, buf1, true);
        step(s + 3, odd, even, buf0, buf2, true);
    };
    if constexpr (SPAN > 4)
        for (; s + SPAN <= common; s += SPAN) {
            for (int b = 0; b < SPAN; b += 4) four(s + b);
            fold();
        }
    for (; s + 4 <= common; s += 4) {
        four(s);
        if constexpr (SPAN <= 4) fold();
    }
    for (; s < nu; s += 4) {
        step(s, even, odd, buf1, buf3, false);
        if (s + 1 < nu) step(s + 1, odd, even, buf2, buf0, false);
        if constexpr (SPAN == 2) fold();
        if (s + 2 < nu) step(s + 2, even, odd, buf3, buf1, false);
        if (s + 3 < nu) step(s + 3, odd, even, buf0, buf2, false);
    }
    __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0): no copy outlives its buffer
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[m][i][r] = __fadd_rn(total[m][i][r], acc[m][i][r]);

    if constexpr (KS == 1) {
        const int64_t t0 = (int64_t)tm * (32 * WG) + wm * 32, r0 = (int64_t)tn * (32 * WG) + wn * 32;
        const int64_t tb[2] = {t0 + 4 * q, t0 + 16 + 4 * q}, rw[2] = {r0 + (lane & 15), r0 + 16 + (lane & 15)};
        store_block(p, tb, rw, acc);
    } else {
        constexpr int NT = 4 * NWS;  // 16 x 16 tiles of the workgroup: [slice][wave of the slice][m, i]
        // the sums in the first stage buffer where it holds them
        constexpr bool FITS = NT * KS * 64 <= ST;
        __shared__ floatx4 own[FITS ? 1 : NT * KS * 64];
        floatx4 *red = FITS ? (floatx4 *)buf0 : own;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int i = 0; i < 2; i++) red[((ks * NWS + ws) * 4 + m * 2 + i) * 64 + lane] = acc[m][i];
        __syncthreads();
        for (int t = wave; t < NT; t += NW) {
            floatx4 v[1][1] = {{red[t * 64 + lane]}};
#pragma unroll
            for (int k = 1; k < KS; k++) {
                const floatx4 o = red[(k * NT + t) * 64 + lane];
#pragma unroll
                for (int r = 0; r < 4; r++) v[0][0][r] = __fadd_rn(v[0][0][r], o[r]);
            }
            const int wt = t / 4, m = t / 2 % 2, i = t % 2;
            const int64_t tb[1] = {(int64_t)tm * (32 * WG) + (wt / WG) * 32 + 16 * m + 4 * q};
            const int64_t rw[1] = {(int64_t)tn * (32 * WG) + (wt % WG) * 32 + 16 * i + (lane & 15)};
            store_block(p, tb, rw, v);
        }
    }
}

// A sum is at most a quarter of K, and 512 columns: no K's error against 64
// bits is then above that of the register-staged kernel's four slices of one
// chain each (13312 columns: 1.03e-6 there, 0.40e-6 here, 2.1e-6 in one chain;
// 896 columns on 1024 tokens: 2.7e-7 there, 2.1e-7 here, 3.8e-7 in two chains).
// Four slices need no shorter sums for it; with fewer, 128 columns from 512 on
// and 64 below.
template <int TF, int WG, int KS>
void launch_tiles(const GemmParams &p, int tiles_m, int64_t tiles, hipStream_t s) {
    const dim3 grid((unsigned)tiles), block(64 * WG * WG * KS);
    if constexpr (KS < 4) {
        if (p.w.units_k < 64) {
            if (p.w.units_k < 16) hipLaunchKernelGGL((f32_tile_kernel<TF, WG, KS, 2>), grid, block, 0, s, p, tiles_m, (int)tiles);
            else hipLaunchKernelGGL((f32_tile_kernel<TF, WG, KS, 4>), grid, block, 0, s, p, tiles_m, (int)tiles);
            return;
        }
    }
    hipLaunchKernelGGL((f32_tile_kernel<TF, WG, KS, 16>), grid, block, 0, s, p, tiles_m, (int)tiles);
}

// 64 x 64 tiles in one slice (0.85 of the fp32 matrix rate over full rounds of
// the 256 CUs, once there are enough for two waves a SIMD) or, up to one round,
// in two slices (0.76); 32 x 32 tiles in four slices (0.63). The cheapest by
// rounds over rate, in units of a 32 x 32 tile a CU. Measured (us, 64 x 64 in
// one or two slices / 32 x 32): 896 x 4864 on 512 tokens 87 / 50, on 1024 80 /
// 97; 4864 x 896 on 256 32 / 32, on 1024 79 / 112; 4096 x 4096 on 64 73 / 23,
// on 256 70 / 81, on 512 136 / 161.
template <int TF>
void launch_staged(const GemmParams &p, hipStream_t s) {
    const int64_t m64 = (p.n + 63) / 64, t64 = m64 * ((p.w.rows + 63) / 64);
    const int64_t m32 = (p.n + 31) / 32, t32 = m32 * ((p.w.rows + 31) / 32);
    const double big = t64 > 256 ? (double)((t64 + 255) / 256) * 4 / 0.85 : 4 / 0.76;
    const double small = (double)((t32 + 255) / 256) / 0.63;
    if (small < big) launch_tiles<TF, 1, 4>(p, (int)m32, t32, s);
    else if (t64 > 256) launch_tiles<TF, 2, 1>(p, (int)m64, t64, s);
    else launch_tiles<TF, 2, 2>(p, (int)m64, t64, s);
}

// rows with bounds on every column
template <int TF>
void launch_tf(const GemmParams &p, hipStream_t s) {
    const int64_t groups = (p.w.rows + 15) / 16;
    const int tiles_m = (int)((p.n + 63) / 64), tiles = tiles_m * (int)((groups + FN - 1) / FN);
    // k slices until the grid gives every SIMD four waves (at least 2 units
    // each; two waves a SIMD measured 7 % slower on C1, eight 1 % slower)
    int ks = 1;
    while (ks < 4 && (int64_t)tiles * ks < 4096 && p.w.units_k / (2 * ks) >= 2) ks *= 2;
    const dim3 grid((unsigned)((tiles + 4 / ks - 1) / (4 / ks)));
    if (ks == 1) hipLaunchKernelGGL((f32_gemm_kernel<TF, 1>), grid, dim3(256), 0, s, p, tiles_m, tiles);
    else if (ks == 2) hipLaunchKernelGGL((f32_gemm_kernel<TF, 2>), grid, dim3(256), 0, s, p, tiles_m, tiles);
    else hipLaunchKernelGGL((f32_gemm_kernel<TF, 4>), grid, dim3(256), 0, s, p, tiles_m, tiles);
}

}  // namespace

bool f32_gemm_takes(const TileView &w, int64_t n) { return (w.tf == TF_F32 || w.tf == TF_F16) && n > 16; }

void launch_f32_gemm(const GemmParams &p, hipStream_t s) {
    DITCH_CHECK(f32_gemm_takes(p.w, p.n) && !p.segs, DITCH_INVALID_ARGUMENT, "f32 product: weight or batch not taken");
    const bool vec = p.w.cols % 32 == 0 && p.ldx % 4 == 0 && ((uintptr_t)p.x & 15) == 0;
    if (vec) p.w.tf == TF_F32 ? launch_staged<TF_F32>(p, s) : launch_staged<TF_F16>(p, s);
    else p.w.tf == TF_F32 ? launch_tf<TF_F32>(p, s) : launch_tf<TF_F16>(p, s);
    DITCH_TRY_HIP(hipGetLastError());
}

}  // namespace ditch
