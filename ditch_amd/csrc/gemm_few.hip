// gemm_few.hip — the product of few tokens: out[n][rows] = x[n][cols] . W^T
// (tensor.matmulT, tensor.zig:1023-1045) for decode steps, short prompts and
// ragged small batches, on tensors the conversion instructions decode exactly
// (TileView::fast: bf16, FP8, MXFP4, INT4, Q8_0).
//
// A call of this size reads every weight once and does little with it, so it
// is bound by the weight read where the matrix is large (14336 x 4096 on one
// token: FP8 13.3 us = 4.4 TB/s) and by one wave's chain of loads and decode
// below that (4096 x 4096: 5 to 7 us). Both ask for many short waves:
//
//   - a workgroup takes NT groups of 16 rows and MT blocks of 16 tokens; its W
//     waves take contiguous slices of K and add them through LDS in wave order
//     (no partial sums in memory, no second launch);
//   - K advances in steps of 128 columns (1, 2 or 4 weight units a row group);
//     two register sets alternate, the next step's codes, scale words and
//     activations requested before the current one is decoded and multiplied.
//     No branch inside the loop, so every wait is a count of later loads;
//   - the weights are decoded by the tiled product's instructions
//     (tile_decode.h). The element decoders of the GEMV (gemv.hip), which
//     follow NaN and infinity rules these tensors cannot meet, took 100 us for
//     FP8 and 29 us for MXFP4 at 4096 x 4096 on one token;
//   - up to 8 tokens (NX) each wave splits its slice of the f32 rows into bf16
//     terms itself, in its own LDS slot; more tokens come as fragments
//     (split_kernel's layout), which producers write directly, or, where the
//     caller has no scratch for them or there are few weights, in chunks of 8 (24
//     tokens: 0.6 to 0.9 of the fragments' time below 4 M weights, 1.2 to 1.9 of
//     it at 14336 x 4096);
//   - one launch may hold up to three matrices over the same activations.
//
// Measured, us a call with its split (before: the GEMV up to 16 tokens, the
// register-staged or the tiled product above), 4096 x 4096:
//   n            1            8           16           24           64
//   FP8     100 -> 6.3   105 -> 9.7  103 -> 10.7  431 -> 12.1  29 -> 15.9
//   MXFP4    29 -> 5.1    35 -> 8.8   32 -> 10.9  175 -> 11.5  28 -> 15.0
//   INT4     47 -> 6.2    54 -> 9.6   51 -> 10.9  302 -> 12.5  31 -> 16.1
#include "gemm_few.h"
#include "tile_decode.h"

namespace ditch {

namespace {

// MATS matrices in one launch; end[i]: row blocks up to and including matrix i
template <int MATS> struct FewParams {
    FewMat mat[MATS];
    int end[MATS];
    int tblocks;  // token blocks (of 16 MT tokens)
    const float *x;
    const uint8_t *xs;
    int64_t n, ldx, ldk;
    // GLU: f32 rows and fragments of act(x mat[0]^T) * (x mat[1]^T)
    float *y;
    uint8_t *ys;
    int64_t ldk_y;
    uint32_t act;
    // SEG: segment blockIdx.y's matrices and rows (mat[] unused)
    const GroupSeg *segs, *segs_up;
    const int32_t *row_index;
    const float *delta_xa;
    int delta_stride;
    float *out;
};

// weight units and side words per row group of a 128-column step
template <int TF> struct Few {
    static constexpr int UPS = TF == TF_BF16 ? 4 : (TF == TF_FP8 || TF == TF_Q8) ? 2 : 1;
    static constexpr int NS = TF == TF_BF16 ? 0 : TF == TF_MX4 ? 1 : 2;
    static constexpr int NSA = NS ? NS : 1;
};

// A wave's activation slot (NX > 0): the words of a step in fragment order,
// [term][k tile][k quarter][token] x 16 bytes, each quarter padded by one word
// (two or more tokens) so that a wave's writes fall in distinct banks.
template <int XT, int NX> struct FewSlot {
    static constexpr int QS = NX > 1 ? NX + 1 : 1;  // words of a (k tile, quarter)
    static constexpr int TS = 4 * QS, ES = 4 * TS;  // of a k tile, of a term
    static constexpr int WORDS = NX > 0 ? XT * ES : 0;
};

// One step's operands of a wave in registers.
template <int TF, int MT, int NT, int XT, int NX> struct FewSet {
    u32x4 raw[NT][Few<TF>::UPS];
    uint32_t side[NT][Few<TF>::NSA];
    u32x4 xa[NX ? 1 : MT][NX ? 1 : 4][NX ? 1 : XT];
    float2 x1;                       // NX = 1: columns 2 lane, 2 lane + 1
    float4 xp[NX > 1 ? NX / 2 : 1];  // NX > 1: token 2 m + lane / 32, columns 4 (lane % 32) .. +4
};

// two f32 values' bf16 term; the values are left holding the remainders
__device__ __forceinline__ uint32_t next_term(float &a, float &b) {
    const uint32_t wd = cvt_pk_bf16(a, b);
    a = __fsub_rn(a, u2f(wd << 16));
    b = __fsub_rn(b, u2f(wd & 0xffff0000u));
    return wd;
}

// GLU: mat[0] and mat[1] are gate and up; a workgroup takes OT row groups of
// both, and its epilogue writes act(gate) * up of the summed tiles.
// SEG: a segment (a routed expert) a blockIdx.y, NX of its rows a blockIdx.z,
// gathered by row_index (or consecutive), from f32 rows.
template <int TF, int MT, int OT, int W, int XT, int NX, int MATS, bool GLU, bool SEG = false>
__global__ __launch_bounds__(64 * W) void few_kernel(FewParams<MATS> p) {
    static_assert(!SEG || (NX > 1 && MT == 1), "segments read f32 rows");
    constexpr int UPS = Few<TF>::UPS, NS = Few<TF>::NS;
    constexpr int NT = GLU ? 2 * OT : OT;  // row groups in registers
    typedef FewSlot<XT, NX> Slot;
    constexpr int RED = W * MT * NT * 64;
    __shared__ u32x4 lds[W * Slot::WORDS > RED ? W * Slot::WORDS : RED];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c16 = lane & 15, kq = lane >> 4;
    // (row block, token block): consecutive workgroups go to the 8 XCDs in
    // turn, so the token blocks of a row block are 8 apart (one XCD reads the
    // row block's weights once from memory and then from its L2)
    int rb = blockIdx.x, tb = 0;
    if (!SEG && p.tblocks > 1) {
        const int nb = p.end[MATS - 1], full = nb / 8 * 8 * p.tblocks, L = blockIdx.x;
        if (L < full) {
            tb = L / 8 % p.tblocks;
            rb = L / (8 * p.tblocks) * 8 + L % 8;
        } else {
            const int rest = nb % 8;
            tb = (L - full) / rest;
            rb = nb / 8 * 8 + (L - full) % rest;
        }
    }
    int mi = 0;
    if constexpr (!GLU && !SEG) {
#pragma unroll
        for (int i = 0; i + 1 < MATS; i++) mi += rb >= p.end[i];
        if (mi) rb -= p.end[mi - 1];
    }
    const FewMat &mat = p.mat[mi];
    const GroupSeg *seg = SEG ? p.segs + blockIdx.y : nullptr;
    const TileView &w = SEG ? seg->w : mat.w;
    // f32 rows: NX of the segment's or of the call's tokens
    const int64_t all = SEG ? seg->cnt : p.n, first = SEG ? (int64_t)blockIdx.z * NX : NX ? (int64_t)tb * NX : 0;
    const int64_t n = NX && all - first > NX ? NX : all - first, off = (SEG ? seg->off : 0) + first;
    if (SEG && n <= 0) return;
    if constexpr (NX > 0) tb = 0;  // (outputs count from row off)
    const int64_t groups = (w.rows + 15) / 16, g0 = (int64_t)rb * OT, units = w.units_k, K = w.cols;
    const int steps = (int)((units + UPS - 1) / UPS), per = (steps + W - 1) / W;
    const int s0 = wave * per < steps ? wave * per : steps, s1 = s0 + per < steps ? s0 + per : steps;

    const uint8_t *wb[NT];
    const uint32_t *sb[NT];
    const uint32_t woff = (uint32_t)lane * 16;
    SideStep st{1, 0};
    if constexpr (TF == TF_FP8 || TF == TF_INT4) st = side_step<TF>(w);
#pragma unroll
    for (int i = 0; i < NT; i++) {
        const TileView &wi = GLU && i >= OT ? (SEG ? p.segs_up[blockIdx.y].w : p.mat[MATS - 1].w) : w;
        const int64_t g = g0 + i % OT < groups ? g0 + i % OT : groups - 1;
        wb[i] = wi.codes + g * units * 1024;
        if constexpr (NS > 0) sb[i] = wi.side + side_row(wi, g, lane);
    }
    // fragment bases of the token blocks; lanes past the tokens repeat the
    // last one (each output row of the MFMA depends on its own token only)
    const uint8_t *xb[MT];
    uint32_t xo[MT];
    if constexpr (NX == 0) {
        const int64_t nblk = (p.n + 15) / 16;
#pragma unroll
        for (int m = 0; m < MT; m++) {
            int64_t blk = (int64_t)tb * MT + m;
            blk = blk < nblk ? blk : nblk - 1;
            const int cnt = (int)(p.n - 16 * blk < 16 ? p.n - 16 * blk : 16);
            xb[m] = p.xs + blk * p.ldk * XT * 1024;
            xo[m] = (uint32_t)((kq * 16 + (c16 < cnt ? c16 : cnt - 1)) * 16);
        }
    }

    const float *xr[SEG ? NX / 2 : 1];
    if constexpr (SEG) {
#pragma unroll
        for (int m = 0; m < NX / 2; m++) {
            const int64_t tok = 2 * m + (lane >> 5), r = off + (tok < n ? tok : n - 1);
            xr[m] = p.x + (p.row_index ? (int64_t)p.row_index[r] : r) * p.ldx;
        }
    }

    typedef FewSet<TF, MT, NT, XT, NX> Set;
    auto fetch = [&](Set &v, int s) __attribute__((always_inline)) {
        if constexpr (NX == 1) {
            const int64_t k = (int64_t)s * 128 + 2 * lane;
            v.x1 = gload<float2>(p.x + (k < K ? k : K - 2));
        } else if constexpr (NX > 1) {
            const int64_t k = (int64_t)s * 128 + 4 * (lane & 31), kc = k < K ? k : K - 4;
#pragma unroll
            for (int m = 0; m < NX / 2; m++) {
                const int64_t tok = 2 * m + (lane >> 5);
                if constexpr (SEG) v.xp[m] = gload<float4>(xr[m] + kc);
                else v.xp[m] = gload<float4>(p.x + (off + (tok < n ? tok : n - 1)) * p.ldx + kc);
            }
        }
#pragma unroll
        for (int i = 0; i < NT; i++) {
#pragma unroll
            for (int j = 0; j < UPS; j++) {
                int64_t u = (int64_t)s * UPS + j;
                u = u < units ? u : units - 1;
                v.raw[i][j] = gload<u32x4>(wb[i] + u * 1024 + woff);
                if constexpr (TF == TF_Q8) v.side[i][j] = gload<uint32_t>(sb[i] + u * 16);
                if constexpr (TF == TF_FP8)
                    v.side[i][j] = gload<uint32_t>(sb[i] + (st.sh >= 0 ? (uint32_t)u >> st.sh : (uint32_t)u / st.per));
            }
            if constexpr (TF == TF_MX4) v.side[i][0] = gload<uint32_t>(sb[i] + s);
            if constexpr (TF == TF_INT4) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t u = 2u * s + j;
                    uint32_t c = st.sh >= 0 ? u >> st.sh : u / st.per;
                    c = c < (uint32_t)w.side_cols ? c : (uint32_t)w.side_cols - 1;  // the step's half past K
                    v.side[i][j] = gload<uint32_t>(sb[i] + c);
                }
            }
        }
        if constexpr (NX == 0) {
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < 4; t++)
#pragma unroll
                    for (int e = 0; e < XT; e++)
                        v.xa[m][t][e] = gload<u32x4>(xb[m] + (((int64_t)s * 4 + t) * XT + e) * 1024 + xo[m]);
        }
    };

    floatx4 acc[MT][NT];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < NT; i++) acc[m][i] = floatx4{0.f, 0.f, 0.f, 0.f};

    u32x4 *slot = lds + wave * Slot::WORDS;
    auto compute = [&](Set &v, int s) __attribute__((always_inline)) {
        // the wave's own slot: its LDS accesses complete in order, no barrier
        if constexpr (NX == 1) {
            const bool in = (int64_t)s * 128 + 2 * lane < K;
            float a = in ? v.x1.x : 0.f, b = in ? v.x1.y : 0.f;
            uint32_t *d = (uint32_t *)slot + lane;  // (k tile lane / 16, quarter lane / 4 % 4, pair lane % 4)
#pragma unroll
            for (int e = 0; e < XT; e++) d[e * Slot::ES * 4] = next_term(a, b);
        } else if constexpr (NX > 1) {
            const int c = lane & 31;
            const bool in = (int64_t)s * 128 + 4 * c < K;
            uint2 *d = (uint2 *)(slot + (c >> 3) * Slot::TS + (c >> 1 & 3) * Slot::QS + (lane >> 5)) + (c & 1);
#pragma unroll
            for (int m = 0; m < NX / 2; m++) {
                float4 a = v.xp[m];
                if (!in) a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                for (int e = 0; e < XT; e++) {
                    const uint32_t lo = next_term(a.x, a.y);
                    d[(e * Slot::ES + 2 * m) * 2] = make_uint2(lo, next_term(a.z, a.w));
                }
            }
        }
#pragma unroll
        for (int j = 1; j < UPS; j++)
            if ((int64_t)s * UPS + j >= units) {  // past the matrix: zero weights
#pragma unroll
                for (int i = 0; i < NT; i++) {
                    v.raw[i][j] = u32x4{0, 0, 0, 0};
                    if constexpr (TF == TF_Q8 || TF == TF_FP8) v.side[i][j] = 0;
                }
            }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            u32x4 xa[MT][XT];
            if constexpr (NX > 0) {
#pragma unroll
                for (int e = 0; e < XT; e++)
                    xa[0][e] = slot[e * Slot::ES + t * Slot::TS + kq * Slot::QS + (c16 < NX ? c16 : NX - 1)];
            } else {
#pragma unroll
                for (int m = 0; m < MT; m++)
#pragma unroll
                    for (int e = 0; e < XT; e++) xa[m][e] = v.xa[m][t][e];
            }
            constexpr int TU = 4 / UPS;  // k tiles of a unit
            const int j = t / TU;
#pragma unroll
            for (int i = 0; i < NT; i++) {
                u32x4 b;
                float ts = 1.f;
                if constexpr (TF == TF_BF16) b = v.raw[i][j];
                else {
                    const u32x4 c[1] = {v.raw[i][j]};
                    const uint32_t sd[2] = {v.side[i][UPS > 1 ? j : 0], v.side[i][UPS > 1 ? j : Few<TF>::NSA - 1]};
                    b = decode_tile_lds<TF>(w, c, sd, t % TU, true);
                    if constexpr (TF == TF_Q8) ts = f16_to_f32_hw((uint16_t)((sd[0] >> (16 * (t % TU))) & 0xffffu));
                }
#pragma unroll
                for (int m = 0; m < MT; m++) mac<TF, XT>(acc[m][i], xa[m], b, b, ts);
            }
        }
    };

    if (s0 < s1) {
        Set a, b;
        fetch(a, s0);
        int s = s0;
        for (; s + 1 < s1; s += 2) {
            fetch(b, s + 1);
            compute(a, s);
            fetch(a, s + 2 < s1 ? s + 2 : s1 - 1);
            compute(b, s + 1);
        }
        if (s < s1) compute(a, s);
    }

    // the W slices added in wave order, a (token block, row group) tile a wave
    floatx4 *red = (floatx4 *)lds;
    __syncthreads();  // the slots are read: their LDS takes the sums
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < NT; i++) red[(wave * MT * NT + m * NT + i) * 64 + lane] = acc[m][i];
    __syncthreads();
    auto total = [&](int q) {  // tile q's slices, in wave order
        floatx4 v = red[q * 64 + lane];
#pragma unroll
        for (int k = 1; k < W; k++) {
            const floatx4 o = red[(k * MT * NT + q) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = __fadd_rn(v[r], o[r]);
        }
        return v;
    };
    if constexpr (GLU) {
        __shared__ float turn[W][16][17];  // a wave's tile, [token][row]
        for (int q = wave; q < MT * OT; q += W) {
            const int m = q / OT, i = q % OT;
            const floatx4 g = total(m * NT + i), u = total(m * NT + OT + i);
            const int64_t blk = (int64_t)tb * MT + m, row = (g0 + i) * 16 + c16;
            floatx4 v;
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = row < w.rows ? __fmul_rn(act_apply(p.act, g[r]), u[r]) : 0.f;
            if (p.y) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int64_t tok = blk * 16 + 4 * kq + r;
                    if (tok < n && row < w.rows) p.y[(off + tok) * w.rows + row] = v[r];
                }
            }
            if (p.ys) {
                // turned in the wave's own LDS (accesses in order): lane = token
                // lane % 16, the tile's columns 8 (lane / 16) .. +8
#pragma unroll
                for (int r = 0; r < 4; r++) turn[wave][4 * kq + r][c16] = v[r];
                __builtin_amdgcn_wave_barrier();
                const int64_t k0 = (g0 + i) * 16 + 8 * kq;
                if (lane < 32 && blk * 16 + c16 < p.n && k0 < w.rows) {
                    float f[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) f[j] = turn[wave][c16][8 * kq + j];
                    u32x4 t[2];
                    a_words_cvt<2>(f, t);
                    u32x4 *d = (u32x4 *)p.ys + (blk * p.ldk_y + k0 / 32) * 128 + k0 % 32 / 8 * 16 + c16;
                    d[0] = t[0];
                    d[64] = t[1];
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        return;
    }
    GemmParams e{};
    e.w.rows = w.rows;
    e.n = n;
    if constexpr (SEG) {
        e.out = p.out + off * w.rows;
        e.delta_b = seg->delta_b;
        e.delta_xa = p.delta_xa + off * p.delta_stride;
        e.delta_rank = seg->delta_rank;
        e.delta_stride = p.delta_stride;
    } else {
        e.out = mat.out + off * w.rows;
        e.bias = mat.bias;
        e.accumulate = mat.accumulate;
        e.delta_b = mat.delta_b;
        e.delta_xa = mat.delta_xa + off * mat.delta_rank;
        e.delta_rank = e.delta_stride = mat.delta_rank;
    }
    for (int q = wave; q < MT * NT; q += W) {
        floatx4 v[1][1] = {{total(q)}};
        const int64_t tok[1] = {((int64_t)tb * MT + q / NT) * 16 + 4 * kq}, row[1] = {(g0 + q % NT) * 16 + c16};
        store_block(e, tok, row, v);
    }
}

struct FewCall {
    const FewMat *mats;
    int nmat;
    const float *x;
    int64_t ldx;
    const void *xs;
    int64_t ldk, n;
    hipStream_t s;
    uint32_t act = 0;
    float *y = nullptr;
    void *ys = nullptr;
    int64_t ldk_y = 0;
};

template <int TF, int MT, int NT, int W, int XT, int NX, int MATS, bool GLU>
void launch_mats(const FewCall &c) {
    FewParams<MATS> p{};
    int end = 0;
    for (int i = 0; i < MATS; i++) {
        if (i < c.nmat) {
            p.mat[i] = c.mats[i];
            if (!GLU || i == 0) end += (int)((c.mats[i].w.rows + 16 * NT - 1) / (16 * NT));
        }
        p.end[i] = end;
    }
    p.y = c.y;
    p.ys = (uint8_t *)c.ys;
    p.ldk_y = c.ldk_y;
    p.act = c.act;
    p.tblocks = NX ? (int)((c.n + NX - 1) / NX) : (int)((c.n + 16 * MT - 1) / (16 * MT));
    p.x = c.x;
    p.xs = (const uint8_t *)c.xs;
    p.n = c.n;
    p.ldx = c.ldx;
    p.ldk = c.ldk;
    hipLaunchKernelGGL((few_kernel<TF, MT, NT, W, XT, NX, MATS, GLU>), dim3((unsigned)(end * p.tblocks)), dim3(64 * W), 0,
                       c.s, p);
}

template <int TF, int MT, int NT, int W, int XT, int NX>
void launch_cfg(const FewCall &c) {
    if (c.nmat == 1) launch_mats<TF, MT, NT, W, XT, NX, 1, false>(c);
    else if constexpr (XT == 2) launch_mats<TF, MT, NT, W, XT, NX, 3, false>(c);
}

// Gate and up: half the row groups of a matrix of their rows together
template <int TF, int MT, int NT, int W, int NX>
void launch_glu_cfg(const FewCall &c) {
    launch_mats<TF, MT, NT, W, 2, NX, 2, true>(c);
}
template <int TF, int NX>
void launch_glu_rows(const FewCall &c, int64_t groups, int64_t steps) {
    if (groups >= 512 || steps <= 8) launch_glu_cfg<TF, 1, 1, 4, NX>(c);
    else launch_glu_cfg<TF, 1, 1, 8, NX>(c);
}
template <int TF>
void launch_glu(const FewCall &c) {
    const int64_t groups = 2 * ((c.mats[0].w.rows + 15) / 16), steps = (c.mats[0].w.cols + 127) / 128, tb = (c.n + 15) / 16;
    if (c.x) {
        if (c.n == 1) launch_glu_rows<TF, 1>(c, groups, steps);
        else if (c.n == 2) launch_glu_rows<TF, 2>(c, groups, steps);
        else if (c.n <= 4) launch_glu_rows<TF, 4>(c, groups, steps);
        else launch_glu_rows<TF, 8>(c, groups, steps);
        return;
    }
    // the plain product's lines (launch_tf) for the two matrices together
    const int64_t units = groups * tb;
    if (units <= 256 && steps > 16) launch_glu_cfg<TF, 1, 1, 8, 0>(c);
    else if (tb == 1 || units < 640) launch_glu_cfg<TF, 1, 1, 4, 0>(c);
    else if (units < 1536 || TF == TF_FP8) launch_glu_cfg<TF, 2, 1, 4, 0>(c);
    else launch_glu_cfg<TF, 2, 2, 4, 0>(c);
}

template <int TF, int XT, int NX>
void launch_rows(const FewCall &c, int64_t groups, int64_t steps) {
    // 32 rows and four K slices where that gives at least 256 workgroups
    // (14336 x 4096 on 8 tokens: MXFP4 12.0 us, 14.8 to 15.4 with 16 rows);
    // below that 16 rows, and eight slices of more than one step each (FP8
    // 4096 x 14336 on 8 tokens 17.4 us, 16 slices 16.6, four 24; 896 x 896
    // 4.7, four slices 4.4)
    if (groups >= 512) launch_cfg<TF, 1, 2, 4, XT, NX>(c);
    else if (steps > 8) launch_cfg<TF, 1, 1, 8, XT, NX>(c);
    else launch_cfg<TF, 1, 1, 4, XT, NX>(c);
}

// The tile of a product from fragments: token blocks x row groups.
// Few row groups x token blocks: eight K slices over 16 rows (1024 x 4096
// on 16 tokens: FP8 8.6 us, 10.3 with four over 32). Otherwise every
// weight decoded feeds MT token blocks and every activation word NT row
// groups; the larger tiles pay once the grid still fills the CUs (4096 x
// 4096: MXFP4 on 48 tokens 13.0 us with 2 x 2, 15.0 with 1 x 2; on 96
// tokens 19.1 with 2 x 4, 20.7; 14336 x 4096 on 16 tokens 15.4 with 1 x 2,
// 19.6 with 2 x 2; FP8 on 128 tokens 55 us with 2 x 2, 66 with 2 x 4).
// Three-term products hold half as many again.
enum FewTile { FT_1x1, FT_1x2, FT_2x2, FT_2x4 };
FewTile few_tile(int tf, int xt, int64_t groups, int64_t steps, int64_t tb) {
    const int64_t units = groups * tb;
    if (units <= 256 && steps > 16) return FT_1x1;
    if (xt == 3 || tb == 1 || units < 640) return FT_1x2;
    return units < 1536 || tf == TF_FP8 ? FT_2x2 : FT_2x4;
}

template <int TF, int XT>
void launch_tf(const FewCall &c) {
    int64_t groups = 0;
    for (int i = 0; i < c.nmat; i++) groups += (c.mats[i].w.rows + 15) / 16;
    const int64_t steps = (c.mats[0].w.cols + 127) / 128, tb = (c.n + 15) / 16;
    if (c.x) {
        if (c.n == 1) launch_rows<TF, XT, 1>(c, groups, steps);
        else if (c.n == 2) launch_rows<TF, XT, 2>(c, groups, steps);
        else if (c.n <= 4) launch_rows<TF, XT, 4>(c, groups, steps);
        else launch_rows<TF, XT, 8>(c, groups * ((c.n + 7) / 8), steps);
        return;
    }
    switch (few_tile(TF, XT, groups, steps, tb)) {
    case FT_1x1: launch_cfg<TF, 1, 1, 8, XT, 0>(c); break;
    case FT_1x2: launch_cfg<TF, 1, 2, 4, XT, 0>(c); break;
    case FT_2x2:
        if constexpr (XT == 2) launch_cfg<TF, 2, 2, 4, XT, 0>(c);
        break;
    case FT_2x4:
        if constexpr (XT == 2 && TF != TF_FP8) launch_cfg<TF, 2, 4, 4, XT, 0>(c);
        break;
    }
}

// 16 rows and four K slices a workgroup: the segments fill the CUs
template <int TF, int NX, bool GLU>
void launch_segs_nx(const FewParams<1> &q, int64_t groups, unsigned nseg, int64_t max_cnt, hipStream_t s) {
    hipLaunchKernelGGL((few_kernel<TF, 1, 1, 4, 2, NX, 1, GLU, true>), dim3((unsigned)groups, nseg, (unsigned)((max_cnt + NX - 1) / NX)),
                       dim3(256), 0, s, q);
}
template <int TF, bool GLU>
void launch_segs(const FewParams<1> &q, int64_t groups, unsigned nseg, int64_t max_cnt, hipStream_t s) {
    if (max_cnt <= 2) launch_segs_nx<TF, 2, GLU>(q, groups, nseg, max_cnt, s);
    else if (max_cnt <= 4) launch_segs_nx<TF, 4, GLU>(q, groups, nseg, max_cnt, s);
    else launch_segs_nx<TF, 8, GLU>(q, groups, nseg, max_cnt, s);
}
template <bool GLU>
void launch_segs_tf(int tf, const FewParams<1> &q, int64_t rows, unsigned nseg, int64_t max_cnt, hipStream_t s) {
    const int64_t groups = (rows + 15) / 16;
    switch (tf) {
    case TF_BF16: launch_segs<TF_BF16, GLU>(q, groups, nseg, max_cnt, s); break;
    case TF_Q8: launch_segs<TF_Q8, GLU>(q, groups, nseg, max_cnt, s); break;
    case TF_FP8: launch_segs<TF_FP8, GLU>(q, groups, nseg, max_cnt, s); break;
    case TF_MX4: launch_segs<TF_MX4, GLU>(q, groups, nseg, max_cnt, s); break;
    case TF_INT4: launch_segs<TF_INT4, GLU>(q, groups, nseg, max_cnt, s); break;
    default: throw Error{DITCH_UNSUPPORTED, "few-token segments: format"};
    }
    DITCH_TRY_HIP(hipGetLastError());
}

}  // namespace

// A call's time by its rounds of 256 workgroups, each an epilogue and a chain
// over K: us a round, and a round and 1024 columns by tile, fitted to 3 900
// calls of 33 to 255 tokens on 80 shapes of 256 to 32768 rows and 256 to 16384
// columns (median error 6 %, MXFP4 from 128 tokens on with three terms).
static double few_us(const TileView &w, int64_t rows, int64_t n, int xt) {
    struct Cost {
        double round, k[4];
    };
    static constexpr Cost bf16{1.6, {1.2, 1.36, 1.9, 3.65}}, q8{2.2, {1.2, 1.2, 1.9, 3.35}}, fp8{0.7, {1.0, 1.3, 1.8, 0}},
        mx4{0.3, {1.0, 1.1, 1.65, 2.45}}, mx4x3{0, {1.6, 1.56, 0, 0}}, int4{0.9, {1.15, 1.6, 2.07, 3.6}};
    static constexpr int MT[4] = {1, 1, 2, 2}, NT[4] = {1, 2, 2, 4};
    const Cost &c = w.tf == TF_BF16 ? bf16 : w.tf == TF_Q8 ? q8 : w.tf == TF_FP8 ? fp8 : w.tf == TF_INT4 ? int4
                    : xt == 3 ? mx4x3 : mx4;
    const int64_t groups = (rows + 15) / 16, tb = (n + 15) / 16;
    const FewTile t = few_tile(w.tf, xt, groups, (w.cols + 127) / 128, tb);
    const int64_t wgs = ((groups + NT[t] - 1) / NT[t]) * ((tb + MT[t] - 1) / MT[t]), rounds = (wgs + 255) / 256;
    return 5.8 - c.round + rounds * (c.round + c.k[t] * w.cols / 1024.0);
}

// Up to 32 tokens every shape but the tallest from 17 on, whose many rounds'
// epilogues outweigh a short K. us here / there, 17 to 31 tokens: bf16 65536 x
// 256 17 / 12, 131072 x 512 41 / 30, 65536 x 512 24 / 25, 65536 x 896 33 / 39;
// Q8_0 131072 x 256 32 / 20, 131072 x 512 39 / 36. 32 tokens, bf16: 65536 x 896
// 34 / 26, 65536 x 4096 136 / 112, 32768 x 896 21 / 23.
// Above 32 where it is ahead of the tiled, scaled-MFMA or mid-batch product by
// the two estimates. Those multiply at twice the rate and more but leave CUs
// idle or pass partial sums through memory on few tokens, so this kernel wins
// while its grid is one round of the CUs, and loses from two (long K) to five
// (short K) rounds on. us here / there: bf16 4096 x 4096 on 128 tokens (one
// round) 20 / 25, on 160 (two) 34 / 34; 16384 x 256 on 64 (two) 9.8 / 11.4, on
// 255 (eight) 27 / 14; 1024 x 14336 on 255 (two) 38 / 44, 4112 x 8192 on 48
// (two) 36 / 29; INT4 16384 x 256 on 160 (five) 16.1 / 16.6. Of 5 850 calls on
// 90 shapes eleven are 7 to 15 % behind the product that runs otherwise (by
// lines in tokens x rows x columns alone 300 of 3 700 were, up to 2.2 times).
static bool few_form(const TileView &w, int64_t n) {
    return w.fast && n >= 1 && n <= 255 && w.cols >= 4 &&
           (w.tf == TF_BF16 || w.tf == TF_MX4 || w.tf == TF_Q8 || w.tf == TF_FP8 || w.tf == TF_INT4);
}
bool few_gemm_takes(const TileView &w, int64_t n, bool exact) {
    if (!few_form(w, n)) return false;
    if (n <= 32) {
        if (exact || n <= 16 || w.rows < 65536) return true;
        return w.tf == TF_BF16 ? n < 32 && w.cols > 512 : w.tf != TF_Q8 || w.cols > 256;
    }
    return !exact && few_us(w, w.rows, n, mx_gemm_takes(w, n) ? 3 : 2) <= 1.02 * large_gemm_us(w, n);
}

// Several matrices in one launch share its rounds and its fragments, which their
// producer writes: above 32 tokens one estimate for all of them against the sum
// of theirs and what the launch saves besides. Matrix by matrix, some went one
// way and some the other: two layers of 896 x 4864 Q8_0 on 40 tokens 104 us with
// all here, 133 mixed; of 4096 x 14336 bf16 350 and 402.
bool few_launch_takes(const TileView *const *w, int count, int64_t n, double saved_us) {
    int64_t rows = 0;
    double other = saved_us;
    for (int i = 0; i < count; i++) {
        if (!few_form(*w[i], n) || w[i]->tf != w[0]->tf || w[i]->cols != w[0]->cols) return false;
        if (n <= 32 && !few_gemm_takes(*w[i], n, false)) return false;
        rows += w[i]->rows;
        if (n > 32) other += large_gemm_us(*w[i], n);
    }
    return n <= 32 || few_us(*w[0], rows, n, 2) <= other;
}

bool few_reads_rows(const TileView &w, int64_t n, const float *x, int64_t ldx) {
    return n <= 32 && w.cols % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0;
}

void launch_few_gemm(const FewMat *mats, int nmat, const float *x, int64_t ldx, const void *xs, int64_t ldk, int64_t n,
                     int xt, hipStream_t s) {
    const FewCall c{mats, nmat, x, ldx, xs, ldk, n, s};
    DITCH_CHECK(nmat >= 1 && nmat <= 3 && n >= 1 && (nmat == 1 || xt == 2), DITCH_INVALID_ARGUMENT,
                "few-token product: 1 to 3 matrices");
    for (int i = 0; i < nmat; i++)
        DITCH_CHECK(mats[i].w.tf == mats[0].w.tf && mats[i].w.cols == mats[0].w.cols && mats[i].w.fast,
                    DITCH_INVALID_ARGUMENT, "few-token product: matrices of one format and width");
    DITCH_CHECK(x ? few_reads_rows(mats[0].w, n, x, ldx) : xs && ldk >= few_ldk(mats[0].w), DITCH_INVALID_ARGUMENT,
                "few-token product: activations not in a form it reads");
#define FEW_TF(TF) \
    case TF: xt == 3 ? launch_tf<TF, 3>(c) : launch_tf<TF, 2>(c); break;
    switch (mats[0].w.tf) {
        FEW_TF(TF_BF16)
        FEW_TF(TF_Q8)
        FEW_TF(TF_FP8)
        FEW_TF(TF_MX4)
        FEW_TF(TF_INT4)
    default: throw Error{DITCH_UNSUPPORTED, "few-token product: format"};
    }
#undef FEW_TF
    DITCH_TRY_HIP(hipGetLastError());
}

bool few_glu_takes(const TileView &gate, const TileView &up, int64_t n) {
    const TileView *const mats[2] = {&gate, &up};  // (saves the down product's split and the activation's launch too)
    return gate.tf == up.tf && gate.rows == up.rows && gate.cols == up.cols && gate.units_k == up.units_k &&
           few_launch_takes(mats, 2, n, 2 * FEW_SPLIT_US + 5) &&
           gate.scale_type == up.scale_type && gate.group == up.group && gate.block_cols == up.block_cols &&
           gate.side_cols == up.side_cols;
}

void launch_few_glu(const TileView &gate, const TileView &up, uint32_t act, float *y, void *ys, int64_t ldk_y,
                    const float *x, int64_t ldx, const void *xs, int64_t ldk, int64_t n, hipStream_t s) {
    DITCH_CHECK(few_glu_takes(gate, up, n) && (y || ys) && (!ys || (gate.rows % 128 == 0 && ldk_y * 32 >= gate.rows)),
                DITCH_INVALID_ARGUMENT, "few-token gate/up: shapes or outputs");
    DITCH_CHECK(x ? n <= 8 && few_reads_rows(gate, n, x, ldx) : xs && ldk >= few_ldk(gate), DITCH_INVALID_ARGUMENT,
                "few-token gate/up: activations not in a form it reads");
    const FewMat mats[2] = {FewMat{gate, nullptr, nullptr, nullptr, nullptr, 0, 0}, FewMat{up, nullptr, nullptr, nullptr, nullptr, 0, 0}};
    FewCall c{mats, 2, x, ldx, xs, ldk, n, s};
    c.act = act;
    c.y = y;
    c.ys = ys;
    c.ldk_y = ldk_y;
    switch (gate.tf) {
    case TF_BF16: launch_glu<TF_BF16>(c); break;
    case TF_Q8: launch_glu<TF_Q8>(c); break;
    case TF_FP8: launch_glu<TF_FP8>(c); break;
    case TF_MX4: launch_glu<TF_MX4>(c); break;
    case TF_INT4: launch_glu<TF_INT4>(c); break;
    default: throw Error{DITCH_UNSUPPORTED, "few-token gate/up: format"};
    }
    DITCH_TRY_HIP(hipGetLastError());
}

// Experts of up to 8 rows, or of up to 32 where most have at most 8 (a chunk of
// 8 rows reads the weights again, from L2): us for gate/up and down of 128
// experts of 2048 x 768, here against the GEMV (20 tokens) and the tiled
// products: INT4 20 tokens 44 + 29 / 190 + 73, FP8 36 tokens 53 + 41 / 61 + 50,
// INT4 64 tokens (86 experts used, 1.3 chunks each) 87 + 61 / 119 + 55.
bool few_grouped_takes(const GroupSeg *segs, unsigned nseg, int64_t max_cnt) {
    if (nseg < 1 || nseg > 65535 || max_cnt > 32) return false;
    const TileView &f = segs[0].w;
    if (max_cnt > 8) {
        int64_t chunks = 0;
        for (unsigned i = 0; i < nseg; i++) chunks += (segs[i].cnt + 7) / 8;
        if (2 * chunks > 3 * (int64_t)nseg) return false;
    }
    for (unsigned i = 0; i < nseg; i++) {
        const TileView &w = segs[i].w;
        if (segs[i].cnt < 1 || segs[i].cnt > max_cnt || !few_gemm_takes(w, 1, false) || w.cols % 4 != 0 ||
            w.tf != f.tf || w.rows != f.rows || w.cols != f.cols)
            return false;
    }
    return true;
}

// (an expert's up is decoded by its gate's scale layout)
bool few_glu_grouped_takes(const GroupSeg *gate, const GroupSeg *up, unsigned nseg, int64_t max_cnt) {
    if (!few_grouped_takes(gate, nseg, max_cnt)) return false;
    for (unsigned i = 0; i < nseg; i++)
        if (!few_glu_takes(gate[i].w, up[i].w, 1)) return false;
    return true;
}

void launch_few_grouped(const GroupSeg *d_segs, const TileView &shape, unsigned nseg, int64_t max_cnt, float *out,
                        const float *x, const float *delta_xa, int delta_stride, hipStream_t s) {
    FewParams<1> q{};
    q.segs = d_segs;
    q.x = x;
    q.ldx = shape.cols;
    q.out = out;
    q.delta_xa = delta_xa;
    q.delta_stride = delta_stride;
    q.tblocks = 1;
    launch_segs_tf<false>(shape.tf, q, shape.rows, nseg, max_cnt, s);
}

void launch_few_glu_grouped(const GroupSeg *d_gate, const GroupSeg *d_up, const TileView &shape, unsigned nseg,
                            int64_t max_cnt, uint32_t act, float *y, const float *x, const int32_t *row_index,
                            hipStream_t s) {
    FewParams<1> q{};
    q.segs = d_gate;
    q.segs_up = d_up;
    q.x = x;
    q.ldx = shape.cols;
    q.row_index = row_index;
    q.y = y;
    q.act = act;
    q.tblocks = 1;
    launch_segs_tf<true>(shape.tf, q, shape.rows, nseg, max_cnt, s);
}

}  // namespace ditch
