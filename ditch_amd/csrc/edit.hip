// edit.hip — the rank-k weight edit in every row-normalisation mode, on the
// device (abliterate.computeDelta, abliterate.zig:223-350): `none`
// (A = V^T W, B = -lambda V), `pre` (row norms, A over the normalised rows,
// B scaled by the norms), `full` (the renormalised edit's delta approximated
// by a rank-r randomised SVD of the implicit operator D = diag(c) W +
// sum_l d_l a_l^T, abliterate.zig:282-349, 353-394, 473-538) and the optional
// input-side ablation (abliterate.zig:234-261).
//
// Every pass over W runs on the resident (re-tiled, still quantised) weight:
// row norms, W^T y for all vectors in one launch, and the exact three-term
// product W x for the q vectors of the SVD. The rest is q or k vectors of
// the matrix's width: up to 24 are orthonormalised over column chunks (wider
// sets by one workgroup), one workgroup runs the Jacobi eigen-solver of the
// q x q Gram matrix.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "internal.h"
#include "zig_random.h"

namespace ditch {

// ---------------------------------------------------------------------------
// helpers (blockDim.x a multiple of 64)

__device__ __forceinline__ double ed_wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ double ed_block_sum(double v, double *sh) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    v = ed_wave_sum(v);
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double r = 0.0;
    for (int w = 0; w < nw; w++) r += sh[w];
    return r;
}

// an f32 dot product accumulated in f64 and rounded once
__device__ float ed_dot(const float *a, const float *b, int64_t n, double *sh) {
    double acc = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc += (double)a[i] * (double)b[i];
    return (float)ed_block_sum(acc, sh);
}

// ---------------------------------------------------------------------------
// kernels

// vn[j][i] = v[j][i] / n_i (0 where n_i = 0)              (abliterate.zig:290-292)
__global__ void edit_vn_kernel(float *vn, const float *v, const float *norms, int64_t k, int64_t rows) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < k * rows; t += (int64_t)gridDim.x * blockDim.x) {
        const float n = norms[t % rows];
        vn[t] = n > 0.f ? __fdiv_rn(v[t], n) : 0.f;
    }
}

// b[i][j] = -lambda v[j][i] (x n_i for `pre`)        (abliterate.zig:275-278, 298-303)
__global__ void edit_b_kernel(float *b, const float *v, const float *norms, int64_t k, int64_t rows, float weight,
                              int64_t ldb) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < k * rows; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = t / k, j = t % k;
        float x = __fmul_rn(-weight, v[j * rows + i]);
        if (norms) x = __fmul_rn(x, norms[i]);
        b[i * ldb + j] = x;
    }
}

// out[j][l] = dot(p_l, x_j) for p [np][len], x [nx][len]: one block per pair
__global__ __launch_bounds__(256) void edit_dots_kernel(float *out, const float *p, const float *x, int64_t np,
                                                        int64_t len) {
    __shared__ double sh[8];
    const int64_t j = blockIdx.y, l = blockIdx.x;
    const float d = ed_dot(p + l * len, x + j * len, len, sh);
    if (threadIdx.x == 0) out[j * np + l] = d;
}

// The full edit's per-row factors (abliterate.zig:318-330): with
// b_ij = -lambda v_ji, s_i^2 = 1 + sum_j (2 b_ij (W_i.a_j)/n_i + sum_l b_ij b_il
// G_jl), c_i = 1/s_i - 1, d_ji = n_i b_ij / s_i.
__global__ void edit_cd_kernel(float *c, float *d, const float *v, const float *norms, const float *wa,
                               const float *gram, int64_t k, int64_t rows, float weight) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += (int64_t)gridDim.x * blockDim.x) {
        const float n = norms[i];
        float s2 = 1.0f;
        for (int64_t j = 0; j < k; j++) {
            const float bij = __fmul_rn(-weight, v[j * rows + i]);
            const float wn_dot_a = n > 0.f ? __fdiv_rn(wa[j * rows + i], n) : 0.f;
            s2 = __fadd_rn(s2, __fmul_rn(__fmul_rn(2.0f, bij), wn_dot_a));
            for (int64_t l = 0; l < k; l++)
                s2 = __fadd_rn(s2, __fmul_rn(__fmul_rn(bij, __fmul_rn(-weight, v[l * rows + i])), gram[j * k + l]));
        }
        const float s = __fsqrt_rn(fmaxf(s2, 1e-12f));
        c[i] = __fsub_rn(__fdiv_rn(1.0f, s), 1.0f);
        for (int64_t j = 0; j < k; j++)
            d[j * rows + i] = __fdiv_rn(__fmul_rn(n, __fmul_rn(-weight, v[j * rows + i])), s);
    }
}

// D X: out[j][i] = (W x_j)_i c_i + sum_l dot(a_l, x_j) d_li (abliterate.zig:363-376)
__global__ void edit_apply_kernel(float *out, const float *c, const float *d, const float *ax, int64_t q, int64_t k,
                                  int64_t rows) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < q * rows; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = t / rows, i = t % rows;
        float o = __fmul_rn(out[t], c[i]);
        for (int64_t l = 0; l < k; l++) o = __fadd_rn(o, __fmul_rn(ax[j * k + l], d[l * rows + i]));
        out[t] = o;
    }
}

// cy[j][i] = c_i y_j[i]                                   (abliterate.zig:383-386)
__global__ void edit_scale_rows_kernel(float *cy, const float *y, const float *c, int64_t q, int64_t rows) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < q * rows; t += (int64_t)gridDim.x * blockDim.x)
        cy[t] = __fmul_rn(c[t % rows], y[t]);
}

// D^T Y: out[j][col] += sum_l dot(d_l, y_j) a_l[col]      (abliterate.zig:387-392)
__global__ void edit_applyT_kernel(float *out, const float *a, const float *dy, int64_t q, int64_t k, int64_t cols) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < q * cols; t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = t / cols, col = t % cols;
        float o = out[t];
        for (int64_t l = 0; l < k; l++) o = __fadd_rn(o, __fmul_rn(dy[j * k + l], a[l * cols + col]));
        out[t] = o;
    }
}

// abliterate.orthonormalize (abliterate.zig:409-423): modified Gram-Schmidt,
// two passes, every row normalised (zeroed at norm <= 1e-20). One block.
__global__ __launch_bounds__(1024) void edit_orthonormalize_kernel(float *vecs, int64_t q, int64_t n) {
    __shared__ double sh[16];
    for (int64_t i = 0; i < q; i++) {
        float *vi = vecs + i * n;
        for (int pass = 0; pass < 2; pass++)
            for (int64_t j = 0; j < i; j++) {
                const float *vj = vecs + j * n;
                const float p = ed_dot(vi, vj, n, sh);
                for (int64_t t = threadIdx.x; t < n; t += blockDim.x) vi[t] = __fadd_rn(vi[t], __fmul_rn(-p, vj[t]));
                __syncthreads();
            }
        const float nrm = __fsqrt_rn(ed_dot(vi, vi, n, sh));
        const float s = nrm > 1e-20f ? __fdiv_rn(1.0f, nrm) : 0.f;
        for (int64_t t = threadIdx.x; t < n; t += blockDim.x) vi[t] = nrm > 1e-20f ? __fmul_rn(vi[t], s) : 0.f;
        __syncthreads();
    }
}

// The same Gram-Schmidt with the vector being orthonormalised held in
// registers (EPT elements a thread, element m * 1024 + tid): each step reads
// only v_j, whose successor is loaded before the step's reduction, and each
// reduction takes one barrier that waits on LDS alone (the wave sums
// alternate between two LDS slots, so a fast wave cannot overwrite sums a
// slow wave is still reading). Per element the arithmetic is the kernel
// above's: f64 dot rounded to f32, then v_i + (-p) v_j rounded twice.
template <int CTRL>
__device__ __forceinline__ double ed_dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// the sum of a wave's 64 values, the same in every lane: DPP butterflies
// within each row of 16 lanes (quad swaps, half-row and row mirrors), then
// the four row sums read as scalars
__device__ __forceinline__ double ed_wave_total(double v) {
    v += ed_dpp<0xB1>(v);
    v += ed_dpp<0x4E>(v);
    v += ed_dpp<0x141>(v);
    v += ed_dpp<0x140>(v);
    double r = 0.0;
#pragma unroll
    for (int row = 0; row < 4; row++)
        r += __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 16 * row),
                              __builtin_amdgcn_readlane(__double2loint(v), 16 * row));
    return r;
}

__device__ __forceinline__ void ed_lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int EPT>
__global__ __launch_bounds__(1024) void edit_orth_reg_kernel(float *vecs, int64_t q, int64_t n) {
    __shared__ double sh[2][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int slot = 0;
    auto block_dot = [&](const float *a, const float *b) -> float {
        double acc = 0.0;
#pragma unroll
        for (int m = 0; m < EPT; m++) acc += (double)a[m] * (double)b[m];
        acc = ed_wave_total(acc);
        if (lane == 0) sh[slot][wave] = acc;
        ed_lds_barrier();
        double r = 0.0;
#pragma unroll
        for (int w = 0; w < 16; w++) r += sh[slot][w];
        slot ^= 1;
        return (float)r;
    };
    auto load = [&](float *dst, const float *src) {
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int64_t t = (int64_t)m * 1024 + tid;
            dst[m] = t < n ? src[t] : 0.f;
        }
    };
    for (int64_t i = 0; i < q; i++) {
        float *vi_g = vecs + i * n;
        float vi[EPT], vj[EPT], vn[EPT];
        load(vi, vi_g);
        if (i > 0) load(vj, vecs);
        for (int pass = 0; pass < 2; pass++)
            for (int64_t j = 0; j < i; j++) {
                const int64_t nj = j + 1 < i ? j + 1 : (pass == 0 ? 0 : -1);
                if (nj >= 0) load(vn, vecs + nj * n);
                const float p = block_dot(vi, vj);
#pragma unroll
                for (int m = 0; m < EPT; m++) vi[m] = __fadd_rn(vi[m], __fmul_rn(-p, vj[m]));
                if (nj >= 0) {
#pragma unroll
                    for (int m = 0; m < EPT; m++) vj[m] = vn[m];
                }
            }
        const float nrm = __fsqrt_rn(block_dot(vi, vi));
        const float s = nrm > 1e-20f ? __fdiv_rn(1.0f, nrm) : 0.f;
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int64_t t = (int64_t)m * 1024 + tid;
            if (t < n) vi_g[t] = nrm > 1e-20f ? __fmul_rn(vi[m], s) : 0.f;
        }
        __syncthreads();  // v_i (global) is read by the later vectors
    }
}

// ---------------------------------------------------------------------------
// Orthonormalisation of few vectors (q <= ED_GRAM_Q) in three short launches
// over column chunks, instead of one workgroup's 2 q^2 dot products in a row
// (10 vectors: 67 us at 896 columns and 100 at 4864, all of it barriers and
// f64 latency). Gram-Schmidt needs only the inner products: a launch leaves
// every chunk's part of the f64 Gram matrix, the next adds the parts, factors
// the Gram matrix (each workgroup the same small Cholesky, whose rows are the
// projections of Gram-Schmidt in f64), applies it to its own columns with one
// rounding an element, and leaves the parts of the new Gram matrix; the third
// does that pass again, which takes the orthogonality from eps * cond to eps
// as the second Gram-Schmidt pass does. A vector that depends on the earlier
// ones to f32 rounding (its remainder at most 1e-7 of it) or whose norm is at
// most 1e-20 is zero and projects nothing; NaN and infinite vectors too.
// The neighbours ride along: the operator's second half on the product the
// chunk is read from (`scale`, `u`), the dot products the next half needs and
// the row-scaled copy it multiplies (`pa`, `cy`).
// 6 to 9 us a launch (latency: the parts, the factorisation, the columns); each
// of the 13 orthonormalisations of an 896 x 4864 edit took 67 to 100 us, and 12
// to 20 us of neighbours.
constexpr int ED_GRAM_Q = 24;  // vectors: LDS for a 256-column chunk and the parts
constexpr int ED_GRAM_K = 8;   // directions of the neighbours
struct OrthArgs {
    float *v;  // [q][n], in place
    int64_t n;
    int q, k, chunk;
    // before: v = v * scale[col] + sum_l (sum of dots_in)[j][l] u[l][col]
    const float *scale, *u;
    const double *dots_in;
    int dots_parts;
    const double *gram_in;  // [chunks][pairs]: orthonormalise by this Gram matrix
    double *gram_out;       // parts of the resulting vectors' Gram matrix
    // after: parts of dot(pa_l, v_j) [chunks][q k], cy = cs[col] v
    const float *pa, *cs;
    double *dots_out;
    float *cy;
    int store;
};

// row and column of the p-th entry of a lower triangle (p below 2^20)
__device__ __forceinline__ void ed_pair(int p, int &i, int &j) {
    i = (int)((__fsqrt_rn(8.f * p + 1.f) - 1.f) * 0.5f);
    while (i * (i + 1) / 2 > p) i--;
    while ((i + 1) * (i + 2) / 2 <= p) i++;
    j = p - i * (i + 1) / 2;
}

__device__ __forceinline__ double ed_lane(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// QM: the vectors, rounded up to the instances below. A thread holds one
// column of every vector; the Cholesky is done by each wave that holds
// columns (lane i: row i), so its factors are scalars for the columns.
template <int QM>
__global__ __launch_bounds__(256) void edit_orth_chunk_kernel(OrthArgs a) {
    extern __shared__ double ed_sh[];
    const int q = a.q, k = a.k, ld = a.chunk + 1, pairs = q * (q + 1) / 2;
    const int np = pairs > q * k ? pairs : q * k;
    double *tmp = ed_sh;
    float *xl = (float *)(tmp + 4 * np), *pr = xl + q * ld;  // [q][ld], [k][ld]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t n = a.n, c0 = (int64_t)blockIdx.x * a.chunk, col = c0 + tid;
    const int nc = (int)(n - c0 < a.chunk ? n - c0 : a.chunk);
    const bool in = tid < nc;
    float x[QM];
#pragma unroll
    for (int j = 0; j < QM; j++) x[j] = in && j < q ? a.v[j * n + col] : 0.f;

    // parts [chunks][count] added by four waves, then in wave order
    auto add_parts = [&](const double *parts, int chunks, int count) {
        for (int p = lane; p < count; p += 64) {
            double r = 0.0;
#pragma unroll 8
            for (int b = wave; b < chunks; b += 4) r += parts[(int64_t)b * count + p];
            tmp[wave * np + p] = r;
        }
        __syncthreads();
    };
    auto part = [&](int p) { return tmp[p] + tmp[np + p] + tmp[2 * np + p] + tmp[3 * np + p]; };

    if (a.u) {
        const float sc = a.scale && in ? a.scale[col] : 1.f;
        add_parts(a.dots_in, a.dots_parts, q * k);
        if (a.scale) {
#pragma unroll
            for (int j = 0; j < QM; j++) x[j] = __fmul_rn(x[j], sc);
        }
        for (int l = 0; l < k; l++) {
            const float u = in ? a.u[l * n + col] : 0.f;
#pragma unroll
            for (int j = 0; j < QM; j++)
                if (j < q) x[j] = __fadd_rn(x[j], __fmul_rn((float)part(j * k + l), u));
        }
        __syncthreads();
    }
    if (a.gram_in) {
        add_parts(a.gram_in, (int)gridDim.x, pairs);
        if (wave * 64 < nc) {
            double row[QM], inv[QM];
            const int i = lane < q ? lane : q - 1;
#pragma unroll
            for (int j = 0; j < QM; j++) row[j] = j <= i ? part(i * (i + 1) / 2 + j) : 0.0;
            const double d0 = part(i * (i + 1) / 2 + i);
#pragma unroll
            for (int j = 0; j < QM; j++) {
                inv[j] = 0.0;
                if (j >= q) continue;
                const double r = ed_lane(row[j], j);
                const bool live = r > 1e-14 * ed_lane(d0, j) && r > 1e-40;
                double y = __builtin_amdgcn_rsq(r);
#pragma unroll
                for (int it = 0; it < 2; it++) y = y * (1.5 - 0.5 * r * y * y);
                inv[j] = live ? y : 0.0;
                row[j] = live ? row[j] * y : 0.0;
#pragma unroll
                for (int c = j + 1; c < QM; c++)
                    if (c < q) row[c] -= row[j] * ed_lane(row[j], c);
            }
            double xd[QM];
#pragma unroll
            for (int r = 0; r < QM; r++) {
                xd[r] = 0.0;
                if (r >= q) continue;
                double acc = (double)x[r];
#pragma unroll
                for (int j = 0; j < r; j++) acc -= ed_lane(row[j], r) * xd[j];
                x[r] = inv[r] > 0.0 ? (float)(acc * inv[r]) : 0.f;
                xd[r] = (double)x[r];
            }
        }
        __syncthreads();
    }
    if (in) {
        const float cs = a.cy ? a.cs[col] : 0.f;
#pragma unroll
        for (int j = 0; j < QM; j++)
            if (j < q) {
                if (a.store) a.v[j * n + col] = x[j];
                if (a.cy) a.cy[j * n + col] = __fmul_rn(cs, x[j]);
                xl[j * ld + tid] = x[j];
            }
        if (a.pa)
            for (int l = 0; l < k; l++) pr[l * ld + tid] = a.pa[l * n + col];
    }
    __syncthreads();
    // dot products of LDS rows over the chunk: a pair a lane, a quarter of the
    // columns a wave
    auto dots = [&](int count, bool gram, double *out) {
        for (int p = lane; p < count; p += 64) {
            int i, j;
            if (gram) ed_pair(p, i, j);
            else i = p / k, j = q + p % k;  // (the rows of pr follow those of x)
            double r = 0.0;
#pragma unroll 8
            for (int c = wave; c < nc; c += 4) r += (double)xl[i * ld + c] * (double)xl[j * ld + c];
            tmp[wave * np + p] = r;
        }
        __syncthreads();
        for (int p = tid; p < count; p += 256) out[(int64_t)blockIdx.x * count + p] = part(p);
        __syncthreads();
    };
    if (a.pa) dots(q * k, false, a.dots_out);
    if (a.gram_out) dots(pairs, true, a.gram_out);
}

// The same two passes by one workgroup, the vectors in registers: up to Q of
// at most 1024 EPT columns (an input-side ablation's, which have no neighbours).
// Bound by the launch and four barriers; three launches and their gaps took
// longer than the vector-by-vector kernels above, us an ablated edit with these,
// the three launches and here: 256 columns 2 directions 58 / 69 / 64, 3072
// columns 2 and 4 64 / 73 / 63 and 83 / 74 / 73; from 14336 columns on equal.
template <int Q, int EPT>
__global__ __launch_bounds__(1024) void edit_orth_small_kernel(float *v, int q, int64_t n) {
    constexpr int P = Q * (Q + 1) / 2;
    __shared__ double parts[16][P], gram[P];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float x[Q][EPT];
#pragma unroll
    for (int i = 0; i < Q; i++)
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int64_t t = (int64_t)m * 1024 + tid;
            x[i][m] = i < q && t < n ? v[i * n + t] : 0.f;
        }
    for (int pass = 0; pass < 2; pass++) {
#pragma unroll
        for (int i = 0; i < Q; i++)
#pragma unroll
            for (int j = 0; j <= i; j++) {
                if (i >= q) continue;
                double r = 0.0;
#pragma unroll
                for (int m = 0; m < EPT; m++) r += (double)x[i][m] * (double)x[j][m];
                r = ed_wave_total(r);
                if (lane == 0) parts[wave][i * (i + 1) / 2 + j] = r;
            }
        __syncthreads();
        if (tid < q * (q + 1) / 2) {
            double r = 0.0;
#pragma unroll
            for (int w = 0; w < 16; w++) r += parts[w][tid];
            gram[tid] = r;
        }
        __syncthreads();
        double l[Q][Q], inv[Q];  // the Cholesky factor, as edit_orth_chunk_kernel's
#pragma unroll
        for (int j = 0; j < Q; j++) {
            inv[j] = 0.0;
            if (j >= q) continue;
            const double d = gram[j * (j + 1) / 2 + j];
            double r = d;
#pragma unroll
            for (int c = 0; c < j; c++) r -= l[j][c] * l[j][c];
            double y = __builtin_amdgcn_rsq(r);
#pragma unroll
            for (int it = 0; it < 2; it++) y = y * (1.5 - 0.5 * r * y * y);
            inv[j] = r > 1e-14 * d && r > 1e-40 ? y : 0.0;
#pragma unroll
            for (int i = j + 1; i < Q; i++) {
                if (i >= q) continue;
                double g = gram[i * (i + 1) / 2 + j];
#pragma unroll
                for (int c = 0; c < j; c++) g -= l[i][c] * l[j][c];
                l[i][j] = inv[j] > 0.0 ? g * y : 0.0;
            }
        }
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            double xd[Q];
#pragma unroll
            for (int i = 0; i < Q; i++) {
                if (i >= q) continue;
                double acc = (double)x[i][m];
#pragma unroll
                for (int j = 0; j < i; j++) acc -= l[i][j] * xd[j];
                x[i][m] = inv[i] > 0.0 ? (float)(acc * inv[i]) : 0.f;
                xd[i] = (double)x[i][m];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < Q; i++)
#pragma unroll
        for (int m = 0; m < EPT; m++) {
            const int64_t t = (int64_t)m * 1024 + tid;
            if (i < q && t < n) v[i * n + t] = x[i][m];
        }
}

// SVD widths up to ED_LDS_Q keep the Jacobi's two q x q matrices in LDS;
// wider ones work on them in place in global memory.
constexpr int ED_LDS_Q = 128;

// abliterate.jacobiEigen (abliterate.zig:427-469): cyclic Jacobi in f32 on the
// q x q matrix m (in place: its diagonal ends as the eigenvalues),
// eigenvectors in the columns of vecs. One block. A sweep takes its pivots in
// rounds of n / 2 disjoint ones (a tournament: entry 0 stays, the others move
// on by one), whose rotations touch different rows and columns: the angles of
// a round together, then every column pair, then every row pair. One pivot at
// a time, a rotation's division and square root chain (0.35 us) came 45 times
// a sweep of 10 x 10; in rounds 9 times.
template <bool LDS>
__global__ __launch_bounds__(1024) void edit_jacobi_kernel(float *m_g, float *vecs_g, float2 *rot_g, int n) {
    extern __shared__ float ed_dyn[];
    __shared__ double sh[16];
    float *m = LDS ? ed_dyn : m_g, *vecs = LDS ? ed_dyn + n * n : vecs_g;
    const int half = (n + 1) / 2, ring = 2 * half - 1;  // odd n: one pivot of a round has no partner
    float2 *rot = LDS ? (float2 *)(ed_dyn + 2 * n * n) : rot_g;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int t = tid; t < n * n; t += nt) {
        if (LDS) m[t] = m_g[t];
        vecs[t] = (t / n == t % n) ? 1.f : 0.f;
    }
    __syncthreads();
    // the pivots (p < q) of pair i of a round; false: none
    auto pivot = [&](int round, int i, int &p, int &q) {
        const int a = i ? 1 + (round + i) % ring : 0, b = 1 + (round + ring - i) % ring;
        p = a < b ? a : b;
        q = a < b ? b : a;
        return q < n;
    };
    for (int sweep = 0; sweep < 50; sweep++) {
        double off = 0;
        for (int t = tid; t < n * n; t += nt)
            if (t / n != t % n) off += (double)m[t] * (double)m[t];
        off = ed_block_sum(off, sh);
        if (off < 1e-18) break;
        for (int round = 0; round < ring; round++) {
            __syncthreads();
            for (int i = tid; i < half; i += nt) {
                int p, q;
                float2 r = make_float2(1.f, 0.f);
                if (pivot(round, i, p, q)) {
                    const float apq = m[p * n + q];
                    if (!(fabsf(apq) < 1e-20f)) {
                        const float app = m[p * n + p], aqq = m[q * n + q];
                        const float theta = __fdiv_rn(__fsub_rn(aqq, app), __fmul_rn(2.0f, apq));
                        const float sg = theta > 0.f ? 1.f : theta < 0.f ? -1.f : 0.f;
                        const float t = __fdiv_rn(sg, __fadd_rn(fabsf(theta), __fsqrt_rn(__fadd_rn(__fmul_rn(theta, theta), 1.0f))));
                        const float tf = theta == 0.f ? 1.0f : t;
                        r.x = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fmul_rn(tf, tf), 1.0f)));
                        r.y = __fmul_rn(tf, r.x);
                    }
                }
                rot[i] = r;
            }
            __syncthreads();
            for (int t = tid; t < n * half; t += nt) {
                const int k = t % n, i = t / n;
                int p, q;
                if (!pivot(round, i, p, q)) continue;
                const float cs = rot[i].x, sn = rot[i].y;
                if (sn == 0.f && cs == 1.f) continue;
                const float akp = m[k * n + p], akq = m[k * n + q];
                m[k * n + p] = __fsub_rn(__fmul_rn(cs, akp), __fmul_rn(sn, akq));
                m[k * n + q] = __fadd_rn(__fmul_rn(sn, akp), __fmul_rn(cs, akq));
                const float vkp = vecs[k * n + p], vkq = vecs[k * n + q];
                vecs[k * n + p] = __fsub_rn(__fmul_rn(cs, vkp), __fmul_rn(sn, vkq));
                vecs[k * n + q] = __fadd_rn(__fmul_rn(sn, vkp), __fmul_rn(cs, vkq));
            }
            __syncthreads();
            for (int t = tid; t < n * half; t += nt) {
                const int k = t % n, i = t / n;
                int p, q;
                if (!pivot(round, i, p, q)) continue;
                const float cs = rot[i].x, sn = rot[i].y;
                if (sn == 0.f && cs == 1.f) continue;
                const float apk = m[p * n + k], aqk = m[q * n + k];
                m[p * n + k] = __fsub_rn(__fmul_rn(cs, apk), __fmul_rn(sn, aqk));
                m[q * n + k] = __fadd_rn(__fmul_rn(sn, apk), __fmul_rn(cs, aqk));
            }
        }
        __syncthreads();
    }
    __syncthreads();
    if (LDS)
        for (int t = tid; t < n * n; t += nt) {
            m_g[t] = m[t];
            vecs_g[t] = vecs[t];
        }
}

// The SVD's factors and the LoRA pair (abliterate.zig:514-547): eigenvalues
// sorted descending (a stable sort), s_t = sqrt(max(lambda, 0)), u_t = Q e,
// v_t = B^T e / s_t; a[t] = sqrt(s_t) v_t, b[i][t] = u_t[i] sqrt(s_t). A
// thread per row and column, a grid row per output component t (rank of them).
__global__ __launch_bounds__(256) void edit_svd_out_kernel(float *a, float *b, const float *evals_m,
                                                           const float *evecs, const float *qy, const float *bt,
                                                           int q, int64_t rows, int64_t cols, int64_t ldb,
                                                           int64_t b_off) {
    extern __shared__ float ed_dyn[];  // the q eigenvalues, then the q entries of the eigenvector
    float *ev = ed_dyn, *e = ed_dyn;
    __shared__ int src_s;
    const int t = blockIdx.y;
    for (int i = threadIdx.x; i < q; i += blockDim.x) ev[i] = evals_m[(int64_t)i * q + i];
    if (threadIdx.x == 0) src_s = t;
    __syncthreads();
    // component t's eigenvalue: t are larger, or equal and before it
    for (int i = threadIdx.x; i < q; i += blockDim.x) {
        int above = 0;
        for (int j = 0; j < q; j++) above += ev[j] > ev[i] || (ev[j] == ev[i] && j < i);
        if (above == t) src_s = i;
    }
    __syncthreads();
    const int src = src_s;
    const float lambda = fmaxf(ev[src], 0.f);
    __syncthreads();
    for (int i = threadIdx.x; i < q; i += blockDim.x) e[i] = evecs[(int64_t)i * q + src];
    __syncthreads();
    const float s = __fsqrt_rn(lambda);
    const float sq = __fsqrt_rn(fmaxf(s, 0.f));
    const float inv = s > 1e-12f ? __fdiv_rn(1.0f, s) : 0.f;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows) {
        float u = 0.f;
#pragma unroll 4
        for (int c = 0; c < q; c++) u = __fadd_rn(u, __fmul_rn(e[c], qy[c * rows + i]));
        b[i * ldb + b_off + t] = __fmul_rn(u, sq);
    }
    if (i < cols) {
        float v = 0.f;
#pragma unroll 4
        for (int c = 0; c < q; c++) v = __fadd_rn(v, __fmul_rn(e[c], bt[c * cols + i]));
        v = s > 1e-12f ? __fmul_rn(v, inv) : 0.f;
        a[t * cols + i] = __fmul_rn(sq, v);
    }
}

// B += B B^T-style Gram of q rows: g[i][j] = dot(x_i, x_j)
// (abliterate.zig:505-508) via edit_dots_kernel.

// ---------------------------------------------------------------------------
// host side

static int ed_grid(int64_t total) {
    int64_t g = (total + 255) / 256;
    return (int)(g < 1 ? 1 : g > 16384 ? 16384 : g);
}

// The full mode's random test matrix: the first n draws of
// Random.floatNorm(f32) from std.Random.DefaultPrng.init(seed), in the
// order the reference fills omega (abliterate.zig:474-479).
void edit_gaussian(float *out, size_t n, uint64_t seed) {
    ZigRandom rng(seed);
    for (size_t t = 0; t < n; t++) out[t] = rng.norm_f32();
}

int64_t edit_rank(int64_t rows, int64_t cols, int64_t k, int mode, int64_t lora_rank, int ablate) {
    int64_t r = k;
    if (mode == 2) {
        const int64_t rr = lora_rank > k ? lora_rank : k;
        int64_t q = 2 * rr + 4;
        q = q < rows ? q : rows;
        q = q < cols ? q : cols;
        r = rr < q ? rr : q;
    }
    return r + (ablate ? k : 0);
}

struct EditWork {
    DevBuf v, norms, vn, a, bp, wa, gram, c, d, omega, qy, qx, cy, dots, bbt, evecs, xs, xa, wu;
    DevBuf gram0, gram1, dpart0, dpart1, rot;
};

// b[i][0..r) = bp[i][0..r), b[i][r + j] = -lambda wu[j][i]  (abliterate.zig:252-257)
__global__ void edit_b_ablate_kernel(float *b, const float *bp, const float *wu, int64_t rows, int64_t r, int64_t k,
                                     float weight) {
    const int64_t rank = r + k;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < rows * rank;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = t / rank, j = t % rank;
        b[t] = j < r ? bp[i * r + j] : __fmul_rn(-weight, wu[(j - r) * rows + i]);
    }
}

static void edit_matmul(const TileView &w, float *out, const float *x, int64_t n, hipStream_t s, DevBuf *ws,
                        const float *delta_a = nullptr, const float *delta_b = nullptr, int delta_rank = 0,
                        float *xa = nullptr) {
    MatmulEpilogue ep;
    ep.exact = 1;  // three bf16 terms: the f32 products of tensor.matmulT
    if (delta_rank > 0) {
        launch_delta_xa(xa, x, delta_a, n, w.cols, delta_rank, s);
        ep.delta_b = delta_b;
        ep.delta_xa = xa;
        ep.delta_rank = delta_rank;
    }
    launch_matmul(w, out, x, n, ep, s, nullptr, ws);
}

// W^T y for q vectors
static void edit_matvecT(const TileView &w, float *out, const float *y, int64_t q, hipStream_t s) {
    launch_matvecT(out, w, y, q, s);
}

// columns a workgroup: 64 up to 4096 (enough workgroups), at most 256
static int orth_chunk(int64_t n) { return (int)(64 * std::min<int64_t>(4, (n + 4095) / 4096)); }
static int64_t orth_chunks(int64_t n) { return (n + orth_chunk(n) - 1) / orth_chunk(n); }
static bool orth_takes(int64_t q, int64_t k) { return q <= ED_GRAM_Q && k <= ED_GRAM_K; }

static void launch_orth_chunk(OrthArgs a, hipStream_t s) {
    a.chunk = orth_chunk(a.n);
    const int64_t pairs = (int64_t)a.q * (a.q + 1) / 2, np = std::max<int64_t>(pairs, (int64_t)a.q * a.k);
    const size_t lds = (size_t)(4 * np * 8 + (a.q + a.k) * (a.chunk + 1) * 4);
    DITCH_CHECK(lds <= 65536, DITCH_INVALID_ARGUMENT, "edit: too many vectors for the chunked orthonormalisation");
    const dim3 grid((unsigned)orth_chunks(a.n));
    if (a.q <= 4) hipLaunchKernelGGL(edit_orth_chunk_kernel<4>, grid, dim3(256), lds, s, a);
    else if (a.q <= 12) hipLaunchKernelGGL(edit_orth_chunk_kernel<12>, grid, dim3(256), lds, s, a);
    else hipLaunchKernelGGL(edit_orth_chunk_kernel<24>, grid, dim3(256), lds, s, a);
    DITCH_TRY_HIP(hipGetLastError());
}

// The three launches: `first` holds what is done before the first Gram matrix,
// `last` what follows the second pass (v, n, q and k are first's).
static void edit_orth_chunks(EditWork &W, OrthArgs first, OrthArgs last, hipStream_t s) {
    const int64_t parts = orth_chunks(first.n) * first.q * (first.q + 1) / 2;
    double *g0 = W.gram0.get<double>(parts), *g1 = W.gram1.get<double>(parts);
    OrthArgs mid{};
    mid.v = last.v = first.v;
    mid.n = last.n = first.n;
    mid.q = last.q = first.q;
    mid.k = last.k = first.k;
    first.gram_out = g0;
    first.store = first.u != nullptr;
    mid.gram_in = g0;
    mid.gram_out = g1;
    mid.store = 1;
    last.gram_in = g1;
    last.store = 1;
    launch_orth_chunk(first, s);
    launch_orth_chunk(mid, s);
    launch_orth_chunk(last, s);
}

static void edit_orth(EditWork &W, float *vecs, int64_t q, int64_t n, hipStream_t s) {
    if ((q <= 4 && n <= 4096) || (q <= 2 && n <= 8192)) {
        if (n <= 1024) hipLaunchKernelGGL((edit_orth_small_kernel<4, 1>), dim3(1), dim3(1024), 0, s, vecs, (int)q, n);
        else if (n <= 4096) hipLaunchKernelGGL((edit_orth_small_kernel<4, 4>), dim3(1), dim3(1024), 0, s, vecs, (int)q, n);
        else hipLaunchKernelGGL((edit_orth_small_kernel<2, 8>), dim3(1), dim3(1024), 0, s, vecs, (int)q, n);
        DITCH_TRY_HIP(hipGetLastError());
        return;
    }
    if (orth_takes(q, 0)) {
        OrthArgs a{};
        a.v = vecs;
        a.n = n;
        a.q = (int)q;
        edit_orth_chunks(W, a, OrthArgs{}, s);
        return;
    }
    const int64_t ept = (n + 1023) / 1024;
    if (ept <= 2)
        hipLaunchKernelGGL(edit_orth_reg_kernel<2>, dim3(1), dim3(1024), 0, s, vecs, q, n);
    else if (ept <= 4)
        hipLaunchKernelGGL(edit_orth_reg_kernel<4>, dim3(1), dim3(1024), 0, s, vecs, q, n);
    else if (ept <= 8)
        hipLaunchKernelGGL(edit_orth_reg_kernel<8>, dim3(1), dim3(1024), 0, s, vecs, q, n);
    else if (ept <= 16)
        hipLaunchKernelGGL(edit_orth_reg_kernel<16>, dim3(1), dim3(1024), 0, s, vecs, q, n);
    else if (ept <= 24)
        hipLaunchKernelGGL(edit_orth_reg_kernel<24>, dim3(1), dim3(1024), 0, s, vecs, q, n);
    else  // vectors above 24 576 elements: the global-memory form
        hipLaunchKernelGGL(edit_orthonormalize_kernel, dim3(1), dim3(1024), 0, s, vecs, q, n);
    DITCH_TRY_HIP(hipGetLastError());
}

static void edit_jacobi(EditWork &W, float *m, float *vecs, int64_t q, hipStream_t s) {
    DITCH_CHECK(q <= 46340, DITCH_UNSUPPORTED, "edit: SVD width above 46340");
    const int64_t items = q * ((q + 1) / 2);  // (row, pair) updates of a round
    const dim3 block((unsigned)std::min<int64_t>(1024, (items + 63) / 64 * 64));
    if (q <= ED_LDS_Q) {
        static const bool attr = [] {
            return hipFuncSetAttribute((const void *)edit_jacobi_kernel<true>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       2 * ED_LDS_Q * ED_LDS_Q * 4 + ED_LDS_Q * 8) == hipSuccess;
        }();
        DITCH_CHECK(attr, DITCH_DEVICE_FAILED, "edit: the Jacobi kernel's LDS size was refused");
        hipLaunchKernelGGL(edit_jacobi_kernel<true>, dim3(1), block, (size_t)(2 * q * q * 4 + (q + 1) * 4), s, m, vecs,
                           (float2 *)nullptr, (int)q);
    } else {
        hipLaunchKernelGGL(edit_jacobi_kernel<false>, dim3(1), block, 0, s, m, vecs, W.rot.get<float2>((q + 1) / 2), (int)q);
    }
    DITCH_TRY_HIP(hipGetLastError());
}

static void edit_dots(float *out, const float *p, int64_t np, const float *x, int64_t nx, int64_t len, hipStream_t s) {
    hipLaunchKernelGGL(edit_dots_kernel, dim3((unsigned)np, (unsigned)nx), dim3(256), 0, s, out, p, x, np, len);
    DITCH_TRY_HIP(hipGetLastError());
}

// The delta of abliterate.computeDelta for the resident weight w and host
// directions v [k][rows]: device buffers da [rank][cols], db [rows][rank]
// (allocated here, owned by the caller), *rank set.
void edit_delta_device(ditch_hip *h, const TileView &w, const float *hv, int64_t k, float weight, int mode,
                       int64_t lora_rank, uint64_t seed, int ablate, hipStream_t s, float **da_out, float **db_out,
                       int64_t *rank_out) {
    const int64_t rows = w.rows, cols = w.cols;
    DITCH_CHECK(k >= 1 && mode >= 0 && mode <= 2, DITCH_INVALID_ARGUMENT, "edit: at least one direction, mode 0..2");
    if (!h->edit_work) h->edit_work = std::make_shared<EditWork>();
    EditWork &W = *static_cast<EditWork *>(h->edit_work.get());
    float *v = W.v.get<float>(k * rows);
    DITCH_TRY_HIP(hipMemcpyAsync(v, hv, k * rows * 4, hipMemcpyHostToDevice, s));
    const int64_t rank = edit_rank(rows, cols, k, mode, lora_rank, ablate);
    const int64_t r_out = rank - (ablate ? k : 0);  // the output-side edit's rank
    float *A = (float *)dev_alloc(rank * cols * 4), *B = (float *)dev_alloc(rows * rank * 4);
    try {
        // the output-side B, [rows][r_out] (a separate buffer when the input
        // side widens the final B)
        float *Bp = ablate ? W.bp.get<float>(rows * r_out) : B;
        float *norms = nullptr;
        float *a = A;  // none / pre: the output-side A is the first k rows of A
        if (mode == 0) {
            edit_matvecT(w, a, v, k, s);
        } else {
            norms = W.norms.get<float>(rows);
            launch_row_norms(norms, w, s);
            float *vn = W.vn.get<float>(k * rows);
            hipLaunchKernelGGL(edit_vn_kernel, dim3(ed_grid(k * rows)), dim3(256), 0, s, vn, v, norms, k, rows);
            DITCH_TRY_HIP(hipGetLastError());
            if (mode == 2) a = W.a.get<float>(k * cols);
            edit_matvecT(w, a, vn, k, s);
        }
        if (mode != 2) {
            hipLaunchKernelGGL(edit_b_kernel, dim3(ed_grid(k * rows)), dim3(256), 0, s, Bp, v, mode == 1 ? norms : nullptr,
                               k, rows, weight, r_out);
            DITCH_TRY_HIP(hipGetLastError());
        } else {
            // D = diag(c) W + sum_l d_l a_l^T and its randomised SVD
            float *wa = W.wa.get<float>(k * rows);
            edit_matmul(w, wa, a, k, s, &W.xs);
            float *gram = W.gram.get<float>(k * k);
            edit_dots(gram, a, k, a, k, cols, s);
            float *c = W.c.get<float>(rows), *d = W.d.get<float>(k * rows);
            hipLaunchKernelGGL(edit_cd_kernel, dim3(ed_grid(rows)), dim3(256), 0, s, c, d, v, norms, wa, gram, k, rows,
                               weight);
            DITCH_TRY_HIP(hipGetLastError());
            const int64_t rr = lora_rank > k ? lora_rank : k;
            int64_t q = 2 * rr + 4;
            q = q < rows ? q : rows;
            q = q < cols ? q : cols;
            std::vector<float> om((size_t)(q * cols));
            edit_gaussian(om.data(), om.size(), seed);
            float *omega = W.omega.get<float>(q * cols);
            DITCH_TRY_HIP(hipMemcpyAsync(omega, om.data(), om.size() * 4, hipMemcpyHostToDevice, s));
            float *qy = W.qy.get<float>(q * rows), *qx = W.qx.get<float>(q * cols), *cy = W.cy.get<float>(q * rows);
            float *dots = W.dots.get<float>(q * k);
            auto apply = [&](float *out, const float *x) {  // out [q][rows] = (D X)^T
                edit_matmul(w, out, x, q, s, &W.xs);
                edit_dots(dots, a, k, x, q, cols, s);
                hipLaunchKernelGGL(edit_apply_kernel, dim3(ed_grid(q * rows)), dim3(256), 0, s, out, c, d, dots, q, k,
                                   rows);
                DITCH_TRY_HIP(hipGetLastError());
            };
            auto applyT = [&](float *out, const float *y) {  // out [q][cols] = (D^T Y)^T
                hipLaunchKernelGGL(edit_scale_rows_kernel, dim3(ed_grid(q * rows)), dim3(256), 0, s, cy, y, c, q, rows);
                DITCH_TRY_HIP(hipGetLastError());
                edit_matvecT(w, out, cy, q, s);
                edit_dots(dots, d, k, y, q, rows, s);
                hipLaunchKernelGGL(edit_applyT_kernel, dim3(ed_grid(q * cols)), dim3(256), 0, s, out, a, dots, q, k,
                                   cols);
                DITCH_TRY_HIP(hipGetLastError());
            };
            if (orth_takes(q, k)) {
                // the operator's halves with the second part of each in the
                // orthonormalisation's launches
                double *ax = W.dpart0.get<double>(orth_chunks(cols) * q * k);
                double *dy = W.dpart1.get<double>(orth_chunks(rows) * q * k);
                OrthArgs in{};  // ax = dot(a_l, omega_j)
                in.v = omega;
                in.n = cols;
                in.q = (int)q;
                in.k = (int)k;
                in.pa = a;
                in.dots_out = ax;
                launch_orth_chunk(in, s);
                for (int it = 0; it < 7; it++) {
                    if (it) {
                        edit_matvecT(w, qx, cy, q, s);
                        OrthArgs f{}, l{};
                        f.v = qx;
                        f.n = cols;
                        f.q = (int)q;
                        f.k = (int)k;
                        f.u = a;
                        f.dots_in = dy;
                        f.dots_parts = (int)orth_chunks(rows);
                        l.pa = a;
                        l.dots_out = ax;
                        edit_orth_chunks(W, f, l, s);
                    }
                    edit_matmul(w, qy, it ? qx : omega, q, s, &W.xs);
                    OrthArgs f{}, l{};
                    f.v = qy;
                    f.n = rows;
                    f.q = (int)q;
                    f.k = (int)k;
                    f.scale = c;
                    f.u = d;
                    f.dots_in = ax;
                    f.dots_parts = (int)orth_chunks(cols);
                    l.pa = d;
                    l.dots_out = dy;
                    l.cs = c;
                    l.cy = cy;
                    edit_orth_chunks(W, f, l, s);
                }
            } else {
                apply(qy, omega);
                edit_orth(W, qy, q, rows, s);
                for (int it = 0; it < 6; it++) {
                    applyT(qx, qy);
                    edit_orth(W, qx, q, cols, s);
                    apply(qy, qx);
                    edit_orth(W, qy, q, rows, s);
                }
            }
            applyT(qx, qy);  // B^T = (Q^T D)^T
            float *bbt = W.bbt.get<float>(q * q), *evecs = W.evecs.get<float>(q * q);
            edit_dots(bbt, qx, q, qx, q, cols, s);
            edit_jacobi(W, bbt, evecs, q, s);
            hipLaunchKernelGGL(edit_svd_out_kernel, dim3((unsigned)((std::max(rows, cols) + 255) / 256), (unsigned)r_out),
                               dim3(256), (size_t)q * 4, s, A, Bp, bbt, evecs, qy, qx, (int)q, rows, cols, r_out,
                               (int64_t)0);
            DITCH_TRY_HIP(hipGetLastError());
        }
        if (ablate) {
            // U = orth(W^T V) [k][cols]; W' U through the primary delta; the
            // rank grows by k (abliterate.zig:234-261)
            float *u = A + r_out * cols;
            edit_matvecT(w, u, v, k, s);
            edit_orth(W, u, k, cols, s);
            float *wu = W.wu.get<float>(k * rows);
            float *xa = W.xa.get<float>(k * r_out);
            edit_matmul(w, wu, u, k, s, &W.xs, A, Bp, (int)r_out, xa);
            hipLaunchKernelGGL(edit_b_ablate_kernel, dim3(ed_grid(rows * rank)), dim3(256), 0, s, B, Bp, wu, rows, r_out,
                               k, weight);
            DITCH_TRY_HIP(hipGetLastError());
        }
        DITCH_TRY_HIP(hipStreamSynchronize(s));
    } catch (...) {
        dev_free(A);
        dev_free(B);
        throw;
    }
    *da_out = A;
    *db_out = B;
    *rank_out = rank;
}

}  // namespace ditch
