// gemm_few.h — products of few tokens (gemm_few.hip).
#pragma once
#include "gemm_common.h"

namespace ditch {

// One matrix of a few-token product: out [n][rows] (+)= x W^T + delta + bias.
struct FewMat {
    TileView w;
    float *out;
    const float *bias;
    const float *delta_b, *delta_xa;  // [rows][rank], [n][rank]
    int delta_rank, accumulate;
};

// Whether the few-token product takes w on n tokens, from f32 rows or from
// fragments (split_kernel's layout, few_ldk(K) k tiles).
bool few_gemm_takes(const TileView &w, int64_t n, bool exact);
// Whether it takes several matrices of one format and K in one launch, over
// fragments that their producer writes, instead of a product and a split each
// (and saved_us of other work).
constexpr double FEW_SPLIT_US = 3;
bool few_launch_takes(const TileView *const *w, int count, int64_t n, double saved_us);
// Estimated us of the product that runs otherwise, 33 to 255 tokens
// (gemm_tile.hip).
double large_gemm_us(const TileView &w, int64_t n);
// k tiles of its fragments: whole 128-column steps (split_ldk)
inline int64_t few_ldk(const TileView &w) { return split_ldk(w.cols); }
// Whether it can read n f32 rows at x itself (no fragments).
bool few_reads_rows(const TileView &w, int64_t n, const float *x, int64_t ldx);
// Products of 1 to 3 matrices of one format and K over the same activations,
// in one launch: from f32 rows x (few_reads_rows) or, with x NULL, from
// fragments xs (xt terms, ldk k tiles per 16-token block).
void launch_few_gemm(const FewMat *mats, int nmat, const float *x, int64_t ldx, const void *xs, int64_t ldk, int64_t n,
                     int xt, hipStream_t s);

// The MLP's first product: act(x gate^T) * (x up^T) (tensor.zig:1309-1337) of
// two matrices of one format and shape the few-token product takes (no
// deltas), as f32 rows y [n][rows] and/or as the next product's fragments
// ys (ldk_y k tiles; rows a multiple of 128). Activations as above.
bool few_glu_takes(const TileView &gate, const TileView &up, int64_t n);
void launch_few_glu(const TileView &gate, const TileView &up, uint32_t act, float *y, void *ys, int64_t ldk_y,
                    const float *x, int64_t ldx, const void *xs, int64_t ldk, int64_t n, hipStream_t s);

// Routed experts of few rows each (16-byte aligned f32 rows of whole float4s),
// every expert one format and shape: the gate/up product with its activation
// into y [pair][rows], the rows gathered by row_index, and the down product
// from consecutive rows, deltas added (delta_xa [pair][stride]). An expert's
// gate and up share their scale layout (few_glu_takes); experts may differ.
bool few_grouped_takes(const GroupSeg *segs, unsigned nseg, int64_t max_cnt);
bool few_glu_grouped_takes(const GroupSeg *gate, const GroupSeg *up, unsigned nseg, int64_t max_cnt);
void launch_few_glu_grouped(const GroupSeg *d_gate, const GroupSeg *d_up, const TileView &shape, unsigned nseg,
                            int64_t max_cnt, uint32_t act, float *y, const float *x, const int32_t *row_index,
                            hipStream_t s);
void launch_few_grouped(const GroupSeg *d_segs, const TileView &shape, unsigned nseg, int64_t max_cnt, float *out,
                        const float *x, const float *delta_xa, int delta_stride, hipStream_t s);

}  // namespace ditch
