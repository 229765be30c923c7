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
// k tiles of its fragments: whole 128-column steps (split_ldk)
inline int64_t few_ldk(const TileView &w) { return split_ldk(w.cols); }
// Whether it reads n f32 rows at x itself (no fragments).
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

}  // namespace ditch
