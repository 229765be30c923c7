// attention_rope.h — the whole-prompt attention's own query rotation and the
// few-row attention (attention.hip), for the forward (model.hip).
#pragma once
#include "internal.h"

namespace ditch {

// RoPE of the queries applied as the whole-prompt kernel loads them, in
// place of the RoPE kernel's pass over q (model.zig:4253-4295): head_dim
// 128 rotated whole in neox order (element d with d + 64), no query head
// norm; cos_t / sin_t [rope_len][64], positions past rope_len - 1 use its
// last row. The per-block kernel, which takes the rows when they are not
// dense, reads q as the RoPE kernel left it (rotated).
struct AttnRope {
    const float *cos_t = nullptr, *sin_t = nullptr;
    int64_t rope_len = 0;
};

// launch_attention_mfma with the queries' rotation in the whole-prompt
// kernel (a.dense set, a.hd == 128).
void launch_attention_mfma_rope(const AttnArgs &a, const AttnRope &rope, int64_t kv_heads, hipStream_t s);

// Few rows (decode steps, short prompts): a workgroup per (row, KV head)
// over the row's own keys. Taken for n < 128 rows, and for any number of rows
// up to the cache's prompt slots nb (a decode step has one row a prompt).
bool attention_rows_takes(int64_t hd, int64_t vd, int64_t groups, int64_t n, int64_t nb, int64_t T);
void launch_attention_rows(const AttnArgs &a, int64_t kv_heads, hipStream_t s);

}  // namespace ditch
