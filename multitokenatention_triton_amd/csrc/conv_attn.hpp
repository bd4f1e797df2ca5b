// The 16-bit kernels of the fused conv-attention path by I/O type; returns 1 when no instance covers the kernel size (the
// caller then uses the general kernel).  scores_only: stop after the conv (o = the score tensor; band_lo, tri_gl and
// fill_upper belong to it), else the attention output (lse may be NULL).
#pragma once

#include "scores_cut.hpp"

namespace mta {
struct conv_attn_args {
    const void *q, *k, *v, *w;
    void *o;
    float *lse;
    int64_t B, H, S, D;
    int R, Sk, causal;
    float scale;
    int fill_upper;
    const int *band_lo;   // scores only: first visible key per row, or NULL
    int tri_gl;           // scores only: > 0 = triangular layout, groups of that many heads
    bool scores_only;
    hipStream_t st;
    row_strides qs = {0, 0, 0};   // a 1x1 kernel's q where its rows do not follow one another
    int64_t rows = 0;             // scores only: rows of q and k where they have fewer than S (0: S)
    scores_stats stats = {nullptr, nullptr, 0, {1, 1, 0}};   // scores only, conv_scores_stats_dispatch: the rows' statistics
};
int conv_attn_mfma_bf16(const conv_attn_args &a);
int conv_attn_mfma_f16(const conv_attn_args &a);
inline int conv_attn_mfma_dispatch(int io_dtype, const conv_attn_args &a)
{
    return io_dtype == MTA_BF16 ? conv_attn_mfma_bf16(a) : io_dtype == MTA_F16 ? conv_attn_mfma_f16(a) : 1;
}
// the scores kernel with the statistics of its rows (causal)
int conv_scores_stats_bf16(const conv_attn_args &a);
int conv_scores_stats_f16(const conv_attn_args &a);
inline int conv_scores_stats_dispatch(int io_dtype, const conv_attn_args &a)
{
    return io_dtype == MTA_BF16 ? conv_scores_stats_bf16(a) : io_dtype == MTA_F16 ? conv_scores_stats_f16(a) : 1;
}
}  // namespace mta
