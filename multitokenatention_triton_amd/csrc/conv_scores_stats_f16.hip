// Instances of the scores kernel with the statistics of its rows, for fp16 data.
#include "conv_scores_mfma.hpp"

namespace {
template <int D> int with_stats(const mta::conv_attn_args &a)
{
    if (a.band_lo) return dispatch_scores<mta::f16_t, D, true, 2>(a);
    return a.stats.key_bias ? dispatch_scores<mta::f16_t, D, false, 2>(a) : dispatch_scores<mta::f16_t, D, false, 1>(a);
}
}  // namespace

int mta::conv_scores_stats_f16(const conv_attn_args &a) { return a.D == 64 ? with_stats<64>(a) : with_stats<128>(a); }
