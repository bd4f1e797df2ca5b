// Instances of the scores kernel with the statistics of its rows, for fp16 data.
#include "conv_scores_mfma.hpp"

namespace {
template <int D> int with_stats(const mta::conv_attn_args &a)
{
    return a.band_lo ? dispatch_scores<mta::f16_t, D, true, true>(a) : dispatch_scores<mta::f16_t, D, false, true>(a);
}
}  // namespace

int mta::conv_scores_stats_f16(const conv_attn_args &a) { return a.D == 64 ? with_stats<64>(a) : with_stats<128>(a); }
