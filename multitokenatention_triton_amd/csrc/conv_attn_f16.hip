// Instances of the fused conv-attention kernels for f16 data.
#include "conv_attn_mfma.hpp"

int mta::conv_attn_mfma_f16(const conv_attn_args &a) { return dispatch_mfma_type<f16_t>(a); }
