// Instances of the fused conv-attention kernels for bf16 data.
#include "conv_attn_mfma.hpp"

int mta::conv_attn_mfma_bf16(const conv_attn_args &a) { return dispatch_mfma_type<bf16_t>(a); }
