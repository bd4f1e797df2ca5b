// fp32 values as sums of bf16 parts, for products on the bf16 matrix cores that keep the 32 bits.
//
// x = x0 + x1 + x2, each part the bf16 value nearest to the remainder of those before it: 8 + 8 + 8 bits, exactly x while the parts
// neither overflow (|x| of 3.39e38 and more rounds to infinity) nor underflow (below about 2^-109).  So the values are split 2^24
// times as large (SPLIT_UP) and the results taken back: every |x| below 2^104 has parts that are normal numbers then, and only sums
// of 2^80 and more overflow.  Of the nine products of parts of a product x w the six x_i w_j with i + j <= 2 are formed; each is exact
// in fp32, and what is left out is below 2^-26 |x w|, a quarter of the last place that one fp32 multiply-add rounds away.
#pragma once

#include "common.hpp"
#include "mfma.hpp"

namespace mta {

constexpr float SPLIT_UP = 16777216.0f;   // 2^24: fp32's last bit, 2^-149, becomes a normal number

// two values' parts, packed.  (The packed dot product with (-1, 0) or (0, -1) takes one of the two values off a remainder without
// unpacking it: one instruction in place of two.  Constants the compiler cannot see: it would fold (-1, 0) into the inline constant
// -1.0, which the instruction takes for (0, -1).)
template <int N> __device__ __forceinline__ void split2(float a, float b, uint32_t (&part)[N])
{
    uint32_t minus_lo = 0x0000bf80u, minus_hi = 0xbf800000u;
    asm("" : "+s"(minus_lo), "+s"(minus_hi));
    const mta_bf16x2 lo = __builtin_bit_cast(mta_bf16x2, minus_lo), hi = __builtin_bit_cast(mta_bf16x2, minus_hi);
#pragma unroll
    for (int s = 0; s < N; ++s) {
        part[s] = pack2<bf16_t>(a, b);
        if (s == N - 1) break;
        const mta_bf16x2 h = __builtin_bit_cast(mta_bf16x2, part[s]);
        a = __builtin_amdgcn_fdot2_f32_bf16(h, lo, a, false);
        b = __builtin_amdgcn_fdot2_f32_bf16(h, hi, b, false);
    }
}

// eight values' parts as operand fragments
__device__ __forceinline__ void split8(f32x4 lo, f32x4 hi, frag8<bf16_t> (&part)[3])
{
    uint32_t w[4][3];
    split2<3>(lo[0], lo[1], w[0]);
    split2<3>(lo[2], lo[3], w[1]);
    split2<3>(hi[0], hi[1], w[2]);
    split2<3>(hi[2], hi[3], w[3]);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        struct { uint32_t v[4]; } f = {{w[0][s], w[1][s], w[2][s], w[3][s]}};
        part[s] = __builtin_bit_cast(frag8<bf16_t>, f);
    }
}

__device__ __forceinline__ void mma4(f32x4 &c, float a, float b) { c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Whether one of a wavefront's sums is not finite: an operand was not, or a part of one overflowed (every product with it is infinite or
// NaN), or the sum itself did.
template <int N> __device__ __forceinline__ bool not_finite(const f32x4 *acc)
{
    float bad = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) bad = fmaf(acc[i][v], 0.0f, bad);
    return __builtin_amdgcn_ballot_w64(bad != 0.0f) != 0;
}
}  // namespace mta
