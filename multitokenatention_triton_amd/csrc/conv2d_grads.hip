// Gradients of the depthwise causal conv with respect to its input and its (C,R,S) kernel in one pass over dy: conv2d_mfma with DW,
// whose comment says what it is for and what it measured.  16-bit data and weights, rows of whole 16-byte vectors; under the causal rule
// square planes.
#include "conv2d_mfma.hpp"

namespace {
// launches it; *bpc: on entry how many partial kernels per channel the workspace holds, then how many were left
template <typename T, int R, int S>
int launch_grads(const void *x, const void *dy, const void *w, void *dx, float *partial, int *bpc, int64_t N, int64_t C, int64_t H, int64_t W,
                 int causal, hipStream_t st)
{
    using G = strip_geom<true>;
    const int64_t tiles_m = (H + G::TM - 1) / G::TM, tiles_n = (W + G::TN - 1) / G::TN;
    if (causal && H != W) return MTA_ERR_UNSUPPORTED;
    const int tri = causal ? 1 : 0;
    const int64_t nbf = tiles_m / G::RPB, kl = tiles_m % G::RPB;
    const int64_t ipp64 = tri ? G::RPB * nbf * (nbf + 1) / 2 + kl * (nbf + 1) : tiles_m * tiles_n;
    if (ipp64 > (1 << 24) || N * ipp64 > 0x3fffffffLL || (H + 128) * W > 0x7fffffffLL) return MTA_ERR_UNSUPPORTED;   // (32-bit counts and offsets)
    const int64_t total = N * ipp64;   // items of a channel
    int64_t b = ((int64_t)2 * device_cu_count() + C - 1) / C;   // workgroups of a channel: two per CU in all
    if (b > *bpc) b = *bpc;
    if (b > total) b = total;
    if (b < 1) b = 1;
    const int64_t per_xcd = (C * b + 7) / 8;
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(per_xcd * 8)), dim3(M_WT), 0, st, (const T *)dy, (const T *)w, (T *)dx, (int)C, (int)H, (int)W, causal,
                           1.0f, (int)tiles_n, (int)ipp64, total, per_xcd, (int)b, tri, (const T *)x, partial);
    };
    go(streams(N, C, H, W, sizeof(T)) ? conv2d_mfma<T, R, S, false, true, true, true, true> : conv2d_mfma<T, R, S, false, true, false, true, true>);
    *bpc = (int)b;
    return launch_status();
}

template <typename T>
int dispatch_grads(const void *x, const void *dy, const void *w, void *dx, float *partial, int *bpc, int64_t N, int64_t C, int64_t H, int64_t W, int R,
                   int S, int causal, hipStream_t st)
{
    if constexpr (sizeof(T) != 2) return MTA_ERR_UNSUPPORTED;
    else {
#define MTA_CONV_CASE(r, s) \
    if (R == r && S == s) return launch_grads<T, r, s>(x, dy, w, dx, partial, bpc, N, C, H, W, causal, st);
    MTA_CONV_CASE(3, 3)
    MTA_CONV_CASE(3, 5)
    MTA_CONV_CASE(5, 5)
    MTA_CONV_CASE(5, 7)
    MTA_CONV_CASE(6, 11)
    MTA_CONV_CASE(7, 7)
    MTA_CONV_CASE(7, 9)
    MTA_CONV_CASE(11, 15)
#undef MTA_CONV_CASE
    return MTA_ERR_UNSUPPORTED;
    }
}
}  // namespace

int mta::conv2d_grads_launch(const void *x, const void *dy, const void *w, void *dx, float *partial, int *bpc, int64_t N, int64_t C, int64_t H,
                             int64_t W, int R, int S, int causal, int io_dtype, hipStream_t st)
{
    MTA_DISPATCH_IO(io_dtype, return dispatch_grads<io_t>(x, dy, w, dx, partial, bpc, N, C, H, W, R, S, causal, st));
    return MTA_ERR_DTYPE;
}
