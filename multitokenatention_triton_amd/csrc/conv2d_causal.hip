// Depthwise causal 2-D convolution over the (N,C,H,W) score tensor.
//
//   y[n,c,p,q] = sum_{i<R,j<S} w[c,i,j] * xm[n,c,p+i-(R-1), q+j-(S-1)/2]
//
// One workgroup owns a TM x TN output tile of one (n,c) plane.  It stages the
// (TM+R-1) x (TN+S-1) query x key halo tile in LDS once (bounds and the causal
// col<=row rule are applied while staging, so the tap loop is mask-free), skips
// tiles that lie entirely above the diagonal (they only receive their +0 fill), and
// applies the causal output rule on store.
//
// Four compute paths:
//   conv2d_valu  fp32 FMAs from an fp32 LDS tile (8 outputs per lane); any I/O and weight dtype, any kernel size.
//   conv2d_rows  fp32 FMAs, sliding down the rows in registers (conv2d_rows.hpp); any I/O and weight dtype, the kernel
//                sizes known at compile time.
//   conv2d_split 11x15, and the larger of the others in 16 bits, of what conv2d_mfma does not take (conv2d_split.hip).
//   conv2d_mfma  16-bit I/O with weights of the same dtype.  The 6x11 conv costs 66 FMAs
//                per output, which on the vector ALU takes longer than moving the tensor
//                through HBM.  Each kernel row is therefore applied as a banded (Toeplitz)
//                matrix product on the matrix cores:
//                    out^T[q, p] += T_i^T[q, k] * X^T[k, p+i-(R-1)]      i = 0..R-1
//                with T_i[k, q] = w[i, k-q-shift] held in registers for the whole kernel
//                and X^T fragments read straight from the row-major LDS tile (a lane reads
//                16 contiguous bytes of one query row).  ~4x the multiply-adds, on a unit
//                with ~16x the rate: the kernel becomes HBM-bound.  Products of 16-bit
//                values are exact in fp32 and accumulation is fp32, as in the VALU path.
#include "common.hpp"
#include "conv2d_mfma.hpp"
#include "conv2d_rows.hpp"

#include <stdlib.h>

#include <atomic>
#include <type_traits>
#include <utility>

namespace {
using namespace mta;

constexpr int NT = 256;

// ------------------------------------------------------------------------------------
// VALU path
// ------------------------------------------------------------------------------------
constexpr int V_TM = 32;  // tile rows   (thread t: row t/8)
constexpr int V_TN = 64;  // tile cols   (thread t: cols 8*(t%8) .. +7)

template <typename T>
__device__ __forceinline__ void store_row8(T *yp, int64_t W, int H, int p, int q, const float *acc,
                                           bool causal)
{
    if (p >= H) return;
    T *dst = yp + (int64_t)p * W + q;
    if (q + 8 <= W && (reinterpret_cast<uintptr_t>(dst) % (8 * sizeof(T))) == 0) {
        struct alignas(8 * sizeof(T)) chunk { T v[8]; } c;
#pragma unroll
        for (int u = 0; u < 8; ++u) c.v[u] = from_float<T>((causal && q + u > p) ? 0.0f : acc[u]);
        *reinterpret_cast<chunk *>(dst) = c;
    } else {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (q + u < W) dst[u] = from_float<T>((causal && q + u > p) ? 0.0f : acc[u]);
    }
}

// BWD: the gradient with respect to the input,
//   dx[h,w] = sum_{i,j} w[i,j] * dym[h-i+(R-1), w-j+(S-1)/2]        (dym = dy with q>p read as 0 when causal)
// which is the same tile computation with the kernel reversed in both axes, the row halo below the tile instead of
// above it and the key halos swapped; dx is +0 above the diagonal (those inputs were never read).
template <typename T, bool BWD>
__global__ __launch_bounds__(NT) void conv2d_valu(const T *__restrict__ x, const void *__restrict__ w,
                                                  T *__restrict__ y, int C, int H, int W, int R,
                                                  int S, int causal, float in_scale, int use_scale,
                                                  int w_dtype, int tiles_n)
{
    const int pad_h = BWD ? 0 : R - 1, pad_w = BWD ? S - 1 - (S - 1) / 2 : (S - 1) / 2;
    const int LD = V_TN + S;  // S-1 halo columns + 1 pad
    extern __shared__ float smem[];
    float *wsm = smem;                        // R*S weights of this channel
    float *tile = smem + ((R * S + 3) & ~3);  // (V_TM+R-1) x LD

    const int tid = threadIdx.x;
    const int64_t plane = blockIdx.y;
    const int c = (int)(plane % C);
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
    const int p0 = tm * V_TM, q0 = tn * V_TN;
    const T *xp = x + plane * (int64_t)H * W;
    T *yp = y + plane * (int64_t)H * W;
    const int tr = tid >> 3, tc = (tid & 7) * 8;

    float acc[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = 0.0f;

    if (causal && q0 > p0 + V_TM - 1) {  // wholly above the diagonal: fill only
        store_row8<T>(yp, W, H, p0 + tr, q0 + tc, acc, true);
        return;
    }

    for (int t = tid; t < R * S; t += NT) wsm[t] = load_any(w, w_dtype, (int64_t)c * R * S + (BWD ? R * S - 1 - t : t));

    const int rows = V_TM + R - 1, cols = V_TN + S - 1;
    for (int rr = tid / 64; rr < rows; rr += NT / 64) {
        const int h = p0 - pad_h + rr;
        const bool row_ok = h >= 0 && h < H;
        for (int cc = tid % 64; cc < cols; cc += 64) {
            const int k = q0 - pad_w + cc;
            float v = 0.0f;
            if (row_ok && k >= 0 && k < W && (!causal || k <= h)) {
                v = to_float(xp[(int64_t)h * W + k]);
                if (use_scale) v = round_to<T>(v * in_scale);
            }
            tile[rr * LD + cc] = v;
        }
    }
    __syncthreads();

    for (int i = 0; i < R; ++i) {
        const float *src = tile + (tr + i) * LD + tc;
        for (int j = 0; j < S; ++j) {
            const float wv = wsm[i * S + j];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc[u] = fmaf(wv, src[u + j], acc[u]);
        }
    }
    store_row8<T>(yp, W, H, p0 + tr, q0 + tc, acc, causal != 0);
}

template <typename T, bool BWD>
int launch_valu(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int R,
                int S, int causal, float in_scale, int use_scale, int w_dtype, hipStream_t st)
{
    const int tiles_m = (int)((H + V_TM - 1) / V_TM), tiles_n = (int)((W + V_TN - 1) / V_TN);
    const size_t lds = sizeof(float) * (((R * S + 3) & ~3) + (size_t)(V_TM + R - 1) * (V_TN + S));
    dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)(N * C));
    if (lds > 160 * 1024) return MTA_ERR_KERNEL_SIZE;
    if (lds > 48 * 1024) {  // per device, so set on every such launch (a cheap host-side call)
        hipError_t e = hipFuncSetAttribute((const void *)conv2d_valu<T, BWD>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL((conv2d_valu<T, BWD>), grid, dim3(NT), lds, st, (const T *)x, w, (T *)y, (int)C,
                       (int)H, (int)W, R, S, causal, in_scale, use_scale, w_dtype, tiles_n);
    return launch_status();
}

template <typename T, int R, int S, bool BWD, bool NARROW>
int launch_mfma(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int causal,
                float in_scale, int use_scale, hipStream_t st)
{
    using G = strip_geom<NARROW>;
    const int64_t tiles_m = (H + G::TM - 1) / G::TM, tiles_n = (W + G::TN - 1) / G::TN;
    // causal, square, and the caller wants nothing written above the diagonal: only the strips that touch the lower triangle
    const int tri = (causal == 2 && H == W) ? 1 : 0;
    const int64_t nbf = tiles_m / G::RPB, kl = tiles_m % G::RPB;
    const int64_t ipp64 = tri ? G::RPB * nbf * (nbf + 1) / 2 + kl * (nbf + 1) : tiles_m * tiles_n;
    if (ipp64 > (1 << 24)) return MTA_ERR_SHAPE;  // decode_item's float sqrt is exact well beyond this
    const int ipp = (int)ipp64;
    const int64_t total = N * C * ipp64;
    const int64_t per_xcd = (total + 7) / 8;
    // persistent workgroups per XCD: as many as fit when only the strips of the lower triangle are walked; with the zero
    // strips in the list three per CU move the tensor fastest (measured at (2,16,2048,2048): 84 us against 85.5 with four)
    int nw = device_cu_count() * (tri ? wg_per_cu<R, NARROW>() : 3) / 8;
    if (nw < 1) nw = 1;
    if (per_xcd < nw) nw = (int)per_xcd;
    dim3 grid((unsigned)(nw * 8));
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, grid, dim3(M_WT), 0, st, (const T *)x, (const T *)w, (T *)y, (int)C, (int)H, (int)W, causal, in_scale,
                           (int)tiles_n, ipp, total, per_xcd, nw, tri, (const T *)nullptr, (float *)nullptr);
    };
    const bool stream = streams(N, C, H, W, sizeof(T));
    if constexpr (BWD) {
        go(stream ? conv2d_mfma<T, R, S, false, true, true, NARROW> : conv2d_mfma<T, R, S, false, true, false, NARROW>);
    } else if (use_scale) {
        go(stream ? conv2d_mfma<T, R, S, true, false, true, NARROW> : conv2d_mfma<T, R, S, true, false, false, NARROW>);
    } else {
        go(stream ? conv2d_mfma<T, R, S, false, false, true, NARROW> : conv2d_mfma<T, R, S, false, false, false, NARROW>);
    }
    return launch_status();
}

// returns 1 when no MFMA instantiation covers (R,S) -- the caller then takes the VALU path
template <typename T, bool BWD>
int dispatch_mfma(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int R, int S,
                  int causal, float in_scale, int use_scale, hipStream_t st)
{
    if constexpr (sizeof(T) != 2) return 1;
    else {
#define MTA_CONV_CASE(r, s)                                       \
    static_assert(mfma_geom<r, s, true>::fits, "window exceeds 32 keys");                                                  \
    if (R == r && S == s) {                                                                                                \
        if constexpr (r <= 7) {                                                                                            \
            if (!narrow_strips(N, C, H, W, causal, r))                                                                       \
                return launch_mfma<T, r, s, BWD, false>(x, w, y, N, C, H, W, causal, in_scale, use_scale, st);             \
        }                                                                                                                  \
        return launch_mfma<T, r, s, BWD, true>(x, w, y, N, C, H, W, causal, in_scale, use_scale, st);                      \
    }
    MTA_CONV_CASE(3, 3)
    MTA_CONV_CASE(3, 5)
    MTA_CONV_CASE(5, 5)
    MTA_CONV_CASE(5, 7)
    MTA_CONV_CASE(6, 11)
    MTA_CONV_CASE(7, 7)
    MTA_CONV_CASE(7, 9)
    MTA_CONV_CASE(11, 15)
#undef MTA_CONV_CASE
    return 1;
    }
}

template <bool BWD>
int conv2d_entry(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int R,
                 int S, int causal, float in_scale, int use_scale, int io_dtype, int w_dtype, void *stream)
{
    // MTA_CONV_FORCE_VALU=1 in the environment keeps everything on the fp32-FMA kernels (for comparisons)
    static const bool force_valu = [] { const char *e = getenv("MTA_CONV_FORCE_VALU"); return e && e[0] == '1'; }();
    if (!x || !w || !y) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (N <= 0 || C <= 0 || H <= 0 || W <= 0) return MTA_ERR_SHAPE;
    if (H > (1 << 24) || W > (1 << 24) || N * C > 0x7fffffffLL / 2) return MTA_ERR_SHAPE;
    if (R < 1 || S < 1 || R > MTA_MAX_KERNEL_R || S > MTA_MAX_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (!aligned_to(x, dtype_size(io_dtype)) || !aligned_to(y, dtype_size(io_dtype)) ||
        !aligned_to(w, dtype_size(w_dtype)))
        return MTA_ERR_ALIGN;
    const int64_t tiles = ((H + V_TM - 1) / V_TM) * ((W + V_TN - 1) / V_TN);
    if (tiles > 0x7fffffffLL || N * C > 65535) return MTA_ERR_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    const bool mfma_ok = io_dtype != MTA_F32 && w_dtype == io_dtype && W % 8 == 0 && aligned_to(x, 16) &&
                         aligned_to(y, 16) && !force_valu;
    MTA_DISPATCH_IO(io_dtype, {
        if (mfma_ok) {
            const int rc = dispatch_mfma<io_t, BWD>(x, w, y, N, C, H, W, R, S, causal, in_scale, use_scale, st);
            if (rc != 1) return rc;
        }
        if (!force_valu) {
            const int rc = conv2d_split_dispatch(x, w, y, N, C, H, W, R, S, BWD, causal, in_scale, use_scale, io_dtype, w_dtype, st);
            if (rc != 1) return rc;
        }
        const int rc = dispatch_rows<io_t, BWD>(x, w, y, N, C, H, W, R, S, causal, in_scale, use_scale, w_dtype, st);
        if (rc != 1) return rc;
        return launch_valu<io_t, BWD>(x, w, y, N, C, H, W, R, S, causal, in_scale, use_scale, w_dtype, st);
    });
    return MTA_ERR_DTYPE;
}
// the `causal` argument of the entry points: 0 = no mask, 2 = causal with the output above the diagonal left to the
// caller (MTA_CAUSAL_LOWER_ONLY), anything else = causal with +0 written there
inline int causal_mode(int causal) { return causal == MTA_CAUSAL_LOWER_ONLY ? 2 : (causal ? 1 : 0); }
}  // namespace

extern "C" int mta_conv2d_fwd(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H,
                              int64_t W, int R, int S, int causal, int io_dtype, int w_dtype, void *stream)
{
    return conv2d_entry<false>(x, w, y, N, C, H, W, R, S, causal_mode(causal), 1.0f, 0, io_dtype, w_dtype, stream);
}

// (causal == 2 inside this file: causal, and the kernel that enumerates the lower triangle's strips only - the
// matrix-core one on square tensors - does not write their images above the diagonal; every other path fills as usual)
extern "C" int mta_conv2d_tril_fwd(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W,
                                   int R, int S, int io_dtype, int w_dtype, void *stream)
{
    return conv2d_entry<false>(x, w, y, N, C, H, W, R, S, 2, 1.0f, 0, io_dtype, w_dtype, stream);
}

extern "C" int mta_conv2d_bwd_input(const void *dy, const void *w, void *dx, int64_t N, int64_t C, int64_t H,
                                    int64_t W, int R, int S, int causal, int io_dtype, int w_dtype, void *stream)
{
    return conv2d_entry<true>(dy, w, dx, N, C, H, W, R, S, causal_mode(causal), 1.0f, 0, io_dtype, w_dtype, stream);
}

extern "C" int mta_conv2d_scaled_fwd(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H,
                                     int64_t W, int R, int S, int causal, float in_scale, int io_dtype,
                                     int w_dtype, void *stream)
{
    return conv2d_entry<false>(x, w, y, N, C, H, W, R, S, causal_mode(causal), in_scale, 1, io_dtype, w_dtype, stream);
}
