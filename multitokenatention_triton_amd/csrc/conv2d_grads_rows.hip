// Gradients of the depthwise causal conv with respect to its input and its (C,R,S) kernel in one pass over dy, for what the matrix-core
// kernel (conv2d_grads.hip) does not take: fp32 data, 16-bit data with fp32 weights or with rows that are not whole vectors.
//
// The row-sliding kernels of conv2d_rows.hpp in one: a wavefront walks down the rows of dy, and the window that a lane has of a row
// serves the R rows of dx above it (times the weights) and the R rows of x above it (into R*S sums per lane, added up over the
// wavefront at the very end).  dx is formed as there, sum by sum.  What bounds it: load instructions (dy and x once, where the two
// kernels take dy twice) and fp32 FMAs, 2 R S per position.  A wavefront's last steps fetch the first rows of its next strip.
// us with the sum of the partial kernels, the two kernels -> this, nothing in the caches: fp32 5x5 lower triangle B1 H32 S1024 84 -> 70, B1 H16
// S512 26 -> 20, B1 H16 S1712 106 -> 87, 3x3 B1 H16 S2048 148 -> 125, whole rows 162 -> 144, 5x7 B1 H16 S2048 154 -> 137, B2 H12 S640 44 -> 34; fp32
// weights, bf16 5x5 B1 H16 S1024 36.8 -> 34.0, fp16 3x3 B2 H16 S1504 81 -> 65; fp16 5x5 B2 H12 S777 49 -> 36.  Kernels of up to 35 taps, whose
// weights fit the scalar registers: 6x11 B1 H16 S1024 75 -> 76, 7x7 60 -> 47, but B2 H16 S2048 fp16 246 -> 281, 7x9 B4 H12 S640 91 -> 146.
// (Unrolled whole, as the kernel gradient alone is: as fast, or with the next strip's rows spilled.)
#include "conv2d_rows.hpp"

namespace {
template <int R, int S> constexpr int grads_occ() { return R * S > 25 || S > R ? 3 : 4; }   // workgroups per CU
// y (the gradient of x) may be x: a row of x is in registers before the row of y is written, by the same lanes
template <typename T, int R, int S, int M>
__global__ __launch_bounds__(256, (grads_occ<R, S>())) void conv2d_grads_rows(const T *x, const T *__restrict__ dy, const void *__restrict__ w, T *y,
                                                                          float *__restrict__ partial, int N, int C, int H, int W, int causal, int bpc,
                                                                          int tiles, int w_dtype)
{
    using G = row_window<S, true>;
    constexpr int STEPS = M + R - 1;
    constexpr int RW_AHEAD = STEPS % 4 == 0 ? 4 : STEPS % 5 == 0 ? 5 : 3;   // rows fetched ahead, the next strip's behind this one's
    static_assert(STEPS % RW_AHEAD == 0, "the next strip's rows in the places where it looks for them");
    constexpr bool SREG = R * S <= 35;        // weights in scalar registers (more of them spill)
    constexpr int LDW = (S + 3) & ~3;
    __shared__ __align__(16) float wsm[R * LDW];
    __shared__ float red[4][R * S];
    const int c = blockIdx.x / bpc, b = blockIdx.x % bpc;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    for (int t = threadIdx.x; t < R * LDW; t += 256) {
        const int i = t / LDW, j = t % LDW;
        wsm[t] = j < S ? load_any(w, w_dtype, (int64_t)c * R * S + (R * S - 1 - (i * S + j))) : 0.0f;
    }
    __syncthreads();
    float ws[SREG ? R * S : 1];
    if constexpr (SREG) {
#pragma unroll
        for (int t = 0; t < R * S; ++t)
            ws[t] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wsm[t / S * LDW + t % S])));
    }
    if (causal == 1) {   // +0 over the strips wholly above the diagonal, row by row
        for (int64_t r = (int64_t)wave * bpc + b; r < (int64_t)N * H; r += (int64_t)bpc * 4) {
            const int n_ = (int)(r / H), p = (int)(r - (int64_t)n_ * H);
            T *row = y + (((int64_t)n_ * C + c) * H + p) * (int64_t)W;
            const float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            // (the strips of M rows that reach row p's strip start at keys of up to its last row)
            for (int64_t q = ((int64_t)(p / M * M + M - 1) / G::KEYS + 1) * G::KEYS + lane * 4; q < W; q += 256) store_quad<T>(row, (int)q, W, z);
        }
    }
    float sum[R][S];                          // of tap (R-1-i, S-1-j)
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < S; ++j) sum[i][j] = 0.0f;
    struct strip_at { int64_t plane; int p0, q0; unsigned off; };   // off: where in a row a lane's vector starts, in bytes
    auto locate = [&](int it) {
        const int n_ = it / tiles;
        strip_at s{((int64_t)n_ * C + c) * H * (int64_t)W, 0, 0, 0u};
        strips<G, M>::at(it - n_ * tiles, H, causal, s.p0, s.q0);
        const int k = s.q0 + (lane - G::LL) * 4;   // (as load_quad)
        s.off = (unsigned)(k < 0 ? 0 : (k > W - 4 ? W - 4 : k)) * (unsigned)sizeof(T);
        return s;
    };
    quad4<T> xr[RW_AHEAD], gr[RW_AHEAD];
    auto fetch = [&](const strip_at &s, int n, int slot) __attribute__((always_inline)) {
        const int h = s.p0 + n < H ? s.p0 + n : H - 1;
        const int64_t row = s.plane + (int64_t)h * W;
        __builtin_memcpy(&gr[slot], reinterpret_cast<const char *>(dy + row) + s.off, sizeof(gr[slot]));
        __builtin_memcpy(&xr[slot], reinterpret_cast<const char *>(x + row) + s.off, sizeof(xr[slot]));
    };
    const int items = N * tiles, stride = bpc * 4;
    int it = wave * bpc + b;
    strip_at cur = locate(it < items ? it : 0);
    if (it < items) {
#pragma unroll
        for (int d = 0; d < RW_AHEAD - 1; ++d) fetch(cur, d, d);
    }
    for (; it < items; it += stride) {
        const strip_at next = it + stride < items ? locate(it + stride) : cur;
        const int p0 = cur.p0, q0 = cur.q0, q = q0 + (lane - G::LL) * 4;
        const bool mine = lane >= G::LL && lane < 64 - G::LR && q < W;
        T *yp = y + cur.plane;
        const bool cols_inside = q0 - 4 * G::LL >= 0 && q0 + G::KEYS + 4 * G::LR <= W;
        // [k]: row (step n) - (R-1) + k of the strip, of x (0 outside it) and of dx
        float xv[R][4], acc[R][4];
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int u = 0; u < 4; ++u) xv[k][u] = acc[k][u] = 0.0f;
        auto step = [&](int n, int slot) __attribute__((always_inline)) {
            const float *wp = wsm + (SREG ? 0 : opaque(0));   // (opaque: the weights are not to be kept in registers across rows)
#pragma unroll
            for (int k = 0; k + 1 < R; ++k)
#pragma unroll
                for (int u = 0; u < 4; ++u) xv[k][u] = xv[k + 1][u];
            const int h = p0 + n;
            const bool inside = cols_inside && h < H && (!causal || q0 + G::KEYS + 4 * G::LR - 1 <= h);
            masked_quad<T>(xr[slot], q, W, (!mine || n >= M || h >= H) ? -1 : (causal && h < W - 1 ? h : W - 1), xv[R - 1]);
            float own[4];
            if (inside) {
#pragma unroll
                for (int u = 0; u < 4; ++u) own[u] = to_float(gr[slot].v[u]);
            } else {
                masked_quad<T>(gr[slot], q, W, h >= H ? -1 : (causal && h < W - 1 ? h : W - 1), own);
            }
            float win[G::WIN];
            window_of<G>(own, win);
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int o = n - (R - 1) + k;    // (uniform) row within the strip
                if (o < 0 || o >= M) continue;
                const int i = R - 1 - k;
#pragma unroll
                for (int j = 0; j < S; ++j) {
                    const float wv = SREG ? ws[SREG ? i * S + j : 0] : wp[i * LDW + j];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        acc[k][u] = fmaf(wv, win[j + u], acc[k][u]);
                        sum[i][j] = fmaf(xv[k][u], win[j + u], sum[i][j]);
                    }
                }
            }
            const int p = p0 + n - (R - 1);       // complete now
            if (n >= R - 1 && p < H && mine && !(causal == 2 && q > p)) {
                float out[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) out[u] = (causal && q + u > p) ? 0.0f : acc[0][u];
                store_quad<T>(yp + (int64_t)p * W, q, W, out);
            }
#pragma unroll
            for (int k = 0; k + 1 < R; ++k)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[k][u] = acc[k + 1][u];
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[R - 1][u] = 0.0f;
        };
#pragma unroll 1
        for (int n = 0; n < STEPS; n += RW_AHEAD) {
#pragma unroll
            for (int d = 0; d < RW_AHEAD; ++d) {
                const int ahead = n + d + RW_AHEAD - 1;
                const bool beyond = ahead >= STEPS;
                fetch(beyond ? next : cur, beyond ? ahead - STEPS : ahead, (d + RW_AHEAD - 1) % RW_AHEAD);
                step(n + d, d);
            }
        }
        cur = next;
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const float s = wave_total(sum[i][j]);
            if (lane == 63) red[wave][(R - 1 - i) * S + S - 1 - j] = s;
        }
    __syncthreads();
    for (int t = threadIdx.x; t < R * S; t += 256)
        partial[(int64_t)blockIdx.x * (R * S) + t] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

template <typename T>
int dispatch_grads_rows(const void *x, const void *dy, const void *w, void *dx, float *partial, int *bpc, int64_t N, int64_t C, int64_t H, int64_t W,
                        int R, int S, int causal, int w_dtype, hipStream_t st)
{
    if (W < 4) return MTA_ERR_UNSUPPORTED;
    const int m = rows_per_strip(N * C, H, W, R, S, causal);
    auto go = [&](auto kern, int occ, int64_t total) {
        if (N * total > 0x3fffff00LL) return (int)MTA_ERR_UNSUPPORTED;   // (32-bit counts)
        int64_t most = ((int64_t)occ * device_cu_count() + C - 1) / C;   // (one round of resident workgroups)
        if (most > (N * total + 3) / 4) most = (N * total + 3) / 4;
        if (*bpc > most) *bpc = (int)most;
        hipLaunchKernelGGL(kern, dim3((unsigned)(C * *bpc)), dim3(256), 0, st, (const T *)x, (const T *)dy, w, (T *)dx, partial, (int)N, (int)C, (int)H,
                           (int)W, causal, *bpc, (int)total, w_dtype);
        return launch_status();
    };
#define MTA_ROWS(r, s, m) go(conv2d_grads_rows<T, r, s, m>, grads_occ<r, s>(), strips<row_window<s, true>, m>::count((int)H, (int)W, causal))
#define MTA_CONV_CASE(r, s) \
    if (R == r && S == s) return m == 4 ? MTA_ROWS(r, s, 4) : MTA_ROWS(r, s, 8);
    MTA_CONV_CASE(3, 3)
    MTA_CONV_CASE(3, 5)
    MTA_CONV_CASE(5, 5)
    MTA_CONV_CASE(5, 7)
#undef MTA_CONV_CASE
#undef MTA_ROWS
    return MTA_ERR_UNSUPPORTED;
}
}  // namespace

int mta::conv2d_grads_rows_launch(const void *x, const void *dy, const void *w, void *dx, float *partial, int *bpc, int64_t N, int64_t C, int64_t H,
                                  int64_t W, int R, int S, int causal, int io_dtype, int w_dtype, hipStream_t st)
{
    MTA_DISPATCH_IO(io_dtype, return dispatch_grads_rows<io_t>(x, dy, w, dx, partial, bpc, N, C, H, W, R, S, causal, w_dtype, st));
    return MTA_ERR_DTYPE;
}
