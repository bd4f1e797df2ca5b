// Row-sliding fp32-FMA kernels of the depthwise conv: forward, input gradient and kernel gradient for the I/O types, weight
// types and widths the matrix-core kernels do not take (fp32; 16-bit data with weights of another dtype or with rows that are
// not whole 16-byte vectors), kernel sizes known at compile time.  conv2d_split.hip comes first in the forward and the input gradient of
// 11x15, and of 6x11, 7x9, 7x7 (bf16) and small 5x7 (bf16) in 16 bits: those instances here are what MTA_CONV_FORCE_VALU=1 takes.
//
// A wavefront owns a strip of M rows and walks down the input rows.  A lane loads four consecutive keys of a row (one load
// instruction per row: 256 keys), several rows ahead, and takes the halo from its neighbours' registers (DPP shifts by one
// lane; the first and last one or two lanes carry halo only).  An input row is used once for all R output rows that it
// reaches, whose sums sit in registers and shift up by one per row.  No LDS tile, no barrier.
//   forward, input gradient: R*S*4 FMAs per row and lane; weights in scalar registers up to 35 taps, else read from LDS
//   kernel gradient:         the same FMAs into R*S sums per lane, against the R rows of dy that slide along; summed over the
//                            wavefront at the very end
// What bounds them: load instructions for small kernels (about 39 ns per 1 KB instruction and CU on this part, cache hit or
// not: fetching each lane's whole window, three to five loads per row, took 100 us where this takes 60 at 16 planes of
// 2048^2, 3x3), fp32 FMAs for large ones.  The 32x64-tile kernels these replace fetched element by element, one predicate
// each, and re-read every window from LDS.
// us, those -> these, fp32, forward | kernel gradient: 16 planes of 512^2 3x3 14 -> 11 | 23 -> 16, 6x11 20 -> 14 | 44 -> 22;
// 32 of 1024^2 3x3 82 -> 29 | 132 -> 36, 6x11 110 -> 51 | 172 -> 67, 11x15 168 -> 104 | 791 -> 142; 16 of 2048^2 3x3 229 -> 67 |
// 296 -> 61, 11x15 345 -> 174 | 1585 -> 232.
#pragma once

#include "common.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

template <typename T> struct alignas(sizeof(T)) quad4 { T v[4]; };   // (aligned to an element: rows of any width)

template <int S, bool REV> struct row_window {
    static constexpr int PADW = REV ? S - 1 - (S - 1) / 2 : (S - 1) / 2;   // keys to the left of an output key
    static constexpr int PADR = S - 1 - PADW;                             // ... to the right
    static constexpr int LL = (PADW + 3) / 4, LR = (PADR + 3) / 4;        // lanes that carry the left / right halo
    static constexpr int KEYS = 4 * (64 - LL - LR);                       // output keys per wavefront
    static constexpr int WIN = PADW + 4 + PADR;
};

// a neighbour's register: lane - 1 (lane + 1) of the wavefront, 0 beyond its end
__device__ __forceinline__ float from_left(float v) { return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x138, 0xf, 0xf, true)); }
__device__ __forceinline__ float from_right(float v) { return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x130, 0xf, 0xf, true)); }

// the window of a lane's four keys out of the lanes' own values
template <typename G> __device__ __forceinline__ void window_of(const float (&own)[4], float (&win)[G::WIN])
{
#pragma unroll
    for (int u = 0; u < 4; ++u) win[G::PADW + u] = own[u];
    float l[4] = {own[0], own[1], own[2], own[3]}, r[4] = {own[0], own[1], own[2], own[3]};
#pragma unroll
    for (int v = 0; v < G::LL; ++v)
#pragma unroll
        for (int u = 3; u >= 0; --u) {
            const int at = G::PADW - 4 * (v + 1) + u;
            if (at >= 0) win[at] = l[u] = from_left(l[u]);
        }
#pragma unroll
    for (int v = 0; v < G::LR; ++v)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int at = G::PADW + 4 * (v + 1) + u;
            if (at < G::WIN) win[at] = r[u] = from_right(r[u]);
        }
}

// four elements from key k (a multiple of 4) of a row; k outside the row re-reads the nearest vector inside (W >= 4)
template <typename T> __device__ __forceinline__ quad4<T> load_quad(const T *row, int k, int W)
{
    const int kc = k < 0 ? 0 : (k > W - 4 ? W - 4 : k);
    quad4<T> r;
    __builtin_memcpy(&r, row + kc, sizeof(r));
    return r;
}

// the values of such a vector where it may reach beyond the row or the diagonal: what lies outside [0, limit] counts as 0
template <typename T> __device__ __forceinline__ void masked_quad(const quad4<T> &r, int k, int W, int limit, float (&v)[4])
{
    const int sh = k > W - 4 ? k - (W - 4) : 0;   // (the load was moved back by so much)
    float l[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) l[u] = to_float(r.v[u]);
    if (sh & 1) { l[0] = l[1]; l[1] = l[2]; l[2] = l[3]; }
    if (sh & 2) { l[0] = l[2]; l[1] = l[3]; }
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = (k + u >= 0 && k + u <= limit) ? l[u] : 0.0f;
}

template <typename T> __device__ __forceinline__ void store_quad(T *row, int q, int W, const float (&v)[4])
{
    quad4<T> o;
#pragma unroll
    for (int u = 0; u < 4; ++u) o.v[u] = from_float<T>(v[u]);
    if (q + 4 <= W) {
        __builtin_memcpy(row + q, &o, sizeof(o));
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q + u < W) row[q + u] = o.v[u];
    }
}

// Strips of M rows x G::KEYS output keys of a plane that touch the lower triangle (all of them without the causal rule), column
// of strips by column of strips; strip number `id` of them.
template <typename G, int M> struct strips {
    static __host__ __device__ int first(int tn, int causal) { return causal ? tn * G::KEYS / M : 0; }   // its last row reaches key tn*KEYS
    static __host__ __device__ int64_t count(int H, int W, int causal)
    {
        const int tiles_m = (H + M - 1) / M, tiles_n = (W + G::KEYS - 1) / G::KEYS;
        int64_t n = 0;
        for (int tn = 0; tn < tiles_n; ++tn) n += tiles_m > first(tn, causal) ? tiles_m - first(tn, causal) : 0;
        return n;
    }
    static __device__ __forceinline__ void at(int id, int H, int causal, int &p0, int &q0)
    {
        const int tiles_m = (H + M - 1) / M;
        int tn = 0;
        for (int n; id >= (n = tiles_m > first(tn, causal) ? tiles_m - first(tn, causal) : 0); ++tn) id -= n;
        p0 = (first(tn, causal) + id) * M;
        q0 = tn * G::KEYS;
    }
};

// rows fetched ahead (the loop is unrolled by as many); 8 where a short strip has many halo rows (11x15, 8 planes of 256^2: 15.1 -> 13.0 us,
// under MTA_CONV_FORCE_VALU=1)
template <int R, int M> constexpr int rows_ahead() { return M == 4 && R > 7 ? 8 : 4; }

// y = conv(x) (BWD: the gradient with respect to x: kernel reversed in both axes, row halo below); M rows per strip
template <typename T, int R, int S, bool BWD, int M>
__global__ __launch_bounds__(256) void conv2d_rows(const T *__restrict__ x, const void *__restrict__ w, T *__restrict__ y, int C, int H, int W,
                                                   int causal, float in_scale, int use_scale, int w_dtype, int total)
{
    using G = row_window<S, BWD>;
    constexpr int RW_AHEAD = rows_ahead<R, M>();
    constexpr bool SREG = R * S <= 35;        // weights in scalar registers (more of them spill)
    constexpr int LDW = (S + 3) & ~3;
    __shared__ __align__(16) float wsm[R * LDW];
    const int64_t plane = blockIdx.y;
    const int c = (int)(plane % C);
    for (int t = threadIdx.x; t < R * LDW; t += 256) {
        const int i = t / LDW, j = t % LDW;
        wsm[t] = j < S ? load_any(w, w_dtype, (int64_t)c * R * S + (BWD ? R * S - 1 - (i * S + j) : i * S + j)) : 0.0f;
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + wave;
    if (tile >= total) return;
    int p0, q0;                                                             // first row and output key
    strips<G, M>::at(tile, H, causal == 2, p0, q0);                         // (causal == 1: the strips above the diagonal too)
    const int q = q0 + (lane - G::LL) * 4;                                  // this lane's keys
    const bool mine = lane >= G::LL && lane < 64 - G::LR && q < W;          // ... are output keys
    T *yp = y + plane * (int64_t)H * W;
    if (causal && q0 > p0 + M - 1) {          // wholly above the diagonal: +0, or nobody's business
        if (causal != 2) {
            const float z[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int r = 0; r < M; ++r)
                if (p0 + r < H && mine) store_quad<T>(yp + (int64_t)(p0 + r) * W, q, W, z);
        }
        return;
    }
    float ws[SREG ? R * S : 1];
    if constexpr (SREG) {
#pragma unroll
        for (int t = 0; t < R * S; ++t)
            ws[t] = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(wsm[t / S * LDW + t % S])));
    }
    const T *xp = x + plane * (int64_t)H * W;
    const int h0 = BWD ? p0 : p0 - (R - 1);   // input row of step 0
    const bool cols_inside = q0 - 4 * G::LL >= 0 && q0 + G::KEYS + 4 * G::LR <= W;
    quad4<T> ring[RW_AHEAD];
    auto fetch = [&](int n, int slot) __attribute__((always_inline)) {
        const int h = h0 + n, hc = h < 0 ? 0 : (h >= H ? H - 1 : h);
        ring[slot] = load_quad<T>(xp + (int64_t)hc * W, q, W);
    };
    float acc[R][4];                          // acc[k]: output row of step n - (R-1) + k
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[k][u] = 0.0f;
    constexpr int STEPS = M + R - 1;
    auto step = [&](int n, int slot) __attribute__((always_inline)) {
        const float *wp = wsm + (SREG ? 0 : opaque(0));   // (opaque: the weights are not to be kept in registers across rows)
        const int h = h0 + n;
        float own[4];
        if (cols_inside && h >= 0 && h < H && (!causal || q0 + G::KEYS + 4 * G::LR - 1 <= h)) {
#pragma unroll
            for (int u = 0; u < 4; ++u) own[u] = to_float(ring[slot].v[u]);
        } else {
            masked_quad<T>(ring[slot], q, W, (h < 0 || h >= H) ? -1 : (causal && h < W - 1 ? h : W - 1), own);
        }
        if (use_scale) {
#pragma unroll
            for (int u = 0; u < 4; ++u) own[u] = round_to<T>(own[u] * in_scale);
        }
        float win[G::WIN];
        window_of<G>(own, win);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int o = n - (R - 1) + k;    // (uniform) output row within the strip
            if (o < 0 || o >= M) continue;
            const int i = R - 1 - k;
            float wr[S];
#pragma unroll
            for (int j = 0; j < S; ++j) wr[j] = SREG ? ws[SREG ? i * S + j : 0] : wp[i * LDW + j];
#pragma unroll
            for (int j = 0; j < S; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[k][u] = fmaf(wr[j], win[j + u], acc[k][u]);
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
#pragma unroll
    for (int d = 0; d < RW_AHEAD - 1; ++d) fetch(d, d);
    for (int n = 0; n < STEPS; n += RW_AHEAD) {
#pragma unroll
        for (int d = 0; d < RW_AHEAD; ++d) {
            fetch(n + d + RW_AHEAD - 1, (d + RW_AHEAD - 1) % RW_AHEAD);
            if (n + d < STEPS) step(n + d, d);
        }
    }
}

// Rows per strip: enough strips for the chip (at 8 rows: `strips8` of them over all planes), then long ones, which fetch their
// R-1 halo rows less often.  us with 4 / 8 / 16 rows, forward: 8 planes of 256^2 (270 strips) 6x11 11.8 / 12.9 / 20.9; 16 of 512^2 (1600)
// 6x11 17.6 / 18.3 / 24.6; 16 of 1024^2 (5300) 3x3 19.6 / 18.3 / 17.3, 11x15 83 / 81 / 73; 16 of 2048^2 (19000) 3x3 58 / 57 / 64,
// 7x7 102 / 83 / 82, 11x15 246 / 214 / 202
inline int rows_per_strip(int64_t planes, int64_t H, int64_t W, int R, int S, int causal)
{
    const int64_t strips8 = planes * ((H + 7) / 8) * ((W + 239) / 240) / (causal && W > 240 ? 2 : 1);
    return strips8 < (R * S > 100 ? 3200 : 1600) ? 4 : (strips8 < 4000 || R <= 5) ? 8 : 16;
}

// returns 1 when (R,S) has no instance
template <typename T, bool BWD>
int dispatch_rows(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int R, int S, int causal, float in_scale,
                  int use_scale, int w_dtype, hipStream_t st)
{
    if (W < 4) return 1;
    const int m = rows_per_strip(N * C, H, W, R, S, causal);
    auto go = [&](auto kern, int64_t total) {
        if (total > 0x7fffff00LL) return (int)MTA_ERR_SHAPE;
        hipLaunchKernelGGL(kern, dim3((unsigned)((total + 3) / 4), (unsigned)(N * C)), dim3(256), 0, st, (const T *)x, w, (T *)y, (int)C, (int)H,
                           (int)W, causal, in_scale, use_scale, w_dtype, (int)total);
        return launch_status();
    };
#define MTA_ROWS(r, s, m) go(conv2d_rows<T, r, s, BWD, m>, strips<row_window<s, BWD>, m>::count((int)H, (int)W, causal == 2))
#define MTA_CONV_CASE(r, s) \
    if (R == r && S == s) return m == 4 ? MTA_ROWS(r, s, 4) : m == 8 ? MTA_ROWS(r, s, 8) : MTA_ROWS(r, s, (r <= 5 ? 8 : 16));
    MTA_CONV_CASE(3, 3)
    MTA_CONV_CASE(3, 5)
    MTA_CONV_CASE(5, 5)
    MTA_CONV_CASE(5, 7)
    MTA_CONV_CASE(6, 11)
    MTA_CONV_CASE(7, 7)
    MTA_CONV_CASE(7, 9)
    MTA_CONV_CASE(11, 15)
#undef MTA_CONV_CASE
#undef MTA_ROWS
    return 1;
}

// ---- kernel gradient ------------------------------------------------------------------------------------------------
// the sum over the wavefront, in its last lane (a fixed order; DPP adds: a row of 16, then rows into the rows behind them)
__device__ __forceinline__ float wave_total(float v)
{
#define MTA_DPP_ADD(ctrl, rows) v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), ctrl, rows, 0xf, false))
    MTA_DPP_ADD(0x111, 0xf);   // row_shr:1
    MTA_DPP_ADD(0x112, 0xf);
    MTA_DPP_ADD(0x114, 0xf);
    MTA_DPP_ADD(0x118, 0xf);
    MTA_DPP_ADD(0x142, 0xa);   // row_bcast:15 into rows 1 and 3
    MTA_DPP_ADD(0x143, 0xc);   // row_bcast:31 into rows 2 and 3
#undef MTA_DPP_ADD
    return v;
}

// dw[i,j] = sum over p, q of dy[p,q] * x[p+i-(R-1), q+j-pad], both with what lies above the diagonal (causal) or outside as 0.
// Workgroup b of a channel takes the channel's strips wave*bpc + b, + 4*bpc, ... and leaves one partial kernel.
// PARTS = 2 (11x15: 165 sums, the sliding rows and the window do not fit twice per SIMD): workgroups of part 0 form the first
// RP = (R+1)/2 kernel rows, those of part 1 the last RP; row RP-1 of an odd R is taken from part 0.
template <int R, int S> constexpr int weight_parts() { return R * S > 100 ? 2 : 1; }
template <typename T, int R, int S, int M>
__global__ __launch_bounds__(256) void conv2d_bwd_weight_rows(const T *__restrict__ x, const T *__restrict__ dy, float *__restrict__ partial, int N,
                                                              int C, int H, int W, int causal, int bpc, int tiles)
{
    using G = row_window<S, false>;
    constexpr int RW_AHEAD = 4;               // rows fetched ahead
    constexpr int PARTS = weight_parts<R, S>(), RP = PARTS == 2 ? (R + 1) / 2 : R;
    __shared__ float red[4][RP * S];
    const int part = blockIdx.y, c = blockIdx.x / bpc, b = blockIdx.x % bpc;
    const int up = (PARTS == 2 && part == 0) ? R - RP : 0;   // x rows of this part lie so much further up
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    float acc[RP][S];
#pragma unroll
    for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < S; ++j) acc[i][j] = 0.0f;
    constexpr int STEPS = M + RP - 1;
    for (int64_t it = (int64_t)wave * bpc + b; it < (int64_t)N * tiles; it += (int64_t)bpc * 4) {
        const int n_ = (int)(it / tiles);
        int p0, q0;
        strips<G, M>::at((int)(it - (int64_t)n_ * tiles), H, causal, p0, q0);
        const int q = q0 + (lane - G::LL) * 4;
        const bool mine = lane >= G::LL && lane < 64 - G::LR && q < W;
        const int64_t plane = ((int64_t)n_ * C + c) * H * (int64_t)W;
        const T *xp = x + plane, *gp = dy + plane;
        const int h0 = p0 - (RP - 1) - up;
        const bool cols_inside = q0 - 4 * G::LL >= 0 && q0 + G::KEYS + 4 * G::LR <= W;
        quad4<T> xr[RW_AHEAD], gr[RW_AHEAD];
        auto fetch = [&](int n, int slot) __attribute__((always_inline)) {
            const int h = h0 + n, hc = h < 0 ? 0 : (h >= H ? H - 1 : h);
            xr[slot] = load_quad<T>(xp + (int64_t)hc * W, q, W);
            const int p = p0 + n < H ? p0 + n : H - 1;
            gr[slot] = load_quad<T>(gp + (int64_t)p * W, q, W);
        };
        float g[RP][4];   // g[k]: dy of output row (step n) - (RP-1) + k within the strip, 0 outside it
#pragma unroll
        for (int k = 0; k < RP; ++k)
#pragma unroll
            for (int u = 0; u < 4; ++u) g[k][u] = 0.0f;
        auto step = [&](int n, int slot) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k + 1 < RP; ++k)
#pragma unroll
                for (int u = 0; u < 4; ++u) g[k][u] = g[k + 1][u];
            {   // the row of dy that enters (halo lanes: 0)
                const int p = p0 + n;
                masked_quad<T>(gr[slot], q, W, (!mine || n >= M || p >= H) ? -1 : (causal && p < W - 1 ? p : W - 1), g[RP - 1]);
            }
            const int h = h0 + n;
            float own[4];
            if (cols_inside && h >= 0 && h < H && (!causal || q0 + G::KEYS + 4 * G::LR - 1 <= h)) {
#pragma unroll
                for (int u = 0; u < 4; ++u) own[u] = to_float(xr[slot].v[u]);
            } else {
                masked_quad<T>(xr[slot], q, W, (h < 0 || h >= H) ? -1 : (causal && h < W - 1 ? h : W - 1), own);
            }
            float win[G::WIN];
            window_of<G>(own, win);
#pragma unroll
            for (int k = 0; k < RP; ++k) {
                const int o = n - (RP - 1) + k;
                if (o < 0 || o >= M) continue;   // (uniform; g is 0 there)
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int j = 0; j < S; ++j) acc[RP - 1 - k][j] = fmaf(g[k][u], win[j + u], acc[RP - 1 - k][j]);
            }
        };
#pragma unroll
        for (int d = 0; d < RW_AHEAD - 1; ++d) fetch(d, d);
        // (unrolled whole, the steps at both ends lose their dead FMAs: 3x3 at 16 planes of 1024^2 31 -> 23 us; not where that takes
        // the registers of the second wavefront per SIMD)
        constexpr int UNROLL = R * S > 100 || (R * S > 40 && M > 4) ? 1 : STEPS;
#pragma unroll UNROLL
        for (int n = 0; n < STEPS; n += RW_AHEAD) {
#pragma unroll
            for (int d = 0; d < RW_AHEAD; ++d) {
                fetch(n + d + RW_AHEAD - 1, (d + RW_AHEAD - 1) % RW_AHEAD);
                if (n + d < STEPS) step(n + d, d);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < RP; ++i)
#pragma unroll
        for (int j = 0; j < S; ++j) {
            const float s = wave_total(acc[i][j]);
            if (lane == 63) red[wave][i * S + j] = s;
        }
    __syncthreads();
    const int skip = (PARTS == 2 && part == 1 && 2 * RP > R) ? S : 0;   // (the row that part 0 has)
    for (int t = threadIdx.x + skip; t < RP * S; t += 256)
        partial[(int64_t)blockIdx.x * (R * S) + (part ? (R - RP) * S : 0) + t] = ((red[0][t] + red[1][t]) + red[2][t]) + red[3][t];
}

// returns false when (R,S) has no instance (nothing launched); bpc: partial kernels per channel, may be lowered
template <typename T>
bool launch_weight_rows(const void *x, const void *dy, float *partial, int &bpc, int64_t N, int64_t C, int64_t H, int64_t W, int R, int S,
                        int causal, hipStream_t st)
{
    if (W < 4) return false;
    const int m = rows_per_strip(N * C * (R * S > 100 ? 4 : 1), H, W, R, S, causal);   // (two workgroups a strip, see weight_parts, and each with half the rows)
    causal = causal ? 1 : 0;
    auto go = [&](auto kern, int parts, int64_t total) {
        if (total > 0x7fffff00LL) return false;
        // (one round of resident workgroups: up to four per CU, two or three for the kernels with more sums)
        int64_t most = ((R * S > 60 ? 512 : 1024) / parts + C - 1) / C;
        if (most > (N * total + 3) / 4) most = (N * total + 3) / 4;
        if (bpc > most) bpc = (int)most;
        hipLaunchKernelGGL(kern, dim3((unsigned)(C * bpc), (unsigned)parts), dim3(256), 0, st, (const T *)x, (const T *)dy, partial, (int)N, (int)C,
                           (int)H, (int)W, causal, bpc, (int)total);
        return true;
    };
#define MTA_ROWS(r, s, m) go(conv2d_bwd_weight_rows<T, r, s, m>, weight_parts<r, s>(), strips<row_window<s, false>, m>::count((int)H, (int)W, causal))
#define MTA_CONV_CASE(r, s) \
    if (R == r && S == s) return m == 4 ? MTA_ROWS(r, s, 4) : m == 8 ? MTA_ROWS(r, s, 8) : MTA_ROWS(r, s, (r <= 5 ? 8 : 16));
    MTA_CONV_CASE(3, 3)
    MTA_CONV_CASE(3, 5)
    MTA_CONV_CASE(5, 5)
    MTA_CONV_CASE(5, 7)
    MTA_CONV_CASE(6, 11)
    MTA_CONV_CASE(7, 7)
    MTA_CONV_CASE(7, 9)
    MTA_CONV_CASE(11, 15)
#undef MTA_CONV_CASE
#undef MTA_ROWS
    return false;
}
}  // namespace
