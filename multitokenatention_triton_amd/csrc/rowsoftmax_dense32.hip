// head mix -> row softmax -> head mix in one pass for 16-bit scores and dense groups of 9 to 32 heads, both mixes on the matrix
// cores (groups of 16 have a kernel of their own that walks lists of rows, rowsoftmax_dense16.hip; fp32: rowsoftmax_dense_f32.hip).
//
// A workgroup owns one query row of one mixing group; a wavefront takes 128 keys of every head per pass and keeps them in registers
// until they are written.  Lane (ln, kg) fetches keys 8ln .. 8ln+7 of the heads 16b + 4kg + v (16 bytes each) and forms the
// column of a key from them with byte permutes: the B operand of a 16x16x16 product per 16 input and 16 output heads, which leaves
// the heads 16b + 4kg + v of the same key with the lane: what the second mix takes, and whole vectors to store, without a move
// between lanes.  Wavefronts without an attended key end at once (a barrier does not wait for them).
// Rounding points are those of the stages one by one: mixed scores (plus bias, rounded again), probabilities, mixed probabilities.
//
// Bound by memory: one read and one write of the attended scores, where a mixing kernel and a softmax kernel make two of each.
// What keeps it from that is the row's chain (load, reduce, barrier, reduce, barrier, store) with three to seven wavefronts per SIMD to
// cover it: the scores wait as packed pairs and their exponentials are formed twice; kept as fp32 (128 registers) 4 x 32 x 680^2 took 63
// us, not 47.  us, bf16, triangles, mixing and softmax kernels -> this: 4 x 32 x 680^2 99 -> 47 (band of S/4: 163 -> 44), 1 x 32 x 1024^2
// 44 -> 27, 2048^2 157 -> 96, 1 x 12 x 2048^2 66 -> 34, 4096^2 188 -> 103, 1 x 24 x 1024^2 354 -> 24; 4 or 8 wavefronts of a row alike.
#include "common.hpp"
#include "mfma.hpp"
#include "strip_common.hpp"

#include <type_traits>

namespace {
using namespace mta;

typedef short d32_s4 __attribute__((ext_vector_type(4)));
typedef _Float16 d32_h4 __attribute__((ext_vector_type(4)));
typedef unsigned int d32_u2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x4 mma4(bf16_t, d32_u2 a, d32_u2 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(d32_s4, a), __builtin_bit_cast(d32_s4, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma4(f16_t, d32_u2 a, d32_u2 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(d32_h4, a), __builtin_bit_cast(d32_h4, b), c, 0, 0, 0);
}

// over the 16 lanes of a DPP row, result in all of them
template <bool IS_MAX> __device__ __forceinline__ float over_row(float v)
{
#define MTA_FOLD(ctrl)                                                                                                     \
    {                                                                                                                      \
        const float o = __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), ctrl, 0xf, 0xf, false)); \
        v = IS_MAX ? fmaxf(v, o) : v + o;                                                                                  \
    }
    MTA_FOLD(0xB1)    // quad_perm [1,0,3,2]
    MTA_FOLD(0x4E)    // quad_perm [2,3,0,1]
    MTA_FOLD(0x141)   // row_half_mirror
    MTA_FOLD(0x140)   // row_mirror
#undef MTA_FOLD
    return v;
}

constexpr int TK = 128;   // keys per wavefront and pass

// wavefronts per SIMD that the registers are kept to
template <int HB, int NV, bool HAS2, bool MASKED> constexpr int dense_waves()
{
    return HB * NV == 1 ? 8 : HB * NV == 2 ? (HAS2 || MASKED ? 5 : 6) : HB == 2 && HAS2 ? 3 : 4;
}

// HB: blocks of 16 heads; NW: wavefronts; NV: passes (rows of up to TK * NW * NV keys)
template <typename T, int HB, int NW, int NV, bool HAS2, bool MASKED>
__global__ __launch_bounds__(64 * NW, (dense_waves<HB, NV, HAS2, MASKED>())) void mix_softmax_dense(const T *__restrict__ x, const T *__restrict__ w1, const T *__restrict__ w2,
                                                             const float *__restrict__ kb, const int *__restrict__ row_lo, T *__restrict__ y,
                                                             int C, int HG, int P, int Q, int causal, int fill_upper, int stream)
{
    __shared__ __align__(16) float red[2][NW][16 * HB];   // [0] maxima, [1] sums
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, ln = lane & 15, kg = lane >> 4;
    const unsigned groups = C / HG;
    unsigned b = blockIdx.x;
    const int p = P - 1 - (int)(b % (unsigned)P);   // the longest rows first
    b /= (unsigned)P;
    const int g = (int)(b % groups);
    const int64_t n = b / groups;
    const int64_t plane = (int64_t)P * Q, base = (n * C + (int64_t)g * HG) * plane + (int64_t)p * Q;
    const int last = causal ? (p < Q - 1 ? p : Q - 1) : Q - 1;   // last attended key
    const int lo = MASKED && row_lo ? first_key(row_lo, n * P + p, last) : 0;   // band mask: first visible key
    // tiles with a visible key: [first, end)
    const int first = lo / TK, end = last / TK + 1;
    auto tile = [&](int k) { return k * NW + wave; };
    auto live = [&](int k) { return tile(k) >= first && tile(k) < end; };
    auto head = [&](int t) { return 16 * (t >> 2) + 4 * kg + (t & 3); };   // t: head of this lane
    constexpr int NS = 4 * HB;
    // vector of head(t) from key `key` on: a uniform base and an offset per lane
    const int64_t lane_heads = 8 * kg * plane;
    auto at = [&](auto *tensor, int t, int key) {
        const int u = 16 * (t >> 2) + (t & 3);
        return reinterpret_cast<std::conditional_t<std::is_const<std::remove_pointer_t<decltype(tensor)>>::value, const u32x4, u32x4> *>(
            (char *)(tensor + base + (u < HG ? u : 0) * plane) + ((head(t) < HG ? lane_heads : 0) + 2 * key));
    };

    bool any = false;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        any |= live(k);
        if (live(k)) continue;
        const int key = tile(k) * TK + 8 * ln;   // +0 (NaN) ahead of the visible keys, and +0 beyond the attended ones on request
        if (key >= Q || (key > last && !fill_upper)) continue;
        const unsigned z = tile(k) < end ? hidden_bits(lo, last) : 0u;
#pragma unroll
        for (int t = 0; t < NS; ++t)
            if (head(t) < HG) store_out(at(y, t, key), u32x4{z, z, z, z}, stream);
    }
    if (!any) return;

    // (a lane beyond the attended keys re-reads the row start; what is no head counts as 0)
    u32x4 xv[NV][NS];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (!live(k)) continue;
        const int key = tile(k) * TK + 8 * ln;
#pragma unroll
        for (int t = 0; t < NS; ++t) xv[k][t] = *at(x, t, key <= last ? key : 0);
    }
    auto weights = [&](const T *w, d32_u2 (&f)[HB][HB]) {   // f[ob][ib]: output head 16 ob + ln, input heads 16 ib + 4 kg ..
#pragma unroll
        for (int ob = 0; ob < HB; ++ob)
#pragma unroll
            for (int ib = 0; ib < HB; ++ib) {
                const int o = 16 * ob + ln;
                unsigned e[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int i = 16 * ib + 4 * kg + v;
                    const bool in = o < HG && i < HG;
                    const unsigned raw = reinterpret_cast<const unsigned short *>(w)[(unsigned)(in ? (g * HG + o) * C + g * HG + i : 0)];
                    e[v] = in ? raw : 0u;
                }
                f[ob][ib] = d32_u2{e[0] | e[1] << 16, e[2] | e[3] << 16};
            }
    };
    auto mix = [&](const d32_u2 (&f)[HB][HB], const d32_u2 (&col)[HB], float (&out)[NS]) {
#pragma unroll
        for (int ob = 0; ob < HB; ++ob) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ib = 0; ib < HB; ++ib) acc = mma4(T{}, f[ob][ib], col[ib], acc);
#pragma unroll
            for (int v = 0; v < 4; ++v) out[4 * ob + v] = acc[v];
        }
    };
    d32_u2 f1[HB][HB];
    if (w1) weights(w1, f1);

    // mixed scores, rounded: pm[k][j][t/2]: key 8 ln + j of the tile, heads head(t) and head(t + 1); -inf where they are hidden
    unsigned pm[NV][8][NS / 2];
    const unsigned hidden = pack2<T>(-INFINITY, -INFINITY);
    float m[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) m[t] = -INFINITY;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (!live(k)) continue;
        const int key = tile(k) * TK + 8 * ln;
#pragma unroll
        for (int t = 0; t < NS; ++t)
            if (head(t) >= HG) xv[k][t] = u32x4{0u, 0u, 0u, 0u};
        float bias[8] = {};   // additive key bias, added in the I/O dtype (without one: 0, which changes no score)
        if (MASKED && kb) __builtin_memcpy(bias, kb + n * Q + (key <= last ? key : 0), sizeof(bias));
        const bool edge = tile(k) * TK + TK - 1 > last || tile(k) * TK < lo;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const unsigned sel = (j & 1) ? 0x07060302u : 0x05040100u;
            d32_u2 col[HB];
#pragma unroll
            for (int ib = 0; ib < HB; ++ib)
                col[ib] = d32_u2{__builtin_amdgcn_perm(xv[k][4 * ib + 1][j >> 1], xv[k][4 * ib][j >> 1], sel),
                                 __builtin_amdgcn_perm(xv[k][4 * ib + 3][j >> 1], xv[k][4 * ib + 2][j >> 1], sel)};
            if (w1) {
                float out[NS];
                mix(f1, col, out);
#pragma unroll
                for (int ib = 0; ib < HB; ++ib)
                    col[ib] = d32_u2{pack2<T>(out[4 * ib], out[4 * ib + 1]), pack2<T>(out[4 * ib + 2], out[4 * ib + 3])};
            }
#pragma unroll
            for (int t = 0; t < NS; t += 2) {
                unsigned v = col[t / 4][t / 2 % 2];
                float e0, e1;
                unpack2<T>(v, e0, e1);
                if constexpr (MASKED) {
                    v = pack2<T>(e0 + bias[j], e1 + bias[j]);
                    unpack2<T>(v, e0, e1);
                }
                if (edge && (key + j > last || key + j < lo)) {
                    v = hidden;
                    e0 = e1 = -INFINITY;
                }
                pm[k][j][t / 2] = v;
                m[t] = fmaxf(m[t], e0);
                m[t + 1] = fmaxf(m[t + 1], e1);
            }
            if (j & 1) __builtin_amdgcn_sched_barrier(0);   // (or all 32 products' results would be held at once)
        }
    }

    // over the 16 lanes of a group, then over the wavefronts that have a tile (the maxima and the sums have a barrier each)
    const int n_live = end - first < NW ? end - first : NW;
    auto combine = [&](auto is_max, float (&v)[NS]) {
        constexpr bool IS_MAX = decltype(is_max)::value;
#pragma unroll
        for (int t = 0; t < NS; ++t) v[t] = over_row<IS_MAX>(v[t]);
        if (n_live == 1) return;
        float (&r)[NW][16 * HB] = red[IS_MAX ? 0 : 1];
        if (ln == 0) {
#pragma unroll
            for (int ib = 0; ib < HB; ++ib)
                *reinterpret_cast<f32x4 *>(&r[wave][16 * ib + 4 * kg]) = f32x4{v[4 * ib], v[4 * ib + 1], v[4 * ib + 2], v[4 * ib + 3]};
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NS; ++t) v[t] = IS_MAX ? -INFINITY : 0.0f;
        for (int i = 0; i < n_live; ++i) {
#pragma unroll
            for (int ib = 0; ib < HB; ++ib) {
                const f32x4 e = *reinterpret_cast<const f32x4 *>(&r[(first + i) % NW][16 * ib + 4 * kg]);
#pragma unroll
                for (int u = 0; u < 4; ++u) v[4 * ib + u] = IS_MAX ? fmaxf(v[4 * ib + u], e[u]) : v[4 * ib + u] + e[u];
            }
        }
    };
    // (what the packed scores unpack to, and the exponentials, are not to be kept from one phase to the next: scratch)
    auto forget = [&]() {
#pragma unroll
        for (int k = 0; k < NV; ++k)
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int t = 0; t < NS / 2; ++t) asm volatile("" : "+v"(pm[k][j][t]));
    };
    combine(std::true_type{}, m);
    forget();
    constexpr float LOG2E = 1.4426950408889634f;
    // (m is -inf only where a mask hides every key of the row: NaN, as a softmax of all -inf gives)
    float sum[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        sum[t] = 0.0f;
        m[t] = -m[t] * LOG2E;
    }
    // the exponentials of a key's heads (formed twice, for the sums and for the probabilities: half the registers of keeping them)
    auto exponentials = [&](int k, int j, float (&e)[NS]) {
#pragma unroll
        for (int t = 0; t < NS; t += 2) {
            unpack2<T>(pm[k][j][t / 2], e[t], e[t + 1]);
            e[t] = __builtin_amdgcn_exp2f(fmaf(e[t], LOG2E, m[t]));   // (-inf -> 0)
            e[t + 1] = __builtin_amdgcn_exp2f(fmaf(e[t + 1], LOG2E, m[t + 1]));
        }
    };
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (!live(k)) continue;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float e[NS];
            exponentials(k, j, e);
#pragma unroll
            for (int t = 0; t < NS; ++t) sum[t] += e[t];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    combine(std::false_type{}, sum);
    forget();
#pragma unroll
    for (int t = 0; t < NS; ++t) {   // 1/sum: the hardware reciprocal and one Newton step
        const float rc = __builtin_amdgcn_rcpf(sum[t]);
        sum[t] = fmaf(fmaf(-sum[t], rc, 1.0f), rc, rc);
    }

    d32_u2 f2[HB][HB];
    if constexpr (HAS2) weights(w2, f2);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (!live(k)) continue;
        const int key = tile(k) * TK + 8 * ln;
        u32x4 out[NS];
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
            float e[2][NS];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                exponentials(k, j + u, e[u]);
#pragma unroll
                for (int t = 0; t < NS; ++t) e[u][t] *= sum[t];
                if (HAS2) {
                    d32_u2 col[HB];
#pragma unroll
                    for (int ib = 0; ib < HB; ++ib)
                        col[ib] = d32_u2{pack2<T>(e[u][4 * ib], e[u][4 * ib + 1]), pack2<T>(e[u][4 * ib + 2], e[u][4 * ib + 3])};
                    mix(f2, col, e[u]);
                }
            }
#pragma unroll
            for (int t = 0; t < NS; ++t) out[t][j / 2] = pack2<T>(e[0][t], e[1][t]);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (tile(k) * TK + TK - 1 > last) {   // +0 beyond the last attended key: 0 * NaN where the row's sum is NaN, 0 * inf in the second mix
#pragma unroll
            for (int t = 0; t < NS; ++t) zero_beyond<T>(out[t], key, last);
        }
        if (key >= Q || (key > last && !fill_upper)) continue;
#pragma unroll
        for (int t = 0; t < NS; ++t)
            if (head(t) < HG) store_out(at(y, t, key), out[t], stream);
    }
}
}  // namespace

// Longest row of the kernel above for 16-bit scores and dense groups of `group_size` heads; 0: none.  (A row's scores stay in
// registers: 16 heads x 4096 keys over 1024 threads, 32 heads x 2048.)
extern "C" int64_t mta_headmix_softmax_dense16_keys(int group_size)
{
    return group_size < 9 || group_size > 32 ? 0 : group_size <= 16 ? 4096 : 2048;
}

namespace mta {
// MTA_ERR_UNSUPPORTED where no instance covers the sizes (the caller has checked the arguments)
int mix_softmax_dense_launch(const void *x, const void *w1, const void *w2, const float *kb, const int *row_lo, void *y, int64_t N,
                             int64_t C, int64_t P, int64_t Q, int HG, int causal, int io_dtype, int w_dtype, int fill_upper, hipStream_t st)
{
    if (w_dtype != io_dtype || Q % 8 != 0 || !aligned_to(x, 16) || !aligned_to(y, 16) || Q > mta_headmix_softmax_dense16_keys(HG))
        return MTA_ERR_UNSUPPORTED;
    const int64_t blocks = N * (C / HG) * P;
    const int stream = streams(N, C, P, Q, 2);
    auto go = [&](auto type) -> int {
        using T = decltype(type);
        const bool masked = kb || row_lo;
        auto run = [&](auto kern, int nw) {
            hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * nw), 0, st, (const T *)x, (const T *)w1, (const T *)w2, kb, row_lo,
                               (T *)y, (int)C, HG, (int)P, (int)Q, causal, fill_upper, stream);
            return launch_status();
        };
#define MTA_MSD_CASE(hb, nw, nv)                                                                                                   \
    if (HG <= 16 * (hb) && Q <= TK * (nw) * (nv))                                                                                  \
        return w2 ? (masked ? run(mix_softmax_dense<T, hb, nw, nv, true, true>, nw) : run(mix_softmax_dense<T, hb, nw, nv, true, false>, nw)) \
                  : (masked ? run(mix_softmax_dense<T, hb, nw, nv, false, true>, nw) : run(mix_softmax_dense<T, hb, nw, nv, false, false>, nw));
        MTA_MSD_CASE(1, 2, 1) MTA_MSD_CASE(1, 4, 1) MTA_MSD_CASE(1, 4, 2) MTA_MSD_CASE(1, 4, 4) MTA_MSD_CASE(1, 8, 4)
        MTA_MSD_CASE(2, 2, 1) MTA_MSD_CASE(2, 4, 1) MTA_MSD_CASE(2, 4, 2) MTA_MSD_CASE(2, 8, 2)
#undef MTA_MSD_CASE
        return MTA_ERR_UNSUPPORTED;
    };
    return io_dtype == MTA_BF16 ? go(bf16_t{}) : io_dtype == MTA_F16 ? go(f16_t{}) : (int)MTA_ERR_UNSUPPORTED;
}
}  // namespace mta
