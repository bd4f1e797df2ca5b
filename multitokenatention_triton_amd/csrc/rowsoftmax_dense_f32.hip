// head mix -> row softmax -> head mix in one pass for fp32 scores and dense groups of 9 to 32 heads, both mixes on the
// matrix cores (v_mfma_f32_16x16x4f32: exact fp32 products, fp32 sums).
//
// A workgroup owns one query row of one mixing group; a wavefront takes 64 keys of every head per pass and keeps them in
// registers until they are written.  Lane (ln, kg) fetches keys 4ln .. 4ln+3 of head 16b + 4kg + v (16 bytes; an instruction
// covers 4 heads x 256 contiguous bytes).  Product j of step (b, v) has keys 4ln + j as columns and the heads 16b + 4kg + v,
// one per lane group, as contraction index; its result leaves the lane with the heads 16b + 4kg + v of the same keys: the
// operands of the second mix, and whole 16-byte vectors to store, without a move between lanes.
//
// Bound by memory: one read and one write of the attended scores, where a mixing kernel and a softmax kernel make two of each.
#include "common.hpp"
#include "mfma.hpp"

namespace {
using namespace mta;

// HB: blocks of 16 heads; NW: wavefronts; NV: passes of 64 keys per wavefront (rows of up to 64 * NW * NV keys)
template <int HB, int NW, int NV>
__global__ __launch_bounds__(64 * NW) void mix_softmax_dense_f32(const float *__restrict__ x, const void *__restrict__ w1,
                                                                 const void *__restrict__ w2, const float *__restrict__ kb,
                                                                 const int *__restrict__ row_lo, float *__restrict__ y, int C, int HG,
                                                                 int P, int Q, int causal, int w_dtype, int fill_upper, int stream)
{
    constexpr int NS = 4 * HB;   // heads per lane
    __shared__ float red[2][NW][16 * HB];   // [0] maxima, [1] sums
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, ln = lane & 15, kg = lane >> 4;
    const unsigned groups = C / HG;
    unsigned b = blockIdx.x;
    const int p = P - 1 - (int)(b % (unsigned)P);   // the longest rows first
    b /= (unsigned)P;
    const int g = (int)(b % groups);
    const int64_t n = b / groups;
    const int64_t plane = (int64_t)P * Q, base = (n * C + (int64_t)g * HG) * plane + (int64_t)p * Q;
    const int last = causal ? (p < Q - 1 ? p : Q - 1) : Q - 1;   // last attended key
    const int lo = row_lo ? first_key(row_lo, n * P + p, last) : 0;   // band mask: first visible key
    auto head = [&](int t) { return 16 * (t >> 2) + 4 * kg + (t & 3); };
    auto key0 = [&](int k) { return (k * NW + wave) * 64; };
    // a pass wholly beyond the attended keys, or wholly ahead of the first visible one, is neither read nor computed
    auto dead = [&](int k) { return key0(k) > last; };
    auto gone = [&](int k) { return dead(k) || key0(k) + 64 <= lo; };

    auto weights = [&](const void *w, float (&f)[HB][NS]) {   // f[ob][t]: output head 16 ob + ln, input head(t); 0 where there is none
#pragma unroll
        for (int ob = 0; ob < HB; ++ob)
#pragma unroll
            for (int t = 0; t < NS; ++t) {
                const int o = 16 * ob + ln, i = head(t);
                f[ob][t] = o < HG && i < HG ? load_any(w, w_dtype, (int64_t)(g * HG + o) * C + g * HG + i) : 0.0f;
            }
    };
    auto mix = [&](const float (&f)[HB][NS], const f32x4 (&in)[NS], f32x4 (&out)[NS]) {   // in[t][j], out[t][j]: head(t), key 4 ln + j
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int ob = 0; ob < HB; ++ob) {
                f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int t = 0; t < NS; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(f[ob][t], in[t][j], acc, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) out[4 * ob + v][j] = acc[v];
            }
    };

    f32x4 s[NV][NS];
    // (a lane beyond the attended keys re-reads the row start; what is no head counts as 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (gone(k)) continue;
        const int key = key0(k) + 4 * ln;
        const float *xp = x + base + (key <= last ? key : 0);
#pragma unroll
        for (int t = 0; t < NS; ++t) {
            const int h = head(t);
            const f32x4 v = *reinterpret_cast<const f32x4 *>(xp + (h < HG ? h : 0) * plane);
            s[k][t] = h < HG ? v : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    if (w1) {
        float f[HB][NS];
        weights(w1, f);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if (gone(k)) continue;
            f32x4 m[NS];
            mix(f, s[k], m);
#pragma unroll
            for (int t = 0; t < NS; ++t) s[k][t] = m[t];
        }
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        if (gone(k)) continue;
        const int key = key0(k) + 4 * ln;
        if (kb) {   // additive key bias of this batch entry
            const int at = key <= last ? key : 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float bias = kb[n * Q + at + j];
#pragma unroll
                for (int t = 0; t < NS; ++t) s[k][t][j] += bias;
            }
        }
        if (key + 3 > last || key < lo) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (key + j > last || key + j < lo) {
#pragma unroll
                    for (int t = 0; t < NS; ++t) s[k][t][j] = -INFINITY;
                }
        }
    }

    // over the 16 lanes of a group, then over the wavefronts (the maxima and the sums have a barrier each)
    float m[NS], inv[NS];
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        float v = -INFINITY;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if (gone(k)) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) v = fmaxf(v, s[k][t][j]);
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
        if (ln == 0) red[0][wave][head(t)] = v;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        float v = red[0][0][head(t)];
#pragma unroll
        for (int i = 1; i < NW; ++i) v = fmaxf(v, red[0][i][head(t)]);
        m[t] = v;
    }
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        // (m is -inf only where a mask hides every key of the row: NaN, as a softmax of all -inf gives)
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if (gone(k)) continue;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                s[k][t][j] = __builtin_amdgcn_exp2f((s[k][t][j] - m[t]) * 1.4426950408889634f);
                sum += s[k][t][j];
            }
        }
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        if (ln == 0) red[1][wave][head(t)] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        float v = red[1][0][head(t)];
#pragma unroll
        for (int i = 1; i < NW; ++i) v += red[1][i][head(t)];
        inv[t] = 1.0f / v;
    }

    float f2[HB][NS];
    if (w2) weights(w2, f2);
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int key = key0(k) + 4 * ln;
        f32x4 out[NS];
        if (gone(k)) {
            const float z = dead(k) ? 0.0f : __uint_as_float(hidden_bits(lo, last));
#pragma unroll
            for (int t = 0; t < NS; ++t) out[t] = f32x4{z, z, z, z};
        } else {
#pragma unroll
            for (int t = 0; t < NS; ++t)   // (what is no head has weight 0 and must be finite: its row sums are over zeros)
#pragma unroll
                for (int j = 0; j < 4; ++j) out[t][j] = head(t) < HG ? s[k][t][j] * inv[t] : 0.0f;
            if (w2) {
                f32x4 mixed[NS];
                mix(f2, out, mixed);
#pragma unroll
                for (int t = 0; t < NS; ++t) out[t] = mixed[t];
            }
            if (key + 3 > last) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (key + j > last) {
#pragma unroll
                        for (int t = 0; t < NS; ++t) out[t][j] = 0.0f;
                    }
            }
        }
        if (key >= Q || (key > last && !fill_upper)) continue;
#pragma unroll
        for (int t = 0; t < NS; ++t)
            if (head(t) < HG) store_out(reinterpret_cast<f32x4 *>(y + base + head(t) * plane + key), out[t], stream);
    }
}
}  // namespace

namespace mta {
// MTA_ERR_UNSUPPORTED where no instance covers the sizes (the caller has checked the arguments)
int mix_softmax_dense_f32_launch(const float *x, const void *w1, const void *w2, const float *kb, const int *row_lo, float *y, int64_t N,
                                 int64_t C, int64_t P, int64_t Q, int HG, int causal, int w_dtype, int fill_upper, hipStream_t st)
{
    if (HG < 9 || HG > 32 || Q % 4 != 0 || !aligned_to(x, 16) || !aligned_to(y, 16) || Q > mta_headmix_softmax_dense_f32_keys(HG))
        return MTA_ERR_UNSUPPORTED;
    const int64_t blocks = N * (C / HG) * P;
    const int stream = streams(N, C, P, Q, 4);
#define MTA_MSD_CASE(hb, nw, nv)                                                                                                   \
    if (HG <= 16 * (hb) && Q <= 64 * (nw) * (nv)) {                                                                                \
        hipLaunchKernelGGL((mix_softmax_dense_f32<hb, nw, nv>), dim3((unsigned)blocks), dim3(64 * (nw)), 0, st, x, w1, w2, kb,     \
                           row_lo, y, (int)C, HG, (int)P, (int)Q, causal, w_dtype, fill_upper, stream);                            \
        return launch_status();                                                                                                    \
    }
    MTA_MSD_CASE(1, 4, 1) MTA_MSD_CASE(1, 4, 2) MTA_MSD_CASE(1, 4, 4) MTA_MSD_CASE(1, 8, 4) MTA_MSD_CASE(1, 8, 8)
    MTA_MSD_CASE(2, 4, 1) MTA_MSD_CASE(2, 4, 2) MTA_MSD_CASE(2, 4, 4) MTA_MSD_CASE(2, 8, 4)
#undef MTA_MSD_CASE
    return MTA_ERR_UNSUPPORTED;
}
}  // namespace mta

// Longest row of the one-pass kernel above for fp32 scores and dense groups of `group_size` heads; 0: none.  (A row's scores
// stay in registers: 16 heads x 4096 keys over 512 threads, 32 heads x 2048.)
extern "C" int64_t mta_headmix_softmax_dense_f32_keys(int group_size)
{
    return group_size < 9 || group_size > 32 ? 0 : group_size <= 16 ? 4096 : 2048;
}
