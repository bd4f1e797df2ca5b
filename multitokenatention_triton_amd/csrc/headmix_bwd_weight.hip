// Gradient of the head mixing with respect to its (C,C) weight:
//
//   dw[o,i] = sum_{n,p,q} dy[n,o,p,q] * x[n,i,p,q]          (causal: only q <= p take part)
//
// i.e. dW = dY X^T with the contraction running over every attended position of the (N,*,P,Q) tensors.  Both tensors
// are read exactly once.  Accumulation is fp32 and hierarchical (registers over a persistent wavefront's share, one
// partial matrix per workgroup in a scratch buffer, a second kernel adds the partials in a fixed order); the
// reference accumulates with fp32 tl.dot and fp64 atomics (triton_linear_head.py:193-278).
//
// Up to 32 heads take the matrix cores: A = dY (rows = output heads), B = X (columns = input heads), positions as the
// contraction index (v_mfma_f32_16x16x32 for 16-bit data, v_mfma_f32_16x16x4f32 - exact fp32 products, fp32 sums - for
// fp32).  Which position feeds which contraction slot is free as long as both operands agree: a lane (row r, group g) loads
// 16 contiguous bytes of a head's row and feeds them as they lie, so that a load instruction covers 64 contiguous bytes per
// row.  With at most 8 (4) heads the 16 operand rows are two (four) sets of the heads at different positions; the blocks of
// the product in which the sets meet themselves are the result, added up at the end, the others are dropped.  HBM-bound:
// B1 H32 S1024 fp32 422 -> 36 us against the generic kernel (one thread per pair of heads over an LDS tile), B1 H8 S256
// bf16 31 -> 15 us (both launches).  More heads take that kernel.
#include "common.hpp"
#include "mfma.hpp"

namespace {
using namespace mta;

constexpr int NT = 256;
// Rows are visited in an order that interleaves short and long ones (0, P-1, 1, P-2, ...), so that under the causal
// mask a pair of consecutive rows always carries P+1 positions.
__device__ __forceinline__ int interleaved_row(int j, int P) { return (j & 1) ? P - 1 - (j >> 1) : (j >> 1); }

typedef unsigned int u4 __attribute__((ext_vector_type(4)));

// One chunk of one query row: where it starts and where the row's attended positions end.
struct hm_unit {
    int64_t rowbase;
    int q0, last;
};

// How a wavefront reads a chunk of T x heads.  NB blocks of 16 operand rows; SETS sets of 16/SETS heads each per block (one
// block if more than one set); TT products (16 bit) or groups of four products (fp32) per chunk.
template <typename T, int NB, int SETS> struct hm_shape {
    static_assert(SETS == 1 || NB == 1, "sets of heads within one block");
    static constexpr int V = vec_of<T>::n;             // positions per load
    static constexpr int TT = (NB == 1 && SETS == 1 && V == 8) ? 8 : 4;
    static constexpr int STEP = 4 * V * SETS;          // positions per load instruction (and head)
    static constexpr int CHUNK = STEP * TT;            // positions per chunk
    static constexpr int HEADS = SETS == 1 ? 16 * NB : 16 / SETS;
};

// The chunk's operands of a lane: load t the V positions from q0 + STEP*t + V*(g + 4*set) on, of head 16a + (r % heads).
template <typename T, int NB, int SETS> struct hm_operands {
    u4 dy[NB][hm_shape<T, NB, SETS>::TT], x[NB][hm_shape<T, NB, SETS>::TT];
};

// 16 bytes from an address that is aligned to an element only; `total`: elements of the tensor (nothing beyond is read)
template <typename T> __device__ __forceinline__ u4 load_unaligned(const T *base, int64_t at, int64_t total)
{
    constexpr int V = vec_of<T>::n;
    u4 v = {0u, 0u, 0u, 0u};
    if (at + V <= total) {
        __builtin_memcpy(&v, base + at, 16);
    } else {
        T e[V];
#pragma unroll
        for (int i = 0; i < V; ++i) e[i] = at + i < total ? base[at + i] : from_float<T>(0.0f);
        __builtin_memcpy(&v, e, 16);
    }
    return v;
}

template <typename T, int NB, int SETS, bool ALIGNED>
__device__ __forceinline__ void hm_load(hm_operands<T, NB, SETS> &o, const T *x, const T *dy, const hm_unit &u, int64_t plane, int C,
                                        int r, int g, int64_t total)
{
    using G = hm_shape<T, NB, SETS>;
    const int q = u.q0 + G::V * (g + 4 * (r / (16 / SETS)));
    // every load is unconditional: a vector wholly beyond `last` re-reads the row start and is zeroed before use; a row of
    // the operands without a head repeats the last head's (what it leads to is dropped)
#pragma unroll
    for (int a = 0; a < NB; ++a) {
        const int h = a * 16 + r % (16 / SETS), hc = h < C ? h : C - 1;
        const int64_t at = u.rowbase + hc * plane;
        auto fetch = [&](const T *p, int t) -> u4 {
            const int qq = (q + G::STEP * t <= u.last) ? q + G::STEP * t : 0;
            if constexpr (ALIGNED) return *reinterpret_cast<const u4 *>(p + at + qq);
            else return load_unaligned<T>(p, at + qq, total);
        };
#pragma unroll
        for (int t = 0; t < G::TT; ++t) o.dy[a][t] = fetch(dy, t);
#pragma unroll
        for (int t = 0; t < G::TT; ++t) o.x[a][t] = fetch(x, t);
    }
}

template <typename T, int NB, int SETS>
__device__ __forceinline__ void hm_consume(f32x4 (&acc)[NB][NB], hm_operands<T, NB, SETS> &o, const hm_unit &u, int r, int g)
{
    using G = hm_shape<T, NB, SETS>;
    if (u.q0 + G::CHUNK - 1 > u.last) {  // the chunk straddles the end of the row: zero what lies beyond it, in both operands
                                         // (what x holds there need not even be finite)
        const int q = u.q0 + G::V * (g + 4 * (r / (16 / SETS)));
#pragma unroll
        for (int t = 0; t < G::TT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                unsigned keep;
                if constexpr (G::V == 8) {
                    const int e = q + G::STEP * t + 2 * v;
                    keep = (e <= u.last ? 0x0000ffffu : 0u) | (e + 1 <= u.last ? 0xffff0000u : 0u);
                } else {
                    keep = q + G::STEP * t + v <= u.last ? 0xffffffffu : 0u;
                }
#pragma unroll
                for (int a = 0; a < NB; ++a) {
                    o.dy[a][t][v] &= keep;
                    o.x[a][t][v] &= keep;
                }
            }
    }
#pragma unroll
    for (int t = 0; t < G::TT; ++t)
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (G::V == 8) {
                    mma16(acc[a][b], __builtin_bit_cast(frag8<T>, o.dy[a][t]), __builtin_bit_cast(frag8<T>, o.x[b][t]));
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(o.dy[a][t][v]), __uint_as_float(o.x[b][t][v]), acc[a][b], 0, 0, 0);
                }
            }
}

template <typename T, int NB, int SETS, bool ALIGNED>
__global__ __launch_bounds__(NT) void headmix_bwd_weight_mfma(const T *__restrict__ x, const T *__restrict__ dy, float *__restrict__ partial,
                                                              int N, int C, int P, int Q, int causal, int slots)
{
    using G = hm_shape<T, NB, SETS>;
    constexpr int LD = 16 * NB;
    __shared__ float red[NT / 64][LD * LD];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int64_t plane = (int64_t)P * Q, total = (int64_t)N * C * plane;
    f32x4 acc[NB][NB];
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Rows are taken in pairs (2k, 2k+1) of the interleaved order, a pair's chunks one after the other in `slots` places (the
    // most a pair has; few are empty), and the places of all pairs are dealt to the wavefronts one by one: wavefront i takes
    // the places i, i + nwaves, ... - the same number of chunks for each whatever the length, and neighbours read side by side.
    // The loads of a chunk are issued before the products of the chunk ahead of it (two operand sets take turns).
    const int64_t rows = (int64_t)N * P, pairs = (rows + 1) / 2;
    const int nwaves = gridDim.x * (NT / 64), wid = __builtin_amdgcn_readfirstlane(blockIdx.x * (NT / 64) + wave);
    const int pair_step = nwaves / slots, slot_step = nwaves % slots;
    int64_t k = wid / slots;
    int i = wid % slots;
    auto advance = [&] {
        k += pair_step;
        i += slot_step;
        if (i >= slots) {
            i -= slots;
            ++k;
        }
    };
    // the chunk of the place at or after (k, i); false where nothing is left
    auto unit_at = [&](hm_unit &u) -> bool {
        while (k < pairs) {
            int c = i;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int64_t rid = 2 * k + half;
                if (rid >= rows) break;
                const int n = (int)(rid / P), p = interleaved_row((int)(rid % P), P);
                u.last = causal ? (p < Q - 1 ? p : Q - 1) : Q - 1;  // last position of the row that takes part
                if (c * G::CHUNK <= u.last) {
                    u.rowbase = (int64_t)n * C * plane + (int64_t)p * Q;
                    u.q0 = c * G::CHUNK;
                    return true;
                }
                c -= u.last / G::CHUNK + 1;
            }
            advance();
        }
        return false;
    };
    hm_unit ua, ub;
    hm_operands<T, NB, SETS> oa, ob;
    bool ha = unit_at(ua);
    if (ha) hm_load<T, NB, SETS, ALIGNED>(oa, x, dy, ua, plane, C, r, g, total);
    while (ha) {
        advance();
        const bool hb = unit_at(ub);
        if (!hb) ub = ua;  // nothing follows: fetch the same chunk again, so that the loads in flight never depend on a branch
        hm_load<T, NB, SETS, ALIGNED>(ob, x, dy, ub, plane, C, r, g, total);
        hm_consume<T, NB, SETS>(acc, oa, ua, r, g);
        if (!hb) break;
        advance();
        ha = unit_at(ua);
        if (!ha) ua = ub;
        hm_load<T, NB, SETS, ALIGNED>(oa, x, dy, ua, plane, C, r, g, total);
        hm_consume<T, NB, SETS>(acc, ob, ub, r, g);
    }
    // acc[a][b][v] = product of operand rows 16a + 4g + v (dY) and 16b + r (X)
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[wave][(a * 16 + 4 * g + v) * LD + b * 16 + r] = acc[a][b][v];
    __syncthreads();
    for (int e = threadIdx.x; e < C * C; e += NT) {
        const int o = e / C, i = e % C;
        float s = 0.0f;
#pragma unroll
        for (int wv = 0; wv < NT / 64; ++wv)
#pragma unroll
            for (int k = 0; k < SETS; ++k) s += red[wv][(k * (LD / SETS) + o) * LD + k * (LD / SETS) + i];
        partial[(int64_t)blockIdx.x * (C * C) + e] = s;
    }
}

// Any dtype and head count up to 128: a workgroup stages KC positions of every head of both tensors in LDS (fp32,
// masked positions as 0) and keeps the C*C running sums in LDS as well; thread t owns pairs t, t+256, ...
constexpr int KC = 32;
template <typename T>
__global__ __launch_bounds__(NT) void headmix_bwd_weight_any(const T *__restrict__ x, const T *__restrict__ dy,
                                                             float *__restrict__ partial, int N, int C, int P, int Q,
                                                             int causal)
{
    extern __shared__ float smem[];
    float *xs = smem;                // C x (KC+1)
    float *gs = xs + C * (KC + 1);   // C x (KC+1)
    float *sums = gs + C * (KC + 1); // C x C
    const int tid = threadIdx.x;
    const int CC = C * C;
    const int64_t plane = (int64_t)P * Q;
    for (int pair = tid; pair < CC; pair += NT) sums[pair] = 0.0f;
    const int qchunks = (Q + KC - 1) / KC;
    const int64_t items = (int64_t)N * P * qchunks;
    for (int64_t it = blockIdx.x; it < items; it += gridDim.x) {
        const int qc = (int)(it % qchunks);
        const int64_t rid = it / qchunks;
        const int n = (int)(rid / P), p = interleaved_row((int)(rid % P), P);
        const int q0 = qc * KC;
        const int last = causal ? (p < Q - 1 ? p : Q - 1) : Q - 1;
        if (q0 > last) continue;
        __syncthreads();
        for (int e = tid; e < C * KC; e += NT) {
            const int h = e / KC, k = e % KC;
            const bool ok = q0 + k <= last;
            const int64_t idx = ((int64_t)n * C + h) * plane + (int64_t)p * Q + q0 + k;
            xs[h * (KC + 1) + k] = ok ? to_float(x[idx]) : 0.0f;
            gs[h * (KC + 1) + k] = ok ? to_float(dy[idx]) : 0.0f;
        }
        __syncthreads();
#pragma unroll 1
        for (int pair = tid; pair < CC; pair += NT) {
            const float *go = gs + (pair / C) * (KC + 1), *xi = xs + (pair % C) * (KC + 1);
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < KC; ++k) s = fmaf(go[k], xi[k], s);
            sums[pair] += s;  // only the owner thread touches this entry
        }
    }
    for (int pair = tid; pair < CC; pair += NT) partial[(int64_t)blockIdx.x * CC + pair] = sums[pair];
}

constexpr int64_t MAX_WS_BYTES = 8 << 20;  // partial matrices never take more than this

// Persistent workgroups (= partial matrices) for a problem, at most.  Matrix-core kernels: one per CU, which has 64 to 128 KB
// of loads in flight; more is slower (256 | 512 | 1024, us: bf16 B1 H16 S1024 10.2 | 11.6 | 13.2, S2048 25.9 | 28.9 | 34.0, B2 H32
// S2048 112 | 115 | 122, fp32 B1 H32 S1024 27.8 | 34.2 | 40.0).  launch_partials takes fewer where there are fewer chunks.
inline int num_blocks(int64_t N, int64_t C, int64_t P, int64_t Q)
{
    int64_t nb = C <= 32 ? 256 : 1024;
    const int64_t pairs = (N * P + 1) / 2;
    if (nb > pairs) nb = pairs;
    const int64_t cap = MAX_WS_BYTES / (C * C * (int64_t)sizeof(float));
    if (nb > cap) nb = cap;
    return (int)(nb < 1 ? 1 : nb);
}
}  // namespace

extern "C" int64_t mta_headmix_bwd_weight_workspace(int64_t N, int64_t C, int64_t P, int64_t Q)
{
    if (N <= 0 || C <= 0 || P <= 0 || Q <= 0 || C > 128) return 0;
    return (int64_t)num_blocks(N, C, P, Q) * C * C * (int64_t)sizeof(float);
}

namespace {
template <typename T>
int launch_partials(const T *x, const T *dy, float *partial, int &nb, int N, int C, int P, int Q, int causal, hipStream_t st)
{
    if (C <= 32) {
        const bool aligned = Q % vec_of<T>::n == 0 && aligned_to(x, 16) && aligned_to(dy, 16);
        auto go = [&](auto kern, int chunk) {
            // the most chunks that the two rows of a pair have: together they hold at most P + 2 attended positions when causal
            const int full = 2 * ((Q + chunk - 1) / chunk), slots = causal && P / chunk + 2 < full ? P / chunk + 2 : full;
            const int64_t places = ((int64_t)N * P + 1) / 2 * slots, enough = (places + NT / 64 - 1) / (NT / 64);
            if (nb > enough) nb = (int)enough;
            hipLaunchKernelGGL(kern, dim3(nb), dim3(NT), 0, st, x, dy, partial, N, C, P, Q, causal, slots);
        };
#define MTA_HM_CASE(nb_, sets)                                                                    \
    aligned ? go(headmix_bwd_weight_mfma<T, nb_, sets, true>, hm_shape<T, nb_, sets>::CHUNK)      \
            : go(headmix_bwd_weight_mfma<T, nb_, sets, false>, hm_shape<T, nb_, sets>::CHUNK)
        if (C <= 4) MTA_HM_CASE(1, 4);
        else if (C <= 8) MTA_HM_CASE(1, 2);
        else if (C <= 16) MTA_HM_CASE(1, 1);
        else MTA_HM_CASE(2, 1);
#undef MTA_HM_CASE
        return launch_status();
    }
    const size_t lds = sizeof(float) * (2 * (size_t)C * (KC + 1) + (size_t)C * C);
    auto kern = headmix_bwd_weight_any<T>;
    if (lds > 48 * 1024) {  // per device, so set on every such launch (a cheap host-side call)
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL(kern, dim3(nb), dim3(NT), lds, st, x, dy, partial, N, C, P, Q, causal);
    return launch_status();
}
}  // namespace

extern "C" int mta_headmix_bwd_weight_as(const void *x, const void *dy, void *dw, void *workspace, int64_t workspace_bytes, int64_t N,
                                         int64_t C, int64_t P, int64_t Q, int group_size, int causal, int io_dtype, int w_dtype, void *stream)
{
    if (!x || !dy || !dw || !workspace) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (N <= 0 || C <= 0 || P <= 0 || Q <= 0 || P > (1 << 24) || Q > (1 << 24) || N * P > 0x7fffffffLL) return MTA_ERR_SHAPE;
    if (C > 128) return MTA_ERR_SHAPE;
    if (group_size < 0 || (group_size > 0 && C % group_size != 0)) return MTA_ERR_GROUP;
    if (!aligned_to(x, dtype_size(io_dtype)) || !aligned_to(dy, dtype_size(io_dtype)) || !aligned_to(dw, dtype_size(w_dtype)) ||
        !aligned_to(workspace, 16))
        return MTA_ERR_ALIGN;
    int nb = num_blocks(N, C, P, Q);
    if (workspace_bytes < (int64_t)nb * C * C * (int64_t)sizeof(float)) return MTA_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    float *partial = (float *)workspace;
    int rc = MTA_OK;
    MTA_DISPATCH_IO(io_dtype, {
        rc = launch_partials<io_t>((const io_t *)x, (const io_t *)dy, partial, nb, (int)N, (int)C, (int)P, (int)Q, causal, st);
    });
    if (rc != MTA_OK) return rc;
    const mta_partials job{partial, dw, (int32_t)C, (int32_t)(C * C), nb, (int32_t)C, group_size, w_dtype, 1.0f};
    return mta_sum_partials(1, &job, stream);
}

extern "C" int mta_headmix_bwd_weight(const void *x, const void *dy, void *dw, void *workspace, int64_t workspace_bytes,
                                      int64_t N, int64_t C, int64_t P, int64_t Q, int causal, int io_dtype, void *stream)
{
    return mta_headmix_bwd_weight_as(x, dy, dw, workspace, workspace_bytes, N, C, P, Q, 0, causal, io_dtype, MTA_F32, stream);
}
