// Fused conv-attention forward:  O = softmax( mask( conv( mask0(Q K^T) ) ) * scale ) V
//
// One workgroup (4 wavefronts) owns a block of query rows of one (batch, head) and
// streams over the keys left to right.  No S x S tensor touches global memory: score
// tiles live in LDS, the conv reads them there, probabilities stay in registers.
//
// Orientation.  Every matrix product is issued "transposed" so that a lane always
// owns one query row:
//     S^T = K Q^T     A = K tile (LDS),        B = Q^T (registers, loaded once)
//     O^T = V^T P^T   A = V^T tile (LDS),      B = P^T (registers, straight from softmax)
// With the 32x32 MFMA accumulator layout (lane = column, 16 rows per lane) this puts the
// 16 keys of a score block that belong to one query row into one lane, so the softmax
// row reductions are in-lane plus one exchange with lane^32, the running max / sum and
// the O rescale are per-lane scalars, and P needs no LDS round trip: the MFMA contraction
// index may be permuted freely as long as both operands agree, so V^T is stored in LDS in
// the key order in which the accumulator layout hands out P.
//
// Tile geometry.  The score tile has 128 rows: HR = roundup(R-1, 8) halo rows above the
// block (recomputed, their outputs are discarded) + BQ = 128-HR output rows.  Keys are
// consumed in blocks of 64.  The conv's key halo is NOT recomputed: the last HC =
// roundup(Sk-1, 8) score columns of the previous block stay in LDS, and the conv /
// softmax / PV of a block lag the scores by the right-hand pad so that every tap is
// already there.  One extra leading key block (mostly out-of-range keys) primes that halo.
#include <algorithm>
#include <cmath>

#include <algorithm>

#include <type_traits>
#include <utility>

#include "conv_attn.hpp"
#include "mfma.hpp"

#include <stdlib.h>

namespace {
using namespace mta;

constexpr int NT = 256;  // 4 wavefronts
constexpr int SR = 128;  // score-tile rows (32 per wavefront)
constexpr int BK = 64;   // keys per iteration

// position of key offset k16 (0..15) inside its 16-key group of the V^T tile: the order in
// which a lane's accumulator registers enumerate the keys of a 32x32 block (see header).
__device__ __forceinline__ int vt_pos16(int k16) { return ((k16 >> 2) & 1) * 8 + (k16 >> 3) * 4 + (k16 & 3); }

template <typename T> struct lds_pad { static constexpr int n = 16 / sizeof(T); };  // 16 bytes of padding per row

// RT, SKT: the kernel size where it is known at compile time (fp32 instances), 0 = any (R and Sk from the arguments).  With
// it the conv keeps its 32 outputs in registers, reads a kernel row's weights once for all of them and the score windows as
// 16-byte vectors; read element by element behind run-time loop bounds the conv was a chain of LDS latencies (B1 H12 S64
// D128, 5x7, fp32: 41 us for two key blocks).
template <typename T, int D, int RT, int SKT>
__global__ __launch_bounds__(NT) void conv_attn_fwd_kernel(const T *__restrict__ Q, const T *__restrict__ K,
                                                           const T *__restrict__ V, const void *__restrict__ Wt,
                                                           T *__restrict__ O, float *__restrict__ Lse, int S, int R_,
                                                           int Sk_, int causal, float scale, int w_dtype, int H, int nqb)
{
    static_assert((RT > 0) == (SKT > 0) && (RT == 0 || sizeof(T) == 4), "compile-time sizes: fp32 only");
    const int R = RT > 0 ? RT : R_, Sk = SKT > 0 ? SKT : Sk_;
    constexpr int VEC = vec_of<T>::n;           // elements per 16-byte vector
    constexpr int PAD = lds_pad<T>::n;
    constexpr int KLD = D + PAD;                // K tile row stride
    constexpr int VLD = BK + PAD;               // V^T tile row stride
    constexpr int KS = D / 16;                  // contraction steps over the head dim
    constexpr int DB = D / 32;                  // 32-wide blocks of the head dim
    constexpr int KV_IT = BK * D / VEC / NT;    // 16-byte vectors per thread per K (or V) tile

    const int HR = (R - 1 + 7) & ~7;
    const int HC = (Sk - 1 + 7) & ~7;
    const int BQ = SR - HR;
    const int pw = (Sk - 1) / 2, pwr = Sk - 1 - pw;
    const int SLD = HC + BK + PAD;              // score tile row stride

    extern __shared__ __align__(16) unsigned char smem_raw[];
    T *Ks = reinterpret_cast<T *>(smem_raw);
    T *Vt = Ks + BK * KLD;
    T *Sc = Vt + D * VLD;
    float *Ws = reinterpret_cast<float *>(Sc + SR * SLD);

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, ln = lane & 31, hf = lane >> 5;
    const int qb = nqb - 1 - (int)blockIdx.x;   // longest blocks first
    const int64_t bh = blockIdx.y;
    const int head = (int)(bh % H);
    const int q0 = qb * BQ;
    const int tr = wave * 32 + ln;              // this lane's row in the score tile
    const int p = q0 - HR + tr;                 // ... and its query row
    const T *Qp = Q + bh * (int64_t)S * D;
    const T *Kp = K + bh * (int64_t)S * D;
    const T *Vp = V + bh * (int64_t)S * D;
    T *Op = O + bh * (int64_t)S * D;

    for (int t = tid; t < R * Sk; t += NT) Ws[t] = load_any(Wt, w_dtype, (int64_t)head * R * Sk + t);

    // Q^T fragments of this lane's row, kept for the whole kernel
    frag8<T> qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        if (p >= 0 && p < S) {
            qf[ks] = *reinterpret_cast<const frag8<T> *>(Qp + (int64_t)p * D + ks * 16 + hf * 8);
        } else {
            qf[ks] = zero_frag<T>();
        }
    }

    f32x16 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[db][v] = 0.0f;
    float m_i = -INFINITY, l_i = 0.0f;

    const int q_last = (q0 + BQ - 1 < S - 1) ? q0 + BQ - 1 : S - 1;
    const int j_end = causal ? q_last / BK : (S - 1) / BK;
    const int j_start = pwr > 0 ? -1 : 0;
    const int tail_vecs = SR * (HC / VEC);      // 16-byte vectors in the retained score columns
    constexpr int TAIL_IT = RT > 0 ? (SR * ((SKT - 1 + 7) & ~7) / VEC + NT - 1) / NT : SR * 64 / VEC / NT;  // (any size: HC <= 64)

    using V16 = pack16<T>;
    for (int j = j_start; j <= j_end; ++j) {
        const int cb = j * BK + pwr;            // first key of the new score block
        // ---- global loads of the K block (keys cb..) and the V block (keys j*BK..) -------
        V16 kreg[KV_IT], vreg[KV_IT];
#pragma unroll
        for (int it = 0; it < KV_IT; ++it) {
            const int idx = it * NT + tid;
            const int row = idx / (D / VEC), vc = idx % (D / VEC);
            // unconditional loads (an out-of-range key re-reads key 0) so that they are issued back to back;
            // out-of-range rows are zeroed when they are written to LDS
            const int kr = cb + row;
            const int vr = j * BK + row;
            kreg[it] = *reinterpret_cast<const V16 *>(Kp + (int64_t)((kr >= 0 && kr < S) ? kr : 0) * D + vc * VEC);
            vreg[it] = *reinterpret_cast<const V16 *>(Vp + (int64_t)((vr >= 0 && vr < S) ? vr : 0) * D + vc * VEC);
        }
        // ---- retained score columns: read the tail of the previous tile ----------------------
        V16 tailreg[TAIL_IT];
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it) {
            const int idx = it * NT + tid;
            if (idx < tail_vecs) {
                const int row = idx / (HC / VEC), vc = idx % (HC / VEC);
                tailreg[it] = *reinterpret_cast<const V16 *>(Sc + row * SLD + BK + vc * VEC);
            }
        }
        __syncthreads();  // everyone is done reading the previous K, V^T and score tiles
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it) {
            const int idx = it * NT + tid;
            if (idx < tail_vecs) {
                const int row = idx / (HC / VEC), vc = idx % (HC / VEC);
                *reinterpret_cast<V16 *>(Sc + row * SLD + vc * VEC) = tailreg[it];
            }
        }
#pragma unroll
        for (int it = 0; it < KV_IT; ++it) {
            const int idx = it * NT + tid;
            const int row = idx / (D / VEC), vc = idx % (D / VEC);
            const int kr = cb + row, vr = j * BK + row;
            const bool k_ok = kr >= 0 && kr < S, v_ok = vr >= 0 && vr < S;
            V16 kv = kreg[it];
            if (!k_ok) {
#pragma unroll
                for (int u = 0; u < VEC; ++u) kv.v[u] = from_float<T>(0.0f);
            }
            *reinterpret_cast<V16 *>(Ks + row * KLD + vc * VEC) = kv;
            const int pos = (row & ~15) + vt_pos16(row & 15);
#pragma unroll
            for (int u = 0; u < VEC; ++u) Vt[(vc * VEC + u) * VLD + pos] = v_ok ? vreg[it].v[u] : from_float<T>(0.0f);
        }
        __syncthreads();

        // ---- S^T = K Q^T for this wavefront's 32 rows; causal zero; to LDS in the I/O dtype ----
#pragma unroll
        for (int kb = 0; kb < BK / 32; ++kb) {
            f32x16 sacc;
#pragma unroll
            for (int v = 0; v < 16; ++v) sacc[v] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const frag8<T> kf = *reinterpret_cast<const frag8<T> *>(Ks + (kb * 32 + ln) * KLD + ks * 16 + hf * 8);
                mma32(sacc, kf, qf[ks]);
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct alignas(sizeof(T) * 4) quad { T v[4]; } out;
                const int xo = kb * 32 + g * 8 + hf * 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int col = cb + xo + r;
                    out.v[r] = from_float<T>((causal && col > p) ? 0.0f : sacc[g * 4 + r]);
                }
                *reinterpret_cast<quad *>(Sc + tr * SLD + HC + xo) = out;
            }
        }
        __syncthreads();
        if (j < 0) continue;

        // ---- conv over the LDS score tile (fp32 FMAs), scale, mask ---------------------------------
        float s[BK / 32][4][4];
        float mloc = -INFINITY;
        if constexpr (RT > 0) {
            constexpr int SH = ((SKT - 1 + 7) & ~7) - (SKT - 1);   // first tap's column for output column 0 of the block
            constexpr int W0 = SH & ~3, WOFF = SH & 3;             // the aligned start of a window, and the tap's place in it
            constexpr int WV = (WOFF + 4 + SKT - 1 + 3) / 4;       // vectors per window
#pragma unroll
            for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[kb][g][r] = 0.0f;
#pragma unroll 1
            for (int i = 0; i < RT; ++i) {
                float w[SKT];
#pragma unroll
                for (int jj = 0; jj < SKT; ++jj) w[jj] = Ws[i * SKT + jj];
                const int srow = tr - (RT - 1) + i;                // (above the tile: a halo row, its result is dropped)
                const float *src = reinterpret_cast<const float *>(Sc) + (srow < 0 ? 0 : srow) * SLD + W0 + hf * 4;
#pragma unroll
                for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        float x[WV * 4];
#pragma unroll
                        for (int u = 0; u < WV; ++u) {
                            const float4 t4 = *reinterpret_cast<const float4 *>(src + kb * 32 + g * 8 + u * 4);
                            x[u * 4] = t4.x; x[u * 4 + 1] = t4.y; x[u * 4 + 2] = t4.z; x[u * 4 + 3] = t4.w;
                        }
#pragma unroll
                        for (int jj = 0; jj < SKT; ++jj)
#pragma unroll
                            for (int r = 0; r < 4; ++r) s[kb][g][r] = fmaf(w[jj], x[WOFF + jj + r], s[kb][g][r]);
                    }
            }
        } else {
#pragma unroll
        for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int xo = kb * 32 + g * 8 + hf * 4;
                const int xb = HC - (Sk - 1) + xo;
                float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
                for (int i = 0; i < R; ++i) {
                    const int srow = tr - (R - 1) + i;
                    if (srow < 0) continue;
                    const T *src = Sc + srow * SLD + xb;
                    float w0 = to_float(src[0]), w1 = to_float(src[1]), w2 = to_float(src[2]);
                    for (int jj = 0; jj < Sk; ++jj) {
                        const float w3 = to_float(src[jj + 3]);
                        const float wv = Ws[i * Sk + jj];
                        a0 = fmaf(wv, w0, a0);
                        a1 = fmaf(wv, w1, a1);
                        a2 = fmaf(wv, w2, a2);
                        a3 = fmaf(wv, w3, a3);
                        w0 = w1; w1 = w2; w2 = w3;
                    }
                }
                s[kb][g][0] = a0; s[kb][g][1] = a1; s[kb][g][2] = a2; s[kb][g][3] = a3;
            }
        }
#pragma unroll
        for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int xo = kb * 32 + g * 8 + hf * 4;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int col = j * BK + xo + r;
                    const bool ok = col < S && (!causal || col <= p);
                    const float val = round_to<T>(round_to<T>(s[kb][g][r]) * scale);
                    s[kb][g][r] = ok ? val : -INFINITY;
                    mloc = fmaxf(mloc, s[kb][g][r]);
                }
            }

        // ---- online softmax: this row is split over lanes ln and ln+32 -----------------------------
        const float mrow = fmaxf(mloc, __shfl_xor(mloc, 32));
        const float m_new = fmaxf(m_i, mrow);
        const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
        const float alpha = __expf(m_i - m_use);
        m_i = m_new;
        float lsum = 0.0f;
        frag8<T> pf[BK / 32][2];
#pragma unroll
        for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float e = __expf(s[kb][g][r] - m_use);
                    const T et = from_float<T>(e);
                    lsum += to_float(et);
                    pf[kb][g >> 1].v[(g & 1) * 4 + r] = et;
                }
        l_i = l_i * alpha + lsum;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int v = 0; v < 16; ++v) oacc[db][v] *= alpha;

        // ---- O^T += V^T P^T -----------------------------------------------------------------------
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int kb = 0; kb < BK / 32; ++kb)
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    const frag8<T> vf =
                        *reinterpret_cast<const frag8<T> *>(Vt + (db * 32 + ln) * VLD + kb * 32 + ks * 16 + hf * 8);
                    mma32(oacc[db], vf, pf[kb][ks]);
                }
    }

    // ---- normalise and store this lane's row (halo rows are dropped) -----------------------------------
    const float l_row = l_i + __shfl_xor(l_i, 32);
    if (tr >= HR && p < S) {
        const float inv = 1.0f / l_row;
        if (Lse != nullptr && hf == 0) Lse[bh * (int64_t)S + p] = m_i + __logf(l_row);
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct alignas(sizeof(T) * 4) quad { T v[4]; } out;
#pragma unroll
                for (int r = 0; r < 4; ++r) out.v[r] = from_float<T>(oacc[db][g * 4 + r] * inv);
                *reinterpret_cast<quad *>(Op + (int64_t)p * D + db * 32 + g * 8 + hf * 4) = out;
            }
    }
}

template <typename T, int D, int RT = 0, int SKT = 0>
int launch(const void *q, const void *k, const void *v, const void *w, void *o, float *lse, int64_t B, int64_t H,
           int64_t S, int R, int Sk, int causal, float scale, int w_dtype, hipStream_t st)
{
    constexpr int PAD = lds_pad<T>::n;
    const int HR = (R - 1 + 7) & ~7, HC = (Sk - 1 + 7) & ~7;
    const int BQ = SR - HR;
    const int nqb = (int)((S + BQ - 1) / BQ);
    const size_t lds = sizeof(T) * ((size_t)BK * (D + PAD) + (size_t)D * (BK + PAD) + (size_t)SR * (HC + BK + PAD)) +
                       sizeof(float) * (size_t)R * Sk;
    auto kern = conv_attn_fwd_kernel<T, D, RT, SKT>;
    if (lds > 160 * 1024) return MTA_ERR_KERNEL_SIZE;
    if (lds > 48 * 1024) {  // per device, so set on every such launch (a cheap host-side call)
        hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    dim3 grid((unsigned)nqb, (unsigned)(B * H));
    hipLaunchKernelGGL(kern, grid, dim3(NT), lds, st, (const T *)q, (const T *)k, (const T *)v, w, (T *)o, lse, (int)S,
                       R, Sk, causal, scale, w_dtype, (int)H, nqb);
    return launch_status();
}

// the general kernel with the kernel size known at compile time; 1 when there is no instance
template <int D>
int dispatch_fp32(const void *q, const void *k, const void *v, const void *w, void *o, float *lse, int64_t B, int64_t H, int64_t S, int R, int Sk,
                  int causal, float scale, int w_dtype, hipStream_t st)
{
#define MTA_FP32_CASE(r, s) \
    if (R == r && Sk == s) return launch<float, D, r, s>(q, k, v, w, o, lse, B, H, S, R, Sk, causal, scale, w_dtype, st);
    MTA_FP32_CASE(3, 3)
    MTA_FP32_CASE(3, 5)
    MTA_FP32_CASE(5, 5)
    MTA_FP32_CASE(5, 7)
    MTA_FP32_CASE(6, 11)
    MTA_FP32_CASE(7, 7)
    MTA_FP32_CASE(7, 9)
    MTA_FP32_CASE(11, 15)
#undef MTA_FP32_CASE
    return 1;
}
}  // namespace

extern "C" int mta_conv_attn_fwd_lse(const void *q, const void *k, const void *v, const void *w, void *o, void *lse_out,
                                     int64_t B, int64_t H, int64_t S, int64_t D, int R, int Sk, int causal, float scale,
                                     int io_dtype, int w_dtype, void *stream)
{
    if (!q || !k || !v || !w || !o) return MTA_ERR_NULL;
    float *lse = (float *)lse_out;
    if (lse && !aligned_to(lse, 4)) return MTA_ERR_ALIGN;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(v, 16) || !aligned_to(o, 16) ||
        !aligned_to(w, dtype_size(w_dtype)))
        return MTA_ERR_ALIGN;
    hipStream_t st = (hipStream_t)stream;
    // MTA_FUSED_FORCE_GENERAL=1 in the environment keeps 16-bit inputs on the general kernel (for comparisons)
    static const bool force_general = [] { const char *e = getenv("MTA_FUSED_FORCE_GENERAL"); return e && e[0] == '1'; }();
    const bool fast_ok = io_dtype != MTA_F32 && w_dtype == io_dtype && !force_general;
    if (fast_ok) {
        const int rc = conv_attn_mfma_dispatch(io_dtype, {q, k, v, w, o, lse, B, H, S, D, R, Sk, causal, scale, 0, nullptr, 0, false, st});
        if (rc != 1) return rc;
    }
    MTA_DISPATCH_IO(io_dtype, {
        if constexpr (sizeof(io_t) == 4) {
            const int rc = D == 64 ? dispatch_fp32<64>(q, k, v, w, o, lse, B, H, S, R, Sk, causal, scale, w_dtype, st)
                                   : dispatch_fp32<128>(q, k, v, w, o, lse, B, H, S, R, Sk, causal, scale, w_dtype, st);
            if (rc != 1) return rc;
        }
        if (D == 64) return launch<io_t, 64>(q, k, v, w, o, lse, B, H, S, R, Sk, causal, scale, w_dtype, st);
        return launch<io_t, 128>(q, k, v, w, o, lse, B, H, S, R, Sk, causal, scale, w_dtype, st);
    });
    return MTA_ERR_DTYPE;
}

extern "C" int mta_conv_attn_fwd(const void *q, const void *k, const void *v, const void *w, void *o, int64_t B,
                                 int64_t H, int64_t S, int64_t D, int R, int Sk, int causal, float scale,
                                 int io_dtype, int w_dtype, void *stream)
{
    return mta_conv_attn_fwd_lse(q, k, v, w, o, nullptr, B, H, S, D, R, Sk, causal, scale, io_dtype, w_dtype, stream);
}

// kernel sizes that the 16-bit scores kernel has an instance for (the cases of dispatch_scores)
static bool scores_instance(int R, int Sk)
{
    return (R == 3 && (Sk == 3 || Sk == 5)) || (R == 5 && (Sk == 5 || Sk == 7)) || (R == 6 && Sk == 11) ||
           (R == 7 && (Sk == 7 || Sk == 9)) || (R == 11 && Sk == 15);
}

// Whether fp32 conv-attention runs as four kernels with the scores in memory.  In the fused kernel a workgroup of 128 rows walks the keys
// alone, conv and softmax on the vector units between two products: a chain of key blocks of 8 to 20 us, and no faster in all with two
// workgroups per CU.  The four kernels spread over the chip at any size, but move 16 bytes of scores per position and cost four launches
// (22 us), lengths that are no multiple of 8 two more copies.  The estimates below follow what was measured on 200 sizes; us, fused | four:
// 3x3 D64 B1 H4 S64 14.6 | 21.7, S192 30 | 22, S1024 129 | 39, H16 S2048 360 | 220; 6x11 D128 B1 H4 S65 43 | 31, S512 143 | 30, S2048 545 | 109;
// 7x9 D64 B4 H8 S65 28 | 31, S2048 713 | 474; 11x15 D64 B2 H12 S2048 1036 | 502; fused is left with small D = 64 grids and with many planes of
// small kernels: 5x5 D64 B4 H32 S192 34 | 46, S777 288 | 369, S1024 401 | 472.  The error against 64 bits is smaller in four kernels throughout.
extern "C" int mta_conv_attn_in_stages(int64_t B, int64_t H, int64_t S, int64_t D, int R, int Sk, int causal, int io_dtype)
{
    // (the kernel sizes that have instances of both)
    if (io_dtype != MTA_F32 || !causal || B <= 0 || H <= 0 || B * H > 65535 || S < 64 || S > (1 << 20) || (D != 64 && D != 128) || !scores_instance(R, Sk)) return 0;
    const double planes = (double)(B * H), s = (double)S, taps = (double)(R * Sk), positions = planes * s * s * 1e-6, blocks = (double)((S + 63) / 64);
    const double rows = (double)(128 - (R - 1 + 7) / 8 * 8), items = planes * std::ceil(s / rows);
    const double chain = std::max(blocks, items * (blocks + 1) / 2 * 1.25 / device_cu_count());   // key blocks one after the other on a CU
    const double fused = D == 64 ? 6 + (7 + 0.073 * taps) * chain : 10 + (13.5 + 0.047 * taps) * chain;
    const double four = std::max(22.0, 16 + 0.09 * planes + (D == 64 ? 3.3 : 3.9) * positions) + (S % 8 ? 9 + 6.4e-6 * planes * s * (double)D : 0);
    return four < 0.95 * fused ? 1 : 0;
}

extern "C" int mta_qk_conv_supported(int64_t S, int64_t D, int R, int Sk, int io_dtype, int w_dtype)
{
    return (io_dtype == MTA_BF16 || io_dtype == MTA_F16) && w_dtype == io_dtype && S > 0 && S % 8 == 0 && (D == 64 || D == 128) &&
                   scores_instance(R, Sk)
               ? 1
               : 0;
}

extern "C" int mta_qk_conv_fwd(const void *q, const void *k, const void *w, void *s_out, int64_t B, int64_t H, int64_t S,
                               int64_t D, int R, int Sk, int causal, float scale, int fill_upper, int io_dtype,
                               int w_dtype, void *stream)
{
    if (!q || !k || !w || !s_out) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(s_out, 16) || !aligned_to(w, dtype_size(w_dtype)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || w_dtype != io_dtype || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int rc = conv_attn_mfma_dispatch(io_dtype, {q, k, nullptr, w, s_out, nullptr, B, H, S, D, R, Sk, causal, scale, fill_upper, nullptr, 0, true, st});
    // (mta_qk_conv_supported must agree with the dispatch: a kernel size it names always has an instance)
    if (rc == 1 && scores_instance(R, Sk)) return MTA_ERR_KERNEL_SIZE;
    return rc == 1 ? MTA_ERR_UNSUPPORTED : rc;
}

// round(a b^T) on and below the diagonal (first_visible: only inside the band): the scores kernel without its conv
extern "C" int mta_lower_scores_fwd(const void *a, const void *b, const void *first_visible, void *out, int64_t B, int64_t H, int64_t S,
                                    int64_t D, int io_dtype, void *stream)
{
    if (!a || !b || !out) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(a, 16) || !aligned_to(b, 16) || !aligned_to(out, 16) || (first_visible && !aligned_to(first_visible, 4))) return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32) return first_visible ? MTA_ERR_UNSUPPORTED : mta_lower_scores_f32(a, b, out, B, H, S, D, stream);
    if (S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    return conv_attn_mfma_dispatch(io_dtype, {a, b, nullptr, nullptr, out, nullptr, B, H, S, D, 1, 1, 1, 1.0f, 0, (const int *)first_visible, 0, true,
                                              (hipStream_t)stream});
}

extern "C" int mta_lower_scores_rows_fwd(const void *a, int64_t a_batch, int64_t a_head, int64_t a_row, const void *b, const void *first_visible,
                                         void *out, int64_t B, int64_t H, int64_t S, int64_t D, int io_dtype, void *stream)
{
    if (!a || !b || !out) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535 || a_batch < 0 || a_head < 0 || a_row <= 0) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(a, 16) || !aligned_to(b, 16) || !aligned_to(out, 16) || (first_visible && !aligned_to(first_visible, 4)) || a_batch % 8 != 0 ||
        a_head % 8 != 0 || a_row % 8 != 0)
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    return conv_attn_mfma_dispatch(io_dtype, {a, b, nullptr, nullptr, out, nullptr, B, H, S, D, 1, 1, 1, 1.0f, 0, (const int *)first_visible, 0, true,
                                              (hipStream_t)stream, {a_batch, a_head, a_row}});
}

// mta_qk_conv_fwd (causal) / mta_qk_conv_band_fwd (first_visible not NULL) with the scores stored in the triangular
// layout (see tri_rowoff in common.hpp), groups of `group` heads interleaved by rows: B*H*tri_rowoff(S) elements, nothing
// above the diagonal.
extern "C" int mta_qk_conv_tri_fwd(const void *q, const void *k, const void *w, const void *first_visible, void *s_out,
                                   int64_t B, int64_t H, int64_t S, int64_t D, int R, int Sk, float scale, int group,
                                   int io_dtype, int w_dtype, void *stream)
{
    if (!q || !k || !w || !s_out) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (group <= 0 || H % group != 0) return MTA_ERR_GROUP;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(s_out, 16) || !aligned_to(w, dtype_size(w_dtype)) ||
        (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || w_dtype != io_dtype || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    if ((int64_t)group * tri_rowoff((int)S) > 0x7fffffffLL) return MTA_ERR_UNSUPPORTED;  // (32-bit offsets inside a group)
    hipStream_t st = (hipStream_t)stream;
    const int *lo = (const int *)first_visible;
    const int rc = conv_attn_mfma_dispatch(io_dtype, {q, k, nullptr, w, s_out, nullptr, B, H, S, D, R, Sk, 1, scale, 0, lo, group, true, st});
    if (rc == 1 && scores_instance(R, Sk)) return MTA_ERR_KERNEL_SIZE;
    return rc == 1 ? MTA_ERR_UNSUPPORTED : rc;
}

extern "C" int mta_qk_conv_stats_slots(int64_t B, int64_t H, int64_t S, int R)
{
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535 || R < 1 || R > MTA_MAX_FUSED_KERNEL_R) return 0;
    bool table;
    return scores_slots(S, R, scores_cut_of(B * H, S, R, true, table));
}

// mta_qk_conv_tri_fwd (group > 0) or mta_qk_conv_fwd / mta_qk_conv_band_fwd without a fill (group = 0), causal, that also leaves the maximum and the
// sum of exponentials of every row's scores item by item
extern "C" int mta_qk_conv_stats_fwd(const void *q, const void *k, const void *w, const void *key_bias, const void *first_visible, void *s_out, void *stats,
                                     int64_t B, int64_t H, int64_t S, int64_t D, int R, int Sk, float scale, int group, int io_dtype, int w_dtype, void *stream)
{
    if (!q || !k || !w || !s_out || !stats) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (group < 0 || (group > 0 && H % group != 0)) return MTA_ERR_GROUP;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(s_out, 16) || !aligned_to(w, dtype_size(w_dtype)) || !aligned_to(stats, 8) ||
        (key_bias && !aligned_to(key_bias, 4)) || (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || w_dtype != io_dtype || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    if (group > 0 && (int64_t)group * tri_rowoff((int)S) > 0x7fffffffLL) return MTA_ERR_UNSUPPORTED;  // (32-bit offsets inside a group)
    bool table;
    const scores_cut cut = scores_cut_of(B * H, S, R, true, table);
    conv_attn_args a = {q, k, nullptr, w, s_out, nullptr, B, H, S, D, R, Sk, 1, scale, 0, (const int *)first_visible, group, true, (hipStream_t)stream};
    a.stats = {(float2 *)stats, (const float *)key_bias, scores_slots(S, R, cut), cut};
    const int rc = conv_scores_stats_dispatch(io_dtype, a);
    if (rc == 1 && scores_instance(R, Sk)) return MTA_ERR_KERNEL_SIZE;
    return rc == 1 ? MTA_ERR_UNSUPPORTED : rc;
}

// The causal entry points above for q and k of `rows` rows, S - 7 <= rows <= S: group > 0 the triangular layout, 0 planes without a fill; stats or NULL
extern "C" int mta_qk_conv_ragged_fwd(const void *q, const void *k, const void *w, const void *first_visible, void *s_out, void *stats, int64_t B, int64_t H,
                                      int64_t S, int64_t rows, int64_t D, int R, int Sk, float scale, int group, int io_dtype, int w_dtype, void *stream)
{
    if (!q || !k || !w || !s_out) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535 || rows <= 0 || rows > S || rows < S - 7) return MTA_ERR_SHAPE;
    if (group < 0 || (group > 0 && H % group != 0)) return MTA_ERR_GROUP;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(s_out, 16) || !aligned_to(w, dtype_size(w_dtype)) || (stats && !aligned_to(stats, 8)) ||
        (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || w_dtype != io_dtype || S % 8 != 0 || !scores_instance(R, Sk)) return MTA_ERR_UNSUPPORTED;
    if (group > 0 && (int64_t)group * tri_rowoff((int)S) > 0x7fffffffLL) return MTA_ERR_UNSUPPORTED;  // (32-bit offsets inside a group)
    conv_attn_args a = {q, k, nullptr, w, s_out, nullptr, B, H, S, D, R, Sk, 1, scale, 0, (const int *)first_visible, group, true, (hipStream_t)stream};
    a.rows = rows;
    if (stats) {
        bool table;
        const scores_cut cut = scores_cut_of(B * H, S, R, true, table);
        a.stats = {(float2 *)stats, nullptr, scores_slots(S, R, cut), cut};
    }
    const int rc = stats ? conv_scores_stats_dispatch(io_dtype, a) : conv_attn_mfma_dispatch(io_dtype, a);
    return rc == 1 ? MTA_ERR_KERNEL_SIZE : rc;
}

// mta_qk_conv_fwd under a band mask: key k of query row p of batch entry b is visible iff first_visible[b, p] <= k <= p
// (int32, (B, S)); the scores of hidden keys enter the conv as 0.  Causal by construction.
extern "C" int mta_qk_conv_band_fwd(const void *q, const void *k, const void *w, const void *first_visible, void *s_out,
                                    int64_t B, int64_t H, int64_t S, int64_t D, int R, int Sk, float scale, int fill_upper,
                                    int io_dtype, int w_dtype, void *stream)
{
    if (!q || !k || !w || !s_out || !first_visible) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (R < 1 || Sk < 1 || R > MTA_MAX_FUSED_KERNEL_R || Sk > MTA_MAX_FUSED_KERNEL_S) return MTA_ERR_KERNEL_SIZE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(s_out, 16) || !aligned_to(w, dtype_size(w_dtype)) ||
        !aligned_to(first_visible, 4))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || w_dtype != io_dtype || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int *lo = (const int *)first_visible;
    const int rc = conv_attn_mfma_dispatch(io_dtype, {q, k, nullptr, w, s_out, nullptr, B, H, S, D, R, Sk, 1, scale, fill_upper, lo, 0, true, st});
    if (rc == 1 && scores_instance(R, Sk)) return MTA_ERR_KERNEL_SIZE;
    return rc == 1 ? MTA_ERR_UNSUPPORTED : rc;
}
