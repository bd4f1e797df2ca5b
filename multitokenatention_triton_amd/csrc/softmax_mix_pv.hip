// O = (W2 softmax(x)) V in one pass over the scores:  x is the score tensor behind the conv (16 bits, planes or the triangular layout), the row
// statistics come from the kernel that wrote it (conv_scores_mfma.hpp), the probabilities exist in registers only.
//
// A wavefront owns 16 query rows of a mixing group of G heads and the results of GO of them (GO * D / 16 accumulators).  A step is 32 keys: a
// lane (row ln, eight keys kg) loads the G heads' scores of its keys, turns them into probabilities - a multiply-add, an exponential
// and a multiplication each -, rounds them, mixes the G heads key by key on 4x4x4 matrix products, whose contraction
// lies within a lane, and rounds the result: what the softmax stage would have stored is then in the lane that supplies it as operand of O^T
// += V^T P^T.  V comes in blocks of 32 keys of GO heads, copied global -> LDS asynchronously a step ahead, read by transpose reads.  The
// probabilities of the next step are formed between the products of this one.
// What it saves is writing and reading the probabilities, half of what the three kernels of this route move: bf16 6x11 B2 H16 S4096 D128 groups of 4,
// softmax + mixing 183 us, P V 148 -> 196 (with a key bias 197; the scores kernel pays 7 to 21 for the statistics); B4 H16 S1024 30 + 22 -> 39; D64 B2 H16 S4096
// 177 + 134 -> 161.  What bounds it: at B2 H16 S4096 D128, where it took 189 with the sum in the exponent, 108 us without loads, 97 for the scores alone as tiles of 16
// rows, 69 for V and the products - they overlap in part only, a barrier a step holding eight wavefronts to the slowest load.  Not better there (us, against
// those 189): scores non-temporal 218, blocks of V asked for three steps ahead and one wavefront per SIMD 232, 128 rows 254, results of two of the four heads per
// workgroup 237 to 273 (twice the exponentials; where the grid is short they win, form_of), packed dot products in place of the 4x4x4 ones (as fast, more vector
// instructions).
#include <type_traits>

#include <stdlib.h>

#include "mfma.hpp"
#include "scores_cut.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

constexpr int BK = 32;               // keys per step
constexpr int MOST_KEYS = 1 << 15;   // under a key bias

// 16 independent 4 x 4 x 4 products: a lane's four values of b (one position's) times the matrix whose row l % 4 lane l holds in a
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ f32x4 mix4(u32x2 a, u32x2 b)
{
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (std::is_same<T, bf16_t>::value)
        return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(s16x4_t, a), __builtin_bit_cast(s16x4_t, b), zero, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(f16x4_t, a), __builtin_bit_cast(f16x4_t, b), zero, 0, 0, 0);
}

struct pv_args {
    const void *x, *w2, *v;
    const float2 *stats;     // [batch * head][slot][row]: scores_stats
    const float *key_bias;   // (B,S) or NULL
    const int *band_lo;      // (B,S) or NULL
    void *o;
    int S, SV, H, groups, nrb, cus, tri, slots;   // SV: rows that v has, at most S
    scores_items items;
    float per_gph;           // reciprocal of H / G
};

template <typename T, int D, int G, int GO, int RW, int GR, int OCC, bool KB>
__global__ __launch_bounds__(64 * RW * GR, OCC) void softmax_mix_pv(const pv_args a)
{
    constexpr int CPR = D / 8, HEAD = BK * D, TILE = GO * HEAD, GT = 64 * RW, ROUNDS = TILE / 8 / GT, RPH = HEAD / 8 / GT, DB = D / 16, ROWS = 16 * RW;
    static_assert(RPH >= 1, "whole copy rounds");
    __shared__ __align__(16) T lds[GR * 2 * TILE];
    __shared__ uint32_t hidden[KB ? MOST_KEYS / BK : 1];   // a bit per key that the bias hides
    const int S = a.S, tid = threadIdx.x % GT, grp = GR == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    int bg, rank;
    if (!longest_first(a.groups * (G / GO), a.nrb, a.cus, bg, rank)) return;
    const int h0 = bg % (G / GO) * GO;   // the first of the group's heads whose results are formed here
    bg /= G / GO;
    const int q0 = (a.nrb - 1 - rank) * ROWS, w0 = q0 + wave * 16, prow = w0 + ln, pc = prow < S ? prow : S - 1;
    const int b = quotient(bg, a.per_gph), g = bg - b * (a.H / G);   // batch entry, group of its
    T *const mine = lds + grp * 2 * TILE;

    // the group's scores: a row of head i lies i * between elements behind the first head's (the same distance for the 16 rows of a wavefront)
    const T *const xg = static_cast<const T *>(a.x) + (a.tri ? (int64_t)bg * (G * tri_rowoff(S)) + G * tri_rowoff(w0 < S ? w0 : S - 1) : ((int64_t)bg * G * S + (w0 < S ? w0 : S - 1)) * S);
    const int64_t between = a.tri ? tri_rowlen(w0 < S ? w0 : S - 1) : (int64_t)S * S;
    const unsigned row_at = (unsigned)(pc - (w0 < S ? w0 : S - 1)) * (unsigned)(a.tri ? G * (int)between : S) + kg * 8;
    const T *const Vg = static_cast<const T *>(a.v) + (int64_t)(bg * G + h0) * a.SV * D;

    // The mixing weights, row lane % 4: of four heads; of two heads twice on the diagonal, for two keys at a time
    u32x2 wm = {0u, 0u};
    {
        const T *const w2 = static_cast<const T *>(a.w2) + (int64_t)(g * G + h0 + lane % GO) * a.H + g * G;
        if constexpr (G == 4) wm = u32x2{*reinterpret_cast<const uint32_t *>(w2), *reinterpret_cast<const uint32_t *>(w2 + 2)};
        else wm = lane & 2 ? u32x2{0u, *reinterpret_cast<const uint32_t *>(w2)} : u32x2{*reinterpret_cast<const uint32_t *>(w2), 0u};
    }

    const int q_last = (q0 + ROWS - 1 < S - 1) ? q0 + ROWS - 1 : S - 1;
    int j_end = q_last / BK, j0 = 0;
    int lo = 0, lo_max = 0;
    if (a.band_lo) {   // the steps ahead of the first key any of these rows sees are not visited (their scores may be undefined)
        int f = S;
        for (int r = lane; r < ROWS; r += 64)
            if (q0 + r < S) f = min(f, a.band_lo[(int64_t)b * S + q0 + r]);
        lo = first_key(a.band_lo, (int64_t)b * S + pc, pc);
        int m = lo;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            f = min(f, __shfl_xor(f, off));
            m = max(m, __shfl_xor(m, off));
        }
        f = __builtin_amdgcn_readfirstlane(f);
        lo_max = __builtin_amdgcn_readfirstlane(m);
        j0 = min((f > 0 ? f : 0) / BK, j_end);
    }
    const int jg = j0 + ((grp - j0) & (GR - 1)), n = jg <= j_end ? (j_end - jg) / GR + 1 : 0, nall = (j_end - j0) / GR + 1;

    const int row0 = tid / CPR;
    int voff[RPH];
#pragma unroll
    for (int r = 0; r < RPH; ++r) {
        const int row = row0 + r * (GT / CPR);
        voff[r] = (row * D + ((tid % CPR) ^ v_swizzle<D>(row)) * 8) * (int)sizeof(T);
    }
    auto issue_v = [&](int j, int buf) __attribute__((always_inline)) {
        T *const dst = mine + buf * TILE;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
            copy_to_lds(Vg + (int64_t)(r / RPH) * a.SV * D, a.SV * D * (int)sizeof(T), dst + (r * GT + wave * 64) * 8, voff[r % RPH] + j * HEAD * (int)sizeof(T));
    };
    auto load_x = [&](int j, u32x4 (&x)[G]) __attribute__((always_inline)) {   // beyond the row: its start
        const unsigned at = (j * BK + kg * 8 <= pc ? (unsigned)(j * BK) : 0u - kg * 8) + row_at;
#pragma unroll
        for (int i = 0; i < G; ++i) x[i] = *reinterpret_cast<const u32x4 *>(xg + i * between + at);
    };
    // Every step asks for the same number of things, behind the last one again for its own: the waits count them.
    u32x4 x[2][G];   // scores of two steps
    auto block = [&](int i) { return min(jg + i * GR, j_end); };
    load_x(block(0), x[0]);
    in_order();
    issue_v(block(0), 0);
    in_order();
    load_x(block(1), x[1]);
    in_order();

    // The rows' factors: p = exp2(x log2(e) - m) / sum, head kg (kg % G) of row ln here, all heads of it in every lane below.  The sum does not go into
    // the exponent: m is log2(e) times a score, rounded, and what the rounding takes away is in the sum as well and cancels; m + log2(sum) would be rounded once
    // more, by 2^-24 of the score's size, which then stays (4 % of a probability at scores of 1e6).  The multiplication that this takes: forward of bf16 6x11
    // groups of 4, D128, B2 H16 S4096 433 -> 435 us, B4 H16 S1024 padded 94.8 -> 96.0.
    constexpr float LOG2E = 1.4426950408889634f;
    float ref[G], inv[G];
    {
        const int items = a.items.of_row(pc, S);
        const float2 *const at = a.stats + ((int64_t)(bg * G + kg % G) * a.slots) * S + pc;
        float m = NO_SCORE, l = 0.0f;
        constexpr int AT_ONCE = 8;
        for (int i = 0; i < items; i += AT_ONCE) {
            float2 s[AT_ONCE];
#pragma unroll
            for (int k = 0; k < AT_ONCE; ++k) s[k] = at[(int64_t)min(i + k, items - 1) * S];
            float most = m;
#pragma unroll
            for (int k = 0; k < AT_ONCE; ++k) most = fmaxf(most, s[k].x);
            l *= __builtin_amdgcn_exp2f(m - most);
#pragma unroll
            for (int k = 0; k < AT_ONCE; ++k) l += i + k < items ? s[k].y * __builtin_amdgcn_exp2f(s[k].x - most) : 0.0f;
            m = most;
        }
        // (a row that sees no key: NaN, as the softmax of -inf alone gives)
        const float per_l = l == 0.0f ? __builtin_nanf("") : 1.0f / l;
#pragma unroll
        for (int i = 0; i < G; ++i) ref[i] = __shfl(m, (i << 4) + ln), inv[i] = __shfl(per_l, (i << 4) + ln);
    }
    if constexpr (KB) {   // a bit per key that the bias hides
        const float *const kb = a.key_bias + (int64_t)b * S;
        for (int w = (int)(threadIdx.x >> 6); w < (j_end + 2) / 2; w += RW * GR) {
            const uint64_t h = __builtin_amdgcn_ballot_w64(kb[min(w * 64 + lane, S - 1)] == -INFINITY);
            if (lane == 0) reinterpret_cast<uint2 *>(hidden)[w] = make_uint2((uint32_t)h, (uint32_t)(h >> 32));
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
    f32x4 oacc[GO][DB];
#pragma unroll
    for (int i = 0; i < GO; ++i)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[i][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int vrow = kg * 8 + (ln >> 2), vat = vrow * D + ((((ln & 3) >> 1) ^ v_swizzle<D>(vrow)) * 8) + (ln & 1) * 4;
    unsigned va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = lds_at(mine + (vat ^ (db * 16)));
    constexpr uint32_t NINF = std::is_same<T, bf16_t>::value ? 0xff80ff80u : 0xfc00fc00u;
    auto hide = [&](u32x4 (&xs)[G], const uint32_t (&keep)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < G; ++i)
#pragma unroll
            for (int d = 0; d < 4; ++d) xs[i][d] = (xs[i][d] & keep[d]) | (NINF & ~keep[d]);
    };
    // what a mask hides among the scores of step j becomes -inf
    auto masks = [&](int j, u32x4 (&xs)[G]) __attribute__((always_inline)) {
        if (j * BK + BK - 1 > w0 || j * BK < lo_max) {   // keys beyond the row, or ahead of its first one
            asm volatile("" ::: "memory");
            const int key = j * BK + kg * 8;
            uint32_t keep[4];
#pragma unroll
            for (int d = 0; d < 4; ++d)
                keep[d] = (key + 2 * d <= pc && key + 2 * d >= lo ? 0xffffu : 0u) | (key + 2 * d + 1 <= pc && key + 2 * d + 1 >= lo ? 0xffff0000u : 0u);
            hide(xs, keep);
        }
        if constexpr (KB) {
            const uint32_t all = __builtin_amdgcn_readfirstlane(hidden[j]);
            if (all != 0) {
                asm volatile("" ::: "memory");
                const uint32_t bits = all >> (kg * 8);
                uint32_t keep[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) keep[d] = (bits >> (2 * d) & 1u ? 0u : 0xffffu) | (bits >> (2 * d + 1) & 1u ? 0u : 0xffff0000u);
                hide(xs, keep);
            }
        }
    };
    // Scores -> mixed probabilities as operands, in 32 pieces of a few instructions, four for a key: the probabilities of half the heads, of the
    // others, rounded and packed; mixed; rounded and packed key by key.
    float e[4];
    u32x2 pk;
    f32x4 mx[2];
    auto piece = [&](auto kc, const u32x4 (&xs)[G], u32x4 (&p)[G]) __attribute__((always_inline)) {
        constexpr int t = decltype(kc)::value / 4, s = decltype(kc)::value % 4, d = t / 2, u = t % 2;   // (two heads: keys t and t + 1 at an even t)
        auto prob = [&](int h, int hi) {
            float x0, x1;
            unpack2<T>(xs[h][d], x0, x1);
            return __builtin_amdgcn_exp2f(fmaf(hi ? x1 : x0, LOG2E, -ref[h]));
        };
        if constexpr (G == 4) {
            if constexpr (s < 2) e[2 * s] = prob(2 * s, u), e[2 * s + 1] = prob(2 * s + 1, u);
            else if constexpr (s == 2) pk = u32x2{pack2<T>(e[0] * inv[0], e[1] * inv[1]), pack2<T>(e[2] * inv[2], e[3] * inv[3])};
            else mx[u] = mix4<T>(wm, pk);
            if constexpr (s == 3 && u == 1) {
#pragma unroll
                for (int o = 0; o < GO; ++o) p[o][d] = pack2<T>(mx[0][o], mx[1][o]);
            }
        } else if constexpr (u == 0) {
            if constexpr (s < 2) e[2 * s] = prob(0, s), e[2 * s + 1] = prob(1, s);
            else if constexpr (s == 2) pk = u32x2{pack2<T>(e[0] * inv[0], e[1] * inv[1]), pack2<T>(e[2] * inv[0], e[3] * inv[1])};
            else mx[0] = mix4<T>(wm, pk);
        } else if constexpr (s == 3) {
#pragma unroll
            for (int o = 0; o < GO; ++o) p[o][d] = pack2<T>(mx[0][o], mx[0][2 + o]);
        }
    };
    // The products of a step and, between them, the probabilities of the next one: matrix cores, LDS and vector units side by side.
    auto product = [&](auto bufc, const u32x4 (&p)[G], const u32x4 (&xs)[G], u32x4 (&pn)[G]) __attribute__((always_inline)) {
        constexpr int buf = decltype(bufc)::value, N = GO * DB, AHEAD = (GO * D > 256 && OCC == 2) || OCC == 3 ? 2 : 4;
        u32x2 fa[AHEAD + 1], fb[AHEAD + 1];
        auto read = [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, off = (buf * TILE + i / DB * HEAD) * (int)sizeof(T);
            fa[i % (AHEAD + 1)] = lds_load_tr8_at(va[i % DB], off);
            fb[i % (AHEAD + 1)] = lds_load_tr8_at(va[i % DB], off + 4 * D * (int)sizeof(T));
        };
        static_for<AHEAD>(read);
        static_for<N>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            if constexpr (i + AHEAD < N) read(std::integral_constant<int, i + AHEAD>{});
            constexpr int younger = 2 * ((i + AHEAD < N ? i + AHEAD : N - 1) - i);
            lds_wait_upto<younger>(fa[i % (AHEAD + 1)], fb[i % (AHEAD + 1)]);
            struct { u32x2 a, b; } both = {fa[i % (AHEAD + 1)], fb[i % (AHEAD + 1)]};
            mma16(oacc[i / DB][i % DB], __builtin_bit_cast(frag8<T>, both), __builtin_bit_cast(frag8<T>, p[i / DB]));
            static_for<32 / N>([&](auto kc) __attribute__((always_inline)) { piece(std::integral_constant<int, i * (32 / N) + decltype(kc)::value>{}, xs, pn); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Step i: key block jg + i GR; its probabilities are formed, its block of V was asked for a step ago, the scores of the next one one and a
    // half.  Behind the barrier nobody reads the other buffer any more; registers whose scores have become probabilities get those of the
    // step after the next two.
    u32x4 p[2][G];
    auto live = [&](int i) { return i < n && (jg + i * GR) * BK <= w0 + 15; };
    auto step = [&](auto nowc, auto full, int i) __attribute__((always_inline)) {
        constexpr int now = decltype(nowc)::value;
        constexpr bool FULL = decltype(full)::value;   // three more steps follow, and no row of this wavefront ends before the next one
        copies_wait<G>();                              // V of this step has come (behind it only G loads of scores)
        wg_barrier();
        const int j = jg + i * GR;
        issue_v(FULL ? j + GR : block(i + 1), now ^ 1);
        in_order();
        if (FULL || live(i)) {   // (behind the last step of a row: probabilities of scores that nobody wants)
            if (FULL || live(i + 1)) masks(j + GR, x[now ^ 1]);
            product(nowc, p[now], x[now ^ 1], p[now ^ 1]);
        }
        load_x(FULL ? j + 3 * GR : block(i + 3), x[now ^ 1]);
        in_order();
    };
    if (live(0)) {
        masks(jg, x[0]);
        static_for<32>([&](auto kc) __attribute__((always_inline)) { piece(kc, x[0], p[0]); });
    }
    in_order();
    load_x(block(2), x[0]);
    in_order();
    const std::integral_constant<int, 0> b0{};
    const std::integral_constant<int, 1> b1{};
    const int full = n - 4 - (ROWS / BK + GR) / GR;   // (the first wavefront's rows end ROWS / BK key blocks before the last one's)
    int i = 0;
    for (; i + 2 <= full; i += 2) {
        step(b0, std::true_type{}, i);
        step(b1, std::true_type{}, i + 1);
    }
    for (; i < nall; i += 2) {
        step(b0, std::false_type{}, i);
        if (i + 1 < nall) step(b1, std::false_type{}, i + 1);
    }
    copies_wait<0>();   // (nothing may come into LDS that is no longer this workgroup's)
    if constexpr (GR > 1) {   // the groups' sums, the upper half's to the lower half by way of the buffers until one is left
        static_assert(GR * 2 * TILE * sizeof(T) >= (size_t)GR / 2 * GT * GO * DB * 16, "half the groups' sums fit the buffers");
        __syncthreads();
        f32x4 *const part = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
        for (int h = GR / 2; h > 0; h /= 2) {
            if (grp >= h && grp < 2 * h) {
#pragma unroll
                for (int k = 0; k < GO * DB; ++k) part[((grp - h) * GO * DB + k) * GT + tid] = oacc[k / DB][k % DB];
            }
            __syncthreads();
            if (grp < h) {
#pragma unroll
                for (int k = 0; k < GO * DB; ++k) oacc[k / DB][k % DB] += part[(grp * GO * DB + k) * GT + tid];
            }
            if (h > 1) __syncthreads();
        }
        if (grp > 0) return;
    }
    if (prow >= S) return;
#pragma unroll
    for (int h = 0; h < GO; ++h)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            struct alignas(8) quad { T v[4]; } out;
#pragma unroll
            for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[h][db][v]);
            *reinterpret_cast<quad *>(static_cast<T *>(a.o) + ((int64_t)(bg * G + h0 + h) * S + prow) * D + db * 16 + kg * 4) = out;
        }
}

// ---- which form --------------------------------------------------------------------------------------------------------
// Of how many heads a workgroup forms the results, of how many rows, and how many groups of wavefronts share the keys: WHOLE all, 64, two; HALF_LONG half of them,
// 64, one (groups of 4 at D64: all, 32, two); HALF_SHORT half, 32, two; HALF_SPLIT half, 16, four.  With half of the heads the exponentials
// are formed twice, but there are twice the workgroups and a step is shorter; more groups of wavefronts shorten the chain of steps.  The
// line runs by n, the 64-row blocks over the groups of heads.  us of the forward, bf16 or fp16, several kernel sizes, the four in this order:
//   groups of 4, D128  n 24 (B4 H12 S72) 21.2 | 16.3 | 15.8, 36 (B2 H12 S352) 32.3 | 27.8 | 24.6, 96 (B2 H32 S360) 38.7 | 34.2 | 32.2, 168 (B2 H16 S1296) 84.5 |
//     82.1 | 69.7, 200 (B4 H8 S1600) 104 | 99.6 | 95.5, 240 (B2 H16 S1864) 121 | 116 | 119, 320 (B2 H16 S2552) 198 | 195 | 208, 408 (B2 H16 S3256) 275 | 312 | 322,
//     504 (B2 H16 S3976) 408 | 454 | 487.  HALF_SPLIT has one workgroup per CU there: from 257 on (n 36, B4 H12 S184 18.4 against 24.6) a second round, and
//     where it wins (few long rows, n 28, B1 H16 S440 26.1 against 25.4) three kernels are faster than two.
//   groups of 4, D64   n 8 (B1 H16 S72) 17.4 | 14.9 | 14.1 | 14.0, 32 (B4 H16 S128) 19.3 | 16.4 | 15.1 | 14.8, 64 (B1 H32 S464) 31.6 | 27.1 | 24.7 | 23.7, 104 (B1 H32 S800)
//     51.3 | 45.7 | 42.3 | 46.2, 168 (B2 H16 S1296) 67.7 | 59.8 | 56.5 | 67.1, 208 (B2 H16 S1608) 93.0 | 83.4 | 85.0 | 99.4, 256 (B1 H16 S4048) 224 | 194 | 215 | 239, 400 (B4 H16
//     S1560) 116 | 120 | 130 | 163
//   groups of 2, D128  n 26 (B1 H4 S816) 28.6 | 27.6 | 22.3 | 20.5, 64 (B1 H4 S2032) 56.8 | 56.9 | 43.8 | 41.4, 88 (B1 H16 S664) 29.9 | 28.8 | 24.6 | 28.6, 188 (B1 H8 S2952)
//     85.6 | 88.9 | 78.6 | 91.4, 256 (B1 H16 S2032) 73.1 | 74.5 | 74.9 | 91.7, 416 (B4 H4 S3328) 148 | 166 | 167 | 203;  D64  24 (B1 H8 S336) 17.3 | 17.6 | 15.2 | 14.0, 72 (B1
//     H16 S560) 23.7 | 24.4 | 21.5 | 20.8, 80 (B2 H16 S264) 18.9 | 18.9 | 16.8 | 17.6, 144 (B2 H16 S544) 27.2 | 27.8 | 25.5 | 27.9, 228 (B1 H12 S2432) 67.6 | 76.8 | 70.9 | 74.5, 456 (B2 H8 S3600) 139 | 159 | 157 | 173
//     Few heads with long rows: HALF_SPLIT beyond n 64 too, HALF_SHORT | HALF_SPLIT, B1 H4: D128 S2112 (66) 42.0 | 38.9, S2752 (86) 53.4 | 53.1, S3000 (94) 55.8 | 58.5;
//     D64 S2112 39.7 | 35.0 (right-padded 46.2 | 40.9, three kernels 42.2), S3712 (116) 63.1 | 61.8, S4096 (128) 68.3 | 69.4, B1 H12 S768 (72) 24.2 | 22.5
enum pv_form { WHOLE = 1, HALF_LONG, HALF_SHORT, HALF_SPLIT };

pv_form form_of(int64_t groups, int64_t S, int D, int G)
{
    static const int force = [] { const char *e = getenv("MTA_SOFTMAX_PV_FORM"); return e ? atoi(e) : 0; }();   // (comparison switch: always that form)
    if (force >= WHOLE && force <= HALF_SPLIT) return (pv_form)force;
    const int64_t n = groups * ((S + 63) / 64);
    if (G == 2) return n >= 200 ? WHOLE : n <= 64 || (D == 64 ? n <= 116 && S >= 512 : n <= 86 && S > 24 * n) ? HALF_SPLIT : HALF_SHORT;
    if (n >= 400) return WHOLE;
    if (D == 64) return n >= 190 ? HALF_LONG : n > 64 ? HALF_SHORT : HALF_SPLIT;
    return n >= 240 ? HALF_LONG : HALF_SHORT;
}

template <typename T, int D, int G, int GO, int RW, int GR, int OCC> int go(pv_args a, int64_t groups, int resident, hipStream_t st)
{
    const int64_t blocks = (a.S + 16 * RW - 1) / (16 * RW), wg = (groups * (G / GO) * blocks + 7) / 8 * 8;
    if (wg > 0x7fffffffLL) return MTA_ERR_SHAPE;
    a.groups = (int)groups, a.nrb = (int)blocks;
    a.cus = wg <= (int64_t)resident * device_cu_count() ? device_cu_count() / 8 : 0;
    if (a.key_bias) hipLaunchKernelGGL((softmax_mix_pv<T, D, G, GO, RW, GR, OCC, true>), dim3((unsigned)wg), dim3(64 * RW * GR), 0, st, a);
    else hipLaunchKernelGGL((softmax_mix_pv<T, D, G, GO, RW, GR, OCC, false>), dim3((unsigned)wg), dim3(64 * RW * GR), 0, st, a);
    return launch_status();
}

template <typename T, int D, int G> int launch(const pv_args &a, int64_t groups, hipStream_t st)
{
    switch (form_of(groups, a.S, D, G)) {
    case WHOLE: return go<T, D, G, G, 4, 2, 2>(a, groups, 1, st);
    case HALF_LONG:
        if constexpr (G == 4 && D == 64) return go<T, D, G, G, 2, 2, 2>(a, groups, 2, st);
        else return go<T, D, G, G / 2, 4, 1, 3>(a, groups, 3, st);
    case HALF_SPLIT:
        if constexpr (G == 2 || D == 64) return go<T, D, G, G / 2, 1, 4, D == 64 ? 2 : 1>(a, groups, D == 64 ? 2 : 1, st);
        [[fallthrough]];
    default: return go<T, D, G, G / 2, 2, 2, D == 64 ? 3 : 2>(a, groups, D == 64 ? 3 : 2, st);
    }
}
template <typename T> int launch_type(const pv_args &a, int64_t groups, int64_t D, int group, hipStream_t st)
{
    if (D == 64) return group == 2 ? launch<T, 64, 2>(a, groups, st) : launch<T, 64, 4>(a, groups, st);
    return group == 2 ? launch<T, 128, 2>(a, groups, st) : launch<T, 128, 4>(a, groups, st);
}
}  // namespace

extern "C" int mta_softmax_mix_pv_supported(int64_t H, int64_t S, int64_t D, int group, int io_dtype, int w_dtype, int key_bias)
{
    return (io_dtype == MTA_BF16 || io_dtype == MTA_F16) && w_dtype == io_dtype && (group == 2 || group == 4) && H > 0 && H % group == 0 && S > 0 && S % 8 == 0 &&
           S <= (key_bias ? MOST_KEYS : 1 << 19) && (D == 64 || D == 128);
}

// v of v_rows rows, S - 7 <= v_rows <= S (o has S; what those beyond v_rows hold is not defined)
extern "C" int mta_softmax_mix_pv_ragged_fwd(const void *x, const void *stats, const void *w2, const void *key_bias, const void *first_visible, const void *v, void *o,
                                      int64_t B, int64_t H, int64_t S, int64_t v_rows, int64_t D, int R, int group, int tri, int io_dtype, int w_dtype, void *stream)
{
    if (!x || !stats || !w2 || !v || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535 || v_rows <= 0 || v_rows > S || v_rows < S - 7) return MTA_ERR_SHAPE;
    if (R < 1 || R > MTA_MAX_FUSED_KERNEL_R) return MTA_ERR_KERNEL_SIZE;
    if (group <= 0 || H % group != 0) return MTA_ERR_GROUP;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(x, 16) || !aligned_to(v, 16) || !aligned_to(o, 16) || !aligned_to(stats, 8) || !aligned_to(w2, 4) || (key_bias && !aligned_to(key_bias, 4)) ||
        (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (!mta_softmax_mix_pv_supported(H, S, D, group, io_dtype, w_dtype, key_bias != nullptr)) return MTA_ERR_UNSUPPORTED;
    bool table;
    const scores_cut cut = scores_cut_of(B * H, S, R, true, table);
    const pv_args a{x, w2, v, (const float2 *)stats, (const float *)key_bias, (const int *)first_visible, o, (int)S, (int)v_rows, (int)H, 0, 0, 0, tri != 0,
                    scores_slots(S, R, cut), scores_items(cut, scores_rows(R)), (float)group / (float)H};
    const int64_t groups = B * (H / group);
    return io_dtype == MTA_BF16 ? launch_type<bf16_t>(a, groups, D, group, (hipStream_t)stream) : launch_type<f16_t>(a, groups, D, group, (hipStream_t)stream);
}

extern "C" int mta_softmax_mix_pv_fwd(const void *x, const void *stats, const void *w2, const void *key_bias, const void *first_visible, const void *v, void *o,
                                      int64_t B, int64_t H, int64_t S, int64_t D, int R, int group, int tri, int io_dtype, int w_dtype, void *stream)
{
    return mta_softmax_mix_pv_ragged_fwd(x, stats, w2, key_bias, first_visible, v, o, B, H, S, S, D, R, group, tri, io_dtype, w_dtype, stream);
}
