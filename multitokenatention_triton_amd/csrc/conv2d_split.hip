// Depthwise conv of large kernels, forward and input gradient, for what the kernels of conv2d_causal.hip on the matrix cores do not
// take (11x15: fp32 data; that and smaller ones: 16-bit data with weights of another dtype or rows that are not whole 16-byte
// vectors): on the bf16 matrix cores, with the 32 bits kept.
//
// Every fp32 value is the sum of three bf16 values (8 + 8 + 8 bits of its significand; each one the rounded remainder of those
// before it), exactly: x = x0 + x1 + x2, w = w0 + w1 + w2 (fp16: two parts, bf16: one).  Of the products of parts the six (bf16 data with
// fp32 weights: three) with i + j <= 2 are formed; each is exact in fp32, what is left out is below 2^-26 |x w|, a quarter of the last place that one fp32
// multiply-add rounds away.  A product takes the outputs of two rows and eight keys
// of sixteen pairs of rows; its 32 slots are four rows of the pair's window, eight columns each, and three such chunks hold the taps of eight keys:
// an operand from LDS serves the three groups of keys whose windows it is part of.  Once per pair of parts: w0 x0 adds into two accumulators
// (16-bit data: one), the small ones into another, and a result is their sum.  So an output takes 9 roundings of its own size or less (11x15) where
// multiply-adds took R*S: the error against 64 bits
// (2-norm) is 0.48e-7 forward and 0.73e-7 for the input gradient, where they left 1.3e-7 and 2.9e-7 (scores, 333^2 and 512^2; random taps
// 0.58e-7 and 0.59e-7; with one accumulator for w0 x0 1.0e-7 and 1.1e-7).
//
// Why: R*S multiply-adds on the vector units (0.079 PFLOP/s without packed fp32 forms) bound the row-sliding kernels from about 50
// taps on.  This form executes 6 * 64 * 9 flops for the 2 * 165 of an output of 11x15, at 2.5 PFLOP/s.
// One kernel row and sixteen keys per product (11 products and as many operands per 256 outputs, 9 and 4 now) -> this, fp32 11x15, whole
// rows: 16 planes of 512^2 19.9 -> 18.9, 16 of 1024^2 41.3 -> 37.9, 32 of 1024^2 66.6 -> 60.5, 16 of 2048^2 142 either way.
// 16-bit data gains by that only if it is also stored well: two groups at a time, four keys a lane, stores are 16 rows x 32 bytes and two wavefronts
// complete a line; without stores this form was the faster one everywhere, with them the slower one up to 333^2.  So all four groups leave together,
// eight keys a lane: 16 rows x 64 bytes in half the instructions and fewer registers.  One row and sixteen keys, two workgroups per CU | two rows,
// 32 bytes, three and four workgroups | 64 bytes, at most three (split_occ), lower triangle (input gradient), us: bf16 6x11 16 of 333^2 6.0 | 6.9 | 6.3
// (6.9 | 7.8 | 7.0), 12 of 801^2 12.4 | 14.4 | 12.1 (15.9 | 18.4 | 15.1), 16 of 1023^2 17.9 | 17.2 | 16.0 (23.4 | 21.6 | 20.6), 32 of 1023^2 28.0 | 30.6 |
// 25.9 (36.4 | 38.8 | 32.9), 16 of 2047^2 51.0 | 47.3 | 42.8 (65.8 | 55.7 | 52.3); with fp32 weights 7x7 12 of 801^2 14.5 | 15.2 | 13.6 (17.4 | 18.2 |
// 16.3), 16 of 1023^2 20.3 | 19.0 | 17.7 (25.5 | 23.3 | 22.2); fp16 7x9 16 of 333^2 7.6 | 7.9 | 7.3, 16 of 1023^2 23.4 | 21.6 | 20.0 (28.7 | 24.5 |
// 23.9), with fp32 weights 6x11 16 of 2047^2 74.6 | 74.0 | 67.2 (84.1 | 83.9 | 81.3).  Left behind the first by 0.2 to 0.5 us: 5x7 and 6x11 of planes up to
// 333^2, of a strip or two per CU.
// us, conv2d_rows -> the former, fp32: lower triangle 16 planes of 512^2 23 -> 18.5, 12 of 801^2 32 -> 28.5, 16 of 1024^2 58 -> 38, 32 of
// 1024^2 105 -> 68, 16 of 2048^2 177 -> 128; whole rows 31 -> 20, 34 -> 31, 86 -> 43, 152 -> 80, 260 -> 151.  Smaller kernels stay
// there, lower triangle | whole rows: 7x9 16 of 1024^2 29.7 | 39.4 against 29.4 | 34.5 here, 16 of 512^2 13.9 | 16.4 against 15.3 |
// 16.5, 16 of 2048^2 92 | 128 against 98 | 140; 6x11 and 5x7 alike or slower.
// 16-bit data with fp32 weights, lower triangle of 16 planes of 1024^2, bf16 | fp16: 5x7 22.2 -> 18.6 | 22.2 -> 22.7, 7x7 26.0 -> 20.6 | (kept) 26.4,
// 6x11 29.4 -> 19.5 | 29.6 -> 24.6, 7x9 28.9 -> 20.8 | 29.4 -> 25.8; bf16 16 of 512^2 6x11 13.0 -> 10.8, 32 of 2048^2 6x11 152 -> 115, 7x7 121 -> 117 (5x7
// 109 -> 114: kept); weights of the data's type, whole rows of 16 planes of 1001^2: bf16 7x7 34.6 -> 23.3, 6x11 40.4 -> 22.9, fp16 6x11 40.8 -> 28.1.
// What bounds it (16 of 1024^2, 40 us): without products 24, without loads and splitting 35, without stores 39; 16 of 2048^2, 145 us: 137, 96, 111 -
// the CU's path to the L2 (1.5 times the strip in, the strip out), and at 1024^2 five rounds of strips with the products' 17 us in them.
// Values that have three parts are split 2^24 times as large, results taken back: every fp32 value below 2^104 then has parts that are normal
// numbers (the smallest denormal's only bit is 2^-125), however small it is and whatever lies beside it, and the products of parts of
// small values stay above the denormals as well.  Results that are not finite then - an operand was not, or is larger, or a sum of
// scaled products is beyond 2^128, one of 2^80 and more - take multiply-adds after all, one by one.  (An infinite part makes every result
// non-finite whose window of slots holds it, also under a zero of the Toeplitz fragment: what is finite is exact.)
// (A look at every strip's largest value, with strips of tiny values staged once more, cost 2 to 4 % in fp32 and 4 to 8 % in 16 bits and could
// not see small values beside ordinary ones: lower triangle of 16 planes, fp32 512^2 19.2 -> 18.5 us, 2048^2 130.9 -> 127.9, bf16 with fp32
// weights 1024^2 6x11 20.6 -> 19.5, fp16 7x9 26.4 -> 25.1.)
//
// Shape.  A workgroup of four wavefronts takes strips of 32 rows x 128 keys of one plane, one after the other, two or three workgroups per
// CU (split_occ).  A strip and its halo are loaded four keys per lane, two strips ahead, into registers; split and written to one of two LDS
// buffers (a plane of bf16 per part) a vector at a time between the products of the strip before.  The fragments of the plane's kernel stay in
// registers (11x15: 3 parts * 3 quads * 3 chunks * 4 of them); they come out of a table of all windows of every kernel row.
#include <algorithm>

#include "conv2d_rows.hpp"
#include "split.hpp"

namespace {
using namespace mta;

constexpr int P_TM = 32, P_TN = 128;       // strip
constexpr int P_HL = 8;                    // keys staged left (and right) of it
constexpr int P_LD = P_TN + 2 * P_HL;      // keys of a staged row
constexpr int P_RS = P_LD + 8;             // its length in LDS, an odd number of 16-byte chunks: operand reads free of bank conflicts (two rows between lanes)
constexpr int P_QUADS = P_LD / 4;

typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

// strips that touch the lower triangle (all of them unless `tri`), column of strips by column of strips
__host__ __device__ __forceinline__ int p_first(int tn, int tri) { return tri ? tn * P_TN / P_TM : 0; }
inline int64_t p_count(int64_t H, int64_t W, int tri)
{
    const int tiles_m = (int)((H + P_TM - 1) / P_TM), tiles_n = (int)((W + P_TN - 1) / P_TN);
    int64_t n = 0;
    for (int tn = 0; tn < tiles_n; ++tn) n += tiles_m > p_first(tn, tri) ? tiles_m - p_first(tn, tri) : 0;
    return n;
}

template <typename T> constexpr int parts_of() { return __is_same(T, float) ? 3 : __is_same(T, f16_t) ? 2 : 1; }

// Workgroups per CU: a strip is a chain of loads, splitting, products and stores between two barriers, and what hides it is the other
// workgroups; as many as registers and LDS hold (fp16 data with three parts of a tap: with some values in scratch memory), at most
// three.  bf16 data and taps leave room for four, whose strips come in fewer and emptier rounds.  us, 6x11, two | three | four, lower triangle
// (whole planes): 12 of 801^2 12.3 | 11.8 | 13.4 (16.2 | 15.2 | 17.1), 32 of 511^2 12.6 | 11.0 | 13.2 (15.7 | 14.5 | 14.2), 4 of 2047^2 16.2 | 15.5 | 18.4
// (25.8 | 23.4 | 22.3), 16 of 2047^2 39.6 | 40.0 | 38.6 (74.8 | 66.9 | 71.9); the other way only 8 of 801^2 9.1 | 8.8 | 8.1 (11.9 | 12.1 | 10.9).
template <typename T, int WP, int R> constexpr int split_occ() { return parts_of<T>() * WP == 1 || (parts_of<T>() * WP <= 6 && R <= 7) ? 3 : 2; }

template <typename T, int WP, int R, int S, bool BWD>
__global__ __launch_bounds__(256, (split_occ<T, WP, R>())) void conv2d_split(const T *__restrict__ x, const void *__restrict__ w, T *__restrict__ y, int C, int H,
                                                       int W, int causal, float in_scale, int use_scale, int w_dtype, int planes, int total, int per_plane)
{
    constexpr int PAD = BWD ? S - 1 - (S - 1) / 2 : (S - 1) / 2, SHIFT = P_HL - PAD;   // first tap's column in a window of 24
    static_assert(SHIFT >= 0 && SHIFT + 8 + S - 1 <= 24, "the taps of 8 outputs in three chunks of 8 columns");
    constexpr int NQ = (R + 4) / 4;                    // quads of rows in the window of a pair of rows
    constexpr bool OVER = 4 * NQ > R + 1;              // ... whose last one reaches beyond it
    constexpr int ROWS = P_TM + R - 1, RPI = 256 / P_QUADS, IT = (ROWS + RPI - 1) / RPI;   // a round of loads: RPI rows, four threads idle
    constexpr int PLANE = ROWS * P_RS;                 // bf16 values of one part
    constexpr int NE = S + 7;                          // windows of a kernel row that hold a tap: first slot - SHIFT - ln = -7 .. S-1
    constexpr int XP = parts_of<T>();                  // parts of a value (WP: of a tap)
    __shared__ __align__(16) uint16_t xs[2][XP * PLANE];
    static_assert(WP * R * (NE + 1) * 8 + WP * R * (S + 16) <= 2 * XP * PLANE, "the table of windows borrows the strips' LDS");
    constexpr float UP_X = XP == 3 ? SPLIT_UP : 1.0f, UP_W = WP == 3 ? SPLIT_UP : 1.0f, DOWN = 1.0f / (UP_X * UP_W);   // (see above)
    const float by = use_scale ? in_scale * UP_X : UP_X;   // fp32 data: factor and scale in one

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // (planes dealt to the XCDs where they divide evenly: a plane's strips share their halo rows in one L2)
    int plane, first;
    if (planes % 8 == 0) {
        const int pos = (int)(blockIdx.x >> 3);
        plane = (int)(blockIdx.x & 7) * (planes / 8) + pos / per_plane;
        first = pos % per_plane;
    } else {
        plane = (int)blockIdx.x / per_plane;
        first = (int)blockIdx.x % per_plane;
    }
    const int c = plane % C;
    const T *xp = x + plane * (int64_t)H * W;
    T *yp = y + plane * (int64_t)H * W;
    const bool tri = causal != 0;

    struct strip { int p0, q0; };
    // strips in the order that this workgroup takes them: `per_plane` further on each time (a column holds many of those steps: found
    // afresh from its number, a strip cost a loop over the columns)
    const int tiles_m = (H + P_TM - 1) / P_TM;
    int col = 0, at = first;
    auto next_strip = [&]() {
        for (int n; at >= (n = tiles_m > p_first(col, tri) ? tiles_m - p_first(col, tri) : 0); ++col) at -= n;
        const strip t{(p_first(col, tri) + at) * P_TM, col * P_TN};
        at += per_plane;
        return t;
    };
    auto top_row = [](strip t) { return BWD ? t.p0 : t.p0 - (R - 1); };
    // no value of the strip or its halo lies outside the plane or above the diagonal
    auto inside = [&](strip t) {
        const int h0 = top_row(t);
        return h0 >= 0 && h0 + ROWS <= H && t.q0 >= P_HL && t.q0 + P_TN + P_HL <= W && (!causal || t.q0 + P_TN + P_HL - 1 <= h0);
    };
    quad4<T> raw[IT];
    const int lr = tid / P_QUADS, lk = tid % P_QUADS * 4;      // this lane's row in a round of loads, and its keys
    // (rows and keys outside the plane re-read the nearest inside)
    auto fetch = [&](strip t, int it) __attribute__((always_inline)) {
        const int h0 = top_row(t), base = h0 < 0 ? 0 : h0, k = t.q0 - P_HL + lk, h = h0 + lr + it * RPI;
        const char *from = reinterpret_cast<const char *>(xp + (int64_t)base * W);
        const int hc = h < base ? base : (h >= H ? H - 1 : h), kc = k < 0 ? 0 : (k > W - 4 ? W - 4 : k);
        __builtin_memcpy(&raw[it], from + (unsigned)((hc - base) * W + kc) * (unsigned)sizeof(T), sizeof(raw[it]));
    };
    // vector `it` of a strip: masked, scaled, split, to LDS
    auto stage = [&](strip t, bool plain, int it, uint16_t *to) __attribute__((always_inline)) {
        const int r = lr + it * RPI;
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = to_float(raw[it].v[u]);
        if (!plain) {
            asm volatile("" : : : "memory");   // (kept a branch)
            const int k = t.q0 - P_HL + lk, h = top_row(t) + r;
            masked_quad<T>(raw[it], k, W, (h < 0 || h >= H) ? -1 : (causal && h < W - 1 ? h : W - 1), v);
        }
        if constexpr (XP == 3) {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] *= by;
        } else if (use_scale) {
            asm volatile("" : : : "memory");
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = round_to<T>(v[u] * in_scale);
        }
        uint32_t a[XP], b[XP];
        split2<XP>(v[0], v[1], a);
        split2<XP>(v[2], v[3], b);
        if (lr < RPI && ((it + 1) * RPI <= ROWS || r < ROWS)) {
#pragma unroll
            for (int s = 0; s < XP; ++s) *reinterpret_cast<uint2 *>(to + s * PLANE + r * P_RS + lk) = make_uint2(a[s], b[s]);
        }
    };
    strip t{0, 0}, next{0, 0};
    if (first < total) {
        t = next_strip();
#pragma unroll
        for (int it = 0; it < IT; ++it) fetch(t, it);     // in flight while the kernel is prepared
    }

    // ---- the kernel's fragments, quad q, chunk c: lane (ln, kg) is output row ln/8 of a pair and key ln%8 of a group, slot t the window's row
    // 4q + kg and column 8c + t: tap (4q + kg - ln/8, 8c + t - SHIFT - ln%8) ----
    frag8<bf16_t> tz[WP][NQ * 3];
    {
        constexpr int NT = (R * (S + 16) + 255) / 256;
        uint16_t *const table = xs[0], *const taps = table + WP * R * (NE + 1) * 8;   // [part][row][8 zeros, S taps, 8 zeros]
        float v[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int e = n * 256 + tid, i = e / (S + 16), j = e % (S + 16) - 8;
            v[n] = i < R && j >= 0 && j < S ? load_any(w, w_dtype, (int64_t)c * R * S + (BWD ? R * S - 1 - (i * S + j) : i * S + j)) : 0.0f;
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int e = n * 256 + tid;
            uint32_t part[WP];
            split2<WP>(v[n] * UP_W, 0.0f, part);
            if (e < R * (S + 16)) {
#pragma unroll
                for (int s = 0; s < WP; ++s) taps[s * R * (S + 16) + e] = (uint16_t)part[s];
            }
        }
        __syncthreads();
        for (int e = tid; e < WP * R * (NE + 1); e += 256) {
            const int row = e / (NE + 1), k = e % (NE + 1);   // window k: taps k-7 .. k; the last one: none
            u16x8 win;
#pragma unroll
            for (int u = 0; u < 8; ++u) win[u] = k < NE ? taps[row * (S + 16) + 1 + k + u] : (uint16_t)0;
            *reinterpret_cast<u16x8 *>(table + e * 8) = win;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < WP; ++s)
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int i = 4 * q + kg - (ln >> 3), from = 8 * c - SHIFT - (ln & 7) + 7;
                    const bool some = i >= 0 && i < R && from >= 0 && from < NE;
                    tz[s][q * 3 + c] = *reinterpret_cast<const frag8<bf16_t> *>(table + ((s * R + (some ? i : 0)) * (NE + 1) + (some ? from : NE)) * 8);
                }
        __syncthreads();
    }
    if (first < total) {
        const bool plain = inside(t);
#pragma unroll
        for (int it = 0; it < IT; ++it) stage(t, plain, it, xs[0]);
        if (first + per_plane < total) {
            next = next_strip();
#pragma unroll
            for (int it = 0; it < IT; ++it) fetch(next, it);
        }
    }
    __syncthreads();

    for (int id = first, n = 0; id < total; id += per_plane, n ^= 1) {
        const bool more = id + per_plane < total, more2 = id + 2 * per_plane < total;
        const strip after = more2 ? next_strip() : t;   // (asked for either way: behind a branch around the loads their waits would be waits for all)
        const bool plain = inside(next);
        // ---- 32 rows x 32 keys per wavefront: four groups of 8 keys of 16 pairs of rows.  Chunk by chunk and quad by quad, each an operand of the
        // three groups whose windows hold the chunk, read while the one before is multiplied (the order is pinned).  In between the next
        // strip's vectors go to the other buffer, one by one, and those of the strip behind it are asked for ----
        constexpr int NG = 4, NX = NG + 2, NSTEP = NX * NQ;
        const uint16_t *const xw = xs[n] + (2 * ln + kg) * P_RS + wave * 32;
        const int over = OVER ? (2 * ln + 4 * (NQ - 1) + kg < ROWS ? 0 : ROWS - 1 - (2 * ln + 4 * (NQ - 1) + kg)) * P_RS : 0;   // (rows that were not staged: one that was)
        frag8<bf16_t> f[2][XP];
        auto read = [&](int m) __attribute__((always_inline)) {
            const int q = m % NQ;
#pragma unroll
            for (int s = 0; s < XP; ++s)
                f[m & 1][s] = *reinterpret_cast<const frag8<bf16_t> *>(xw + s * PLANE + 4 * q * P_RS + m / NQ * 8 + (OVER && q == NQ - 1 ? over : 0));
        };
        const int lower = causal ? (t.p0 + P_TM - 1 - t.q0 - wave * 32) >> 3 : NG - 1;   // last group that touches the triangle
        // (address of a lane's results: a uniform base and a byte offset within the strip)
        constexpr int LK = sizeof(T) == 2 ? 8 : 4;   // keys of a row that a lane stores at a time
        const int pl = 2 * ln, ql = wave * 32 + kg * LK;
        char *const ybase = reinterpret_cast<char *>(yp + (int64_t)t.p0 * W + t.q0);
        const unsigned yoff = (unsigned)(pl * W + ql) * (unsigned)sizeof(T);
        const bool whole = t.p0 + P_TM <= H && t.q0 + P_TN <= W && (!causal || t.q0 + P_TN - 1 <= t.p0);
        float bad = 0.0f;   // not 0: a result that is not finite
        uint32_t out[sizeof(T) == 2 ? NG : 1][2];   // 16-bit data: the groups' results, packed
        // sums of the large products, fp32 data: of the middle chunk, which holds the taps next to the output's own position, and of the other two,
        // so that a sum is rounded fewer times and that of a kernel near the identity once or twice; and of the small ones
        constexpr bool TWO = XP == 3;
        f32x4 big[NG], small[NG], rim_[TWO ? NG : 1], *const rim = TWO ? rim_ : big;
        read(0);
#pragma unroll
        for (int x = 0; x < NX; ++x) {
            if (x < NG) big[x] = small[x] = rim[x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int m = x * NQ + q;
                if (x - 2 <= lower) {
                    if (m + 1 < NSTEP) read(m + 1);
                    // part ws of the taps times part s of the values, for the groups that take this chunk
                    auto products = [&](f32x4 *acc, int ws, int s) __attribute__((always_inline)) {
#pragma unroll
                        for (int c = 2; c >= 0; --c)
                            if (x - c >= 0 && x - c < NG) mma16(acc[x - c], tz[ws][q * 3 + c], f[m & 1][s]);
                    };
                    if constexpr (XP > 2) products(small, 0, 2);
                    if constexpr (WP > 2) products(small, 2, 0);
                    if constexpr (XP > 1 && WP > 1) products(small, 1, 1);
#pragma unroll
                    for (int c = 2; c >= 0; --c)
                        if (x - c >= 0 && x - c < NG) mma16(c == 1 ? big[x - c] : rim[x - c], tz[0][q * 3 + c], f[m & 1][0]);
                    if constexpr (WP > 1) products(small, 1, 0);
                    if constexpr (XP > 1) products(small, 0, 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                constexpr int LEAD = NSTEP / 4;  // (not ahead of the last strip's stores: loads and stores complete on one counter)
#pragma unroll
                for (int it = 0; it < IT; ++it)
                    if (m == LEAD + it * (NSTEP - LEAD) / IT) {
                        if (more) stage(next, plain, it, xs[n ^ 1]);
                        fetch(after, it);
                        __builtin_amdgcn_sched_barrier(0);
                    }
            }
            if (x == 3 || x == 5) {   // two groups are complete
                const int w = x - 3;
                float v[2][4];
#pragma unroll
                for (int g = 0; g < 2; ++g)
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        v[g][u] = (big[w + g][u] + (TWO ? rim[w + g][u] + small[w + g][u] : small[w + g][u])) * DOWN;
                        bad = fmaf(v[g][u], 0.0f, bad);
                    }
                if constexpr (sizeof(T) == 2) {
                    // all four groups leave together: a lane gets the eight keys of group kg in each row of its pair, stores of 16 rows x 64 bytes
#pragma unroll
                    for (int g = 0; g < 2; ++g)
#pragma unroll
                        for (int n = 0; n < 2; ++n) out[w + g][n] = pack2<T>(v[g][2 * n], v[g][2 * n + 1]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) swap16(out[w][n], out[w + 1][n]);   // (afterwards: [w] keys 0-3, [w + 1] keys 4-7 of group w + kg%2)
                    if (w == 0) continue;
#pragma unroll
                    for (int n = 0; n < 4; ++n) swap32(out[n >> 1][n & 1], out[2 + (n >> 1)][n & 1]);   // ([0], [1] the pair's first row, [2], [3] the second)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        mta_u32x4 o = {out[2 * h][0], out[2 * h][1], out[2 * h + 1][0], out[2 * h + 1][1]};
                        if (whole) {
                            asm volatile("" : "+v"(o));   // (one store, not one shared in part with the other branch)
                            __builtin_memcpy(ybase + (yoff + (unsigned)(h * W) * (unsigned)sizeof(T)), &o, sizeof(o));
                        } else {
                            const int p = t.p0 + pl + h, q = t.q0 + ql;
#pragma unroll
                            for (int n = 0; n < 4; ++n) {
                                if (causal && q + 2 * n > p) o[n] &= 0xffff0000u;
                                if (causal && q + 2 * n + 1 > p) o[n] &= 0x0000ffffu;
                            }
                            // (asked for by quads; mostly both)
                            const bool one = p < H && q < W && !(causal == 2 && q > p), two = p < H && q + 4 < W && !(causal == 2 && q + 4 > p);
                            if (two && q + 8 <= W) {
                                __builtin_memcpy(yp + (int64_t)p * W + q, &o, sizeof(o));
                            } else {
#pragma unroll
                                for (int g = 0; g < 2; ++g) {
                                    unpack2<T>(o[2 * g], v[g][0], v[g][1]);
                                    unpack2<T>(o[2 * g + 1], v[g][2], v[g][3]);
                                    if (g ? two : one) store_quad<T>(yp + (int64_t)p * W, q + 4 * g, W, v[g]);
                                }
                            }
                        }
                    }
                } else {   // a lane gets four keys of each row of its pair, stores of 16 rows x 64 bytes
#pragma unroll
                    for (int u = 0; u < 4; ++u) swap32(v[0][u], v[1][u]);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (whole) {
                            asm volatile("" : "+v"(v[h][0]), "+v"(v[h][1]), "+v"(v[h][2]), "+v"(v[h][3]));
                            __builtin_memcpy(ybase + (yoff + (unsigned)(h * W + w * 8) * (unsigned)sizeof(T)), v[h], sizeof(v[h]));
                        } else {
                            const int p = t.p0 + pl + h, q = t.q0 + ql + w * 8;
                            if (p < H && q < W && !(causal == 2 && q > p)) {
#pragma unroll
                                for (int u = 0; u < 4; ++u) v[h][u] = causal && q + u > p ? 0.0f : v[h][u];
                                store_quad<T>(yp + (int64_t)p * W, q, W, v[h]);
                            }
                        }
                    }
                }
            }
        }
        if (__builtin_amdgcn_ballot_w64(bad != 0.0f) != 0) {   // this lane's results that are not finite: multiply-adds, tap by tap
#pragma unroll 1
            for (int e = opaque(0); e < 16; ++e) {
                const int pe = t.p0 + pl + (LK == 8 ? e >> 3 : e >> 2 & 1), q = t.q0 + ql + (LK == 8 ? e & 7 : (e >> 3) * 16 + (e & 3));
                if (pe >= H || q >= W || (causal && q > pe)) continue;
                T *const at = yp + (int64_t)pe * W + q;
                if (__builtin_isfinite(to_float(*at))) continue;
                float sum = 0.0f;
                for (int i = 0; i < R; ++i) {
                    const int h = BWD ? pe + i : pe - (R - 1) + i;
                    if (h < 0 || h >= H) continue;
                    for (int j = 0; j < S; ++j) {
                        const int k = q - PAD + j;
                        if (k < 0 || k >= W || (causal && k > h)) continue;
                        float v = to_float(xp[(int64_t)h * W + k]);
                        if (use_scale) v = round_to<T>(v * in_scale);
                        sum = fmaf(load_any(w, w_dtype, (int64_t)c * R * S + (BWD ? R * S - 1 - (i * S + j) : i * S + j)), v, sum);
                    }
                }
                *at = from_float<T>(sum);
            }
        }
        t = next;
        next = after;
        __syncthreads();
    }
    if (causal == 1) {     // the strips wholly above the diagonal
        const int tiles = tiles_m * ((W + P_TN - 1) / P_TN);
        for (int id = first; id < tiles; id += per_plane) {
            const int p0 = id % tiles_m * P_TM, q0 = id / tiles_m * P_TN;
            if (q0 <= p0 + P_TM - 1) continue;
            for (int e = tid; e < P_TM * (P_TN / 4); e += 256) {
                const int p = p0 + e / (P_TN / 4), q = q0 + e % (P_TN / 4) * 4;
                T *dst = yp + (int64_t)p * W + q;
                const T zero = from_float<T>(0.0f);
                const quad4<T> z = {{zero, zero, zero, zero}};
                if (p >= H || q >= W) continue;
                if (q + 4 <= W) {
                    __builtin_memcpy(dst, &z, sizeof(z));
                } else {
                    asm volatile("" : : : "memory");
                    for (int u = 0; u < W - q; ++u) dst[u] = zero;
                }
            }
        }
    }
}

template <typename T, int WP, int R, int S, bool BWD>
int launch_split(const void *x, const void *w, void *y, int64_t planes, int64_t C, int64_t H, int64_t W, int causal, float in_scale, int use_scale,
                 int w_dtype, hipStream_t st)
{
    const int64_t total = p_count(H, W, causal != 0);
    if (total > 0x3fffffffLL) return MTA_ERR_SHAPE;
    // One round of resident workgroups, rounded down: those beyond it would start when the others end.  fp32 11x15, lower triangle, us, rounded up ->
    // down: 12 planes of 801^2 26.0 -> 23.7, 24 of 1023^2 62.0 -> 49.0, 12 of 1501^2 68.8 -> 55.9.
    int64_t per_plane = std::max<int64_t>(split_occ<T, WP, R>() * device_cu_count() / planes, 1);
    if (per_plane > total) per_plane = total;
    hipLaunchKernelGGL((conv2d_split<T, WP, R, S, BWD>), dim3((unsigned)(planes * per_plane)), dim3(256), 0, st, (const T *)x, w, (T *)y, (int)C, (int)H,
                       (int)W, causal, in_scale, use_scale, w_dtype, (int)planes, (int)total, (int)per_plane);
    return launch_status();
}

// weights of the data's own type have its parts, others three
template <typename T>
int dispatch_split(const void *x, const void *w, void *y, int64_t planes, int64_t C, int64_t H, int64_t W, int R, int S, bool bwd, int causal,
                   float in_scale, int use_scale, bool same, int w_dtype, hipStream_t st)
{
#define MTA_SPLIT(wp, r, s)                                                                                                     \
    (bwd ? launch_split<T, wp, r, s, true>(x, w, y, planes, C, H, W, causal, in_scale, use_scale, w_dtype, st)                  \
         : launch_split<T, wp, r, s, false>(x, w, y, planes, C, H, W, causal, in_scale, use_scale, w_dtype, st))
#define MTA_CONV_CASE(r, s)                                                                                                     \
    if (R == r && S == s) {                                                                                                     \
        if constexpr (sizeof(T) == 2) {                                                                                         \
            if (same) return MTA_SPLIT(parts_of<T>(), r, s);                                                                    \
        }                                                                                                                       \
        return MTA_SPLIT(3, r, s);                                                                                              \
    }
    MTA_CONV_CASE(11, 15)
    // 16-bit data: fewer parts, so that smaller kernels gain as well.  bf16: from 49 taps on, 5x7 up to 32 M elements; fp16, with twice the parts:
    // from 60 taps on (7x7: S1024 26.4 | 25.4, but B2 H12 S640 19.1 | 21.7, B2 H16 S2048 123 | 143)
    if constexpr (sizeof(T) == 2) {
        MTA_CONV_CASE(6, 11)
        MTA_CONV_CASE(7, 9)
        if constexpr (parts_of<T>() == 1) {
            MTA_CONV_CASE(7, 7)
            if (planes * H * W <= 32 << 20) {
                MTA_CONV_CASE(5, 7)
            }
        }
    }
#undef MTA_CONV_CASE
#undef MTA_SPLIT
    return 1;
}
}  // namespace

int mta::conv2d_split_dispatch(const void *x, const void *w, void *y, int64_t N, int64_t C, int64_t H, int64_t W, int R, int S, bool bwd, int causal,
                               float in_scale, int use_scale, int io_dtype, int w_dtype, hipStream_t st)
{
    if (W < 4) return 1;
    MTA_DISPATCH_IO(io_dtype, return dispatch_split<io_t>(x, w, y, N * C, C, H, W, R, S, bwd, causal, in_scale, use_scale, w_dtype == io_dtype, w_dtype, st));
    return 1;
}
