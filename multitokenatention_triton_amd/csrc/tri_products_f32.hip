// The three lower-triangle products around an fp32 (B,H,S,S) score tensor of the causal pipeline:
//
//   scores   C[p,q]  = sum_d A[p,d] B[q,d]              q <= p     (Q K^T; dP = dO V^T)
//   pv       O[p,d]  = scale * sum_{q<=p} P[p,q] V[q,d]             (P V; dQ)
//   ptx      O[q,d]  = scale * sum_{p>=q} P[p,q] X[p,d]             (dV, dK)
//
// on v_mfma_f32_16x16x4f32 (fp32 products, fp32 sums), nothing above the diagonal read or - beyond the 16-byte vector that
// straddles it, as zeros - written.  The library's batched GEMMs they replace work on the full square, and at one batch of 16
// heads on a few dozen 256x256 tiles.
//
// Small grids use no LDS in the loops: which element feeds which operand slot is free as long as both operands agree, and each product has an
// assignment in which every operand is 16 (P of ptx: 8) contiguous bytes per lane -
//   scores: contraction d = 16s + 4g + t for slot group g at step t: a lane's vector of its row is four steps' operand;
//   pv:     contraction q = 16j + 4g + t (P's vector), output column d = 64b + 4r + u for operand row r of product u (V's
//           vector of key q is four products' operand);
//   ptx:    contraction p = 4j + g, output row q = 2r + w of product w (P's pair), column d as above (X's vector)
// (lane = 16g + r).  A line fetched by one lane's load is used up by its neighbours in the same instruction.
// us against the library GEMM (scores / pv / ptx): B1 H4 S256 D64 3.9 / 4.4 / 5.5 against 24 / 21 / 22, where launching is all
// there is; B1 H16 S512 10 / 8 / 9 against 21 / 20 / 21; B1 H32 S1024 38 / 38 / 31 against 55 / 36 / 35 (the library's operand
// has to be filled above the diagonal first, which is another 15 us).
#include "common.hpp"
#include "mfma.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

__device__ __forceinline__ void mma4(f32x4 &c, float a, float b) { c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// ---- scores: a wavefront owns 16 W query rows x 32 W keys, a workgroup 32 W x 64 W ----------------------------------------
template <int W> constexpr int sc_rows() { return 32 * W; }

// tiles on or below the diagonal of the first n rows of tiles, two tile rows per tile column
__host__ __device__ __forceinline__ int sc_tiles(int n) { return (n / 2) * (n / 2 + 1) + (n & 1) * (n / 2 + 1); }

template <int D, int W>
__global__ __launch_bounds__(256) void lower_scores_f32(const float *__restrict__ A, const float *__restrict__ Bm, float *__restrict__ C,
                                                        int S, int heads, int tiles, int cus)
{
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    // tile row: the largest n with sc_tiles(n) <= tile
    int tr = (int)(2.0f * sqrtf((float)tile));
    while (sc_tiles(tr) > tile) --tr;
    while (sc_tiles(tr + 1) <= tile) ++tr;
    const int tc = tile - sc_tiles(tr);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int p0 = tr * sc_rows<W>() + (wave & 1) * 16 * W, q0 = tc * 2 * sc_rows<W>() + (wave >> 1) * 32 * W;
    if (p0 >= S || q0 >= S || q0 > p0 + 16 * W - 1) return;   // (outside, or wholly above the diagonal)
    const float *Ap = A + (int64_t)bh * S * D + g * 4, *Bp = Bm + (int64_t)bh * S * D + g * 4;
    int arow[W], brow[2 * W];
#pragma unroll
    for (int i = 0; i < W; ++i) arow[i] = (p0 + 16 * i + r < S ? p0 + 16 * i + r : S - 1) * D;
#pragma unroll
    for (int i = 0; i < 2 * W; ++i) brow[i] = (q0 + 16 * i + r < S ? q0 + 16 * i + r : S - 1) * D;
    f32x4 acc[2 * W][W];
#pragma unroll
    for (int i = 0; i < 2 * W; ++i)
#pragma unroll
        for (int k = 0; k < W; ++k) acc[i][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 a[2][W], b[2][2 * W];
    auto fetch = [&](int s, int set) {
#pragma unroll
        for (int i = 0; i < W; ++i) a[set][i] = *reinterpret_cast<const f32x4 *>(Ap + arow[i] + 16 * s);
#pragma unroll
        for (int i = 0; i < 2 * W; ++i) b[set][i] = *reinterpret_cast<const f32x4 *>(Bp + brow[i] + 16 * s);
    };
    fetch(0, 0);
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
        if (s + 1 < D / 16) fetch(s + 1, (s + 1) & 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 2 * W; ++i)
#pragma unroll
                for (int k = 0; k < W; ++k) mma4(acc[i][k], b[s & 1][i][t], a[s & 1][k][t]);
    }
    // acc[i][k][v]: key q0 + 16i + 4g + v of query row p0 + 16k + r
    float *Cp = C + (int64_t)bh * S * S;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const int p = p0 + 16 * k + r;
        if (p >= S) continue;
#pragma unroll
        for (int i = 0; i < 2 * W; ++i) {
            const int q = q0 + 16 * i + 4 * g;
            if (q > p) continue;
            f32x4 o = acc[i][k];
#pragma unroll
            for (int v = 1; v < 4; ++v)
                if (q + v > p) o[v] = 0.0f;
            *reinterpret_cast<f32x4 *>(Cp + (int64_t)p * S + q) = o;
        }
    }
}

// ---- scores of large grids: a workgroup owns 128 query rows x 128 keys, its wavefronts 64 x 64 each ------------------------
// The kernel above pulls 6 KB through the L1 for every 32 products.  Here slabs of 16 head dims of both operands are copied
// global -> LDS asynchronously, one slab ahead, and serve all four wavefronts: a third of the bytes per product.  What bounds it
// now is the fp32 matrix rate (64 more head dims cost 25 us at B1 H32 S1024, 91 TFLOP/s) with the write of the scores behind it.  A slab row is four 16-byte
// chunks, XOR-swizzled by bits 2 and 3 of the row: the lanes that the LDS serves together (0-7 with 24-31, ...) then cover its
// banks once.
constexpr int SL_TILE = 128, SL_D = 16;
template <int D>
__global__ __launch_bounds__(256, 3) void lower_scores_f32_slabs(const float *__restrict__ A, const float *__restrict__ Bm, float *__restrict__ C,
                                                                 int S, int heads, int tiles, int cus)
{
    __shared__ __align__(16) float a_buf[2][SL_TILE * SL_D];
    __shared__ __align__(16) float b_buf[2][SL_TILE * SL_D];
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    int tr = (int)(sqrtf(2.0f * (float)tile + 0.25f) - 0.5f);   // tile row: tr (tr + 1) / 2 tiles lie ahead of it
    while (tr * (tr + 1) / 2 > tile) --tr;
    while ((tr + 1) * (tr + 2) / 2 <= tile) ++tr;
    const int tc = tile - tr * (tr + 1) / 2;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
    const float *Ap = A + (int64_t)bh * S * D, *Bp = Bm + (int64_t)bh * S * D;
    // slab s: 128 rows of four chunks, two slots per thread and operand (rows past the sequence re-read the last one)
    auto issue = [&](int s, int set) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int slot = i * 256 + tid, row = slot >> 2, c = (slot & 3) ^ ((row >> 2) & 3);
            const int ra = tr * SL_TILE + row < S ? tr * SL_TILE + row : S - 1, rb = tc * SL_TILE + row < S ? tc * SL_TILE + row : S - 1;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Ap + (int64_t)ra * D + SL_D * s + 4 * c), (lds_void_t *)(a_buf[set] + (i * 256 + wave * 64) * 4), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Bp + (int64_t)rb * D + SL_D * s + 4 * c), (lds_void_t *)(b_buf[set] + (i * 256 + wave * 64) * 4), 16, 0, 0);
        }
    };
    const int wp = (wave & 1) * 64, wq = (wave >> 1) * 64, p0 = tr * SL_TILE + wp, q0 = tc * SL_TILE + wq;
    const bool live = p0 < S && q0 < S && q0 <= p0 + 63;   // (else outside, or wholly above the diagonal)
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[i][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    issue(0, 0);
#pragma unroll
    for (int s = 0; s < D / SL_D; ++s) {
        __builtin_amdgcn_s_waitcnt(0);   // slab s has arrived
        __syncthreads();                 // for every wavefront; reads of the other buffers are finished
        if (s + 1 < D / SL_D) issue(s + 1, (s + 1) & 1);
        if (!live) continue;
        f32x4 a[4], b[4];
        const int at = (g ^ ((r >> 2) & 3)) * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] = *reinterpret_cast<const f32x4 *>(a_buf[s & 1] + (wp + 16 * i + r) * SL_D + at);
            b[i] = *reinterpret_cast<const f32x4 *>(b_buf[s & 1] + (wq + 16 * i + r) * SL_D + at);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k) mma4(acc[i][k], b[i][t], a[k][t]);
    }
    if (!live) return;
    // acc[i][k][v]: key q0 + 16i + 4g + v of query row p0 + 16k + r
    float *Cp = C + (int64_t)bh * S * S;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int p = p0 + 16 * k + r;
        if (p >= S) continue;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = q0 + 16 * i + 4 * g;
            if (q > p) continue;
            f32x4 o = acc[i][k];
#pragma unroll
            for (int v = 1; v < 4; ++v)
                if (q + v > p) o[v] = 0.0f;
            *reinterpret_cast<f32x4 *>(Cp + (int64_t)p * S + q) = o;
        }
    }
}

// the sums of a workgroup's four wavefronts, N vectors per lane each, added in wavefront order: wavefront w takes vectors
// w, w+4, ... ; `part`: 4 * CH * 64 vectors of LDS, CH vectors at a time
template <int N, int CH, typename GET, typename STORE>
__device__ __forceinline__ void reduce_waves(f32x4 *part, int wave, int lane, GET &&get, STORE &&store)
{
    static_assert(N % CH == 0 && CH % 4 == 0, "whole chunks, a quarter per wavefront");
#pragma unroll
    for (int c = 0; c < N; c += CH) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < CH; ++i) part[(wave * CH + i) * 64 + lane] = get(c + i);
        __syncthreads();
#pragma unroll
        for (int i = 0; i < CH / 4; ++i) {
            const int e = i * 4 + wave, at = e * 64 + lane;
            const f32x4 sum = ((part[at] + part[CH * 64 + at]) + part[2 * CH * 64 + at]) + part[3 * CH * 64 + at];
            store(c, i, sum);
        }
    }
}

// ---- pv: a workgroup owns 16 query rows, its wavefronts every fourth step of 16 keys ---------------------------------------
// (Short grids: a wavefront's chain of steps is what they wait for, and with 32 rows a step takes twice as long.  us, 32 rows | 16: B1
// H4 S256 D64 5.5 | 4.4, S1024 12.2 | 8.2, B1 H8 S512 D128 11.6 | 7.5, B1 H16 S512 D64 8.4 | 7.7, B1 H4 S768 D128 15.7 | 9.7.)
constexpr int RB = 1, PV_ROWS = 16 * RB;
template <int D>
__global__ __launch_bounds__(256, 2) void causal_pv_f32(const float *__restrict__ P, const float *__restrict__ V, float *__restrict__ O, int S,
                                                     int heads, int tiles, int cus, float scale)
{
    constexpr int NB = D / 64, CH = 4 * RB * NB < 8 ? 4 * RB * NB : 8;
    __shared__ f32x4 part[4 * CH * 64];
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    const int p0 = (tiles - 1 - tile) * PV_ROWS;   // longest rows first
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const float *Vp = V + (int64_t)bh * S * D + 4 * r;
    int prow[RB];
    const float *Pp[RB];
#pragma unroll
    for (int k = 0; k < RB; ++k) {
        prow[k] = p0 + 16 * k + r;
        Pp[k] = P + (int64_t)bh * S * S + (int64_t)(prow[k] < S ? prow[k] : S - 1) * S;
    }
    const int last = p0 + PV_ROWS - 1 < S - 1 ? p0 + PV_ROWS - 1 : S - 1, j_end = last / 16;
    f32x4 acc[RB][NB][4];
#pragma unroll
    for (int k = 0; k < RB; ++k)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[k][b][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int DEPTH = NB == 1 ? 4 : 2;   // steps in flight
    f32x4 pa[DEPTH][RB], va[DEPTH][4][NB];
    auto step_of = [&](int n) { return 4 * n + wave; };
    auto fetch = [&](int j, int set) __attribute__((always_inline)) {
        const int q = 16 * j + 4 * g;
#pragma unroll
        for (int k = 0; k < RB; ++k) pa[set][k] = *reinterpret_cast<const f32x4 *>(Pp[k] + (q <= prow[k] && q < S ? q : 0));
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int b = 0; b < NB; ++b) va[set][t][b] = *reinterpret_cast<const f32x4 *>(Vp + (int64_t)(q + t < S ? q + t : S - 1) * D + 64 * b);
    };
    auto work = [&](int j, int set) __attribute__((always_inline)) {
        const int q = 16 * j + 4 * g;
        if (16 * j + 15 > p0) {   // (wavefront-uniform) keys beyond the row: 0
#pragma unroll
            for (int k = 0; k < RB; ++k)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (q + t > (prow[k] < S - 1 ? prow[k] : S - 1)) pa[set][k][t] = 0.0f;
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int k = 0; k < RB; ++k) mma4(acc[k][b][u], va[set][t][b][u], pa[set][k][t]);
    };
    // this wavefront's steps, one of every four: fetched DEPTH - 1 ahead (a step past the end re-reads what is in bounds)
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) fetch(step_of(d), d);
    for (int n = 0; step_of(n) <= j_end; n += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            fetch(step_of(n + d + DEPTH - 1), (d + DEPTH - 1) % DEPTH);
            const int j = step_of(n + d);
            if (j <= j_end) work(j, d);
        }
    }
    // vectors over u (four consecutive columns): acc[k][b][.][v] of row prow[k] is columns 64b + 16g + 4v .. + 3
    float *Op = O + (int64_t)bh * S * D;
    reduce_waves<4 * RB * NB, CH>(part, wave, lane,
        [&](int e) {
            const int k = e / (4 * NB), b = e / 4 % NB, v = e % 4;
            return f32x4{acc[k][b][0][v], acc[k][b][1][v], acc[k][b][2][v], acc[k][b][3][v]};
        },
        [&](int c, int i, f32x4 sum) {
            const int e = c + i * 4 + wave, k = e / (4 * NB), b = e / 4 % NB, v = e % 4, p = p0 + 16 * k + r;
            if (p < S) *reinterpret_cast<f32x4 *>(Op + (int64_t)p * D + 64 * b + 16 * g + 4 * v) = sum * scale;
        });
}

// ---- ptx: a workgroup owns 32 keys, its wavefronts every fourth step of 4 query rows ---------------------------------------
constexpr int PT_KW = 2, PT_KEYS = 16 * PT_KW;   // keys per lane (operand row), per workgroup
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int D>
__global__ __launch_bounds__(256, 2) void causal_ptx_f32(const float *__restrict__ P, const float *__restrict__ X, float *__restrict__ O, int S,
                                                      int heads, int tiles, int cus, float scale)
{
    constexpr int NB = D / 64;
    __shared__ f32x4 part[4 * 8 * 64];
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    const int k0 = tile * PT_KEYS;   // the first keys have the most query rows
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int key = k0 + PT_KW * r;   // this lane's keys: key, key + 1
    const float *Pp = P + (int64_t)bh * S * S + (key < S ? key : k0), *Xp = X + (int64_t)bh * S * D + 4 * r;
    f32x4 acc[PT_KW][NB][4];
#pragma unroll
    for (int w = 0; w < PT_KW; ++w)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[w][b][u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int DEPTH = NB == 1 ? 8 : 4;   // steps in flight
    f32x2 pa[DEPTH];
    f32x4 xa[DEPTH][NB];
    const int j0 = k0 / 4, j_end = (S - 1) / 4;
    auto fetch = [&](int j, int set) __attribute__((always_inline)) {
        const int p = 4 * j + g < S ? 4 * j + g : S - 1;
        pa[set] = *reinterpret_cast<const f32x2 *>(Pp + (int64_t)p * S);
#pragma unroll
        for (int b = 0; b < NB; ++b) xa[set][b] = *reinterpret_cast<const f32x4 *>(Xp + (int64_t)p * D + 64 * b);
    };
    auto work = [&](int j, int set) __attribute__((always_inline)) {
        if (4 * j < k0 + PT_KEYS || 4 * j + 4 > S) {   // (wavefront-uniform) query rows above the key, or past the sequence: 0
            const int p = 4 * j + g;
#pragma unroll
            for (int w = 0; w < PT_KW; ++w)
                if (p < key + w || p >= S) pa[set][w] = 0.0f;
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int w = 0; w < PT_KW; ++w) mma4(acc[w][b][u], xa[set][b][u], pa[set][w]);
    };
    // this wavefront's steps j0 + wave, + 4, ...: fetched DEPTH ahead (a step past the end re-reads the last row)
    const int jw = j0 + wave;
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d) fetch(jw + 4 * d, d);
    for (int j = jw; j <= j_end; j += 4 * DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            fetch(j + 4 * (d + DEPTH - 1), (d + DEPTH - 1) % DEPTH);
            if (j + 4 * d <= j_end) work(j + 4 * d, d);
        }
    }
    float *Op = O + (int64_t)bh * S * D;
    reduce_waves<4 * PT_KW * NB, 8>(part, wave, lane,
        [&](int e) {
            const int w = e / (4 * NB), b = e / 4 % NB, v = e % 4;
            return f32x4{acc[w][b][0][v], acc[w][b][1][v], acc[w][b][2][v], acc[w][b][3][v]};
        },
        [&](int c, int i, f32x4 sum) {
            const int e = c + i * 4 + wave, w = e / (4 * NB), b = e / 4 % NB, v = e % 4;
            if (key + w < S) *reinterpret_cast<f32x4 *>(Op + (int64_t)(key + w) * D + 64 * b + 16 * g + 4 * v) = sum * scale;
        });
}

// ---- pv and ptx of larger grids ---------------------------------------------------------------------------------------------
// The kernels above pull V (X) through the L1 again for every 32 rows and wavefront.  Here RW wavefronts of 16 rows share a block of it
// in LDS (BK keys, PB query rows; copied asynchronously, one block ahead) and GR groups of them take every GR-th block; a
// wavefront's rows of P come straight from memory (ptx: through LDS, column-wise).  What bounds them is the fp32 matrix rate of
// one CU - 64 rows of 1024 keys keep it busy for 15 us - so that the grid has to be even: blocks as long as the chip is filled
// with, and the order of longest_first().  us, the kernel above | RW GR = 2 4 | 4 2 | 4 1:
//   pv   B1 H8 S1024 D128 (n32 = 256 blocks of 32 rows) 20.8 | 23.7 | 37.5 | 39.0, B1 H12 S768 D128 (288) 25.9 | 18.9 | 29.5 | 30.2,
//        B1 H16 S1024 D64 (512) 19.7 | 15.4 | 22.5 | 22.8, D128 36.5 | 25.8 | 38.8 | 40.6, B1 H32 S1024 D64 (n64 = 512 blocks of 64)
//        40.2 | 29.0 | 25.6 | 25.4, D128 82.5 | 50.7 | 43.3 | 43.4, B1 H16 S2048 D64 (512) 72.9 | 61.1 | 50.6 | 55.2, B4 H16 S768 D64 (768)
//        45.0 | 33.9 | 32.3 | 29.0, B4 H16 S1024 D64 (1024) 71.4 | 56.3 | 50.8 | 46.3, B2 H32 S1024 D128 148 | 91.5 | 86.9 | 82.7
//   ptx  (no RW = 2) B4 H8 S768 D64 (n64 = 384) 18.0 | - | 19.4 | 21.3, B1 H32 S1024 D64 (512) 29.2 | - | 26.3 | 28.5, D128 50.5 | - | 44.6 |
//        46.8, B1 H16 S2048 D128 (512) 91.1 | - | 81.2 | 86.1, B4 H16 S1024 D64 (1024) 56.0 | - | 52.5 | 49.9
// The line of ptx at 512 is two blocks for every CU, where RW GR = 4 2 is ahead at both head sizes.  Between 384 and 512, the kernel above |
// 4 2, us: D64 416 (S1024) 28.8 | 26.6, (S2048) 51.0 | 45.2, 480 (S3072) 73.8 | 68.1, 488 (S3904) 86.8 | 83.5, 496 (S512) 20.9 | 16.4; D128 416
// (S1024) 47.0 | 46.0, (S2048) 82.5 | 85.3, 448 (S1024) 46.0 | 46.3, (S2048) 86.6 | 85.6, 480 (S1024) 51.4 | 46.9, (S3072) 127 | 126, 488 (S3904)
// 154 | 158, 496 (S512) 32.1 | 27.7: head size 64 would gain from 416 on.
// The sums of GR groups of GT threads, N vectors each, added up in the first group (true there): the upper half of the groups hand
// theirs to the lower half through LDS until one is left.
template <int N, int GT, int GR> __device__ __forceinline__ bool group_sums(float *lds, f32x4 (&acc)[N], int grp, int tid)
{
    f32x4 *const part = reinterpret_cast<f32x4 *>(lds);
    __syncthreads();   // nobody reads operands any more
#pragma unroll
    for (int h = GR / 2; h > 0; h /= 2) {
        if (grp >= h && grp < 2 * h) {
#pragma unroll
            for (int i = 0; i < N; ++i) part[((grp - h) * N + i) * GT + tid] = acc[i];
        }
        __syncthreads();
        if (grp < h) {
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i] += part[(grp * N + i) * GT + tid];
        }
        if (h > 1) __syncthreads();
    }
    return grp == 0;
}

template <int D, int RW, int GR, int BK>
__global__ __launch_bounds__(64 * RW * GR, 4) void causal_pv_f32_shared(const float *__restrict__ P, const float *__restrict__ V, float *__restrict__ O,
                                                                        int S, int heads, int tiles, int cus, float scale)
{
    constexpr int NB = D / 64, GT = 64 * RW, ROWS = 16 * RW, CPR = D / 4, ROUNDS = BK * CPR / GT, STEPS = BK / 16, N = 4 * NB;
    static_assert(BK * CPR % GT == 0 && GT % CPR == 0 && N * GT * 16 * GR / 2 <= GR * BK * D * 4, "whole copy rounds; the sums fit a buffer");
    __shared__ __align__(16) float v_a_all[GR * BK * D];
    __shared__ __align__(16) float v_b_all[GR * BK * D];
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
    float *const v_a = v_a_all + grp * (BK * D), *const v_b = v_b_all + grp * (BK * D);
    const int p0 = (tiles - 1 - tile) * ROWS, w0 = p0 + wave * 16, prow = w0 + r, lim = prow < S ? prow : S - 1;
    const float *Vp = V + (int64_t)bh * S * D, *Pp = P + (int64_t)bh * S * S + (int64_t)lim * S;
    const int row0 = tid / CPR, col0 = tid % CPR * 4;
    auto issue = [&](int j, float *dst) {   // keys past the sequence re-read the last one: their probabilities are masked
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) {
            const int key = j * BK + row0 + i * (GT / CPR);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Vp + (int64_t)(key < S ? key : S - 1) * D + col0), (lds_void_t *)(dst + (i * GT + wave * 64) * 4),
                                             16, 0, 0);
        }
    };
    auto load_p = [&](int j, f32x4 (&pf)[STEPS]) {
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int key = j * BK + 16 * s + 4 * g;
            pf[s] = *reinterpret_cast<const f32x4 *>(Pp + (key <= lim ? key : 0));
        }
    };
    const int last = p0 + ROWS - 1 < S - 1 ? p0 + ROWS - 1 : S - 1, j_end = last / BK, nsteps = j_end / GR + 1;
    f32x4 acc[N];   // acc[4b + u][v]: column 64b + 16g + 4v + u of row prow
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 p_a[STEPS], p_b[STEPS];
    if (grp <= j_end) issue(grp, v_a);
    load_p(grp, p_a);
    auto step = [&](int j, const float *Vb, float *Vn, f32x4 (&pf)[STEPS], f32x4 (&pn)[STEPS]) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // V block j and the rows' vectors have arrived
        __syncthreads();                 // for every wavefront; reads of the other buffer are finished
        if (j > j_end) return;
        if (j + GR <= j_end) {
            issue(j + GR, Vn);
            load_p(j + GR, pn);
        }
        if (j * BK > w0 + 15) return;   // wholly above the diagonal for these rows
        if (j * BK + BK - 1 > w0) {
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (j * BK + 16 * s + 4 * g + t > lim) pf[s][t] = 0.0f;
        }
        const float *at = Vb + 4 * g * D + 4 * r;
        f32x4 part[N];   // the block's own sums: chains of BK / 4 products, and a step of the total per block
#pragma unroll
        for (int i = 0; i < N; ++i) part[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 av[2][NB];
        auto read = [&](int i, f32x4 (&dst)[NB]) {
#pragma unroll
            for (int b = 0; b < NB; ++b) dst[b] = *reinterpret_cast<const f32x4 *>(at + (16 * (i >> 2) + (i & 3)) * D + 64 * b);
        };
        read(0, av[0]);
#pragma unroll
        for (int i = 0; i < 4 * STEPS; ++i) {
            if (i + 1 < 4 * STEPS) read(i + 1, av[(i + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);   // (the reads stay ahead of the products)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < 4; ++u) mma4(part[4 * b + u], av[i & 1][b][u], pf[i >> 2][i & 3]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] += part[i];
    };
    for (int i = 0, j = grp;;) {
        step(j, v_a, v_b, p_a, p_b);
        if (++i >= nsteps) break;
        j += GR;
        step(j, v_b, v_a, p_b, p_a);
        if (++i >= nsteps) break;
        j += GR;
    }
    if constexpr (GR > 1) {
        if (!group_sums<N, GT, GR>(v_a_all, acc, grp, tid)) return;
    }
    if (prow >= S) return;
    float *Op = O + (int64_t)bh * S * D + (int64_t)prow * D + 16 * g;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            *reinterpret_cast<f32x4 *>(Op + 64 * b + 4 * v) = f32x4{acc[4 * b][v], acc[4 * b + 1][v], acc[4 * b + 2][v], acc[4 * b + 3][v]} * scale;
}

// ptx: a P tile row holds 16-byte chunk c at position c ^ 4 (row % 4), so that the four rows of a product's operand lie in different
// banks
template <int D, int RW, int GR, int PB>
__global__ __launch_bounds__(64 * RW * GR, 4) void causal_ptx_f32_shared(const float *__restrict__ P, const float *__restrict__ X, float *__restrict__ O,
                                                                         int S, int heads, int tiles, int cus, float scale)
{
    constexpr int NB = D / 64, GT = 64 * RW, KB = 16 * RW, XC = D / 4, PC = KB / 4, XR = PB * XC / GT, PR = PB * PC / GT, N = 4 * NB;
    static_assert(PB * XC % GT == 0 && PB * PC % GT == 0 && GT / PC % 4 == 0, "whole copy rounds that keep the swizzle phase");
    constexpr int BUF = PB * (D + KB);   // floats of a block: X, then P
    constexpr int SUMS = N * GT * 4 * GR / 2;        // floats of half the groups' sums
    __shared__ __align__(16) float a_all[GR * BUF > SUMS ? GR * BUF : SUMS];
    __shared__ __align__(16) float b_all[GR * BUF];
    int bh, tile;
    if (!longest_first(heads, tiles, cus, bh, tile)) return;
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
    float *const a = a_all + grp * BUF, *const b = b_all + grp * BUF;
    const int k0 = tile * KB, w0 = k0 + wave * 16, krow = w0 + r;   // (the first keys have the most query rows)
    const float *Pp = P + (int64_t)bh * S * S, *Xp = X + (int64_t)bh * S * D;
    const int xrow0 = tid / XC, xcol = tid % XC * 4, prow0 = tid / PC, pcol = ((tid % PC) ^ (4 * (prow0 & 3))) * 4;
    const int pfrom = k0 + pcol < S ? k0 + pcol : k0;   // (keys past the sequence: rows of the result that nobody stores)
    auto issue = [&](int j, float *dst) {   // rows past the sequence re-read the last one: they are masked
#pragma unroll
        for (int i = 0; i < XR; ++i) {
            const int row = j * PB + xrow0 + i * (GT / XC);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Xp + (int64_t)(row < S ? row : S - 1) * D + xcol), (lds_void_t *)(dst + (i * GT + wave * 64) * 4), 16,
                                             0, 0);
        }
#pragma unroll
        for (int i = 0; i < PR; ++i) {
            const int row = j * PB + prow0 + i * (GT / PC);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Pp + (int64_t)(row < S ? row : S - 1) * S + pfrom),
                                             (lds_void_t *)(dst + PB * D + (i * GT + wave * 64) * 4), 16, 0, 0);
        }
    };
    const int j_start = k0 / PB, j_end = (S - 1) / PB, jg = j_start + ((grp - j_start) & (GR - 1)), nsteps = (j_end - j_start) / GR + 1;
    f32x4 acc[N];   // acc[4b + u][v]: column 64b + 16g + 4v + u of key krow
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (jg <= j_end) issue(jg, a);
    const int xat = g * D + 4 * r, pat = PB * D + g * KB + (((wave * 4 + (r >> 2)) ^ (4 * g)) * 4) + (r & 3);
    auto step = [&](int j, const float *cur, float *next) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // block j has arrived
        __syncthreads();                 // for every wavefront; reads of the other buffer are finished
        if (j > j_end) return;
        if (j + GR <= j_end) issue(j + GR, next);
        const int pbase = j * PB;
        if (pbase + PB - 1 < w0) return;   // every row of the block lies above these keys
        const bool edge = pbase + PB > S || pbase < w0 + 15;
        f32x4 part[N];   // (as in pv)
#pragma unroll
        for (int i = 0; i < N; ++i) part[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        f32x4 xv[2][NB];
        float pv[2];
        auto read = [&](int i, int set) {
            pv[set] = cur[pat + 4 * i * KB];
#pragma unroll
            for (int c = 0; c < NB; ++c) xv[set][c] = *reinterpret_cast<const f32x4 *>(cur + xat + 4 * i * D + 64 * c);
        };
        read(0, 0);
#pragma unroll
        for (int i = 0; i < PB / 4; ++i) {
            if (i + 1 < PB / 4) read(i + 1, (i + 1) & 1);
            float p = pv[i & 1];
            if (edge) {   // query rows above the key (P is undefined there) or past the sequence count as 0
                const int row = pbase + 4 * i + g;
                if (row < krow || row >= S) p = 0.0f;
            }
            __builtin_amdgcn_sched_barrier(0);   // (the reads stay ahead of the products)
#pragma unroll
            for (int c = 0; c < NB; ++c)
#pragma unroll
                for (int u = 0; u < 4; ++u) mma4(part[4 * c + u], xv[i & 1][c][u], p);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < N; ++i) acc[i] += part[i];
    };
    for (int i = 0, j = jg;;) {
        step(j, a, b);
        if (++i >= nsteps) break;
        j += GR;
        step(j, b, a);
        if (++i >= nsteps) break;
        j += GR;
    }
    if constexpr (GR > 1) {
        if (!group_sums<N, GT, GR>(a_all, acc, grp, tid)) return;
    }
    if (krow >= S) return;
    float *Op = O + (int64_t)bh * S * D + (int64_t)krow * D + 16 * g;
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            *reinterpret_cast<f32x4 *>(Op + 64 * c + 4 * v) = f32x4{acc[4 * c][v], acc[4 * c + 1][v], acc[4 * c + 2][v], acc[4 * c + 3][v]} * scale;
}

int check(const void *a, const void *b, const void *c, int64_t B, int64_t H, int64_t S, int64_t D)
{
    if (!a || !b || !c) return MTA_ERR_NULL;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 20) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(a, 16) || !aligned_to(b, 16) || !aligned_to(c, 16)) return MTA_ERR_ALIGN;
    if (S % 4 != 0) return MTA_ERR_UNSUPPORTED;
    return MTA_OK;
}

// Scores on tiles of 128 x 128 in LDS slabs from half a workgroup per CU on, on the bf16 matrix cores (tri_products_split.hip) from 300 tiles on, and
// at D = 128 instead of the slabs: us, direct | slabs | split: D64 B1 H8 S512 (80 tiles) 6.2 | 9.4 | 8.5, B1 H16 S512 (160) 14.8 | 9.4 | 9.1, B2 H16
// S512 (320) - | 15.1 | 13.2, B1 H16 S1024 (576) 24.7 | 22.2 | 18.3; D128 (80) 8.4 | 13.2 | 11.1, (160) 17.5 | 14.7 | 12.1, (576) 39.5 | 34.4 | 26.2.

// resident: workgroups that a CU holds at once
template <typename K, typename... ARGS>
int launch(K kern, int64_t heads, int64_t tiles, int threads, int resident, hipStream_t st, const void *a, const void *b, void *c, int64_t S,
           ARGS... more)
{
    const int64_t total = heads * tiles, grid = (total + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return MTA_ERR_SHAPE;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(threads), 0, st, (const float *)a, (const float *)b, (float *)c, (int)S, (int)heads, (int)tiles,
                       total <= (int64_t)resident * device_cu_count() ? device_cu_count() / 8 : 0, more...);
    return launch_status();
}
}  // namespace

extern "C" int mta_lower_scores_f32(const void *a, const void *b, void *out, int64_t B, int64_t H, int64_t S, int64_t D, void *stream)
{
    const int rc = check(a, b, out, B, H, S, D);
    if (rc != MTA_OK) return rc;
    const int64_t n = (S + SL_TILE - 1) / SL_TILE;
    const int64_t tiles = B * H * (n * (n + 1) / 2);
    if (tiles >= (D == 64 ? 300 : 128)) return lower_scores_split_launch(a, b, out, B * H, S, D, (hipStream_t)stream);
    if (tiles >= 128) return launch(lower_scores_f32_slabs<64>, B * H, n * (n + 1) / 2, 256, 0, (hipStream_t)stream, a, b, out, S);
    // Grids that leave most of the chip idle: tiles of a quarter, whose wavefronts are done in a quarter of the time (us, 64 x 128 | 32 x 64:
    // B1 H4 S256 D64 (24 workgroups of 64 x 128) 5.7 | 3.9, H8 (48) 5.7 | 3.9, H4 S512 (80) 6.2 | 5.2, H8 S512 (160) 6.4 | 6.8).
    const int64_t large = sc_tiles((int)((S + sc_rows<2>() - 1) / sc_rows<2>())), small = sc_tiles((int)((S + sc_rows<1>() - 1) / sc_rows<1>()));
    auto go = [&](auto d64, auto d128, int64_t tiles) { return launch(D == 64 ? d64 : d128, B * H, tiles, 256, 0, (hipStream_t)stream, a, b, out, S); };
    return B * H * large <= 100 ? go(lower_scores_f32<64, 1>, lower_scores_f32<128, 1>, small) : go(lower_scores_f32<64, 2>, lower_scores_f32<128, 2>, large);
}

extern "C" int mta_causal_pv_f32(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int64_t D, float scale, void *stream)
{
    const int rc = check(p, v, o, B, H, S, D);
    if (rc != MTA_OK) return rc;
    const int64_t b32 = (S + 31) / 32, b64 = (S + 63) / 64;
    auto go = [&](auto d64, auto d128, int64_t blocks, int threads, int resident) {
        return launch(D == 64 ? d64 : d128, B * H, blocks, threads, resident, (hipStream_t)stream, p, v, o, S, scale);
    };
    if (B * H * b32 <= 256) return go(causal_pv_f32<64>, causal_pv_f32<128>, (S + PV_ROWS - 1) / PV_ROWS, 256, 3);
    if (B * H * b64 < 512) return go(causal_pv_f32_shared<64, 2, 4, 32>, causal_pv_f32_shared<128, 2, 4, 16>, b32, 512, 2);
    if (B * H * b64 < 768) return go(causal_pv_f32_shared<64, 4, 2, 64>, causal_pv_f32_shared<128, 4, 2, 32>, b64, 512, 2);
    return go(causal_pv_f32_shared<64, 4, 1, 64>, causal_pv_f32_shared<128, 4, 1, 32>, b64, 256, 4);
}

extern "C" int mta_causal_ptx_f32(const void *p, const void *x, void *o, int64_t B, int64_t H, int64_t S, int64_t D, float scale, void *stream)
{
    const int rc = check(p, x, o, B, H, S, D);
    if (rc != MTA_OK) return rc;
    const int64_t b64 = (S + 63) / 64;
    auto go = [&](auto d64, auto d128, int64_t blocks, int threads, int resident) {
        return launch(D == 64 ? d64 : d128, B * H, blocks, threads, resident, (hipStream_t)stream, p, x, o, S, scale);
    };
    if (B * H * b64 < 512) return go(causal_ptx_f32<64>, causal_ptx_f32<128>, (S + PT_KEYS - 1) / PT_KEYS, 256, D == 64 ? 5 : 4);
    if (B * H * b64 < 768) return go(causal_ptx_f32_shared<64, 4, 2, 32>, causal_ptx_f32_shared<128, 4, 2, 16>, b64, 512, 2);
    return go(causal_ptx_f32_shared<64, 4, 1, 32>, causal_ptx_f32_shared<128, 4, 1, 32>, b64, 256, D == 64 ? 5 : 3);
}
