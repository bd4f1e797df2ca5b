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
// No LDS in the loops: which element feeds which operand slot is free as long as both operands agree, and each product has an
// assignment in which every operand is 16 (P of ptx: 8) contiguous bytes per lane -
//   scores: contraction d = 16s + 4g + t for slot group g at step t: a lane's vector of its row is four steps' operand;
//   pv:     contraction q = 16j + 4g + t (P's vector), output column d = 64b + 4r + u for operand row r of product u (V's
//           vector of key q is four products' operand);
//   ptx:    contraction p = 4j + g, output row q = 2r + w of product w (P's pair), column d as above (X's vector)
// (lane = 16g + r).  A line fetched by one lane's load is used up by its neighbours in the same instruction.
// us against the library GEMM (scores / pv / ptx): B1 H4 S256 D64 5.8 / 5.5 / 5.5 against 24 / 21 / 22, where launching is all
// there is; B1 H16 S512 11 / 8 / 9 against 21 / 20 / 21; B1 H32 S1024 38 / 38 / 31 against 55 / 36 / 35 (the library's operand
// has to be filled above the diagonal first, which is another 15 us).  Tried for pv and not kept: 64 rows per workgroup, pairs
// of adjacent steps per wavefront, non-temporal loads of P (38 -> 44, 40, 42 us at the last size).
#include "common.hpp"
#include "mfma.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

__device__ __forceinline__ void mma4(f32x4 &c, float a, float b) { c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// (batch*head, tile) of a workgroup: XCD x (workgroup id % 8) takes the x-th eighth of the list, so that the workgroups of a
// head share an L2; where the heads divide evenly (hpx of them per XCD) their tiles are started rank by rank, the longest of
// every head first (tile 0), so that the short ones fill the end of the grid
__device__ __forceinline__ bool place(int tiles, int64_t total, int64_t per_xcd, int hpx, int64_t &bh, int &tile)
{
    const int64_t pos = blockIdx.x >> 3, lid = (int64_t)(blockIdx.x & 7) * per_xcd + pos;
    if (lid >= total) return false;
    if (hpx > 0) {
        bh = (int64_t)(blockIdx.x & 7) * hpx + pos % hpx;
        tile = (int)(pos / hpx);
    } else {
        bh = lid / tiles;
        tile = (int)(lid - bh * tiles);
    }
    return true;
}

// ---- scores: a wavefront owns 32 query rows x 64 keys, a workgroup 64 x 128 -----------------------------------------------
constexpr int SC_ROWS = 64, SC_KEYS = 128;

// tiles on or below the diagonal of the first n rows of tiles, two tile rows per tile column
__host__ __device__ __forceinline__ int sc_tiles(int n) { return (n / 2) * (n / 2 + 1) + (n & 1) * (n / 2 + 1); }

template <int D>
__global__ __launch_bounds__(256) void lower_scores_f32(const float *__restrict__ A, const float *__restrict__ Bm, float *__restrict__ C,
                                                        int S, int tiles, int64_t total, int64_t per_xcd, int hpx)
{
    static_assert(SC_KEYS == 2 * SC_ROWS, "two tile rows per tile column");
    int64_t bh;
    int tile;
    if (!place(tiles, total, per_xcd, hpx, bh, tile)) return;
    // tile row: the largest n with sc_tiles(n) <= tile
    int tr = (int)(2.0f * sqrtf((float)tile));
    while (sc_tiles(tr) > tile) --tr;
    while (sc_tiles(tr + 1) <= tile) ++tr;
    const int tc = tile - sc_tiles(tr);
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int p0 = tr * SC_ROWS + (wave & 1) * 32, q0 = tc * SC_KEYS + (wave >> 1) * 64;
    if (p0 >= S || q0 >= S || q0 > p0 + 31) return;   // (outside, or wholly above the diagonal)
    const float *Ap = A + bh * (int64_t)S * D + g * 4, *Bp = Bm + bh * (int64_t)S * D + g * 4;
    int arow[2], brow[4];
#pragma unroll
    for (int i = 0; i < 2; ++i) arow[i] = (p0 + 16 * i + r < S ? p0 + 16 * i + r : S - 1) * D;
#pragma unroll
    for (int i = 0; i < 4; ++i) brow[i] = (q0 + 16 * i + r < S ? q0 + 16 * i + r : S - 1) * D;
    f32x4 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k) acc[i][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 a[2][2], b[2][4];
    auto fetch = [&](int s, int set) {
#pragma unroll
        for (int i = 0; i < 2; ++i) a[set][i] = *reinterpret_cast<const f32x4 *>(Ap + arow[i] + 16 * s);
#pragma unroll
        for (int i = 0; i < 4; ++i) b[set][i] = *reinterpret_cast<const f32x4 *>(Bp + brow[i] + 16 * s);
    };
    fetch(0, 0);
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
        if (s + 1 < D / 16) fetch(s + 1, (s + 1) & 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int k = 0; k < 2; ++k) mma4(acc[i][k], b[s & 1][i][t], a[s & 1][k][t]);
    }
    // acc[i][k][v]: key q0 + 16i + 4g + v of query row p0 + 16k + r
    float *Cp = C + bh * (int64_t)S * S;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
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

// ---- scores of large grids: a workgroup owns 128 query rows x 128 keys, its wavefronts 64 x 64 each ------------------------
// The kernel above pulls 6 KB through the L1 for every 32 products.  Here slabs of 16 head dims of both operands are copied
// global -> LDS asynchronously, one slab ahead, and serve all four wavefronts: a third of the bytes per product.  What bounds it
// now is the fp32 matrix rate (64 more head dims cost 25 us at B1 H32 S1024, 91 TFLOP/s) with the write of the scores behind it.  A slab row is four 16-byte
// chunks, XOR-swizzled by bits 2 and 3 of the row: the lanes that the LDS serves together (0-7 with 24-31, ...) then cover its
// banks once.
constexpr int SL_TILE = 128, SL_D = 16;
template <int D>
__global__ __launch_bounds__(256, 3) void lower_scores_f32_slabs(const float *__restrict__ A, const float *__restrict__ Bm, float *__restrict__ C,
                                                                 int S, int tiles, int64_t total, int64_t per_xcd, int hpx)
{
    __shared__ __align__(16) float a_buf[2][SL_TILE * SL_D];
    __shared__ __align__(16) float b_buf[2][SL_TILE * SL_D];
    int64_t bh;
    int tile;
    if (!place(tiles, total, per_xcd, hpx, bh, tile)) return;
    int tr = (int)(sqrtf(2.0f * (float)tile + 0.25f) - 0.5f);   // tile row: tr (tr + 1) / 2 tiles lie ahead of it
    while (tr * (tr + 1) / 2 > tile) --tr;
    while ((tr + 1) * (tr + 2) / 2 <= tile) ++tr;
    const int tc = tile - tr * (tr + 1) / 2;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, g = lane >> 4;
    const float *Ap = A + bh * (int64_t)S * D, *Bp = Bm + bh * (int64_t)S * D;
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
    float *Cp = C + bh * (int64_t)S * S;
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

// ---- pv: a workgroup owns 32 query rows, its wavefronts every fourth step of 16 keys ---------------------------------------
constexpr int RB = 2, PV_ROWS = 16 * RB;
template <int D>
__global__ __launch_bounds__(256, 2) void causal_pv_f32(const float *__restrict__ P, const float *__restrict__ V, float *__restrict__ O, int S,
                                                     int tiles, int64_t total, int64_t per_xcd, int hpx, float scale)
{
    constexpr int NB = D / 64;
    __shared__ f32x4 part[4 * 8 * 64];
    int64_t bh;
    int tile;
    if (!place(tiles, total, per_xcd, hpx, bh, tile)) return;
    const int p0 = (tiles - 1 - tile) * PV_ROWS;   // longest rows first
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const float *Vp = V + bh * (int64_t)S * D + 4 * r;
    int prow[RB];
    const float *Pp[RB];
#pragma unroll
    for (int k = 0; k < RB; ++k) {
        prow[k] = p0 + 16 * k + r;
        Pp[k] = P + bh * (int64_t)S * S + (int64_t)(prow[k] < S ? prow[k] : S - 1) * S;
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
    float *Op = O + bh * (int64_t)S * D;
    reduce_waves<4 * RB * NB, 8>(part, wave, lane,
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
                                                      int tiles, int64_t total, int64_t per_xcd, int hpx, float scale)
{
    constexpr int NB = D / 64;
    __shared__ f32x4 part[4 * 8 * 64];
    int64_t bh;
    int tile;
    if (!place(tiles, total, per_xcd, hpx, bh, tile)) return;
    const int k0 = tile * PT_KEYS;   // the first keys have the most query rows
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int key = k0 + PT_KW * r;   // this lane's keys: key, key + 1
    const float *Pp = P + bh * (int64_t)S * S + (key < S ? key : k0), *Xp = X + bh * (int64_t)S * D + 4 * r;
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
    float *Op = O + bh * (int64_t)S * D;
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

int check(const void *a, const void *b, const void *c, int64_t B, int64_t H, int64_t S, int64_t D)
{
    if (!a || !b || !c) return MTA_ERR_NULL;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 20) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(a, 16) || !aligned_to(b, 16) || !aligned_to(c, 16)) return MTA_ERR_ALIGN;
    if (S % 4 != 0) return MTA_ERR_UNSUPPORTED;
    return MTA_OK;
}

// Whether the scores run on tiles of 128 x 128 in LDS slabs: from half a workgroup per CU on (us, direct | slabs, D64 / D128:
// B1 H8 S512, 80 tiles, 6.7 | 9.4 / 9.5 | 13.2; B1 H16 S512, 160, 14.8 | 9.9 / 17.5 | 14.2; B1 H16 S1024, 576, 24.7 | 23.5 / 39.5 | 35.5;
// B1 H32 S1024, 1152, 40.7 | 38.8 / 69.3 | 63.8; B1 H16 S2048, 2176, 73.2 | 62.5 / 127 | 105).
bool scores_slabs(int64_t tiles) { return tiles >= 128; }

template <typename K, typename... ARGS>
int launch(K kern, int64_t bh, int64_t tiles, hipStream_t st, const void *a, const void *b, void *c, int64_t S, ARGS... more)
{
    const int64_t total = bh * tiles, per_xcd = (total + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL || tiles > 0x7fffffffLL) return MTA_ERR_SHAPE;
    hipLaunchKernelGGL(kern, dim3((unsigned)(per_xcd * 8)), dim3(256), 0, st, (const float *)a, (const float *)b, (float *)c, (int)S, (int)tiles,
                       total, per_xcd, bh % 8 == 0 ? (int)(bh / 8) : 0, more...);
    return launch_status();
}
}  // namespace

extern "C" int mta_lower_scores_f32(const void *a, const void *b, void *out, int64_t B, int64_t H, int64_t S, int64_t D, void *stream)
{
    const int rc = check(a, b, out, B, H, S, D);
    if (rc != MTA_OK) return rc;
    const int64_t n = (S + SL_TILE - 1) / SL_TILE;
    if (scores_slabs(B * H * n * (n + 1) / 2))
        return D == 64 ? launch(lower_scores_f32_slabs<64>, B * H, n * (n + 1) / 2, (hipStream_t)stream, a, b, out, S)
                       : launch(lower_scores_f32_slabs<128>, B * H, n * (n + 1) / 2, (hipStream_t)stream, a, b, out, S);
    const int64_t tiles = sc_tiles((int)((S + SC_ROWS - 1) / SC_ROWS));
    return D == 64 ? launch(lower_scores_f32<64>, B * H, tiles, (hipStream_t)stream, a, b, out, S)
                   : launch(lower_scores_f32<128>, B * H, tiles, (hipStream_t)stream, a, b, out, S);
}

extern "C" int mta_causal_pv_f32(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int64_t D, float scale, void *stream)
{
    const int rc = check(p, v, o, B, H, S, D);
    if (rc != MTA_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const int64_t tiles = (S + PV_ROWS - 1) / PV_ROWS;
    return D == 64 ? launch(causal_pv_f32<64>, B * H, tiles, st, p, v, o, S, scale) : launch(causal_pv_f32<128>, B * H, tiles, st, p, v, o, S, scale);
}

extern "C" int mta_causal_ptx_f32(const void *p, const void *x, void *o, int64_t B, int64_t H, int64_t S, int64_t D, float scale, void *stream)
{
    const int rc = check(p, x, o, B, H, S, D);
    if (rc != MTA_OK) return rc;
    const int64_t tiles = (S + PT_KEYS - 1) / PT_KEYS;
    return D == 64 ? launch(causal_ptx_f32<64>, B * H, tiles, (hipStream_t)stream, p, x, o, S, scale)
                   : launch(causal_ptx_f32<128>, B * H, tiles, (hipStream_t)stream, p, x, o, S, scale);
}
