// The 16-bit kernels of conv_attn_fwd.hip (fused conv-attention and its scores-only half, everything on the matrix cores),
// a template over the I/O type: one translation unit per type instantiates it (conv_attn_bf16.hip, conv_attn_f16.hip).
#pragma once

#include <algorithm>
#include <type_traits>
#include <utility>

#include "conv_attn.hpp"
#include "mfma.hpp"

#include <stdlib.h>

namespace {
using namespace mta;

// =======================================================================================
// 16-bit fast path: everything on 16x16x32 MFMAs, conv included.
//
//  * 4 wavefronts own 128 score rows (HR halo rows + 128-HR output rows); a wavefront owns two
//    blocks of 16 rows.  Lane (r = lane%16, g = lane/16) owns query row r of a block; the
//    16x16 accumulator layout gives it keys 4g..4g+3 of every 16-key block, so a query row is
//    spread over 4 lanes and row reductions cost two lane exchanges.
//  * K and V blocks (64 keys) are copied global -> LDS asynchronously (global_load_lds), double
//    buffered, row-major, 16-byte chunks XOR-swizzled by the key index instead of padded.
//  * S^T = K Q^T -> causal/range zero -> LDS score tile (I/O dtype) -> conv as Toeplitz MFMAs
//    (out^T = T_i^T X^T per kernel row, the fragments of T_i^T live in registers) -> online
//    softmax in registers -> O^T += V^T P^T, where the V^T fragments come straight out of the
//    row-major V block through the LDS transpose read (ds_read_b64_tr_b16): within 16 lanes,
//    lane c supplies the address of 4 head-dim values of key c/4 and lane i receives head-dim
//    value i of 4 consecutive keys.
// =======================================================================================
typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void glb_void_t;
typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

// The workgroup has NW = 4 wavefronts and owns 128 score rows; two workgroups per CU for the attention kernel (three at D = 64 up
// to 7 kernel rows), three for the scores-only one, which overlap each other's barriers and memory latency.  Attention over small
// grids: NW = 8 with one block of 16 rows each, see launch_mfma.  (The scores-only kernel on eight, with the fragments of K read twice as
// often: 6x11 B2 H16 S512 D64 12.5 -> 17.4 us, B4 H16 S1024 D128 38.4 -> 43.2.)
// What bounds the attention kernel: matrix products (896 flops executed per score at 6x11, D = 128: Q K^T and P V 256 each, the
// conv as Toeplitz products 384) beside the vector ALU (the exponentials) and the LDS, which would each take 35 to 50 % of its
// time alone (6x11 B1 H32 S8192 D128, by counters: the matrix cores are busy 47 % of the cycles at about 2.1 GHz, the LDS 42 %, the vector ALU
// 37 %): what is left is how far the two wavefronts of a SIMD overlap them between two barriers per key block.  So the vector work is kept small (one maximum, one multiply-add, one exponential and half a conversion and a sum
// per score: no rounding between the conv and the probabilities) and is written between the products of the same wavefront:
// the first row block's probabilities among the second one's conv products, half of the second one's among those of P V.
// The loop has one body: K, V and the buffer the next block goes to are offsets into one LDS array (all reads of it are issued
// from assembly, so that the compiler cannot wait for the copy in flight), a key block that the diagonal or the end of the
// sequence does not touch branches around its masks, and every LDS operand is read several products ahead into a ring of
// registers.  211 registers (248 before, with three bodies): 11 kernel rows run two workgroups per CU as well.
// us, with the logits rounded twice in the I/O dtype and the softmax of a row block in one piece -> now: bf16 6x11 B1 H32 S8192
// D128 1067 -> 990 (executed 1.0 PFLOP/s; an 8192^3 library product reaches 1.08), 3x3 B1 H32 S4096 D128 276 -> 246, 7x7 B1 H16
// S2048 D128 98.9 -> 87.0, 6x11 B1 H8 S2048 D64 78.8 -> 66.7, 5x5 B2 H32 S4096 D64 378 -> 341; fp16 7x9 B4 H12 S2048 D64 120 -> 93,
// 11x15 B1 H32 S4096 D128 595 -> 360.
constexpr int F_BK = 64;   // keys per iteration
constexpr int QK_OCC = 3;     // wavefronts per SIMD the scores-only kernel is compiled for (three workgroups per CU)
constexpr int QK_CHUNK = 32;  // key blocks per work item of the scores-only kernel when no item table is built
// with an item table: long and short items (key blocks), and the share of a query block's key range that goes into short
// ones (MTA_QK_CHUNK_LONG / MTA_QK_CHUNK_SHORT / MTA_QK_SHORT_PERCENT in the environment override them, for comparisons)
// (long items measured at B2 H16 S4096 D128: 32/32/0 237 us, 16/16/0 231, 64/16/50 238, 48/24/50 228, 52/26/50 227, 48/24/35 243)
constexpr int QK_SHORT_PERCENT = 50;
constexpr int ITEM_TABLE_MAX = 768;
struct qk_chunks { int big, small; };
// How long the items are, from the launch's key blocks over all heads (768 workgroups are resident).  From 16000 on the grid
// runs in several rounds whatever the length and 48/24 keeps the rebuilt columns few; below, items as short as it takes to
// have two or three per CU, down to one key block, win although each rebuilds one key block's worth of columns: the grid is
// otherwise a fraction of the chip, each workgroup walking its keys alone.  us, 48/24 | as short as the rule makes them:
// B1 H8 S256 D64 3x3 (80 blocks) 13.3 | 7.6; B1 H16 S512 D128 5x5 (448) 23.3 | 11.5; B2 H16 S512 D64 6x11 (896) 22.6 | 13.4;
// B4 H16 S512 (1792) 26.3 | 22.0; B1 H8 S2048 D64 (2450) 48.9 | 23.9.
// Where the line lies, the kernel alone (in brackets the forward with groups of 4 heads / with all weights dense; three processes
// a side, which differ by up to 3 on the kernel and 2 on a forward), 48/24 | 16/8: B1 H16 S2048 D128 7x7 (5216) 62 | 51 (117 | 108 /
// 184 | 171); B1 H32 S2048 D64 5x5 (10432) 58 | 56 (158 | 156 / 394 | 392); B2 H16 S2048 D128 6x11 (10432) 68 | 69 (165 | 166 /
// 298 | 293); B1 H16 S3072 D128 3x3 (10688) 65 | 63 (199 | 190 / 309 | 297); B1 H16 S3712 D64 7x9 (15088) 82 | 81 (236 | 235 /
// 386 | 383); B3 H16 S2048 D128 7x7 (15648) 99 | 103 (241 | 245 / 395 | 396); B1 H16 S4096 D128 7x7 (19104) 121 | 126 (300 | 299 /
// 485 | 490); B4 H16 S2048 D64 3x3 (20864) 87 | 90 (242 | 246 / 462 | 471); B2 H16 S3072 D128 6x11 (21376) 133 | 136 (332 | 331 /
// 536 | 545); B2 H16 S4096 D128 6x11 (38208) 225 | 236 (538 | 546 / 887 | 898).
inline qk_chunks qk_chunk_rule(int64_t blocks, int64_t head_blocks, int nqb)
{
    if (blocks >= 16000) return {48, 24};
    if (blocks < 600) return {1, 1};
    int small = (int)std::min<int64_t>(std::max<int64_t>((blocks + 400) / 800, 1), 8);
    while (head_blocks / small + 2 * nqb > ITEM_TABLE_MAX && small < 24) small *= 2;   // (the table holds one head's items)
    return {2 * small, small};
}
constexpr int F_SLD = 80;  // score-tile row stride (elements): exactly the retained columns + one key block.  A wider
                           // row costs the scores-only kernel its third workgroup per CU, and with this one a fragment
                           // read (16 consecutive rows x 64 bytes) is free of bank conflicts as it is: the LDS serves
                           // lanes 0-7 together with lanes 24-31 (8-15 with 16-23, ...), and rows 160 bytes apart put
                           // those on the even and the odd 16-byte positions (measured; 144 or 176 bytes halve the rate)

// LDS accesses issued from assembly: the compiler neither reorders them nor waits for the asynchronous copy in flight
// ahead of them (it cannot tell a read of the score tile from the copy's target), and the wait points are placed by
// hand.  LDS operations of a wavefront complete in order, so "at most n operations outstanding" names the oldest ones
// as complete; a loaded value is tied to the wait that covers it through an in/out operand.
__device__ __forceinline__ unsigned lds_addr(const void *p) { return (unsigned)(uintptr_t)(lds_void_t *)p; }
__device__ __forceinline__ u32x4_t lds_read16_at(unsigned addr, int off)
{
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
__device__ __forceinline__ void lds_write8_at(unsigned addr, int off, uint32_t lo, uint32_t hi)
{
    const u32x2_t v = {lo, hi};
    asm volatile("ds_write_b64 %0, %1 offset:%2" : : "v"(addr), "v"(v), "n"(off) : "memory");
}
__device__ __forceinline__ void lds_write16_at(unsigned addr, int off, u32x4_t v)
{
    asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(addr), "v"(v), "n"(off) : "memory");
}
// the transpose read of 8 bytes
__device__ __forceinline__ u32x2_t lds_read_tr8_at(unsigned addr, int off)
{
    u32x2_t v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
template <int N> __device__ __forceinline__ void lds_wait_upto(u32x4_t &v)
{
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(v) : "n"(N) : "memory");
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>), in order
template <int... I, typename F> __device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}
// The scores-only kernel writes the scores of 16-key blocks cb-1 and cb (cb odd, both row blocks: two writes) right
// after step (cb+1)*KS + LAG - 1 of its score phase; the last pair after the loop.  Number of those writes issued at the
// end of a step in [lo, hi).
constexpr int score_writes_between(int lo, int hi, int KS, int NCB, int LAG, int RB)
{
    int c = 0;
    for (int cb = 1; cb + 1 < NCB; cb += 2) {
        const int s = (cb + 1) * KS + LAG - 1;
        if (s >= lo && s < hi) c += RB;
    }
    return c;
}

// a.lo*b.lo + a.hi*b.hi + c for two packed pairs of the 16-bit type T, accumulated in fp32
template <typename T> __device__ __forceinline__ float dot2_io(uint32_t a, uint32_t b, float c)
{
    if constexpr (std::is_same<T, bf16_t>::value) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(mta_bf16x2, a), __builtin_bit_cast(mta_bf16x2, b), c, false);
    } else {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(mta_f16x2, a), __builtin_bit_cast(mta_f16x2, b), c, false);
    }
}

// max / sum over the four lane groups (lanes l, l^16, l^32, l^48) that share a query row, in every lane: two
// exchanges between whole rows of lanes on the vector ALU (no LDS permute, so the LDS counter stays ours to count)
__device__ __forceinline__ float max_across_groups(float v)
{
    u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_across_groups(float v)
{
    u32x2_t r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// A tap of the attention kernel, whose softmax takes maxima ahead of the factor and therefore a factor > 0: the tap carries its
// sign (an exact change of the sign bit), and for 0 its value.
template <typename T> __device__ __forceinline__ T signed_tap(T w, float scale)
{
    uint16_t b = __builtin_bit_cast(uint16_t, w);
    if (scale < 0.0f) b ^= 0x8000u;
    if (scale == 0.0f) return from_float<T>(to_float(w) * 0.0f);
    return __builtin_bit_cast(T, b);
}

// Inside a rarely taken, wavefront-uniform `if`: keeps it a branch.  Without it the compiler turns the masks of the
// diagonal key blocks into selects that every key block executes (a third of the attention kernel's vector
// instructions).
#define MTA_KEEP_BRANCH() asm volatile("" ::: "memory")

// Returns its argument, opaquely: what is derived from the result cannot be hoisted out of the block that computes it.
__device__ __forceinline__ int opaque_lane(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

// Swizzle of a V block for the attention kernel's transpose reads, whose 16-lane groups are 4 keys apart (keys
// 4kg + 0..3): the 8 consecutive keys that may be served in one cycle must land in 8 different 8-bank regions.
// D = 128: region = chunk pair ^ key%8.  D = 64 (a row is half the banks, odd keys take the other half):
// region = chunk pair ^ (key/2)%4.
template <int D> __device__ __forceinline__ int v_swizzle4(int key)
{
    if constexpr (D == 128) return 2 * (key & 7);
    else return 2 * ((key >> 1) & 3);
}

template <int R, int SK> struct fused_geom {
    static constexpr int F_SR = 128;
    static constexpr int HR = (R - 1 + 7) & ~7;    // halo rows above the block (recomputed)
    static constexpr int HC = (SK - 1 + 7) & ~7;   // score columns kept from the previous key block
    static constexpr int BQ = F_SR - HR;           // output rows per workgroup
    static constexpr int PW = (SK - 1) / 2, PWR = SK - 1 - PW;
    static constexpr int SHIFT = HC - (SK - 1);    // first tap's offset in a block's 32-key window
    static constexpr bool fits = SHIFT + 16 + SK - 1 <= 32 && HC + F_BK <= 80;
    static constexpr int WZ_OFF = SHIFT + 16, WZ_LD = WZ_OFF + 32;
};

// A head's work items (query block, range of key blocks) in the order they are to be started: longest first, so that the
// long items all start early and the short ones fill the end of the grid.  Built on the host for every launch (a
// counting sort over at most ITEM_TABLE_MAX items) and passed by value as a kernel argument; n = 0: no table, the kernel
// cuts every query block's key range into chunks of jc_len blocks and walks the query blocks from the last to the first.
// The chunks need not be equal: the first part of a query block's key range goes into long items (one extra key block
// per item rebuilds the retained score columns, and an item costs a few microseconds to set up), the rest into short
// ones, which are started last and even out the end of the grid.
struct item_table {
    int n;
    uint32_t e[ITEM_TABLE_MAX];  // query block (11 bits) | first key block << 11 (11 bits) | key blocks << 22
};

// RAW (scores only, a 1x1 kernel): no conv at all - round(round(Q K^T) * scale) goes from the accumulators to memory: the
// plain lower-triangle product of the training route (raw scores, dP = dO V^T).  No score tile, no retained columns, no halo.
// SCORES_ONLY: stop after the conv and write  conv(mask0(scale * Q K^T))  as an (S,S) plane per (batch, head)
// (`O` is then the score tensor, V is unused).  Only q <= p is written when causal, plus +0 above the
// diagonal when `fill_upper` is set.
// BAND (scores-only kernel): a mask of the form "key k of query row p is visible iff band_lo[b, p] <= k <= p" - the
// scores of the hidden keys enter the conv as 0, as the reference's masked_fill ahead of its conv leaves them
// (mta_attention_triton.py:70-73).
template <typename T, int D, int R, int SK, bool SCORES_ONLY, int NW, bool BAND>
__global__ __launch_bounds__(64 * NW, SCORES_ONLY ? ((R > 7 || (BAND && R >= 7)) ? 2 : QK_OCC) : 2) void conv_attn_fwd_mfma(const T *__restrict__ Q, const T *__restrict__ K,
                                                             const T *__restrict__ V, const T *__restrict__ Wt,
                                                             T *__restrict__ O, float *__restrict__ Lse, int S, int causal,
                                                             float scale, int H, int nqb, int fill_upper, unsigned total_wg,
                                                             unsigned heads, unsigned per_xcd, int jc_len,
                                                             item_table tbl, const int *__restrict__ band_lo, int tri_gl, row_strides qs)
{
    static_assert(!BAND || SCORES_ONLY, "the band mask belongs to the scores-only kernel");
    using G = fused_geom<R, SK>;
    constexpr bool RAW = SCORES_ONLY && R == 1 && SK == 1;
    constexpr int F_NT = 64 * NW, F_SR = 128, RB = F_SR / (16 * NW);   // (RB: blocks of 16 rows per wavefront)
    static_assert(RB == 2 || (RB == 1 && !SCORES_ONLY), "the scores-only kernel is written for two");
    constexpr int CPR = D / 8;                     // 16-byte chunks per K/V row
    constexpr int TILE = F_BK * D;                 // elements per K or V block
    constexpr int ROUNDS = TILE / 8 / F_NT;        // copy instructions per block per lane
    constexpr int KS = D / 32;                     // contraction steps over the head dim
    constexpr int DB = D / 16;                     // 16-wide blocks of the head dim
    constexpr int NCB = F_BK / 16;                 // 16-key blocks per iteration
    static_assert(ROUNDS >= 1, "block smaller than one copy round");

    // The scores-only kernel double-buffers K in B0 / B1, arrays of their own with a loop body each: the compiler then sees that LDS
    // reads never touch the asynchronous copy in flight into the other one.  The attention kernel rotates K and V through the
    // three buffers of KV: in an iteration K(j) sits in one, V(j) in another; K(j+1) is copied into the third from the top of the
    // iteration on, and V(j+1) into K(j)'s buffer once the score phase is over (the barrier in the middle of the iteration).
    // Three 16 KB buffers and the score tile are 68 KB: two workgroups per CU.
    __shared__ __align__(16) T B0[SCORES_ONLY ? TILE : 8];
    __shared__ __align__(16) T B1[SCORES_ONLY ? TILE : 8];
    __shared__ __align__(256) T KV[SCORES_ONLY ? 8 : 3 * TILE];
    __shared__ __align__(16) T Sc[RAW ? 8 : F_SR * F_SLD];                // score tile
    // zero-padded kernel rows, only needed until the Toeplitz fragments are built: they borrow a buffer that
    // receives its first copy after that (LDS is granted in 1280-byte units; the array's own 648 bytes were the
    // difference between two and three workgroups per CU for the scores-only kernel)
    static_assert(R * G::WZ_LD <= TILE, "kernel rows do not fit the borrowed buffer");
    T *const wz = SCORES_ONLY ? B1 : KV + 2 * TILE;

    const int tid = threadIdx.x;
    // (the wavefront index through readfirstlane: everything derived from it is then scalar, branches included)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // The items are taken rank by rank - the longest item of every head, then the second longest of each, ... - so that the long items
    // all start early and the short ones fill the end of the grid (workgroups start in index order as slots free up).
    // Workgroup ids are dealt round-robin to the 8 XCDs: with heads in multiples of 8 an XCD keeps its own, whose K and V stay in its L2
    // (of 12 heads an XCD sees 3, of 4 one).  With other numbers of heads an XCD used to take an eighth of the list head by head - of 4
    // heads one XCD a head's long items and another its short ones.  us, that -> this, bf16 6x11, scores | attention: B1 H4 S3008 D128
    // 26.5 -> 24.1 | 117 -> 117, B1 H12 S2048 D64 33.7 -> 27.7 | 66.7 -> 67.2, S3712 D64 76.3 -> 67.5 | 152 -> 122, S4096 D128 101 -> 93 | 210 -> 170,
    // B1 H20 S2048 D128 53.2 -> 45.8 | 106 -> 88.6; without a conv B1 H12 S2048 D64 16.9 -> 14.4, S2560 23.8 -> 20.1.  per_xcd: the old deal, see
    // launch_mfma.
    // Work item = (batch*head, query block, chunk of jc_len key blocks).  The scores-only kernel splits the key
    // range of a query block (its output columns are independent; a chunk starts one key block early to rebuild
    // the retained halo columns), so that items are short and equal and the grid runs in several even rounds;
    // the attention kernel accumulates over all keys and gets jc_len = all of them.
    // (a 32-bit division: the 64-bit ones that this took were half a microsecond of a workgroup's start)
    unsigned id = blockIdx.x;
    if (RAW && per_xcd) id = (id & 7) * per_xcd + (id >> 3);
    if (id >= total_wg) return;
    int item = (int)(id / heads), bh = (int)(id - (unsigned)item * heads);
    if (RAW && per_xcd) {
        const unsigned items = total_wg / heads;
        bh = (int)(id / items);
        item = (int)(id - (unsigned)bh * items);
    }
    int qb = nqb - 1, jc = 0;
    int tbl_lo = -1, tbl_len = 0;
    if (tbl.n > 0) {
        const unsigned e = tbl.e[item];
        qb = (int)(e & 2047u);
        tbl_lo = (int)((e >> 11) & 2047u);
        tbl_len = (int)(e >> 22);
    } else {
        for (; qb > 0; --qb) {  // longest query blocks first
            const int ql = (qb * G::BQ + G::BQ - 1 < S - 1) ? qb * G::BQ + G::BQ - 1 : S - 1;
            const int nch = ((causal ? ql / F_BK : (S - 1) / F_BK) + jc_len) / jc_len;
            if (item < nch) break;
            item -= nch;
        }
        jc = item;
    }
    const int head = (int)((unsigned)bh % (unsigned)H);
    const int q0 = qb * G::BQ;
    const bool q_strided = RAW && qs.row != 0;
    const T *Qp = Q + (q_strided ? (int64_t)(bh / H) * qs.batch + head * qs.head : (int64_t)bh * S * D);
    const int64_t q_row = q_strided ? qs.row : D;
    const T *Kp = K + (int64_t)bh * S * D;
    const T *Vp = SCORES_ONLY ? Kp : V + (int64_t)bh * S * D;
    // (scores only, tri_gl > 0: the scores go out in the triangular layout, groups of tri_gl heads interleaved by rows;
    // nothing above the diagonal is stored then)
    const bool tri = SCORES_ONLY && tri_gl > 0;
    T *Op = tri ? O + ((unsigned)bh / (unsigned)(tri ? tri_gl : 1)) * ((tri ? tri_gl : 1) * tri_rowoff(S)) : O + (int64_t)bh * S * (SCORES_ONLY ? S : D);
    const int tri_i = tri ? (int)((unsigned)bh % (unsigned)tri_gl) : 0;

    // asynchronous copy of key block j into buffer `buf`: K rows cb.., V rows j*BK..; out-of-range keys
    // re-read a valid row (their scores are zeroed / their probabilities are 0 later)
    // slot r*512+tid of a block is row kv_row[r], 16-byte chunk kv_c of that row (fixed per lane)
    // (a round advances the row by F_NT/CPR, a multiple of CPR: the swizzled chunk is the same in every round)
    static_assert((F_NT / CPR) % CPR == 0 && F_NT % CPR == 0, "copy rounds must keep the swizzle phase");
    const int kv_row0 = tid / CPR;
    const int kv_off0 = kv_row0 * D + ((tid % CPR) ^ (kv_row0 & (CPR - 1))) * 8;
    // V blocks use the swizzle that keeps the transpose reads free of bank conflicts (it only depends on key bits
    // below 4, which a copy round does not change either)
    static_assert((F_NT / CPR) % 16 == 0, "copy rounds must keep the V swizzle phase");
    const int v_off0 = kv_row0 * D + ((tid % CPR) ^ v_swizzle4<D>(kv_row0)) * 8;
    auto issue_k = [&](int j, T *Kdst) {
        const int cb = j * F_BK + G::PWR;
        const bool inside = cb >= 0 && cb + F_BK <= S;  // no key needs clamping
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int kv_row = kv_row0 + r * (F_NT / CPR), kv_off = kv_off0 + r * (F_NT / CPR) * D;
            int koff = cb * D + kv_off;
            if (!inside) {
                int kr = cb + kv_row;
                kr = kr < 0 ? 0 : (kr >= S ? S - 1 : kr);
                koff = kv_off + (kr - kv_row) * D;
            }
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Kp + koff),
                                             (lds_void_t *)(Kdst + (r * F_NT + wave * 64) * 8), 16, 0, 0);
        }
    };
    auto issue_v = [&](int j, T *Vdst) {
        const bool inside = j >= 0 && (j + 1) * F_BK <= S;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int kv_row = kv_row0 + r * (F_NT / CPR), v_off = v_off0 + r * (F_NT / CPR) * D;
            int voff = j * F_BK * D + v_off;
            if (!inside) {
                int vr = j * F_BK + kv_row;
                vr = vr < 0 ? 0 : (vr >= S ? S - 1 : vr);
                voff = v_off + (vr - kv_row) * D;
            }
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Vp + voff),
                                             (lds_void_t *)(Vdst + (r * F_NT + wave * 64) * 8), 16, 0, 0);
        }
    };

    const int q_last = (q0 + G::BQ - 1 < S - 1) ? q0 + G::BQ - 1 : S - 1;
    const int j_last = causal ? q_last / F_BK : (S - 1) / F_BK;  // last key block of the query block
    int j_lo = tbl_lo >= 0 ? tbl_lo : jc * jc_len;                // first key block whose outputs this item produces
    const int j_len = tbl_lo >= 0 ? tbl_len : jc_len;
    const int j_end = (j_lo + j_len - 1 < j_last) ? j_lo + j_len - 1 : j_last;
    if constexpr (BAND) {
        // Key blocks that lie wholly ahead of the first key any row of this query block sees are skipped: no visible
        // position takes a tap from them, and what they would hold is hidden from every row (left unwritten).  Every
        // wavefront reduces all the rows (the same answer in each: no exchange).
        const int64_t brow = (bh / H) * (int64_t)S;
        int fmin = S;
        for (int r = lane; r < G::BQ + G::HR; r += 64) {
            const int p = q0 - G::HR + r;
            if (p >= 0 && p < S) {
                const int f = band_lo[brow + p];
                fmin = f < fmin ? f : fmin;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(fmin, off);
            fmin = o < fmin ? o : fmin;
        }
        fmin = __builtin_amdgcn_readfirstlane(fmin);
        const int j_first = (fmin > 0 ? fmin : 0) / F_BK;
        if (j_first > j_lo) j_lo = j_first;
        if (j_lo > j_end) return;
    }
    // one key block earlier only fills the retained score columns (before the first one: the right pad, if any)
    const int j_start = RAW ? j_lo : j_lo > 0 ? j_lo - 1 : (G::PWR > 0 ? -1 : 0);
    // What the start waits for is asked for at once, this wavefront's rows of Q and the kernel's taps ahead of the first blocks of K and V:
    // behind them, the taps waited for the blocks and Q was asked for when those had come.  With the 32-bit divisions above, scores
    // kernel, us: bf16 6x11 B2 H16 S1008 D64 22.3 -> 21.1, B4 H16 S1024 D128 40.6 -> 40.1, 7x7 B1 H16 S1024 D64 18.6 -> 17.7, B1 H16 S2048 D128 42.1 ->
    // 40.9, 6x11 B2 H16 S2048 D128 69.7 -> 67.5, S4096 240 -> 236, 11x15 B2 H16 S640 D128 21.1 -> 19.8.
    int trow[RB], prow[RB];   // this lane's query rows
    frag8<T> qf[RB][KS];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        trow[rb] = wave * (16 * RB) + rb * 16 + ln;
        prow[rb] = q0 - G::HR + trow[rb];
        const int pc = prow[rb] < 0 ? 0 : (prow[rb] >= S ? S - 1 : prow[rb]);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[rb][ks] = *reinterpret_cast<const frag8<T> *>(Qp + pc * q_row + ks * 32 + kg * 8);
    }
    constexpr int WZ_IT = (R * G::WZ_LD + F_NT - 1) / F_NT;
    T taps[RAW ? 1 : WZ_IT];
    if constexpr (!RAW) {
#pragma unroll
        for (int n = 0; n < WZ_IT; ++n) {
            const int e = n * F_NT + tid, i = e / G::WZ_LD, jj = e % G::WZ_LD - G::WZ_OFF;
            taps[n] = Wt[head * R * SK + (i < R && jj >= 0 && jj < SK ? i * SK + jj : 0)];
        }
    }
    asm volatile("" : : : "memory");
    issue_k(j_start, SCORES_ONLY ? B0 : KV);
    if (!SCORES_ONLY) issue_v(j_start, KV + TILE);

    if constexpr (!RAW) {
    // zero the score tile once (columns past HC+BK are read by the last window but never written)
    for (int e = tid; e < F_SR * F_SLD / 8; e += F_NT) {
        pack16<T> z;
#pragma unroll
        for (int u = 0; u < 8; ++u) z.v[u] = from_float<T>(0.0f);
        *reinterpret_cast<pack16<T> *>(Sc + e * 8) = z;
    }
#pragma unroll
    for (int n = 0; n < WZ_IT; ++n) {
        const int e = n * F_NT + tid, jj = e % G::WZ_LD - G::WZ_OFF;
        if (e < R * G::WZ_LD) wz[e] = jj >= 0 && jj < SK ? signed_tap<T>(taps[n], SCORES_ONLY ? 1.0f : scale) : from_float<T>(0.0f);
    }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (prow[rb] < 0 || prow[rb] >= S) qf[rb][ks] = zero_frag<T>();  // rows outside the sequence are conv padding
    // band mask: first visible key of this lane's two rows, and the largest of them over the wavefront's 32 rows (a key
    // block that starts at or beyond it is visible to all of them)
    int flo[2] = {0, 0}, fmax_w = 0;   // (scores only: two row blocks)
    if constexpr (BAND) {
        const int64_t brow = (bh / H) * (int64_t)S;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) flo[rb] = (prow[rb] >= 0 && prow[rb] < S) ? band_lo[brow + prow[rb]] : 0;
        int m = flo[0] > flo[1] ? flo[0] : flo[1];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(m, off);
            m = o > m ? o : m;
        }
        fmax_w = __builtin_amdgcn_readfirstlane(m);
    }
    __syncthreads();

    // Toeplitz fragments T_i^T: accumulator row m = ln, slots k = 8*kg + t, tap = k - SHIFT - m
    frag8<T> tz[R];
#pragma unroll
    for (int i = 0; i < (RAW ? 0 : R); ++i) {
        const T *src = wz + i * G::WZ_LD + G::WZ_OFF + kg * 8 - G::SHIFT - ln;
#pragma unroll
        for (int t = 0; t < 8; ++t) tz[i].v[t] = src[t];
    }

    f32x4 oacc[RB][DB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m_i[RB], l_i[RB];   // (maxima of the conv's results, ahead of the factor)
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        m_i[rb] = -INFINITY;
        l_i[rb] = 0.0f;
    }
    const float scale_abs = scale == 0.0f ? 1.0f : fabsf(scale), scale2 = scale_abs * 1.4426950408889634f;

    // retained columns: each thread moves one 16-byte vector per round (HC/8 vectors per row)
    constexpr int TAIL_VECS = F_SR * (G::HC / 8);
    constexpr int TAIL_IT = (TAIL_VECS + F_NT - 1) / F_NT;

    int tail_off[TAIL_IT > 0 ? TAIL_IT : 1];  // element offset of this thread's retained vector(s) in the tile's head
#pragma unroll
    for (int it = 0; it < TAIL_IT; ++it) {
        constexpr int VPRW = G::HC / 8 > 0 ? G::HC / 8 : 1;
        const int idx = it * F_NT + tid;
        tail_off[it] = idx < TAIL_VECS ? (idx / VPRW) * F_SLD + (idx % VPRW) * 8 : -1;
    }
    // the 16-row blocks of this wavefront span rows pmin .. pmin + 16 RB - 1 of the sequence
    const int pmin = q0 - G::HR + wave * (16 * RB);
    // Rows of the conv (and of everything after it: softmax, P V, the stores).  The first wavefront's rows are taken
    // R-1 further down than the rows it computes scores for: its conv windows then start at tile row 0 instead of
    // above the tile, every fragment address is the same affine function of (row block, kernel row), and what it
    // leaves out are halo rows nobody stores.  Its last R-1 rows belong to the second wavefront too and are not
    // stored from here.
    const int cshift = wave == 0 ? R - 1 : 0;
    int cprow[RB];
    bool row_stored[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const int tr_ = trow[rb] + cshift;
        cprow[rb] = prow[rb] + cshift;
        row_stored[rb] = tr_ >= G::HR && tr_ < (wave + 1) * (16 * RB) && cprow[rb] < S;
    }

    auto plain = [&](int j) {
        const int cbase = j * F_BK + G::PWR;
        return j >= 0 && cbase + F_BK <= S && (!causal || cbase + F_BK - 1 <= pmin) && (!BAND || cbase >= fmax_w);
    };
    // PLAIN: the key block (its scores and its conv outputs) lies inside the sequence and on or below the diagonal
    // for all 32 rows of this wavefront: no masks and no per-sub-block tests (most blocks of a long sequence)
    auto block = [&](auto plain_tag, int j, const T *Kb, const T *Vb, T *Kn, T *Vn) __attribute__((always_inline)) {
        constexpr bool PLAIN = decltype(plain_tag)::value;
        const int cbase = j * F_BK + G::PWR;  // first key of the new score block
        const bool whole = PLAIN || (!SCORES_ONLY && plain(j));   // (the attention kernel has one body, with a branch around its masks)
        // (a vector type, read by every lane: a struct read under a lane condition travels through scratch memory)
        u32x4_t tailreg[TAIL_IT > 0 ? TAIL_IT : 1];
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it)
            tailreg[it] = *reinterpret_cast<const u32x4_t *>(Sc + (tail_off[it] >= 0 ? tail_off[it] : 0) + F_BK);
        __builtin_amdgcn_s_waitcnt(0);  // this wavefront's part of block j has landed in LDS
        __syncthreads();                // ... and everybody's; all reads of the previous tiles are done
        // (Leaving the previous iteration's result stores in flight here - vmcnt(number of stores) instead of 0 - was
        // measured: no gain.)
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it)
            if (tail_off[it] >= 0) *reinterpret_cast<u32x4_t *>(Sc + tail_off[it]) = tailreg[it];
        if (j < j_end) issue_k(j + 1, Kn);  // lands while this block is being worked on

        // ---- S^T = K Q^T, zero above the diagonal / outside the sequence, to the score tile ----
        {
            // Pipelined like the conv phase below: K fragments are read from assembly KLD steps (one or two 16-key
            // blocks) ahead into a ring of registers, a step being one fragment and the two products it feeds (both row
            // blocks); a block's scores are rounded, scaled, masked and written LAG steps into the next block.
            constexpr int NSTEP = NCB * KS, KLD = SCORES_ONLY ? 2 * KS : KS, KSLOT = KLD + 1, LAG = 2;  // (attention kernel: one block ahead; two spill)
            static_assert(NSTEP > KLD && KS >= LAG && NCB % 2 == 0, "pipeline deeper than the work; blocks are written in pairs");
            unsigned ka[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                ka[ks] = lds_addr(Kb) + (unsigned)((ln * D + (((ks * 4 + kg) ^ (ln & (CPR - 1))) * 8)) * (int)sizeof(T));
            const unsigned wa = lds_addr(Sc) + (unsigned)((trow[0] * F_SLD + G::HC + (kg & 1) * 16 + (kg >> 1) * 8) * (int)sizeof(T));
            u32x4_t kring[KSLOT];
            f32x4 sacc[2][RB];
            uint32_t held[RB][2];
            auto kissue = [&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value;
                kring[n % KSLOT] = lds_read16_at(ka[n % KS], (n / KS) * 16 * D * (int)sizeof(T));
            };
            auto epilogue = [&](auto cbc) __attribute__((always_inline)) {
                constexpr int cb = decltype(cbc)::value;
                // key block wholly inside the sequence and on or below the diagonal for all 32 rows: no masks
                const bool s_plain = PLAIN || !SCORES_ONLY ? PLAIN || whole : (cbase + cb * 16 >= 0 && cbase + cb * 16 + 16 <= S && (!causal || cbase + cb * 16 + 15 <= pmin) &&
                                               (!BAND || cbase + cb * 16 >= fmax_w));
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const f32x4 a = sacc[cb & 1][rb];
                    uint32_t lo = pack2<T>(a[0], a[1]), hi = pack2<T>(a[2], a[3]);
                    if (SCORES_ONLY) {  // MTA scales the scores before the conv, in the I/O dtype: round, scale, round again
                        float a0, a1, a2, a3;
                        unpack2<T>(lo, a0, a1);
                        unpack2<T>(hi, a2, a3);
                        lo = pack2<T>(a0 * scale, a1 * scale);
                        hi = pack2<T>(a2 * scale, a3 * scale);
                    }
                    if (!s_plain) {
                        MTA_KEEP_BRANCH();
                        const int col = cbase + cb * 16 + kg * 4;
                        const int lim = causal ? (prow[rb] < S - 1 ? prow[rb] : S - 1) : S - 1;  // last key kept
                        const int first = BAND ? (flo[rb] > 0 ? flo[rb] : 0) : 0;  // first key kept
                        if (col < first || col > lim) lo &= 0xffff0000u;
                        if (col + 1 < first || col + 1 > lim) lo &= 0x0000ffffu;
                        if (col + 2 < first || col + 2 > lim) hi &= 0xffff0000u;
                        if (col + 3 < first || col + 3 > lim) hi &= 0x0000ffffu;
                    }
                    // Two 16-key blocks go to the tile together.  A lane holds keys 4kg..4kg+3 of each; after the
                    // exchange between neighbouring lane groups (even groups give their second block's part and take
                    // the neighbour's first block's part) it holds 8 consecutive keys of one block: one 16-byte write
                    // per lane and block pair instead of two 8-byte ones, which conflicted four ways in the banks.
                    if constexpr ((cb & 1) == 0) {
                        held[rb][0] = lo;
                        held[rb][1] = hi;
                    } else {
                        const u32x2_t s0 = __builtin_amdgcn_permlane16_swap(held[rb][0], lo, false, false);
                        const u32x2_t s1 = __builtin_amdgcn_permlane16_swap(held[rb][1], hi, false, false);
                        if constexpr (RAW) {
                            const int kg_o = opaque_lane(kg);
                            const int col = cbase + (cb - 1 + (kg_o & 1)) * 16 + (kg_o >> 1) * 8, p_ = prow[rb];
                            if (p_ < S && (PLAIN || (col < S && (!causal || fill_upper || col <= p_))))
                                *reinterpret_cast<u32x4_t *>(Op + (int64_t)p_ * S + col) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
                        } else
                        lds_write16_at(wa, (rb * 16 * F_SLD + (cb - 1) * 16) * (int)sizeof(T), u32x4_t{s0[0], s1[0], s0[1], s1[1]});
                    }
                }
            };
            static_for<KLD>(kissue);
            static_for<NSTEP>([&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value;
                constexpr int cb = n / KS, ks = n % KS;
                if constexpr (n + KLD < NSTEP) kissue(std::integral_constant<int, n + KLD>{});
                // LDS operations younger than read n: the reads issued after it and the score writes issued since
                constexpr int younger = (n + KLD < NSTEP ? n + KLD : NSTEP - 1) - n + (RAW ? 0 : score_writes_between(n > KLD ? n - KLD : 0, n, KS, NCB, LAG, RB));
                lds_wait_upto<(younger < 15 ? younger : 15)>(kring[n % KSLOT]);
                if constexpr (ks == 0) {
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb) sacc[cb & 1][rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) mma16(sacc[cb & 1][rb], __builtin_bit_cast(frag8<T>, kring[n % KSLOT]), qf[rb][ks]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (cb >= 1 && ks == LAG - 1) {
                    epilogue(std::integral_constant<int, cb - 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
            epilogue(std::integral_constant<int, NCB - 1>{});
        }
        if constexpr (RAW) return;
        else {
        // score tile complete for everybody.  Only the LDS counter is waited for: a fence would also wait for the
        // copy of the next key block, in flight since the top of the iteration
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // (attention kernel: nobody reads K(j) any more, the next V block may land in its buffer)
        if (!SCORES_ONLY && j < j_end) issue_v(j + 1, Vn);
        if (j < j_lo) return;

        // ---- conv (Toeplitz MFMAs over the score tile) -> global (scores only) / -> online softmax ----
        // One product needs one fresh 1 KB score fragment from LDS, and a wavefront that waits for each fragment
        // where it is used spends four times the products' own time here.  The reads are therefore issued NLD
        // products ahead, from assembly (see lds_read16_at), into a ring of registers; every product is preceded by
        // a wait that leaves exactly the younger operations outstanding.  The R products of one output block add into the same
        // registers, each waiting for the one before; with TURNS = 2 two neighbouring blocks are worked on in turns, which gives the
        // scores kernels up to 1.5 % (1 | 2, us: bf16 6x11 B1 H16 S2048 D64 34.3 | 33.9, B4 H16 S1024 D128 39.8 | 39.3, fp16 7x7 B1 H16
        // S2048 D128 41.6 | 41.2) and the attention kernel nothing (bf16 6x11 B1 H32 S8192 D128 986 | 994, D64 B1 H8 S2048 66.7 | 67.2, fp16
        // 7x9 D64 B4 H12 93.6 | 93.5, 11x15 D128 B1 H32 S4096 362 | 359).  A block's results are taken up LAG products into the next turn,
        // when they are long complete.
        constexpr int TURNS = SCORES_ONLY ? 2 : 1;
        constexpr int NB = RB * NCB, NREAD = NB * R;
        // score fragments in flight (scores only: 8 and 12 measure the same, 15 spills; attention: 4 and 8 the same, and 8 with 7 kernel
        // rows at D = 64 takes the third workgroup of a CU: fp16 7x9 B4 H12 S2048 92.7 | 105.4 us)
        constexpr int NLD = SCORES_ONLY ? 8 : 4;
        constexpr int NSLOT = NLD + 1;
        constexpr int LAG = 2;
        static_assert(NREAD > NLD && R >= LAG && NLD <= 15, "pipeline deeper than the work or than the counter");
        const unsigned xa = lds_addr(Sc) + (unsigned)(((trow[0] + cshift - (R - 1)) * F_SLD + kg * 8) * (int)sizeof(T));
        u32x4_t ring[NSLOT];
        f32x4 cacc[2 * TURNS];
        auto issue = [&](auto ic) __attribute__((always_inline)) {
            constexpr int n = decltype(ic)::value;
            constexpr int blk = n / (TURNS * R) * TURNS + n % TURNS, i = n % (TURNS * R) / TURNS;   // output block, kernel row
            ring[n % NSLOT] = lds_read16_at(xa, (((blk / NCB) * 16 + i) * F_SLD + (blk % NCB) * 16) * (int)sizeof(T));
        };
        // what happens to output block b = rb*NCB + cb (rows crow[rb], keys j*64 + 16cb ..) once it is complete
        uint32_t held[2];           // scores only: the even block of a pair, packed
        float sv[RB][NCB][4], mloc, mneg[RB];   // attention: a row block's logits, their maximum; minus the running maximum as the exponent takes it
        frag8<T> pf[RB][2];         // attention: probabilities, in the operand layout of the P V products
        auto finish = [&](auto bc) __attribute__((always_inline)) {
            constexpr int b = decltype(bc)::value;
            constexpr int rb = b / NCB, cb = b % NCB;
            const f32x4 a = cacc[b % (2 * TURNS)];
            const int p_ = cprow[rb];
            if constexpr (SCORES_ONLY) {
                // Blocks leave in pairs, like the scores above: after the exchange a lane holds 8 consecutive keys of
                // one of the two blocks and stores them itself, 16 rows x 64 bytes per instruction; no staging through LDS.
                // (Ordinary stores: a 128-byte line is completed by two instructions a few hundred cycles apart, and the L2
                // merges them.  Marked non-temporal, each 64-byte half went to memory on its own and the write counter
                // read 1.38 times the bytes; the price of the merge is that the scores displace some of the head's K blocks
                // from the L2 - fetches 79 -> 196 MB per launch at the benchmark shape, 825 -> 736 MB in total, 4 % faster.)
                uint32_t lo = pack2<T>(a[0], a[1]), hi = pack2<T>(a[2], a[3]);
                if (!PLAIN && causal && j * F_BK + cb * 16 + 15 > pmin) {  // block touches the diagonal for some row
                    const int col = j * F_BK + cb * 16 + kg * 4;
                    if (col > p_) lo &= 0xffff0000u;
                    if (col + 1 > p_) lo &= 0x0000ffffu;
                    if (col + 2 > p_) hi &= 0xffff0000u;
                    if (col + 3 > p_) hi &= 0x0000ffffu;
                }
                if constexpr ((cb & 1) == 0) {
                    held[0] = lo;
                    held[1] = hi;
                } else {
                    const u32x2_t s0 = __builtin_amdgcn_permlane16_swap(held[0], lo, false, false);
                    const u32x2_t s1 = __builtin_amdgcn_permlane16_swap(held[1], hi, false, false);
                    // (column from a laundered lane index: the address is then formed here, 64-bit adds and all, instead
                    // of being kept in registers across the key-block loop - the kernel is at its register limit)
                    const int kg_o = opaque_lane(kg);
                    const int col = j * F_BK + (cb - 1 + (kg_o & 1)) * 16 + (kg_o >> 1) * 8;
                    if (row_stored[rb] && (PLAIN || (col < S && (!causal || fill_upper || col <= p_)))) {
                        // (triangular layout: the row's start from a laundered row number, for the same reason)
                        T *dst = tri ? Op + (tri_row_start(opaque_lane(p_), tri_gl, tri_i) + (unsigned)col) : Op + (int64_t)p_ * S + col;
                        *reinterpret_cast<u32x4_t *>(dst) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
                    }
                }
            } else {
                // (fp32 from here to the probabilities: the factor goes into the exponential's multiply-add)
                float v4[4] = {a[0], a[1], a[2], a[3]};
                if (!whole) {
                    MTA_KEEP_BRANCH();
                    // (the column from a laundered lane index: formed here, not by every key block)
                    const int left = (causal ? (p_ < S - 1 ? p_ : S - 1) : S - 1) - (j * F_BK + cb * 16) - opaque_lane(kg) * 4;
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (v > left) v4[v] = -INFINITY;
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) sv[rb][cb][v] = v4[v];
                const float m4 = fmaxf(fmaxf(v4[0], v4[1]), v4[2]);
                mloc = cb == 0 ? fmaxf(m4, v4[3]) : fmaxf(fmaxf(mloc, m4), v4[3]);
                if constexpr (cb == NCB - 1) {  // the row block is complete: its running maximum (a row lives in 4 lanes)
                    const float m_new = fmaxf(m_i[rb], max_across_groups(mloc));
                    const float m_use = (m_new == -INFINITY) ? 0.0f : m_new;
                    // exp(scale*(x - m)) = exp2(x*scale*log2(e) - m*scale*log2(e)): one multiply-add and one v_exp per element
                    mneg[rb] = -m_use * scale2;
                    // Where no row's maximum has moved (most key blocks, once the maxima have settled) the 4*DB multiplications are skipped.
                    // The factor of a row whose maximum stays is 1 by that, not by its exponent: mneg is rounded, and the sums would drift
                    // by that rounding at every key block (0.5 % of a row of 8192 keys at logits of 772) and be multiplied at nearly every one.
                    // us: 6x11 B1 H32 S8192 D128 1007 -> 989, 5x5 B2 H32 S4096 D64 354 -> 345, 3x3 B1 H32 S4096 D128 244 -> 240.
                    if (__builtin_amdgcn_ballot_w64(m_new != m_i[rb]) != 0) {
                        const float alpha = m_new != m_i[rb] ? __builtin_amdgcn_exp2f(fmaf(m_i[rb], scale2, mneg[rb])) : 1.0f;
                        l_i[rb] *= alpha;
#pragma unroll
                        for (int db = 0; db < DB; ++db) oacc[rb][db] *= alpha;
                    }
                    m_i[rb] = m_new;
                }
            }
        };
        // two of a row block's probabilities: keys 16*(h/2) + 4*kg + 2*(h%2), + 1.  The row sum runs over the rounded ones (what
        // the P V products see): a packed dot product with (1, 1).  The empty statements keep the work where it is written,
        // among the matrix products; the compiler moves it down to where the probabilities are used.
        auto probs = [&](auto rbc, auto hc) __attribute__((always_inline)) {
            constexpr int rb = decltype(rbc)::value, h = decltype(hc)::value, c = h / 2, v = h % 2 * 2;
            const float e0 = __builtin_amdgcn_exp2f(fmaf(sv[rb][c][v], scale2, mneg[rb]));
            const float e1 = __builtin_amdgcn_exp2f(fmaf(sv[rb][c][v + 1], scale2, mneg[rb]));
            uint32_t pk = pack2<T>(e0, e1);
            l_i[rb] = dot2_io<T>(pk, pack2<T>(1.0f, 1.0f), l_i[rb]);
            asm volatile("" : "+v"(pk), "+v"(l_i[rb]));
            reinterpret_cast<uint32_t *>(&pf[rb][c >> 1])[(c & 1) * 2 + h % 2] = pk;
        };
        static_for<NLD>(issue);
        static_for<NREAD>([&](auto ic) __attribute__((always_inline)) {
            constexpr int n = decltype(ic)::value;
            constexpr int blk = n / (TURNS * R) * TURNS + n % TURNS, i = n % (TURNS * R) / TURNS;
            if constexpr (n + NLD < NREAD) issue(std::integral_constant<int, n + NLD>{});
            // LDS operations younger than read n: exactly the reads issued after it
            constexpr int younger = (n + NLD < NREAD ? n + NLD : NREAD - 1) - n;
            lds_wait_upto<younger>(ring[n % NSLOT]);
            if constexpr (i == 0) cacc[blk % (2 * TURNS)] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            mma16(cacc[blk % (2 * TURNS)], tz[i], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (blk >= TURNS && i == LAG - 1) {
                finish(std::integral_constant<int, blk - TURNS>{});
                __builtin_amdgcn_sched_barrier(0);
            }
            // the first row block's probabilities, a pair at a time among the second one's products
            if constexpr (!SCORES_ONLY && RB == 2) {
                constexpr int n0 = NREAD / 2 + TURNS * LAG - 1, every = (NREAD - 1 - n0) / 8;
                static_assert(every >= 1, "fewer products than pairs");
                if constexpr (n > n0 && (n - n0) % every == 0 && (n - n0) / every <= 8) {
                    probs(std::integral_constant<int, 0>{}, std::integral_constant<int, (n - n0) / every - 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        });
        if constexpr (SCORES_ONLY) {
            static_for<TURNS>([&](auto b) __attribute__((always_inline)) { finish(std::integral_constant<int, NB - TURNS + decltype(b)::value>{}); });
            return;
        } else {
            // ---- O^T += V^T P^T ; V^T fragments via the LDS transpose read of the row-major V block, VLD of them ahead ----
            // slots 0..3 of a fragment: keys 32ks+4kg+(0..3); slots 4..7: keys 32ks+16+4kg+(0..3) -- the order of pf.
            // A lane reads at key 4kg + ln/4 (its swizzle is the same 16 keys on) and the 16-byte chunk 2db + (ln%4)/2 of the
            // row; the swizzle and the block number db meet in address bits 5..7, which nothing else touches.
            constexpr int NV = 2 * DB, VLD = 4, VSLOT = VLD + 1;
            static_assert(NV > VLD && 2 * VLD <= 15, "pipeline deeper than the work or than the counter");
            const int key_a = kg * 4 + (ln >> 2);
            const unsigned va = lds_addr(Vb) + (unsigned)((key_a * D + v_swizzle4<D>(key_a) * 8 + ((ln & 3) >> 1) * 8 + (ln & 1) * 4) * (int)sizeof(T));
            struct { u32x2_t a, b; } vring[VSLOT];
            auto vissue = [&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value, ks = n / DB, db = n % DB;
                const unsigned at = va ^ (unsigned)(db * 32);
                vring[n % VSLOT].a = lds_read_tr8_at(at, ks * 32 * D * (int)sizeof(T));
                vring[n % VSLOT].b = lds_read_tr8_at(at, (ks * 32 + 16) * D * (int)sizeof(T));
            };
            static_for<VLD>(vissue);
            static_for<TURNS>([&](auto b) __attribute__((always_inline)) { finish(std::integral_constant<int, NB - TURNS + decltype(b)::value>{}); });
            // the last row block's probabilities: those of the first 32 keys, then the rest among the products with these
            static_for<4>([&](auto h) __attribute__((always_inline)) { probs(std::integral_constant<int, RB - 1>{}, h); });
            static_for<NV>([&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value, ks = n / DB, db = n % DB;
                if constexpr (n + VLD < NV) vissue(std::integral_constant<int, n + VLD>{});
                constexpr int younger = 2 * ((n + VLD < NV ? n + VLD : NV - 1) - n);
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(vring[n % VSLOT].a), "+v"(vring[n % VSLOT].b) : "n"(younger) : "memory");
                const frag8<T> vf = __builtin_bit_cast(frag8<T>, vring[n % VSLOT]);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) mma16(oacc[rb][db], vf, pf[rb][ks]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (ks == 0 && db % (DB / 4) == 0) {
                    probs(std::integral_constant<int, RB - 1>{}, std::integral_constant<int, 4 + db / (DB / 4)>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        }
        }
    };
    if constexpr (SCORES_ONLY) {
        for (int j = j_start;;) {  // block(tag, j, K(j), V(j), where K(j+1) goes, where V(j+1) goes)
            if (plain(j)) block(std::true_type{}, j, B0, B0, B1, B1);
            else block(std::false_type{}, j, B0, B0, B1, B1);
            if (++j > j_end) break;
            if (plain(j)) block(std::true_type{}, j, B1, B1, B0, B0);
            else block(std::false_type{}, j, B1, B1, B0, B0);
            if (++j > j_end) break;
        }
    } else {
        int kb = 0, vb = TILE, nb = 2 * TILE;   // where K(j) and V(j) are, and the third buffer
        for (int j = j_start; j <= j_end; ++j) {
            block(std::false_type{}, j, KV + kb, KV + vb, KV + nb, KV + kb);
            const int k_next = nb;
            nb = vb;
            vb = kb;
            kb = k_next;
        }
    }

    if constexpr (SCORES_ONLY) {
        // +0 for the key blocks to the right of the last one visited (all above the diagonal)
        if (causal && fill_upper && j_end == j_last) {
            pack16<T> z;
#pragma unroll
            for (int u = 0; u < 8; ++u) z.v[u] = from_float<T>(0.0f);
            const int c_first = (j_end + 1) * F_BK;
            const int vec_per_row = (S - c_first + 7) / 8;
            for (int r = wave; r < G::BQ; r += F_NT / 64) {
                const int p_ = q0 + r;
                if (p_ >= S) break;
                for (int vc = lane; vc < vec_per_row; vc += 64) {
                    const int col = c_first + vc * 8;
                    if (col < S) *reinterpret_cast<pack16<T> *>(Op + (int64_t)p_ * S + col) = z;
                }
            }
        }
        return;
    }
    // ---- normalise and store (halo rows are dropped) ----
    // (row and column from a lane index counted afresh: the store addresses are then formed here, after the key-block
    // loop, and nothing has to be kept - or spilled - across the loop for them)
    const int lane_e = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int ln_o = lane_e & 15, kg_o = lane_e >> 4;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        const float l_row = sum_across_groups(l_i[rb]);
        const int tr_ = wave * (16 * RB) + rb * 16 + ln_o + cshift, p_ = q0 - G::HR + tr_;
        if (tr_ >= G::HR && tr_ < (wave + 1) * (16 * RB) && p_ < S) {
            const float inv = 1.0f / l_row;
            if (Lse != nullptr && kg_o == 0) Lse[bh * (int64_t)S + p_] = m_i[rb] * scale_abs + __logf(l_row);
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                const uint32_t lo = pack2<T>(oacc[rb][db][0] * inv, oacc[rb][db][1] * inv);
                const uint32_t hi = pack2<T>(oacc[rb][db][2] * inv, oacc[rb][db][3] * inv);
                *reinterpret_cast<uint2 *>(Op + (int64_t)p_ * D + db * 16 + kg_o * 4) = make_uint2(lo, hi);
            }
        }
    }
}

template <typename T, int D, int R, int SK, bool SCORES_ONLY, bool BAND = false>
int launch_mfma(const void *q, const void *k, const void *v, const void *w, void *o, float *lse, int64_t B, int64_t H,
                int64_t S, int causal, float scale, int fill_upper, hipStream_t st, const int *band_lo = nullptr, int tri_gl = 0,
                row_strides qs = {0, 0, 0})
{
    using G = fused_geom<R, SK>;
    constexpr bool RAW = SCORES_ONLY && R == 1 && SK == 1;
    static_assert(G::fits, "conv window exceeds the 32-key MFMA contraction");
    const int nqb = (int)((S + G::BQ - 1) / G::BQ);
    // Attention kernel: eight wavefronts of 16 rows instead of four of 32 - the chain of steps that a workgroup is gets a fifth shorter, a CU
    // holds two of these at D = 64 and one at 128 - up to 2 1/4 and 1 3/4 workgroups per CU.  us, four | eight: 6x11 B1 H8 S296 D128 (24
    // workgroups) 19.0 | 15.8, B1 H16 S640 D64 (96) 26.3 | 21.6, D128 32.4 | 27.1, B1 H32 S1300 D64 (352) 49.7 | 41.0, D128 61.9 | 49.6, B1 H24 S2048
    // D128 (432) 91.5 | 78.8, H26 (468) 91.8 | 88.1, H28 (504) 92.0 | 91.9, H32 (576) 94.4 | 103.5, D64 (504) 73.7 | 63.4, (576) 76.0 | 68.2, B2 H60 S600
    // D64 (600) 31.9 | 31.6, B4 H32 S512 (640) 27.7 | 30.6; 3x3, 7x9 and 11x15 alike.
    const bool few = !SCORES_ONLY && 4 * B * H * nqb <= (D == 64 ? 9 : 7) * (int64_t)device_cu_count();
    auto kern = conv_attn_fwd_mfma<T, D, R, SK, SCORES_ONLY, 4, BAND>;
    if constexpr (!SCORES_ONLY) {
        if (few) kern = conv_attn_fwd_mfma<T, D, R, SK, false, 8, BAND>;
    }
    // key blocks per work item: all of them for the attention kernel; QK_CHUNK for the scores-only kernel
    const int jc_len = SCORES_ONLY ? QK_CHUNK : (int)((S + F_BK - 1) / F_BK) + 1;
    int64_t items_per_bh = 0;
    for (int qb = 0; qb < nqb; ++qb) {
        const int64_t ql = std::min<int64_t>((int64_t)qb * G::BQ + G::BQ - 1, S - 1);
        items_per_bh += ((causal ? ql / F_BK : (S - 1) / F_BK) + jc_len) / jc_len;
    }
    // the items of a head, longest first (the number of key blocks an item visits, as the kernel computes it)
    item_table tbl;
    tbl.n = 0;
    if (SCORES_ONLY && nqb <= 2047 && (S + F_BK - 1) / F_BK <= 2047) {
        constexpr int MAXLEN = 1023;
        static thread_local int count[MAXLEN + 2];
        static thread_local uint32_t items[ITEM_TABLE_MAX];
        static thread_local int lens[ITEM_TABLE_MAX];
        // long chunks for the first part of a query block's key range, short ones for the last QK_SHORT_SHARE of it
        static const int env_big = [] { const char *e = getenv("MTA_QK_CHUNK_LONG"); return e ? atoi(e) : 0; }();
        static const int env_small = [] { const char *e = getenv("MTA_QK_CHUNK_SHORT"); return e ? atoi(e) : 0; }();
        static const int share = [] { const char *e = getenv("MTA_QK_SHORT_PERCENT"); return e ? atoi(e) : QK_SHORT_PERCENT; }();
        int64_t head_blocks = 0;
        for (int qb = 0; qb < nqb; ++qb) {
            const int64_t ql = std::min<int64_t>((int64_t)qb * G::BQ + G::BQ - 1, S - 1);
            head_blocks += (causal ? ql / F_BK : (S - 1) / F_BK) + 1;
        }
        const qk_chunks cut = qk_chunk_rule(B * H * head_blocks, head_blocks, nqb);
        const int big = env_big ? env_big : cut.big, small = env_small ? env_small : cut.small;
        int n = 0;
        bool ok = big >= 1 && small >= 1 && big <= MAXLEN && small <= MAXLEN && share >= 0 && share <= 100;
        for (int qb = 0; qb < nqb && ok; ++qb) {
            const int64_t ql = std::min<int64_t>((int64_t)qb * G::BQ + G::BQ - 1, S - 1);
            const int nk = (int)(causal ? ql / F_BK : (S - 1) / F_BK) + 1;  // key blocks 0 .. j_last
            const int nshort = std::min(nk, (nk * share / 100 + small / 2) / small * small);
            const int nlong = nk - nshort;
            for (int j0 = 0; j0 < nk && ok;) {
                const int len = j0 < nlong ? std::min(big, nlong - j0) : std::min(small, nk - j0);
                if (n >= ITEM_TABLE_MAX) { ok = false; break; }
                // what the kernel visits: one key block earlier rebuilds the retained columns (ahead of the first: the right pad)
                lens[n] = len + (!RAW && (j0 > 0 || G::PWR > 0) ? 1 : 0);
                items[n++] = (uint32_t)qb | ((uint32_t)j0 << 11) | ((uint32_t)len << 22);
                j0 += len;
            }
        }
        if (ok && n > 1) {
            std::fill(count, count + MAXLEN + 2, 0);
            for (int i = 0; i < n; ++i) ++count[lens[i]];
            int pos = 0;
            for (int len = MAXLEN + 1; len >= 0; --len) {  // positions: longer items first
                const int c = count[len];
                count[len] = pos;
                pos += c;
            }
            for (int i = n - 1; i >= 0; --i) tbl.e[count[lens[i]]++] = items[i];  // among equal lengths later query blocks first
            tbl.n = n;
            items_per_bh = n;
        }
    }
    const int64_t total_wg = B * H * items_per_bh;
    if (total_wg > 0x7ffffff0LL) return MTA_ERR_SHAPE;
    // Raw scores of long rows that are not whole 128-byte lines, of heads in other numbers than multiples of 8: an XCD takes an eighth of the
    // list, head by head.  Rank by rank, neighbouring items of a row end the same lines on two XCDs.  us, rank by rank | head by head, nothing in the
    // caches, D64: B1 H12 S3344 63.7 | 60.4, S3400 73.7 | 68.9, S4008 100 | 94.6, H20 105 | 102, 122 | 117, 164 | 160, H28 S4008 234 | 221, B3 H12 302 | 287;
    // either way at up to 3072 keys (H28 S3000 133 | 126, H12 55.8 | 58.0, H20 S1704 30.9 | 34.0); slower from 5000 on (H12 151 | 157, H20 263 | 267),
    // with 4 heads (S4008 31.7 | 32.8), of whole lines (H12 S3008 37.4 | 44.7, H28 S4096 160 | 175), and mostly with a conv (6x11 H12 S4008 102 |
    // 109).
    const bool by_head = RAW && S % 64 != 0 && S > 3072 && S <= 4096 && (B * H) % 8 != 0 && B * H > 8;
    const int64_t per_xcd = by_head ? (total_wg + 7) / 8 : 0;
    dim3 grid((unsigned)(by_head ? per_xcd * 8 : total_wg));
    hipLaunchKernelGGL(kern, grid, dim3(few ? 512 : 256), 0, st, (const T *)q, (const T *)k, (const T *)v, (const T *)w, (T *)o,
                       lse, (int)S, causal, scale, (int)H, nqb, fill_upper, (unsigned)total_wg, (unsigned)(B * H), (unsigned)per_xcd, jc_len, tbl, band_lo, tri_gl, qs);
    return launch_status();
}

// returns 1 when no instantiation covers the kernel size (the caller then uses the general kernel)
template <typename T, int D, bool SCORES_ONLY, bool BAND = false>
int dispatch_mfma(const void *q, const void *k, const void *v, const void *w, void *o, float *lse, int64_t B, int64_t H,
                  int64_t S, int R, int Sk, int causal, float scale, int fill_upper, hipStream_t st, const int *band_lo = nullptr,
                  int tri_gl = 0, row_strides qs = {0, 0, 0})
{
    if constexpr (sizeof(T) == 2) {
        if constexpr (SCORES_ONLY) {   // no conv (weights are not read)
            if (R == 1 && Sk == 1)
                return launch_mfma<T, D, 1, 1, true, BAND>(q, k, v, w, o, lse, B, H, S, causal, scale, fill_upper, st, band_lo, 0, qs);
        }
#define MTA_FUSED_CASE(r, s) \
    if (R == r && Sk == s) return launch_mfma<T, D, r, s, SCORES_ONLY, BAND>(q, k, v, w, o, lse, B, H, S, causal, scale, fill_upper, st, band_lo, tri_gl);
        MTA_FUSED_CASE(3, 3)
        MTA_FUSED_CASE(3, 5)
        MTA_FUSED_CASE(5, 5)
        MTA_FUSED_CASE(5, 7)
        MTA_FUSED_CASE(6, 11)
        MTA_FUSED_CASE(7, 7)
        MTA_FUSED_CASE(7, 9)
        // (the 44 registers of its Toeplitz fragments leave both kernels two workgroups per CU)
        MTA_FUSED_CASE(11, 15)
#undef MTA_FUSED_CASE
    }
    return 1;
}

template <typename T, int D> int dispatch_mfma_d(const conv_attn_args &a)
{
    if (!a.scores_only) return dispatch_mfma<T, D, false>(a.q, a.k, a.v, a.w, a.o, a.lse, a.B, a.H, a.S, a.R, a.Sk, a.causal, a.scale, 0, a.st);
    if (a.band_lo)
        return dispatch_mfma<T, D, true, true>(a.q, a.k, nullptr, a.w, a.o, nullptr, a.B, a.H, a.S, a.R, a.Sk, 1, a.scale, a.fill_upper, a.st, a.band_lo, a.tri_gl, a.qs);
    return dispatch_mfma<T, D, true>(a.q, a.k, nullptr, a.w, a.o, nullptr, a.B, a.H, a.S, a.R, a.Sk, a.causal, a.scale, a.fill_upper, a.st, nullptr, a.tri_gl, a.qs);
}
template <typename T> int dispatch_mfma_type(const conv_attn_args &a) { return a.D == 64 ? dispatch_mfma_d<T, 64>(a) : dispatch_mfma_d<T, 128>(a); }
}  // namespace
