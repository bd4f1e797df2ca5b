// The scores kernel of conv_attn_fwd.hip for 16-bit types: products and conv on the matrix cores.  A template over the I/O type,
// instantiated in conv_attn_bf16.hip and conv_attn_f16.hip by way of conv_attn_mfma.hpp.
#pragma once

#include <algorithm>

#include <stdlib.h>

#include "conv_attn_lds.hpp"
#include "scores_cut.hpp"

namespace {

// 4 wavefronts own 128 score rows (HR halo rows + 128-HR output rows); a wavefront scores two blocks of 16 rows and takes the 32 rows as
// 16 pairs of neighbours from the conv on.  K blocks (64 keys) are copied global -> LDS asynchronously (global_load_lds), double buffered,
// row-major, 16-byte chunks XOR-swizzled by the key index instead of padded; S^T = K Q^T -> scale, causal/range zero -> LDS score tile
// (I/O dtype) -> conv as MFMAs of a zero-padded tap matrix (scores_geom; its operands live in registers) -> global.  Three workgroups per
// CU overlap each other's barriers and memory latency.  (Eight wavefronts, with the fragments of K read twice as often: 6x11 B2 H16 S512 D64
// 12.5 -> 17.4 us, B4 H16 S1024 D128 38.4 -> 43.2.)
// us, a conv product for one row and sixteen keys -> for a pair of rows and eight, bf16 6x11 B2 H16 S4096 D128 220 -> 207, fp16 7x7 B1 H16
// 126 -> 102 (in a loop, warm: 244 -> 229, 132 -> 115): the matrix cores are busy 41 % (50), the LDS 42 % (54), the vector ALU 40 % of the
// cycles (42: addresses of the stores formed once, by 32-bit offset).
// What bounds it: without its stores it takes 155 us of 229, without products and copies of K 147: the sum is what the clock, not a unit,
// bounds - non-temporal stores (207 in a loop, the forward unchanged), whole lines per instruction, stores left in flight, copies of K asked
// for half a block earlier, deeper or shallower reads: no gain in a forward.
// The fused attention kernel keeps one row x sixteen keys: with pairs (two maxima a key block, exchanges between the rows' lanes) it gained
// on long grids, B1 H32 S8192 D128 1004 -> 953, and lost where a workgroup's chain of steps counts, 6x11 B1 H8 S2048 D64 52 -> 70, B1 H32
// S1300 43 -> 56.
constexpr int QK_OCC = 3;     // wavefronts per SIMD the kernel is compiled for (three workgroups per CU)
__device__ __forceinline__ uint32_t lds_read4_at(unsigned addr, int off)
{
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
}
template <int N> __device__ __forceinline__ void lds_wait_upto(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t &d)
{
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(a), "+v"(b), "+v"(c), "+v"(d) : "n"(N) : "memory");
}
// a in lanes 32-63, b in lanes 0-31
__device__ __forceinline__ uint32_t upper_half_of(uint32_t a, uint32_t b)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)b, (int)a, 0xe4, 0xc, 0xf, false);   // (0xe4: every lane its own)
}
// The conv on the matrix cores.  A product (16x16x32) takes two query rows x eight keys of output (its 16 rows) for sixteen pairs of
// query rows (its 16 columns): the pair's window has R + 1 rows, the eight keys' SK + 7 columns, and the 32 slots of the contraction
// hold 8-column chunks of the window's rows, 8 slots a lane group.  6x11 needs 7 x 18 = 126 slots for 256 outputs, four products;
// one row x sixteen keys at a time, 26 of whose 32 slots a kernel row uses, took six.  And the operand that comes from LDS - four rows of
// one chunk (`quad`) - serves the windows of NP neighbouring groups of eight keys, each with taps of its own.
//   columns of the score tile (a row of the window in the tile's own columns): HC kept from the key block before, then 64 new ones;
//   group c of eight keys has its first tap at column 8c + SHIFT, its last at 8c + HC + 7.
//   R + 1 rows = NQ quads, then: 2 rows left -> one operand of 2 rows x 2 chunks (PAIR);  3 rows left and two columns of a chunk
//   ahead of two whole ones (LEFT: 11 taps, columns 8c + 6, 8c + 7) -> PAIR, and one operand (LAST) of the seventh row's two chunks in lane groups
//   0 and 1 and the two columns of all seven rows, one dword a row, in 2 and 3: rows 0, 2, 4, 6 and 1, 3, 5.  Those dwords are the last ones of
//   operands that the products of the groups before have just used: the quad of chunk c - 1 (four rows, a lane group each) and the second half of
//   PAIR of group c - 2 (two rows); three moves bring them to their place in LAST.  The first two groups of a key block gather them from LDS.
// Products | LDS operands per 256 outputs, now (one row at a time: R | R): 3x3, 3x5 2 | 1.1, 5x5, 5x7 3 | 2.1, 6x11 4 | 3.1, 7x7, 7x9 4 | 2.3, 11x15 9 | 3.8.
// The order of the operand reads, computed at compile time: read i is a quad of chunk at (kind < NQ), or PAIR or LAST of group at.
struct conv_reads {
    int n = 0, kind[80] = {}, at[80] = {}, last[16] = {};   // last: a group's last read
    bool gathered[80] = {};
    constexpr void add(int k, int a, bool g) { kind[n] = k, at[n] = a, gathered[n] = g, ++n; }
    constexpr int ops(int lo, int hi) const   // LDS operations of reads lo .. hi - 1
    {
        int c = 0;
        for (int i = lo; i < hi && i < n; ++i) c += gathered[i] ? 4 : 1;
        return c;
    }
};
template <int R, int SK> struct scores_geom {
    static constexpr int F_SR = 128;
    static constexpr int HR = (R - 1 + 7) & ~7;    // halo rows above the block (recomputed)
    static constexpr int HC = (SK - 1 + 7) & ~7;   // score columns that the first group of a key block reaches back
    static constexpr int BQ = F_SR - HR;           // output rows per workgroup
    static constexpr int PW = (SK - 1) / 2, PWR = SK - 1 - PW;
    static constexpr int SHIFT = HC - (SK - 1);    // first tap's column in a group's window
    static constexpr bool LEFT = R == 6 && HC == 16 && SHIFT == 6;
    static constexpr int C0 = LEFT ? 8 : 0;        // first column that the tile holds
    static constexpr int KEPT = HC - C0;           // of which this many are kept
    // A row's length: in an operand read neighbouring lanes are two rows apart and lane groups a row or a chunk, and the LDS serves lanes
    // 0-7 together with lanes 24-31 (8-15 with 16-23).  With rows of an odd number of chunks two rows are an odd multiple of 32 bytes, so
    // that the lanes of one group meet the eight even 16-byte positions of the banks and those of the other the odd ones.
    static constexpr int SLD = KEPT <= 8 ? 72 : 88;
    static constexpr int NP = KEPT / 8 + 1;        // chunks of a window
    static constexpr int WR = R + 1, NQ = WR / 4, REST = WR % 4;
    static constexpr bool PAIR = REST >= 2;
    static constexpr bool fits = (R == 1 && SK == 1) || ((REST == 0 || (REST == 2 && NP == 2) || LEFT) && KEPT > 0 && KEPT + 64 <= SLD);
    // zero-padded kernel rows -1 .. R and zeros around the taps, from which the operands are gathered
    static constexpr int WZ_OFF = SHIFT + 8, WZ_LD = 40;
    static constexpr int KPAIR = NQ, KLAST = NQ + 1, NTZ = NQ * NP + (PAIR ? 1 : 0) + (LEFT ? 1 : 0);   // operands of taps
    static constexpr conv_reads reads(int nwin)
    {
        conv_reads p;
        if (LEFT) p.add(KLAST, 0, true);
        for (int x = 0; x < nwin + NP - 1; ++x) {
            for (int q = 0; q < NQ; ++q) p.add(q, x, false);
            const int w = x - (NP - 1);   // the group whose last chunk this is
            if (PAIR && w >= 0) p.add(KPAIR, w, false);
            if (w >= 0) p.last[w] = p.n - 1;
            if (LEFT && x + 1 < nwin) p.add(KLAST, x + 1, x == 0);
        }
        return p;
    }
};

// A head's work items (query block, range of key blocks) in the order they are to be started: longest first, so that the
// long items all start early and the short ones fill the end of the grid.  Built on the host for every launch (a
// counting sort over at most ITEM_TABLE_MAX items) and passed by value as a kernel argument; n = 0: no table, the kernel
// cuts every query block's key range into chunks of jc_len blocks and walks the query blocks from the last to the first.
// The chunks need not be equal: the first part of a query block's key range goes into long items (an item costs a few
// microseconds to set up), the rest into short
// ones, which are started last and even out the end of the grid.
struct item_table {
    int n;
    uint32_t e[ITEM_TABLE_MAX];  // query block (11 bits) | first key block << 11 (11 bits) | key blocks << 22
};

// RAW (a 1x1 kernel): no conv at all - round(round(Q K^T) * scale) goes from the accumulators to memory: the
// plain lower-triangle product of the training route (raw scores, dP = dO V^T).  No score tile, no retained columns, no halo.
// Writes  conv(mask0(scale * Q K^T))  as an (S,S) plane per (batch, head).  Only q <= p is written when causal, plus +0 above the
// diagonal when `fill_upper` is set.
// BAND: a mask of the form "key k of query row p is visible iff band_lo[b, p] <= k <= p" - the
// scores of the hidden keys enter the conv as 0, as the reference's masked_fill ahead of its conv leaves them
// (mta_attention_triton.py:70-73).
// STATS (causal): the statistics of each row's scores of the item, as they are stored (scores_stats): 32 more vector instructions and eight exponentials per
// eight scores of a lane, us without | with them | and a key bias: bf16 6x11 B2 H16 S4096 D128 226 | 247 | 255 (in a loop: the clock), B4 H16 S1024
// 37.6 | 44.2 | 46.0, B1 H16 S2048 37.7 | 46.1 | 47.4, 7x7 B2 H16 S4096 D64 180 | 195 | 203.  With the maximum so far taken at every eight, and a factor for the sum, B2 H16 S4096 took 22 us more.
// STATS 2: with a key bias, which an instance of its own has to look for.
template <typename T, int D, int R, int SK, bool BAND, int STATS>
__global__ __launch_bounds__(256, R <= 7 && !(STATS && BAND && R >= 6 && D == 128) ? QK_OCC : 2) void conv_scores_mfma(const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ Wt,
                                                           T *__restrict__ O, int S, int SR, int causal, float scale, int H, int nqb, int fill_upper,
                                                           unsigned total_wg, unsigned heads, unsigned per_xcd, int jc_len,
                                                           item_table tbl, const int *__restrict__ band_lo, int tri_gl, row_strides qs, scores_stats st)
{
    using G = scores_geom<R, SK>;
    constexpr bool RAW = R == 1 && SK == 1, KB = STATS == 2;
    static_assert(!RAW || !STATS, "raw scores have no statistics");
    constexpr int NW = 4, F_NT = 64 * NW, F_SR = 128, RB = F_SR / (16 * NW);   // (RB: blocks of 16 rows per wavefront)
    constexpr int CPR = D / 8;                     // 16-byte chunks per K row
    constexpr int TILE = F_BK * D;                 // elements per K block
    constexpr int ROUNDS = TILE / 8 / F_NT;        // copy instructions per block per lane
    constexpr int KS = D / 32;                     // contraction steps over the head dim
    constexpr int NCB = F_BK / 16;                 // 16-key blocks per iteration
    static_assert(ROUNDS >= 1, "block smaller than one copy round");

    // K is double-buffered in B0 / B1, arrays of their own with a loop body each: the compiler then sees that LDS reads never touch the
    // asynchronous copy in flight into the other one.
    __shared__ __align__(16) T B0[TILE];
    __shared__ __align__(16) T B1[TILE];
    __shared__ __align__(16) T tile[RAW ? 8 : F_SR * G::SLD];   // score tile
    // the two columns ahead of the tile's first, for the first group's window (one dword a row)
    __shared__ uint32_t side[G::LEFT ? F_SR : 1];
    // zero-padded kernel rows, only needed until the taps' operands are built: they borrow a buffer that
    // receives its first copy after that (LDS is granted in 1280-byte units; the array's own 648 bytes were the
    // difference between two and three workgroups per CU)
    static_assert((R + 2) * G::WZ_LD <= TILE, "kernel rows do not fit the borrowed buffer");
    T *const wz = B1;

    const int tid = threadIdx.x;
    // (the wavefront index through readfirstlane: everything derived from it is then scalar, branches included)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // The items are taken rank by rank - the longest item of every head, then the second longest of each, ... - so that the long items
    // all start early and the short ones fill the end of the grid (workgroups start in index order as slots free up).
    // Workgroup ids are dealt round-robin to the 8 XCDs: with heads in multiples of 8 an XCD keeps its own, whose K and V stay in its L2
    // (of 12 heads an XCD sees 3, of 4 one).  With other numbers of heads an XCD used to take an eighth of the list head by head - of 4
    // heads one XCD a head's long items and another its short ones.  us, that -> this, bf16 6x11: B1 H4 S3008 D128
    // 26.5 -> 24.1, B1 H12 S2048 D64 33.7 -> 27.7, S3712 D64 76.3 -> 67.5, S4096 D128 101 -> 93,
    // B1 H20 S2048 D128 53.2 -> 45.8; without a conv B1 H12 S2048 D64 16.9 -> 14.4, S2560 23.8 -> 20.1.  per_xcd: the old deal, see
    // launch_scores.
    // Work item = (batch*head, query block, chunk of jc_len key blocks).  The key range of a query block is split (its output columns are
    // independent; a chunk starts with the 16 keys ahead of it, for the kept columns), so that items are short and equal and the grid
    // runs in several even rounds.
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
    const T *Qp = Q + (q_strided ? (int64_t)(bh / H) * qs.batch + head * qs.head : (int64_t)bh * SR * D);
    const int64_t q_row = q_strided ? qs.row : D;
    const T *Kp = K + (int64_t)bh * SR * D;   // (SR: rows that q and k have, at most S; those beyond re-read the last one)
    // (tri_gl > 0: the scores go out in the triangular layout, groups of tri_gl heads interleaved by rows;
    // nothing above the diagonal is stored then)
    const bool tri = tri_gl > 0;
    T *Op = tri ? O + ((unsigned)bh / (unsigned)(tri ? tri_gl : 1)) * ((tri ? tri_gl : 1) * tri_rowoff(S)) : O + (int64_t)bh * S * S;
    const int tri_i = tri ? (int)((unsigned)bh % (unsigned)tri_gl) : 0;
    // Scores go to memory from the start of row o_row of the plane (the same for the whole workgroup), with a 32-bit offset per lane for the
    // row, formed once: forming the addresses at each store was a quarter of the vector instructions.
    const int o_row = q0 - G::HR > 0 ? q0 - G::HR : 0;
    char *const o_at = reinterpret_cast<char *>(Op + (tri ? tri_gl * tri_rowoff(o_row) + tri_i * (int64_t)tri_rowlen(o_row) : (int64_t)o_row * S));
    auto o_offset = [&](int row) {   // bytes from o_at to the row's start; rows of this workgroup's
        return (tri ? tri_row_start(row, tri_gl, tri_i) - tri_row_start(o_row, tri_gl, tri_i) : (unsigned)(row - o_row) * (unsigned)S) * (unsigned)sizeof(T);
    };

    // asynchronous copy of key block j into a buffer; out-of-range keys re-read a valid row (their scores are zeroed later)
    // slot r*256+tid of a block is row kv_row[r], 16-byte chunk kv_c of that row (fixed per lane)
    // (a round advances the row by F_NT/CPR, a multiple of CPR: the swizzled chunk is the same in every round)
    static_assert((F_NT / CPR) % CPR == 0 && F_NT % CPR == 0, "copy rounds must keep the swizzle phase");
    const int kv_row0 = tid / CPR;
    const int kv_off0 = kv_row0 * D + ((tid % CPR) ^ (kv_row0 & (CPR - 1))) * 8;
    // (a block inside the sequence: a uniform address and this lane's offset, which the copy adds by itself)
    auto issue_k = [&](int j, T *dst) __attribute__((always_inline)) {
        const int first = j * F_BK + G::PWR;
        if (first >= 0 && first + F_BK <= SR) {
            const char *at = reinterpret_cast<const char *>(Kp + (int64_t)first * D);
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r)
                __builtin_amdgcn_global_load_lds((glb_void_t *)(at + r * (F_NT / CPR) * D * (int)sizeof(T) + (unsigned)(kv_off0 * (int)sizeof(T))),
                                                 (lds_void_t *)(dst + (r * F_NT + wave * 64) * 8), 16, 0, 0);
        } else {
            MTA_KEEP_BRANCH();
#pragma unroll
            for (int r = 0; r < ROUNDS; ++r) {
                int row = first + kv_row0 + r * (F_NT / CPR);
                row = row < 0 ? 0 : (row >= SR ? SR - 1 : row);
                __builtin_amdgcn_global_load_lds((glb_void_t *)(Kp + (kv_off0 + (row - kv_row0) * D)),
                                                 (lds_void_t *)(dst + (r * F_NT + wave * 64) * 8), 16, 0, 0);
            }
        }
    };

    const int q_last = (q0 + G::BQ - 1 < S - 1) ? q0 + G::BQ - 1 : S - 1;
    const int j_last = causal ? q_last / F_BK : (S - 1) / F_BK;  // last key block of the query block
    int j_lo = tbl_lo >= 0 ? tbl_lo : jc * jc_len;                // first key block whose outputs this item produces
    const int j_len = tbl_lo >= 0 ? tbl_len : jc_len;
    const int j_end = (j_lo + j_len - 1 < j_last) ? j_lo + j_len - 1 : j_last;
    float2 *const stats_at = STATS ? st.at + ((int64_t)bh * st.slots + st.cut.index(j_last + 1, j_lo)) * S : nullptr;   // the item's, row 0
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
        if (j_lo > j_end) {
            if constexpr (STATS) {
                for (int r = tid; r < G::BQ; r += F_NT)
                    if (q0 + r < S) stats_at[q0 + r] = make_float2(NO_SCORE, 0.0f);
            }
            return;
        }
    }
    // What the start waits for is asked for at once, this wavefront's rows of Q and the kernel's taps ahead of the first block of K:
    // behind it, the taps waited for the block and Q was asked for when that had come.  With the 32-bit divisions above, scores
    // kernel, us: bf16 6x11 B2 H16 S1008 D64 22.3 -> 21.1, B4 H16 S1024 D128 40.6 -> 40.1, 7x7 B1 H16 S1024 D64 18.6 -> 17.7, B1 H16 S2048 D128 42.1 ->
    // 40.9, 6x11 B2 H16 S2048 D128 69.7 -> 67.5, S4096 240 -> 236, 11x15 B2 H16 S640 D128 21.1 -> 19.8.
    int trow[RB], prow[RB];   // this lane's query rows
    frag8<T> qf[RB][KS];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        trow[rb] = wave * (16 * RB) + rb * 16 + ln;
        prow[rb] = q0 - G::HR + trow[rb];
        const int pc = prow[rb] < 0 ? 0 : (prow[rb] >= SR ? SR - 1 : prow[rb]);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[rb][ks] = *reinterpret_cast<const frag8<T> *>(Qp + pc * q_row + ks * 32 + kg * 8);
    }
    constexpr int WZ_IT = ((R + 2) * G::WZ_LD + F_NT - 1) / F_NT;
    T taps[RAW ? 1 : WZ_IT];
    if constexpr (!RAW) {
#pragma unroll
        for (int n = 0; n < WZ_IT; ++n) {
            const int e = n * F_NT + tid, i = e / G::WZ_LD - 1, jj = e % G::WZ_LD - G::WZ_OFF;
            taps[n] = Wt[head * R * SK + (i >= 0 && i < R && jj >= 0 && jj < SK ? i * SK + jj : 0)];
        }
    }
    asm volatile("" : : : "memory");
    // The score columns kept from the key block ahead of the first one are the last of its 16 keys: those rows of K go to their place in
    // the buffer that the block behind the first gets (the zero-padded taps lie at its other end).  They used to be the by-product of a whole
    // key block with a copy and barriers of its own: us, scores bf16 6x11 D128, in a loop, B1 H4 S200 8.1 -> 7.0, B1 H8 S512 8.8 -> 7.6, B2 H16
    // S1008 26.7 -> 24.7, B1 H16 S2048 43.7 -> 41.9, B4 H16 S1024 44.9 -> 44.0, B2 H16 S4096 224 -> 221; shorter or longer items: no gain.
    if constexpr (!RAW) {
        static_assert((R + 2) * G::WZ_LD <= (F_BK - 16) * D && 64 / CPR <= 16 && F_NT / CPR >= 16, "16 rows of K beside the taps; whole wavefronts copy them");
        const int first = (j_lo - 1) * F_BK + G::PWR, row = kv_row0 + (ROUNDS - 1) * (F_NT / CPR);
        if (__builtin_amdgcn_readfirstlane(row) >= F_BK - 16) {
            const int key = first + row < 0 ? 0 : (first + row >= SR ? SR - 1 : first + row);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Kp + (kv_off0 + (key - kv_row0) * D)),
                                             (lds_void_t *)(wz + ((ROUNDS - 1) * F_NT + wave * 64) * 8), 16, 0, 0);
        }
    }
    issue_k(j_lo, B0);

    if constexpr (!RAW) {
    // zero the score tile once (the columns kept from the key block before the first one; 15 taps: columns nobody writes)
    for (int e = tid; e < F_SR * G::SLD / 8; e += F_NT) {
        pack16<T> z;
#pragma unroll
        for (int u = 0; u < 8; ++u) z.v[u] = from_float<T>(0.0f);
        *reinterpret_cast<pack16<T> *>(tile + e * 8) = z;
    }
    if (G::LEFT && tid < F_SR) side[tid] = 0;
#pragma unroll
    for (int n = 0; n < WZ_IT; ++n) {
        const int e = n * F_NT + tid, i = e / G::WZ_LD - 1, jj = e % G::WZ_LD - G::WZ_OFF;
        if (e < (R + 2) * G::WZ_LD)
            wz[e] = i >= 0 && i < R && jj >= 0 && jj < SK ? taps[n] : from_float<T>(0.0f);
    }
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (prow[rb] < 0 || prow[rb] >= S) qf[rb][ks] = zero_frag<T>();  // rows outside the sequence are conv padding
    // band mask: first visible key of this lane's two rows, and the largest of them over the wavefront's 32 rows (a key
    // block that starts at or beyond it is visible to all of them)
    int flo[2] = {0, 0}, fmax_w = 0;
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
    __builtin_amdgcn_s_waitcnt(0);   // this wavefront's 16 rows of K, the first block
    __syncthreads();

    // The conv's taps as operands: product row m = ln is the output of row m/8 of the pair and key m%8 of the group; a slot that holds column
    // col of the window's row `row` takes tap (row - m/8, col - SHIFT - m%8), 0 where there is none.
    frag8<T> tz[RAW ? 1 : G::NTZ];
    if constexpr (!RAW) {
        const T *const src = wz + G::WZ_LD + G::WZ_OFF - G::SHIFT - (ln >> 3) * G::WZ_LD - (ln & 7);
#pragma unroll
        for (int q = 0; q < G::NQ; ++q)
#pragma unroll
            for (int c = 0; c < G::NP; ++c)
#pragma unroll
                for (int t = 0; t < 8; ++t) tz[q * G::NP + c].v[t] = src[(4 * q + kg) * G::WZ_LD + G::C0 + 8 * c + t];
        if constexpr (G::PAIR) {
#pragma unroll
            for (int t = 0; t < 8; ++t) tz[G::NQ * G::NP].v[t] = src[(4 * G::NQ + (kg & 1)) * G::WZ_LD + G::C0 + 8 * (kg >> 1) + t];
        }
        if constexpr (G::LEFT) {
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int row = kg < 2 ? G::WR - 1 : (kg & 1) + t / 2 * 2, col = kg < 2 ? G::C0 + 8 * kg + t : G::C0 - 2 + t % 2;
                tz[G::NTZ - 1].v[t] = row < G::WR ? src[row * G::WZ_LD + col] : from_float<T>(0.0f);
            }
        }
    }

    // Kept columns: each thread moves one 16-byte vector per round (KEPT/8 vectors per row); LEFT: the next 128 threads the two columns
    // ahead of the kept ones, for the first group's window.
    constexpr int VPRW = G::KEPT / 8 > 0 ? G::KEPT / 8 : 1, TAIL_VECS = F_SR * (G::KEPT / 8), TAIL_ALL = TAIL_VECS + (G::LEFT ? F_SR : 0);
    constexpr int TAIL_IT = (TAIL_ALL + F_NT - 1) / F_NT;
    static_assert(!G::LEFT || TAIL_IT == 1, "one vector per thread");
    int tail_off[TAIL_IT > 0 ? TAIL_IT : 1];  // where this thread's vector(s) go in the tile's rows; LEFT: where they come from
#pragma unroll
    for (int it = 0; it < TAIL_IT; ++it) {
        const int idx = it * F_NT + tid;
        tail_off[it] = idx < TAIL_VECS ? (idx / VPRW) * G::SLD + (idx % VPRW) * 8 : idx < TAIL_ALL ? (idx - TAIL_VECS) * G::SLD - 8 : -1;
    }
    // the 16-row blocks of this wavefront span rows pmin .. pmin + 16 RB - 1 of the sequence
    const int pmin = q0 - G::HR + wave * (16 * RB);
    // Rows of the conv and of the stores.  The first wavefront's rows are taken
    // R-1 further down than the rows it computes scores for: its conv windows then start at tile row 0 instead of
    // above the tile, every operand's address is the same affine function of (row pair, window row), and what it
    // leaves out are halo rows nobody stores.  Its last R-1 rows belong to the second wavefront too and are not
    // stored from here.
    const int cshift = wave == 0 ? R - 1 : 0;
    static_assert(RAW || G::HR >= R - 1, "the first wavefront's first conv row would be a stored one");
    // A product's column ln is a pair of rows: rows 2ln, 2ln + 1 of the wavefront's 32.  Its result lies with row kg/2 of the pair and keys
    // 4(kg%2) .. + 3 of the group.
    const int pair_row = wave * (16 * RB) + cshift + 2 * ln;
    // where this lane's vectors of 8 keys go: two rows - of its two row blocks (RAW), of its pair - and a column of 32 or 64 bytes' worth
    const int o_col = RAW ? (kg & 1) * 16 + (kg >> 1) * 8 : kg * 8;
    unsigned o_off[2] = {0, 0};
    bool stored[2] = {false, false};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int tr_ = RAW ? trow[h] : pair_row + h, p_ = q0 - G::HR + tr_;
        stored[h] = tr_ >= G::HR && tr_ < (wave + 1) * 32 && p_ < S;
        o_off[h] = o_offset(p_) + (unsigned)(o_col * (int)sizeof(T));
    }

    // four scores of row block rb, keys col .. col + 3, as the tile holds them
    auto score4 = [&](int rb, f32x4 a, int col, bool masked, uint32_t &lo, uint32_t &hi) __attribute__((always_inline)) {
        lo = pack2<T>(a[0], a[1]), hi = pack2<T>(a[2], a[3]);
        // MTA scales the scores before the conv, in the I/O dtype: round, scale, round again
        float a0, a1, a2, a3;
        unpack2<T>(lo, a0, a1);
        unpack2<T>(hi, a2, a3);
        lo = pack2<T>(a0 * scale, a1 * scale);
        hi = pack2<T>(a2 * scale, a3 * scale);
        if (masked) {
            MTA_KEEP_BRANCH();
            const int prow_ = STATS ? q0 - G::HR + wave * (16 * RB) + rb * 16 + (opaque_lane(lane) & 15) : prow[rb];   // (formed here: registers)
            const int lim = causal ? (prow_ < S - 1 ? prow_ : S - 1) : S - 1;  // last key kept
            const int first = BAND ? (flo[rb] > 0 ? flo[rb] : 0) : 0;  // first key kept
            if (col < first || col > lim) lo &= 0xffff0000u;
            if (col + 1 < first || col + 1 > lim) lo &= 0x0000ffffu;
            if (col + 2 < first || col + 2 > lim) hi &= 0xffff0000u;
            if (col + 3 < first || col + 3 > lim) hi &= 0x0000ffffu;
        }
    };
    if constexpr (!RAW) {   // the kept columns: scores of the last 16 keys of the block ahead of the first
        f32x4 sacc[RB];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const frag8<T> kf = *reinterpret_cast<const frag8<T> *>(wz + (F_BK - 16 + ln) * D + (((ks * 4 + kg) ^ (ln & (CPR - 1))) * 8));
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                if (ks == 0) sacc[rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                mma16(sacc[rb], kf, qf[rb][ks]);
            }
        }
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            uint32_t lo, hi;
            score4(rb, sacc[rb], (j_lo - 1) * F_BK + G::PWR + F_BK - 16 + kg * 4, true, lo, hi);
            *reinterpret_cast<uint2 *>(tile + trow[rb] * G::SLD + G::KEPT + F_BK - 16 + kg * 4) = make_uint2(lo, hi);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }

    auto plain = [&](int j) {
        const int cbase = j * F_BK + G::PWR;
        return j >= 0 && cbase + F_BK <= S && (!causal || cbase + F_BK - 1 <= pmin) && (!BAND || cbase >= fmax_w);
    };
    // STATS, of this lane's keys of the rows of its pair: minus a reference, in powers of two, and the sum of exponentials relative to it
    float row_neg[2] = {-NO_SCORE, -NO_SCORE}, row_sum[2] = {0.0f, 0.0f};
    int row_lo[2] = {0, 0};
    uint64_t hidden = 0;                                              // keys of the block that the key bias hides
    const float *const kb = KB && st.key_bias ? st.key_bias + (int64_t)(bh / H) * S : nullptr;
    float kb_next = 0.0f;
    auto load_bias = [&](int j) __attribute__((always_inline)) {
        const int key = j * F_BK + lane;
        kb_next = kb[key < S ? key : S - 1];
    };
    if constexpr (STATS) {
        if (KB && kb) load_bias(j_lo);
        if constexpr (BAND) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int p_ = q0 - G::HR + pair_row + h;
                row_lo[h] = p_ >= 0 && p_ < S ? band_lo[(bh / H) * (int64_t)S + p_] : 0;
            }
        }
    }
    // Eight scores of the row h of the pair, keys col .., into the row's statistics.  The reference is the maximum of the lane's first eight
    // (FIRST) and stays: exponentials of what follows may be large, and where they are too large for 32 bits (the sum is infinite or NaN) all of
    // it is done again with the maximum so far (EVERY), as it is under a band mask, whose rows' first scores may be hidden.  Where a key bias hides all
    // of a lane's eight, the next ones are its first (`fresh`: some lane of the wavefront has none yet): the items that start within the padding of a left-padded
    // sequence were all done again, forward of B1 H12 S1808 D64 bf16 7x7 83.7 -> 77.0 us.
    bool fresh = true;
    constexpr float LOG2E = 1.4426950408889634f;
    const std::integral_constant<int, 0> rest{};
    const std::integral_constant<int, 1> first_ones{};
    const std::integral_constant<int, 2> every{};
    auto take = [&](auto mode, auto plain_tag, int h, u32x4_t v, int col, uint64_t hide, int shift) __attribute__((always_inline)) {
        constexpr int MODE = BAND ? 2 : decltype(mode)::value;
        if (!decltype(plain_tag)::value || BAND || (KB && hide != 0)) {
            MTA_KEEP_BRANCH();
            const uint32_t gone = (uint32_t)(hide >> shift) >> ((opaque_lane(lane) >> 4) * 8) & 255u;
            const int last = q0 - G::HR + wave * (16 * RB) + cshift + 2 * (opaque_lane(lane) & 15) + h - col, first = BAND ? row_lo[h] - col : 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                constexpr uint32_t NINF = std::is_same<T, bf16_t>::value ? 0xff80u : 0xfc00u;
                if (2 * u > last || 2 * u < first || (gone >> (2 * u) & 1u)) v[u] = (v[u] & 0xffff0000u) | NINF;
                if (2 * u + 1 > last || 2 * u + 1 < first || (gone >> (2 * u + 1) & 1u)) v[u] = (v[u] & 0x0000ffffu) | NINF << 16;
            }
        }
        if constexpr (MODE != 0) {
            float m = -3.402823466e38f;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float x0, x1;
                unpack2<T>(v[u], x0, x1);
                asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(m), "v"(x0), "v"(x1));
            }
            const float neg = fminf(-m * LOG2E, row_neg[h]);   // (no score yet: NO_SCORE stays)
            if constexpr (MODE == 2) row_sum[h] *= __builtin_amdgcn_exp2f(neg - row_neg[h]);
            if (MODE == 2 || !KB || row_neg[h] == -NO_SCORE) row_neg[h] = neg;
        }
        float sum = row_sum[h];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float x0, x1;
            unpack2<T>(v[u], x0, x1);
            sum += __builtin_amdgcn_exp2f(fmaf(x0, LOG2E, row_neg[h]));
            sum += __builtin_amdgcn_exp2f(fmaf(x1, LOG2E, row_neg[h]));
        }
        row_sum[h] = sum;
    };
    float nan = 0.0f;   // NaN once a product of the key block has met a value that is not finite
    // PLAIN: the key block (its scores and its conv outputs) lies inside the sequence and on or below the diagonal
    // for all 32 rows of this wavefront: no masks and no per-sub-block tests (most blocks of a long sequence)
    auto block = [&](auto plain_tag, int j, const T *Kb, T *Kn) __attribute__((always_inline)) {
        constexpr bool PLAIN = decltype(plain_tag)::value;
        const int cbase = j * F_BK + G::PWR;  // first key of the new score block
        char *const o_block = o_at + (int64_t)(RAW ? cbase : j * F_BK) * (int)sizeof(T);
        // (a vector type, read by every lane: a struct read under a lane condition travels through scratch memory)
        u32x4_t tailreg[TAIL_IT > 0 ? TAIL_IT : 1];
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it)
            tailreg[it] = *reinterpret_cast<const u32x4_t *>(tile + (G::LEFT ? (tid < TAIL_ALL ? tail_off[it] : 0) : tail_off[it] >= 0 ? tail_off[it] : 0) + F_BK);
        __builtin_amdgcn_s_waitcnt(0);  // this wavefront's part of block j has landed in LDS
        __syncthreads();                // ... and everybody's; all reads of the previous tiles are done
        // (Leaving the previous iteration's result stores in flight here - vmcnt(number of stores) instead of 0 - was
        // measured: no gain.)
#pragma unroll
        for (int it = 0; it < TAIL_IT; ++it) {
            if constexpr (G::LEFT) {
                if (tid < TAIL_VECS) *reinterpret_cast<u32x4_t *>(tile + tail_off[it]) = tailreg[it];
                else if (tid < TAIL_ALL) side[tid - TAIL_VECS] = tailreg[it][3];
            } else if (tail_off[it] >= 0) {
                *reinterpret_cast<u32x4_t *>(tile + tail_off[it]) = tailreg[it];
            }
        }
        if (j < j_end) issue_k(j + 1, Kn);  // lands while this block is being worked on
        if (KB && kb) {
            hidden = __builtin_amdgcn_ballot_w64(kb_next == -INFINITY);
            if (j < j_end) load_bias(j + 1);
        }

        // ---- S^T = K Q^T, zero above the diagonal / outside the sequence, to the score tile ----
        {
            // Pipelined like the conv phase below: K fragments are read from assembly KLD steps (two 16-key
            // blocks) ahead into a ring of registers, a step being one fragment and the two products it feeds (both row
            // blocks); a block's scores are rounded, scaled, masked and written LAG steps into the next block.
            constexpr int NSTEP = NCB * KS, KLD = STATS && D == 128 && (R == 6 || BAND) ? 5 : 2 * KS, KSLOT = KLD + 1, LAG = 2;
            static_assert(NSTEP > KLD && KS >= LAG && NCB % 2 == 0, "pipeline deeper than the work; blocks are written in pairs");
            unsigned ka[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                ka[ks] = lds_addr(Kb) + (unsigned)((ln * D + (((ks * 4 + kg) ^ (ln & (CPR - 1))) * 8)) * (int)sizeof(T));
            const unsigned wa = lds_addr(tile) + (unsigned)((trow[0] * G::SLD + G::KEPT + (kg & 1) * 16 + (kg >> 1) * 8) * (int)sizeof(T));
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
                const bool s_plain = PLAIN || (cbase + cb * 16 >= 0 && cbase + cb * 16 + 16 <= S && (!causal || cbase + cb * 16 + 15 <= pmin) &&
                                               (!BAND || cbase + cb * 16 >= fmax_w));
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const f32x4 a = sacc[cb & 1][rb];
                    uint32_t lo, hi;
                    score4(rb, a, cbase + cb * 16 + kg * 4, !s_plain, lo, hi);
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
                            const int col = cbase + (cb - 1) * 16 + o_col, p_ = prow[rb];
                            if (p_ < S && (PLAIN || (col < S && (!causal || fill_upper || col <= p_))))
                                *reinterpret_cast<u32x4_t *>(o_block + o_off[rb] + (cb - 1) * 16 * (int)sizeof(T)) = u32x4_t{s0[0], s1[0], s0[1], s1[1]};
                        } else
                        lds_write16_at(wa, (rb * 16 * G::SLD + (cb - 1) * 16) * (int)sizeof(T), u32x4_t{s0[0], s1[0], s0[1], s1[1]});
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

        // ---- conv (products over the score tile) -> global ----
        // A product needs taps from registers and an operand from LDS, and a wavefront that waits for each operand where it is used
        // spends far more than the products' own time here.  The reads are therefore issued NLD ahead, from assembly (see
        // lds_read16_at), into a ring of registers; the products of a read are preceded by a wait that leaves exactly the younger
        // operations outstanding.  A quad's products go to NP different groups.  A group's results are taken up LAG reads later, when
        // they are long complete.
        constexpr int NWIN = F_BK / 8;   // groups of eight keys
        constexpr conv_reads plan = G::reads(NWIN);
        constexpr int NREAD = plan.n;
        constexpr int NLD = STATS && D == 128 && R == 6 && !BAND ? 3 : 6, NSLOT = NLD + 3, LAG = 2, NACC = 4;   // (LAST takes dwords of the two operands before it)
        static_assert(NREAD > NLD, "pipeline deeper than the work");
        static_assert(G::LEFT || G::NP + (LAG + G::NQ + G::PAIR - 1) / (G::NQ + G::PAIR) <= NACC, "groups in flight share registers");
        const unsigned row0 = lds_addr(tile) + (unsigned)((pair_row - (R - 1)) * G::SLD * (int)sizeof(T));
        const unsigned xq = row0 + (unsigned)(kg * G::SLD * (int)sizeof(T));                                          // row kg of a quad
        const unsigned xp = row0 + (unsigned)((((kg & 1) + 4 * G::NQ) * G::SLD + (kg >> 1) * 8) * (int)sizeof(T));    // PAIR: rows, chunks
        // LAST: lane groups 0 and 1 read the last row's two chunks, 2 the chunk ahead of them, whose last dword it keeps (3: something)
        const unsigned xl = row0 + (unsigned)(((G::WR - 1) * G::SLD + (kg < 3 ? (kg & 1) - (kg >> 1) : 0) * 8) * (int)sizeof(T));
        u32x4_t ring[NSLOT];
        uint32_t gath[2][4];
        f32x4 cacc[NACC];
        auto issue = [&](auto ic) __attribute__((always_inline)) {
            constexpr int n = decltype(ic)::value, k = plan.kind[n], at = plan.at[n];
            if constexpr (k < G::NQ) {
                ring[n % NSLOT] = lds_read16_at(xq, (4 * k * G::SLD + 8 * at) * (int)sizeof(T));
            } else if constexpr (k == G::KPAIR) {
                ring[n % NSLOT] = lds_read16_at(xp, 8 * at * (int)sizeof(T));
            } else if constexpr (!plan.gathered[n]) {
                ring[n % NSLOT] = lds_read16_at(xl, 8 * at * (int)sizeof(T));
            } else {
                constexpr bool in_side = at == 0;   // (the first group's two columns are not in the tile)
                const unsigned first = in_side ? lds_addr(side) + (unsigned)(pair_row - (R - 1)) * 4 : row0 + 8 * at * (int)sizeof(T) - 4;
                const int row_step = in_side ? 4 : G::SLD * (int)sizeof(T);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 2 * i + (kg & 1) < G::WR ? 2 * i + (kg & 1) : G::WR - 1;
                    gath[at][i] = lds_read4_at(kg < 2 ? xl + 4 * i + 8 * at * (int)sizeof(T) : first + (unsigned)(row * row_step), 0);
                }
            }
        };
        nan = 0.0f;
        uint32_t held[4][2];        // four groups, packed
        // what happens to group w (rows crow, keys j*64 + 8w ..) once it is complete
        auto finish = [&](auto wc) __attribute__((always_inline)) {
            constexpr int w = decltype(wc)::value;
            const f32x4 a = cacc[w % NACC];
            // Groups leave four at a time, exchanged like the scores above and then between the rows of a pair: a lane holds 8
            // consecutive keys of one row and stores them itself, 16 rows x 64 bytes per instruction; no staging through LDS.
            // (Ordinary stores: a 128-byte line is completed by two instructions a few hundred cycles apart, and the L2
            // merges them.  Marked non-temporal, each 64-byte half went to memory on its own and the write counter
            // read 1.38 times the bytes; the price of the merge is that the scores displace some of the head's K blocks
            // from the L2 - at the benchmark shape 541 MB are written and 294 fetched per launch, for 68 MB of Q and K.)
            // (a value that is not finite reaches all results of its products, and each chunk the products of two groups, the last one those of
            // the last group: one of four results of every other group tells)
            if constexpr (w % 2 == 0 || w == NWIN - 1) nan = fmaf(a[0], 0.0f, nan);
            uint32_t lo = pack2<T>(a[0], a[1]), hi = pack2<T>(a[2], a[3]);
            if (!PLAIN && causal && j * F_BK + w * 8 + 7 > pmin) {  // the group touches the diagonal for some row
                const int lane_ = STATS ? opaque_lane(lane) : lane;
                const int col = j * F_BK + w * 8 + (lane_ >> 4 & 1) * 4, crow = q0 - G::HR + wave * (16 * RB) + cshift + 2 * (lane_ & 15) + (lane_ >> 5);   // this lane's row
                if (col > crow) lo &= 0xffff0000u;
                if (col + 1 > crow) lo &= 0x0000ffffu;
                if (col + 2 > crow) hi &= 0xffff0000u;
                if (col + 3 > crow) hi &= 0x0000ffffu;
            }
            held[w & 3][0] = lo;
            held[w & 3][1] = hi;
            if constexpr (w & 1) {   // afterwards: [w-1] keys 0-3, [w] keys 4-7 of group w - 1 + kg%2
                swap16(held[(w & 3) - 1][0], held[w & 3][0]);
                swap16(held[(w & 3) - 1][1], held[w & 3][1]);
            }
            if constexpr ((w & 3) == 3) {   // afterwards: [0], [1] the first row of the pair, [2], [3] the second, group w - 3 + kg
#pragma unroll
                for (int n = 0; n < 4; ++n) swap32(held[n >> 1][n & 1], held[2 + (n >> 1)][n & 1]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int p_ = q0 - G::HR + pair_row + h, col = j * F_BK + (w - 3) * 8 + o_col;
                    const u32x4_t eight = {held[2 * h][0], held[2 * h][1], held[2 * h + 1][0], held[2 * h + 1][1]};
                    if (stored[h] && (PLAIN || (col < S && (!causal || fill_upper || col <= p_))))
                        *reinterpret_cast<u32x4_t *>(o_block + o_off[h] + (w - 3) * 8 * (int)sizeof(T)) = eight;
                    if constexpr (STATS) {
                        if (KB && !BAND ? fresh : w == 3 && j == j_lo) {
                            MTA_KEEP_BRANCH();
                            take(first_ones, plain_tag, h, eight, col, hidden, (w - 3) * 8);
                        } else {
                            take(rest, plain_tag, h, eight, col, hidden, (w - 3) * 8);
                        }
                    }
                }
                if (KB && !BAND && fresh) fresh = __builtin_amdgcn_ballot_w64(row_neg[0] == -NO_SCORE || row_neg[1] == -NO_SCORE) != 0;
            }
        };
        static_for<NLD>(issue);
        static_for<NREAD>([&](auto ic) __attribute__((always_inline)) {
            constexpr int n = decltype(ic)::value, k = plan.kind[n], at = plan.at[n];
            if constexpr (n + NLD < NREAD) issue(std::integral_constant<int, n + NLD>{});
            // LDS operations younger than read n: exactly those of the reads issued after it
            constexpr int younger = plan.ops(n + 1, n + NLD + 1);
            if constexpr (plan.gathered[n]) {
                uint32_t *const g = gath[at];
                lds_wait_upto<(younger < 15 ? younger : 15)>(g[0], g[1], g[2], g[3]);
                ring[n % NSLOT] = u32x4_t{g[0], g[1], g[2], g[3]};
            } else {
                lds_wait_upto<(younger < 15 ? younger : 15)>(ring[n % NSLOT]);
            }
            if constexpr (k < G::NQ) {
                static_for<G::NP>([&](auto pc) __attribute__((always_inline)) {
                    constexpr int c = G::NP - 1 - decltype(pc)::value, w = at - c;   // chunk `at` is chunk c of group w's window
                    if constexpr (w >= 0 && w < NWIN) {
                        if constexpr (c == 0 && k == 0 && !G::LEFT) cacc[w % NACC] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                        mma16(cacc[w % NACC], tz[k * G::NP + c], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
                    }
                });
            } else if constexpr (k == G::KPAIR) {
                mma16(cacc[at % NACC], tz[G::NQ * G::NP], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
            } else {
                if constexpr (!plan.gathered[n]) {   // (read n - 2: the quad of chunk at - 1, n - 1: PAIR of group at - 2)
                    static_assert(plan.kind[n - 1] == G::KPAIR && plan.at[n - 1] == at - 2 && plan.kind[n - 2] == 0 && plan.at[n - 2] == at - 1, "operands in another order");
                    u32x4_t &l = ring[n % NSLOT];
                    uint32_t quad = ring[(n - 2) % NSLOT][3], l0 = l[0];
                    l[1] = upper_half_of(quad, l[1]);
                    l[2] = upper_half_of(ring[(n - 1) % NSLOT][3], l[2]);
                    swap32(l0, quad);   // (the lower half of quad comes to the upper half)
                    l[0] = l0;
                }
                cacc[at % NACC] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};   // (a group's first product)
                mma16(cacc[at % NACC], tz[G::NTZ - 1], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
            }
            __builtin_amdgcn_sched_barrier(0);
            static_for<NWIN>([&](auto wc) __attribute__((always_inline)) {
                if constexpr (plan.last[decltype(wc)::value] + LAG == n) {
                    finish(wc);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
        });
        static_for<NWIN>([&](auto wc) __attribute__((always_inline)) {
            if constexpr (plan.last[decltype(wc)::value] + LAG >= NREAD) finish(wc);
        });
        }
    };
    // A row of a pair meets taps 0 in the window row that only the other one takes, a key of a group in the columns that only others take,
    // and an infinity or a NaN there turns those into NaN.  Results that are NaN are formed again, tap by tap, all others stay the products'
    // own.  A lane reads back the vectors that it has stored and takes eight keys of one row at a time, a window row after the other,
    // until none of its wavefront's sums can become a number any more.  us, all values finite | one row of Q NaN | all of Q (in brackets with
    // all 32 rows of such a block formed again, a key per lane): bf16 6x11 B2 H16 S4096 D128 254 | 527 | 789 (4608 | 14361), fp16 7x7 B1 H16
    // S4096 102 | 464 | 468 (3123 | 6370), bf16 11x15 B1 H16 S2048 D64 39 | 296 | 158 (3417 | 6939), 3x3 B2 H16 S1024 D64 18 | 40 | 63 (65 | 199).
    // Keeping the groups' NaN masks instead of reading back: all of Q 395, 189, 128, 36, but every launch 2 % slower.
    auto form_again = [&](int j) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // the stores come first
        const int lane_ = opaque_lane(lane), key0 = (lane_ >> 4) * 8, first = wave * (16 * RB) + cshift + 2 * (lane_ & 15);   // (rare: nothing of it is kept in registers outside)
        char *const o_block = o_at + (int64_t)j * F_BK * (int)sizeof(T);
        unsigned wanted = 0;             // bit 8n + u: NaN in row n/2 of the pair, key 32 (n%2) + key0 + u
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int col = j * F_BK + (n & 1) * 32 + key0;
            u32x4_t back = {0, 0, 0, 0};
            if (stored[n >> 1] && col < S && (!causal || fill_upper || col <= q0 - G::HR + first + (n >> 1)))
                back = *reinterpret_cast<const u32x4_t *>(o_block + o_off[n >> 1] + (n & 1) * 32 * (int)sizeof(T));
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float a, b;
                unpack2<T>(back[u], a, b);
                wanted |= (a != a ? 1u : 0u) << (8 * n + 2 * u) | (b != b ? 2u : 0u) << (8 * n + 2 * u);
            }
        }
#pragma unroll 1
        for (int n = 0; n < 4; ++n) {
            const unsigned want = wanted >> (8 * n) & 255u;
            if (__builtin_amdgcn_ballot_w64(want != 0) == 0) continue;
            const int q = (n & 1) * 32 + key0, row = first + (n >> 1) - (R - 1);
            float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int i = 0; i < R; ++i) {
                const T *const from = tile + (row + i) * G::SLD + q + G::SHIFT - G::C0, *const ahead = reinterpret_cast<const T *>(side) + (row + i) * 2;
                float x[SK + 7];
#pragma unroll
                for (int e = 0; e < SK + 7; ++e) x[e] = to_float(e < G::C0 - G::SHIFT && q == 0 ? ahead[e] : from[e]);   // (LEFT: two columns of the first group)
#pragma unroll
                for (int t = 0; t < SK; ++t) {
                    const float tap = to_float(Wt[(head * R + i) * SK + t]);
#pragma unroll
                    for (int u = 0; u < 8; ++u) acc[u] = fmaf(tap, x[t + u], acc[u]);
                }
                unsigned open = 0;
#pragma unroll
                for (int u = 0; u < 8; ++u) open |= (acc[u] == acc[u] ? 1u : 0u) << u;
                if (__builtin_amdgcn_ballot_w64((open & want) != 0) == 0) break;
            }
            T *const at = reinterpret_cast<T *>(o_block + (n >> 1 ? o_off[1] : o_off[0])) + (n & 1) * 32;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (want >> u & 1) at[u] = from_float<T>(acc[u]);
        }
    };
    bool again = false;   // STATS: results have been formed again, the statistics are those of what they were
    auto check = [&](int j) __attribute__((always_inline)) {
        if constexpr (!RAW)
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan != nan) != 0, 0)) form_again(j), again = true;
    };
    for (int j = j_lo;;) {  // block(tag, j, K(j), where K(j+1) goes)
        if (plain(j)) block(std::true_type{}, j, B0, B1);
        else block(std::false_type{}, j, B0, B1);
        check(j);
        if (++j > j_end) break;
        if (plain(j)) block(std::true_type{}, j, B1, B0);
        else block(std::false_type{}, j, B1, B0);
        check(j);
        if (++j > j_end) break;
    }

    if constexpr (STATS) {
        const int lane_ = opaque_lane(lane), kg_ = lane_ >> 4, pair = wave * (16 * RB) + cshift + 2 * (lane_ & 15);   // (nothing of it is kept in registers)
        if (!BAND) again = again || __builtin_amdgcn_ballot_w64(!(row_sum[0] < 1e30f) || !(row_sum[1] < 1e30f)) != 0;
        if (__builtin_expect(again, 0)) {   // the statistics of what is stored now, read back
            __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
            for (int h = 0; h < 2; ++h) row_neg[h] = -NO_SCORE, row_sum[h] = 0.0f;
#pragma unroll 1
            for (int j = j_lo; j <= j_end; ++j) {
                const int key = j * F_BK + lane_;
                const uint64_t gone = KB && kb ? __builtin_amdgcn_ballot_w64(kb[key < S ? key : S - 1] == -INFINITY) : 0;
#pragma unroll
                for (int n = 0; n < 4; ++n) {
                    const int h = n >> 1, col = j * F_BK + (n & 1) * 32 + kg_ * 8;
                    if (stored[h] && col < S && col <= q0 - G::HR + pair + h)
                        take(every, std::false_type{}, h, *reinterpret_cast<const u32x4_t *>(o_at + (int64_t)j * F_BK * (int)sizeof(T) + o_off[h] + (n & 1) * 32 * (int)sizeof(T)), col, gone, (n & 1) * 32);
                }
            }
        }
        // the keys of a row lie with four lanes, 16 apart
#pragma unroll
        for (int off = 16; off < 64; off *= 2)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float neg = __shfl_xor(row_neg[h], off), sum = __shfl_xor(row_sum[h], off), least = fminf(neg, row_neg[h]);
                row_sum[h] = row_sum[h] * __builtin_amdgcn_exp2f(least - row_neg[h]) + sum * __builtin_amdgcn_exp2f(least - neg);
                row_neg[h] = least;
            }
        if (kg_ < 2 && (kg_ == 0 ? stored[0] : stored[1]))
            stats_at[q0 - G::HR + pair + kg_] = kg_ == 0 ? make_float2(-row_neg[0], row_sum[0]) : make_float2(-row_neg[1], row_sum[1]);
    }

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
}

template <typename T, int D, int R, int SK, bool BAND, int STATS>
int launch_scores(const conv_attn_args &a)
{
    using G = scores_geom<R, SK>;
    constexpr bool RAW = R == 1 && SK == 1;
    static_assert(G::fits, "no arrangement of the conv's window");
    const int64_t B = a.B, H = a.H, S = a.S;
    const int causal = BAND ? 1 : a.causal, tri_gl = RAW ? 0 : a.tri_gl;
    const int nqb = (int)((S + G::BQ - 1) / G::BQ);
    static_assert(G::BQ == scores_rows(R), "rows of a query block");
    constexpr int jc_len = QK_CHUNK;
    bool table;
    const scores_cut cut = scores_cut_of(B * H, S, R, causal, table);
    int64_t items_per_bh = 0;
    // the items of a head, longest first (the number of key blocks an item visits, as the kernel computes it): long chunks for the first part
    // of a query block's key range, short ones for the rest
    item_table tbl;
    tbl.n = 0;
    constexpr int MAXLEN = 1023;
    static thread_local int count[MAXLEN + 2];
    static thread_local uint32_t items[ITEM_TABLE_MAX];
    static thread_local int lens[ITEM_TABLE_MAX];
    int n = 0;
    for (int qb = 0; qb < nqb; ++qb) {
        const int nk = causal ? scores_key_blocks(qb, G::BQ, (int)S) : (int)((S - 1) / F_BK) + 1, nlong = cut.longs(nk);
        items_per_bh += cut.items(nk);
        if (!table) continue;
        for (int j0 = 0; j0 < nk;) {
            const int len = j0 < nlong ? std::min(cut.big, nlong - j0) : std::min(cut.small, nk - j0);
            lens[n] = len;
            items[n++] = (uint32_t)qb | ((uint32_t)j0 << 11) | ((uint32_t)len << 22);
            j0 += len;
        }
    }
    if (n > 1) {
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
    hipLaunchKernelGGL((conv_scores_mfma<T, D, R, SK, BAND, STATS>), grid, dim3(256), 0, a.st, (const T *)a.q, (const T *)a.k, (const T *)a.w, (T *)a.o,
                       (int)S, (int)(a.rows ? a.rows : S), causal, a.scale, (int)H, nqb, a.fill_upper, (unsigned)total_wg, (unsigned)(B * H), (unsigned)per_xcd, jc_len, tbl, a.band_lo, tri_gl,
                       RAW ? a.qs : row_strides{0, 0, 0}, a.stats);
    return launch_status();
}

// returns 1 when no instantiation covers the kernel size (the caller then uses the general kernel)
template <typename T, int D, bool BAND, int STATS> int dispatch_scores(const conv_attn_args &a)
{
    if constexpr (!STATS)
        if (a.R == 1 && a.Sk == 1) return launch_scores<T, D, 1, 1, BAND, 0>(a);   // no conv (weights are not read)
#define MTA_SCORES_CASE(r, s) \
    if (a.R == r && a.Sk == s) return launch_scores<T, D, r, s, BAND, STATS>(a);
    MTA_SCORES_CASE(3, 3)
    MTA_SCORES_CASE(3, 5)
    MTA_SCORES_CASE(5, 5)
    MTA_SCORES_CASE(5, 7)
    MTA_SCORES_CASE(6, 11)
    MTA_SCORES_CASE(7, 7)
    MTA_SCORES_CASE(7, 9)
    // (the 36 registers of its taps' operands leave three workgroups per CU at D = 64, two at 128)
    MTA_SCORES_CASE(11, 15)
#undef MTA_SCORES_CASE
    return 1;
}
}  // namespace
