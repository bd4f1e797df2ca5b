// How the scores kernel (conv_scores_mfma.hpp) cuts the key range of a block of query rows into work items, for it and for the kernel that
// puts the items' row statistics together (softmax_mix_pv.hip).
#pragma once

#include <algorithm>

#include <stdlib.h>

#include "common.hpp"

namespace mta {

constexpr int QK_BK = 64;            // keys per block
constexpr int ITEM_TABLE_MAX = 768;  // a head's items at most, for them to be started from a table

// The first part of a query block's key blocks goes into items of `big` key blocks, about `share` percent of it into items of `small`.
struct scores_cut {
    int big, small, share;
    __host__ __device__ int longs(int nk) const   // key blocks of nk in long items
    {
        const int nshort = (nk * share / 100 + small / 2) / small * small;
        return nk - (nshort < nk ? nshort : nk);
    }
    __host__ __device__ int items(int nk) const
    {
        const int nlong = longs(nk);
        return (nlong + big - 1) / big + (nk - nlong + small - 1) / small;
    }
    __host__ __device__ int index(int nk, int first) const   // of the item that starts with key block `first`
    {
        const int nlong = longs(nk);
        return first < nlong ? first / big : (nlong + big - 1) / big + (first - nlong) / small;
    }
};

// rows of a query block: 128 score rows without the ones that only the conv's window takes
__host__ __device__ constexpr int scores_rows(int R) { return 128 - ((R - 1 + 7) & ~7); }
// key blocks that query block qb sees under the causal rule
__host__ __device__ inline int scores_key_blocks(int qb, int rows, int S)
{
    const int last = qb * rows + rows - 1;
    return (last < S - 1 ? last : S - 1) / QK_BK + 1;
}

// x / n by the reciprocal of n: exact for x below 2^20 (x + 1/2 keeps 1 / 2n away from every multiple, the product is off by 2^-22 of it)
__host__ __device__ inline int quotient(int x, float per_n) { return (int)(((float)x + 0.5f) * per_n); }
// The same numbers where dividing by what is only known at run time costs too much: a row's items, by reciprocals
struct scores_items {
    scores_cut cut;
    int rows;                           // of a query block
    float per_rows, per_big, per_small; // reciprocals of rows, cut.big, cut.small
    scores_items(const scores_cut &c, int r) : cut(c), rows(r), per_rows(1.0f / (float)r), per_big(1.0f / (float)c.big), per_small(1.0f / (float)c.small) {}
    __host__ __device__ int of_row(int p, int S) const   // = cut.items(scores_key_blocks(p / rows, rows, S))
    {
        const int nk = scores_key_blocks(quotient(p, per_rows), rows, S), want = quotient(quotient(nk * cut.share, 0.01f) + cut.small / 2, per_small) * cut.small;
        const int nshort = want < nk ? want : nk;
        return quotient(nk - nshort + cut.big - 1, per_big) + quotient(nshort + cut.small - 1, per_small);
    }
};

constexpr int QK_CHUNK = 32;  // key blocks per work item of the kernel when no item table is built
// with an item table: long and short items (key blocks), and the share of a query block's key range that goes into short
// ones (MTA_QK_CHUNK_LONG / MTA_QK_CHUNK_SHORT / MTA_QK_SHORT_PERCENT in the environment override them, for comparisons)
// (long items measured at B2 H16 S4096 D128: 32/32/0 237 us, 16/16/0 231, 64/16/50 238, 48/24/50 228, 52/26/50 227, 48/24/35 243)
constexpr int QK_SHORT_PERCENT = 50;
// How long the items are, from the launch's key blocks over all heads (768 workgroups are resident).  From 16000 on the grid
// runs in several rounds whatever the length and 48/24 keeps the starts few; below, items as short as it takes to
// have two or three per CU, down to one key block, win although each forms the 16 columns ahead of it again: the grid is
// otherwise a fraction of the chip, each workgroup walking its keys alone.  us, the kernel in a loop, bf16, 48/24 | as short as the rule makes them:
// B1 H8 S256 D64 3x3 (80 blocks) 10.9 | 6.0; B1 H16 S512 D128 5x5 (448) 19.4 | 9.2; B2 H16 S512 D64 6x11 (896) 20.4 | 12.1;
// B4 H16 S512 (1792) 22.1 | 17.9; B1 H8 S2048 D64 (2450) 46.1 | 22.9.
// Where the line lies, 48/24 | 16/8 (two processes a side, which differ by up to 4, at S3712 by 12): B1 H16 S2048 D128 7x7 (5216) 50.4 | 40.0; B1 H32 S2048
// D64 5x5 (10432) 51.0 | 46.8; B2 H16 S2048 D128 6x11 (10432) 70.5 | 71.0; B1 H16 S3072 D128 3x3 (10688) 62.6 | 62.8; B1 H16 S3712 D64 7x9 (15088)
// 79.0 | 75.4; B3 H16 S2048 D128 7x7 (15648) 94.8 | 98.5; B1 H16 S4096 D128 7x7 (19104) 116.5 | 117.2; B4 H16 S2048 D64 3x3 (20864) 85.0 | 89.8; B2 H16
// S3072 D128 6x11 (21376) 144 | 143; B2 H16 S4096 D128 6x11 (38208) 238 | 250.
inline scores_cut scores_cut_rule(int64_t blocks, int64_t head_blocks, int nqb, int share)
{
    if (blocks >= 16000) return {48, 24, share};
    if (blocks < 600) return {1, 1, share};
    int small = (int)std::min<int64_t>(std::max<int64_t>((blocks + 400) / 800, 1), 8);
    while (head_blocks / small + 2 * nqb > ITEM_TABLE_MAX && small < 24) small *= 2;   // (the table holds one head's items)
    return {2 * small, small, share};
}
// A launch's cut; table: whether a head's items fit the table (else they are QK_CHUNK key blocks each).
inline scores_cut scores_cut_of(int64_t heads, int64_t S, int R, bool causal, bool &table)
{
    constexpr int MAXLEN = 1023;
    static const int env_big = [] { const char *e = getenv("MTA_QK_CHUNK_LONG"); return e ? atoi(e) : 0; }();
    static const int env_small = [] { const char *e = getenv("MTA_QK_CHUNK_SHORT"); return e ? atoi(e) : 0; }();
    static const int share = [] { const char *e = getenv("MTA_QK_SHORT_PERCENT"); return e ? atoi(e) : QK_SHORT_PERCENT; }();
    const int rows = scores_rows(R), nqb = (int)((S + rows - 1) / rows), all = (int)((S + QK_BK - 1) / QK_BK);
    int64_t head_blocks = 0;
    for (int qb = 0; qb < nqb; ++qb) head_blocks += causal ? scores_key_blocks(qb, rows, (int)S) : all;
    scores_cut cut = scores_cut_rule(heads * head_blocks, head_blocks, nqb, share);
    if (env_big) cut.big = env_big;
    if (env_small) cut.small = env_small;
    table = nqb <= 2047 && all <= 2047 && cut.big >= 1 && cut.small >= 1 && cut.big <= MAXLEN && cut.small <= MAXLEN && share >= 0 && share <= 100;
    int items = 0;
    for (int qb = 0; qb < nqb && table; ++qb) {
        items += cut.items(causal ? scores_key_blocks(qb, rows, (int)S) : all);
        table = items <= ITEM_TABLE_MAX;
    }
    return table ? cut : scores_cut{QK_CHUNK, QK_CHUNK, 0};
}

// items of a query block, at most (causal: later blocks see more keys; a longer row is not always more items)
inline int scores_slots(int64_t S, int R, const scores_cut &cut)
{
    const int rows = scores_rows(R), nqb = (int)((S + rows - 1) / rows);
    int most = 0;
    for (int qb = 0; qb < nqb; ++qb) most = std::max(most, cut.items(scores_key_blocks(qb, rows, (int)S)));
    return most;
}

// Row statistics that a scores kernel leaves for the softmax behind it, [batch * head][item of the row's query block][row]: a reference r in
// powers of two (the maximum of some of the item's scores times log2(e)) and the sum of exp2(score log2(e) - r) over the item's scores.
constexpr float NO_SCORE = -3.3e38f;   // the reference of no score at all (a number: differences of two are 0)
struct scores_stats {
    float2 *at;              // NULL: none
    const float *key_bias;   // (B,S) or NULL: 0, or -inf for a key that no row sees
    int slots;               // items of a query block, at most
    scores_cut cut;
};

}  // namespace mta
