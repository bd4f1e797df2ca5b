// The 16-bit kernel of the fused conv-attention (conv_attn_fwd.hip), everything on the matrix cores, and the dispatch to it and to the
// scores kernel: a template over the I/O type; one translation unit per type instantiates it (conv_attn_bf16.hip, conv_attn_f16.hip).
#pragma once

#include "conv_scores_mfma.hpp"

namespace {

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

// The workgroup has NW = 4 wavefronts and owns 128 score rows; two workgroups per CU (three at D = 64 up
// to 7 kernel rows), which overlap each other's barriers and memory latency.  Small grids: NW = 8 with one block of 16 rows each, see launch_attn.
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
// A launch without the scores kernel's table of work items (3 KB of kernel arguments) and an item that is its query block, of which the table's
// search found the number by walking: B1 H32 S8192 D128 970 -> 957, 7x7 B1 H24 S2048 D128 80.9 -> 76.3, 3x3 B1 H32 S1024 D64 28.2 -> 27.0, B1 H4 S100
// 7.8 -> 7.1.  The columns ahead of the first key block from 16 keys instead of a key block (as the scores kernel does): 26.5, 77.9, and on large
// grids 1 % slower (3x3 B1 H32 S4096 D128 238 | 239): not kept.
constexpr int F_SLD = 80;  // score-tile row stride (elements): exactly the retained columns + one key block.  With this one a fragment
                           // read (16 consecutive rows x 64 bytes) is free of bank conflicts as it is: the LDS serves
                           // lanes 0-7 together with lanes 24-31 (8-15 with 16-23, ...), and rows 160 bytes apart put
                           // those on the even and the odd 16-byte positions (measured; 144 or 176 bytes halve the rate)

// the transpose read of 8 bytes
__device__ __forceinline__ u32x2_t lds_read_tr8_at(unsigned addr, int off)
{
    u32x2_t v;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(off) : "memory");
    return v;
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

template <typename T, int D, int R, int SK, int NW>
__global__ __launch_bounds__(64 * NW, 2) void conv_attn_fwd_mfma(const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ V, const T *__restrict__ Wt,
                                                             T *__restrict__ O, float *__restrict__ Lse, int S, int causal, float scale, int H, int nqb,
                                                             unsigned total_wg, unsigned heads)
{
    using G = fused_geom<R, SK>;
    constexpr int F_NT = 64 * NW, F_SR = 128, RB = F_SR / (16 * NW);   // (RB: blocks of 16 rows per wavefront)
    constexpr int CPR = D / 8;                     // 16-byte chunks per K/V row
    constexpr int TILE = F_BK * D;                 // elements per K or V block
    constexpr int ROUNDS = TILE / 8 / F_NT;        // copy instructions per block per lane
    constexpr int KS = D / 32;                     // contraction steps over the head dim
    constexpr int DB = D / 16;                     // 16-wide blocks of the head dim
    constexpr int NCB = F_BK / 16;                 // 16-key blocks per iteration
    static_assert(ROUNDS >= 1, "block smaller than one copy round");

    // K and V rotate through the three buffers of KV: in an iteration K(j) sits in one, V(j) in another; K(j+1) is copied into the third
    // from the top of the iteration on, and V(j+1) into K(j)'s buffer once the score phase is over (the barrier in the middle of the
    // iteration).  Three 16 KB buffers and the score tile are 68 KB: two workgroups per CU.
    __shared__ __align__(256) T KV[3 * TILE];
    __shared__ __align__(16) T Sc[F_SR * F_SLD];                // score tile
    // zero-padded kernel rows, only needed until the Toeplitz fragments are built: they borrow a buffer that
    // receives its first copy after that
    static_assert(R * G::WZ_LD <= TILE, "kernel rows do not fit the borrowed buffer");
    T *const wz = KV + 2 * TILE;

    const int tid = threadIdx.x;
    // (the wavefront index through readfirstlane: everything derived from it is then scalar, branches included)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // Work item = (batch*head, query block), taken rank by rank: the last (longest) query block of every head, then the one before of each,
    // ... - so that the long items all start early (workgroups start in index order as slots free up).  Workgroup ids are dealt
    // round-robin to the 8 XCDs: with heads in multiples of 8 an XCD keeps its own, whose K and V stay in its L2 (of 12 heads an XCD sees
    // 3, of 4 one).  An eighth of the list per XCD, head by head, instead -> this, us, bf16 6x11: B1 H4 S3008 D128 117 -> 117, B1 H12 S2048 D64
    // 66.7 -> 67.2, S3712 D64 152 -> 122, S4096 D128 210 -> 170, B1 H20 S2048 D128 106 -> 88.6.
    // (a 32-bit division: the 64-bit ones that this took were half a microsecond of a workgroup's start)
    const unsigned id = blockIdx.x;
    if (id >= total_wg) return;
    const int item = (int)(id / heads), bh = (int)(id - (unsigned)item * heads);
    const int qb = nqb - 1 - item;
    const int head = (int)((unsigned)bh % (unsigned)H);
    const int q0 = qb * G::BQ;
    const T *Qp = Q + (int64_t)bh * S * D;
    const T *Kp = K + (int64_t)bh * S * D;
    const T *Vp = V + (int64_t)bh * S * D;
    T *Op = O + (int64_t)bh * S * D;

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
    // one key block earlier only fills the retained score columns of the first one's right pad, if there is one
    const int j_start = G::PWR > 0 ? -1 : 0;
    // What the start waits for is asked for at once, this wavefront's rows of Q and the kernel's taps ahead of the first blocks of K and V:
    // behind them, the taps waited for the blocks and Q was asked for when those had come.
    int trow[RB], prow[RB];   // this lane's query rows
    frag8<T> qf[RB][KS];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        trow[rb] = wave * (16 * RB) + rb * 16 + ln;
        prow[rb] = q0 - G::HR + trow[rb];
        const int pc = prow[rb] < 0 ? 0 : (prow[rb] >= S ? S - 1 : prow[rb]);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) qf[rb][ks] = *reinterpret_cast<const frag8<T> *>(Qp + pc * D + ks * 32 + kg * 8);
    }
    constexpr int WZ_IT = (R * G::WZ_LD + F_NT - 1) / F_NT;
    T taps[WZ_IT];
#pragma unroll
    for (int n = 0; n < WZ_IT; ++n) {
        const int e = n * F_NT + tid, i = e / G::WZ_LD, jj = e % G::WZ_LD - G::WZ_OFF;
        taps[n] = Wt[head * R * SK + (i < R && jj >= 0 && jj < SK ? i * SK + jj : 0)];
    }
    asm volatile("" : : : "memory");
    issue_k(j_start, KV);
    issue_v(j_start, KV + TILE);

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
        if (e < R * G::WZ_LD) wz[e] = jj >= 0 && jj < SK ? signed_tap<T>(taps[n], scale) : from_float<T>(0.0f);
    }
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (prow[rb] < 0 || prow[rb] >= S) qf[rb][ks] = zero_frag<T>();  // rows outside the sequence are conv padding
    __syncthreads();

    // Toeplitz fragments T_i^T: accumulator row m = ln, slots k = 8*kg + t, tap = k - SHIFT - m
    frag8<T> tz[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
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
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) cprow[rb] = prow[rb] + cshift;

    auto block = [&](int j, const T *Kb, const T *Vb, T *Kn, T *Vn) __attribute__((always_inline)) {
        const int cbase = j * F_BK + G::PWR;  // first key of the new score block
        // The key block (its scores and its conv outputs) lies inside the sequence and on or below the diagonal for all rows of this
        // wavefront: no masks (most blocks of a long sequence)
        const bool whole = j >= 0 && cbase + F_BK <= S && (!causal || cbase + F_BK - 1 <= pmin);
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
        if (j < j_last) issue_k(j + 1, Kn);  // lands while this block is being worked on

        // ---- S^T = K Q^T, zero above the diagonal / outside the sequence, to the score tile ----
        {
            // Pipelined like the conv phase below: K fragments are read from assembly KLD steps (one 16-key
            // block) ahead into a ring of registers, a step being one fragment and the two products it feeds (both row
            // blocks); a block's scores are rounded, masked and written LAG steps into the next block.
            constexpr int NSTEP = NCB * KS, KLD = KS, KSLOT = KLD + 1, LAG = 2;  // (two blocks ahead spill)
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
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const f32x4 a = sacc[cb & 1][rb];
                    uint32_t lo = pack2<T>(a[0], a[1]), hi = pack2<T>(a[2], a[3]);
                    if (!whole) {
                        MTA_KEEP_BRANCH();
                        const int col = cbase + cb * 16 + kg * 4;
                        const int lim = causal ? (prow[rb] < S - 1 ? prow[rb] : S - 1) : S - 1;  // last key kept
                        if (col < 0 || col > lim) lo &= 0xffff0000u;
                        if (col + 1 < 0 || col + 1 > lim) lo &= 0x0000ffffu;
                        if (col + 2 < 0 || col + 2 > lim) hi &= 0xffff0000u;
                        if (col + 3 < 0 || col + 3 > lim) hi &= 0x0000ffffu;
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
                constexpr int younger = (n + KLD < NSTEP ? n + KLD : NSTEP - 1) - n + score_writes_between(n > KLD ? n - KLD : 0, n, KS, NCB, LAG, RB);
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
        // score tile complete for everybody.  Only the LDS counter is waited for: a fence would also wait for the
        // copy of the next key block, in flight since the top of the iteration
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // nobody reads K(j) any more, the next V block may land in its buffer
        if (j < j_last) issue_v(j + 1, Vn);
        if (j < 0) return;

        // ---- conv (Toeplitz MFMAs over the score tile) -> online softmax ----
        // One product needs one fresh 1 KB score fragment from LDS, and a wavefront that waits for each fragment
        // where it is used spends four times the products' own time here.  The reads are therefore issued NLD
        // products ahead, from assembly (see lds_read16_at), into a ring of registers; every product is preceded by
        // a wait that leaves exactly the younger operations outstanding.  The R products of one output block add into the same
        // registers, each waiting for the one before (two neighbouring blocks worked on in turns: bf16 6x11 B1 H32 S8192 D128 986 | 994 us, D64 B1
        // H8 S2048 66.7 | 67.2, fp16 7x9 D64 B4 H12 93.6 | 93.5, 11x15 D128 B1 H32 S4096 362 | 359).  A block's results are taken up LAG
        // products into the next one, when they are long complete.
        constexpr int NB = RB * NCB, NREAD = NB * R;
        // score fragments in flight (4 and 8 measure the same, and 8 with 7 kernel rows at D = 64 takes the third workgroup of a CU: fp16 7x9
        // B4 H12 S2048 92.7 | 105.4 us)
        constexpr int NLD = 4;
        constexpr int NSLOT = NLD + 1;
        constexpr int LAG = 2;
        static_assert(NREAD > NLD && R >= LAG && NLD <= 15, "pipeline deeper than the work or than the counter");
        const unsigned xa = lds_addr(Sc) + (unsigned)(((trow[0] + cshift - (R - 1)) * F_SLD + kg * 8) * (int)sizeof(T));
        u32x4_t ring[NSLOT];
        f32x4 cacc[2];
        auto issue = [&](auto ic) __attribute__((always_inline)) {
            constexpr int n = decltype(ic)::value;
            constexpr int blk = n / R, i = n % R;   // output block, kernel row
            ring[n % NSLOT] = lds_read16_at(xa, (((blk / NCB) * 16 + i) * F_SLD + (blk % NCB) * 16) * (int)sizeof(T));
        };
        // what happens to output block b = rb*NCB + cb (rows crow[rb], keys j*64 + 16cb ..) once it is complete
        float sv[RB][NCB][4], mloc, mneg[RB];   // a row block's logits, their maximum; minus the running maximum as the exponent takes it
        frag8<T> pf[RB][2];         // probabilities, in the operand layout of the P V products
        auto finish = [&](auto bc) __attribute__((always_inline)) {
            constexpr int b = decltype(bc)::value;
            constexpr int rb = b / NCB, cb = b % NCB;
            const f32x4 a = cacc[b % 2];
            const int p_ = cprow[rb];
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
            constexpr int blk = n / R, i = n % R;
            if constexpr (n + NLD < NREAD) issue(std::integral_constant<int, n + NLD>{});
            // LDS operations younger than read n: exactly the reads issued after it
            constexpr int younger = (n + NLD < NREAD ? n + NLD : NREAD - 1) - n;
            lds_wait_upto<younger>(ring[n % NSLOT]);
            if constexpr (i == 0) cacc[blk % 2] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            mma16(cacc[blk % 2], tz[i], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (blk >= 1 && i == LAG - 1) {
                finish(std::integral_constant<int, blk - 1>{});
                __builtin_amdgcn_sched_barrier(0);
            }
            // the first row block's probabilities, a pair at a time among the second one's products
            if constexpr (RB == 2) {
                constexpr int n0 = NREAD / 2 + LAG - 1, every = (NREAD - 1 - n0) / 8;
                static_assert(every >= 1, "fewer products than pairs");
                if constexpr (n > n0 && (n - n0) % every == 0 && (n - n0) / every <= 8) {
                    probs(std::integral_constant<int, 0>{}, std::integral_constant<int, (n - n0) / every - 1>{});
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        });
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
        finish(std::integral_constant<int, NB - 1>{});
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
    };
    int kb = 0, vb = TILE, nb = 2 * TILE;   // where K(j) and V(j) are, and the third buffer
    for (int j = j_start; j <= j_last; ++j) {
        block(j, KV + kb, KV + vb, KV + nb, KV + kb);
        const int k_next = nb;
        nb = vb;
        vb = kb;
        kb = k_next;
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

template <typename T, int D, int R, int SK>
int launch_attn(const conv_attn_args &a)
{
    using G = fused_geom<R, SK>;
    static_assert(G::fits, "conv window exceeds the 32-key MFMA contraction");
    const int64_t B = a.B, H = a.H, S = a.S;
    const int nqb = (int)((S + G::BQ - 1) / G::BQ);
    // Eight wavefronts of 16 rows instead of four of 32 - the chain of steps that a workgroup is gets a fifth shorter, a CU
    // holds two of these at D = 64 and one at 128 - up to 2 1/4 and 1 3/4 workgroups per CU.  us, four | eight: 6x11 B1 H8 S296 D128 (24
    // workgroups) 19.0 | 15.8, B1 H16 S640 D64 (96) 26.3 | 21.6, D128 32.4 | 27.1, B1 H32 S1300 D64 (352) 49.7 | 41.0, D128 61.9 | 49.6, B1 H24 S2048
    // D128 (432) 91.5 | 78.8, H26 (468) 91.8 | 88.1, H28 (504) 92.0 | 91.9, H32 (576) 94.4 | 103.5, D64 (504) 73.7 | 63.4, (576) 76.0 | 68.2, B2 H60 S600
    // D64 (600) 31.9 | 31.6, B4 H32 S512 (640) 27.7 | 30.6; 3x3, 7x9 and 11x15 alike.
    const bool few = 4 * B * H * nqb <= (D == 64 ? 9 : 7) * (int64_t)device_cu_count();
    auto kern = few ? conv_attn_fwd_mfma<T, D, R, SK, 8> : conv_attn_fwd_mfma<T, D, R, SK, 4>;
    const int64_t total_wg = B * H * nqb;
    if (total_wg > 0x7ffffff0LL) return MTA_ERR_SHAPE;
    hipLaunchKernelGGL(kern, dim3((unsigned)total_wg), dim3(few ? 512 : 256), 0, a.st, (const T *)a.q, (const T *)a.k, (const T *)a.v, (const T *)a.w, (T *)a.o,
                       a.lse, (int)S, a.causal, a.scale, (int)H, nqb, (unsigned)total_wg, (unsigned)(B * H));
    return launch_status();
}

// returns 1 when no instantiation covers the kernel size (the caller then uses the general kernel)
template <typename T, int D> int dispatch_attn(const conv_attn_args &a)
{
#define MTA_FUSED_CASE(r, s) \
    if (a.R == r && a.Sk == s) return launch_attn<T, D, r, s>(a);
    MTA_FUSED_CASE(3, 3)
    MTA_FUSED_CASE(3, 5)
    MTA_FUSED_CASE(5, 5)
    MTA_FUSED_CASE(5, 7)
    MTA_FUSED_CASE(6, 11)
    MTA_FUSED_CASE(7, 7)
    MTA_FUSED_CASE(7, 9)
    // (the 44 registers of its Toeplitz fragments leave two workgroups per CU)
    MTA_FUSED_CASE(11, 15)
#undef MTA_FUSED_CASE
    return 1;
}

template <typename T, int D> int dispatch_mfma_d(const conv_attn_args &a)
{
    if (!a.scores_only) return dispatch_attn<T, D>(a);
    return a.band_lo ? dispatch_scores<T, D, true, 0>(a) : dispatch_scores<T, D, false, 0>(a);
}
template <typename T> int dispatch_mfma_type(const conv_attn_args &a) { return a.D == 64 ? dispatch_mfma_d<T, 64>(a) : dispatch_mfma_d<T, 128>(a); }
}  // namespace
