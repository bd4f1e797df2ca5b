// The depthwise causal conv on the matrix cores: strips of a plane in LDS, Toeplitz fragments of the channel's kernel, and with DW the
// kernel gradient in the same pass (conv2d_causal.hip, conv2d_grads.hip).
#pragma once

#include "common.hpp"
#include "mfma.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

// ------------------------------------------------------------------------------------
// MFMA (Toeplitz) path
// ------------------------------------------------------------------------------------
// The output is written once and not read again by this kernel: for large tensors non-temporal stores keep it from displacing
// the input rows that neighbouring strips re-read (halos) in the L2.
#define MTA_CONV_STORE(ptr, val) store_out((ptr), (val), STREAM)

constexpr int M_NW = 4;            // wavefronts per workgroup, each with 16 rows x 128 keys of the workgroup's strip
constexpr int M_WT = 64 * M_NW;    // threads per workgroup
constexpr int M_HALF = 128;        // keys per wavefront: 8 column blocks of 16
constexpr int M_TURN = 5;          // DW: a workgroup's place within a round of items moves on by so much
// A strip: 64 rows x 128 keys (NARROW) or 32 x 256; which one, see narrow_strips()
template <bool NARROW> struct strip_geom {
    static constexpr int TM = NARROW ? 64 : 32, TN = NARROW ? 128 : 256;
    static constexpr int RB = TM / 16;     // row blocks of 16
    static constexpr int RPB = TN / TM;    // row strips per TN x TN block of the lower triangle
    static_assert(RB * (TN / M_HALF) == M_NW, "a wavefront for each 16 x 128 outputs");
};
// Persistent workgroups per CU: four, as long as two strip buffers take a quarter of the LDS (five copy rounds, 20 KB) and a
// wavefront 128 registers; three for wide strips of more than 6 kernel rows, and for more than 7.  They are what hides the latency:
// the kernel of 6 x 11 over the lower triangle of B1 H16 S2048 fp16 took 41.6, 39.9, 33.7 us with two, three, four (from cache).
template <int R, bool NARROW, bool DW = false> constexpr int wg_per_cu() { return DW ? 2 : R > (NARROW ? 7 : 6) ? 3 : 4; }

// 16 outputs + S-1 taps (+ alignment shift) must fit the 32-key contraction of one 16x16x32 MFMA
template <int R, int S, bool NARROW> struct mfma_geom : strip_geom<NARROW> {
    using strip_geom<NARROW>::TM;
    using strip_geom<NARROW>::TN;
    static constexpr int PADW = (S - 1) / 2;
    static constexpr int HL = (PADW + 7) & ~7;             // left halo, rounded so 16-byte loads stay aligned
    static constexpr int SHIFT = HL - PADW;                // first tap's offset inside a block's 32-key window
    static constexpr bool fits = SHIFT + 16 + S - 1 <= 32;
    static constexpr int TW = TN - 16 + 32;                // staged columns
    // Row stride in LDS.  A fragment read takes 16 bytes per lane from 16 consecutive rows (lane group kg at byte offset
    // 16 kg); the LDS serves lanes 0-7 together with lanes 24-31 (8-15 with 16-23, ...), i.e. rows 0-7 at one offset with
    // rows 8-15 at the next: with a stride of 2 (mod 8) 16-byte slots those sixteen accesses fall on sixteen different
    // slots of the 256-byte bank line (3 (mod 8), one padding slot after the data, put rows 3 and 8 on the same one).
    static constexpr int LD = TW;
    static_assert((LD / 8) % 8 == 2, "row stride of the staged strip");
    static constexpr int ROWS = TM + R - 1;
    // Where a wavefront's results wait in LDS.  NARROW: in its own row block, once every wavefront has read its input.  Else the
    // results of key half `h` go back to LDS columns h * RES_OFF .. + M_HALF - 1 of rows that the other row block does not read,
    // which no wavefront of the other half reads as input (half 0 reads columns 0 .. M_HALF+15, half 1 columns M_HALF ..).
    static constexpr int RES_OFF = M_HALF + 16;
    static_assert(NARROW || RES_OFF + M_HALF <= LD, "result columns of the second half");
};

// Position t of a work item inside its plane -> (strip row tm (TM rows), strip col tn (TN keys)).
// `tri` (causal, square, lower triangle only): the strips that touch the lower triangle, row strip by row strip from
// the top, each from the left up to the diagonal: row strip tm has tm / RPB + 1 of them, so RPB/2 * b * (b+1) items
// precede block row b.  Otherwise: all strips, row-major.
template <bool NARROW> __device__ __forceinline__ void decode_item(int t, int tiles_n, int tri, int &tm, int &tn)
{
    if (tri) {
        constexpr int RPB = strip_geom<NARROW>::RPB, HB = RPB / 2;
        static_assert(RPB % 2 == 0, "row strips per block row");
        int b = (int)((sqrtf((float)t / (float)HB + 0.25f) - 0.5f));
        while (HB * (b + 1) * (b + 2) <= t) ++b;
        while (HB * b * (b + 1) > t) --b;
        const int rem = t - HB * b * (b + 1);
        tm = b * RPB + rem / (b + 1);
        tn = rem % (b + 1);
    } else {
        tm = t / tiles_n;
        tn = t % tiles_n;
    }
}

// +0 over a TM x TN region (of strips that write whole rows), all threads of the workgroup.  FULL: the region lies inside the tensor; the stores are
// then unconditional (exactly TM*TN/8/M_WT vector-memory instructions per lane)
template <typename T, bool NARROW, bool STREAM, bool FULL = false>
__device__ __forceinline__ void zero_fill_strip(T *yp, int H, int W, int p0, int q0, int tid)
{
    constexpr int M_TM = strip_geom<NARROW>::TM, M_TN = strip_geom<NARROW>::TN;
    constexpr int VEC = 8, VPRW = M_TN / VEC, RPP = M_WT / VPRW;  // vectors per row, rows per pass
    pack16<T> z;
#pragma unroll
    for (int u = 0; u < VEC; ++u) z.v[u] = from_float<T>(0.0f);
    tid = opaque(tid);
    // thread t covers rows t/VPRW + RPP*k, vector t%VPRW: a uniform base, one 32-bit per-lane byte offset, uniform row steps
    static_assert(M_WT % VPRW == 0 && M_TM % RPP == 0, "region rows per pass");
    char *base = reinterpret_cast<char *>(yp + (int64_t)p0 * W + q0);
    const int r0 = tid / VPRW, cv = (tid % VPRW) * VEC;
    const unsigned off = (unsigned)(r0 * W + cv) * (unsigned)sizeof(T);
    const int64_t rstep = (int64_t)RPP * W * (int64_t)sizeof(T);
#pragma unroll
    for (int k = 0; k < M_TM / RPP; ++k) {
        if (FULL || (p0 + r0 + k * RPP < H && q0 + cv < W))
            MTA_CONV_STORE(reinterpret_cast<u32x4 *>(base + k * rstep + off), __builtin_bit_cast(u32x4, z));
    }
}

// Persistent four-wavefront workgroups: each walks a run of M_TM x M_TN strips dealt round-robin within its XCD's share
// of the item list.  A wavefront owns a row block of 16 rows and 128 keys of the strip: it issues a quarter of the staging
// copies and computes its 16 x 128 outputs.  The wavefronts meet at two barriers per strip (the strip has landed and the
// previous strip's buffer may be overwritten; the strip is no longer needed as input, or the results are in LDS); latency is
// hidden by the other workgroups resident on the CU, each in its own phase (loading / matrix cores / storing) with its own
// two LDS strip buffers of (M_TM + R - 1) rows x (M_TN + 16) keys.
//
// Item order.  Strips are taken row strip by row strip, each from the left, so that an XCD's workgroups sweep whole
// rows of the output together, zero strips included: under the causal rule a strip wholly above the diagonal is an
// item like the others, whose workgroup stores +0 over it (no copy, no products).  Written this way - every row of the
// output completed within a short time - the tensor moves through memory a tenth faster than with strips taken block by
// block and the part above the diagonal filled by workgroups of their own.  Odd planes are walked backwards, so that a workgroup's share alternates between the cheap strips above the
// diagonal and the others.  MTA_CAUSAL_LOWER_ONLY on a square tensor enumerates the strips that touch the lower
// triangle only.
//
// Per 16x16 output block and kernel row i:  out^T[q, p] += T_i^T[q, k] X^T[k, p+i-(R-1)], one
// v_mfma_f32_16x16x32 whose 32-key contraction window holds the 16 outputs' taps.  A operand =
// Toeplitz fragment (4 VGPRs per kernel row, kept while the channel is unchanged), B operand = 16 contiguous
// bytes of one staged row per lane.  A wavefront sustains about one such 1 KB LDS operand per 35 cycles whatever the
// addresses, against 16 cycles for the product: the products of a strip are therefore split over four wavefronts (on
// four SIMDs).  Results go back through LDS rows that are no longer needed as input.  NARROW: after a barrier a wavefront
// writes its row block's own 16 rows and stores them, four 256-byte rows per instruction.  Else row block 0 takes the
// strip's first 16 staged rows, row block 1 the last 16 of its window (see mfma_geom::RES_OFF for the columns); after a
// barrier wavefront w stores strip rows 8w .. 8w+7 whole, two 512-byte rows per instruction.
//
// Staging.  A strip whose halo lies wholly inside the tensor and on or below the diagonal (the common case, decided per
// workgroup) is copied global -> LDS by global_load_lds_dwordx4: no registers, no masks, no LDS store instructions.
// The LDS row stride is 34 or 18 16-byte slots (see mfma_geom::LD), and thread t of copy round `it` owns slot it*256+t.  Any
// other strip is copied slot by slot under a predicate - a slot inside the plane and on or below the diagonal is
// copied, any other is written as zeros while the buffer waits for its data - and after landing only the one vector
// per row that straddles the diagonal is masked in LDS.  Nothing is read from outside the tensor.
//
// Kernel rows.  The channel's R*S taps are copied global -> LDS the same way, one strip ahead, as the dwords that hold
// them (from the 4-byte aligned address at or below the first tap: such a dword holds at least one tap, so it lies in
// mapped memory); the copy is older than the strip's, so the wait for the strip covers it, and no register carries a
// value that is still in flight.  The Toeplitz fragments are gathered from there when the channel changes.
//
// SCALED: every strip is staged through registers, where x*in_scale is rounded to the I/O dtype before it
// reaches LDS (what a separate elementwise scale pass would have produced).
//
// BWD: the gradient with respect to the input (see conv2d_valu): kernel rows reversed in both axes, the R-1 halo rows
// below the strip instead of above it.  Key sizes are odd here, so the key halos are the same on both sides.
// DW: the input gradient (x: dy) together with the kernel gradient, whose other operand is `xin`.  Alone the two read dy twice and move
// four tensors where three do, and the kernel gradient alone keeps the vector ALU busy shifting its operands.  A strip brings its own
// 64 x 128 positions of xin with it; dy with its halo is in LDS anyway.  The kernel gradient's products contract over 32 rows: both
// operands are transpose reads, the row offset is an address, and all key offsets of 16 x 16 keys come out of one product - 2 R products
// per 512 positions, and 2 R accumulators that live in registers for the whole kernel (with the keys as contraction index, as in
// conv2d_bwd_weight.hip, 2 S of both and a shift in registers for each).  So a workgroup stays with one channel; it walks every
// nw-th strip of its planes, its place in the round moving on by M_TURN so that nobody gets only the strips at the left, and leaves one
// partial kernel.  y may be xin: a strip of xin is read by its own workgroup only, and is in LDS before the strip of y is written.
// Strips wholly above the diagonal are no items here: each strip of a row takes its share of them.  2 workgroups per CU
// (LDS: two buffers of 36 KB); what bounds it is memory.  us with the sum of the partial kernels, the two kernels -> this, bf16,
// nothing in the caches: whole rows 6x11 B2 H16 S2048 146 -> 121 (537 MB, 110 at the rate of a copy; keys as contraction index 130),
// 11x15 B1 H16 S2048 97 -> 73; lower triangle 7x7 B1 H16 S2048 72 -> 58, 5x7 B1 H32 S2048 121 -> 103, 6x11 S1024 34.4 -> 27.3,
// 11x15 S1024 41.9 -> 33.4, 7x9 B4 H12 S640 44.5 -> 37.5, 3x3 B1 H12 S1000 29.3 -> 22.1.
template <typename T, int R, int S, bool SCALED, bool BWD, bool STREAM, bool NARROW, bool DW = false>
__global__ __launch_bounds__(M_WT, (wg_per_cu<R, NARROW, DW>())) void conv2d_mfma(
    const T *__restrict__ x, const T *__restrict__ w, T *y, int C, int H, int W, int causal, float in_scale,
    int tiles_n, int ipp, int64_t total, int64_t per_xcd, int nw, int tri, const T *xin, float *__restrict__ partial)
{
    static_assert(!DW || (BWD && NARROW), "the kernel gradient comes with the input gradient, over strips of 64 x 128");
    using G = mfma_geom<R, S, NARROW>;
    constexpr int M_TM = G::TM, M_TN = G::TN;
    static_assert(!BWD || (S % 2 == 1 && !SCALED), "the backward instance assumes symmetric key halos and no scale");
    static_assert(sizeof(T) == 2, "16-bit data");
    constexpr int TOP = BWD ? 0 : R - 1;                    // halo rows above the strip (the others lie below it)
    constexpr int LD = G::LD, VEC = 8;
    constexpr int VPR = G::TW / VEC;                        // data vectors per staged row (34 or 18)
    constexpr int SPR = LD / VEC;                           // 16-byte slots per LDS row
    constexpr int SLOTS = G::ROWS * SPR;
    constexpr int STAGE_IT = (SLOTS + M_WT - 1) / M_WT;     // copies per strip and lane (the last round may be partial)
    static_assert(SPR == VPR, "no padding slots");
    // the channel's kernel as it lies in memory (see above) travels with its strip: behind the strip's last slot
    constexpr int WRAW_DW = (R * S + 2) / 2;                 // dwords that cover R*S taps starting in either half of the first
    constexpr int WRAW_IT = (WRAW_DW + 63) / 64;
    constexpr int WRAW_SLOT = (SLOTS + 3) & ~3;              // (64-byte aligned)
    constexpr int NEED_SLOTS = WRAW_SLOT + WRAW_IT * 16;     // (a copy instruction of the kernel rows covers 16 slots)
    constexpr int BUF_SLOTS = NEED_SLOTS > STAGE_IT * M_WT ? (NEED_SLOTS + 15) / 16 * 16 : STAGE_IT * M_WT;
    constexpr int BUF = BUF_SLOTS * VEC;                     // elements per LDS strip buffer
    // DW: behind it x over the strip's own positions, a wavefront's 16 rows after the other; 16-byte piece c of row r at c ^ 2 (r % 8):
    // a transpose read takes 32 bytes of 8 consecutive rows at a time, which lie in different banks then
    constexpr int XBUF = DW ? 16 * M_HALF : 0;               // elements per wavefront
    constexpr int BUFX = BUF + M_NW * XBUF;
    static_assert(!DW || (BUF * sizeof(T) % 256 == 0 && BUFX * sizeof(T) % 256 == 0), "the exclusive or on an address of x is one on its place in 256 bytes");
    __shared__ __align__(256) T tiles[2 * BUFX];              // double buffer: strip n is computed while strip n+1 lands
    using V16 = pack16<T>;

    // XCD-aware split: workgroup ids are dealt round-robin to the 8 XCDs; each XCD gets one
    // contiguous chunk of the item list (whole planes, mostly), so halo re-reads stay in its L2.
    const int64_t c0 = DW ? 0 : (int64_t)(blockIdx.x & 7) * per_xcd;
    const int64_t c1 = (c0 + per_xcd < total) ? c0 + per_xcd : total;
    // within the chunk the items are dealt round-robin to the XCD's workgroups, so that at any moment
    // they sweep the same few hundred rows together (DRAM pages are consumed whole, as by a linear copy)
    const unsigned vb = DW ? (blockIdx.x & 7) * ((unsigned)per_xcd) + (blockIdx.x >> 3) : 0u;
    const int channel0 = DW ? (int)(vb / (unsigned)nw) : 0;
    int sub = DW ? (int)(vb - (unsigned)channel0 * (unsigned)nw) : 0;
    if (DW && channel0 >= C) return;
    const int64_t first = DW ? (int64_t)sub : c0 + (int64_t)(blockIdx.x >> 3);
    const int64_t last = c1;
    const int step = nw;
    if (!DW && (c0 >= total || first >= last)) return;
    int n_items;
    if constexpr (DW) {
        const unsigned all = (unsigned)total, rounds = all / (unsigned)nw;
        n_items = (int)rounds + (((unsigned)sub + rounds % (unsigned)nw * M_TURN) % (unsigned)nw < all - rounds * (unsigned)nw ? 1 : 0);
    } else {
        n_items = (int)((last - first + step - 1) / step);
    }
    const int64_t HW = (int64_t)H * W, plane_step = DW ? C * HW : HW;

    const int tid = threadIdx.x, lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // (the wavefront index through readfirstlane: everything derived from it is then scalar)
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb0 = (wave % G::RB) * 16;     // first strip row of this wavefront's row block
    const int ch = wave / G::RB;             // its key half
    frag8<T> tz[R];
    int cur_channel = -1;
    const bool reflect = !DW && causal != 0 && !tri;  // odd planes backwards

    // per-thread geometry of the staging copies, fixed for the whole kernel: slot it*M_WT+tid is row srow,
    // vector svc of the strip; padding slots re-read a neighbouring valid vector
    unsigned goff[STAGE_IT];  // byte offsets from the strip's first staged element (uniform base + 32-bit lane offset)
#pragma unroll
    for (int it = 0; it < STAGE_IT; ++it) {
        const int slot = it * M_WT + tid;
        int rr = slot / SPR, vc = slot % SPR;
        if (rr >= G::ROWS) { rr = 0; vc = 0; }
        if (vc >= VPR) vc = VPR - 1;
        goff[it] = (unsigned)(rr * W + vc * VEC) * (unsigned)sizeof(T);
    }

    // a strip is `interior` when its whole halo lies inside the tensor and on or below the diagonal
    auto is_interior = [&](int p0_, int q0_) {
        if (SCALED) return false;
        const int h0 = p0_ - TOP, k0 = q0_ - G::HL;
        return h0 >= 0 && h0 + G::ROWS <= H && k0 >= 0 && k0 + G::TW <= W && (!causal || k0 + G::TW - 1 <= h0);
    };
    // (a plane is named by the offset of its first element, `pbase`: kept up to date by additions, no 64-bit divisions)
    // 0: a strip to convolve, 1: wholly above the diagonal, +0 to be stored, 2: wholly above it, nothing to do
    auto kind_of = [&](int p0_, int q0_) { return (!DW && causal && q0_ > p0_ + M_TM - 1) ? (causal == 2 ? 2 : 1) : 0; };
    // Asynchronous copy of a strip into LDS buffer `buf` (this wavefront's quarter of the slots).  Interior strip: every
    // slot is copied.  Any other strip: a slot is copied only if it lies inside the plane and on or below the diagonal;
    // the others - what lies outside the plane (borders), above the diagonal (which is then not read from memory at
    // all), and the padding slots - are written as zeros right here, while the buffer is still waiting for its data.
    // What remains to be done once the copy has landed is the one vector of a row that straddles the diagonal.
    auto slot_valid = [&](int slot, int h0_, int k0_) {
        const int rr = slot / SPR, vc = slot % SPR;
        const int h = h0_ + rr, col = k0_ + vc * VEC;
        return rr < G::ROWS && vc < VPR && h >= 0 && h < H && col >= 0 && col < W && !(causal && col > h);
    };
    auto prefetch = [&](int64_t pbase_, int p0_, int q0_, T *buf, bool interior_) {
        const char *base = reinterpret_cast<const char *>(x) +
                           (pbase_ + (int64_t)(p0_ - TOP) * W + (q0_ - G::HL)) * (int64_t)sizeof(T);
        if (interior_) {
#pragma unroll
            for (int it = 0; it < STAGE_IT; ++it)
                if ((it + 1) * M_WT <= SLOTS || it * M_WT + tid < SLOTS)
                    __builtin_amdgcn_global_load_lds((glb_void_t *)(base + goff[it]),
                                                     (lds_void_t *)(buf + (it * M_WT + wave * 64) * VEC), 16, 0, 0);
        } else {
            const int tid_ = opaque(tid);
            const int h0_ = p0_ - TOP, k0_ = q0_ - G::HL;
            const unsigned buf_lds = (unsigned)(uintptr_t)(lds_void_t *)buf;
            const u32x4 zero4 = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int it = 0; it < STAGE_IT; ++it) {
                const int slot = it * M_WT + tid_;
                if (slot_valid(slot, h0_, k0_))
                    __builtin_amdgcn_global_load_lds((glb_void_t *)(base + goff[it]),
                                                     (lds_void_t *)(buf + (it * M_WT + wave * 64) * VEC), 16, 0, 0);
                else if (slot < SLOTS)
                    lds_store16(buf_lds + (unsigned)slot * 16u, zero4);
            }
        }
    };
    // asynchronous copy of a channel's kernel into the spare slots of strip buffer `par` (first wavefront); the taps start
    // wshift(channel) 16-bit elements into them
    auto wshift = [&](int channel_) { return (int)((reinterpret_cast<uintptr_t>(w + (int64_t)channel_ * (R * S)) >> 1) & 1u); };
    auto fetch_weights = [&](int channel_, int par) {
        if (wave != 0) return;
        const uintptr_t a0 = reinterpret_cast<uintptr_t>(w + (int64_t)channel_ * (R * S));
        const char *base = reinterpret_cast<const char *>(a0 & ~(uintptr_t)3);
        const int ndw = ((int)((a0 >> 1) & 1u) + R * S + 1) / 2;  // dwords that hold a tap (at most WRAW_DW)
#pragma unroll
        for (int k = 0; k < WRAW_IT; ++k)
            if (k * 64 + lane < ndw)
                __builtin_amdgcn_global_load_lds((glb_void_t *)(base + (k * 64 + lane) * 4),
                                                 (lds_void_t *)(tiles + par * BUFX + (WRAW_SLOT + k * 16) * VEC), 4, 0, 0);
    };
    // current and next work item: position inside the plane, plane (as element offset, and its parity) and channel
    int t_nx;
    int64_t pbase_nx;
    int chan_nx, podd_nx;
    {
        const int64_t plane0 = DW ? (unsigned)first / (unsigned)ipp : first / ipp;
        t_nx = (int)(first - plane0 * ipp);
        pbase_nx = plane0 * plane_step + channel0 * HW;
        chan_nx = DW ? channel0 : (int)(plane0 % C);
        podd_nx = (int)(plane0 & 1);
    }
    // DW: asynchronous copy of this wavefront's inputs; a piece that is masked as a whole reads the start of the plane instead
    auto fetch_x = [&](int64_t pbase_, int p0_, int q0_, T *buf, bool interior_) {
        if constexpr (DW) {
            const int lane_ = opaque(lane), r_ = lane_ >> 4;
            const char *plane = reinterpret_cast<const char *>(xin + pbase_);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int row = 4 * k + r_, h = p0_ + rb0 + row, col = q0_ + ch * M_HALF + (((lane_ & 15) ^ (row & 7) * 2) * VEC);
                const bool ok = interior_ || (h < H && col < W && !(causal && col > h));
                __builtin_amdgcn_global_load_lds((glb_void_t *)(plane + (ok ? (size_t)(unsigned)(h * W + col) * sizeof(T) : (size_t)0)),
                                                 (lds_void_t *)(buf + BUF + wave * XBUF + k * 4 * M_HALF), 16, 0, 0);
            }
        }
    };
    f32x4 dwacc[DW ? R : 1][2];
    if constexpr (DW) {
#pragma unroll
        for (int u = 0; u < R; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) dwacc[u][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    int tm = 0, tn = 0;
    if (n_items > 0) {
    decode_item<NARROW>((reflect && podd_nx) ? ipp - 1 - t_nx : t_nx, tiles_n, tri, tm, tn);
    if (kind_of(tm * M_TM, tn * M_TN) == 0) {
        fetch_weights(chan_nx, 0);
        if (!SCALED) prefetch(pbase_nx, tm * M_TM, tn * M_TN, tiles, is_interior(tm * M_TM, tn * M_TN));
        fetch_x(pbase_nx, tm * M_TM, tn * M_TN, tiles, is_interior(tm * M_TM, tn * M_TN));
    }
    }

    constexpr int ST = 16 * (M_HALF / VEC) / 64;  // stores per strip and lane (a wavefront's 16 x 128 outputs) ...
    static_assert(ST == M_TM * (M_TN / VEC) / M_WT && ST == 4, "... and per zero strip");
    int younger = -1;                      // stores certainly issued after the copy in flight (-1: unknown)
    int parity = 0;
    for (int item = 0; item < n_items; ++item, parity ^= 1) {
        T *tile = tiles + parity * BUFX;
        T *other = tiles + (parity ^ 1) * BUFX;
        const int p0 = tm * M_TM, q0 = tn * M_TN;
        const int64_t pbase = pbase_nx;
        const T *xp = x + pbase;
        T *yp = y + pbase;
        const int channel = chan_nx;
        const int kind = kind_of(p0, q0);
        const bool interior = kind == 0 && is_interior(p0, q0);
        const int h0 = p0 - TOP, k0 = q0 - G::HL;
        // the strip's outputs all lie inside the tensor: its stores are unconditional then, and their number is known
        const bool full_out = p0 + M_TM <= H && q0 + M_TN <= W;
        // (opaque: the addresses derived from it are then formed where they are used instead of being kept, dozens of
        // them, in registers across the loop)
        const unsigned tile_lds = (unsigned)opaque((int)(unsigned)(uintptr_t)(lds_void_t *)tile);

        // This wavefront's part of the strip's copy (if any) and of its kernel rows has landed.  Vector-memory operations
        // complete in issue order, and the only ones this wavefront issued after that copy are the previous strip's
        // stores: when their number is known exactly (`younger`), they may stay in flight.
        if (younger == ST) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(ST) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        younger = 0;

        if (!SCALED && kind == 0 && !interior && causal && k0 + G::TW - 1 > h0) {
            // the copy has landed: in the one vector of a row that straddles the diagonal, zero the keys beyond it (all
            // reads first, one wait, then the writes)
            const int tid_ = opaque(tid);
            constexpr int GRP = 3;  // slots per batch (each holds four registers between its read and its write)
#pragma unroll
            for (int g0 = 0; g0 < STAGE_IT; g0 += GRP) {
                u32x4 raw[GRP];
#pragma unroll
                for (int it = g0; it < g0 + GRP && it < STAGE_IT; ++it) {
                    const int slot = it * M_WT + tid_;
                    const int h = h0 + slot / SPR, col = k0 + (slot % SPR) * VEC;
                    if (slot_valid(slot, h0, k0) && col + VEC - 1 > h) raw[it - g0] = lds_load16(tile_lds + (unsigned)slot * 16u);
                }
                lds_wait();
#pragma unroll
                for (int it = g0; it < g0 + GRP && it < STAGE_IT; ++it) {
                    const int slot = it * M_WT + tid_;
                    const int h = h0 + slot / SPR, col = k0 + (slot % SPR) * VEC;
                    if (slot_valid(slot, h0, k0) && col + VEC - 1 > h) {
                        asm volatile("" : "+v"(raw[it - g0]));  // (the value is defined from the wait above on)
                        V16 v = __builtin_bit_cast(V16, raw[it - g0]);
#pragma unroll
                        for (int u = 0; u < VEC; ++u)
                            if (col + u > h) v.v[u] = from_float<T>(0.0f);
                        lds_store16(tile_lds + (unsigned)slot * 16u, __builtin_bit_cast(u32x4, v));
                    }
                }
            }
        } else if (SCALED && kind == 0) {
            // through registers.  Loads are unconditional and issued back to back (an invalid
            // slot re-reads a valid address); what a slot really holds is decided on the way to LDS
            V16 stage[STAGE_IT];
            const int tid_ = opaque(tid);
#pragma unroll
            for (int it = 0; it < STAGE_IT; ++it) {
                const int slot = it * M_WT + tid_;
                const int rr = slot / SPR, vc = slot % SPR;
                const int h = h0 + rr, col = k0 + vc * VEC;
                stage[it] = *reinterpret_cast<const V16 *>(xp + (slot_valid(slot, h0, k0) ? (int64_t)h * W + col : 0));
            }
#pragma unroll
            for (int it = 0; it < STAGE_IT; ++it) {
                const int slot = it * M_WT + tid_;
                const int rr = slot / SPR, vc = slot % SPR;
                const int h = h0 + rr, col = k0 + vc * VEC;
                const bool ok = slot_valid(slot, h0, k0);
                V16 v = stage[it];
#pragma unroll
                for (int u = 0; u < VEC; ++u) v.v[u] = from_float<T>(to_float(v.v[u]) * in_scale);
                if (!ok) {
#pragma unroll
                    for (int u = 0; u < VEC; ++u) v.v[u] = from_float<T>(0.0f);
                } else if (causal && col + VEC - 1 > h) {  // the one vector of a row that straddles the diagonal
#pragma unroll
                    for (int u = 0; u < VEC; ++u)
                        if (col + u > h) v.v[u] = from_float<T>(0.0f);
                }
                if (slot < SLOTS) lds_store16(tile_lds + (unsigned)slot * 16u, __builtin_bit_cast(u32x4, v));
            }
        }
        lds_wait();    // this wavefront's LDS stores above are complete
        wg_barrier();  // the strip and its kernel rows are in LDS; every wavefront is done with the previous strip

        if (kind == 0 && channel != cur_channel) {  // Toeplitz fragments T_i^T for this lane's accumulator row
            cur_channel = channel;
            const int lane_ = opaque(lane);
            const int ln_ = lane_ & 15, kg_ = lane_ >> 4;
            const unsigned wa = tile_lds + (unsigned)(WRAW_SLOT * 16) + 2u * (unsigned)wshift(channel);
#pragma unroll
            for (int i = 0; i < R; ++i) {  // row m = ln, slots k = 8*kg + t, tap j = k-SHIFT-m
                unsigned tap[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int j = kg_ * 8 + t - G::SHIFT - ln_;
                    const bool ok = j >= 0 && j < S;
                    const int idx = BWD ? (R - 1 - i) * S + (S - 1 - j) : i * S + j;
                    tap[t] = lds_load_u16(wa + 2u * (unsigned)(ok ? idx : 0));
                }
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(tap[0]), "+v"(tap[1]), "+v"(tap[2]), "+v"(tap[3]), "+v"(tap[4]), "+v"(tap[5]), "+v"(tap[6]), "+v"(tap[7])
                             :
                             : "memory");
                unsigned pk[4];
#pragma unroll
                for (int t = 0; t < 8; t += 2) {
                    const int j = kg_ * 8 + t - G::SHIFT - ln_;
                    const unsigned lo = (j >= 0 && j < S) ? tap[t] : 0u, hi = (j + 1 >= 0 && j + 1 < S) ? tap[t + 1] : 0u;
                    pk[t / 2] = lo | (hi << 16);
                }
                tz[i] = __builtin_bit_cast(frag8<T>, u32x4{pk[0], pk[1], pk[2], pk[3]});
            }
        }

        // put the next strip's copy in flight (into the buffer the previous iteration has just released)
        if (item + 1 < n_items) {
            t_nx += step;
            if constexpr (DW) {
                const int before = sub;
                sub = (sub + M_TURN) % nw;
                t_nx += sub - before;
            }
            while (t_nx >= ipp) {  // (at most once, unless a plane holds fewer items than there are workgroups)
                t_nx -= ipp;
                pbase_nx += plane_step;
                if (!DW) chan_nx = chan_nx + 1 == C ? 0 : chan_nx + 1;
                podd_nx ^= 1;
            }
            decode_item<NARROW>((reflect && podd_nx) ? ipp - 1 - t_nx : t_nx, tiles_n, tri, tm, tn);
            if (kind_of(tm * M_TM, tn * M_TN) == 0) {
                fetch_weights(chan_nx, parity ^ 1);  // (before the copy: the loop-top wait counts what is younger than the copy)
                if (!SCALED) prefetch(pbase_nx, tm * M_TM, tn * M_TN, other, is_interior(tm * M_TM, tn * M_TN));
                fetch_x(pbase_nx, tm * M_TM, tn * M_TN, other, is_interior(tm * M_TM, tn * M_TN));
            }
        }
        if constexpr (DW) {
            // the strips wholly above the diagonal, dealt among the others of their row of strips (ahead of the strip's own stores: the
            // wait at the top of the loop counts those)
            if (causal == 1) {
                const int nr = p0 / M_TN + 1;
                for (int z = nr + q0 / M_TN; z < tiles_n; z += nr) {
                    if (p0 + M_TM <= H && (z + 1) * M_TN <= W) zero_fill_strip<T, NARROW, STREAM, true>(yp, H, W, p0, z * M_TN, tid);
                    else zero_fill_strip<T, NARROW, STREAM>(yp, H, W, p0, z * M_TN, tid);
                }
            }
        } else if (kind != 0) {
            if (kind == 1) {
                if (full_out) {
                    zero_fill_strip<T, NARROW, STREAM, true>(yp, H, W, p0, q0, tid);
                    younger = ST;
                } else {
                    zero_fill_strip<T, NARROW, STREAM>(yp, H, W, p0, q0, tid);
                    younger = -1;
                }
            }
            continue;
        }

        // ---- this wavefront's 16 x 128 outputs: 8 column blocks of 16x16 on 16x16x32 MFMAs (one per kernel row: the
        // 32-key window holds the 16 outputs' taps).  Lane (row ln, group kg) holds keys 4*kg..4*kg+3 of each block.
        if constexpr (DW) {
            // ---- the kernel gradient's products: this wavefront's 32 rows x 64 keys of x, the rows as contraction index.  For row offset
            // u, keys m of x against keys n of dy, u rows further down and from 8 keys further left on (16 h more):
            //     D_u,h[m][n] += sum_p x[p, qa + m] dy[p + u, qa - 8 + 16 h + n]
            // Both operands are transpose reads; a block of 16 keys of dy serves the blocks of x on either side of its start.
            const int lane_ = opaque(lane), ln_ = lane_ & 15, kg_ = lane_ >> 4;
            const int row_a = (wave >> 1) * 32 + kg_ * 4 + (ln_ >> 2);
            const unsigned xa = tile_lds + (unsigned)((BUF + row_a * M_HALF) * sizeof(T)) + (unsigned)((row_a & 7) * 32 + (ln_ & 3) * 8);
            const unsigned da = tile_lds + (unsigned)((row_a * LD + (wave & 1) * 64 + (ln_ & 3) * 4) * sizeof(T));
            struct tr_frag { u32x2 a, b; };
            tr_frag xf[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const unsigned at = xa ^ (unsigned)(((wave & 1) * 4 + b) * 32);
                xf[b].a = lds_load_tr8_at(at, 0);
                xf[b].b = lds_load_tr8_at(at, (int)(16 * M_HALF * sizeof(T)));
            }
            constexpr int NF = R * 5, AHEAD = 4, NS = AHEAD + 1;
            tr_frag ring[NS];
            auto issue = [&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value, u = n / 5, c = n % 5;
                ring[n % NS].a = lds_load_tr8_at(da, (int)((u * LD + c * 16) * sizeof(T)));
                ring[n % NS].b = lds_load_tr8_at(da, (int)(((u + 16) * LD + c * 16) * sizeof(T)));
            };
            static_for<AHEAD>(issue);
            asm volatile("s_waitcnt lgkmcnt(%8)" : "+v"(xf[0].a), "+v"(xf[0].b), "+v"(xf[1].a), "+v"(xf[1].b), "+v"(xf[2].a), "+v"(xf[2].b), "+v"(xf[3].a), "+v"(xf[3].b) : "n"(2 * AHEAD) : "memory");
            frag8<T> xv[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) xv[b] = __builtin_bit_cast(frag8<T>, xf[b]);
            if (!interior) {   // what lies outside the plane or above the diagonal counts as zero
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const int k = q0 + (wave & 1) * 64 + b * 16 + ln_, h = p0 + (wave >> 1) * 32 + kg_ * 4;
                    u32x4 v = __builtin_bit_cast(u32x4, xv[b]);
                    const int lo = k < W ? (causal && k > h ? k - h : 0) : 64, hi = H - h;   // rows h + lo .. h + hi - 1 count
#pragma unroll
                    for (int t = 0; t < 8; t += 2) {
                        const int e = (t >> 2) * 16 + (t & 3);
                        v[t / 2] &= (e >= lo && e < hi ? 0x0000ffffu : 0u) | (e + 1 >= lo && e + 1 < hi ? 0xffff0000u : 0u);
                    }
                    xv[b] = __builtin_bit_cast(frag8<T>, v);
                }
            }
            static_for<NF>([&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value, u = n / 5, c = n % 5;
                if constexpr (n + AHEAD < NF) issue(std::integral_constant<int, n + AHEAD>{});
                constexpr int newer = 2 * ((n + AHEAD < NF ? n + AHEAD : NF - 1) - n);
                asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(ring[n % NS].a), "+v"(ring[n % NS].b) : "n"(newer) : "memory");
                const frag8<T> b = __builtin_bit_cast(frag8<T>, ring[n % NS]);
                if constexpr (c < 4) mma16(dwacc[u][0], xv[c < 4 ? c : 0], b);
                if constexpr (c > 0) mma16(dwacc[u][1], xv[c > 0 ? c - 1 : 0], b);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        const int res0 = NARROW || rb0 == 0 ? rb0 : rb0 + R - 1;        // staged rows that receive the results
        const int qw = q0 + ch * M_HALF;                             // first key of this wavefront's outputs
        {
            constexpr int NCB = M_HALF / 16;
            f32x4 acc[NCB];
            const unsigned xa = tile_lds + (unsigned)((rb0 + ln) * LD + ch * M_HALF + kg * 8) * sizeof(T);
            // Column blocks in pairs, kernel row by kernel row (two independent accumulation chains).  A wavefront issues
            // in order, so a run of LDS reads followed by a run of products leaves the matrix cores idle during the first
            // and the LDS idle during the second: the operand of product n + NLD is read right before product n is issued,
            // into a ring of registers, and a product waits only for its own operand (LDS operations complete in order:
            // exactly the reads issued after it may be outstanding).  Source order is pinned (the scheduler would regroup
            // reads and products).  Blocks above the diagonal are computed like the others and masked below.
            // (operands in flight: 6, or 4 beside the fragments of 7 rows, where four workgroups per CU leave a wavefront 128
            // registers; 12 where three do, 9 beside the fragments of 11 rows)
            constexpr int NLD_MAX = DW ? (R > 7 ? 6 : 10) : wg_per_cu<R, NARROW>() < 4 ? (R > 7 ? 9 : 12) : (R > 6 ? 4 : 6);
            constexpr int NPROD = NCB * R, NLD = 2 * R < NLD_MAX ? 2 * R : NLD_MAX, NSLOT = NLD + 1;
            static_assert(NLD <= 15 && NPROD > NLD, "lgkmcnt field; pipeline deeper than the work");
            u32x4 ring[NSLOT];
            // product n: column block 2*(n / 2R) + n % 2, kernel row (n % 2R) / 2
            auto issue = [&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value;
                constexpr int cb = 2 * (n / (2 * R)) + n % 2, i = (n % (2 * R)) / 2;
                ring[n % NSLOT] = lds_load16_at(xa, (int)((i * LD + cb * 16) * sizeof(T)));
            };
            static_for<NLD>(issue);
            static_for<NPROD>([&](auto ic) __attribute__((always_inline)) {
                constexpr int n = decltype(ic)::value;
                constexpr int cb = 2 * (n / (2 * R)) + n % 2, i = (n % (2 * R)) / 2;
                if constexpr (n + NLD < NPROD) issue(std::integral_constant<int, n + NLD>{});
                constexpr int newer = (n + NLD < NPROD ? n + NLD : NPROD - 1) - n;
                asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(ring[n % NSLOT]) : "n"(newer) : "memory");
                if constexpr (i == 0) acc[cb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                mma16(acc[cb], tz[i], __builtin_bit_cast(frag8<T>, ring[n % NSLOT]));
                __builtin_amdgcn_sched_barrier(0);
            });
            // results into the staged rows res0.. (NARROW: once every wavefront has read what it needs of them; else read by this
            // wavefront only, and no longer needed by it)
            if (NARROW) wg_barrier();
            const int prow = p0 + rb0 + ln;
            const unsigned ra = tile_lds + (unsigned)((res0 + ln) * LD + ch * G::RES_OFF + kg * 4) * sizeof(T);
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                const int q = qw + cb * 16 + kg * 4;
                uint32_t lo = pack2<T>(acc[cb][0], acc[cb][1]), hi = pack2<T>(acc[cb][2], acc[cb][3]);
                if (!interior && causal && q + 3 > prow) {
                    if (q > prow) lo &= 0xffff0000u;
                    if (q + 1 > prow) lo &= 0x0000ffffu;
                    if (q + 2 > prow) hi &= 0xffff0000u;
                    if (q + 3 > prow) hi &= 0x0000ffffu;
                }
                lds_store8_at(ra, (int)(cb * 16 * sizeof(T)), lo, hi);
            }
        }
        // ---- coalesced stores.  NARROW: a wavefront stores the 16 rows that it computed, four 256-byte pieces of rows per
        // instruction.  Else, after a barrier, wavefront w stores rows 8w .. 8w+7 of the strip in full, two 512-byte rows per
        // instruction (the halves of a row come from two wavefronts' results): whole rows in one instruction move a few percent
        // faster through memory ----
        lds_wait();
        if (!NARROW) wg_barrier();
        {
            // (uniform row base + one 32-bit per-lane byte offset: no 64-bit address arithmetic per store)
            const int sr0 = NARROW ? rb0 : wave * 8;                       // first strip row this wavefront stores
            const int sres = NARROW || sr0 < 16 ? sr0 : sr0 + R - 1;       // ... and where its results lie (see res0)
            constexpr int RPS = NARROW ? 4 : 2;                            // rows per instruction
            char *ybase = reinterpret_cast<char *>(yp + (int64_t)(p0 + sr0) * W + q0);
            const int lane_o = opaque(lane);  // (row offsets formed here, not kept in registers across the loop)
            const int r_l = NARROW ? lane_o >> 4 : lane_o >> 5, hf = NARROW ? 0 : (lane_o >> 4) & 1, cv = (lane_o & 15) * VEC;
            const unsigned yoff = (unsigned)(r_l * W + hf * M_HALF + cv) * (unsigned)sizeof(T);
            const int64_t ystep = (int64_t)RPS * W * (int64_t)sizeof(T);
            u32x4 v[4];
            const unsigned va = tile_lds + (unsigned)((sres + r_l) * LD + hf * G::RES_OFF + cv) * sizeof(T);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = lds_load16_at(va, (int)(k * RPS * LD * sizeof(T)));
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : : "memory");
            if (full_out) {  // unconditional: exactly ST vector-memory instructions
#pragma unroll
                for (int k = 0; k < 4; ++k) MTA_CONV_STORE(reinterpret_cast<u32x4 *>(ybase + k * ystep + yoff), v[k]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int r = k * RPS + r_l;
                    if (p0 + sr0 + r < H && q0 + hf * M_HALF + cv < W) MTA_CONV_STORE(reinterpret_cast<u32x4 *>(ybase + k * ystep + yoff), v[k]);
                }
            }
            younger = full_out ? ST : -1;
        }
    }
    if constexpr (DW) {
        // tap (i,j) = sum over m of D_u[m][m + 8 + PW - j], u = R-1-i.  The wavefronts' sums pass through the LDS, as many at a time as it
        // holds; every tap is added up in a fixed order.
        constexpr int PER = 2 * R * 16 * 17, RED = M_NW * R * S, AT_ONCE = (M_NW * PER + RED) * 4 <= 2 * BUFX * (int)sizeof(T) ? M_NW : M_NW / 2;
        static_assert((AT_ONCE * PER + RED) * 4 <= 2 * BUFX * (int)sizeof(T), "the sums pass through the strips' memory");
        float *red = reinterpret_cast<float *>(tiles), *sums = red + RED;
        for (int w0 = 0; w0 < M_NW; w0 += AT_ONCE) {
            __syncthreads();
            if (wave >= w0 && wave < w0 + AT_ONCE) {
#pragma unroll
                for (int u = 0; u < R; ++u)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int v = 0; v < 4; ++v) sums[(wave - w0) * PER + ((2 * u + h) * 16 + 4 * kg + v) * 17 + ln] = dwacc[u][h][v];
            }
            __syncthreads();
            for (int e = tid; e < AT_ONCE * R * S; e += M_WT) {
                const int wv = e / (R * S), tap = e % (R * S), i = tap / S, j = tap % S;
                const float *from = sums + wv * PER + (R - 1 - i) * (2 * 16 * 17);
                float s = 0.0f;
#pragma unroll
                for (int m = 0; m < 16; ++m) {
                    const int n = m + 8 + G::PADW - j;
                    s += from[((n >> 4) * 16 + m) * 17 + (n & 15)];
                }
                red[(w0 + wv) * (R * S) + tap] = s;
            }
        }
        __syncthreads();
        float s = 0.0f;
        if (tid < R * S) {
#pragma unroll
            for (int wv = 0; wv < M_NW; ++wv) s += red[wv * (R * S) + tid];
        }
        if (tid < R * S) partial[vb * (unsigned)(R * S) + tid] = s;
    }
}

// 64 x 128 strips of 7 kernel rows need a quarter of the LDS (32 x 256 ones a little more: three workgroups per CU, not four), and
// they cover the triangle with less beside it; but their rows are written in pieces of 256 bytes, not 512, which costs where whole
// rows are written and where the stores are non-temporal.  32 x 256 | 64 x 128, us, bf16, nothing in the caches:
//   only the lower triangle   B1 H16 S1024  B1 H16 S2048  B2 H16 S2048  B4 H16 S2048  B1 H8 S4096  B1 H16 S4096
//     3x3                       14.8 | 14.1   40.4 | 37.9     62 | 65      120 | 128    58.3 | 60.3   110 | 111
//     6x11                      15.6 | 15.2   41.2 | 39.4     67 | 67      130 | 132    60.3 | 62.0   113 | 116
//     7x7                       18.6 | 15.8   46.3 | 39.9     83 | 68      160 | 134    65.5 | 62.7   119 | 118
//     11x15 (two per CU)        22.5 | 20.4   54   | 45.7    104 | 82      195 | 156    81.8 | 74.5   155 | 139
//   whole rows
//     6x11                      18.6 | 17.5   50.9 | 52.3     84 | 95      159 | 175     102 | 106    154 | 173
//     7x7                       19.8 | 17.8   51.5 | 52.3     84 | 95      161 | 176     105 | 106    155 | 173
//     11x15 (two per CU)        24   | 21     56   | 54      102 | 96      193 | 179     129 | 117    181 | 175
inline bool narrow_strips(int64_t N, int64_t C, int64_t H, int64_t W, int causal, int R)
{
    return R > 7 || (causal == 2 && H == W && (R > 6 || !streams(N, C, H, W, 2)));
}
}  // namespace
