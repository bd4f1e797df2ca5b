// O = P V for the MTA pipeline:  P is the (B,H,S,S) post-softmax tensor, V is (B,H,S,D), O is (B,H,S,D).
//
// When causal, only keys q <= p of P are read: nothing above the diagonal is touched (it may be
// uninitialised memory), which halves the traffic of the plain batched GEMM this replaces.
// What bounds it is the bytes through a CU's path to the L2: the P triangle once, V once per block of rows; product_form() says
// which kernel a grid takes.
//
// The wide one: P_WAVES wavefronts own a block of 32 query rows each; a wavefront owns two blocks of 16 rows.  O^T += V^T P^T on
// 16x16x32 MFMAs: lane (r = lane%16, g = lane/16) owns query row r of a block and supplies P^T
// fragments straight from global memory (16 contiguous bytes = 8 keys of its row, loaded one key
// block ahead), V blocks of 64 keys are copied global -> LDS asynchronously (double buffered,
// 16-byte chunks XOR-swizzled by key) and V^T fragments come out of them through the LDS transpose
// read: within 16 lanes, lane c supplies the address of 4 head-dim values of key c/4 and lane i
// receives head-dim value i of 4 consecutive keys.
#include <type_traits>

#include <cstdlib>

#include "common.hpp"
#include "mfma.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

constexpr int P_WAVES = 4;          // wavefronts per workgroup (8, i.e. half the V re-reads, measured no faster)
constexpr int P_NT = 64 * P_WAVES;
constexpr int P_BQ = 32 * P_WAVES;  // query rows per block: 32 per wavefront
constexpr int P_OCC = 2;            // workgroups per CU the kernel is compiled for
constexpr int P_BK = 64;  // keys per iteration (128 measured no faster): each lane reads P_BK/4 contiguous bytes of its row per
                                 // iteration, back to back, so that DRAM pages are used in long runs
constexpr int P_KS = P_BK / 32;  // 32-key contraction steps per iteration

// This kernel stays for (B,H,S,S) planes of 4096 keys and more in grids of 2048 row blocks and more (product_form()).
template <typename T, int D>
__global__ __launch_bounds__(P_NT, P_OCC) void causal_pv_kernel(
    const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S, int causal, int nqb, int64_t total_wg,
    int64_t per_xcd, const int *__restrict__ band_lo, int H, int tri_gl, float scale, int SV)
{
    constexpr int CPR = D / 8;               // 16-byte chunks per V row
    constexpr int TILE = P_BK * D;           // elements per V block
    constexpr int ROUNDS = (TILE / 8 + P_NT - 1) / P_NT;
    constexpr int DB = D / 16;
    // Double buffer as two separate arrays, and a loop body instantiated once per array: the compiler then sees that
    // the LDS reads of one block never touch the asynchronous copy in flight into the other.  With one array it
    // cannot, and waits for the copy (and for every load issued before it) ahead of the first LDS read.
    __shared__ __align__(16) T v_a[TILE];
    __shared__ __align__(16) T v_b[TILE];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    // XCD-aware order: XCD x (workgroup id % 8) takes the x-th eighth of the (batch*head, query block) list, so
    // the workgroups that share one head's V run on one L2; within a head the longest query blocks come first
    const int64_t lid = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (lid >= total_wg) return;
    // A workgroup takes two blocks of query rows of one (batch, head): block nqb-1-pi and block pi.  With causal
    // rows the first has the most keys and the second the fewest: every workgroup gets the same amount of work
    // (the whole grid is resident at once, so the longest workgroup would otherwise set the kernel's duration).
    const int npairs = (nqb + 1) / 2;
    const int pi = (int)(lid % npairs);
    const int64_t bh = lid / npairs;
    // (tri_gl > 0: P in the triangular layout, groups of tri_gl heads interleaved by rows)
    const T *Pp = tri_gl > 0 ? P + (bh / tri_gl) * (tri_gl * tri_rowoff(S)) : P + bh * (int64_t)S * S;
    const T *Vp = V + bh * (int64_t)SV * D;   // (SV: rows that V has, at most S)
    T *Op = O + bh * (int64_t)S * D;
  for (int half = 0; half < 2; ++half) {
    const int qb = half == 0 ? nqb - 1 - pi : pi;
    if (half == 1 && qb == nqb - 1 - pi) break;  // odd number of blocks: the middle one is alone
    const int q0 = qb * P_BQ;
    if (half == 1) __syncthreads();  // the V buffers are reused: everybody has finished reading them

    auto issue_v = [&](int j, T *dst) {
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int slot = r * P_NT + tid;
            if (TILE / 8 % P_NT != 0 && slot >= TILE / 8) break;
            const int row = slot / CPR, c = (slot % CPR) ^ v_swizzle<D>(row);
            int vr = j * P_BK + row;
            vr = vr >= SV ? SV - 1 : vr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Vp + (int64_t)vr * D + c * 8),
                                             (lds_void_t *)(dst + (r * P_NT + wave * 64) * 8), 16, 0, 0);
        }
    };

    int prow[2];
    const T *prow_ptr[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        prow[rb] = q0 + wave * 32 + rb * 16 + ln;
        const int pc = prow[rb] < S ? prow[rb] : S - 1;
        prow_ptr[rb] = tri_gl > 0 ? Pp + tri_gl * tri_rowoff(pc) + (int)(bh % tri_gl) * tri_rowlen(pc) + kg * 8
                                  : Pp + (int64_t)pc * S + kg * 8;
    }
    // P^T fragments of key block j: slots t = 0..7 of k-step ks are keys j*64 + 32ks + 8kg + t; out-of-range
    // vectors re-read the row start, the values are masked when used
    auto load_p = [&](int j, frag8<T> (&pf)[2][P_KS]) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int ks = 0; ks < P_KS; ++ks) {
                const int key = j * P_BK + ks * 32 + kg * 8;
                const bool ok = key < S && !(causal && key > prow[rb]);
                // (non-temporal: P is streamed, every element is read once)
                typedef unsigned int u4 __attribute__((ext_vector_type(4)));
                pf[rb][ks] = __builtin_bit_cast(frag8<T>, __builtin_nontemporal_load(reinterpret_cast<const u4 *>(
                                                              prow_ptr[rb] + (ok ? j * P_BK + ks * 32 : -kg * 8))));
            }
    };

    const int q_last = (q0 + P_BQ - 1 < S - 1) ? q0 + P_BQ - 1 : S - 1;
    const int j_end = causal ? q_last / P_BK : (S - 1) / P_BK;
    // band mask (band_lo[b, p]: first key row p sees, P is 0 ahead of it): the key blocks ahead of the first key any row
    // of this query block sees are not visited (every wavefront reduces all the rows: the same answer in each)
    int j0 = 0;
    if (band_lo) {
        const int64_t brow = (bh / H) * (int64_t)S;
        int fmin = S;
        for (int r = lane; r < P_BQ; r += 64) {
            if (q0 + r < S) {
                const int f = band_lo[brow + q0 + r];
                fmin = f < fmin ? f : fmin;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(fmin, off);
            fmin = o < fmin ? o : fmin;
        }
        fmin = __builtin_amdgcn_readfirstlane(fmin);
        j0 = (fmin > 0 ? fmin : 0) / P_BK;
        if (j0 > j_end) j0 = j_end;
    }
    issue_v(j0, v_a);
    // P fragments are fetched one key block ahead, alternately into two register sets
    frag8<T> p_a[2][P_KS], p_b[2][P_KS];
    load_p(j0, p_a);

    f32x4 oacc[2][DB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto step = [&](int j, const T *Vb, T *Vn, frag8<T> (&pcur)[2][P_KS], frag8<T> (&pnext)[2][P_KS]) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);  // V block j and the P fragments have arrived
        __syncthreads();                // for every wavefront; reads of the other buffer are finished
        if (j + 1 <= j_end) {
            issue_v(j + 1, Vn);
            load_p(j + 1, pnext);
        }
        // mask the fragments of this block: keys beyond the row (causal) or the sequence count as 0
        frag8<T> pf[2][P_KS];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int ks = 0; ks < P_KS; ++ks) {
                const int key0 = j * P_BK + ks * 32 + kg * 8;
                pf[rb][ks] = pcur[rb][ks];
                const int lim = causal ? (prow[rb] < S - 1 ? prow[rb] : S - 1) : S - 1;
                if (key0 + 7 > lim) {
#pragma unroll
                    for (int t = 0; t < 8; ++t)
                        if (key0 + t > lim) pf[rb][ks].v[t] = from_float<T>(0.0f);
                }
            }
        // V^T fragments of block blk = ks*DB + db are read from LDS while the matrix cores work on block blk-1 (left to
        // itself the compiler issues read, wait, product, read, wait, ... : an LDS latency per group of products)
        auto load_vf = [&](int blk, frag8<T> &dst) {
            const int ks = blk / DB, db = blk % DB;
            const int key_a = ks * 32 + kg * 8 + (ln >> 2);  // slots 0..3: keys 8kg+(0..3); slots 4..7: +4
            const int key_b = key_a + 4;
            const int ch = db * 2 + ((ln & 3) >> 1);
            const int sub = (ln & 1) * 4;
            const T *pa = Vb + key_a * D + ((ch ^ v_swizzle<D>(key_a)) * 8) + sub;
            const T *pb = Vb + key_b * D + ((ch ^ v_swizzle<D>(key_b)) * 8) + sub;
            struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pa),
                                           __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pb)};
            dst = __builtin_bit_cast(frag8<T>, both);
        };
        frag8<T> vf[2];
        load_vf(0, vf[0]);
#pragma unroll
        for (int blk = 0; blk < P_KS * DB; ++blk) {
            const int ks = blk / DB, db = blk % DB;
            if (blk + 1 < P_KS * DB) load_vf(blk + 1, vf[(blk + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);  // (the instruction scheduler would move the reads back behind the products)
            mma16(oacc[0][db], vf[blk & 1], pf[0][ks]);
            mma16(oacc[1][db], vf[blk & 1], pf[1][ks]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int j = j0;;) {
        step(j, v_a, v_b, p_a, p_b);
        if (++j > j_end) break;
        step(j, v_b, v_a, p_b, p_a);
        if (++j > j_end) break;
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        if (prow[rb] >= S) continue;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            struct alignas(8) quad { T v[4]; } out;
#pragma unroll
            for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[rb][db][v] * scale);
            *reinterpret_cast<quad *>(Op + (int64_t)prow[rb] * D + db * 16 + kg * 4) = out;
        }
    }
  }
}

// ---- small grids ----------------------------------------------------------------------------------------------------
// The two products with 32 output rows per workgroup, whose four wavefronts take every fourth 32-row step of the contraction
// each, on operands of their own in LDS (no barrier in the loop), and add their sums up at the end.  With 128 rows per
// wavefront group a short sequence is a few dozen workgroups that each walk their keys alone; this is 8 times as many with a
// quarter of the steps.  The price is that a V (X) block serves 32 rows, so only grids that fill the chip in no other way
// take it (product_form()).
constexpr int RB = 2, N_ROWS = 16 * RB;   // 16-row blocks, output rows per workgroup (64 rows: the sums leave too few registers)
constexpr int N_STEP = 32;                // contraction rows per step
// the sums of the four wavefronts, added in their order: wavefront w takes 16-wide blocks w, w+4, ... of the head dim
template <typename T, int D, typename STORE>
__device__ __forceinline__ void narrow_reduce(T *a, T *b, const f32x4 (&oacc)[RB][D / 16], int wave, int lane, STORE &&store)
{
    constexpr int DB = D / 16, PART = RB * DB * 64;   // 16-byte vectors of one wavefront's sums: half a buffer
    static_assert((size_t)PART * 16 * 2 <= (size_t)4 * N_STEP * D * sizeof(T), "two wavefronts' sums fit a buffer");
    f32x4 *const part[4] = {reinterpret_cast<f32x4 *>(a), reinterpret_cast<f32x4 *>(a) + PART, reinterpret_cast<f32x4 *>(b),
                            reinterpret_cast<f32x4 *>(b) + PART};
    __syncthreads();   // nobody reads operands any more
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) part[wave][(rb * DB + db) * 64 + lane] = oacc[rb][db];
    __syncthreads();
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int i = 0; i < DB / 4; ++i) {
            const int db = i * 4 + wave, at = (rb * DB + db) * 64 + lane;
            store(rb, db, ((part[0][at] + part[1][at]) + part[2][at]) + part[3][at]);
        }
}

template <typename T, int D>
__device__ __forceinline__ void pv_narrow(T *lds, unsigned wg, const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S, int causal,
                                          int heads, int nrb, int cus, const int *__restrict__ band_lo, int H, int tri_gl, float scale, int SV)
{
    constexpr int CPR = D / 8, TILE = N_STEP * D, ROUNDS = TILE / 8 / 64, DB = D / 16;
    T *const v_a_all = lds, *const v_b_all = lds + 4 * TILE;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const v_a = v_a_all + wave * TILE;
    T *const v_b = v_b_all + wave * TILE;
    int bh, rank;
    if (!longest_first(wg, heads, nrb, cus, bh, rank)) return;
    const int q0 = (nrb - 1 - rank) * N_ROWS;
    const T *Pp = tri_gl > 0 ? P + (bh / tri_gl) * (tri_gl * tri_rowoff(S)) : P + bh * (int64_t)S * S;
    const T *Vp = V + bh * (int64_t)SV * D;   // (SV: rows that V has, at most S)
    T *Op = O + bh * (int64_t)S * D;

    auto issue_v = [&](int j, T *dst) {   // keys past the sequence re-read the last one: their probabilities are masked
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int slot = r * 64 + lane, row = slot / CPR, c = (slot % CPR) ^ v_swizzle<D>(row);
            int vr = j * N_STEP + row;
            vr = vr >= SV ? SV - 1 : vr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Vp + (int64_t)vr * D + c * 8), (lds_void_t *)(dst + r * 64 * 8), 16, 0, 0);
        }
    };
    int prow[RB];
    const T *prow_ptr[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        prow[rb] = q0 + rb * 16 + ln;
        const int pc = prow[rb] < S ? prow[rb] : S - 1;
        prow_ptr[rb] = tri_gl > 0 ? Pp + tri_gl * tri_rowoff(pc) + (int)(bh % tri_gl) * tri_rowlen(pc) + kg * 8
                                  : Pp + (int64_t)pc * S + kg * 8;
    }
    auto load_p = [&](int j, frag8<T> (&pf)[RB]) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int key = j * N_STEP + kg * 8;
            const bool ok = key < S && !(causal && key > prow[rb]);
            pf[rb] = *reinterpret_cast<const frag8<T> *>(prow_ptr[rb] + (ok ? j * N_STEP : -kg * 8));
        }
    };
    const int q_last = (q0 + N_ROWS - 1 < S - 1) ? q0 + N_ROWS - 1 : S - 1;
    const int j_end = causal ? q_last / N_STEP : (S - 1) / N_STEP;
    int j0 = 0;
    if (band_lo) {   // the steps ahead of the first key any of these rows sees hold zeros
        const int fr = q0 + (lane & 31);
        int f = fr < S ? band_lo[(bh / H) * (int64_t)S + fr] : S;
#pragma unroll
        for (int off = N_ROWS / 2; off > 0; off >>= 1) {
            const int o = __shfl_xor(f, off);
            f = o < f ? o : f;
        }
        f = __builtin_amdgcn_readfirstlane(f);
        j0 = (f > 0 ? f : 0) / N_STEP;
        if (j0 > j_end) j0 = j_end;
    }
    // this wavefront's steps: j = wave (mod 4), by the step's own number (what a band mask skips leaves every sum as it is)
    const int jw = j0 + ((wave - j0) & 3);
    f32x4 oacc[RB][DB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    frag8<T> p_a[RB], p_b[RB];
    auto step = [&](int j, const T *Vb, T *Vn, frag8<T> (&pcur)[RB], frag8<T> (&pnext)[RB]) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // this wavefront's V block and P fragments have arrived
        asm volatile("" ::: "memory");
        if (j + 4 <= j_end) {
            issue_v(j + 4, Vn);
            load_p(j + 4, pnext);
        }
        frag8<T> pf[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int key0 = j * N_STEP + kg * 8;
            pf[rb] = pcur[rb];
            const int lim = causal ? (prow[rb] < S - 1 ? prow[rb] : S - 1) : S - 1;
            if (key0 + 7 > lim) {
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (key0 + t > lim) pf[rb].v[t] = from_float<T>(0.0f);
            }
        }
        auto load_vf = [&](int db, frag8<T> &dst) {
            const int key_a = kg * 8 + (ln >> 2), key_b = key_a + 4, ch = db * 2 + ((ln & 3) >> 1), sub = (ln & 1) * 4;
            const T *pa = Vb + key_a * D + ((ch ^ v_swizzle<D>(key_a)) * 8) + sub;
            const T *pb = Vb + key_b * D + ((ch ^ v_swizzle<D>(key_b)) * 8) + sub;
            struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pa),
                                           __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pb)};
            dst = __builtin_bit_cast(frag8<T>, both);
        };
        frag8<T> vf[2];
        load_vf(0, vf[0]);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (db + 1 < DB) load_vf(db + 1, vf[(db + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) mma16(oacc[rb][db], vf[db & 1], pf[rb]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (jw <= j_end) {
        issue_v(jw, v_a);
        load_p(jw, p_a);
        for (int j = jw;;) {
            step(j, v_a, v_b, p_a, p_b);
            if ((j += 4) > j_end) break;
            step(j, v_b, v_a, p_b, p_a);
            if ((j += 4) > j_end) break;
        }
    }
    narrow_reduce<T, D>(v_a_all, v_b_all, oacc, wave, lane, [&](int rb, int db, const f32x4 &sum) {
        if (prow[rb] >= S) return;
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(sum[v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)prow[rb] * D + db * 16 + kg * 4) = out;
    });
}

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void causal_pv_narrow_kernel(const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S,
                                                                  int causal, int heads, int nrb, int cus, const int *__restrict__ band_lo, int H, int tri_gl,
                                                                  float scale, int SV)
{
    __shared__ __align__(16) T lds[8 * N_STEP * D];
    pv_narrow<T, D>(lds, blockIdx.x, P, V, O, S, causal, heads, nrb, cus, band_lo, H, tri_gl, scale, SV);
}

// The sums of GR groups of GT threads added up in the first group (true there): the upper half of the groups hand theirs to the
// lower half through the two operand buffers, which together hold just that, until one is left.
template <typename T, int DB, int GT, int GR> __device__ __forceinline__ bool mid_sums(T *a, T *b, f32x4 (&oacc)[DB], int grp, int tid)
{
    __syncthreads();   // nobody reads operands any more
#pragma unroll
    for (int h = GR / 2; h > 0; h /= 2) {
        auto place = [&](int g, int db) -> f32x4 & {
            const int at = g * DB + db;
            return at < h * DB / 2 ? reinterpret_cast<f32x4 *>(a)[at * GT + tid] : reinterpret_cast<f32x4 *>(b)[(at - h * DB / 2) * GT + tid];
        };
        if (grp >= h && grp < 2 * h) {
#pragma unroll
            for (int db = 0; db < DB; ++db) place(grp - h, db) = oacc[db];
        }
        __syncthreads();
        if (grp < h) {
#pragma unroll
            for (int db = 0; db < DB; ++db) oacc[db] += place(grp, db);
        }
        if (h > 1) __syncthreads();
    }
    return grp == 0;
}

// ---- grids between the two --------------------------------------------------------------------------------------------
// RW wavefronts of 16 rows share a block of V (64 keys) in LDS, GR groups of them take every GR-th block; 16 wavefronts per CU in
// every form (two workgroups of 8 or one of 16).  A wavefront of 16 rows instead of 32 reads its V fragments from LDS for one
// product each instead of two, which the LDS has room for, and leaves the registers (95 instead of 180) for twice the
// wavefronts: the reads of P and V that one waits for fly beside the others' products.
template <typename T, int D, int RW, int GR>
__global__ __launch_bounds__(64 * RW * GR, RW * GR / 4 * (RW * GR <= 8 ? 2 : 1)) void causal_pv_mid_kernel(
    const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S, int causal, int heads, int nrb, int cus,
    const int *__restrict__ band_lo, int H, int tri_gl, float scale, int SV)
{
    constexpr int CPR = D / 8, TILE = P_BK * D, GT = 64 * RW, ROUNDS = TILE / 8 / GT, DB = D / 16, ROWS = 16 * RW;
    static_assert(TILE / 8 % GT == 0 && (GT / CPR) % 16 == 0, "whole copy rounds that keep the swizzle phase");
    __shared__ __align__(16) T v_a_all[GR * TILE];
    __shared__ __align__(16) T v_b_all[GR * TILE];
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const v_a = v_a_all + grp * TILE;
    T *const v_b = v_b_all + grp * TILE;
    int bh, rank;
    if (!longest_first(heads, nrb, cus, bh, rank)) return;
    const int q0 = (nrb - 1 - rank) * ROWS;
    const T *Pp = tri_gl > 0 ? P + (bh / tri_gl) * (tri_gl * tri_rowoff(S)) : P + bh * (int64_t)S * S;
    const T *Vp = V + bh * (int64_t)SV * D;   // (SV: rows that V has, at most S)
    T *Op = O + bh * (int64_t)S * D;

    const int row0 = tid / CPR, voff0 = row0 * D + ((tid % CPR) ^ v_swizzle<D>(row0)) * 8;
    auto issue_v = [&](int j, T *dst) {   // keys past the sequence re-read the last one: their probabilities are masked
        const bool inside = (j + 1) * P_BK <= SV;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            int off = j * TILE + voff0 + r * (GT / CPR) * D;
            if (!inside) {
                const int key = j * P_BK + row0 + r * (GT / CPR);
                off -= (key >= SV ? key - (SV - 1) : 0) * D;
            }
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Vp + off), (lds_void_t *)(dst + (r * GT + wave * 64) * 8), 16, 0, 0);
        }
    };
    const int w0 = q0 + wave * 16, prow = w0 + ln;
    const int pc = prow < S ? prow : S - 1;
    const T *prow_ptr = tri_gl > 0 ? Pp + tri_gl * tri_rowoff(pc) + (int)(bh % tri_gl) * tri_rowlen(pc) : Pp + (int64_t)pc * S;
    const int lim = causal ? pc : S - 1;   // last key of this lane's row
    auto load_p = [&](int j, frag8<T> (&pf)[P_KS]) {
#pragma unroll
        for (int ks = 0; ks < P_KS; ++ks) {
            const int key = j * P_BK + ks * 32 + kg * 8;
            pf[ks] = *reinterpret_cast<const frag8<T> *>(prow_ptr + (key <= lim ? key : 0));
        }
    };
    const int q_last = (q0 + ROWS - 1 < S - 1) ? q0 + ROWS - 1 : S - 1;
    const int j_end = causal ? q_last / P_BK : (S - 1) / P_BK;
    int j0 = 0;
    if (band_lo) {   // the blocks ahead of the first key any of these rows sees hold zeros
        int f = S;
        for (int r = lane; r < ROWS; r += 64)
            if (q0 + r < S) {
                const int b = band_lo[(bh / H) * (int64_t)S + q0 + r];
                f = b < f ? b : f;
            }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(f, off);
            f = o < f ? o : f;
        }
        f = __builtin_amdgcn_readfirstlane(f);
        j0 = (f > 0 ? f : 0) / P_BK;
        if (j0 > j_end) j0 = j_end;
    }
    // this group's blocks, by the block's own number (what a band mask skips leaves every sum as it is)
    const int jg = j0 + ((grp - j0) & (GR - 1)), nsteps = (j_end - j0) / GR + 1;
    f32x4 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    frag8<T> p_a[P_KS], p_b[P_KS];
    if (jg <= j_end) issue_v(jg, v_a);
    load_p(jg, p_a);
    // lane's place in a block of V for the transpose reads: rows kg*8 + ln/4 (+4), whose swizzle no other part of the row
    // number touches; head-dim block db is an exclusive or away
    const int vrow = kg * 8 + (ln >> 2), vat = vrow * D + ((((ln & 3) >> 1) ^ v_swizzle<D>(vrow)) * 8) + (ln & 1) * 4;
    auto step = [&](int j, const T *Vb, T *Vn, frag8<T> (&pf)[P_KS], frag8<T> (&pn)[P_KS]) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // V block j and the P fragments have arrived
        __syncthreads();                 // for every wavefront; reads of the other buffer are finished
        if (j > j_end) return;
        if (j + GR <= j_end) {
            issue_v(j + GR, Vn);
            load_p(j + GR, pn);
        }
        if (causal && j * P_BK > w0 + 15) return;   // wholly above the diagonal for these rows
        if (j * P_BK + P_BK - 1 > (causal ? w0 : S - 1)) {
#pragma unroll
            for (int ks = 0; ks < P_KS; ++ks) {
                const int left = lim - (j * P_BK + ks * 32 + kg * 8);
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (t > left) pf[ks].v[t] = from_float<T>(0.0f);
            }
        }
        auto load_vf = [&](int blk, frag8<T> &dst) {
            const int ks = blk / DB, db = blk % DB;
            const T *pa = Vb + (vat ^ (db * 16)) + ks * 32 * D;
            struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pa),
                                           __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(pa + 4 * D))};
            dst = __builtin_bit_cast(frag8<T>, both);
        };
        constexpr int AHEAD = 2;
        frag8<T> vf[AHEAD + 1];
#pragma unroll
        for (int b = 0; b < AHEAD; ++b) load_vf(b, vf[b]);
#pragma unroll
        for (int blk = 0; blk < P_KS * DB; ++blk) {
            if (blk + AHEAD < P_KS * DB) load_vf(blk + AHEAD, vf[(blk + AHEAD) % (AHEAD + 1)]);
            __builtin_amdgcn_sched_barrier(0);
            mma16(oacc[blk % DB], vf[blk % (AHEAD + 1)], pf[blk / DB]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int i = 0, j = jg;;) {
        step(j, v_a, v_b, p_a, p_b);
        if (++i >= nsteps) break;
        j += GR;
        step(j, v_b, v_a, p_b, p_a);
        if (++i >= nsteps) break;
        j += GR;
    }
    if constexpr (GR > 1) {
        if (!mid_sums<T, DB, GT, GR>(v_a_all, v_b_all, oacc, grp, tid)) return;
    }
    if (prow >= S) return;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[db][v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)prow * D + db * 16 + kg * 4) = out;
    }
}

// swizzle of a P tile of 32 keys (4 chunks per row): the transpose read serves rows 0..3 and 8..11 (+4, +16) together, and
// rows 8 apart share banks
__device__ __forceinline__ int p_swizzle(int row) { return 2 * ((row >> 3) & 1); }

template <typename T, int D>
__device__ __forceinline__ void ptx_narrow(T *lds, unsigned wg, const T *__restrict__ P, const T *__restrict__ X, T *__restrict__ O, int S, int causal,
                                           int heads, int nkb, int cus, float scale, int H, row_strides xs)
{
    constexpr int XC = D / 8, XT = N_STEP * D, PCH = N_ROWS / 8, XR = XT / 8 / 64, PT = N_STEP * N_ROWS, PR = PT / 8 / 64, DB = D / 16;
    T *const x_a_all = lds, *const x_b_all = lds + 4 * XT, *const p_a_all = lds + 8 * XT, *const p_b_all = p_a_all + 4 * PT;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const x_a = x_a_all + wave * XT;
    T *const x_b = x_b_all + wave * XT;
    T *const p_a = p_a_all + wave * PT;
    T *const p_b = p_b_all + wave * PT;
    int bh, rank;
    if (!longest_first(wg, heads, nkb, cus, bh, rank)) return;
    const int k0 = rank * N_ROWS;   // under the causal rule the first keys have the most query rows
    const T *Pp = P + bh * (int64_t)S * S;
    const T *Xp = X + bh / H * xs.batch + bh % H * xs.head;
    const int xrow = (int)xs.row;
    T *Op = O + bh * (int64_t)S * D;
    auto issue = [&](int j, T *xdst, T *pdst) {   // rows past the sequence re-read the last row, keys past it the first chunk
#pragma unroll
        for (int r = 0; r < XR; ++r) {
            const int slot = r * 64 + lane, row = slot / XC, c = (slot % XC) ^ v_swizzle<D>(row);
            int pr = j * N_STEP + row;
            pr = pr >= S ? S - 1 : pr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Xp + (int64_t)pr * xrow + c * 8), (lds_void_t *)(xdst + r * 64 * 8), 16, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < PR; ++r) {
            const int slot = r * 64 + lane, row = slot / PCH;
            int c = (slot % PCH) ^ p_swizzle(row);
            if (k0 + c * 8 >= S) c = 0;
            int pr = j * N_STEP + row;
            pr = pr >= S ? S - 1 : pr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Pp + (int64_t)pr * S + k0 + c * 8), (lds_void_t *)(pdst + r * 64 * 8), 16, 0, 0);
        }
    };
    auto read_tr = [&](const T *tile, int ld, int sw_a, int sw_b, int blk) {   // rows 8kg + t of a row-major block, column 16*blk + ln
        const int row_a = kg * 8 + (ln >> 2), row_b = row_a + 4, ch = blk * 2 + ((ln & 3) >> 1), sub = (ln & 1) * 4;
        const T *pa = tile + row_a * ld + ((ch ^ sw_a) * 8) + sub;
        const T *pb = tile + row_b * ld + ((ch ^ sw_b) * 8) + sub;
        struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pa),
                                       __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pb)};
        return __builtin_bit_cast(frag8<T>, both);
    };
    const int ra = kg * 8 + (ln >> 2);
    const int xs_a = v_swizzle<D>(ra), xs_b = v_swizzle<D>(ra + 4), ps_a = p_swizzle(ra), ps_b = p_swizzle(ra + 4);
    int krow[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) krow[rb] = k0 + rb * 16 + ln;
    const int j_end = (S - 1) / N_STEP, j_start = causal ? k0 / N_STEP : 0;
    const int jw = j_start + ((wave - j_start) & 3);
    f32x4 oacc[RB][DB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto step = [&](int j, const T *Xb, const T *Pb, T *Xn, T *Pn) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);
        asm volatile("" ::: "memory");
        if (j + 4 <= j_end) issue(j + 4, Xn, Pn);
        const int pbase = j * N_STEP;
        const bool edge = pbase + N_STEP > S || (causal && pbase < k0 + N_ROWS - 1);   // (wavefront-uniform)
        frag8<T> pf[RB];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            pf[rb] = read_tr(Pb, N_ROWS, ps_a, ps_b, rb);
            if (edge) {   // query rows above the key (causal: P is undefined there) or past the sequence count as 0
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int p = pbase + kg * 8 + t;
                    if (p >= S || (causal && p < krow[rb])) pf[rb].v[t] = from_float<T>(0.0f);
                }
            }
        }
        frag8<T> xf[2];
        xf[0] = read_tr(Xb, D, xs_a, xs_b, 0);
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (db + 1 < DB) xf[(db + 1) & 1] = read_tr(Xb, D, xs_a, xs_b, db + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) mma16(oacc[rb][db], xf[db & 1], pf[rb]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (jw <= j_end) {
        issue(jw, x_a, p_a);
        for (int j = jw;;) {
            step(j, x_a, p_a, x_b, p_b);
            if ((j += 4) > j_end) break;
            step(j, x_b, p_b, x_a, p_a);
            if ((j += 4) > j_end) break;
        }
    }
    narrow_reduce<T, D>(x_a_all, x_b_all, oacc, wave, lane, [&](int rb, int db, const f32x4 &sum) {
        if (krow[rb] >= S) return;
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(sum[v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)krow[rb] * D + db * 16 + kg * 4) = out;
    });
}

template <typename T, int D> constexpr int ptx_narrow_lds() { return 8 * N_STEP * D + 8 * N_STEP * N_ROWS; }   // elements
template <typename T, int D>
__global__ __launch_bounds__(256, 2) void causal_ptx_narrow_kernel(const T *__restrict__ P, const T *__restrict__ X, T *__restrict__ O, int S,
                                                                   int causal, int heads, int nkb, int cus, float scale, int H, row_strides xs)
{
    __shared__ __align__(16) T lds[ptx_narrow_lds<T, D>()];
    ptx_narrow<T, D>(lds, blockIdx.x, P, X, O, S, causal, heads, nkb, cus, scale, H, xs);
}

// Both products of one P, a workgroup of each in turns within an XCD: what a training step has left behind the gradient of the
// scores.  Two small grids, each bound by its own latency, and two launches of a step that the host bounds; one | two, us, bf16:
// B1 H8 S256 D64 4.5 | 8.5, B1 H16 S512 D128 8.1 | 13.8, B1 H16 S1024 D64 13.2 | 15.6, B1 H8 S2048 D64 19.7 | 26.2, D128 29.6 | 33.3.
template <typename T, int D>
__global__ __launch_bounds__(256, 2) void causal_products_narrow_kernel(const T *__restrict__ P, const T *__restrict__ V, const T *__restrict__ X,
                                                                        T *__restrict__ O, T *__restrict__ Ot, int S, int causal, int heads, int blocks,
                                                                        int cus, float scale)
{
    __shared__ __align__(16) T lds[ptx_narrow_lds<T, D>()];
    const unsigned wg = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7);
    if (blockIdx.x & 8) ptx_narrow<T, D>(lds, wg, P, X, Ot, S, causal, heads, blocks, cus, scale, heads, row_strides{0, (int64_t)S * D, D});
    else pv_narrow<T, D>(lds, wg, P, V, O, S, causal, heads, blocks, cus, nullptr, 1, 0, scale, S);
}

// ---- the transposed product --------------------------------------------------------------------------------------
// O[k, :] = sum over p of P[p, k] X[p, :], p >= k only when causal: the gradients that the two matrix products of the
// attention leave on their right-hand operands (dV = P^T dO, dK = G^T Q), whose left factor is only defined - and only
// read - on and below the diagonal.  O^T += X^T P on 16x16x32 MFMAs with the query rows as contraction index: both operands are
// copied global -> LDS asynchronously as row-major blocks (double buffered, 16-byte chunks XOR-swizzled by row) and both
// fragments come out of them through the LDS transpose read, which hands a lane four consecutive rows of one column.
// Grids between the two: RW wavefronts of 16 keys share a block of PB query rows (X and P), GR groups of them take every GR-th
// block; grid order and sums as in causal_pv_mid_kernel.
template <typename T, int D, int RW, int GR, int PB>
__global__ __launch_bounds__(64 * RW * GR, 4) void causal_ptx_mid_kernel(const T *__restrict__ P, const T *__restrict__ X, T *__restrict__ O, int S,
                                                                         int causal, int heads, int nkb, int cus,
                                                                         float scale, int H, row_strides xs)
{
    constexpr int XC = D / 8, KB = 16 * RW, PC = KB / 8, XT = PB * D, PT = PB * KB, GT = 64 * RW, XR = XT / 8 / GT, PR = PT / 8 / GT, DB = D / 16,
                  KS = PB / 32;
    static_assert(XT / 8 % GT == 0 && PT / 8 % GT == 0 && GT / XC % 16 == 0 && GT / PC % 16 == 0, "whole copy rounds that keep the swizzle phase");
    __shared__ __align__(16) T x_a_all[GR * XT];
    __shared__ __align__(16) T x_b_all[GR * XT];
    __shared__ __align__(16) T p_a_all[GR * PT];
    __shared__ __align__(16) T p_b_all[GR * PT];
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const x_a = x_a_all + grp * XT;
    T *const x_b = x_b_all + grp * XT;
    T *const p_a = p_a_all + grp * PT;
    T *const p_b = p_b_all + grp * PT;
    int bh, kb;
    if (!longest_first(heads, nkb, cus, bh, kb)) return;
    const int k0 = kb * KB;   // (the first keys have the most query rows)
    const T *Pp = P + bh * (int64_t)S * S;
    const T *Xp = X + bh / H * xs.batch + bh % H * xs.head;
    const int xrow = (int)xs.row;
    T *Op = O + bh * (int64_t)S * D;

    const int xrow0 = tid / XC, xoff0 = xrow0 * xrow + ((tid % XC) ^ v_swizzle<D>(xrow0)) * 8;
    const int prow0 = tid / PC;
    int pchunk = (tid % PC) ^ v_swizzle<KB>(prow0);
    if (k0 + pchunk * 8 >= S) pchunk = 0;   // (keys past the sequence: rows of the result that nobody stores)
    auto issue = [&](int j, T *xdst, T *pdst) {   // rows past the sequence re-read the last one: they are masked
        const bool inside = (j + 1) * PB <= S;
#pragma unroll
        for (int r = 0; r < XR; ++r) {
            const int row = j * PB + xrow0 + r * (GT / XC), back = inside || row < S ? 0 : row - (S - 1);
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Xp + ((int64_t)j * PB * xrow + xoff0 + (r * (GT / XC) - back) * xrow)),
                                             (lds_void_t *)(xdst + (r * GT + wave * 64) * 8), 16, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < PR; ++r) {
            const int row = j * PB + prow0 + r * (GT / PC), from = inside || row < S ? row : S - 1;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Pp + (int64_t)from * S + k0 + pchunk * 8), (lds_void_t *)(pdst + (r * GT + wave * 64) * 8), 16,
                                             0, 0);
        }
    };
    // a lane's place in a block for the transpose reads: rows kg*8 + ln/4 (+4; 32 further per step), whose swizzle no other part
    // of the row number touches; 16-wide column block c is an exclusive or away
    const int trow = kg * 8 + (ln >> 2), half = (ln & 3) >> 1, sub = (ln & 1) * 4;
    const int xat = trow * D + ((half ^ v_swizzle<D>(trow)) * 8) + sub, pat = trow * KB + (((wave * 2 + half) ^ v_swizzle<KB>(trow)) * 8) + sub;
    auto read_tr = [&](const T *at, int ld) {
        struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)at),
                                       __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(at + 4 * ld))};
        return __builtin_bit_cast(frag8<T>, both);
    };
    const int w0 = k0 + wave * 16, krow = w0 + ln;
    const int j_start = causal ? k0 / PB : 0, j_end = (S - 1) / PB;
    const int jg = j_start + ((grp - j_start) & (GR - 1)), nsteps = (j_end - j_start) / GR + 1;
    f32x4 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (jg <= j_end) issue(jg, x_a, p_a);
    auto step = [&](int j, const T *Xb, const T *Pb, T *Xn, T *Pn) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);   // block j has arrived
        __syncthreads();                 // for every wavefront; reads of the other buffers are finished
        if (j > j_end) return;
        if (j + GR <= j_end) issue(j + GR, Xn, Pn);
        const int pbase = j * PB;
        if (causal && pbase + PB - 1 < w0) return;   // every row of the block lies above these keys
        const bool edge = pbase + PB > S || (causal && pbase < w0 + 15);
        frag8<T> pf[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            pf[ks] = read_tr(Pb + pat + ks * 32 * KB, KB);
            if (edge) {   // query rows above the key (causal: P is undefined there) or past the sequence count as 0
                const int first = (causal ? krow : 0) - (pbase + ks * 32 + kg * 8), end = S - (pbase + ks * 32 + kg * 8);
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (t < first || t >= end) pf[ks].v[t] = from_float<T>(0.0f);
            }
        }
        constexpr int AHEAD = 2;
        frag8<T> xf[AHEAD + 1];
#pragma unroll
        for (int b = 0; b < AHEAD; ++b) xf[b] = read_tr(Xb + (xat ^ (b % DB * 16)) + b / DB * 32 * D, D);
#pragma unroll
        for (int blk = 0; blk < KS * DB; ++blk) {
            constexpr int N = KS * DB;
            const int nb = blk + AHEAD;
            if (nb < N) xf[nb % (AHEAD + 1)] = read_tr(Xb + (xat ^ (nb % DB * 16)) + nb / DB * 32 * D, D);
            __builtin_amdgcn_sched_barrier(0);
            mma16(oacc[blk % DB], xf[blk % (AHEAD + 1)], pf[blk / DB]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int i = 0, j = jg;;) {
        step(j, x_a, p_a, x_b, p_b);
        if (++i >= nsteps) break;
        j += GR;
        step(j, x_b, p_b, x_a, p_a);
        if (++i >= nsteps) break;
        j += GR;
    }
    if constexpr (GR > 1) {
        if (!mid_sums<T, DB, GT, GR>(x_a_all, x_b_all, oacc, grp, tid)) return;
    }
    if (krow >= S) return;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[db][v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)krow * D + db * 16 + kg * 4) = out;
    }
}

// ---- rings ------------------------------------------------------------------------------------------------------------
// The two products with NB buffers instead of two: NB - 1 blocks are in flight at every time, where the kernels above wait for all they
// asked for at each step and have one.  What a step waits for is counted, so every step asks for the same number of things, also past
// the last block (then at the end of the buffer the copies come from, where nothing is read), and the copies come from buffers:
// beside copies from addresses the compiler waits for everything in flight ahead of each use of a loaded register.  Few wavefronts per CU
// are enough for that, so that a short grid gets by without groups; a long one has the wavefronts anyway (product_form()).
// The sums of GR groups of GT threads added up in the first group (true there), the upper half's handed to the lower half through LDS
template <int DB, int GT, int GR> __device__ __forceinline__ bool ring_sums(void *lds, f32x4 (&oacc)[DB], int grp, int tid)
{
    f32x4 *const part = static_cast<f32x4 *>(lds);
    __syncthreads();   // nobody reads operands any more
#pragma unroll
    for (int h = GR / 2; h > 0; h /= 2) {
        if (grp >= h && grp < 2 * h) {
#pragma unroll
            for (int db = 0; db < DB; ++db) part[((grp - h) * DB + db) * GT + tid] = oacc[db];
        }
        __syncthreads();
        if (grp < h) {
#pragma unroll
            for (int db = 0; db < DB; ++db) oacc[db] += part[(grp * DB + db) * GT + tid];
        }
        if (h > 1) __syncthreads();
    }
    return grp == 0;
}

template <typename T, int D, int RW, int GR, int NB, int OCC>
__global__ __launch_bounds__(64 * RW * GR, OCC) void causal_pv_ring_kernel(
    const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S, int causal, int heads, int nrb, int cus,
    const int *__restrict__ band_lo, int H, int tri_gl, float scale, int SV)
{
    constexpr int CPR = D / 8, TILE = P_BK * D, GT = 64 * RW, ROUNDS = TILE / 8 / GT, DB = D / 16, ROWS = 16 * RW, L = ROUNDS + P_KS;
    static_assert(TILE / 8 % GT == 0 && (GT / CPR) % 16 == 0, "whole copy rounds that keep the swizzle phase");
    static_assert(GR * NB * TILE * (int)sizeof(T) >= GR / 2 * DB * GT * 16, "half the groups' sums fit the buffers");
    __shared__ __align__(16) T lds[GR * NB * TILE];
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    int bh, rank;
    if (!longest_first(heads, nrb, cus, bh, rank)) return;
    const int q0 = (nrb - 1 - rank) * ROWS;
    const T *Pp = tri_gl > 0 ? P + (bh / tri_gl) * (tri_gl * tri_rowoff(S)) : P + bh * (int64_t)S * S;
    const T *Vp = V + bh * (int64_t)SV * D;   // (SV: rows that V has, at most S)
    T *Op = O + bh * (int64_t)S * D;
    T *const mine = lds + grp * NB * TILE;

    const int row0 = tid / CPR, voff = (row0 * D + ((tid % CPR) ^ v_swizzle<D>(row0)) * 8) * (int)sizeof(T);
    const int w0 = q0 + wave * 16, prow = w0 + ln;
    const int pc = prow < S ? prow : S - 1;
    const T *prow_ptr = tri_gl > 0 ? Pp + tri_gl * tri_rowoff(pc) + (int)(bh % tri_gl) * tri_rowlen(pc) : Pp + (int64_t)pc * S;
    const int lim = causal ? pc : S - 1;   // last key of this lane's row
    const int q_last = (q0 + ROWS - 1 < S - 1) ? q0 + ROWS - 1 : S - 1;
    const int j_end = causal ? q_last / P_BK : (S - 1) / P_BK;
    int j0 = 0;
    if (band_lo) {   // the blocks ahead of the first key any of these rows sees hold zeros
        int f = S;
        for (int r = lane; r < ROWS; r += 64)
            if (q0 + r < S) {
                const int b = band_lo[(bh / H) * (int64_t)S + q0 + r];
                f = b < f ? b : f;
            }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const int o = __shfl_xor(f, off);
            f = o < f ? o : f;
        }
        f = __builtin_amdgcn_readfirstlane(f);
        j0 = (f > 0 ? f : 0) / P_BK;
        if (j0 > j_end) j0 = j_end;
    }
    // this group's blocks, by the block's own number (what a band mask skips leaves every sum as it is)
    const int jg = j0 + ((grp - j0) & (GR - 1)), nsteps = (j_end - j0) / GR + 1;
    frag8<T> p[NB][P_KS];
    // block j, to buffer b: the same number of loads whatever j is, so that the waits can count; rows past the sequence are zeros,
    // a block past the last one is all of it past the end of the buffer (nothing is read), and so are the rows' vectors (their start again)
    auto fetch = [&](int j, auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value;
        const int left = j <= j_end ? SV - j * P_BK : 0;
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r)
            copy_to_lds(Vp + (int64_t)j * TILE, left * D * (int)sizeof(T), mine + b * TILE + (r * GT + wave * 64) * 8, voff + r * (GT / CPR) * D * (int)sizeof(T));
        in_order();
#pragma unroll
        for (int ks = 0; ks < P_KS; ++ks) {
            const int key = j * P_BK + ks * 32 + kg * 8;
            p[b][ks] = *reinterpret_cast<const frag8<T> *>(prow_ptr + (key <= lim ? key : 0));
        }
        in_order();
    };
    f32x4 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // lane's place in a block of V for the transpose reads: rows kg*8 + ln/4 (+4), whose swizzle no other part of the row
    // number touches; head-dim block db is an exclusive or away
    const int vrow = kg * 8 + (ln >> 2), vat = vrow * D + ((((ln & 3) >> 1) ^ v_swizzle<D>(vrow)) * 8) + (ln & 1) * 4;
    unsigned va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = lds_at(mine + (vat ^ (db * 16)));
    static_for<NB - 1>([&](auto bc) __attribute__((always_inline)) { fetch(jg + decltype(bc)::value * GR, bc); });
    auto step = [&](int j, auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value, N = P_KS * DB, AHEAD = DB == 8 ? 6 : 4;
        copies_wait<(NB - 2) * L>();   // V block j and the rows' vectors have arrived
        wg_barrier();                  // for every wavefront; reads of the buffer ahead of it are finished
        fetch(j + (NB - 1) * GR, std::integral_constant<int, (b + NB - 1) % NB>{});
        if (j > j_end || (causal && j * P_BK > w0 + 15)) return;   // wholly above the diagonal for these rows
        if (j * P_BK + P_BK - 1 > (causal ? w0 : S - 1)) {
#pragma unroll
            for (int ks = 0; ks < P_KS; ++ks) {
                const int left = lim - (j * P_BK + ks * 32 + kg * 8);
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (t > left) p[b][ks].v[t] = from_float<T>(0.0f);
            }
        }
        u32x2 ta[AHEAD + 1], tb[AHEAD + 1];
        auto read = [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, off = (b * TILE + i / DB * 32 * D) * (int)sizeof(T);
            ta[i % (AHEAD + 1)] = lds_load_tr8_at(va[i % DB], off);
            tb[i % (AHEAD + 1)] = lds_load_tr8_at(va[i % DB], off + 4 * D * (int)sizeof(T));
        };
        static_for<AHEAD>(read);
        static_for<N>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, younger = 2 * ((i + AHEAD < N ? i + AHEAD : N - 1) - i);
            if constexpr (i + AHEAD < N) read(std::integral_constant<int, i + AHEAD>{});
            lds_wait_upto<younger>(ta[i % (AHEAD + 1)], tb[i % (AHEAD + 1)]);
            const struct { u32x2 a, b; } both = {ta[i % (AHEAD + 1)], tb[i % (AHEAD + 1)]};
            mma16(oacc[i % DB], __builtin_bit_cast(frag8<T>, both), p[b][i / DB]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    for (int i = 0; i < nsteps; i += NB)
        static_for<NB>([&](auto bc) __attribute__((always_inline)) { step(jg + (i + decltype(bc)::value) * GR, bc); });
    copies_wait<0>();   // (nothing may come into LDS that is no longer this workgroup's)
    if constexpr (GR > 1) {
        if (!ring_sums<DB, GT, GR>(lds, oacc, grp, tid)) return;
    }
    if (prow >= S) return;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[db][v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)prow * D + db * 16 + kg * 4) = out;
    }
}

template <typename T, int D, int RW, int GR, int PB, int NB, int OCC>
__global__ __launch_bounds__(64 * RW * GR, OCC) void causal_ptx_ring_kernel(const T *__restrict__ P, const T *__restrict__ X, T *__restrict__ O, int S,
                                                                          int causal, int heads, int nkb, int cus, float scale, int H, row_strides xs)
{
    constexpr int XC = D / 8, KB = 16 * RW, PC = KB / 8, XT = PB * D, PT = PB * KB, GT = 64 * RW, XR = XT / 8 / GT, PR = PT / 8 / GT, DB = D / 16,
                  KS = PB / 32, BUF = XT + PT, L = XR + PR;
    static_assert(XT / 8 % GT == 0 && PT / 8 % GT == 0 && GT / XC % 16 == 0 && GT / PC % 16 == 0, "whole copy rounds that keep the swizzle phase");
    static_assert(GR * NB * BUF * (int)sizeof(T) >= GR / 2 * DB * GT * 16, "half the groups' sums fit the buffers");
    __shared__ __align__(16) T lds[GR * NB * BUF];
    const int tid = threadIdx.x % GT, grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / GT));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const mine = lds + grp * NB * BUF;
    int bh, kb;
    if (!longest_first(heads, nkb, cus, bh, kb)) return;
    const int k0 = kb * KB;   // (the first keys have the most query rows)
    const T *Pp = P + bh * (int64_t)S * S + k0;
    const T *Xp = X + bh / H * xs.batch + bh % H * xs.head;
    const int xrow = (int)xs.row;
    T *Op = O + bh * (int64_t)S * D;

    const int xrow0 = tid / XC, xoff = (xrow0 * xrow + ((tid % XC) ^ v_swizzle<D>(xrow0)) * 8) * (int)sizeof(T);
    const int prow0 = tid / PC;
    int pchunk = (tid % PC) ^ v_swizzle<KB>(prow0);
    if (k0 + pchunk * 8 >= S) pchunk = 0;   // (keys past the sequence: rows of the result that nobody stores)
    const int poff = (prow0 * S + pchunk * 8) * (int)sizeof(T);
    const int j_start = causal ? k0 / PB : 0, j_end = (S - 1) / PB;
    // block j of X and P to buffer b, the same number of copies whatever j is; rows past the sequence are zeros
    auto fetch = [&](int j, int b) __attribute__((always_inline)) {
        const int left = j <= j_end ? (S - j * PB < PB ? S - j * PB : PB) : 0;
        const int xbytes = left > 0 ? ((left - 1) * xrow + D) * (int)sizeof(T) : 0, pbytes = left > 0 ? (left * S - k0) * (int)sizeof(T) : 0;
#pragma unroll
        for (int r = 0; r < XR; ++r)
            copy_to_lds(Xp + (int64_t)j * PB * xrow, xbytes, mine + b * BUF + (r * GT + wave * 64) * 8, xoff + r * (GT / XC) * xrow * (int)sizeof(T));
#pragma unroll
        for (int r = 0; r < PR; ++r)
            copy_to_lds(Pp + (int64_t)j * PB * S, pbytes, mine + b * BUF + XT + (r * GT + wave * 64) * 8, poff + r * (GT / PC) * S * (int)sizeof(T));
        in_order();
    };
    // a lane's place in a block for the transpose reads: rows kg*8 + ln/4 (+4; 32 further per step), whose swizzle no other part
    // of the row number touches; 16-wide column block c is an exclusive or away
    const int trow = kg * 8 + (ln >> 2), half = (ln & 3) >> 1, sub = (ln & 1) * 4;
    const int xat = trow * D + ((half ^ v_swizzle<D>(trow)) * 8) + sub, pat = trow * KB + (((wave * 2 + half) ^ v_swizzle<KB>(trow)) * 8) + sub;
    unsigned xa[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) xa[db] = lds_at(mine + (xat ^ (db * 16)));
    const unsigned pa = lds_at(mine + XT + pat);
    const int w0 = k0 + wave * 16, krow = w0 + ln;
    const int jg = j_start + ((grp - j_start) & (GR - 1)), nsteps = (j_end - j_start) / GR + 1;
    f32x4 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    static_for<NB - 1>([&](auto bc) __attribute__((always_inline)) { fetch(jg + decltype(bc)::value * GR, decltype(bc)::value); });
    auto step = [&](int j, auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value, N = KS * DB, AHEAD = 4;
        copies_wait<(NB - 2) * L>();   // block j has arrived
        wg_barrier();                  // for every wavefront; reads of the buffer ahead of it are finished
        fetch(j + (NB - 1) * GR, (b + NB - 1) % NB);
        const int pbase = j * PB;
        if (j > j_end || (causal && pbase + PB - 1 < w0)) return;   // every row of the block lies above these keys
        const bool edge = pbase + PB > S || (causal && pbase < w0 + 15);
        u32x2 qa[KS], qb[KS], ta[AHEAD + 1], tb[AHEAD + 1];
        static_for<KS>([&](auto kc) __attribute__((always_inline)) {
            constexpr int ks = decltype(kc)::value, off = (b * BUF + ks * 32 * KB) * (int)sizeof(T);
            qa[ks] = lds_load_tr8_at(pa, off);
            qb[ks] = lds_load_tr8_at(pa, off + 4 * KB * (int)sizeof(T));
        });
        auto read = [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, off = (b * BUF + i / DB * 32 * D) * (int)sizeof(T);
            ta[i % (AHEAD + 1)] = lds_load_tr8_at(xa[i % DB], off);
            tb[i % (AHEAD + 1)] = lds_load_tr8_at(xa[i % DB], off + 4 * D * (int)sizeof(T));
        };
        static_for<AHEAD>(read);
        frag8<T> pf[KS];
        static_for<KS>([&](auto kc) __attribute__((always_inline)) {
            constexpr int ks = decltype(kc)::value;
            lds_wait_upto<2 * AHEAD + 2 * (KS - 1 - ks)>(qa[ks], qb[ks]);
            const struct { u32x2 a, b; } both = {qa[ks], qb[ks]};
            pf[ks] = __builtin_bit_cast(frag8<T>, both);
            if (edge) {   // query rows above the key (causal: P is undefined there) or past the sequence count as 0
                const int first = (causal ? krow : 0) - (pbase + ks * 32 + kg * 8), end = S - (pbase + ks * 32 + kg * 8);
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    if (t < first || t >= end) pf[ks].v[t] = from_float<T>(0.0f);
            }
        });
        static_for<N>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, younger = 2 * ((i + AHEAD < N ? i + AHEAD : N - 1) - i);
            if constexpr (i + AHEAD < N) read(std::integral_constant<int, i + AHEAD>{});
            lds_wait_upto<younger>(ta[i % (AHEAD + 1)], tb[i % (AHEAD + 1)]);
            const struct { u32x2 a, b; } both = {ta[i % (AHEAD + 1)], tb[i % (AHEAD + 1)]};
            mma16(oacc[i % DB], __builtin_bit_cast(frag8<T>, both), pf[i / DB]);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    for (int i = 0; i < nsteps; i += NB)
        static_for<NB>([&](auto bc) __attribute__((always_inline)) { step(jg + (i + decltype(bc)::value) * GR, bc); });
    copies_wait<0>();   // (nothing may come into LDS that is no longer this workgroup's)
    if constexpr (GR > 1) {
        if (!ring_sums<DB, GT, GR>(lds, oacc, grp, tid)) return;
    }
    if (krow >= S) return;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        struct alignas(8) quad { T v[4]; } out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[db][v] * scale);
        *reinterpret_cast<quad *>(Op + (int64_t)krow * D + db * 16 + kg * 4) = out;
    }
}

// ---- which kernel ------------------------------------------------------------------------------------------------------
// What bounds both products is the latency and the bytes of a CU's path to the L2 (about 9 TB/s over the chip): the scores once, and the
// other operand (V, X) once for every block of output rows.  Larger blocks need less of it, smaller ones fill the chip: the line
// runs by the number n of 64-row blocks.  RING kernels are the rings of three (P^T X of 128 rows: four) buffers with 64 or 128 rows, _2 with
// two groups; R kernels have two buffers.  us, rotating P tensors; P V, narrow | R64_2 | R128_1 | RING64 | RING64_2 | RING128 (R figures of
// grids beyond 512 blocks: the kernel taken there):
//   n  256  B1 H8 S2048 D128   15.8 | -- | -- | 16.0 | 18.2 | 23.2         320  B1 H5 S4096 D128   -- | -- | -- | 35.4 | 32.0 | 45.6  (four groups 37.4)
//      288  B1 H12 S1536 D128  16.1 | -- | -- | 15.4 | 14.4 | 18.7             384  B1 H8 S3072 D64    -- | -- | -- | 22.5 | 23.2 | 29.4 (four groups 24.1)
//      512  B1 H16 S2048 D128  34.2 | 23.1 | 41.9 | 19.5 | 23.6 | 24.3         512  B1 H16 S2048 D64   -- | 19.2 | -- | 15.3 | 18.4 | 21.3
//      512  B2 H16 S1008 D64   16.3 | 10.6 | 15.3 | 9.8 | 11.9 | 11.5          512  B4 H16 S512 D128   -- | 10.1 | -- | 10.8 | 15.6 | 11.3
//      768  B1 H16 S3072 D64   -- | 47.4 | -- | 39.7 | 41.7 | 41.6             768  B1 H16 S3072 D128  -- | 50.6 | -- | 51.9 | 53.9 | 51.8
//     1024  B1 H16 S4096 D128  118 | 91.7 | 101 | 97.8 | 108 | 77.0            1024 B4 H16 S1024 D128  45.1 | 28.0 | 23.8 | 26.3 | 35.6 | 23.8
//     1536  B2 H16 S3072 D64   105 | 76.4 | 86.3 | 75.9 | 79.5 | 70.4          2048 B1 H32 S4096 D128  -- | -- | 137 | 163 | 176 | 144
//          in the triangular layout B2 H16 S4096 D128 (2048) narrow 236, R64_2 167, R128_1 145, wide 152
//   P^T X, narrow | R64_2 | R128_1 | RING64_2 (D64: RING64, four buffers of 64 rows) | RING128 | RING128_2
//   n  256  B1 H8 S2048 D128   16.4 | -- | -- | 18.3 | 30.8 | 26.3             384  B1 H8 S3072 D64    -- | -- | -- | 20.3 (four groups 25.8)
//      512  B1 H16 S2048 D128  -- | 25 | -- | 20.5 | 31.4 | 26.8               512  B4 H16 S512 D128   -- | 10.5 | -- | 10.6 | 12.3 | 12.6
//      512  B1 H16 S2048 D64   25.8 | 26.1 | 29.7 | 15.5                       768  B1 H16 S3072 D128  66.7 | 53.2 | 56.2 | 46.8 | 49.1 | 42.9
//     1024  B1 H16 S4096 D128  -- | -- | 78.4 | 79.9 | 73.4 | 71.4             1024 B2 H16 S2048 D128  64.8 | 49.9 | 50.4 | 49.0 | 46.4 | 49.8
//     1024  B4 H16 S1024 D64   27.2 | 16.5 | 19.5 | 18.4                       2048 B4 H32 S1024 D128  -- | -- | 43.9 | 51.4 | 43.3 | 54.1
// Over 120 random grids of 257 to 2500 blocks these lines give 0.935 (P V) and 0.914 (P^T X) of the time that kernels of two buffers took.
// The fp32 sums of a row have three orders: block by block (one group), the even and the odd blocks apart (two groups), every fourth
// block apart (the narrow kernel's four wavefronts).  So a head's last bit may differ between batch sizes that take different kernels.
enum product_kernel { WIDE = 1, R64_2, NARROW, RING64_2, RING128, R128_1, RING64, RING128_2 };

product_kernel product_form(int64_t heads, int64_t S, int D, bool transposed, bool tri, bool band)
{
    // MTA_PV_SPLIT in the environment: 1 .. 8 = always that kernel of the list above (comparison switch), or the next to it where a product
    // has no such form
    static const int force = [] { const char *e = getenv("MTA_PV_SPLIT"); return e ? atoi(e) : 0; }();
    if (force >= WIDE && force <= RING128_2) return force == WIDE && transposed ? R128_1 : (product_kernel)force;
    const int64_t n = heads * ((S + 63) / 64);
    if (n <= 256) return NARROW;   // (resident at once: a CU gets a long and a short block)
    // Many short sequences end their rings soon after they have filled them: P V of B4 H16 S832 D64 (832 blocks) 13.0 on two groups, 15.7 as
    // a ring; P^T X of B4 H16 S640 D128 (640) 13.0 | 15.2.
    const bool longer = S > (D == 64 ? 2 : 3) * (n - 256);
    if (transposed) {
        if (D == 64) return n < 2048 && (S > 1024 || (n < 1024 && longer)) ? RING64 : R64_2;
        if (n < 704) return longer ? RING64_2 : R64_2;
        if (n < 1024) return S > 1024 ? RING128_2 : R64_2;
        return n <= 1536 && S > 768 ? RING128 : R128_1;
    }
    // (Under a band mask a block of rows has few key blocks: two workgroups of two groups per CU in place of one whose ring is deeper, with the
    // same sums.  Window of S/4, B1 H12 S2256 D128 (432): 15.5 | 18.9.)
    if (n < 450 && D == 128) return S > 4 * n ? (band ? R64_2 : RING64_2) : S > 1000 ? RING64 : R64_2;
    if (n < 640 && D == 128) return longer ? RING64 : R64_2;
    if (n < 1024) return D == 64 && (n < 544 ? longer : 2 * S > 5 * n) ? RING64 : R64_2;
    if (D == 64 ? n < 2048 && S >= 2304 : n < 1600 && S >= 2048) return RING128;
    return n >= 2048 ? S >= 4096 && !tri ? WIDE : R128_1 : D == 64 ? R64_2 : R128_1;
}

// A kernel's grid: a workgroup per block of `rows` output rows, `resident` of them on a CU at once; f(grid, blocks per head, cus as
// longest_first() takes it).  A grid that is resident at once but for one more round, which then comes longest first again, pairs
// long and short blocks as well: P V | P^T X of B2 H12 S2784 D128 (528 workgroups of two per CU) 66.8 | 60.2 -> 58.2 | 55.0 us, B2 H16
// S2072 54.9 | 50.1 -> 47.3 | 43.8; two more rounds, or one on top of a reversed round: up to 11 % slower.  False where the grid is too large.
template <typename F> bool product_grid(int64_t heads, int64_t S, int rows, int resident, int causal, F &&f)
{
    const int64_t blocks = (S + rows - 1) / rows, wg = (heads * blocks + 7) / 8 * 8;
    if (wg > 0x7fffffffLL) return false;
    f(dim3((unsigned)wg), (int)blocks, causal && wg <= (int64_t)(resident + (resident % 2 == 0)) * device_cu_count() ? device_cu_count() / 8 : 0);
    return true;
}

template <typename T, int D>
int launch_t(const void *p, const void *x, row_strides xs, void *o, int64_t B, int64_t H, int64_t S, int causal, float scale, hipStream_t st)
{
    auto go = [&](auto kern, int rows, int threads, int resident) {
        const bool fits = product_grid(B * H, S, rows, resident, causal, [&](dim3 grid, int blocks, int cus) {
            hipLaunchKernelGGL(kern, grid, dim3(threads), 0, st, (const T *)p, (const T *)x, (T *)o, (int)S, causal, (int)(B * H), blocks, cus, scale, (int)H,
                               xs);
        });
        return fits ? launch_status() : MTA_ERR_SHAPE;
    };
    const product_kernel form = product_form(B * H, S, D, true, false, false);
    if constexpr (D == 128) {
        switch (form) {
        case RING64:
        case RING64_2: return go(causal_ptx_ring_kernel<T, D, 4, 2, 32, 3, 4>, 64, 512, 2);
        case RING128: return go(causal_ptx_ring_kernel<T, D, 8, 1, 32, 4, 4>, 128, 512, 2);
        case RING128_2: return go(causal_ptx_ring_kernel<T, D, 8, 2, 32, 3, 4>, 128, 1024, 1);
        case R128_1: return go(causal_ptx_mid_kernel<T, D, 8, 1, 64>, 128, 512, 2);
        default: break;
        }
    } else if (form >= RING64_2) return go(causal_ptx_ring_kernel<T, D, 4, 1, 64, 4, 2>, 64, 256, 2);
    return form == NARROW ? go(causal_ptx_narrow_kernel<T, D>, N_ROWS, 256, D == 64 ? 3 : 2) : go(causal_ptx_mid_kernel<T, D, 4, 2, 32>, 64, 512, 2);
}

template <typename T, int D>
int launch(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int causal, hipStream_t st,
           const int *band_lo = nullptr, int tri_gl = 0, float scale = 1.0f, int64_t v_rows = 0)
{
    auto go = [&](auto kern, int rows, int threads, int resident) {
        const bool fits = product_grid(B * H, S, rows, resident, causal, [&](dim3 grid, int blocks, int cus) {
            hipLaunchKernelGGL(kern, grid, dim3(threads), 0, st, (const T *)p, (const T *)v, (T *)o, (int)S, causal, (int)(B * H), blocks, cus, band_lo, (int)H,
                               tri_gl, scale, (int)(v_rows ? v_rows : S));
        });
        return fits ? launch_status() : MTA_ERR_SHAPE;
    };
    switch (product_form(B * H, S, D, false, tri_gl > 0, band_lo != nullptr)) {
    case NARROW: return go(causal_pv_narrow_kernel<T, D>, N_ROWS, 256, D == 64 ? 4 : 2);
    case RING64_2:
        if constexpr (D == 128) return go(causal_pv_ring_kernel<T, D, 4, 2, 3, 2>, 64, 512, 1);
        [[fallthrough]];
    case RING64: return go(causal_pv_ring_kernel<T, D, 4, 1, 3, 3>, 64, 256, D == 64 ? 6 : 3);
    case RING128:
    case RING128_2: return go(causal_pv_ring_kernel<T, D, 8, 1, 3, 4>, 128, 512, D == 64 ? 3 : 2);
    case R64_2: return go(causal_pv_mid_kernel<T, D, 4, 2>, 64, 512, 2);
    case R128_1: return go(causal_pv_mid_kernel<T, D, 8, 1>, 128, 512, 2);
    case WIDE: break;
    }
    const int nqb = (int)((S + P_BQ - 1) / P_BQ);
    const int64_t total_wg = B * H * ((nqb + 1) / 2), per_xcd = (total_wg + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL) return MTA_ERR_SHAPE;
    hipLaunchKernelGGL((causal_pv_kernel<T, D>), dim3((unsigned)(per_xcd * 8)), dim3(P_NT), 0, st, (const T *)p, (const T *)v, (T *)o, (int)S, causal, nqb,
                       total_wg, per_xcd, band_lo, (int)H, tri_gl, scale, (int)(v_rows ? v_rows : S));
    return launch_status();
}
}  // namespace

namespace {
int pv_entry(const void *p, const void *v, const void *first_visible, void *o, int64_t B, int64_t H, int64_t S, int64_t D, int causal,
             float scale, int io_dtype, void *stream)
{
    if (!p || !v || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(p, 16) || !aligned_to(v, 16) || !aligned_to(o, 16) || (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || S % 8 != 0 || (first_visible && !causal)) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int *lo = (const int *)first_visible;
    if (io_dtype == MTA_BF16)
        return D == 64 ? launch<bf16_t, 64>(p, v, o, B, H, S, causal, st, lo, 0, scale) : launch<bf16_t, 128>(p, v, o, B, H, S, causal, st, lo, 0, scale);
    return D == 64 ? launch<f16_t, 64>(p, v, o, B, H, S, causal, st, lo, 0, scale) : launch<f16_t, 128>(p, v, o, B, H, S, causal, st, lo, 0, scale);
}
}  // namespace

// first_visible (int32, (B,S); NULL = none): P[b,h,p,k] is 0 for k < first_visible[b,p] (what the softmax stage leaves
// under a band mask); the key blocks ahead of a query block's first visible key are not read.  Implies causal.
extern "C" int mta_causal_pv_band_fwd(const void *p, const void *v, const void *first_visible, void *o, int64_t B, int64_t H,
                                      int64_t S, int64_t D, int causal, int io_dtype, void *stream)
{
    return pv_entry(p, v, first_visible, o, B, H, S, D, causal, 1.0f, io_dtype, stream);
}

extern "C" int mta_causal_pv_scaled_fwd(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int64_t D, int causal,
                                        float scale, int io_dtype, void *stream)
{
    return pv_entry(p, v, nullptr, o, B, H, S, D, causal, scale, io_dtype, stream);
}

// P in the triangular layout (see tri_rowoff in common.hpp), groups of `group` heads interleaved by rows; causal.
extern "C" int mta_causal_pv_tri_fwd(const void *p, const void *v, const void *first_visible, void *o, int64_t B, int64_t H,
                                     int64_t S, int64_t D, int group, int io_dtype, void *stream)
{
    if (!p || !v || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (group <= 0 || H % group != 0) return MTA_ERR_GROUP;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(p, 16) || !aligned_to(v, 16) || !aligned_to(o, 16) || (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int *lo = (const int *)first_visible;
    if (io_dtype == MTA_BF16)
        return D == 64 ? launch<bf16_t, 64>(p, v, o, B, H, S, 1, st, lo, group) : launch<bf16_t, 128>(p, v, o, B, H, S, 1, st, lo, group);
    return D == 64 ? launch<f16_t, 64>(p, v, o, B, H, S, 1, st, lo, group) : launch<f16_t, 128>(p, v, o, B, H, S, 1, st, lo, group);
}

// V of `rows` rows, S - 7 <= rows <= S, whose probabilities beyond them are not read by the rows up to there (causal): group > 0 P in the
// triangular layout, 0 planes.  O has S rows; what those beyond `rows` hold is not defined.
extern "C" int mta_causal_pv_ragged_fwd(const void *p, const void *v, const void *first_visible, void *o, int64_t B, int64_t H, int64_t S, int64_t rows,
                                        int64_t D, int group, int io_dtype, void *stream)
{
    if (!p || !v || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535 || rows <= 0 || rows > S || rows < S - 7) return MTA_ERR_SHAPE;
    if (group < 0 || (group > 0 && H % group != 0)) return MTA_ERR_GROUP;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(p, 16) || !aligned_to(v, 16) || !aligned_to(o, 16) || (first_visible && !aligned_to(first_visible, 4)))
        return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int *lo = (const int *)first_visible;
    if (io_dtype == MTA_BF16)
        return D == 64 ? launch<bf16_t, 64>(p, v, o, B, H, S, 1, st, lo, group, 1.0f, rows) : launch<bf16_t, 128>(p, v, o, B, H, S, 1, st, lo, group, 1.0f, rows);
    return D == 64 ? launch<f16_t, 64>(p, v, o, B, H, S, 1, st, lo, group, 1.0f, rows) : launch<f16_t, 128>(p, v, o, B, H, S, 1, st, lo, group, 1.0f, rows);
}

extern "C" int mta_causal_pv_fwd(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int64_t D,
                                 int causal, int io_dtype, void *stream)
{
    return mta_causal_pv_band_fwd(p, v, nullptr, o, B, H, S, D, causal, io_dtype, stream);
}

extern "C" int mta_causal_ptx_fwd(const void *p, const void *x, void *o, int64_t B, int64_t H, int64_t S, int64_t D,
                                  int causal, int io_dtype, void *stream)
{
    return mta_causal_ptx_scaled_fwd(p, x, o, B, H, S, D, causal, 1.0f, io_dtype, stream);
}

extern "C" int mta_causal_ptx_scaled_fwd(const void *p, const void *x, void *o, int64_t B, int64_t H, int64_t S, int64_t D, int causal,
                                         float scale, int io_dtype, void *stream)
{
    return mta_causal_ptx_rows_fwd(p, x, H * S * D, S * D, D, o, B, H, S, D, causal, scale, io_dtype, stream);
}

extern "C" int mta_causal_ptx_rows_fwd(const void *p, const void *x, int64_t x_batch, int64_t x_head, int64_t x_row, void *o, int64_t B, int64_t H,
                                       int64_t S, int64_t D, int causal, float scale, int io_dtype, void *stream)
{
    if (!p || !x || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(p, 16) || !aligned_to(x, 16) || !aligned_to(o, 16) || x_batch % 8 != 0 || x_head % 8 != 0 || x_row % 8 != 0) return MTA_ERR_ALIGN;
    if (x_batch < 0 || x_head < 0 || x_row <= 0) return MTA_ERR_SHAPE;
    if (io_dtype == MTA_F32 || S % 8 != 0 || x_row > (1 << 20)) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const row_strides xs{x_batch, x_head, x_row};
    if (io_dtype == MTA_BF16)
        return D == 64 ? launch_t<bf16_t, 64>(p, x, xs, o, B, H, S, causal, scale, st) : launch_t<bf16_t, 128>(p, x, xs, o, B, H, S, causal, scale, st);
    return D == 64 ? launch_t<f16_t, 64>(p, x, xs, o, B, H, S, causal, scale, st) : launch_t<f16_t, 128>(p, x, xs, o, B, H, S, causal, scale, st);
}

// o = scale * P V and ot = scale * P^T X with the lower triangle of P (causal; else all of it)
extern "C" int mta_causal_products(const void *p, const void *v, const void *x, void *o, void *ot, int64_t B, int64_t H, int64_t S, int64_t D,
                                   int causal, float scale, int io_dtype, void *stream)
{
    if (!p || !v || !x || !o || !ot) return MTA_ERR_NULL;
    const bool one = io_dtype != MTA_F32 && dtype_size(io_dtype) && B > 0 && H > 0 && S > 0 && S <= (1 << 24) && B * H <= 65535 && (D == 64 || D == 128) &&
                     S % 8 == 0 && aligned_to(p, 16) && aligned_to(v, 16) && aligned_to(x, 16) && aligned_to(o, 16) && aligned_to(ot, 16) &&
                     product_form(B * H, S, (int)D, false, false, false) == NARROW && product_form(B * H, S, (int)D, true, false, false) == NARROW;
    if (!one) {
        const int rc = mta_causal_pv_scaled_fwd(p, v, o, B, H, S, D, causal, scale, io_dtype, stream);
        return rc != MTA_OK ? rc : mta_causal_ptx_scaled_fwd(p, x, ot, B, H, S, D, causal, scale, io_dtype, stream);
    }
    const int64_t blocks = (S + N_ROWS - 1) / N_ROWS, wg = (B * H * blocks + 7) / 8 * 8;
    const int cus = causal && 2 * wg <= (int64_t)(D == 64 ? 3 : 2) * device_cu_count() ? device_cu_count() / 16 : 0;
    auto go = [&](auto type, auto d) {
        using T = decltype(type);
        hipLaunchKernelGGL((causal_products_narrow_kernel<T, d()>), dim3((unsigned)(2 * wg)), dim3(256), 0, (hipStream_t)stream, (const T *)p, (const T *)v,
                           (const T *)x, (T *)o, (T *)ot, (int)S, causal, (int)(B * H), (int)blocks, cus, scale);
    };
    const std::integral_constant<int, 64> d64{};
    const std::integral_constant<int, 128> d128{};
    if (io_dtype == MTA_BF16) D == 64 ? go(bf16_t{}, d64) : go(bf16_t{}, d128);
    else D == 64 ? go(f16_t{}, d64) : go(f16_t{}, d128);
    return launch_status();
}
