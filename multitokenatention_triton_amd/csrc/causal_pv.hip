// O = P V for the MTA pipeline:  P is the (B,H,S,S) post-softmax tensor, V is (B,H,S,D), O is (B,H,S,D).
//
// When causal, only keys q <= p of P are read: nothing above the diagonal is touched (it may be
// uninitialised memory), which halves the traffic of the plain batched GEMM this replaces.
// HBM-bound: the P triangle is streamed once, V blocks are re-read from L2.
//
// P_WAVES wavefronts own a block of 32 query rows each; a wavefront owns two blocks of 16 rows.  O^T += V^T P^T on
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

// SPLIT = 2: two such groups of wavefronts in a workgroup share the query rows and take the even and the odd key
// blocks; the second group's sums reach the first through LDS at the end.  For grids that put one workgroup on a CU
// (few heads): twice the loads in flight for the same bytes.
template <typename T, int D, int SPLIT>
__global__ __launch_bounds__(P_NT * SPLIT, SPLIT == 2 ? 1 : P_OCC) void causal_pv_kernel(
    const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S, int causal, int nqb, int64_t total_wg,
    int64_t per_xcd, const int *__restrict__ band_lo, int H, int tri_gl, float scale)
{
    constexpr int CPR = D / 8;               // 16-byte chunks per V row
    constexpr int TILE = P_BK * D;           // elements per V block
    constexpr int ROUNDS = (TILE / 8 + P_NT - 1) / P_NT;
    constexpr int DB = D / 16;
    static_assert(SPLIT == 1 || (size_t)SPLIT * TILE * sizeof(T) == (size_t)DB * P_NT * 16, "the sums of one row block fit one V buffer pair");
    // Double buffer as two separate arrays, and a loop body instantiated once per array: the compiler then sees that
    // the LDS reads of one block never touch the asynchronous copy in flight into the other.  With one array it
    // cannot, and waits for the copy (and for every load issued before it) ahead of the first LDS read.
    __shared__ __align__(16) T v_a_all[SPLIT * TILE];
    __shared__ __align__(16) T v_b_all[SPLIT * TILE];

    const int grp = SPLIT == 2 ? (int)(threadIdx.x >> 8) : 0;  // which key blocks: j % SPLIT == grp
    T *const v_a = v_a_all + grp * TILE;
    T *const v_b = v_b_all + grp * TILE;
    const int tid = threadIdx.x & (P_NT - 1);
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
    const T *Vp = V + bh * (int64_t)S * D;
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
            vr = vr >= S ? S - 1 : vr;
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
    // this group's key blocks: jg, jg + SPLIT, ... (by the block's own parity, whatever the first block is: a band mask
    // that skips blocks of zeros leaves every sum as it is, bit for bit)
    const int jg = SPLIT == 2 ? j0 + ((j0 & 1) != grp) : j0;
    const int nsteps = (j_end - j0) / SPLIT + 1;  // of the group that starts at j0: the other one idles in its last step
    if (jg <= j_end) issue_v(jg, v_a);
    // P fragments are fetched one key block ahead, alternately into two register sets
    frag8<T> p_a[2][P_KS], p_b[2][P_KS];
    load_p(jg, p_a);

    f32x4 oacc[2][DB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto step = [&](int j, const T *Vb, T *Vn, frag8<T> (&pcur)[2][P_KS], frag8<T> (&pnext)[2][P_KS]) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);  // V block j and the P fragments have arrived
        __syncthreads();                // for every wavefront; reads of the other buffer are finished
        if (SPLIT == 2 && j > j_end) return;  // (the other group's last block: this one only meets it at the barrier)
        if (j + SPLIT <= j_end) {
            issue_v(j + SPLIT, Vn);
            load_p(j + SPLIT, pnext);
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
    for (int i = 0, j = jg;; j += SPLIT) {
        step(j, v_a, v_b, p_a, p_b);
        if (++i >= nsteps) break;
        j += SPLIT;
        step(j, v_b, v_a, p_b, p_a);
        if (++i >= nsteps) break;
    }

    if constexpr (SPLIT == 2) {
        // the second group's sums travel through the V buffers (rows' first block in one, second in the other)
        typedef __attribute__((address_space(3))) f32x4 lds_f4;
        __syncthreads();  // nobody reads V any more
        if (grp == 1) {
#pragma unroll
            for (int db = 0; db < DB; ++db) {
                reinterpret_cast<f32x4 *>(v_a_all)[db * P_NT + tid] = oacc[0][db];
                reinterpret_cast<f32x4 *>(v_b_all)[db * P_NT + tid] = oacc[1][db];
            }
        }
        __syncthreads();
        if (grp == 1) continue;  // (the barrier ahead of the second row block is met at the top of the loop)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            oacc[0][db] += reinterpret_cast<const f32x4 *>(v_a_all)[db * P_NT + tid];
            oacc[1][db] += reinterpret_cast<const f32x4 *>(v_b_all)[db * P_NT + tid];
        }
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
// quarter of the steps.  The price is that a V (X) block serves 32 rows instead of 128, so long sequences of many heads,
// whose grids fill the chip anyway, keep the kernels above and below (narrow_grid()).
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
__global__ __launch_bounds__(256, 2) void causal_pv_narrow_kernel(const T *__restrict__ P, const T *__restrict__ V, T *__restrict__ O, int S,
                                                                  int causal, int nrb, int64_t total_wg, int64_t per_xcd,
                                                                  const int *__restrict__ band_lo, int H, int tri_gl, float scale)
{
    constexpr int CPR = D / 8, TILE = N_STEP * D, ROUNDS = TILE / 8 / 64, DB = D / 16;
    __shared__ __align__(16) T v_a_all[4 * TILE];
    __shared__ __align__(16) T v_b_all[4 * TILE];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const v_a = v_a_all + wave * TILE;
    T *const v_b = v_b_all + wave * TILE;
    const int64_t lid = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (lid >= total_wg) return;
    const int64_t bh = lid / nrb;
    const int q0 = (nrb - 1 - (int)(lid % nrb)) * N_ROWS;   // longest rows first
    const T *Pp = tri_gl > 0 ? P + (bh / tri_gl) * (tri_gl * tri_rowoff(S)) : P + bh * (int64_t)S * S;
    const T *Vp = V + bh * (int64_t)S * D;
    T *Op = O + bh * (int64_t)S * D;

    auto issue_v = [&](int j, T *dst) {   // keys past the sequence re-read the last one: their probabilities are masked
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const int slot = r * 64 + lane, row = slot / CPR, c = (slot % CPR) ^ v_swizzle<D>(row);
            int vr = j * N_STEP + row;
            vr = vr >= S ? S - 1 : vr;
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

// swizzle of a P tile of 32 keys (4 chunks per row): the transpose read serves rows 0..3 and 8..11 (+4, +16) together, and
// rows 8 apart share banks
__device__ __forceinline__ int p_swizzle(int row) { return 2 * ((row >> 3) & 1); }

template <typename T, int D>
__global__ __launch_bounds__(256, 2) void causal_ptx_narrow_kernel(const T *__restrict__ P, const T *__restrict__ X, T *__restrict__ O, int S,
                                                                   int causal, int nkb, int64_t total_wg, int64_t per_xcd, float scale)
{
    constexpr int XC = D / 8, XT = N_STEP * D, PCH = N_ROWS / 8, XR = XT / 8 / 64, PT = N_STEP * N_ROWS, PR = PT / 8 / 64, DB = D / 16;
    __shared__ __align__(16) T x_a_all[4 * XT];
    __shared__ __align__(16) T x_b_all[4 * XT];
    __shared__ __align__(16) T p_a_all[4 * PT];
    __shared__ __align__(16) T p_b_all[4 * PT];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    T *const x_a = x_a_all + wave * XT;
    T *const x_b = x_b_all + wave * XT;
    T *const p_a = p_a_all + wave * PT;
    T *const p_b = p_b_all + wave * PT;
    const int64_t lid = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (lid >= total_wg) return;
    const int64_t bh = lid / nkb;
    const int k0 = (int)(lid % nkb) * N_ROWS;   // under the causal rule the first keys have the most query rows
    const T *Pp = P + bh * (int64_t)S * S;
    const T *Xp = X + bh * (int64_t)S * D;
    T *Op = O + bh * (int64_t)S * D;
    auto issue = [&](int j, T *xdst, T *pdst) {   // rows past the sequence re-read the last row, keys past it the first chunk
#pragma unroll
        for (int r = 0; r < XR; ++r) {
            const int slot = r * 64 + lane, row = slot / XC, c = (slot % XC) ^ v_swizzle<D>(row);
            int pr = j * N_STEP + row;
            pr = pr >= S ? S - 1 : pr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Xp + (int64_t)pr * D + c * 8), (lds_void_t *)(xdst + r * 64 * 8), 16, 0, 0);
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

// ---- the transposed product --------------------------------------------------------------------------------------
// O[k, :] = sum over p of P[p, k] X[p, :], p >= k only when causal: the gradients that the two matrix products of the
// attention leave on their right-hand operands (dV = P^T dO, dK = G^T Q), whose left factor is only defined - and only
// read - on and below the diagonal.
//
// A workgroup owns 128 keys (output rows; 32 per wavefront, two blocks of 16) and walks the query rows from its first
// key downwards in blocks of 64.  O^T += X^T P on 16x16x32 MFMAs with the query rows as contraction index: both
// operands are copied global -> LDS asynchronously as row-major blocks (64 rows of X, 64 rows x 128 keys of P; double
// buffered, 16-byte chunks XOR-swizzled by row) and both fragments come out of them through the LDS transpose read,
// which hands a lane four consecutive rows of one column: X^T with the head dim as operand row, P with the key as
// operand column.  P is streamed from memory once; the X blocks are re-read from L2 by every key block above them.
constexpr int T_KB = 32 * P_WAVES;  // keys per workgroup
constexpr int T_PB = 64;            // query rows per step
constexpr int T_KS = T_PB / 32;

template <typename T, int D>
__global__ __launch_bounds__(P_NT, P_OCC) void causal_ptx_kernel(const T *__restrict__ P, const T *__restrict__ X,
                                                                 T *__restrict__ O, int S, int causal, int nkb, int64_t total_wg,
                                                                 int64_t per_xcd, float scale)
{
    constexpr int XT = T_PB * D, PT = T_PB * T_KB;  // elements per X block / P tile
    constexpr int XC = D / 8, PC = T_KB / 8;        // 16-byte chunks per row
    constexpr int XR = XT / 8 / P_NT, PR = PT / 8 / P_NT;
    static_assert(XT / 8 % P_NT == 0 && PT / 8 % P_NT == 0, "whole copy rounds");
    constexpr int DB = D / 16;
    __shared__ __align__(16) T x_a[XT];
    __shared__ __align__(16) T x_b[XT];
    __shared__ __align__(16) T p_a[PT];
    __shared__ __align__(16) T p_b[PT];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    const int64_t lid = (int64_t)(blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (lid >= total_wg) return;
    // two key blocks per workgroup, pi and nkb-1-pi: under the causal rule the first has the most query rows and the
    // second the fewest, so that every workgroup gets the same amount of work
    const int npairs = (nkb + 1) / 2;
    const int pi = (int)(lid % npairs);
    const int64_t bh = lid / npairs;
    const T *Pp = P + bh * (int64_t)S * S;
    const T *Xp = X + bh * (int64_t)S * D;
    T *Op = O + bh * (int64_t)S * D;
  for (int half = 0; half < 2; ++half) {
    const int kb = half == 0 ? pi : nkb - 1 - pi;
    if (half == 1 && kb == pi) break;  // odd number of blocks: the middle one is alone
    const int k0 = kb * T_KB;
    if (half == 1) __syncthreads();    // the buffers are reused: everybody has finished reading them

    // block j = query rows 64j ..; rows past the sequence re-read the last row, keys past it the block's first chunk:
    // what they bring in is masked (rows) or belongs to output rows that are not stored (keys)
    auto issue = [&](int j, T *xdst, T *pdst) {
#pragma unroll
        for (int r = 0; r < XR; ++r) {
            const int slot = r * P_NT + tid;
            const int row = slot / XC, c = (slot % XC) ^ v_swizzle<D>(row);
            int pr = j * T_PB + row;
            pr = pr >= S ? S - 1 : pr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Xp + (int64_t)pr * D + c * 8),
                                             (lds_void_t *)(xdst + (r * P_NT + wave * 64) * 8), 16, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < PR; ++r) {
            const int slot = r * P_NT + tid;
            const int row = slot / PC;
            int c = (slot % PC) ^ v_swizzle<T_KB>(row);
            if (k0 + c * 8 >= S) c = 0;
            int pr = j * T_PB + row;
            pr = pr >= S ? S - 1 : pr;
            __builtin_amdgcn_global_load_lds((glb_void_t *)(Pp + (int64_t)pr * S + k0 + c * 8),
                                             (lds_void_t *)(pdst + (r * P_NT + wave * 64) * 8), 16, 0, 0);
        }
    };
    // operand fragment out of a row-major block of LD columns: contraction slots t = 0..7 of step ks are the block's rows
    // 32ks + 8kg + t, the operand's row / column is column 16*blk + ln of the block
    auto frag_of = [&](const T *tile, auto ldc, int ks, int blk) {
        constexpr int LD = decltype(ldc)::value;
        const int row_a = ks * 32 + kg * 8 + (ln >> 2), row_b = row_a + 4;
        const int ch = blk * 2 + ((ln & 3) >> 1);
        const int sub = (ln & 1) * 4;
        const T *pa = tile + row_a * LD + ((ch ^ v_swizzle<LD>(row_a)) * 8) + sub;
        const T *pb = tile + row_b * LD + ((ch ^ v_swizzle<LD>(row_b)) * 8) + sub;
        struct { v4s_t a, b; } both = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pa),
                                       __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)pb)};
        return __builtin_bit_cast(frag8<T>, both);
    };

    // this lane's two output rows (keys)
    int krow[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) krow[rb] = k0 + (wave * 2 + rb) * 16 + ln;
    const int j_start = causal ? k0 / T_PB : 0, j_end = (S - 1) / T_PB;
    f32x4 oacc[2][DB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[rb][db] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    issue(j_start, x_a, p_a);

    auto step = [&](int j, const T *Xb, const T *Pb, T *Xn, T *Pn) __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0);  // block j has arrived
        __syncthreads();                // for every wavefront; reads of the other buffers are finished
        if (j < j_end) issue(j + 1, Xn, Pn);
        // P fragments of this wavefront's two key blocks; query rows above the key (causal: P is undefined there) or
        // past the sequence count as 0
        frag8<T> pf[2][T_KS];
        const int pbase = j * T_PB;
        const bool edge = pbase + T_PB > S || (causal && pbase < k0 + T_KB - 1);  // (wavefront-uniform)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int ks = 0; ks < T_KS; ++ks) {
                pf[rb][ks] = frag_of(Pb, std::integral_constant<int, T_KB>{}, ks, wave * 2 + rb);
                if (edge) {
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const int p = pbase + ks * 32 + kg * 8 + t;
                        if (p >= S || (causal && p < krow[rb])) pf[rb][ks].v[t] = from_float<T>(0.0f);
                    }
                }
            }
        frag8<T> xf[2];
        xf[0] = frag_of(Xb, std::integral_constant<int, D>{}, 0, 0);
#pragma unroll
        for (int blk = 0; blk < T_KS * DB; ++blk) {
            const int ks = blk / DB, db = blk % DB;
            if (blk + 1 < T_KS * DB) xf[(blk + 1) & 1] = frag_of(Xb, std::integral_constant<int, D>{}, (blk + 1) / DB, (blk + 1) % DB);
            __builtin_amdgcn_sched_barrier(0);  // (the instruction scheduler would move the reads back behind the products)
            mma16(oacc[0][db], xf[blk & 1], pf[0][ks]);
            mma16(oacc[1][db], xf[blk & 1], pf[1][ks]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int j = j_start;;) {
        step(j, x_a, p_a, x_b, p_b);
        if (++j > j_end) break;
        step(j, x_b, p_b, x_a, p_a);
        if (++j > j_end) break;
    }

#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        if (krow[rb] >= S) continue;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            struct alignas(8) quad { T v[4]; } out;
#pragma unroll
            for (int v = 0; v < 4; ++v) out.v[v] = from_float<T>(oacc[rb][db][v] * scale);
            *reinterpret_cast<quad *>(Op + (int64_t)krow[rb] * D + db * 16 + kg * 4) = out;
        }
    }
  }
}

// MTA_PV_SPLIT in the environment: 1 / 2 / 3 = always one group / two groups / the narrow kernels (comparison switch)
int pv_force()
{
    static const int force = [] { const char *e = getenv("MTA_PV_SPLIT"); return e ? atoi(e) : 0; }();
    return force;
}
// Whether a product whose wide grid has that many workgroups (pairs of 128-row blocks) runs on the narrow kernels.  The line
// lies where the two meet (us, wide -> narrow; P V in the triangular layout / P^T X): B1 H16 D128 S512 16.6 -> 6.7 / 17.8 -> 6.6;
// S1024 24.3 -> 12.8 / 25.3 -> 10.8; S2048 (128 workgroups) 48.8 -> 27.3 / 40.8 -> 24.5; S4096 (256) 95 -> 118 / 77 -> 102;
// B4 S1024 (256) 33.4 -> 37.5 / 27.7 -> 34.0; D64, half the bytes per V row: B1 H32 S2048 (256) 45.3 -> 36.1 / 30.1 -> 30.9,
// B1 H16 S4096 (256) 93 -> 88 / 61 -> 70.
bool narrow_grid(int64_t wide_wg, int most)
{
    if (pv_force()) return pv_force() == 3;
    return wide_wg <= most;
}

template <typename T, int D>
int launch_t(const void *p, const void *x, void *o, int64_t B, int64_t H, int64_t S, int causal, float scale, hipStream_t st)
{
    int nkb = (int)((S + T_KB - 1) / T_KB);
    int64_t total_wg = B * H * ((nkb + 1) / 2);
    const bool narrow = narrow_grid(total_wg, 192);
    if (narrow) {
        nkb = (int)((S + N_ROWS - 1) / N_ROWS);
        total_wg = B * H * nkb;
    }
    const int64_t per_xcd = (total_wg + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL) return MTA_ERR_SHAPE;
    dim3 grid((unsigned)(per_xcd * 8));
    if (narrow) {
        auto kern = causal_ptx_narrow_kernel<T, D>;
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (const T *)p, (const T *)x, (T *)o, (int)S, causal, nkb, total_wg, per_xcd, scale);
        return launch_status();
    }
    auto kern = causal_ptx_kernel<T, D>;
    hipLaunchKernelGGL(kern, grid, dim3(P_NT), 0, st, (const T *)p, (const T *)x, (T *)o, (int)S, causal, nkb, total_wg,
                       per_xcd, scale);
    return launch_status();
}

template <typename T, int D>
int launch(const void *p, const void *v, void *o, int64_t B, int64_t H, int64_t S, int causal, hipStream_t st,
           const int *band_lo = nullptr, int tri_gl = 0, float scale = 1.0f)
{
    int nqb = (int)((S + P_BQ - 1) / P_BQ);
    int64_t total_wg = B * H * ((nqb + 1) / 2);
    const bool narrow = narrow_grid(total_wg, D == 64 ? 256 : 192);
    if (narrow) {
        nqb = (int)((S + N_ROWS - 1) / N_ROWS);
        total_wg = B * H * nqb;
    }
    const int64_t per_xcd = (total_wg + 7) / 8;
    if (per_xcd * 8 > 0x7fffffffLL) return MTA_ERR_SHAPE;
    dim3 grid((unsigned)(per_xcd * 8));
    if (narrow) {
        auto kern = causal_pv_narrow_kernel<T, D>;
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, (const T *)p, (const T *)v, (T *)o, (int)S, causal, nqb, total_wg, per_xcd,
                           band_lo, (int)H, tri_gl, scale);
        return launch_status();
    }
    // a grid of at most one workgroup per CU runs the two-group instance (key blocks split between them)
    const bool split = pv_force() ? pv_force() == 2 : total_wg <= device_cu_count();
    if (split) {
        auto kern = causal_pv_kernel<T, D, 2>;
        hipLaunchKernelGGL(kern, grid, dim3(P_NT * 2), 0, st, (const T *)p, (const T *)v, (T *)o, (int)S, causal, nqb,
                           total_wg, per_xcd, band_lo, (int)H, tri_gl, scale);
    } else {
        auto kern = causal_pv_kernel<T, D, 1>;
        hipLaunchKernelGGL(kern, grid, dim3(P_NT), 0, st, (const T *)p, (const T *)v, (T *)o, (int)S, causal, nqb,
                           total_wg, per_xcd, band_lo, (int)H, tri_gl, scale);
    }
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
    if (!p || !x || !o) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (B <= 0 || H <= 0 || S <= 0 || S > (1 << 24) || B * H > 65535) return MTA_ERR_SHAPE;
    if (D != 64 && D != 128) return MTA_ERR_HEAD_DIM;
    if (!aligned_to(p, 16) || !aligned_to(x, 16) || !aligned_to(o, 16)) return MTA_ERR_ALIGN;
    if (io_dtype == MTA_F32 || S % 8 != 0) return MTA_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    if (io_dtype == MTA_BF16)
        return D == 64 ? launch_t<bf16_t, 64>(p, x, o, B, H, S, causal, scale, st) : launch_t<bf16_t, 128>(p, x, o, B, H, S, causal, scale, st);
    return D == 64 ? launch_t<f16_t, 64>(p, x, o, B, H, S, causal, scale, st) : launch_t<f16_t, 128>(p, x, o, B, H, S, causal, scale, st);
}
