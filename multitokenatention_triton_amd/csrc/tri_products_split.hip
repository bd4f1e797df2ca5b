// The lower-triangle scores of fp32 operands (C[p,q] = sum_d A[p,d] B[q,d], q <= p: Q K^T, dP = dO V^T) on the bf16 matrix cores, with
// the 32 bits kept (split.hpp): the larger grids of tri_products_f32.hip.  The result's vectors, and nothing else above the
// diagonal, are written as there.
//
// A workgroup of four wavefronts takes 128 query rows and a run of steps of 64 keys (32 at D = 128).  A wavefront keeps its 32 rows split
// in registers; the keys are loaded four dims per lane, two steps ahead, split on the way to one of two LDS buffers between the
// products of the step before (rows of bf16, 16-byte chunks XOR-swizzled by the key), and serve all four wavefronts.
// What bounds it is the CU's path to the L2, which the scores (out) and the keys (in, half as much at D = 64, as much at 128) pass: 4.6
// TB/s together at B1 H16 S2048 D64.  On v_mfma_f32_16x16x4f32, in slabs of 16 dims of both operands, it was the matrix rate and the
// loads of two operands per tile.  us, those -> this: D64 B2 H16 S512 15.1 -> 13.2, B1 H12 S800 13.9 -> 12.4, B1 H16 S1024 22.2 -> 18.3, B1
// H32 S1024 36.6 -> 27.3, B1 H16 S2048 61.5 -> 41.9; D128 B1 H16 S512 14.7 -> 12.1, B1 H32 S1024 64.5 -> 40.9, B1 H16 S2048 102 -> 62.7.  Error
// against 64 bits (2-norm): D64 1.4e-7 -> 0.5e-7, D128 2.0e-7 -> 0.65e-7.
// Runs of 1 | 2 | 4 steps: D64 B1 H16 S1024 (1152 steps) 18.7 | 17.6 | 20.4, B1 H32 S1024 (2304) 34.4 | 31.9 | 28.8, B1 H16 S2048 (4352) 56.3 | 46.3
// | 42.1; D128, twice as many, B2 H16 S512 17.5 | 17.3 | 18.2, B1 H16 S2048 88.0 | 70.8 | 63.8.
// Operands are split 2^24 times as large (split.hpp); a wavefront with a sum that is not finite then forms its step again with fp32
// products.  (Unscaled, with a look at the sums, which cannot tell small operands against large ones: up to 5 % faster, and up to 12000
// times the error of 32-bit sums.  us with nothing in the caches, that -> this: D64 B1 H16 S512 9.8 -> 9.8, S1024 19.3 -> 20.2, S2048 54.0 -> 53.8;
// D128 11.6 -> 12.1, 27.1 -> 27.4, 68.3 -> 69.1.)
// (P V and P^T X in this form, with a V block per 64 rows: as fast as on the fp32 instructions - B1 H32 S1024 D64 26.1 | 28.3, B1 H32 S2048 D128 155 |
// 138 us - since V passes that path as often as P does.)
#include "split.hpp"
#include "strip_common.hpp"

namespace {
using namespace mta;

constexpr int SS_ROWS = 128;                                    // query rows of a workgroup, 32 per wavefront
template <int D> constexpr int ss_keys() { return 4096 / D; }   // keys of a step

// items of a head: blocks of query rows from the last to the first, each cut into runs of `run` steps
__host__ __device__ __forceinline__ int ss_steps(int block, int S, int keys)
{
    const int last = (block + 1) * SS_ROWS < S ? (block + 1) * SS_ROWS : S;
    return (last + keys - 1) / keys;
}

template <int D>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void lower_scores_split(const float *__restrict__ A, const float *__restrict__ Bm, float *__restrict__ C, int S,
                                                                         int heads, int items, int run)
{
    constexpr int BK = ss_keys<D>(), KS = D / 32, NCB = BK / 16, CPR = D / 8, QUADS = BK * D / 4 / 256, PLANE = BK * D;
    __shared__ __align__(16) uint16_t kt[2][3 * PLANE];
    int bh, rank;
    if (!longest_first(heads, items, 0, bh, rank)) return;
    int block = (S + SS_ROWS - 1) / SS_ROWS - 1;
    for (int n; rank >= (n = (ss_steps(block, S, BK) + run - 1) / run); --block) rank -= n;
    const int j0 = rank * run, j_all = ss_steps(block, S, BK), j_end = j0 + run < j_all ? j0 + run : j_all;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 15, kg = lane >> 4;
    const float *Ap = A + (int64_t)bh * S * D, *Bp = Bm + (int64_t)bh * S * D;
    float *Cp = C + (int64_t)bh * S * S;
    const int w0 = block * SS_ROWS + wave * 32;                  // this wavefront's rows

    // (rows of the scores that lie outside the tensor: their stores are dropped)
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(Cp + (int64_t)(w0 < S ? w0 : 0) * S, 0, (int)(w0 < S ? 32u * (unsigned)S * 4u : 0u), 0x00027000);
    // a step's keys: four dims per lane and round (keys past the sequence re-read the last one: nobody stores their scores)
    f32x4 raw[QUADS];
    auto fetch = [&](int j, int i) __attribute__((always_inline)) {
        const int slot = i * 256 + tid, key = j * BK + slot / (D / 4), kc = key < S ? key : S - 1;
        raw[i] = *reinterpret_cast<const f32x4 *>(Bp + (int64_t)kc * D + slot % (D / 4) * 4);
    };
    // row of a key: 16-byte chunk c at position c ^ key % CPR
    auto stage = [&](int i, uint16_t *to) __attribute__((always_inline)) {
        const int slot = i * 256 + tid, key = slot / (D / 4), q = slot % (D / 4);
        uint32_t a[3], b[3];
        split2<3>(raw[i][0] * SPLIT_UP, raw[i][1] * SPLIT_UP, a);
        split2<3>(raw[i][2] * SPLIT_UP, raw[i][3] * SPLIT_UP, b);
        uint16_t *at = to + key * D + ((q >> 1) ^ (key & (CPR - 1))) * 8 + (q & 1) * 4;
#pragma unroll
        for (int s = 0; s < 3; ++s) *reinterpret_cast<uint2 *>(at + s * PLANE) = make_uint2(a[s], b[s]);
    };
#pragma unroll
    for (int i = 0; i < QUADS; ++i) fetch(j0, i);
    frag8<bf16_t> a[2][KS][3];                                   // this wavefront's rows, split
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
        const int p = w0 + rb * 16 + ln < S ? w0 + rb * 16 + ln : S - 1;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const f32x4 lo = *reinterpret_cast<const f32x4 *>(Ap + (int64_t)p * D + ks * 32 + kg * 8);
            const f32x4 hi = *reinterpret_cast<const f32x4 *>(Ap + (int64_t)p * D + ks * 32 + kg * 8 + 4);
            split8(lo * SPLIT_UP, hi * SPLIT_UP, a[rb][ks]);
        }
    }
#pragma unroll
    for (int i = 0; i < QUADS; ++i) stage(i, kt[0]);
#pragma unroll
    for (int i = 0; i < QUADS; ++i) fetch(j0 + 1 < j_end ? j0 + 1 : j0, i);
    __syncthreads();
    // acc[cb][rb][v]: key q0 + 16 cb + 4 kg + v of query row w0 + 16 rb + ln.  A step's scores are stored at the top of the next one, and
    // with buffer stores, which drop what lies outside: so there are as many of them between the loads of keys and the wait for
    // these on every path, and it does not become a wait for the stores (loads and stores complete on one counter).
    f32x4 acc[NCB][2];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) acc[cb][rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    auto store = [&](int q0, bool none) __attribute__((always_inline)) {
        const bool inside = w0 + 32 <= S && q0 + BK - 1 <= w0 && !none;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const int p = w0 + rb * 16 + ln;
#pragma unroll
            for (int cb = 0; cb < NCB; ++cb) {
                const int q = q0 + cb * 16 + kg * 4;
                unsigned at = (unsigned)((rb * 16 + ln) * S + q) * 4u;
                if (!inside) {
                    if (p >= S || q > p || none) at = 0xffffffffu;
#pragma unroll
                    for (int v = 1; v < 4; ++v) acc[cb][rb][v] = q + v > p ? 0.0f : acc[cb][rb][v];
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[cb][rb]), rows, (int)at, 0, 0);
            }
        }
    };
    bool again = true;      // the step's scores are not in acc
    for (int j = j0, n = 0; j < j_end; ++j, n ^= 1) {
        store((j - 1) * BK, again);
        const int q0 = j * BK, jn = j + 2 < j_end ? j + 2 : j;
        const bool live = w0 < S && q0 <= w0 + 31;
        const uint16_t *from = kt[n] + ln * D;
        frag8<bf16_t> f[2][3];
        auto read = [&](int m) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < 3; ++s)
                f[m & 1][s] = *reinterpret_cast<const frag8<bf16_t> *>(from + s * PLANE + m / KS * 16 * D + (((m % KS) * 4 + kg) ^ (ln & (CPR - 1))) * 8);
        };
        read(0);
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            f32x4 small[2], big[2];
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) small[rb] = big[rb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const int m = cb * KS + ks;
                if (m + 1 < NCB * KS) read(m + 1);
                if (live) {
#pragma unroll
                    for (int t = 0; t < 6; ++t) {
                        constexpr int BX[6] = {2, 0, 1, 1, 0, 0}, AX[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb) mma16(t == 5 ? big[rb] : small[rb], f[m & 1][BX[t]], a[rb][ks][AX[t]]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) acc[cb][rb] = (big[rb] + small[rb]) * (1.0f / SPLIT_UP / SPLIT_UP);
            // the next step's keys to the other buffer, those of the one behind it asked for
#pragma unroll
            for (int i = cb * QUADS / NCB; i < (cb + 1) * QUADS / NCB; ++i) {
                stage(i, kt[n ^ 1]);
                fetch(jn, i);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        again = live && not_finite<NCB * 2>(&acc[0][0]);
        if (again) {   // fp32 products, from memory: contraction d = 16s + 4kg + t, four steps' operand in a lane's vector of its row
#pragma unroll 1
            for (int e = 0; e < NCB * 2; ++e) {
                const int qa = q0 + e / 2 * 16, p = w0 + (e & 1) * 16 + ln;
                const float *ar = Ap + (int64_t)(p < S ? p : S - 1) * D + kg * 4, *br = Bp + (int64_t)(qa + ln < S ? qa + ln : S - 1) * D + kg * 4;
                f32x4 sum{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
                for (int s = 0; s < D / 16; ++s) {
                    const f32x4 av = *reinterpret_cast<const f32x4 *>(ar + 16 * s), bv = *reinterpret_cast<const f32x4 *>(br + 16 * s);
#pragma unroll
                    for (int t = 0; t < 4; ++t) mma4(sum, bv[t], av[t]);
                }
                const int q = qa + kg * 4;
                if (p >= S || q > p) continue;
#pragma unroll
                for (int v = 1; v < 4; ++v) sum[v] = q + v > p ? 0.0f : sum[v];
                *reinterpret_cast<f32x4 *>(Cp + (int64_t)p * S + q) = sum;
            }
        }
        __syncthreads();
    }
    store((j_end - 1) * BK, again);
}

template <int D>
int launch_scores(const void *a, const void *b, void *c, int64_t heads, int64_t S, int64_t steps, hipStream_t st)
{
    const int run = (steps < 2000 ? 2 : 4) * (D / 64), blocks = (int)((S + SS_ROWS - 1) / SS_ROWS);
    int64_t items = 0;
    for (int i = 0; i < blocks; ++i) items += (ss_steps(i, (int)S, ss_keys<D>()) + run - 1) / run;
    const int64_t grid = (heads * items + 7) / 8 * 8;
    if (grid > 0x7fffffffLL) return MTA_ERR_SHAPE;
    hipLaunchKernelGGL(lower_scores_split<D>, dim3((unsigned)grid), dim3(256), 0, st, (const float *)a, (const float *)b, (float *)c, (int)S, (int)heads,
                       (int)items, run);
    return launch_status();
}
}  // namespace

int mta::lower_scores_split_launch(const void *a, const void *b, void *c, int64_t heads, int64_t S, int64_t D, hipStream_t st)
{
    int64_t steps = 0;   // blocks of 128 rows x 64 keys
    for (int i = 0; i < (int)((S + SS_ROWS - 1) / SS_ROWS); ++i) steps += ss_steps(i, (int)S, 64);
    return D == 64 ? launch_scores<64>(a, b, c, heads, S, heads * steps, st) : launch_scores<128>(a, b, c, heads, S, heads * steps, st);
}
