// Both gradients of the head mixing in one read of its output gradient, alone and behind the softmax gradient:
//
//   dx[n,i,p,q] = sum_o w[o,i] dy[n,o,p,q]        dw[o,i] = sum_{n,p,q} dy[n,o,p,q] x[n,i,p,q]      (causal: only q <= p)
//
// and the same with dy = s * (ds - sum_k s ds) formed on the way from a row of probabilities s and their gradient ds
// (rounded to the I/O dtype, as the softmax gradient leaves it in memory).  The reference runs these as three kernels behind
// torch's softmax gradient (triton_linear_head.py:144-278, 330-368; mta_attention_triton.py:75-79).
//
// What bounds them is memory, so what counts is the passes over score tensors: as separate kernels five (dx: two; dw: two, dy
// among them) and seven with the softmax gradient, here three and four.  us, separate | here and the same behind the softmax gradient
// (causal, lower triangle, the summing of dw included): bf16 B2 H8 S2048 51 | 38, 94 | 58; B1 H16 S2048 52 | 39, 98 | 66 (5.2 and
// 4.1 TB/s); B1 H16 S4096 228 | 152, 382 | 292; B1 H32 S2048 120 | 81, 214 | 170; fp32 B1 H32 S1024 60 | 43, 105 | 75; bf16 groups
// of 4 of B2 H32 S2048, filled above the diagonal: 260 | 225.
//
// Two ways to hold a tile, by the size of the mixing group:
//  * 2 or 4 heads (lane_*): a lane owns one 16-byte vector of keys of all heads of its group; the mix and the G x G running sums of
//    dw are products inside the lane (packed dot products where weights and data share a 16-bit type: half the vector
//    instructions of the fp32 form), the lanes' sums are added once at the end.
//  * 8, 12, 16 or 32 heads (dense): a wavefront owns 16 vectors of keys of all heads.  Lane (ln, kg) loads vector ln of a quarter
//    of the heads, which is the B operand of the mix on the matrix cores after two byte permutes (16-bit; fp32: as it lies) -
//    the layout of headmix_dense16.  dw = dy x^T contracts over keys and wants a lane to hold keys of one head: dy goes
//    through a wavefront-private tile in LDS (rows of 288 bytes: conflict-free 16-byte reads), x comes from memory in that
//    layout (64 contiguous bytes per head and instruction, four of them back to back).  8 heads in the lane form hold 64 sums
//    per lane, two wavefronts per SIMD: 60 and 106 us at bf16 B2 S2048 where this one takes 38 and 58.
// Partial sums of dw are fp32: registers over a workgroup's share, one matrix per workgroup, added in a fixed order.
//
// In the kernels behind the softmax gradient a row's workgroup walks "load, sum, barrier, load x, products, store".  Measured
// and not kept (bf16 B1 H16 S2048, 66 us): x loaded ahead of the barrier 69, the next row's vectors loaded ahead 120 (they spill),
// 16 wavefronts of one tile instead of 8 of two 66.  Four tiles per wavefront (rows of more than 2048 keys, fp32 1024) hold 256
// registers and spill: 104 to 120 bytes a lane with 12 and 16 heads in 16 bits, 52 with 16 in fp32; so do 32 heads in 16 bits, 8 bytes
// with one tile and 44 with two.  With the tile-at-a-time order below that is what is left; B1 H16 S4096 runs at 3.7 TB/s all the same
// (4.1 at S2048, which does not spill).
#include "common.hpp"
#include "mfma.hpp"

namespace {
using namespace mta;

typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));

// ---- pieces both layouts share -------------------------------------------------------------------------------------------
// 16 bytes at a wavefront-uniform address plus a lane's 32-bit byte offset (a group of heads is smaller than 4 GB)
template <bool STREAM> __device__ __forceinline__ u4 load_vec(const void *base, unsigned off)
{
    const u4 *p = reinterpret_cast<const u4 *>(static_cast<const char *>(base) + off);
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    return *p;
}
__device__ __forceinline__ u4 *vec_at(void *base, unsigned off) { return reinterpret_cast<u4 *>(static_cast<char *>(base) + off); }

// dword u of a vector as fp32 values (two of a 16-bit type), and back
template <typename T> __device__ __forceinline__ void widen(unsigned v, float (&f)[vec_of<T>::n / 4])
{
    if constexpr (vec_of<T>::n == 8) unpack2<T>(v, f[0], f[1]);
    else f[0] = __uint_as_float(v);
}
template <typename T> __device__ __forceinline__ unsigned narrow(const float (&f)[vec_of<T>::n / 4])
{
    if constexpr (vec_of<T>::n == 8) return pack2<T>(f[0], f[1]);
    else return __float_as_uint(f[0]);
}

// sum over the 16 lanes of a row of lanes, in all of them
template <int CTRL> __device__ __forceinline__ float dpp_add(float v)
{
    return v + __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float row_sum(float v)
{
    v = dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x141>(v);  // row_half_mirror
    return dpp_add<0x140>(v);  // row_mirror
}

__device__ __forceinline__ int last_key(int p, int Q, int causal) { return causal && p < Q - 1 ? p : Q - 1; }

// sum over a vector of s * ds, both masked beyond `last`
template <typename T> __device__ __forceinline__ float dot_vec(u4 &s, u4 &ds, int key, int last, float sum)
{
    if (key + vec_of<T>::n - 1 > last) {
        zero_beyond<T>(s, key, last);
        zero_beyond<T>(ds, key, last);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float a[vec_of<T>::n / 4], b[vec_of<T>::n / 4];
        widen<T>(s[u], a);
        widen<T>(ds[u], b);
#pragma unroll
        for (int e = 0; e < vec_of<T>::n / 4; ++e) sum = fmaf(a[e], b[e], sum);
    }
    return sum;
}

// s * (ds - dot), rounded
template <typename T> __device__ __forceinline__ u4 softmax_grad(const u4 &s, const u4 &ds, float dot)
{
    u4 r;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float a[vec_of<T>::n / 4], b[vec_of<T>::n / 4];
        widen<T>(s[u], a);
        widen<T>(ds[u], b);
#pragma unroll
        for (int e = 0; e < vec_of<T>::n / 4; ++e) a[e] *= b[e] - dot;
        r[u] = narrow<T>(a);
    }
    return r;
}

// The chunks of KEYS keys of all rows (N*P of them), dealt to wavefronts one by one.  Rows are taken in pairs (2k, 2k+1) of an
// order that interleaves short and long ones (0, P-1, 1, P-2, ...), so that under the causal rule every pair holds about P + 1
// attended positions; a pair has `slots` places, of which few are empty.  `whole`: chunks beyond the diagonal count too (they
// get the fill).
template <int KEYS> struct chunk_walk {
    unsigned k, pairs, rows, pair_step, slot_step, slots, i;
    int P, Q, causal;
    bool whole;
    unsigned n;          // the chunk: batch entry, row, its last attended key, first key
    int p, last, q0;

    __device__ __forceinline__ chunk_walk(unsigned rows_, int P_, int Q_, int causal_, bool whole_, unsigned slots_, unsigned wid, unsigned nwaves)
        : k(wid / slots_), pairs((rows_ + 1) / 2), rows(rows_), pair_step(nwaves / slots_), slot_step(nwaves % slots_), slots(slots_),
          i(wid % slots_), P(P_), Q(Q_), causal(causal_), whole(whole_) {}
    __device__ __forceinline__ void advance()
    {
        k += pair_step;
        i += slot_step;
        if (i >= slots) {
            i -= slots;
            ++k;
        }
    }
    __device__ __forceinline__ bool find()   // the chunk of the place at or after (k, i)
    {
        while (k < pairs) {
            int c = (int)i;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const unsigned rid = 2 * k + half;
                if (rid >= rows) break;
                const unsigned j = rid % (unsigned)P;
                n = rid / (unsigned)P;
                p = (j & 1) ? P - 1 - (int)(j >> 1) : (int)(j >> 1);
                last = last_key(p, Q, causal);
                const int reach = whole ? Q - 1 : last;
                if (c * KEYS <= reach) {
                    q0 = c * KEYS;
                    return true;
                }
                c -= reach / KEYS + 1;
            }
            advance();
        }
        return false;
    }
};

// ---- groups of 2 or 4 heads: a lane holds them all -------------------------------------------------------------------------
// The group's weights in scalar registers: fp32 values w[o][i], or (PAIRS: 16-bit data, weights of the same dtype) the pairs
// (w[2j][i], w[2j+1][i]) that the packed dot products take.
template <typename T, int G, bool PAIRS> struct lane_weights {
    unsigned v[PAIRS ? G * G / 2 : G * G];

    __device__ __forceinline__ lane_weights(const void *wp, int w_dtype, int g, int C)
    {
        auto at = [&](int o, int i) { return (int64_t)(g * G + o) * C + g * G + i; };
        if constexpr (PAIRS) {
            const uint16_t *w = reinterpret_cast<const uint16_t *>(wp);
#pragma unroll
            for (int e = 0; e < G * G / 2; ++e)
                v[e] = (unsigned)__builtin_amdgcn_readfirstlane((int)(w[at(2 * (e / G), e % G)] | (unsigned)w[at(2 * (e / G) + 1, e % G)] << 16));
        } else {
#pragma unroll
            for (int e = 0; e < G * G; ++e)
                v[e] = (unsigned)__builtin_amdgcn_readfirstlane((int)__float_as_uint(load_any(wp, w_dtype, at(e / G, e % G))));
        }
    }
};

template <typename T> __device__ __forceinline__ float dot2(unsigned a, unsigned b, float c)
{
    if constexpr (__is_same(T, bf16_t))
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(mta_bf16x2, a), __builtin_bit_cast(mta_bf16x2, b), c, false);
    else
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(mta_f16x2, a), __builtin_bit_cast(mta_f16x2, b), c, false);
}

// out = w^T dy for the keys of a vector; acc += dy x^T
template <typename T, int G, bool PAIRS>
__device__ __forceinline__ void lane_tile(const u4 (&dy)[G], const u4 (&x)[G], const lane_weights<T, G, PAIRS> &w, float (&acc)[G * G], u4 (&out)[G])
{
    constexpr int E = vec_of<T>::n / 4;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if constexpr (PAIRS) {   // two keys: the mix contracts over pairs of heads, dw over the pair of keys
            unsigned lo[G / 2], hi[G / 2];
#pragma unroll
            for (int j = 0; j < G / 2; ++j) {
                lo[j] = __builtin_amdgcn_perm(dy[2 * j + 1][u], dy[2 * j][u], 0x05040100u);
                hi[j] = __builtin_amdgcn_perm(dy[2 * j + 1][u], dy[2 * j][u], 0x07060302u);
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
                for (int j = 0; j < G / 2; ++j) {
                    s0 = dot2<T>(lo[j], w.v[j * G + i], s0);
                    s1 = dot2<T>(hi[j], w.v[j * G + i], s1);
                }
                out[i][u] = pack2<T>(s0, s1);
            }
#pragma unroll
            for (int o = 0; o < G; ++o)
#pragma unroll
                for (int i = 0; i < G; ++i) acc[o * G + i] = dot2<T>(dy[o][u], x[i][u], acc[o * G + i]);
        } else {
            float d[G][E], xx[G][E];
#pragma unroll
            for (int h = 0; h < G; ++h) {
                widen<T>(dy[h][u], d[h]);
                widen<T>(x[h][u], xx[h]);
            }
#pragma unroll
            for (int i = 0; i < G; ++i) {
                float s[E];
#pragma unroll
                for (int e = 0; e < E; ++e) s[e] = 0.0f;
#pragma unroll
                for (int o = 0; o < G; ++o)
#pragma unroll
                    for (int e = 0; e < E; ++e) s[e] = fmaf(__uint_as_float(w.v[o * G + i]), d[o][e], s[e]);
                out[i][u] = narrow<T>(s);
            }
#pragma unroll
            for (int o = 0; o < G; ++o)
#pragma unroll
                for (int i = 0; i < G; ++i)
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[o * G + i] = fmaf(d[o][e], xx[i][e], acc[o * G + i]);
        }
    }
}

// a wavefront's sums into 4 rows of `red` (one per row of 16 lanes)
template <int G> __device__ __forceinline__ void lane_deposit(const float (&acc)[G * G], float (*red)[G * G], int wave, int lane)
{
#pragma unroll
    for (int e = 0; e < G * G; ++e) {
        const float s = row_sum(acc[e]);
        if ((lane & 15) == (e & 15)) red[4 * wave + (lane >> 4)][e] = s;
    }
}

constexpr int NT = 256;

template <typename T, int G, bool PAIRS, bool STREAM>
__global__ __launch_bounds__(NT) void lane_grads(const T *__restrict__ x, const T *__restrict__ dy, const void *__restrict__ w, T *__restrict__ dx,
                                                 float *__restrict__ partial, unsigned rows, int C, int P, int Q, int causal, unsigned slots,
                                                 unsigned parts, int w_dtype)
{
    constexpr int V = vec_of<T>::n, KEYS = 64 * V;
    __shared__ float red[4 * NT / 64][G * G];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int g = (int)(blockIdx.x / parts);
    const unsigned bi = blockIdx.x % parts;
    const int64_t plane = (int64_t)P * Q;
    const lane_weights<T, G, PAIRS> wt(w, w_dtype, g, C);
    float acc[G * G];
#pragma unroll
    for (int e = 0; e < G * G; ++e) acc[e] = 0.0f;
    chunk_walk<KEYS> at(rows, P, Q, causal, causal == 1, slots, bi * (NT / 64) + wave, parts * (NT / 64));
    for (; at.find(); at.advance()) {
        const int64_t base = ((int64_t)at.n * C + (int64_t)g * G) * plane + (int64_t)at.p * Q;
        const int key = at.q0 + lane * V, last = at.last;
        u4 out[G];
        if (at.q0 > last) {
#pragma unroll
            for (int i = 0; i < G; ++i) out[i] = u4{0u, 0u, 0u, 0u};
        } else {
            // a lane beyond the attended keys re-reads the row's start: zeros to either gradient
            const unsigned from = key <= last ? (unsigned)key * sizeof(T) : 0;
            u4 dv[G], xv[G];
#pragma unroll
            for (int h = 0; h < G; ++h) dv[h] = load_vec<STREAM>(dy + base + h * plane, from);
#pragma unroll
            for (int h = 0; h < G; ++h) xv[h] = load_vec<STREAM>(x + base + h * plane, from);
            if (at.q0 + KEYS - 1 > last) {
#pragma unroll
                for (int h = 0; h < G; ++h) {
                    zero_beyond<T>(dv[h], key, last);
                    zero_beyond<T>(xv[h], key, last);
                }
            }
            lane_tile<T, G, PAIRS>(dv, xv, wt, acc, out);
            if (at.q0 + KEYS - 1 > last) {   // (a weight that is not finite makes NaN of those zeros)
#pragma unroll
                for (int i = 0; i < G; ++i) zero_beyond<T>(out[i], key, last);
            }
        }
        if (key < Q && (causal != 2 || key <= last)) {
#pragma unroll
            for (int i = 0; i < G; ++i) store_out(vec_at(dx + base + i * plane, (unsigned)key * sizeof(T)), out[i], STREAM);
        }
    }
    lane_deposit<G>(acc, red, wave, lane);
    __syncthreads();
    for (int e = threadIdx.x; e < G * G; e += NT) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 4 * NT / 64; ++k) s += red[k][e];
        partial[(int64_t)blockIdx.x * (G * G) + e] = s;
    }
}

// The rows of one (batch entry, group) that workgroup `bi` of `parts` takes, longest first; back and forth, so that all of them
// get about as many keys.  -1 at the end.
__device__ __forceinline__ int row_of(int k, int bi, int parts, int P)
{
    const int j = k * parts + ((k & 1) ? parts - 1 - bi : bi);
    return P - 1 - j;
}

// Behind the softmax gradient: a workgroup per row of a group, a wavefront per KEYS keys.  A wavefront beyond the attended keys
// of a row is beyond those of the rows that follow (they are shorter): it leaves its sums in LDS and ends - a barrier waits
// for the wavefronts that are left.
template <typename T, int G, bool PAIRS>
__global__ __launch_bounds__(512) void lane_softmax_grads(const T *__restrict__ s, const T *__restrict__ ds, const T *__restrict__ x,
                                                          const void *__restrict__ w, T *__restrict__ dx, float *__restrict__ partial, int N, int C,
                                                          int P, int Q, int causal, int parts, int w_dtype, int stream)
{
    constexpr int V = vec_of<T>::n, KEYS = 64 * V, MAXW = 8;
    __shared__ __align__(16) float dots[2][G][4 * MAXW];
    __shared__ float red[4 * MAXW][G * G];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int nw = blockDim.x >> 6;
    const int bi = (int)(blockIdx.x % (unsigned)parts), n = (int)(blockIdx.x / (unsigned)parts) % N, g = (int)(blockIdx.x / (unsigned)parts) / N;
    const int64_t plane = (int64_t)P * Q;
    const lane_weights<T, G, PAIRS> wt(w, w_dtype, g, C);
    float acc[G * G];
#pragma unroll
    for (int e = 0; e < G * G; ++e) acc[e] = 0.0f;
    const int key = wave * KEYS + lane * V;
    int live = 0;
    for (int k = 0;; ++k) {
        const int p = row_of(k, bi, parts, P);
        if (p < 0) break;
        const int last = last_key(p, Q, causal);
        if (wave * KEYS > last) {
            lane_deposit<G>(acc, red, wave, lane);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            return;
        }
        live = last / KEYS + 1;
        const int64_t base = ((int64_t)n * C + (int64_t)g * G) * plane + (int64_t)p * Q;
        const unsigned from = key <= last ? (unsigned)key * sizeof(T) : 0;
        u4 sv[G], dv[G], xv[G];
#pragma unroll
        for (int h = 0; h < G; ++h) {
            sv[h] = load_vec<false>(s + base + h * plane, from);
            dv[h] = load_vec<false>(ds + base + h * plane, from);
        }
#pragma unroll
        for (int h = 0; h < G; ++h) xv[h] = load_vec<false>(x + base + h * plane, from);
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const float d = row_sum(dot_vec<T>(sv[h], dv[h], key, last, 0.0f));
            if ((lane & 15) == (h & 15)) dots[k & 1][h][4 * wave + (lane >> 4)] = d;
        }
        __syncthreads();
        u4 out[G];
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float d = 0.0f;
            for (int v = 0; v < live; ++v) {
                const f32x4 four = *reinterpret_cast<const f32x4 *>(&dots[k & 1][h][4 * v]);
                d += (four[0] + four[1]) + (four[2] + four[3]);
            }
            dv[h] = softmax_grad<T>(sv[h], dv[h], d);
        }
        if (wave * KEYS + KEYS - 1 > last) {   // (0 * NaN beyond the row's end, where a sum is NaN)
#pragma unroll
            for (int h = 0; h < G; ++h) {
                zero_beyond<T>(dv[h], key, last);
                zero_beyond<T>(xv[h], key, last);
            }
        }
        lane_tile<T, G, PAIRS>(dv, xv, wt, acc, out);
        if (key <= last) {
#pragma unroll
            for (int i = 0; i < G; ++i) {
                if (key + V - 1 > last) zero_beyond<T>(out[i], key, last);
                store_out(vec_at(dx + base + i * plane, (unsigned)key * sizeof(T)), out[i], stream);
            }
        }
    }
    lane_deposit<G>(acc, red, wave, lane);
    __syncthreads();
    for (int e = threadIdx.x; e < G * G; e += 64 * live) {
        float sum = 0.0f;
        for (int k = 0; k < 4 * nw; ++k) sum += red[k][e];
        partial[(int64_t)blockIdx.x * (G * G) + e] = sum;
    }
}

// ---- groups of 8, 12, 16 or 32 heads: matrix cores ---------------------------------------------------------------------------
template <typename T, int HG> struct dense {
    static constexpr int V = vec_of<T>::n;
    static constexpr bool F32 = V == 4;
    static constexpr int KEYS = 16 * V;                          // of a tile
    static constexpr int OB = (HG + 15) / 16;                    // blocks of 16 heads
    static constexpr int HPL = !F32 && HG == 12 ? 4 : HG / 4;    // heads per lane
    static constexpr int SETS = HG == 8 ? 2 : 1;                 // sets of heads at different keys in the 16 operand rows of dw
    static constexpr int STEPS = 4 / SETS;                       // of dw per tile, 4 * SETS vectors of a head each
    static constexpr int OPL = HG == 8 ? 2 : 4;                  // output heads per lane of a block
    static constexpr int LD = 288;                               // bytes of a row in LDS (256 of them data)
    static constexpr int BYTES = 16 * OB * LD;                   // a wavefront's tile in LDS
    static_assert(HG == 8 || HG == 12 || HG == 16 || HG == 32, "instances");

    int ln, kg;
    int64_t plane;
    unsigned heads_at, rows_at, out_at;   // byte offsets of a lane's first head: load, load_rows, mix
    u2 w16;             // 16-bit, up to 16 heads: w[head(t)][out(ln)], t < 4
    frag8<T> w32[OB];   // 16-bit, 32 heads: w[8kg .. 8kg+7][16ob + ln]
    float wf[OB][HPL];  // fp32: w[4t + kg][16ob + out(ln)]
    f32x4 acc[OB][OB];  // dw: acc[a][b][v] = entry (16a + 4kg + v, 16b + ln)

    // (16 bit: the heads of a lane follow each other, as the products take them; fp32: product t takes heads 4t .. 4t+3)
    __device__ __forceinline__ int head(int t) const { return F32 ? 4 * t + kg : HPL * kg + t; }
    // operand row ln of the mix: output head 4kg + v of a block is what lane group kg gets in its value v (8 heads: 2kg + v of
    // two values, so that all lanes store), and of dw: a head (8 heads: of one set of keys or the other)
    __device__ __forceinline__ int out() const { return OPL == 4 ? ln : (ln & 3) < 2 ? 2 * (ln >> 2) + (ln & 3) : HG; }
    __device__ __forceinline__ int row() const { return SETS == 2 ? ln & 7 : ln < HG ? ln : HG - 1; }
    __device__ __forceinline__ int vec(int s) const { return (SETS == 2 ? 8 * s + 4 * (ln >> 3) : 4 * s) + kg; }   // of step s
    __device__ __forceinline__ bool owns() const { return F32 || HPL * kg < HG; }   // (16 bit, 12 heads: the last lane group has none)

    __device__ __forceinline__ dense(int lane, const void *w, int w_dtype, int g, int C, int64_t plane_) : ln(lane & 15), kg(lane >> 4), plane(plane_)
    {
        const unsigned bytes = (unsigned)(plane * sizeof(T));
        heads_at = owns() ? head(0) * bytes : 0;
        rows_at = row() * bytes;
        out_at = OPL * kg * bytes;
#pragma unroll
        for (int a = 0; a < OB; ++a)
#pragma unroll
            for (int b = 0; b < OB; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (F32) {
#pragma unroll
            for (int ob = 0; ob < OB; ++ob)
#pragma unroll
                for (int t = 0; t < HPL; ++t)
                    wf[ob][t] = 16 * ob + out() < HG ? load_any(w, w_dtype, (int64_t)(g * HG + head(t)) * C + g * HG + 16 * ob + out()) : 0.0f;
        } else if constexpr (HG == 32) {
#pragma unroll
            for (int ob = 0; ob < OB; ++ob)
#pragma unroll
                for (int t = 0; t < 8; ++t) w32[ob].v[t] = ((const T *)w)[(int64_t)(g * HG + head(t)) * C + g * HG + 16 * ob + ln];
        } else {
            struct alignas(8) quad { T v[4]; } col;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                col.v[t] = t < HPL && owns() && out() < HG ? ((const T *)w)[(int64_t)(g * HG + head(t)) * C + g * HG + out()] : from_float<T>(0.0f);
            w16 = __builtin_bit_cast(u2, col);
        }
    }

    // v[t]: vector ln of head(t), base: head 0 of the group, first key of the row (a lane beyond `last` re-reads the row's start)
    template <bool STREAM> __device__ __forceinline__ void load(u4 (&v)[HPL], const T *base, int key, int last) const
    {
        const unsigned from = heads_at + (key <= last ? key * sizeof(T) : 0);
#pragma unroll
        for (int t = 0; t < HPL; ++t) v[t] = load_vec<STREAM>(base + (F32 ? 4 * t : t) * plane, from);
    }

    // x[s]: vector vec(s) of head 16b + row()
    __device__ __forceinline__ void load_rows(u4 (&x)[STEPS], int b, const T *base, int q0, int last) const
    {
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int key = q0 + vec(s) * V;
            x[s] = load_vec<false>(base + 16 * b * plane, rows_at + (key <= last ? key * sizeof(T) : 0));
        }
    }

    // dx = w^T v for the tile's keys (v: zeros beyond `last`), stored up to `last`, or up to Q with zeros behind
    __device__ __forceinline__ void mix(const u4 (&v)[HPL], T *base, int key, int last, int Q, bool whole, bool stream) const
    {
#pragma unroll
        for (int ob = 0; ob < OB; ++ob) {
            f32x4 d[V];   // d[j][e]: head 16ob + OPL*kg + e, key V*ln + j
#pragma unroll
            for (int j = 0; j < V; ++j) {
                d[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (F32) {
#pragma unroll
                    for (int t = 0; t < HPL; ++t) d[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[ob][t], __uint_as_float(v[t][j]), d[j], 0, 0, 0);
                } else {
                    const unsigned sel = (j & 1) ? 0x07060302u : 0x05040100u;
                    if constexpr (HG == 32) {
                        u4 col;
#pragma unroll
                        for (int u = 0; u < 4; ++u) col[u] = __builtin_amdgcn_perm(v[2 * u + 1][j >> 1], v[2 * u][j >> 1], sel);
                        mma16(d[j], w32[ob], __builtin_bit_cast(frag8<T>, col));
                    } else {
                        u2 col = {__builtin_amdgcn_perm(v[1][j >> 1], v[0][j >> 1], sel), 0u};
                        if constexpr (HPL == 4) col[1] = __builtin_amdgcn_perm(v[HPL - 1][j >> 1], v[HPL - 2][j >> 1], sel);
                        if constexpr (__is_same(T, bf16_t))
                            d[j] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, w16), __builtin_bit_cast(s4, col), d[j], 0, 0, 0);
                        else
                            d[j] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(h4, w16), __builtin_bit_cast(h4, col), d[j], 0, 0, 0);
                    }
                }
            }
            if (key >= Q || (!whole && key > last) || 16 * ob + OPL * kg >= HG) continue;
#pragma unroll
            for (int e = 0; e < OPL; ++e) {
                u4 o;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if constexpr (F32) o[u] = __float_as_uint(d[u][e]);
                    else o[u] = pack2<T>(d[2 * u][e], d[2 * u + 1][e]);
                }
                if (key + V - 1 > last) zero_beyond<T>(o, key, last);
                store_out(vec_at(base + (16 * ob + e) * plane, out_at + (unsigned)key * sizeof(T)), o, stream);
            }
        }
    }

    // v into `tile` (this wavefront's), rows of heads.  The LDS operations of a wavefront are done in order; the fences keep the
    // compiler to it.
    __device__ __forceinline__ void to_lds(const u4 (&v)[HPL], char *tile) const
    {
        in_order();
        if (owns()) {
            char *at = tile + head(0) * LD + ln * 16;
#pragma unroll
            for (int t = 0; t < HPL; ++t) *reinterpret_cast<u4 *>(at + (F32 ? 4 * t : t) * LD) = v[t];
        }
        in_order();
    }
    static __device__ __forceinline__ void in_order()
    {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }

    // columns 16b .. 16b+15 of acc += v x^T (both zeros beyond the attended keys)
    __device__ __forceinline__ void weight(const u4 (&x)[STEPS], int b, const char *tile)
    {
        const char *at = tile + row() * LD + vec(0) * 16;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int a = 0; a < OB; ++a) {
                const u4 d = *reinterpret_cast<const u4 *>(at + 16 * a * LD + 64 * SETS * s);
                if constexpr (F32) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(d[e]), __uint_as_float(x[s][e]), acc[a][b], 0, 0, 0);
                } else {
                    mma16(acc[a][b], __builtin_bit_cast(frag8<T>, d), __builtin_bit_cast(frag8<T>, x[s]));
                }
            }
    }

    // both gradients of a tile whose v (dy) is in registers, zeros beyond `last`; LOADED: `first` holds the first block of x
    template <bool LOADED>
    __device__ __forceinline__ void grads(const u4 (&v)[HPL], const u4 (&first)[STEPS], const T *x, T *dx, int q0, int key, int last, int Q, bool whole,
                                          bool stream, char *tile)
    {
        to_lds(v, tile);
        mix(v, dx, key, last, Q, whole, stream);
#pragma unroll
        for (int b = 0; b < OB; ++b) {
            u4 xv[STEPS];
            if (LOADED && b == 0) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) xv[s] = first[s];
            } else {
                load_rows(xv, b, x, q0, last);
            }
            if (q0 + KEYS - 1 > last) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) zero_beyond<T>(xv[s], q0 + vec(s) * V, last);
            }
            weight(xv, b, tile);
        }
    }

    // the sums as a (16 OB) x (16 OB) matrix in the tile
    __device__ __forceinline__ void deposit(char *tile) const
    {
        float *m = reinterpret_cast<float *>(tile);
#pragma unroll
        for (int a = 0; a < OB; ++a)
#pragma unroll
            for (int b = 0; b < OB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) m[(16 * a + 4 * kg + v) * (16 * OB) + 16 * b + ln] = acc[a][b][v];
    }
    // ... and entry e = (o, i) of it (8 heads: the blocks in which a set of keys meets itself)
    static __device__ __forceinline__ float entry(const char *tile, int e)
    {
        const float *m = reinterpret_cast<const float *>(tile) + (e / HG) * (16 * OB) + e % HG;
        return SETS == 2 ? m[0] + m[8 * 16 + 8] : m[0];
    }
};

template <typename T, int HG, bool STREAM>
__global__ __launch_bounds__(NT) void dense_grads(const T *__restrict__ x, const T *__restrict__ dy, const void *__restrict__ w, T *__restrict__ dx,
                                                  float *__restrict__ partial, unsigned rows, int C, int P, int Q, int causal, unsigned slots,
                                                  unsigned parts, int w_dtype)
{
    using D = dense<T, HG>;
    __shared__ __align__(16) char tiles[NT / 64][D::BYTES];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int g = (int)(blockIdx.x / parts);
    const unsigned bi = blockIdx.x % parts;
    const int64_t plane = (int64_t)P * Q;
    D d(lane, w, w_dtype, g, C, plane);
    chunk_walk<D::KEYS> at(rows, P, Q, causal, causal == 1, slots, bi * (NT / 64) + wave, parts * (NT / 64));
    for (; at.find(); at.advance()) {
        const int64_t base = ((int64_t)at.n * C + (int64_t)g * HG) * plane + (int64_t)at.p * Q;
        const int key = at.q0 + d.ln * D::V, last = at.last;
        if (at.q0 > last) {   // beyond the diagonal: zeros
            if (key < Q && d.owns()) {
#pragma unroll
                for (int t = 0; t < D::HPL; ++t)
                    store_out(vec_at(dx + base + (D::F32 ? 4 * t : t) * plane, d.heads_at + (unsigned)key * sizeof(T)), u4{0u, 0u, 0u, 0u}, STREAM);
            }
            continue;
        }
        u4 v[D::HPL], xv[D::STEPS];
        d.template load<STREAM>(v, dy + base, key, last);
        d.load_rows(xv, 0, x + base, at.q0, last);
        if (at.q0 + D::KEYS - 1 > last) {
#pragma unroll
            for (int t = 0; t < D::HPL; ++t) zero_beyond<T>(v[t], key, last);
        }
        if (!d.owns()) {   // (0 times an infinity would reach every head)
#pragma unroll
            for (int t = 0; t < D::HPL; ++t) v[t] = u4{0u, 0u, 0u, 0u};
        }
        d.template grads<true>(v, xv, x + base, dx + base, at.q0, key, last, Q, causal != 2, STREAM, tiles[wave]);
    }
    d.deposit(tiles[wave]);
    __syncthreads();
    for (int e = threadIdx.x; e < HG * HG; e += NT) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < NT / 64; ++k) s += D::entry(tiles[k], e);
        partial[(int64_t)blockIdx.x * (HG * HG) + e] = s;
    }
}

// Behind the softmax gradient; rows and wavefronts as in lane_softmax_grads, TPW tiles per wavefront.
template <typename T, int HG, int TPW>
__global__ __launch_bounds__(512, TPW == 1 ? 4 : 2) void dense_softmax_grads(const T *__restrict__ s, const T *__restrict__ ds, const T *__restrict__ x,
                                                            const void *__restrict__ w, T *__restrict__ dx, float *__restrict__ partial, int N, int C,
                                                            int P, int Q, int causal, int parts, int w_dtype, int stream)
{
    using D = dense<T, HG>;
    constexpr int MAXW = 8;
    extern __shared__ __align__(16) char lds[];   // a tile per wavefront, then dots[2][HG][MAXW]
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int nw = blockDim.x >> 6;
    char *tile = lds + wave * D::BYTES;
    float *dots = reinterpret_cast<float *>(lds + nw * D::BYTES);
    const int bi = (int)(blockIdx.x % (unsigned)parts), n = (int)(blockIdx.x / (unsigned)parts) % N, g = (int)(blockIdx.x / (unsigned)parts) / N;
    const int64_t plane = (int64_t)P * Q;
    D d(lane, w, w_dtype, g, C, plane);
    int live = 0;
    for (int k = 0;; ++k) {
        const int p = row_of(k, bi, parts, P);
        if (p < 0) break;
        const int last = last_key(p, Q, causal);
        if (wave * D::KEYS > last) {
            d.deposit(tile);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            return;
        }
        live = last / D::KEYS + 1 < nw ? last / D::KEYS + 1 : nw;
        asm volatile("" : "+v"(d.ln), "+v"(d.kg));   // (key numbers and their bounds anew for every row: kept, they spill)
        const int64_t base = ((int64_t)n * C + (int64_t)g * HG) * plane + (int64_t)p * Q;
        u4 sv[TPW][D::HPL], dv[TPW][D::HPL];
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const int q0 = (i * nw + wave) * D::KEYS, key = q0 + d.ln * D::V;
            if (i > 0 && q0 > last) continue;
            d.template load<false>(sv[i], s + base, key, last);
            d.template load<false>(dv[i], ds + base, key, last);
        }
        float dot[D::HPL];
#pragma unroll
        for (int t = 0; t < D::HPL; ++t) dot[t] = 0.0f;
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            const int q0 = (i * nw + wave) * D::KEYS, key = q0 + d.ln * D::V;
            if (i > 0 && q0 > last) continue;
#pragma unroll
            for (int t = 0; t < D::HPL; ++t) {
                dot[t] = dot_vec<T>(sv[i][t], dv[i][t], key, last, dot[t]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        float *row = dots + (k & 1) * (HG * MAXW);
#pragma unroll
        for (int t = 0; t < D::HPL; ++t) {
            dot[t] = row_sum(dot[t]);
            if (d.ln == 0 && d.owns()) row[d.head(t) * MAXW + wave] = dot[t];
        }
        __syncthreads();
        // (from here on the vectors as they were loaded: their values widened ahead of the barrier would be kept across it)
#pragma unroll
        for (int i = 0; i < TPW; ++i)
#pragma unroll
            for (int t = 0; t < D::HPL; ++t) asm volatile("" : "+v"(sv[i][t]), "+v"(dv[i][t]));
#pragma unroll
        for (int t = 0; t < D::HPL; ++t) {
            const float *of = row + (d.owns() ? d.head(t) : 0) * MAXW;
            dot[t] = 0.0f;
            for (int v = 0; v < live; ++v) dot[t] += of[v];
        }
#pragma unroll
        for (int i = 0; i < TPW; ++i) {
            asm volatile("" : "+v"(d.ln), "+v"(d.kg));
            const int q0 = (i * nw + wave) * D::KEYS, key = q0 + d.ln * D::V;
            if (i > 0 && q0 > last) continue;
            __builtin_amdgcn_sched_barrier(0);   // (a tile at a time: the next one's loads and values would not fit the registers)
            u4 xv[D::STEPS];
            if constexpr (HG != 32) d.load_rows(xv, 0, x + base, q0, last);   // (32 heads: behind the mix, for want of registers)
#pragma unroll
            for (int t = 0; t < D::HPL; ++t) {
                dv[i][t] = softmax_grad<T>(sv[i][t], dv[i][t], dot[t]);
                if (key + D::V - 1 > last) zero_beyond<T>(dv[i][t], key, last);   // (0 * NaN, where the sum is NaN)
                if (!d.owns()) dv[i][t] = u4{0u, 0u, 0u, 0u};
            }
            d.template grads<HG != 32>(dv[i], xv, x + base, dx + base, q0, key, last, Q, false, stream, tile);
        }
    }
    d.deposit(tile);
    __syncthreads();
    for (int e = threadIdx.x; e < HG * HG; e += 64 * live) {
        float sum = 0.0f;
        for (int k = 0; k < nw; ++k) sum += D::entry(lds + k * D::BYTES, e);
        partial[(int64_t)blockIdx.x * (HG * HG) + e] = sum;
    }
}

// ---- host ------------------------------------------------------------------------------------------------------------------
// What a call is cut into: workgroups per group of heads (= partial matrices per group).  0: no kernel.
struct cut {
    int64_t parts = 0;    // per group
    unsigned slots = 0;   // chunk_walk
    int waves = 0, tiles = 0;   // softmax kernels: wavefronts per row, tiles per wavefront
};

cut cut_of(int64_t N, int64_t C, int64_t P, int64_t Q, int group_size, int causal, int io_dtype, int w_dtype, bool softmax)
{
    cut c;
    const int64_t G = group_size > 0 ? group_size : C, V = io_dtype == MTA_F32 ? 4 : 8;
    const bool lanes = G == 2 || G == 4, mfma = G == 8 || G == 12 || G == 16 || G == 32;
    if (!(lanes || mfma) || C % G || C > 1024 || Q % V || N * P > 0x3fffffffLL) return c;
    if (mfma && io_dtype != MTA_F32 && w_dtype != io_dtype) return c;
    if (G * P * Q >= (int64_t(1) << 32) / (16 / V)) return c;   // (32-bit byte offsets within a group)
    const int64_t groups = C / G, keys = (lanes ? 64 : 16) * V;
    if (softmax) {
        const int64_t tiles = (Q + keys - 1) / keys;
        if (lanes) {
            if (tiles > 8) return c;
            c.waves = (int)tiles;
        } else {
            if (tiles > (G == 32 ? 16 : 32)) return c;
            c.tiles = tiles > 16 ? 4 : tiles > 8 ? 2 : 1;
            c.waves = (int)((tiles + c.tiles - 1) / c.tiles);
        }
        // Workgroups of several rows each, about as many as the chip holds: more cost partial matrices (fp32 B1 H32 S1024 1024 | 512:
        // 81 | 75 us), fewer leave it idle (bf16 B2 H8 S2048 512 | 256: 58 | 67).  Small groups and the longest rows want 1024
        // (bf16 B2 H4 S4096 137 | 145, B1 H16 S4096 292 | 312).
        const int64_t most = (lanes || c.tiles == 4 ? 1024 : 512) / (N * groups);
        c.parts = most < 1 ? 1 : most < P ? most : P;
        if (N * groups * c.parts > 0x7fffffffLL) c.parts = 0;
    } else {
        const int64_t full = 2 * ((Q + keys - 1) / keys), slots = causal == 2 && P / keys + 2 < full ? P / keys + 2 : full;
        const int64_t enough = ((N * P + 1) / 2 * slots + NT / 64 - 1) / (NT / 64), most = lanes ? 2048 : G == 32 ? 512 : 1024;   // (see above; 32 heads, fp32 B1 S1024: 512 | 1024 43 | 54 us)
        c.slots = (unsigned)slots;
        c.parts = most < enough ? most : enough;
    }
    return c;
}

int check_args(const void *a, const void *b, const void *c, const void *w, const void *dx, const void *dw, const void *ws, int64_t N, int64_t C,
               int64_t P, int64_t Q, int group_size, int io_dtype, int w_dtype)
{
    if (!a || !b || !c || !w || !dx || !dw || !ws) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype) || !dtype_size(w_dtype)) return MTA_ERR_DTYPE;
    if (N <= 0 || C <= 0 || P <= 0 || Q <= 0 || P > (1 << 24) || Q > (1 << 24)) return MTA_ERR_SHAPE;
    if (group_size < 0 || (group_size > 0 && C % group_size != 0)) return MTA_ERR_GROUP;
    if (!aligned_to(w, dtype_size(w_dtype)) || !aligned_to(dw, dtype_size(w_dtype)) || !aligned_to(ws, 16)) return MTA_ERR_ALIGN;
    return MTA_OK;
}

// `parts` matrices of G x G per group
mta_partials job_of(const void *ws, void *dw, int64_t C, int64_t G, int64_t parts, int w_dtype)
{
    return {ws, dw, (int32_t)C, (int32_t)(G * G), (int32_t)parts, (int32_t)G, 0, w_dtype, 1.0f};
}

template <typename T>
void launch_grads(const void *x, const void *dy, const void *w, void *dx, void *ws, const cut &c, int64_t N, int64_t C, int64_t P, int64_t Q, int G,
                  int causal, int w_dtype, bool same_dtype, hipStream_t st)
{
    auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(C / G * c.parts)), dim3(NT), 0, st, (const T *)x, (const T *)dy, w, (T *)dx, (float *)ws,
                           (unsigned)(N * P), (int)C, (int)P, (int)Q, causal, c.slots, (unsigned)c.parts, w_dtype);
    };
    constexpr bool P16 = sizeof(T) == 2;
    const bool big = streams(N, C, P, Q, sizeof(T)), pairs = P16 && same_dtype;
    switch (G) {
    case 2: return pairs ? big ? go(lane_grads<T, 2, P16, true>) : go(lane_grads<T, 2, P16, false>) : big ? go(lane_grads<T, 2, false, true>) : go(lane_grads<T, 2, false, false>);
    case 4: return pairs ? big ? go(lane_grads<T, 4, P16, true>) : go(lane_grads<T, 4, P16, false>) : big ? go(lane_grads<T, 4, false, true>) : go(lane_grads<T, 4, false, false>);
    case 8: return big ? go(dense_grads<T, 8, true>) : go(dense_grads<T, 8, false>);
    case 12: return big ? go(dense_grads<T, 12, true>) : go(dense_grads<T, 12, false>);
    case 16: return big ? go(dense_grads<T, 16, true>) : go(dense_grads<T, 16, false>);
    default: return big ? go(dense_grads<T, 32, true>) : go(dense_grads<T, 32, false>);
    }
}

template <typename T>
hipError_t launch_softmax_grads(const void *s, const void *ds, const void *x, const void *w, void *dx, void *ws, const cut &c, int64_t N, int64_t C,
                                int64_t P, int64_t Q, int G, int causal, int w_dtype, bool same_dtype, hipStream_t st)
{
    constexpr bool P16 = sizeof(T) == 2;
    const bool pairs = P16 && same_dtype;
    auto go = [&](auto kern, size_t lds) {
        if (lds > 48 * 1024) {   // per device, so set on every such launch (a cheap host-side call)
            const hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(kern, dim3((unsigned)(N * (C / G) * c.parts)), dim3(64 * c.waves), lds, st, (const T *)s, (const T *)ds, (const T *)x, w,
                           (T *)dx, (float *)ws, (int)N, (int)C, (int)P, (int)Q, causal, (int)c.parts, w_dtype, (int)streams(N, C, P, Q, sizeof(T)));
        return hipSuccess;
    };
    auto lds = [&](int bytes) { return (size_t)c.waves * bytes + 2 * G * 8 * sizeof(float); };
#define MTA_TILES(g) c.tiles == 1 ? dense_softmax_grads<T, g, 1> : c.tiles == 2 ? dense_softmax_grads<T, g, 2>
    switch (G) {
    case 2: return go(pairs ? lane_softmax_grads<T, 2, P16> : lane_softmax_grads<T, 2, false>, 0);
    case 4: return go(pairs ? lane_softmax_grads<T, 4, P16> : lane_softmax_grads<T, 4, false>, 0);
    case 8: return go(MTA_TILES(8) : dense_softmax_grads<T, 8, 4>, lds(dense<T, 8>::BYTES));
    case 12: return go(MTA_TILES(12) : dense_softmax_grads<T, 12, 4>, lds(dense<T, 12>::BYTES));
    case 16: return go(MTA_TILES(16) : dense_softmax_grads<T, 16, 4>, lds(dense<T, 16>::BYTES));
    default: return go(c.tiles == 1 ? dense_softmax_grads<T, 32, 1> : dense_softmax_grads<T, 32, 2>, lds(dense<T, 32>::BYTES));
    }
#undef MTA_TILES
}
}  // namespace

extern "C" int64_t mta_headmix_grads_workspace(int64_t N, int64_t C, int64_t P, int64_t Q, int group_size, int causal, int with_softmax, int io_dtype,
                                               int w_dtype)
{
    if (N <= 0 || C <= 0 || P <= 0 || Q <= 0 || P > (1 << 24) || Q > (1 << 24) || !dtype_size(io_dtype) || !dtype_size(w_dtype) || group_size < 0 ||
        (group_size > 0 && C % group_size))
        return 0;
    const cut c = cut_of(N, C, P, Q, group_size, causal, io_dtype, w_dtype, with_softmax != 0);
    const int64_t G = group_size > 0 ? group_size : C;
    return (with_softmax ? N : 1) * (C / G) * c.parts * G * G * (int64_t)sizeof(float);
}

extern "C" int mta_headmix_grads_partials(const void *x, const void *dy, const void *w, void *dx, void *dw, void *workspace, int64_t workspace_bytes,
                                          int64_t N, int64_t C, int64_t P, int64_t Q, int group_size, int causal, int io_dtype, int w_dtype,
                                          mta_partials *job, void *stream)
{
    if (!job) return MTA_ERR_NULL;
    const int rc = check_args(x, dy, x, w, dx, dw, workspace, N, C, P, Q, group_size, io_dtype, w_dtype);
    if (rc != MTA_OK) return rc;
    causal = causal == MTA_CAUSAL_LOWER_ONLY ? 2 : causal ? 1 : 0;
    const cut c = cut_of(N, C, P, Q, group_size, causal, io_dtype, w_dtype, false);
    if (!c.parts || !aligned_to(x, 16) || !aligned_to(dy, 16) || !aligned_to(dx, 16)) return MTA_ERR_UNSUPPORTED;
    const int G = group_size > 0 ? group_size : (int)C;
    if (workspace_bytes < C / G * c.parts * G * G * (int64_t)sizeof(float)) return MTA_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    MTA_DISPATCH_IO(io_dtype, launch_grads<io_t>(x, dy, w, dx, workspace, c, N, C, P, Q, G, causal, w_dtype, w_dtype == io_dtype, st));
    *job = job_of(workspace, dw, C, G, c.parts, w_dtype);
    return launch_status();
}

extern "C" int mta_headmix_grads(const void *x, const void *dy, const void *w, void *dx, void *dw, void *workspace, int64_t workspace_bytes, int64_t N,
                                 int64_t C, int64_t P, int64_t Q, int group_size, int causal, int io_dtype, int w_dtype, void *stream)
{
    mta_partials job;
    const int rc = mta_headmix_grads_partials(x, dy, w, dx, dw, workspace, workspace_bytes, N, C, P, Q, group_size, causal, io_dtype, w_dtype, &job, stream);
    return rc != MTA_OK ? rc : mta_sum_partials(1, &job, stream);
}

extern "C" int mta_softmax_headmix_grads_partials(const void *s, const void *ds, const void *x, const void *w, void *dx, void *dw, void *workspace,
                                                  int64_t workspace_bytes, int64_t N, int64_t C, int64_t P, int64_t Q, int group_size, int causal,
                                                  int io_dtype, int w_dtype, mta_partials *job, void *stream)
{
    if (!job) return MTA_ERR_NULL;
    const int rc = check_args(s, ds, x, w, dx, dw, workspace, N, C, P, Q, group_size, io_dtype, w_dtype);
    if (rc != MTA_OK) return rc;
    causal = causal ? 1 : 0;
    const cut c = cut_of(N, C, P, Q, group_size, causal, io_dtype, w_dtype, true);
    if (!c.parts || !aligned_to(s, 16) || !aligned_to(ds, 16) || !aligned_to(x, 16) || !aligned_to(dx, 16)) return MTA_ERR_UNSUPPORTED;
    const int G = group_size > 0 ? group_size : (int)C;
    const int64_t blocks = N * (C / G) * c.parts;
    if (workspace_bytes < blocks * G * G * (int64_t)sizeof(float)) return MTA_ERR_WORKSPACE;
    hipStream_t st = (hipStream_t)stream;
    hipError_t attr = hipSuccess;
    MTA_DISPATCH_IO(io_dtype, attr = launch_softmax_grads<io_t>(s, ds, x, w, dx, workspace, c, N, C, P, Q, G, causal, w_dtype, w_dtype == io_dtype, st));
    if (attr != hipSuccess) return (int)attr;
    *job = job_of(workspace, dw, C, G, N * c.parts, w_dtype);
    return launch_status();
}

extern "C" int mta_softmax_headmix_grads(const void *s, const void *ds, const void *x, const void *w, void *dx, void *dw, void *workspace,
                                         int64_t workspace_bytes, int64_t N, int64_t C, int64_t P, int64_t Q, int group_size, int causal, int io_dtype,
                                         int w_dtype, void *stream)
{
    mta_partials job;
    const int rc = mta_softmax_headmix_grads_partials(s, ds, x, w, dx, dw, workspace, workspace_bytes, N, C, P, Q, group_size, causal, io_dtype, w_dtype, &job,
                                                      stream);
    return rc != MTA_OK ? rc : mta_sum_partials(1, &job, stream);
}
