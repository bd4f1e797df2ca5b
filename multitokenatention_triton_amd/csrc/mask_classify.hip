// What a 4-D attention mask amounts to together with the causal rule, in one read of it: hidden keys (every row sees the kept keys up to
// itself), a band (row p sees the keys first[p] .. p), rows that see nothing, or neither.  The reference has no counterpart: it expands any
// mask to a (B,H,S,S) tensor (mta_attention_triton.py:106-127).
//
// A wavefront takes a row: 16 bytes per lane and step (elements one by one where the strides do not allow it, and at a row's end), compared with
// the row that sees most - the last one, without the causal rule the first -, counted, and the first visible key kept.  Causal boolean masks of
// one plane are read up to the diagonal only; others whole, because a value that is neither 0 nor -inf, or a head that differs, anywhere makes
// the mask another kind of mask.  A row adds its findings to one word: an atomic only where a bit is still missing, so that a band, whose rows
// all find "not hidden keys", does not queue up at it.
// Bound by its launch and by the one word read back: B4 S1024 boolean 4 MB.  It takes the place of a dozen elementwise and reduction
// kernels and three to five reads back: a call with a new mask, us, bf16 6x11 H16 D128 groups of 4:
// right-padded B4 S1024 188 -> 135 (103 with a mask seen before), B2 S256 108 -> 52 (26), window B2 S1024 217 -> 93 (53).
#include "common.hpp"

namespace {
using namespace mta;

enum { NOT_KEYS = 1, FIRST_HIDDEN = 2, NOT_BAND = 4, EMPTY_ROW = 8, OTHER_VALUE = 16, HEADS_DIFFER = 32 };   // (also in ops.py)

struct mask_args {
    const unsigned char *mask;
    int64_t sb, sh, sr, sc;   // strides in elements
    int H, S, S_out, causal, vectors, rows;   // vectors: whole 16-byte loads are aligned; rows: per wavefront
    unsigned minus_inf;       // its bits; 0: a boolean mask
    int *flags, *first;
    float *bias;
};

template <int E> struct element;
template <> struct element<1> { typedef uint8_t t; };
template <> struct element<2> { typedef uint16_t t; };
template <> struct element<4> { typedef uint32_t t; };

template <int E> __global__ __launch_bounds__(256) void mask_classify_kernel(mask_args a)
{
    typedef typename element<E>::t T;
    constexpr int V = 16 / E;
    constexpr unsigned SIGN = E == 4 ? 0x80000000u : E == 2 ? 0x8000u : 0u;   // boolean: every bit counts
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int S = a.S, ref = a.causal ? S - 1 : 0;
    const int64_t n = blockIdx.y;
    const bool boolean = E == 1, whole = !boolean || a.H > 1 || !a.causal;
    struct chunk { T e[V]; };
    auto load = [&](int h, int p, int q) {   // keys q .. q+V-1 of a row; 0 beyond it
        chunk c;
        const unsigned char *at = a.mask + (n * a.sb + h * a.sh + p * a.sr + q * a.sc) * E;
        if (a.vectors && q + V <= S) {
            __builtin_memcpy(&c, __builtin_assume_aligned(at, 16), 16);
        } else {
#pragma unroll
            for (int u = 0; u < V; ++u) c.e[u] = q + u < S ? *reinterpret_cast<const T *>(at + u * a.sc * E) : T(0);
        }
        return c;
    };
    // boolean: non-zero; additive: +-0
    auto visible = [&](T e) { return boolean ? e != 0 : (e & ~SIGN) == 0; };
    auto bits_of = [&](const chunk &c) {
        unsigned r = 0;
#pragma unroll
        for (int u = 0; u < V; ++u) r |= (visible(c.e[u]) ? 1u : 0u) << u;
        return r;
    };
    for (int i = 0; i < a.rows; ++i) {
        const int p = (blockIdx.x * 4 + wave) * a.rows + i;   // (wavefront-uniform)
        if (p >= S) return;
        const int end = a.causal ? p + 1 : S;                 // of the keys that count
        int count = 0, first = S;
        unsigned found = 0;
        for (int q = lane * V; q < (whole ? S : end); q += 64 * V) {
            const chunk c = load(0, p, q);
            const int in_row = S - q < V ? S - q : V, in = end - q < V ? (end - q < 0 ? 0 : end - q) : V;
            const unsigned counts = (1u << in) - 1u;
            const unsigned seen = bits_of(c) & counts;
            if ((seen ^ bits_of(load(0, ref, q))) & counts) found |= NOT_KEYS;
            count += __popc(seen);
            if (seen) first = min(first, q + __ffs((int)seen) - 1);
            if (!boolean) {
#pragma unroll
                for (int u = 0; u < V; ++u)
                    if (u < in_row && !visible(c.e[u]) && c.e[u] != (T)a.minus_inf) found |= OTHER_VALUE;
            }
            for (int h = 1; h < a.H; ++h) {
                const chunk o = load(h, p, q);   // (the same value: a NaN, which equals nothing, is an OTHER_VALUE)
#pragma unroll
                for (int u = 0; u < V; ++u)
                    if (u < in_row && !(boolean ? visible(c.e[u]) == visible(o.e[u]) : c.e[u] == o.e[u] || (visible(c.e[u]) && visible(o.e[u]))))
                        found |= HEADS_DIFFER;
            }
            if (p == ref) {
#pragma unroll
                for (int u = 0; u < V; ++u)
                    if (u < in_row) a.bias[n * a.S_out + q + u] = seen >> u & 1u ? 0.0f : -INFINITY;
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            count += __shfl_xor(count, off);
            first = min(first, __shfl_xor(first, off));
            found |= (unsigned)__shfl_xor((int)found, off);
        }
        if (p == ref && lane < a.S_out - S) {   // the padding: keys with no bias, rows that see themselves
            a.bias[n * a.S_out + S + lane] = 0.0f;
            a.first[n * a.S_out + S + lane] = S + lane;
        }
        if (lane != 0) continue;
        if (count == 0) found |= EMPTY_ROW;
        else if (count != p - first + 1) found |= NOT_BAND;
        if (p == ref && (a.causal ? first != 0 : count == 0)) found |= FIRST_HIDDEN;
        a.first[n * a.S_out + p] = count ? first : p + 1;
        if (found & ~(unsigned)__hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(a.flags, (int)found);
    }
}
}  // namespace

extern "C" int mta_mask_classify(const void *mask, int64_t stride_b, int64_t stride_h, int64_t stride_row, int64_t stride_key, int64_t N,
                                 int64_t H, int64_t S, int64_t S_out, int causal, int mask_dtype, void *flags, void *first, void *bias, void *stream)
{
    if (!mask || !flags || !first || !bias) return MTA_ERR_NULL;
    const int size = mask_dtype < 0 ? 1 : dtype_size(mask_dtype);
    if (!size) return MTA_ERR_DTYPE;
    if (N <= 0 || N > 65535 || H <= 0 || H > 4096 || S <= 0 || S > (1 << 24) || S_out < S || S_out > S + 64) return MTA_ERR_SHAPE;
    if (stride_b < 0 || stride_h < 0 || stride_row < 0 || stride_key < 0) return MTA_ERR_SHAPE;
    if (!aligned_to(mask, size) || !aligned_to(flags, 4) || !aligned_to(first, 4) || !aligned_to(bias, 4)) return MTA_ERR_ALIGN;
    mask_args a = {(const unsigned char *)mask, stride_b, stride_h, stride_row, stride_key, (int)H, (int)S, (int)S_out, causal != 0, 0, 1,
                   mask_dtype == MTA_F32 ? 0xff800000u : mask_dtype == MTA_BF16 ? 0xff80u : mask_dtype == MTA_F16 ? 0xfc00u : 0u,
                   (int *)flags, (int *)first, (float *)bias};
    a.vectors = stride_key == 1 && aligned_to(mask, 16) && (stride_b | stride_h | stride_row) * size % 16 == 0;
    a.rows = N * S > 16384 ? 4 : 1;   // (a workgroup per CU 16 times over)
    const dim3 grid((unsigned)((S + 4 * a.rows - 1) / (4 * a.rows)), (unsigned)N);
    hipStream_t st = (hipStream_t)stream;
    auto kern = size == 1 ? mask_classify_kernel<1> : size == 2 ? mask_classify_kernel<2> : mask_classify_kernel<4>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, a);
    return launch_status();
}
