// x[n,c,p,q] = 0 for q < first_visible[n,p]: what the reference's `torch.where(mask == -inf, 0.0, scores)` behind its
// post-softmax conv (mta_attention_triton.py:82-83) does below the diagonal under a band mask (row p sees the keys
// first_visible[n,p] .. p).  The conv spreads probability into the columns a row does not see; this takes it out again
// before the heads are mixed.  Only the hidden stretch of each row is touched, and only written: whole 16-byte vectors
// are stored, the one vector that holds the first visible key is read, cleared in part and written back.
#include "common.hpp"

namespace {
using namespace mta;

typedef unsigned int bz_u4 __attribute__((ext_vector_type(4)));
constexpr int BZ_NT = 256;

// A workgroup takes BZ_ROWS consecutive rows of one plane, a wavefront every fourth of them; rows of S elements of E bytes, whole
// 16-byte vectors (V elements each).  The rows' first visible keys and their vectors in part are fetched together, a row per lane: one
// after the other, each behind its own load, the eight rows of a wavefront were a chain of eight memory latencies (us, bf16, window of
// S/4: 128 planes of 680^2 28.7 -> 17.1, 16 of 4096^2 51.5 -> 36.4).
constexpr int BZ_ROWS = 32, BZ_RPW = BZ_ROWS / (BZ_NT / 64);   // rows per wavefront
template <int E>
__global__ __launch_bounds__(BZ_NT) void band_zero_kernel(unsigned char *__restrict__ x, const int *__restrict__ first, int C,
                                                          int S, int blocks_per_plane)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned plane = blockIdx.x / (unsigned)blocks_per_plane;  // n*C + c
    const int p0 = (int)(blockIdx.x % (unsigned)blocks_per_plane) * BZ_ROWS;
    const int64_t n = plane / (unsigned)C;
    const bz_u4 z = {0u, 0u, 0u, 0u};
    constexpr int V = 16 / E;
    auto row_of = [&](int i) { return p0 + wave + i * (BZ_NT / 64); };
    auto vectors = [&](int p) { return reinterpret_cast<bz_u4 *>(x + ((int64_t)plane * S + p) * S * E); };
    int lo = 0;   // of this lane's row
    if (lane < BZ_RPW && row_of(lane) < S) {
        const int p = row_of(lane);
        lo = first[n * S + p];
        lo = lo < 0 ? 0 : (lo > p + 1 ? p + 1 : lo);  // (a row that sees nothing: everything up to the diagonal)
        const int rest = lo % V;
        if (rest) {
            bz_u4 *at = vectors(p) + lo / V, t = *at;
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (e < rest) t[e * E / 4] &= E == 4 ? 0u : (e & 1) ? 0x0000ffffu : 0xffff0000u;
            *at = t;
        }
    }
#pragma unroll
    for (int i = 0; i < BZ_RPW; ++i) {
        const int full = __builtin_amdgcn_readlane(lo, i) / V;  // whole vectors of hidden keys (0 beyond the last row)
        bz_u4 *row = vectors(row_of(i));
        for (int v = lane; v < full; v += 64) row[v] = z;
    }
}

int band_zero(void *x, const void *first_visible, int64_t N, int64_t C, int64_t S, int size, void *stream)
{
    if (!x || !first_visible) return MTA_ERR_NULL;
    if (N <= 0 || C <= 0 || S <= 0 || S > (1 << 24) || N * C * S > 0x7fffffffLL) return MTA_ERR_SHAPE;
    if (!aligned_to(x, 16) || !aligned_to(first_visible, 4)) return MTA_ERR_ALIGN;
    if (S * size % 16 != 0) return MTA_ERR_UNSUPPORTED;
    const int64_t bpp = (S + BZ_ROWS - 1) / BZ_ROWS;
    auto kern = size == 4 ? band_zero_kernel<4> : band_zero_kernel<2>;
    hipLaunchKernelGGL(kern, dim3((unsigned)(N * C * bpp)), dim3(BZ_NT), 0, (hipStream_t)stream, (unsigned char *)x, (const int *)first_visible,
                       (int)C, (int)S, (int)bpp);
    return launch_status();
}
}  // namespace

extern "C" int mta_band_zero_fwd(void *x, const void *first_visible, int64_t N, int64_t C, int64_t S, int io_dtype, void *stream)
{
    if (!x || !first_visible) return MTA_ERR_NULL;
    if (!dtype_size(io_dtype)) return MTA_ERR_DTYPE;
    if (io_dtype == MTA_F32) return MTA_ERR_UNSUPPORTED;
    return band_zero(x, first_visible, N, C, S, 2, stream);
}

extern "C" int mta_band_zero_f32(void *x, const void *first_visible, int64_t N, int64_t C, int64_t S, void *stream)
{
    return band_zero(x, first_visible, N, C, S, 4, stream);
}
