// The second half of every weight gradient: the partial results that the workgroups of its first kernel left in a workspace, added
// in a fixed order, times a factor, rounded once to the weight's dtype.
//
// What bounds it is its own launch: a few KB to a few MB, and 4 us alone on the stream.  So a launch takes several gradients: the
// backward of a whole module adds up its four at the end (a training step of B1 H8 S256 D64 bf16, bound by the host: 21 launches
// -> 18, 174 -> 168 us; B1 H16 S2048 D128 fp16, where the pre-softmax pair shares one: 607 -> 605).  16 entries per workgroup, an
// entry's partial results dealt to 16 threads, or 64 where there are more than one round of loads of 16 threads takes (256): each adds
// its share in index order, 16 loads in flight whatever is left of it (a loop that unrolls by 16 walked a share of four as a chain of
// four latencies), then four threads of a wavefront, then the wavefronts in order.  With the gradient's first kernel, that loop and 64
// threads always | 16 threads | 64, us: B2 H16 S1001 head weight (256 partial results) 36.8 | 35.4 | 36.2, B1 H32 S1024 (512) 24.9 | 23.1 | 23.2,
// B1 H16 S1024 (1024) 18.0 | 17.7 | 17.8, B2 H32 S2048 groups of 4 (2048) 176 | 180 | 176; B2 H16 S1000 conv 3x3 (32) 26.4 | 26.6 | 27.5.
// One gradient has an argument block of its own (370 bytes less to fetch: 0.2 us).
#include "common.hpp"

namespace {
using namespace mta;

constexpr int ENTRIES = 16, BATCH = 16;
template <int N> struct jobs_arg {
    int first[N + 1];   // workgroups of the jobs ahead
    mta_partials job[N];
};

template <int N, int SHARES> __global__ __launch_bounds__(ENTRIES * SHARES) void sum_partials(const jobs_arg<N> jobs, int count)
{
    __shared__ float red[ENTRIES * SHARES / 64][ENTRIES];
    int n = 0;
    if constexpr (N > 1) {
        while (n + 1 < count && (int)blockIdx.x >= jobs.first[n + 1]) ++n;
    }
    const mta_partials &j = jobs.job[n];
    const int le = threadIdx.x % ENTRIES, sl = threadIdx.x / ENTRIES, e = ((int)blockIdx.x - jobs.first[n]) * ENTRIES + le;
    // entry e of the result: which block, which entry of it
    int block, at, entries = j.entries;
    bool in;
    if (j.side > 0) {   // blocks on the diagonal of a (rows, rows) matrix
        const int o = e / j.rows, i = e % j.rows;
        block = o / j.side;
        at = o % j.side * j.side + i % j.side;
        in = o < j.rows && block == i / j.side && (j.mask <= 0 || o / j.mask == i / j.mask);
    } else {
        block = e / entries;
        at = e % entries;
        in = block < j.rows;
    }
    float s = 0.0f;
    if (in) {
        const float *from = (const float *)j.partial + (int64_t)block * j.parts * entries + at;
        for (int b = sl; b < j.parts; b += BATCH * SHARES) {
            float v[BATCH];
#pragma unroll
            for (int u = 0; u < BATCH; ++u) v[u] = from[(int64_t)(b + u * SHARES < j.parts ? b + u * SHARES : b) * entries];
#pragma unroll
            for (int u = 0; u < BATCH; ++u) s += b + u * SHARES < j.parts ? v[u] : 0.0f;
        }
    }
    static_assert(ENTRIES == 16 && SHARES % 4 == 0, "four shares of an entry in a wavefront");
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    red[threadIdx.x >> 6][le] = s;
    __syncthreads();
    if (sl != 0 || e >= (j.side > 0 ? j.rows * j.rows : j.rows * entries)) return;
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < ENTRIES * SHARES / 64; ++k) t += red[k][le];
    t = in ? t * j.scale : 0.0f;
    if (j.dtype == MTA_F32) ((float *)j.dw)[e] = t;
    else if (j.dtype == MTA_BF16) ((bf16_t *)j.dw)[e] = from_float<bf16_t>(t);
    else ((f16_t *)j.dw)[e] = from_float<f16_t>(t);
}
}  // namespace

extern "C" int mta_sum_partials(int count, const mta_partials *jobs, void *stream)
{
    if (count < 0 || count > MTA_MAX_SUMS) return MTA_ERR_SHAPE;
    if (count == 0) return MTA_OK;
    if (!jobs) return MTA_ERR_NULL;
    jobs_arg<MTA_MAX_SUMS> a{};
    int most = 0;
    for (int i = 0; i < count; ++i) {
        const mta_partials &j = jobs[i];
        if (!j.partial || !j.dw) return MTA_ERR_NULL;
        if (!dtype_size(j.dtype)) return MTA_ERR_DTYPE;
        const int64_t total = j.side > 0 ? (int64_t)j.rows * j.rows : (int64_t)j.rows * j.entries;
        if (j.rows <= 0 || j.entries <= 0 || j.parts <= 0 || total > (1 << 26) || (j.side > 0 && (j.rows % j.side || j.entries != j.side * j.side))) return MTA_ERR_SHAPE;
        a.job[i] = j;
        a.first[i + 1] = a.first[i] + (int)((total + ENTRIES - 1) / ENTRIES);
        most = j.parts > most ? j.parts : most;
    }
    auto go = [&](auto kern, int shares, const auto &arg) {
        hipLaunchKernelGGL(kern, dim3((unsigned)a.first[count]), dim3(ENTRIES * shares), 0, (hipStream_t)stream, arg, count);
        return launch_status();
    };
    const jobs_arg<1> one{{0, a.first[1]}, {a.job[0]}};
    if (most <= 16 * BATCH) return count == 1 ? go(sum_partials<1, 16>, 16, one) : go(sum_partials<MTA_MAX_SUMS, 16>, 16, a);
    return count == 1 ? go(sum_partials<1, 64>, 64, one) : go(sum_partials<MTA_MAX_SUMS, 64>, 64, a);
}
