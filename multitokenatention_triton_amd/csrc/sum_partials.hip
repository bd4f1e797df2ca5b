// The second half of every weight gradient: the partial results that the workgroups of its first kernel left in a workspace, added
// in a fixed order, times a factor, rounded once to the weight's dtype.
//
// What bounds it is its own launch: a few KB to a few MB, and 4 us alone on the stream.  So a launch takes several gradients: the
// backward of a whole module adds up its four at the end (a training step of B1 H8 S256 D64 bf16, bound by the host: 21 launches
// -> 18, 174 -> 168 us; B1 H16 S2048 D128 fp16, where the pre-softmax pair shares one: 607 -> 605).  16 entries per workgroup, an
// entry's partial results dealt to 64 threads (each adds its share in index order, 16 in flight), the 64 sums added in thread order.
#include "common.hpp"

namespace {
using namespace mta;

constexpr int ENTRIES = 16, SHARES = 64;
struct jobs_arg {
    int first[MTA_MAX_SUMS + 1];   // workgroups of the jobs ahead
    mta_partials job[MTA_MAX_SUMS];
};

__global__ __launch_bounds__(ENTRIES * SHARES) void sum_partials(const jobs_arg jobs, int count)
{
    __shared__ float red[SHARES][ENTRIES + 1];
    int n = 0;
    while (n + 1 < count && (int)blockIdx.x >= jobs.first[n + 1]) ++n;
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
#pragma unroll 16
        for (int b = sl; b < j.parts; b += SHARES) s += from[(int64_t)b * entries];
    }
    red[sl][le] = s;
    __syncthreads();
    if (sl != 0 || e >= (j.side > 0 ? j.rows * j.rows : j.rows * entries)) return;
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < SHARES; ++k) t += red[k][le];
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
    jobs_arg a{};
    for (int i = 0; i < count; ++i) {
        const mta_partials &j = jobs[i];
        if (!j.partial || !j.dw) return MTA_ERR_NULL;
        if (!dtype_size(j.dtype)) return MTA_ERR_DTYPE;
        const int64_t total = j.side > 0 ? (int64_t)j.rows * j.rows : (int64_t)j.rows * j.entries;
        if (j.rows <= 0 || j.entries <= 0 || j.parts <= 0 || total > (1 << 26) || (j.side > 0 && (j.rows % j.side || j.entries != j.side * j.side))) return MTA_ERR_SHAPE;
        a.job[i] = j;
        a.first[i + 1] = a.first[i] + (int)((total + ENTRIES - 1) / ENTRIES);
    }
    hipLaunchKernelGGL(sum_partials, dim3((unsigned)a.first[count]), dim3(ENTRIES * SHARES), 0, (hipStream_t)stream, a, count);
    return launch_status();
}
