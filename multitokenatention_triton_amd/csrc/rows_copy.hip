// Rows of up to three (B,H,S,D) tensors copied into dense ones: padded with rows of zeros (or cut), the rows of hidden keys
// zeroed, multiplied by a factor - what the glue needs around the score kernels for lengths that are not whole 16-byte
// vectors of a score row, and for key masks.  Latency-bound: the tensors are D/S of a score tensor's size, so everything a
// call needs goes into one launch (torch's comparison, copy and masked fill were three for a key mask: 29 us of a 155 us
// forward at B4 H16 S1024 D128).
#include "common.hpp"

namespace {
using namespace mta;

constexpr int NT = 256, MOST = 3;

struct rows_job {
    const void *x[MOST];
    void *y[MOST];
    int64_t sb[MOST], sh[MOST], sr[MOST];  // strides of x in elements: batch entry, head, row
    unsigned vecs[MOST];                   // vectors (elements) of y
    int D[MOST];
    float scale[MOST];
    int hide[MOST];
};

// VEC elements per thread; blockIdx.y = tensor
template <typename T, int VEC>
__global__ __launch_bounds__(NT) void rows_copy_kernel(rows_job job, const float *__restrict__ key_bias, int bias_stride, int H, int S_in, int S_out)
{
    const int i = blockIdx.y;
    const unsigned e = blockIdx.x * NT + threadIdx.x;
    if (e >= job.vecs[i]) return;
    struct alignas(sizeof(T) * VEC) V { T v[VEC]; };
    const unsigned per_row = (unsigned)(job.D[i] / VEC);
    const unsigned row = e / per_row, bh = row / (unsigned)S_out, b = bh / (unsigned)H;
    const int c = (int)(e - row * per_row) * VEC, p = (int)(row - bh * S_out);
    V out;
#pragma unroll
    for (int u = 0; u < VEC; ++u) out.v[u] = from_float<T>(0.0f);
    if (p < S_in && !(job.hide[i] && key_bias[(int64_t)b * bias_stride + p] == -INFINITY)) {
        const T *src = (const T *)job.x[i] + b * job.sb[i] + (int64_t)(bh - b * H) * job.sh[i] + p * job.sr[i] + c;
        out = *reinterpret_cast<const V *>(src);
        if (job.scale[i] != 1.0f) {
#pragma unroll
            for (int u = 0; u < VEC; ++u) out.v[u] = from_float<T>(to_float(out.v[u]) * job.scale[i]);
        }
    }
    *reinterpret_cast<V *>((T *)job.y[i] + (int64_t)e * VEC) = out;
}
}  // namespace

extern "C" int mta_rows_copy(int count, const void *const *x, const int64_t *x_strides, void *const *y, const int64_t *D,
                             const float *scale, const int *hide, const void *key_bias, int64_t bias_stride, int64_t B, int64_t H, int64_t S_in,
                             int64_t S_out, int io_dtype, void *stream)
{
    if (!x || !x_strides || !y || !D || !scale || !hide) return MTA_ERR_NULL;
    const int size = dtype_size(io_dtype);
    if (!size) return MTA_ERR_DTYPE;
    if (count < 1 || count > MOST || B <= 0 || H <= 0 || S_in <= 0 || S_out <= 0 || S_in > (1 << 24) || S_out > (1 << 24)) return MTA_ERR_SHAPE;
    rows_job job = {};
    bool vec = true;
    const int V = 16 / size;
    for (int i = 0; i < count; ++i) {
        if (!x[i] || !y[i] || (hide[i] && !key_bias)) return MTA_ERR_NULL;
        if (D[i] <= 0 || D[i] > (1 << 24)) return MTA_ERR_SHAPE;
        if (!aligned_to(x[i], size) || !aligned_to(y[i], size)) return MTA_ERR_ALIGN;
        job.x[i] = x[i];
        job.y[i] = y[i];
        job.sb[i] = x_strides[3 * i];
        job.sh[i] = x_strides[3 * i + 1];
        job.sr[i] = x_strides[3 * i + 2];
        job.D[i] = (int)D[i];
        job.scale[i] = scale[i];
        job.hide[i] = hide[i];
        vec = vec && D[i] % V == 0 && job.sb[i] % V == 0 && job.sh[i] % V == 0 && job.sr[i] % V == 0 && aligned_to(x[i], 16) && aligned_to(y[i], 16);
    }
    int64_t most = 0;
    for (int i = 0; i < count; ++i) {
        const int64_t vecs = B * H * S_out * (D[i] / (vec ? V : 1));
        if (vecs > 0xffff0000LL) return MTA_ERR_SHAPE;
        job.vecs[i] = (unsigned)vecs;
        if (vecs > most) most = vecs;
    }
    const int64_t blocks = (most + NT - 1) / NT;
    const dim3 grid((unsigned)blocks, (unsigned)count);
    MTA_DISPATCH_IO(io_dtype, {
        auto kern = vec ? rows_copy_kernel<io_t, vec_of<io_t>::n> : rows_copy_kernel<io_t, 1>;
        hipLaunchKernelGGL(kern, grid, dim3(NT), 0, (hipStream_t)stream, job, (const float *)key_bias, (int)bias_stride, (int)H, (int)S_in, (int)S_out);
    });
    return launch_status();
}
