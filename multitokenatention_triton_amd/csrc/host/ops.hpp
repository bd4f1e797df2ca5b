// Tensor-level operators over the C ABI for the native routes: torch supplies device memory and the stream, the checks are
// the ones the kernels rely on, every computation is a call into libmta_hip.so.
#pragma once

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cmath>
#include <optional>

#include "../../../include/mta_hip.h"

namespace mta_host {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

inline int code(const Tensor &t, const char *what)
{
    switch (t.scalar_type()) {
    case at::kFloat: return MTA_F32;
    case at::kBFloat16: return MTA_BF16;
    case at::kHalf: return MTA_F16;
    default: C10_THROW_ERROR(TypeError, c10::str(what, ": dtype ", t.scalar_type(), " is not supported (float32, bfloat16, float16)"));
    }
}

inline bool is16(const Tensor &t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }

inline Tensor on_gpu(const Tensor &t, const char *what)
{
    TORCH_CHECK(t.is_cuda(), what, " lives on ", t.device(), ": the MTA kernels only run on an AMD GPU (there is no CPU path)");
    return t.is_contiguous() ? t : t.contiguous();
}

// ... at an address of whole 16-byte vectors: a view into a larger buffer is copied where a library product took it as it was
inline Tensor on_gpu_vectors(const Tensor &t, const char *what)
{
    const Tensor x = on_gpu(t, what);
    return reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16 ? x.clone() : x;
}

inline void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// 0 = ok; negative = argument rejected (ValueError); positive = HIP error (RuntimeError)
inline void check(int rc, const char *what)
{
    if (rc == 0) return;
    TORCH_CHECK_VALUE(rc > 0, what, ": ", mta_strerror(rc), " (code ", rc, ")");
    TORCH_CHECK(false, what, ": ", mta_strerror(rc), " (code ", rc, ")");
}

// the kernels index a weight by the data's heads: (C,R,S) conv kernels, (C,C) head weights
inline void check_conv_weight(const Tensor &w, int64_t heads)
{
    TORCH_CHECK(w.dim() == 3 && w.size(0) == heads, "a conv weight of ", heads, " heads must be (", heads, ",R,S), got ", w.sizes());
}
inline void check_head_weight(const Tensor &w, int64_t heads)
{
    TORCH_CHECK(w.dim() == 2 && w.size(0) == heads && w.size(1) == heads, "Weight must be (", heads, ",", heads, "), got ", w.sizes());
}

inline const void *ptr(const Tensor &t) { return t.const_data_ptr(); }
inline const void *ptr(const OptTensor &t) { return t ? t->const_data_ptr() : nullptr; }
inline void *out_ptr(const Tensor &t) { return t.mutable_data_ptr(); }

// the `causal` argument of the conv / head-mixing entry points
inline int causal_mode(bool causal, bool fill_upper) { return !causal ? 0 : fill_upper ? 1 : MTA_CAUSAL_LOWER_ONLY; }

inline int64_t tri_row_offset(int64_t p)
{
    const int64_t a = p >> 6;
    return 2048 * a * (a + 1) + (p & 63) * 64 * (a + 1);
}

inline Tensor conv2d(const Tensor &x_, const Tensor &w_, bool causal, std::optional<double> in_scale, bool fill_upper)
{
    const Tensor x = on_gpu(x_, "input"), w = on_gpu(w_, "weight");
    TORCH_CHECK_VALUE(x.dim() == 4 && w.dim() == 3, "expected input (N,C,H,W) and weight (C,R,S), got ", x.sizes(), " and ", w.sizes());
    TORCH_CHECK(x.size(1) == w.size(0), "This implementation assumes depthwise convolution (C_in == C_out)");
    Tensor y = at::empty(x.sizes(), x.options());
    const int64_t n = x.size(0), c = x.size(1), h = x.size(2), wd = x.size(3);
    const int r = (int)w.size(1), s = (int)w.size(2), ic = code(x, "input"), wc = code(w, "weight");
    int rc;
    if (in_scale)
        rc = mta_conv2d_scaled_fwd(ptr(x), ptr(w), out_ptr(y), n, c, h, wd, r, s, causal_mode(causal, fill_upper), (float)*in_scale, ic, wc, stream_of(x));
    else
        rc = mta_conv2d_fwd(ptr(x), ptr(w), out_ptr(y), n, c, h, wd, r, s, causal_mode(causal, fill_upper), ic, wc, stream_of(x));
    check(rc, "mta_conv2d_fwd");
    return y;
}

inline Tensor conv2d_bwd_input(const Tensor &dy_, const Tensor &w_, bool causal, bool fill_upper)
{
    const Tensor dy = on_gpu(dy_, "grad_output"), w = on_gpu(w_, "weight");
    check_conv_weight(w, dy.size(1));
    Tensor dx = at::empty(dy.sizes(), dy.options());
    check(mta_conv2d_bwd_input(ptr(dy), ptr(w), out_ptr(dx), dy.size(0), dy.size(1), dy.size(2), dy.size(3), (int)w.size(1), (int)w.size(2),
                               causal_mode(causal, fill_upper), code(dy, "grad_output"), code(w, "weight"), stream_of(dy)),
          "mta_conv2d_bwd_input");
    return dx;
}

// Weight gradients whose partial results one launch adds up (run(); until then the gradients hold nothing).  Keeps the workspaces
// that far; all on the stream of the first one.
struct Sums {
    // the entry of a gradient about to be computed into dw by way of ws
    mta_partials *add(const Tensor &dw, const Tensor &ws)
    {
        if (count == MTA_MAX_SUMS) run();
        kept[count] = {dw, ws};
        if (count == 0) stream = stream_of(ws);
        return &jobs[count++];
    }
    void drop() { kept[--count] = {}; }   // ... and was not, after all
    void run()
    {
        check(mta_sum_partials(count, jobs, stream), "mta_sum_partials");
        while (count) drop();
    }

  private:
    mta_partials jobs[MTA_MAX_SUMS];
    std::pair<Tensor, Tensor> kept[MTA_MAX_SUMS];
    int count = 0;
    void *stream = nullptr;
};

// the gradient of a (C,R,S) kernel, times `scale`, in the dtype of `like` (in `sums`)
inline Tensor conv2d_bwd_weight(const Tensor &x_, const Tensor &dy_, const Tensor &like, bool causal, double scale, Sums &sums)
{
    const Tensor x = on_gpu(x_, "input"), dy = on_gpu(dy_, "grad_output");
    TORCH_CHECK_VALUE(x.sizes() == dy.sizes() && x.scalar_type() == dy.scalar_type(), "input and grad_output must share shape and dtype");
    const int64_t n = x.size(0), c = x.size(1), h = x.size(2), w = x.size(3);
    const int r = (int)like.size(1), s = (int)like.size(2);
    Tensor dw = at::empty({c, r, s}, like.options());
    const int64_t bytes = std::max<int64_t>(mta_conv2d_bwd_weight_workspace(n, c, h, w, r, s), 16);
    Tensor ws = at::empty({bytes}, x.options().dtype(at::kByte));
    check(mta_conv2d_bwd_weight_partials(ptr(x), ptr(dy), out_ptr(dw), out_ptr(ws), bytes, n, c, h, w, r, s, causal, (float)scale, code(x, "input"),
                                         code(like, "weight"), sums.add(dw, ws), stream_of(x)),
          "mta_conv2d_bwd_weight");
    return dw;
}

// Both gradients of the conv in one pass over dy, the kernel's times `scale` (in `sums`); over_x: the input's gradient takes the place of x.
// Nothing where there is no kernel.
inline std::optional<std::pair<Tensor, Tensor>> conv2d_grads(const Tensor &x_, const Tensor &dy_, const Tensor &w_, bool causal, bool fill_upper,
                                                             double scale, Sums &sums, bool over_x = false)
{
    if (dy_.scalar_type() != x_.scalar_type() || dy_.sizes() != x_.sizes()) return std::nullopt;
    const Tensor x = on_gpu(x_, "input"), dy = on_gpu(dy_, "grad_output"), w = on_gpu(w_, "weight");
    check_conv_weight(w, dy.size(1));
    const int64_t n = x.size(0), c = x.size(1), h = x.size(2), wd = x.size(3);
    const int r = (int)w.size(1), s = (int)w.size(2);
    const int64_t bytes = std::max<int64_t>(mta_conv2d_bwd_weight_workspace(n, c, h, wd, r, s), 16);
    Tensor dx = over_x ? x : at::empty(dy.sizes(), dy.options());
    Tensor dw = at::empty(w.sizes(), w.options()), ws = at::empty({bytes}, x.options().dtype(at::kByte));
    const int rc = mta_conv2d_grads_partials(ptr(x), ptr(dy), ptr(w), out_ptr(dx), out_ptr(dw), out_ptr(ws), bytes, n, c, h, wd, r, s,
                                             causal_mode(causal, fill_upper), (float)scale, code(x, "input"), code(w, "weight"), sums.add(dw, ws), stream_of(x));
    if (rc == MTA_ERR_UNSUPPORTED) {
        sums.drop();
        return std::nullopt;
    }
    check(rc, "mta_conv2d_grads");
    return std::make_pair(dx, dw);
}

inline Tensor headmix(const Tensor &x_, const Tensor &w_, bool causal, double fill, int64_t group, bool fill_upper)
{
    const Tensor x = on_gpu(x_, "input"), w = on_gpu(w_, "weight");
    TORCH_CHECK_VALUE(x.dim() == 4, "expected input (N,C,P,Q), got ", x.sizes());
    TORCH_CHECK(w.dim() == 2 && w.size(0) == w.size(1), "Weight must be square matrix, got ", w.sizes());
    TORCH_CHECK(x.size(1) == w.size(0), "Channel dimension ", x.size(1), " must match weight dimension ", w.size(0));
    Tensor y = at::empty(x.sizes(), x.options());
    check(mta_headmix_fwd(ptr(x), ptr(w), out_ptr(y), x.size(0), x.size(1), x.size(2), x.size(3), (int)group, causal_mode(causal, fill_upper),
                          (float)fill, code(x, "input"), code(w, "weight"), stream_of(x)),
          "mta_headmix_fwd");
    return y;
}

inline Tensor headmix_bwd_input(const Tensor &dy_, const Tensor &w_, bool causal, int64_t group, bool fill_upper)
{
    const Tensor dy = on_gpu(dy_, "grad_output"), w = on_gpu(w_, "weight");
    check_head_weight(w, dy.size(1));
    Tensor dx = at::empty(dy.sizes(), dy.options());
    check(mta_headmix_bwd_input(ptr(dy), ptr(w), out_ptr(dx), dy.size(0), dy.size(1), dy.size(2), dy.size(3), (int)group,
                                causal_mode(causal, fill_upper), code(dy, "grad_output"), code(w, "weight"), stream_of(dy)),
          "mta_headmix_bwd_input");
    return dx;
}

// the gradient of a (C,C) head weight in the dtype of `like`; group > 0: confined to the diagonal blocks
inline Tensor headmix_bwd_weight(const Tensor &x_, const Tensor &dy_, const Tensor &like, bool causal, int64_t group)
{
    const Tensor x = on_gpu(x_, "input"), dy = on_gpu(dy_, "grad_output");
    TORCH_CHECK_VALUE(x.sizes() == dy.sizes() && x.scalar_type() == dy.scalar_type(), "input and grad_output must share shape and dtype");
    const int64_t n = x.size(0), c = x.size(1), p = x.size(2), q = x.size(3);
    const int64_t bytes = mta_headmix_bwd_weight_workspace(n, c, p, q);
    TORCH_CHECK_VALUE(bytes > 0, "mta_headmix_bwd_weight: no kernel for ", c, " heads (at most 128)");
    Tensor dw = at::empty({c, c}, like.options()), ws = at::empty({std::max<int64_t>(bytes, 16)}, x.options().dtype(at::kByte));
    check(mta_headmix_bwd_weight_as(ptr(x), ptr(dy), out_ptr(dw), out_ptr(ws), bytes, n, c, p, q, (int)group, causal, code(x, "input"),
                                    code(like, "weight"), stream_of(x)),
          "mta_headmix_bwd_weight");
    return dw;
}

// The gradients of the head mixing with respect to its input and its weight in one pass; with `probs`, dy is the gradient of the
// softmax behind it (of the probabilities `probs`).  Nothing where there is no kernel.  (dw: in `sums`)
inline std::optional<std::pair<Tensor, Tensor>> headmix_grads(const OptTensor &probs_, const Tensor &dy_, const Tensor &x_, const Tensor &w_, bool causal,
                                                              int64_t group, bool fill_upper, Sums &sums)
{
    if (dy_.dim() != 4 || dy_.scalar_type() != x_.scalar_type() || dy_.sizes() != x_.sizes()) return std::nullopt;
    const Tensor x = on_gpu(x_, "input"), dy = on_gpu(dy_, "grad_output"), w = on_gpu(w_, "weight");
    const OptTensor probs = probs_ ? OptTensor(on_gpu(*probs_, "probabilities")) : probs_;
    TORCH_CHECK(!probs || (probs->sizes() == x.sizes() && probs->scalar_type() == x.scalar_type()), "probabilities and input must share shape and dtype");
    check_head_weight(w, x.size(1));
    const int64_t n = x.size(0), c = x.size(1), p = x.size(2), q = x.size(3);
    const int ic = code(x, "input"), wc = code(w, "weight"), mode = causal_mode(causal, fill_upper);
    const int64_t bytes = mta_headmix_grads_workspace(n, c, p, q, (int)group, mode, probs.has_value(), ic, wc);
    if (bytes <= 0) return std::nullopt;
    Tensor dx = at::empty(x.sizes(), x.options()), dw = at::empty(w.sizes(), w.options()), ws = at::empty({bytes}, x.options().dtype(at::kByte));
    mta_partials *job = sums.add(dw, ws);
    const int rc = probs ? mta_softmax_headmix_grads_partials(ptr(probs), ptr(dy), ptr(x), ptr(w), out_ptr(dx), out_ptr(dw), out_ptr(ws), bytes, n, c, p, q,
                                                              (int)group, causal, ic, wc, job, stream_of(x))
                         : mta_headmix_grads_partials(ptr(x), ptr(dy), ptr(w), out_ptr(dx), out_ptr(dw), out_ptr(ws), bytes, n, c, p, q, (int)group, mode,
                                                      ic, wc, job, stream_of(x));
    if (rc == MTA_ERR_UNSUPPORTED) {
        sums.drop();
        return std::nullopt;
    }
    check(rc, "mta_headmix_grads");
    return std::make_pair(dx, dw);
}

inline Tensor headmix_softmax(const Tensor &x_, const OptTensor &w1, const OptTensor &w2, bool causal, int64_t group, bool fill_upper,
                              const OptTensor &key_bias, const OptTensor &first)
{
    const Tensor x = on_gpu(x_, "input");
    TORCH_CHECK_VALUE(x.dim() == 4, "expected input (N,C,P,Q), got ", x.sizes());
    OptTensor a, b;
    if (w1) a = on_gpu(*w1, "weight");
    if (w2) b = on_gpu(*w2, "weight");
    for (const OptTensor *w : {&a, &b})
        if (*w) check_head_weight(**w, x.size(1));
    TORCH_CHECK(!key_bias || (key_bias->numel() == x.size(0) * x.size(3) && key_bias->device() == x.device()), "key_bias must be (", x.size(0), ",", x.size(3), ")");
    TORCH_CHECK(!first || (first->numel() == x.size(0) * x.size(2) && first->device() == x.device()), "first must be (", x.size(0), ",", x.size(2), ")");
    TORCH_CHECK_TYPE(!a || !b || a->scalar_type() == b->scalar_type(), "w1 and w2 must share a dtype");
    const int wc = a ? code(*a, "weight") : b ? code(*b, "weight") : MTA_F32;
    Tensor y = at::empty(x.sizes(), x.options());
    check(mta_headmix_softmax_band_fwd(ptr(x), ptr(a), ptr(b), ptr(key_bias), ptr(first), out_ptr(y), x.size(0), x.size(1), x.size(2), x.size(3),
                                       (int)group, causal, fill_upper, code(x, "input"), wc, stream_of(x)),
          "mta_headmix_softmax_band_fwd");
    return y;
}

inline Tensor softmax_bwd(const Tensor &p_, const Tensor &dp_, bool causal, bool fill_upper)
{
    const Tensor p = on_gpu(p_, "probabilities"), dp = on_gpu(dp_, "grad_output");
    TORCH_CHECK_VALUE(p.dim() == 4 && p.sizes() == dp.sizes() && p.scalar_type() == dp.scalar_type(),
                      "probabilities and grad_output must be (N,C,P,Q) tensors of one shape and dtype");
    Tensor dx = at::empty(p.sizes(), p.options());
    check(mta_softmax_bwd(ptr(p), ptr(dp), out_ptr(dx), p.size(0), p.size(1), p.size(2), p.size(3), causal, fill_upper, code(p, "probabilities"),
                          stream_of(p)),
          "mta_softmax_bwd");
    return dx;
}

// nothing (nullopt) when the library has no kernel for the combination
inline OptTensor conv2d_headmix(const Tensor &x_, const Tensor &wc_, const Tensor &wm_, bool causal, int64_t group, bool fill_upper)
{
    const Tensor x = on_gpu(x_, "input"), wc = on_gpu(wc_, "conv weight"), wm = on_gpu(wm_, "mix weight");
    check_conv_weight(wc, x.size(1));
    check_head_weight(wm, x.size(1));
    Tensor y = at::empty(x.sizes(), x.options());
    const int rc = mta_conv2d_headmix_fwd(ptr(x), ptr(wc), ptr(wm), out_ptr(y), x.size(0), x.size(1), x.size(2), x.size(3), (int)wc.size(1),
                                          (int)wc.size(2), (int)group, causal, fill_upper, code(x, "input"), code(wc, "weight"),
                                          code(wm, "weight"), stream_of(x));
    if (rc == MTA_ERR_UNSUPPORTED) return std::nullopt;
    check(rc, "mta_conv2d_headmix_fwd");
    return y;
}

// (here and below: `s_pad` > 0 is the length of the scores where Q, K and V are rows of a shorter one, at most 7 fewer, that are read where they lie)
inline bool qk_conv_supported(const Tensor &q, const Tensor &k, const Tensor &w, int64_t s_pad = 0)
{
    if (q.dim() != 4 || q.sizes() != k.sizes() || q.scalar_type() != k.scalar_type() || w.dim() != 3 || !is16(q) ||
        w.scalar_type() != q.scalar_type())
        return false;
    return mta_qk_conv_supported(s_pad ? s_pad : q.size(2), q.size(3), (int)w.size(1), (int)w.size(2), code(q, "Q"), code(w, "W")) != 0;
}

inline bool causal_pv_supported(at::ScalarType t, int64_t s, int64_t d)
{
    return (t == at::kBFloat16 || t == at::kHalf) && (d == 64 || d == 128) && s % 8 == 0;
}

// scale * conv(mask0(Q K^T)) as a (B,H,S,S) tensor; the caller has asked qk_conv_supported
inline Tensor qk_conv(const Tensor &q_, const Tensor &k_, const Tensor &w_, bool causal, double scale, bool fill_upper, const OptTensor &first, int64_t s_pad = 0)
{
    const Tensor q = on_gpu(q_, "Q"), k = on_gpu(k_, "K"), w = on_gpu(w_, "W");
    const int64_t b = q.size(0), h = q.size(1), s = s_pad ? s_pad : q.size(2), d = q.size(3);
    check_conv_weight(w, h);
    Tensor y = at::empty({b, h, s, s}, q.options());
    const int r = (int)w.size(1), sk = (int)w.size(2), ic = code(q, "Q"), wc = code(w, "W");
    const int rc = s_pad ? mta_qk_conv_ragged_fwd(ptr(q), ptr(k), ptr(w), ptr(first), out_ptr(y), nullptr, b, h, s, q.size(2), d, r, sk, (float)scale, 0, ic, wc, stream_of(q))
                 : first ? mta_qk_conv_band_fwd(ptr(q), ptr(k), ptr(w), ptr(first), out_ptr(y), b, h, s, d, r, sk, (float)scale, fill_upper, ic, wc, stream_of(q))
                 : mta_qk_conv_fwd(ptr(q), ptr(k), ptr(w), out_ptr(y), b, h, s, d, r, sk, causal, (float)scale, fill_upper, ic, wc, stream_of(q));
    check(rc, "mta_qk_conv_fwd");
    return y;
}

// whether P V and P^T X run as kernels that read (and P's producer need only write) the lower triangle: 16-bit data, which
// the kernels also take without the causal rule, or fp32 under it.  x: the (B,H,S,D) operand.
inline bool lower_products_supported(at::ScalarType t, c10::IntArrayRef x, bool causal)
{
    if (x.size() != 4) return false;
    return causal_pv_supported(t, x[2], x[3]) ||
           (t == at::kFloat && causal && (x[3] == 64 || x[3] == 128) && x[2] % 4 == 0 && x[2] <= (1 << 20));
}

// whether P (B,H,S,S) and X (B,H,S,D) are what the P V and P^T X kernels take: they index P by X's batch, heads and rows, where
// the library product broadcasts
inline bool score_planes_of(c10::IntArrayRef p, c10::IntArrayRef x)
{
    return p.size() == 4 && x.size() == 4 && p[0] == x[0] && p[1] == x[1] && p[2] == x[2] && p[3] == x[2];
}

inline OptTensor causal_pv(const Tensor &p_, const Tensor &v_, bool causal, const OptTensor &first, double scale, int64_t s_pad = 0)
{
    if (s_pad) {   // (16-bit and causal: the caller has checked)
        const Tensor p = on_gpu(p_, "P"), v = on_gpu(v_, "V");
        const int64_t b = v.size(0), h = v.size(1), d = v.size(3);
        TORCH_CHECK(causal && scale == 1.0 && p.scalar_type() == v.scalar_type() && p.sizes() == c10::IntArrayRef({b, h, s_pad, s_pad}));
        Tensor o = at::empty({b, h, s_pad, d}, v.options());
        check(mta_causal_pv_ragged_fwd(ptr(p), ptr(v), ptr(first), out_ptr(o), b, h, s_pad, v.size(2), d, 0, code(p, "P"), stream_of(p)), "mta_causal_pv_fwd");
        return o;
    }
    if (p_.scalar_type() != v_.scalar_type() || !score_planes_of(p_.sizes(), v_.sizes()) ||
        !lower_products_supported(p_.scalar_type(), v_.sizes(), causal))
        return std::nullopt;
    const Tensor p = on_gpu(p_, "P"), v = is16(v_) ? on_gpu(v_, "V") : on_gpu_vectors(v_, "V");
    Tensor o = at::empty(v.sizes(), v.options());
    const int64_t b = v.size(0), h = v.size(1), s = v.size(2), d = v.size(3);
    if (!is16(p)) {   // (the hidden stretch of P holds zeros)
        check(mta_causal_pv_f32(ptr(p), ptr(v), out_ptr(o), b, h, s, d, (float)scale, stream_of(p)), "mta_causal_pv_f32");
    } else if (first) {
        TORCH_CHECK(scale == 1.0);
        check(mta_causal_pv_band_fwd(ptr(p), ptr(v), ptr(first), out_ptr(o), b, h, s, d, causal, code(p, "P"), stream_of(p)), "mta_causal_pv_fwd");
    } else {
        check(mta_causal_pv_scaled_fwd(ptr(p), ptr(v), out_ptr(o), b, h, s, d, causal, (float)scale, code(p, "P"), stream_of(p)), "mta_causal_pv_fwd");
    }
    return o;
}

// whether the rows of a (B,H,S,D) tensor that is not contiguous can be read where they lie (16-bit data, whole 16-byte vectors)
inline bool rows_in_place(const Tensor &x)
{
    return x.dim() == 4 && x.is_cuda() && is16(x) && !x.is_contiguous() && x.stride(3) == 1 && x.stride(2) > 0 && x.stride(2) <= (1 << 20) &&
           x.stride(2) % 8 == 0 && x.stride(1) >= 0 && x.stride(1) % 8 == 0 && x.stride(0) >= 0 && x.stride(0) % 8 == 0 &&
           reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16 == 0;
}

inline OptTensor causal_ptx(const Tensor &p_, const Tensor &x_, bool causal, double scale)
{
    if (p_.scalar_type() != x_.scalar_type() || !score_planes_of(p_.sizes(), x_.sizes()) ||
        !lower_products_supported(p_.scalar_type(), x_.sizes(), causal))
        return std::nullopt;
    const bool in_place = rows_in_place(x_);
    const Tensor p = on_gpu(p_, "P"), x = in_place ? x_ : is16(x_) ? on_gpu(x_, "X") : on_gpu_vectors(x_, "X");
    Tensor o = at::empty(x.sizes(), x.options());
    const int64_t b = x.size(0), h = x.size(1), s = x.size(2), d = x.size(3);
    if (in_place)
        check(mta_causal_ptx_rows_fwd(ptr(p), ptr(x), x.stride(0), x.stride(1), x.stride(2), out_ptr(o), b, h, s, d, causal, (float)scale, code(p, "P"),
                                      stream_of(p)),
              "mta_causal_ptx_fwd");
    else if (is16(p))
        check(mta_causal_ptx_scaled_fwd(ptr(p), ptr(x), out_ptr(o), b, h, s, d, causal, (float)scale, code(p, "P"), stream_of(p)), "mta_causal_ptx_fwd");
    else
        check(mta_causal_ptx_f32(ptr(p), ptr(x), out_ptr(o), b, h, s, d, (float)scale, stream_of(p)), "mta_causal_ptx_f32");
    return o;
}

// P v and P^T x, both times `scale`, of 16-bit tensors and a causal P
inline std::optional<std::pair<Tensor, Tensor>> causal_products(const Tensor &p_, const Tensor &v_, const Tensor &x_, double scale)
{
    if (!is16(p_) || p_.scalar_type() != v_.scalar_type() || p_.scalar_type() != x_.scalar_type() || v_.sizes() != x_.sizes() ||
        !score_planes_of(p_.sizes(), v_.sizes()) || !lower_products_supported(p_.scalar_type(), v_.sizes(), true))
        return std::nullopt;
    const Tensor p = on_gpu(p_, "P"), v = on_gpu(v_, "V"), x = on_gpu(x_, "X");
    Tensor o = at::empty(v.sizes(), v.options()), ot = at::empty(x.sizes(), x.options());
    check(mta_causal_products(ptr(p), ptr(v), ptr(x), out_ptr(o), out_ptr(ot), v.size(0), v.size(1), v.size(2), v.size(3), true, (float)scale,
                              code(p, "P"), stream_of(p)),
          "mta_causal_products");
    return std::make_pair(o, ot);
}

inline void band_zero_(const Tensor &x, const Tensor &first)
{
    TORCH_CHECK(x.dim() == 4 && x.is_contiguous() && first.dim() == 2 && first.size(0) == x.size(0) && first.size(1) == x.size(2) &&
                    first.scalar_type() == at::kInt && first.is_contiguous() && first.device() == x.device(),
                "a band of ", first.sizes(), " does not belong to scores of ", x.sizes());
    if (is16(x))
        check(mta_band_zero_fwd(out_ptr(x), ptr(first), x.size(0), x.size(1), x.size(2), code(x, "input"), stream_of(x)), "mta_band_zero_fwd");
    else
        check(mta_band_zero_f32(out_ptr(x), ptr(first), x.size(0), x.size(1), x.size(2), stream_of(x)), "mta_band_zero_f32");
}

// whether the triangular-layout kernels exist (host-side questions to the library)
inline bool tri_route_supported(const Tensor &q, const Tensor &k, const Tensor &conv_w, int64_t group, const OptTensor &w1, const OptTensor &w2,
                                bool band, bool out_planes, bool key_bias, int64_t s_pad = 0)
{
    if (!qk_conv_supported(q, k, conv_w, s_pad) || (!w1 && !w2)) return false;
    for (const OptTensor *w : {&w1, &w2})
        if (*w && ((*w)->scalar_type() != q.scalar_type() || reinterpret_cast<uintptr_t>(ptr(*w)) % 4)) return false;
    const int64_t h = q.size(1), s = s_pad ? s_pad : q.size(2);
    if (h % group || group * tri_row_offset(s) >= (int64_t(1) << 31) || !causal_pv_supported(q.scalar_type(), s, q.size(3))) return false;
    const int c = code(q, "Q");
    return mta_headmix_softmax_tri_supported(h, s, (int)group, out_planes, c, c, w1.has_value(), w2.has_value(), band, key_bias) != 0;
}

inline Tensor qk_conv_tri(const Tensor &q_, const Tensor &k_, const Tensor &w_, double scale, int64_t group, const OptTensor &first, int64_t s_pad = 0)
{
    const Tensor q = on_gpu(q_, "Q"), k = on_gpu(k_, "K"), w = on_gpu(w_, "W");
    const int64_t b = q.size(0), h = q.size(1), s = s_pad ? s_pad : q.size(2), d = q.size(3);
    check_conv_weight(w, h);
    Tensor y = at::empty({b * h * tri_row_offset(s)}, q.options());
    check(s_pad ? mta_qk_conv_ragged_fwd(ptr(q), ptr(k), ptr(w), ptr(first), out_ptr(y), nullptr, b, h, s, q.size(2), d, (int)w.size(1), (int)w.size(2),
                                         (float)scale, (int)group, code(q, "Q"), code(w, "W"), stream_of(q))
                : mta_qk_conv_tri_fwd(ptr(q), ptr(k), ptr(w), ptr(first), out_ptr(y), b, h, s, d, (int)w.size(1), (int)w.size(2), (float)scale, (int)group,
                                      code(q, "Q"), code(w, "W"), stream_of(q)),
          "mta_qk_conv_tri_fwd");
    return y;
}

inline Tensor headmix_softmax_tri(const Tensor &x, const OptTensor &w1, const OptTensor &w2, int64_t n, int64_t c, int64_t s, int64_t group,
                                  const OptTensor &first, bool out_planes, const OptTensor &key_bias)
{
    OptTensor a, b;
    if (w1) a = on_gpu(*w1, "weight");
    if (w2) b = on_gpu(*w2, "weight");
    for (const OptTensor *w : {&a, &b})
        if (*w) check_head_weight(**w, c);
    TORCH_CHECK_VALUE(x.dim() == 1 && x.numel() == n * c * tri_row_offset(s), "expected a flat tensor of ", n * c * tri_row_offset(s), " elements");
    Tensor y = out_planes ? at::empty({n, c, s, s}, x.options()) : at::empty(x.sizes(), x.options());
    const int ic = code(x, "input");
    check(mta_headmix_softmax_tri_fwd(ptr(x), ptr(a), ptr(b), ptr(key_bias), ptr(first), out_ptr(y), n, c, s, (int)group, out_planes, ic, ic,
                                      stream_of(x)),
          "mta_headmix_softmax_tri_fwd");
    return y;
}

inline Tensor causal_pv_tri(const Tensor &p, const Tensor &v_, int64_t group, const OptTensor &first, int64_t s_pad = 0)
{
    const Tensor v = on_gpu(v_, "V");
    const int64_t s = s_pad ? s_pad : v.size(2);
    TORCH_CHECK_VALUE(v.dim() == 4 && p.numel() == v.size(0) * v.size(1) * tri_row_offset(s) && p.scalar_type() == v.scalar_type(),
                      "P in the triangular layout does not belong to a V of shape ", v.sizes());
    Tensor o = at::empty({v.size(0), v.size(1), s, v.size(3)}, v.options());
    check(s_pad ? mta_causal_pv_ragged_fwd(ptr(p), ptr(v), ptr(first), out_ptr(o), v.size(0), v.size(1), s, v.size(2), v.size(3), (int)group, code(p, "P"),
                                           stream_of(p))
                : mta_causal_pv_tri_fwd(ptr(p), ptr(v), ptr(first), out_ptr(o), v.size(0), v.size(1), s, v.size(3), (int)group, code(p, "P"), stream_of(p)),
          "mta_causal_pv_tri_fwd");
    return o;
}

// scores with the statistics of their rows, and what follows from the two: see mta_qk_conv_stats_fwd.  key_bias: 0 and -inf only
inline bool stats_route_supported(const Tensor &q, const Tensor &k, const Tensor &conv_w, int64_t group, const Tensor &w2, bool key_bias, int64_t s_pad = 0)
{
    if (!qk_conv_supported(q, k, conv_w, s_pad) || w2.scalar_type() != q.scalar_type() || reinterpret_cast<uintptr_t>(ptr(w2)) % 4) return false;
    const int c = code(q, "Q");
    return mta_softmax_mix_pv_supported(q.size(1), s_pad ? s_pad : q.size(2), q.size(3), (int)group, c, c, key_bias) != 0;
}

// (scores, statistics); tri: in the triangular layout
inline std::pair<Tensor, Tensor> qk_conv_stats(const Tensor &q_, const Tensor &k_, const Tensor &w_, double scale, int64_t group, bool tri,
                                               const OptTensor &key_bias, const OptTensor &first, int64_t s_pad = 0)
{
    const Tensor q = on_gpu_vectors(q_, "Q"), k = on_gpu_vectors(k_, "K"), w = on_gpu(w_, "W");
    const int64_t b = q.size(0), h = q.size(1), s = s_pad ? s_pad : q.size(2), d = q.size(3), r = w.size(1);
    check_conv_weight(w, h);
    Tensor y = tri ? at::empty({b * h * tri_row_offset(s)}, q.options()) : at::empty({b, h, s, s}, q.options());
    Tensor stats = at::empty({b * h, mta_qk_conv_stats_slots(b, h, s, (int)r), s, 2}, q.options().dtype(at::kFloat));
    TORCH_CHECK(!s_pad || !key_bias);
    check(s_pad ? mta_qk_conv_ragged_fwd(ptr(q), ptr(k), ptr(w), ptr(first), out_ptr(y), out_ptr(stats), b, h, s, q.size(2), d, (int)r, (int)w.size(2), (float)scale,
                                         tri ? (int)group : 0, code(q, "Q"), code(w, "W"), stream_of(q))
                : mta_qk_conv_stats_fwd(ptr(q), ptr(k), ptr(w), ptr(key_bias), ptr(first), out_ptr(y), out_ptr(stats), b, h, s, d, (int)r, (int)w.size(2), (float)scale,
                                tri ? (int)group : 0, code(q, "Q"), code(w, "W"), stream_of(q)),
          "mta_qk_conv_stats_fwd");
    return {y, stats};
}

inline Tensor softmax_mix_pv(const Tensor &x, const Tensor &stats, const Tensor &w2_, const Tensor &v_, int64_t r, int64_t group, bool tri,
                             const OptTensor &key_bias, const OptTensor &first, int64_t s_pad = 0)
{
    const Tensor v = on_gpu_vectors(v_, "V"), w2 = on_gpu(w2_, "weight");
    check_head_weight(w2, v.size(1));
    const int64_t s = s_pad ? s_pad : v.size(2);
    Tensor o = at::empty({v.size(0), v.size(1), s, v.size(3)}, v.options());
    check(mta_softmax_mix_pv_ragged_fwd(ptr(x), ptr(stats), ptr(w2), ptr(key_bias), ptr(first), ptr(v), out_ptr(o), v.size(0), v.size(1), s, v.size(2), v.size(3), (int)r,
                                 (int)group, tri, code(x, "scores"), code(w2, "weight"), stream_of(x)),
          "mta_softmax_mix_pv_fwd");
    return o;
}

// Rows of up to three (B,H,S,D) tensors, of any strides, into dense ones of S_out rows, one launch (mta_rows_copy).
class RowsCopy {
  public:
    RowsCopy(int64_t s_out, const OptTensor &key_bias) : s_out_(s_out), key_bias_(key_bias) {}

    // hide: the rows of hidden keys count as zeros
    Tensor add(const Tensor &x_, bool hide, double scale)
    {
        TORCH_CHECK(x_.is_cuda(), "input lives on ", x_.device(), ": the MTA kernels only run on an AMD GPU (there is no CPU path)");
        const Tensor x = x_.stride(3) == 1 ? x_ : x_.contiguous();
        TORCH_CHECK_VALUE(n_ == 0 || (x.size(0) == like_[0].size(0) && x.size(1) == like_[0].size(1) && x.size(2) == like_[0].size(2) &&
                                      x.scalar_type() == like_[0].scalar_type()),
                          "Q, K and V must share batch, heads, length and dtype");
        Tensor y = at::empty({x.size(0), x.size(1), s_out_, x.size(3)}, x.options());
        x_ptr_[n_] = ptr(x);
        y_ptr_[n_] = out_ptr(y);
        for (int i = 0; i < 3; ++i) strides_[3 * n_ + i] = x.stride(i);
        d_[n_] = x.size(3);
        scale_[n_] = (float)scale;
        hide_[n_] = hide && key_bias_;
        like_[n_++] = x;
        return y;
    }

    void run()
    {
        if (n_ == 0) return;
        const Tensor &x = like_[0];
        check(mta_rows_copy(n_, x_ptr_, strides_, y_ptr_, d_, scale_, hide_, ptr(key_bias_), key_bias_ ? key_bias_->size(1) : 0, x.size(0), x.size(1),
                            x.size(2), s_out_, code(x, "input"), stream_of(x)),
              "mta_rows_copy");
    }

  private:
    int64_t s_out_;
    OptTensor key_bias_;
    int n_ = 0;
    const void *x_ptr_[3];
    void *y_ptr_[3];
    int64_t strides_[9], d_[3];
    float scale_[3];
    int hide_[3];
    Tensor like_[3];
};

}  // namespace mta_host
