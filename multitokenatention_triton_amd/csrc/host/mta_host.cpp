// Native host path of the modules: one call per forward, one autograd node per module.
//
// At the lengths where a kernel takes a few microseconds the host is what bounds a call: an MTA forward of three kernels
// spent 84 us in Python (argument checks, a device context, a ctypes call and an allocation per stage) and a training step
// 530 us (seven autograd nodes with a Python frame each way).  The routes therefore live here, over the operators of
// ops.hpp; the Python modules keep parameters, masks and the rarely taken routes.
#include <torch/extension.h>

#include <ATen/ExpandUtils.h>
#include <ATen/autocast_mode.h>
#include <torch/csrc/autograd/anomaly_mode.h>

#include "ops.hpp"

namespace py = pybind11;

namespace mta_host {
namespace {

// largest mixing group the one-pass mix/softmax/mix kernel keeps in registers, and what its matrix-core variant takes
constexpr int64_t FUSED_MAX_GROUP = 8, FUSED_MFMA_GROUP = 16;

bool no_row_lists()
{
    const char *e = getenv("MTA_MIX16_NO_ROW_LISTS");
    return e && !strcmp(e, "1");
}

// whether mix -> softmax (-> mix) over mixing groups of `group` heads runs as one kernel
bool one_pass_group(int64_t group, at::ScalarType t, int64_t n_keys, const OptTensor &w1, const OptTensor &w2)
{
    if (group <= FUSED_MAX_GROUP) return true;
    if (w1 && w2 && w1->scalar_type() != w2->scalar_type()) return false;   // (one kernel takes its two weights in one dtype)
    if (t == at::kFloat) return n_keys % 4 == 0 && n_keys <= mta_headmix_softmax_dense_f32_keys((int)std::min<int64_t>(group, 1 << 20));
    return (t == at::kBFloat16 || t == at::kHalf) && n_keys % 8 == 0 && n_keys <= mta_headmix_softmax_dense16_keys((int)std::min<int64_t>(group, 1 << 20)) &&
           (!w1 || w1->scalar_type() == t) && (!w2 || w2->scalar_type() == t);
}

// the 16-bit matrix-core variant for groups of 16 takes a key bias or a band mask in its row-list form only
bool masks_ok(int64_t group, at::ScalarType t, bool masked)
{
    return !masked || group != FUSED_MFMA_GROUP || t == at::kFloat || !no_row_lists();
}

// Whether conv + mixing of 16 heads in one kernel is worth it: its 512 persistent workgroups walk 32 x 64 tiles of all 16
// heads at 16 to 18 us each, so that it takes more than one and a half rounds of tiles to meet the two kernels one after the other, or
// one round that is nearly full and surely fits (what is left to spare takes up an uneven deal over the XCDs).  Groups of 2 or 4 heads take that
// round; dense weights are left on the two kernels: they gain 3 to 6 % from 440 to 490 tiles, nothing at 420, and lose 2 to 4 % at 506.
// us of the forward (H16 D64, the pre-softmax conv 6x11), two kernels | one, fp16 dense 3x3 / 7x7 after the softmax / bf16 groups of 4, 3x3 / fp16 groups
// of 2, 3x3: 272 tiles (B1 S1024) 62.5 | 63.3 / 63.5 | 65.9 / 65.1 | 71.8 / 63.9 | 68.1, 380 (B1 S1216) 73.5 | 72.2 / 76.6 | 75.9 / 73.8 | 77.5 / 73.7 | 73.6,
// 420 (B1 S1280) 74.9 | 73.2 / 78.2 | 76.9 / 75.7 | 77.1 / 75.6 | 75.6, 440 (B4 S640) 79.2 | 75.2 / 83.0 | 79.2 / 81.6 | 78.1 / 83.8 | 76.3, 448 (B8 S448) 81.9 |
// 78.3 / 85.8 | 82.3 / 82.3 | 77.9 / 87.2 | 75.7, 480 (B2 S960) 79.1 | 74.8 / 83.5 | 78.8 / 81.7 | 78.9 / 82.3 | 76.9, 506 (B1 S1408) 83.8 | 85.7 / 87.8 | 91.7 /
// 81.6 | 88.2 / 81.8 | 86.2, 544 (B2 S1008) 80.3 | 81.3 / 84.4 | 87.2 / 85.6 | 85.0 / 86.0 | 83.3, 600 (B1 S1536) 90.5 | 95.3 / 94.8 | 101 / 89.8 | 98.4 / 90.5 |
// 96.8, 702 (B1 S1664) 96.4 | 95.7 / 101 | 101 / 95.9 | 97.8 / 95.5 | 95.9, 756 (B1 S1728) 106 | 106 / 110 | 111 / 103 | 105 / 103 | 103, 816 (B3 S1024) 119 |
// 113 / 126 | 118 / 109 | 109 / 110 | 107, 840 (B2 S1280) 114 | 109 / 120 | 115 / 112 | 114 / 113 | 113, 1056 (B1 S2048) 133 | 126 / 136 | 135 / 134 | 133 / 131 | 130.
bool conv_mix16_fills(int64_t planes, int64_t rows, int64_t keys, bool lower_only, bool dense)
{
    const int64_t tr = (rows + 31) / 32, tk = (keys + 63) / 64, tiles = planes * (lower_only && rows == keys ? tk * (tk + 1) : tr * tk);
    return tiles >= 800 || (!dense && tiles >= 430 && tiles <= 490);
}

// Whether softmax, mixing and P V in one kernel (softmax_mix_pv.hip) beat softmax + mixing, then P V: its workgroups walk a row's keys, a chain that only a
// grid of enough blocks of 64 rows (over the groups of heads) hides, or short rows.  `padded`: a key bias, or rows that see no key - both kernels look for
// hidden keys at every step, and rows that start late are as long as any -, so the line lies higher; under windows and documents the chains are
// short and it lies where it does without a mask.  us of the forward, three kernels | two, several kernel sizes, 16 bits:
//   no mask, groups of 4    D128: 24 blocks (B1 H32 S184) 17.7 | 18.0, 36 (B4 H12 S184) 20.0 | 18.4, (B1 H8 S1152) 37.2 | 44.0, 96 (B4 H16 S376) 36.5 | 35.2, 104 (B4 H8 S832)
//     44.9 | 44.9, 160 (B1 H32 S1256) 74.2 | 70.9, 256 (B2 H16 S2000) 148 | 131;  D64: 12 (B1 H16 S136) 14.7 | 14.1, 32 (B2 H16 S208) 17.2 | 16.5, 36 (B1 H12 S752)
//     25.9 | 27.0, 64 (B1 H32 S464) 27.2 | 23.7, 84 (B4 H4 S1336) 46.9 | 48.3, 136 (B1 H16 S2176) 85.4 | 76.8, 256 (B1 H16 S4048) 236 | 194
//   windows and documents, groups of 4    D128: 36 (B4 H12 S184) 20.9 | 19.3, 64 (B1 H32 S464) 29.7 | 26.7, 132 (B1 H16 S2112) 73.0 | 62.1;  D64: 60 (B2 H12 S584) 27.7 |
//     26.0, 116 (B1 H16 S1856) 55.5 | 53.5, 138 (B1 H12 S2904) 75.1 | 62.2
//   padded, groups of 4    D128, right: 24 (B2 H16 S184) 20.8 | 22.2, 48 (B1 H32 S144) 6 % faster, 72 (B2 H16 S536) 38.1 | 41.1, 96 (B4 H16 S376) 40.7 | 42.6, 128 (B1 H16 S2000)
//     88.0 | 96.6, 160 (B2 H32 S264) 3 % faster, 208 (B1 H16 S3288) 210 | 195; left: 96 (B1 H32 S712) 8 % slower, 136 (B2 H16 S1088) even, 176 (B1 H16 S2760)
//     124 | 109;  D64, right: 72 (B4 H8 S568) 36.3 | 35.6, 76 (B1 H16 S1184) 45.7 | 51.0, 96 (B4 H16 S368) 35.2 | 34.0, 140 (B1 H16 S2200) 99.8 | 94.2, 256 (B1 H16 S4040) 240 |
//     199; left: 81 (B1 H12 S1672) 58.1 | 66.9, 171 (B1 H12 S3616) 163 | 145; up to 24 blocks of up to 256 keys 10 % faster or even (a launch less)
//   groups of 2: everywhere, B1 H4 S2112 D64 38.0 | 34.8, but for padded rows of few heads: B1 H4 D128 S3328 (104) 69.3 | 74.4, left 75.8 | 82.5
bool softmax_pv_pays(int64_t planes, int64_t keys, int64_t head_dim, int64_t group, bool padded)
{
    const int64_t blocks = planes / group * ((keys + 63) / 64);
    if (group == 2) return !padded || keys <= 20 * blocks || blocks > 130 || blocks < (head_dim == 64 ? 117 : 82);
    if (padded) return head_dim == 64 ? blocks >= 130 || keys <= 5 * blocks || (keys <= 256 && blocks <= 24) : blocks >= 140 || 2 * keys <= 7 * blocks;
    return head_dim == 64 ? blocks >= 80 || keys <= 16 * blocks || keys <= 256 : blocks >= 120 || keys <= 8 * blocks;
}

int64_t lcm(int64_t a, int64_t b)
{
    int64_t x = a, y = b;
    while (y) { const int64_t t = x % y; x = y; y = t; }
    return a / x * b;
}

// 1/sqrt(D) as the reference forms it: in fp32
double score_scale(const Tensor &q) { return (double)(1.0f / std::sqrt((float)q.size(-1))); }

// the optional observer of the modules: called with a stage's name right before the kernel (or library call) that does it is
// enqueued; a kernel that does several operators is one stage with a name of its own
struct Mark {
    const py::object &hook;
    void operator()(const char *stage) const
    {
        if (!hook.is_none()) hook(stage);
    }
};

// (B,H,S,D) seen as (B,S,H,D), of its first `rows` rows only if that is not negative, without a view relation that autograd
// would track
Tensor heads_last(const Tensor &o, int64_t rows)
{
    at::AutoDispatchBelowADInplaceOrView guard;
    return (rows < 0 ? o : o.narrow(2, 0, rows)).transpose(1, 2);
}

// int32 (B,S): p + 1 for the rows p that see no key, 0 for the others (mta_band_zero_fwd then clears those rows)
Tensor empty_row_ends(const Tensor &empty_rows)
{
    const Tensor rows = at::arange(1, empty_rows.size(-1) + 1, empty_rows.options().dtype(at::kInt));
    return at::where(empty_rows, rows.unsqueeze(0), at::zeros({}, rows.options())).contiguous();
}

// The dtype that a library product gives data of dtype t: under autocast its own.  The kernels that stand in for library products
// (fp32 products, padded lengths, raw scores as a stage of their own) are taken where that is the data's dtype; the ones that are
// a stage by themselves, with weights of the data's dtype, have never been subject to autocast.
at::ScalarType product_type(at::ScalarType t)
{
    return at::autocast::is_autocast_enabled(at::kCUDA) ? at::autocast::get_autocast_dtype(at::kCUDA) : t;
}

// a b by the library; outside autocast (a backward that runs there) in a's dtype, as it would be inside
Tensor matmul_as(const Tensor &a, const Tensor &b)
{
    return at::matmul(a, b.to(a.scalar_type()));
}

// forward-mode differentiation: the kernels know no tangents
bool has_tangent(const Tensor &t) { return t.defined() && t._fw_grad(0).defined(); }

void no_tangents(std::initializer_list<const Tensor *> ts, const char *what)
{
    for (const Tensor *t : ts) TORCH_CHECK_NOT_IMPLEMENTED(!has_tangent(*t), what, " does not implement forward-mode differentiation");
}

// Q, K and V of one batch, head count, length and dtype, which is what the row copies around the kernels take (of fewer than
// 2^31 elements).  Anything else the library products broadcast, and a V with a tangent they differentiate.
bool alike(const Tensor &q, const Tensor &k, const Tensor &v)
{
    if (has_tangent(v)) return false;
    if (q.dim() != 4 || k.sizes() != q.sizes() || v.dim() != 4 || v.size(0) != q.size(0) || v.size(1) != q.size(1) || v.size(2) != q.size(2))
        return false;
    return k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && std::max(q.numel(), v.numel()) < (int64_t(1) << 31);
}

// The sizes of Q K^T, as torch.matmul broadcasts them; raises where the two products of a call do not exist.
at::DimVector score_sizes(const Tensor &q, const Tensor &k, const Tensor &v)
{
    TORCH_CHECK_VALUE(k.dim() == 4 && q.dim() >= 2 && q.dim() <= 4 && v.dim() >= 1, "expected Q, K, V (B,H,S,D), got ", q.sizes(), ", ", k.sizes(), ", ",
                      v.sizes());
    TORCH_CHECK(q.size(-1) == k.size(-1), "Q and K must share their head size, got ", q.sizes(), " and ", k.sizes());
    TORCH_CHECK(v.size(v.dim() > 1 ? -2 : 0) == k.size(2), "K and V must share their length, got ", k.sizes(), " and ", v.sizes());
    TORCH_CHECK(k.device() == q.device() && v.device() == q.device(), "Q, K and V live on ", q.device(), ", ", k.device(), " and ", v.device());
    at::DimVector s = at::infer_size_dimvector(q.sizes().slice(0, q.dim() - 2), k.sizes().slice(0, 2));
    if (v.dim() > 2) at::infer_size_dimvector(s, v.sizes().slice(0, v.dim() - 2));
    s.push_back(q.size(-2));
    s.push_back(k.size(2));
    return s;
}

// Weights against the heads of the scores: an AssertionError, as the operators raise it, ahead of the first launch.
void check_weight(const Tensor &w, int64_t dim, int64_t heads, const Tensor &q, const char *what)
{
    TORCH_CHECK_VALUE(w.dim() == dim, what, " must have ", dim, " dimensions, got ", w.sizes());
    TORCH_CHECK(w.device() == q.device(), what, " lives on ", w.device(), ", Q on ", q.device());
    if (w.size(0) == heads && (dim == 3 || w.size(1) == heads)) return;
    PyErr_SetString(PyExc_AssertionError, c10::str(what, " ", w.sizes(), " does not match the ", heads, " heads of Q and K").c_str());
    throw py::error_already_set();
}

// The length the score kernels work on.  They move score rows as 16-byte vectors; under the causal rule a length that is not
// a multiple of 8 is padded with zero rows: only padding rows see the padding keys, so every result of a real row is what it
// was (their gradients are zero: the padding rows of the incoming gradient are).
int64_t padded_length(const Tensor &q, const Tensor &k, const Tensor &v, bool causal)
{
    const int64_t s = q.size(-2);
    return causal && alike(q, k, v) && product_type(q.scalar_type()) == q.scalar_type() ? (s + 7) / 8 * 8 : s;
}

// key_bias (fp32), first (int32) and empty_rows (bool): one value per batch entry of the scores and key (row).  Under the causal
// rule they arrive with the columns of a padded length; a call that is not padded takes the first `s` of them.
OptTensor mask_row(const OptTensor &t, at::ScalarType type, const char *what, const at::DimVector &scores, bool causal, int64_t s, const Tensor &q)
{
    if (!t) return t;
    const int64_t given = causal ? (scores[3] + 7) / 8 * 8 : scores[3];
    TORCH_CHECK(t->device() == q.device(), what, " lives on ", t->device(), ", Q on ", q.device());
    TORCH_CHECK_VALUE(t->scalar_type() == type && t->dim() == 2 && t->size(0) == scores[0] && t->size(1) == given, what, " must be ", type, " of shape (",
                      scores[0], ",", given, "), got ", t->scalar_type(), " ", t->sizes());
    return (s == given ? *t : t->narrow(1, 0, s)).contiguous();
}

// (B,H,S,D) with the rows of hidden keys zeroed, where no row copy does it on the way
Tensor zero_hidden(const Tensor &x, const Tensor &key_bias)
{
    return x.masked_fill((key_bias == -INFINITY).unsqueeze(1).unsqueeze(-1), 0);
}

// round(a b^T) on and below the diagonal of a (B,H,S,S) tensor, nothing written above it.  Nothing where there is no kernel.
// `first`: a band mask, zeros ahead of a row's first visible key (the kernel does not visit the key blocks no row of a query
// block sees, fp32 visits all: the hidden stretch of every row is cleared afterwards).
OptTensor lower_scores(const Tensor &a, const Tensor &b, const OptTensor &first)
{
    if (a.sizes() != b.sizes() || a.scalar_type() != b.scalar_type() || !a.is_cuda() ||
        !lower_products_supported(a.scalar_type(), a.sizes(), true))
        return std::nullopt;
    const bool in_place = rows_in_place(a);
    const Tensor x = in_place ? a : on_gpu_vectors(a, "Q"), y = on_gpu_vectors(b, "K");
    Tensor out = at::empty({x.size(0), x.size(1), x.size(2), x.size(2)}, x.options());
    if (in_place)
        check(mta_lower_scores_rows_fwd(ptr(x), x.stride(0), x.stride(1), x.stride(2), ptr(y), ptr(first), out_ptr(out), x.size(0), x.size(1), x.size(2),
                                        x.size(3), code(x, "Q"), stream_of(x)),
              "mta_lower_scores_fwd");
    else check(mta_lower_scores_fwd(ptr(x), ptr(y), is16(x) ? ptr(first) : nullptr, out_ptr(out), x.size(0), x.size(1), x.size(2), x.size(3), code(x, "Q"), stream_of(x)),
          "mta_lower_scores_fwd");
    if (first) band_zero_(out, *first);
    return out;
}

// whether the first and the last kernel of the 16-bit causal route take Q, K and V of fewer rows than the scores have where they lie
bool reads_ragged(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &conv_w, int64_t s_pad)
{
    for (const Tensor *x : {&q, &k, &v})
        if (!x->is_cuda() || !x->is_contiguous() || x->numel() == 0 || x->is_neg() || reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16) return false;
    return alike(q, k, v) && !has_tangent(v) && qk_conv_supported(q, k, conv_w, s_pad) && causal_pv_supported(v.scalar_type(), s_pad, v.size(3));
}

// ---- inference -------------------------------------------------------------------------------------------------------
// The fused route.  `key_bias`: fp32 (B,Sk), added to the mixed scores ahead of the softmax; the K rows of the keys it
// hides (-inf) are zeroed, so that their scores enter the pre-softmax conv as 0, and their V rows too where a post-softmax
// conv that is not the identity writes into their columns (`key_bias_hides`: its values are 0 and -inf).  `first`: int32 (B,S), a band mask (row p sees the keys
// first[p] .. p), applied to the scores inside the first kernel (where the first stage is two: between them) and as -inf inside the softmax kernel, and behind a
// post-softmax conv that is not the identity the hidden stretch of every row is zeroed again; the caller has checked that
// the first stage exists.  `empty_rows`: bool (B,S), the rows of the band that see no key (first[p] = p + 1): the softmax
// leaves NaN in them, which the reference replaces by zeros ahead of its post-softmax conv
// (mta_attention_triton.py:81) - here those rows of the probabilities are cleared ahead of a post-softmax conv that is not
// the identity, and their rows of the output, where nothing else would, at the end.
Tensor forward_inference(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &conv_w, const Tensor &w_pre, const Tensor &post_conv_w,
                         const Tensor &w_post, bool causal, bool pre_identity, int64_t pre_group, bool post_conv_identity, bool post_identity,
                         int64_t post_group, const OptTensor &key_bias_, bool key_bias_hides, const OptTensor &first_, const OptTensor &empty_rows_, bool planes,
                         double dropout, const py::object &hook)
{
    at::NoGradGuard no_grad;
    const c10::OptionalDeviceGuard guard(q_.is_cuda() ? std::optional<c10::Device>(q_.device()) : std::nullopt);
    const Mark mark{hook};
    const at::DimVector planes_of = score_sizes(q_, k_, v_);
    check_weight(conv_w, 3, planes_of[1], q_, "the conv weight");
    if (!pre_identity) check_weight(w_pre, 2, planes_of[1], q_, "the head weight ahead of the softmax");
    if (!post_conv_identity) check_weight(post_conv_w, 3, planes_of[1], q_, "the conv weight behind the softmax");
    if (!post_identity) check_weight(w_post, 2, planes_of[1], q_, "the head weight behind the softmax");
    const int64_t s_real = q_.size(-2), s_pad = padded_length(q_, k_, v_, causal);
    const int64_t columns = s_pad == s_real ? k_.size(2) : s_pad;
    const OptTensor key_bias = mask_row(key_bias_, at::kFloat, "the key mask", planes_of, causal, columns, q_),
                    first = mask_row(first_, at::kInt, "the band mask", planes_of, causal, columns, q_),
                    empty_rows = mask_row(empty_rows_, at::kBool, "the empty rows", planes_of, causal, columns, q_);
    Tensor q = q_, k = k_, v = v_;
    // A length that is not a multiple of 8, in 16 bits: the kernels at both ends read Q, K and V where they lie (`ragged`: the length of the scores).
    // The padded copies cost a launch and 3 to 13 us.  Forwards, us: bf16 6x11 / 3x3 B2 H16 S1001 D64 85.8 -> 79.8, 7x9 / 7x9 B1 H16 S283 32.7 -> 29.8, fp16
    // groups of 8 B1 H16 S1001 D64 41.2 -> 38.8.  Key masks keep the copies, which zero the hidden rows on the way.
    const int64_t ragged = s_pad != s_real && !key_bias && reads_ragged(q_, k_, v_, conv_w, s_pad) ? s_pad : 0;
    if (key_bias && !alike(q_, k_, v_)) {
        k = zero_hidden(k_, *key_bias);
        if (!post_conv_identity) v = zero_hidden(v_, *key_bias);
    } else if ((s_pad != s_real && !ragged) || key_bias) {
        RowsCopy rows(s_pad, key_bias);
        if (s_pad != s_real) q = rows.add(q_, false, 1.0);
        k = rows.add(k_, true, 1.0);
        if (s_pad != s_real || !post_conv_identity) v = rows.add(v_, !post_conv_identity, 1.0);
        rows.run();
    }
    // (what the padding rows hold is nobody's business)
    auto result = [&](const Tensor &out) { return (s_pad == s_real ? out : out.narrow(2, 0, s_real)).transpose(1, 2); };
    const double scale = score_scale(q);
    const int64_t heads = planes_of[1], n_keys = ragged ? ragged : k.size(-2);
    const OptTensor w1 = pre_identity ? OptTensor() : OptTensor(w_pre), w2 = post_identity ? OptTensor() : OptTensor(w_post);
    const int64_t g_pre = pre_identity ? 1 : pre_group ? pre_group : heads, g_post = post_identity ? 1 : post_group ? post_group : heads;
    const int64_t g_both = lcm(g_pre, g_post);
    const bool masked = key_bias || first;
    const bool qk_kernel = qk_conv_supported(q, k, conv_w, ragged), as_is = product_type(q.scalar_type()) == q.scalar_type();
    const auto dtype = qk_kernel ? q.scalar_type() : product_type(q.scalar_type());   // (of the scores)
    const bool one_pass = post_conv_identity && one_pass_group(g_both, dtype, n_keys, w1, w2) && masks_ok(g_both, dtype, masked);
    // the last stage may leave the upper triangle unwritten only if our own P V kernel consumes it
    const bool own_pv = (s_pad != s_real || score_planes_of(planes_of, v.sizes())) && !has_tangent(v) && dtype == v.scalar_type() &&
                        (as_is || dtype != at::kFloat) && (ragged || lower_products_supported(dtype, v.sizes(), causal));
    const bool bias_vectors = !key_bias || reinterpret_cast<uintptr_t>(ptr(*key_bias)) % 16 == 0;

    // Two kernels: the scores with the statistics of their rows, and softmax, mixing and P V in one, the probabilities in registers only (which
    // is why the hook hears of the two stages at once).
    if (causal && pre_identity && post_conv_identity && w2 && qk_kernel && own_pv && dropout <= 0 && !(key_bias && (first || !key_bias_hides)) &&
        softmax_pv_pays(planes_of[0] * heads, n_keys, v.size(-1), g_post, key_bias || empty_rows) && stats_route_supported(q, k, conv_w, g_post, *w2, key_bias.has_value(), ragged)) {
        const bool tri = !planes && g_post * tri_row_offset(n_keys) < (int64_t(1) << 31);
        mark("qk_conv");
        const auto [scores, stats] = qk_conv_stats(q, k, conv_w, scale, g_post, tri, key_bias, first, ragged);
        mark("mix_softmax_mix");
        mark("pv");
        Tensor out = softmax_mix_pv(scores, stats, *w2, v, conv_w.size(1), g_post, tri, key_bias, first, ragged);
        if (empty_rows) out.masked_fill_(empty_rows->unsqueeze(1).unsqueeze(-1), 0);
        mark("end");
        return result(out);
    }

    // Three kernels with nothing elementwise between them: the two score tensors are nobody else's business, and they travel
    // in the triangular layout (what lies on and below the diagonal only, the rows a workgroup of the softmax stage reads
    // side by side): half the footprint, and every stage streams memory in longer runs.
    if (!planes && causal && one_pass && own_pv && dropout <= 0 && (g_both == 2 || g_both == 4 || g_both == 8 || g_both == 16) && bias_vectors &&
        tri_route_supported(q, k, conv_w, g_both, w1, w2, first.has_value(), false, key_bias.has_value(), ragged)) {
        mark("qk_conv");
        Tensor scores = qk_conv_tri(q, k, conv_w, scale, g_both, first, ragged);
        mark("mix_softmax_mix");
        scores = headmix_softmax_tri(scores, w1, w2, q.size(0), heads, n_keys, g_both, first, false, key_bias);
        mark("pv");
        Tensor out = causal_pv_tri(scores, v, g_both, first, ragged);
        if (empty_rows) out.masked_fill_(empty_rows->unsqueeze(1).unsqueeze(-1), 0);
        mark("end");
        return result(out);
    }

    Tensor scores;
    // (dense groups of 16 heads ahead of a post-softmax conv: the first score tensor still travels in the triangular layout,
    // the softmax stage hands the conv (B,H,S,S) planes)
    const bool tri_first = !planes && causal && !one_pass && g_pre == 16 && masks_ok(16, dtype, masked) && w1 &&
                           !(post_conv_identity && !w2 && !own_pv) &&
                           tri_route_supported(q, k, conv_w, 16, w1, OptTensor(), first.has_value(), true, key_bias.has_value(), ragged);
    if (tri_first) {
        mark("qk_conv");
        scores = qk_conv_tri(q, k, conv_w, scale, 16, first, ragged);
    } else if (qk_kernel) {
        mark("qk_conv");
        scores = qk_conv(q, k, conv_w, causal, scale, false, first, ragged);
    } else {
        mark("qk");
        const OptTensor raw = causal && as_is ? lower_scores(q, k, first) : OptTensor();
        TORCH_CHECK(raw || !first, "the band mask needs the lower-triangle products");
        scores = raw ? *raw : at::matmul(q, k.transpose(2, 3));
        mark("conv_pre");   // (the stage that follows never reads above the diagonal)
        scores = conv2d(scores, conv_w, causal, scale, false);
    }

    if (one_pass) {
        mark("mix_softmax_mix");
        scores = headmix_softmax(scores, w1, w2, causal, g_both, !own_pv, key_bias, first);
    } else {
        const bool fill = post_conv_identity && !w2 && !own_pv;
        if (tri_first) {
            mark("mix_softmax");
            scores = headmix_softmax_tri(scores, w1, OptTensor(), q.size(0), heads, n_keys, g_pre, first, true, key_bias);
        } else if (one_pass_group(g_pre, dtype, n_keys, w1, OptTensor()) && masks_ok(g_pre, dtype, masked)) {
            mark("mix_softmax");
            scores = headmix_softmax(scores, w1, OptTensor(), causal, g_pre, fill, key_bias, first);
        } else {
            mark("mix_pre");   // (the softmax kernel that follows never reads above the diagonal)
            scores = headmix(scores, w_pre, causal, 0.0, g_pre, false);
            mark("softmax");
            scores = headmix_softmax(scores, OptTensor(), OptTensor(), causal, 0, fill, key_bias, first);
        }
        if (empty_rows && !post_conv_identity) band_zero_(scores, empty_row_ends(*empty_rows));
        // conv and mix in one pass, the conv result never written: taken where it measures at least as fast as the two
        // kernels.  Under a band mask the conv's result is zeroed at the hidden positions ahead of the mixing: two kernels.
        // - 16 heads at a time (dense groups of 16, or groups of 2 or 4) on the matrix cores, where there are tiles enough.
        // - groups of up to 4 heads and the sizes with a vector-staged instance, on the vector units: 3x3 in fp32, and while the
        //   tensor is so small that a launch counts.  One kernel | two, us, the lower triangle, 3x3 / 7x7: bf16 groups of 4, 12 x 768^2
        //   13 | 21 / 21 | 21, 12 x 1024^2 24 | 24 / 37 | 25, 32 x 1448^2 75 | 60 / 104 | 64, 12 x 2912^2 103 | 95 / 146 | 101; fp32 groups
        //   of 2, 16 x 512^2 13 | 20 / 22 | 22, 12 x 1024^2 27 | 30 / 54 | 36, 16 x 1536^2 52 | 70 / 106 | 81, 16 x 2048^2 115 | 117 / 268 | 141.
        const int64_t r = post_conv_w.size(1), s = post_conv_w.size(2);
        const bool mix16 = (g_post == 16 || ((g_post == 2 || g_post == 4) && heads % 16 == 0)) && ((r == 3 && s == 3) || (r == 5 && s == 5) || (r == 7 && s == 7)) && is16(scores) &&
                           post_conv_w.scalar_type() == scores.scalar_type() && w_post.scalar_type() == scores.scalar_type() && n_keys % 8 == 0;
        const bool small_groups = g_post <= 4 && g_post != 3 &&
                                  ((r == 3 && s == 3 && (dtype == at::kFloat || scores.numel() <= 12 << 20)) || (r == 7 && s == 7 && scores.numel() <= 6 << 20));
        OptTensor done;
        if (!first && !post_conv_identity && w2 &&
            (small_groups || (mix16 && conv_mix16_fills(scores.size(0) * (heads / 16), scores.size(2), n_keys, causal && own_pv, g_post == 16)))) {
            mark("conv_mix_post");
            done = conv2d_headmix(scores, post_conv_w, w_post, causal, g_post, !own_pv);
        }
        if (done) {
            scores = *done;
        } else {
            // neither our head mixing nor our P V reads above the diagonal: whoever feeds them need not write there
            if (!post_conv_identity) {
                mark("conv_post");
                scores = conv2d(scores, post_conv_w, causal, std::nullopt, !w2 && !own_pv);
                // (the conv has spread probability into columns the rows do not see: mta_attention_triton.py:82-83)
                if (first) band_zero_(scores, *first);
            }
            if (w2) {
                mark("mix_post");
                scores = headmix(scores, w_post, causal, 0.0, g_post, !own_pv);
            }
        }
    }
    if (dropout > 0) scores = at::dropout(scores, dropout, true);
    mark("pv");
    OptTensor out = own_pv ? causal_pv(scores, v, causal, first, 1.0, ragged) : OptTensor();
    if (!out) out = at::matmul(scores, v);
    if (empty_rows) out->masked_fill_(empty_rows->unsqueeze(1).unsqueeze(-1), 0);
    mark("end");
    return result(*out);
}

// ---- training ----------------------------------------------------------------------------------------------------------
struct TrainOptions {
    bool causal, pre_causal, post_causal;
    double pre_fill, post_fill;
    int64_t pre_group, post_group;   // 0 = dense (the weight gradient is then dense too)
    OptTensor first;       // int32 (B,S), a band mask
    OptTensor key_bias;    // fp32 (B,S): added ahead of the softmax; the K and V rows of the keys it hides (-inf) count as zeros
                           // and receive no gradient, as in the reference, whose masked_fill / where cut it
    OptTensor empty_rows;  // bool (B,S), the rows of the band that see no key: their probabilities are cleared
};

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

OptTensor option(const Tensor &t) { return t.defined() ? OptTensor(t) : OptTensor(); }
Tensor tensor(const OptTensor &t) { return t ? *t : Tensor(); }

// The reference's operator sequence (mta_attention_triton.py:68-92) in pieces, forward and backward.  Between two stages nothing
// reads above the diagonal when causal (the kernels never do, in either direction), so nothing is written there, except what goes
// into a library GEMM.

// Q K^T -> factor -> conv -> head mixing -> softmax.  raw: the raw scores, kept where the first stage is two operators; x: the
// conv's result.
Tensor probabilities(const Tensor &q, const Tensor &k, const Tensor &conv_w, const Tensor &w_pre, const TrainOptions &o, const Mark &mark, Tensor &raw,
                     Tensor &x)
{
    const double scale = score_scale(q);
    const bool fill = !o.causal;
    if (qk_conv_supported(q, k, conv_w)) {
        mark("qk_conv");
        x = qk_conv(q, k, conv_w, o.causal, scale, false, o.first);
        // The kernel leaves the key blocks that no row of a query block sees unwritten.  The softmax stage does not read
        // a row's hidden stretch, but its weight gradient multiplies what is stored there by a gradient that is 0: the
        // stretch is cleared, so that the product is 0 too.
        if (o.first) band_zero_(x, *o.first);
    } else {
        mark("qk");
        const bool as_is = product_type(q.scalar_type()) == q.scalar_type();
        const OptTensor lower_raw = o.causal && as_is ? lower_scores(q, k, o.first) : OptTensor();
        TORCH_CHECK(lower_raw || !o.first, "the band mask needs the lower-triangle products");
        raw = lower_raw ? *lower_raw : at::matmul(q, k.transpose(2, 3));
        mark("conv_pre");
        x = conv2d(raw, conv_w, o.causal, scale, false);
    }
    const int64_t heads = w_pre.size(0), n_keys = k.size(-2), g_eff = o.pre_group ? o.pre_group : heads;
    const auto dtype = x.scalar_type();
    Tensor p;
    // (groups of more than 8 heads, but for 16 in 16 bits: with the head weight's own causal rule apart from the module's the mixing
    // stays alone)
    if ((g_eff <= FUSED_MAX_GROUP || (dtype != at::kFloat && g_eff == FUSED_MFMA_GROUP) || o.pre_causal == o.causal) && one_pass_group(g_eff, dtype, n_keys, w_pre, OptTensor()) &&
        masks_ok(g_eff, dtype, o.key_bias || o.first)) {
        mark("mix_softmax");
        p = headmix_softmax(x, w_pre, OptTensor(), o.causal, o.pre_group, fill, o.key_bias, o.first);
    } else {
        mark("mix_pre");
        const Tensor m = headmix(x, w_pre, o.pre_causal, fill ? o.pre_fill : 0.0, o.pre_group, fill);
        mark("softmax");
        p = headmix_softmax(m, OptTensor(), OptTensor(), o.causal, 0, fill, o.key_bias, o.first);
    }
    if (o.empty_rows) band_zero_(p, empty_row_ends(*o.empty_rows));
    return p;
}

// The gradients of a head mixing with respect to its input and its weight (those that are wanted).  One kernel where it is both;
// small: also for one of them, which costs nothing there and gives the bits that it has beside the other.
std::pair<Tensor, Tensor> headmix_bwd(const Tensor &dy, const Tensor &x, const Tensor &w, bool causal, int64_t group, bool fill_upper, bool need_x,
                                      bool need_w, bool small, Sums &sums)
{
    if ((need_x && need_w) || (small && (need_x || need_w))) {
        if (auto both = headmix_grads(std::nullopt, dy, x, w, causal, group, fill_upper, sums))
            return {need_x ? both->first : Tensor(), need_w ? both->second : Tensor()};
    }
    return {need_x ? headmix_bwd_input(dy, w, causal, group, fill_upper) : Tensor(),
            need_w ? headmix_bwd_weight(x, dy.to(x.scalar_type()), w, causal, group) : Tensor()};
}

// the gradients of q, k, conv_w and w_pre (need[i]: wanted) from the one of the probabilities p.  small: as in headmix_bwd
void probabilities_bwd(const Tensor &q, const Tensor &k, const Tensor &conv_w, const Tensor &w_pre, Tensor raw, const Tensor &x, const Tensor &p,
                       const OptTensor &first, bool causal, bool pre_causal, int64_t pre_group, Tensor dp, const bool (&need)[4], Tensor *(&&out)[4], bool small, Sums &sums)
{
    const double scale = score_scale(q);
    // (the head mixing's gradient kernels never read above the diagonal when causal)
    Tensor dx;
    const bool need_x = need[0] || need[1] || need[2];
    // (one kernel for the three gradients, also where one of them is for nobody: it reads less than the two that it takes otherwise)
    const auto all = causal == pre_causal ? headmix_grads(p, dp, x, w_pre, causal, pre_group, !causal, sums) : std::nullopt;
    if (all) {
        dp.reset();
        if (need[3]) *out[3] = all->second;
        if (!need_x) return;
        dx = all->first;
    } else {
        Tensor ds = softmax_bwd(p, dp, causal, false);
        dp.reset();
        if (need[3]) *out[3] = headmix_bwd_weight(x, ds, w_pre, pre_causal, pre_group);
        if (!need_x) return;
        dx = headmix_bwd_input(ds, w_pre, pre_causal, pre_group, !causal);
    }
    auto stage_input = [&] {   // (the kernel gradient reads its first argument on and below the diagonal only)
        if (raw.defined()) return;
        const OptTensor lower_raw = causal ? lower_scores(q, k, first) : OptTensor();
        TORCH_CHECK(lower_raw || !first);
        raw = lower_raw ? *lower_raw : at::matmul(q, k.transpose(2, 3));
    };
    const bool lower = causal && q.sizes() == k.sizes() && dx.scalar_type() == q.scalar_type() && lower_products_supported(q.scalar_type(), q.sizes(), true);
    Tensor g;
    if (need[2] && (need[0] || need[1] || small)) {
        const bool formed = !raw.defined();   // (formed here: no further tensor for the gradient)
        stage_input();
        if (auto both = conv2d_grads(raw, dx, conv_w, causal, !lower, scale, sums, formed)) {
            std::tie(g, *out[2]) = *both;
            raw.reset();
        }
    }
    if (need[0] || need[1]) {
        if (!g.defined()) g = conv2d_bwd_input(dx, conv_w, causal, !lower);
        if (first) band_zero_(g, *first);
        Tensor dq, dk;
        OptTensor own_q, own_k;
        if (lower && need[0] && need[1]) {
            if (const auto both = causal_products(g, k, q, scale)) std::tie(own_q, own_k) = *both;
        }
        if (need[0] && !own_q) own_q = lower ? causal_pv(g, k, true, OptTensor(), scale) : OptTensor();
        if (need[0]) dq = own_q ? *own_q : matmul_as(g, k);
        if (need[1] && !own_k) own_k = lower ? causal_ptx(g, q, true, scale) : OptTensor();
        if (need[1]) dk = own_k ? *own_k : matmul_as(g.transpose(2, 3), q);
        // the factor, where the products were the library's
        if (need[0] && need[1] && !own_q && !own_k && dq.sizes() == dk.sizes()) {
            RowsCopy rows(dq.size(2), OptTensor());
            dq = rows.add(dq, false, scale);
            dk = rows.add(dk, false, scale);
            rows.run();
        } else {
            if (need[0] && !own_q) dq = dq * scale;
            if (need[1] && !own_k) dk = dk * scale;
        }
        *out[0] = dq;
        *out[1] = dk;
    }
    if (need[2] && !out[2]->defined()) {
        stage_input();
        *out[2] = conv2d_bwd_weight(raw, dx, conv_w, causal, scale, sums);
    }
}

// whether M V and its gradients run on the lower triangle of M (the last stage's output): by the library GEMM M is read in full
bool lower_values(const Tensor &m, const Tensor &v, const TrainOptions &o)
{
    const bool lower = o.causal && o.post_causal && m.scalar_type() == v.scalar_type() && score_planes_of(m.sizes(), v.sizes()) &&
                       lower_products_supported(v.scalar_type(), v.sizes(), true);
    TORCH_CHECK(!o.first || lower, "the band mask needs the lower-triangle products");
    return lower;
}

// M V, seen as (B,S,H,D), its first s_real rows
Tensor values(const Tensor &m, const Tensor &v, bool lower, int64_t s_real, const OptTensor &first)
{
    const Tensor out = lower ? *causal_pv(m, v, true, first, 1.0) : at::matmul(m, v);
    return heads_last(out, s_real == m.size(2) ? -1 : s_real);
}

// the incoming gradient as (B,H,S,D), padded with zero rows; a copy (6 us at B1 H16 S2048 D128 in 16 bits, and a launch of a small step)
// only where rows are added or the products do not take rows where they lie
Tensor value_rows(const Tensor &grad, int64_t s_pad, const Tensor &m, bool lower)
{
    const Tensor go = grad.transpose(1, 2);
    // (the lower-triangle kernels read 16-bit rows where they lie)
    if (lower && go.dim() == 4 && go.size(2) == s_pad && go.scalar_type() == m.scalar_type() && rows_in_place(go)) return go;
    if (go.dim() != 4 || go.numel() >= (int64_t(1) << 31)) return go.contiguous();   // (beyond what a padded length is used for)
    RowsCopy rows(s_pad, OptTensor());
    const Tensor out = rows.add(go, false, 1.0);
    rows.run();
    return out;
}

Tensor values_bwd_v(const Tensor &m, const Tensor &go, bool lower)
{
    const OptTensor own = lower ? causal_ptx(m, go, true, 1.0) : OptTensor();
    return own ? *own : matmul_as(m.transpose(2, 3), go);
}

// (first: the gradient is formed inside the band)
Tensor values_bwd_m(const Tensor &go, const Tensor &v, bool lower, const OptTensor &first)
{
    const OptTensor own = lower ? lower_scores(go, v, first) : OptTensor();
    TORCH_CHECK(own || !first);
    return own ? *own : matmul_as(go, v.transpose(2, 3));
}

// The pieces as one node: the host's time is what bounds a step of small tensors (a node costs about 8.6 us of it, forward and
// backward together).  Everything saved stays to the end of backward, so only for score tensors of up to WHOLE_STEP_BYTES, where
// that is at most five of them more at the peak (80 MB); beyond, the step is the kernels' time and a node per score tensor costs
// nothing.  us a step, one node | four (timed in turn; from process to process the host's part differs by as much): B1 H8 S256 D64
// bf16 (1 MB a score tensor) 181 | 205, B1 H16 S512 D128 (8 MB) 174 | 191, B1 H16 S1024 D64 (32 MB) 239 | 239.
constexpr int64_t WHOLE_STEP_BYTES = int64_t(16) << 20;

struct WholeStep : torch::autograd::Function<WholeStep> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &conv_w, const Tensor &w_pre,
                          const Tensor &post_conv_w, const Tensor &w_post, int64_t s_pad, double dropout, const TrainOptions *opt, const Mark *mark_)
    {
        const TrainOptions &o = *opt;
        const Mark &mark = *mark_;
        const int64_t s_real = q_.size(2);
        Tensor q = q_, k = k_, v = v_;
        if (s_pad != s_real || o.key_bias) {
            RowsCopy rows(s_pad, o.key_bias);
            if (s_pad != s_real) q = rows.add(q_, false, 1.0);
            k = rows.add(k_, true, 1.0);
            v = rows.add(v_, true, 1.0);
            rows.run();
        }
        Tensor raw, x, keep;
        const Tensor p = probabilities(q, k, conv_w, w_pre, o, mark, raw, x);
        mark("conv_post");
        const Tensor c = conv2d(p, post_conv_w, o.causal, std::nullopt, !o.causal);
        if (o.first) band_zero_(c, *o.first);
        mark("mix_post");
        const bool lower = lower_values(c, v, o);
        Tensor m = headmix(c, w_post, o.post_causal, lower ? 0.0 : o.post_fill, o.post_group, !lower);
        if (dropout > 0) std::tie(m, keep) = at::native_dropout(m, dropout, true);
        mark("pv");
        const Tensor out = values(m, v, lower, s_real, o.first);
        mark("end");
        ctx->save_for_backward({q, k, v, conv_w, w_pre, post_conv_w, w_post, raw, x, p, c, m, keep, tensor(o.first), tensor(o.key_bias)});
        ctx->saved_data["s_real"] = s_real;
        ctx->saved_data["causal"] = o.causal;
        ctx->saved_data["pre_causal"] = o.pre_causal;
        ctx->saved_data["post_causal"] = o.post_causal;
        ctx->saved_data["pre_group"] = o.pre_group;
        ctx->saved_data["post_group"] = o.post_group;
        ctx->saved_data["dropout"] = dropout;
        ctx->saved_data["lower"] = lower;
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &conv_w = saved[3], &w_pre = saved[4], &post_conv_w = saved[5],
                     &w_post = saved[6], &raw = saved[7], &x = saved[8], &p = saved[9], &c = saved[10], &m = saved[11], &keep = saved[12];
        const OptTensor first = option(saved[13]), key_bias = option(saved[14]);
        const int64_t s_real = ctx->saved_data["s_real"].toInt(), s_pad = q.size(2);
        const bool causal = ctx->saved_data["causal"].toBool(), pre_causal = ctx->saved_data["pre_causal"].toBool(),
                   post_causal = ctx->saved_data["post_causal"].toBool(), lower = ctx->saved_data["lower"].toBool();
        const int64_t pre_group = ctx->saved_data["pre_group"].toInt(), post_group = ctx->saved_data["post_group"].toInt();
        const double dropout = ctx->saved_data["dropout"].toDouble();
        const c10::OptionalDeviceGuard guard(q.device());
        bool need[7];
        for (int i = 0; i < 7; ++i) need[i] = ctx->needs_input_grad(i);
        const bool need_x = need[0] || need[1] || need[3], need_p = need_x || need[4], need_c = need_p || need[5];
        const bool small = (int64_t)p.nbytes() <= WHOLE_STEP_BYTES;   // (anomaly mode takes this node at any size)
        variable_list out(11);
        Sums sums;
        const Tensor go = value_rows(grads[0], s_pad, m, lower);
        if (need[2]) out[2] = values_bwd_v(m, go, lower);
        if (need_c || need[6]) {
            Tensor dm = values_bwd_m(go, v, lower, first);
            if (dropout > 0) dm = at::native_dropout_backward(dm, keep, dropout < 1 ? 1.0 / (1.0 - dropout) : 0.0);
            Tensor dc;
            std::tie(dc, out[6]) = headmix_bwd(dm, c, w_post, post_causal, post_group, !causal, need_c, need[6], small, sums);
            dm.reset();
            Tensor dp;
            if (need[5] && (need_p || small)) {   // (alone, too: see headmix_bwd)
                if (auto both = conv2d_grads(p, dc, post_conv_w, causal, !causal, 1.0, sums)) std::tie(dp, out[5]) = *both;
            }
            if (need[5] && !out[5].defined()) out[5] = conv2d_bwd_weight(p, dc, post_conv_w, causal, 1.0, sums);
            if (need_p) {
                if (!dp.defined()) dp = conv2d_bwd_input(dc, post_conv_w, causal, !causal);
                dc.reset();
                probabilities_bwd(q, k, conv_w, w_pre, raw, x, p, first, causal, pre_causal, pre_group, std::move(dp), {need[0], need[1], need[3], need[4]},
                                  {&out[0], &out[1], &out[3], &out[4]}, small, sums);
            }
        }
        sums.run();
        // the gradients of Q, K and V leave without the padding and without what the hidden keys' rows hold
        RowsCopy rows(s_real, key_bias);
        for (int i = 0; i < 3; ++i)
            if (out[i].defined() && (s_pad != s_real || (i > 0 && key_bias))) out[i] = rows.add(out[i], i > 0, 1.0);
        rows.run();
        return out;
    }
};

// ---- ... and as one node per score tensor that is kept: the engine frees what a node has saved and the gradient it was given
// when the node is done, so that backward holds the four saved tensors (x, p, c, m; raw too where there is one) and one or two
// gradients at a time.

// The tensors in a padded length, the rows of hidden keys zeroed from the `hide_from`th on; backward: without the padding and
// without what those rows got.
struct PadRows : torch::autograd::Function<PadRows> {
    static variable_list forward(AutogradContext *ctx, at::TensorList xs, int64_t hide_from, int64_t s_pad, const OptTensor *key_bias)
    {
        ctx->save_for_backward({tensor(*key_bias)});
        ctx->saved_data["s_real"] = xs[0].size(2);
        ctx->saved_data["hide_from"] = hide_from;
        variable_list out;
        RowsCopy rows(s_pad, *key_bias);
        for (const Tensor &x : xs) out.push_back(rows.add(x, (int64_t)out.size() >= hide_from, 1.0));
        rows.run();
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const OptTensor key_bias = option(ctx->get_saved_variables()[0]);
        const int64_t s_real = ctx->saved_data["s_real"].toInt(), hide_from = ctx->saved_data["hide_from"].toInt();
        const c10::OptionalDeviceGuard guard(grads[0].device());
        RowsCopy rows(s_real, key_bias);
        variable_list out(grads.size() + 3);
        for (size_t i = 0; i < grads.size(); ++i) {
            if (!ctx->needs_input_grad(i)) continue;
            const bool hide = (int64_t)i >= hide_from && key_bias;
            out[i] = hide || grads[i].size(2) != s_real ? rows.add(grads[i], hide, 1.0) : grads[i];
        }
        rows.run();
        return out;
    }
};

struct Probabilities : torch::autograd::Function<Probabilities> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &conv_w, const Tensor &w_pre, const TrainOptions *o,
                          const Mark *mark)
    {
        Tensor raw, x;
        const Tensor p = probabilities(q, k, conv_w, w_pre, *o, *mark, raw, x);
        ctx->save_for_backward({q, k, conv_w, w_pre, raw, x, p, tensor(o->first)});
        ctx->saved_data["causal"] = o->causal;
        ctx->saved_data["pre_causal"] = o->pre_causal;
        ctx->saved_data["pre_group"] = o->pre_group;
        return p;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto s = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(s[0].device());
        variable_list out(6);
        Sums sums;
        probabilities_bwd(s[0], s[1], s[2], s[3], s[4], s[5], s[6], option(s[7]), ctx->saved_data["causal"].toBool(),
                          ctx->saved_data["pre_causal"].toBool(), ctx->saved_data["pre_group"].toInt(), grads[0].to(s[6].scalar_type()),
                          {ctx->needs_input_grad(0), ctx->needs_input_grad(1), ctx->needs_input_grad(2), ctx->needs_input_grad(3)},
                          {&out[0], &out[1], &out[2], &out[3]}, false, sums);
        sums.run();
        return out;
    }
};

// the two operators: nodes of their own, and the post-softmax conv and head mixing of a training step
struct Conv2d : torch::autograd::Function<Conv2d> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &w, bool causal, bool fill_upper, bool grad_fill_upper)
    {
        ctx->save_for_backward({x, w});
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["grad_fill_upper"] = grad_fill_upper;
        return conv2d(x, w, causal, std::nullopt, fill_upper);
    }
    // convolution_2d_trit.py:336-378.  The reference returns the weight gradient in fp64 and lets autograd cast it; here it
    // is accumulated in fp32 and cast to the weight's dtype.
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(saved[0].device());
        const bool causal = ctx->saved_data["causal"].toBool();
        torch::autograd::variable_list out(5);
        const Tensor dy = on_gpu(grads[0], "grad_output");
        const bool fill_upper = ctx->saved_data["grad_fill_upper"].toBool();
        Sums sums;
        if (ctx->needs_input_grad(0) && ctx->needs_input_grad(1)) {
            if (auto both = conv2d_grads(saved[0], dy, saved[1], causal, fill_upper, 1.0, sums)) std::tie(out[0], out[1]) = *both;
        }
        if (ctx->needs_input_grad(0) && !out[0].defined()) out[0] = conv2d_bwd_input(dy, saved[1], causal, fill_upper);
        if (ctx->needs_input_grad(1) && !out[1].defined()) out[1] = conv2d_bwd_weight(saved[0], dy.to(saved[0].scalar_type()), saved[1], causal, 1.0, sums);
        sums.run();
        return out;
    }
};

struct HeadMix : torch::autograd::Function<HeadMix> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &w, bool causal, double fill, int64_t group,
                          bool fill_upper, bool grad_fill_upper)
    {
        ctx->save_for_backward({x, w});
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["group"] = group;
        ctx->saved_data["grad_fill_upper"] = grad_fill_upper;
        return headmix(x, w, causal, fill_upper || !causal ? fill : 0.0, group, fill_upper);
    }
    // triton_linear_head.py:322-370.  Above the diagonal the input gradient is 0 (the reference leaves torch.empty_like
    // memory there); the weight gradient is accumulated in fp32 and cast.
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(saved[0].device());
        const bool causal = ctx->saved_data["causal"].toBool();
        const int64_t group = ctx->saved_data["group"].toInt();
        torch::autograd::variable_list out(7);
        const Tensor dy = on_gpu(grads[0], "grad_output");
        Sums sums;
        std::tie(out[0], out[1]) = headmix_bwd(dy, saved[0], saved[1], causal, group, ctx->saved_data["grad_fill_upper"].toBool(),
                                               ctx->needs_input_grad(0), ctx->needs_input_grad(1), false, sums);
        sums.run();
        return out;
    }
};

struct Values : torch::autograd::Function<Values> {
    static Tensor forward(AutogradContext *ctx, const Tensor &m, const Tensor &v, bool lower, int64_t s_real, const OptTensor *first)
    {
        ctx->save_for_backward({m, v, tensor(*first)});
        ctx->saved_data["lower"] = lower;
        return values(m, v, lower, s_real, *first);
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto s = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(s[0].device());
        const bool lower = ctx->saved_data["lower"].toBool();
        const Tensor go = value_rows(grads[0], s[0].size(2), s[0], lower);
        variable_list out(5);
        if (ctx->needs_input_grad(1)) out[1] = values_bwd_v(s[0], go, lower);
        if (ctx->needs_input_grad(0)) out[0] = values_bwd_m(go, s[1], lower, option(s[2]));
        return out;
    }
};

Tensor forward_training(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &conv_w, const Tensor &w_pre, const Tensor &post_conv_w,
                        const Tensor &w_post, bool causal, bool pre_causal, bool post_causal, double pre_fill, double post_fill,
                        int64_t pre_group, int64_t post_group, const OptTensor &key_bias, const OptTensor &first, const OptTensor &empty_rows,
                        double dropout, const py::object &hook)
{
    const c10::OptionalDeviceGuard guard(q_.is_cuda() ? std::optional<c10::Device>(q_.device()) : std::nullopt);
    no_tangents({&q_, &k_, &v_, &conv_w, &w_pre, &post_conv_w, &w_post}, "MTAAttentionTriton");
    const at::DimVector planes_of = score_sizes(q_, k_, v_);
    const int64_t heads = planes_of[1], s_real = q_.size(-2), s_pad = padded_length(q_, k_, v_, causal), columns = s_pad == s_real ? k_.size(2) : s_pad;
    check_weight(conv_w, 3, heads, q_, "the conv weight");
    check_weight(w_pre, 2, heads, q_, "the head weight ahead of the softmax");
    check_weight(post_conv_w, 3, heads, q_, "the conv weight behind the softmax");
    check_weight(w_post, 2, heads, q_, "the head weight behind the softmax");
    const TrainOptions o{causal, pre_causal, post_causal, pre_fill, post_fill, pre_group, post_group,
                         mask_row(first, at::kInt, "the band mask", planes_of, causal, columns, q_),
                         mask_row(key_bias, at::kFloat, "the key mask", planes_of, causal, columns, q_),
                         mask_row(empty_rows, at::kBool, "the empty rows", planes_of, causal, columns, q_)};
    const Mark mark{hook};
    const bool rows_alike = alike(q_, k_, v_);
    // (anomaly mode looks for NaN in what goes from node to node, also above the diagonal, where nobody writes)
    if (rows_alike && (planes_of[0] * heads * s_pad * s_pad * (int64_t)q_.element_size() <= WHOLE_STEP_BYTES || torch::autograd::AnomalyMode::is_enabled()))
        return WholeStep::apply(q_, k_, v_, conv_w, w_pre, post_conv_w, w_post, s_pad, dropout, &o, &mark);
    Tensor q = q_, k = k_, v = v_;
    if (o.key_bias && !rows_alike) {
        k = zero_hidden(k_, *o.key_bias);
        v = zero_hidden(v_, *o.key_bias);
    } else if (s_pad != s_real || o.key_bias) {
        const bool pad = s_pad != s_real;
        const Tensor given[3] = {q_, k_, v_};
        const auto rows = PadRows::apply(at::TensorList(given + !pad, 2 + pad), (int64_t)pad, s_pad, &o.key_bias);
        if (pad) q = rows[0];
        k = rows[pad];
        v = rows[1 + pad];
    }
    Tensor t = Probabilities::apply(q, k, conv_w, w_pre, &o, &mark);
    mark("conv_post");
    t = Conv2d::apply(t, post_conv_w, causal, !causal, !causal);
    // (the hidden stretch receives a gradient of 0: the one with respect to the last scores is formed inside the band)
    if (o.first) band_zero_(t, *o.first);
    mark("mix_post");
    const bool lower = lower_values(t, v, o);
    t = HeadMix::apply(t, w_post, post_causal, post_fill, post_group, !lower, !causal);
    if (dropout > 0) t = at::dropout(t, dropout, true);
    mark("pv");
    t = Values::apply(t, v, lower, s_real, &o.first);
    mark("end");
    return t;
}

// ---- the two operators ---------------------------------------------------------------------------------------------
bool wants_grad(const Tensor &a, const Tensor &b) { return at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad()); }

Tensor conv2d_apply(const Tensor &x, const Tensor &w, bool causal, bool fill_upper, bool grad_fill_upper)
{
    const c10::OptionalDeviceGuard guard(x.is_cuda() ? std::optional<c10::Device>(x.device()) : std::nullopt);
    no_tangents({&x, &w}, "Conv2dTriton");
    if (!wants_grad(x, w)) return conv2d(x, w, causal, std::nullopt, fill_upper);
    return Conv2d::apply(x, w, causal, fill_upper, grad_fill_upper);
}

Tensor headmix_apply(const Tensor &x, const Tensor &w, bool causal, double fill, int64_t group, bool fill_upper, bool grad_fill_upper)
{
    const c10::OptionalDeviceGuard guard(x.is_cuda() ? std::optional<c10::Device>(x.device()) : std::nullopt);
    no_tangents({&x, &w}, "TritonLinearHead");
    if (!wants_grad(x, w)) return headmix(x, w, causal, fill_upper || !causal ? fill : 0.0, group, fill_upper);
    return HeadMix::apply(x, w, causal, fill, group, fill_upper, grad_fill_upper);
}

// Conv-attention in fp32 as scores, conv, softmax and P V, one kernel each, over as many planes at a time as 256 MB hold (one of S = 8192).
// us, parts of 128 MB | 256: 6x11 B1 H32 S4096 D128 2755 | 2234, B8 H32 S1024 D128 1391 | 1237, 7x9 B3 H4 S2300 D64 310 | 246.  Scratch: 512 MB
// at most, for scores, conv and softmax, or, where three do not fit, the softmax where the scores were (two | three: 3x3 B1 H4 S1024 D64
// 39.4 | 37.1, B1 H8 51.9 | 49.3, 7x7 B1 H8 S768 D128 54.9 | 53.0; from 100 MB a tensor on alike).  Nothing where the fused kernel is taken.
OptTensor conv_attn_stages(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &w, bool causal, double scale)
{
    constexpr int64_t SCRATCH = 256 << 20;
    if (q_.scalar_type() != at::kFloat || !causal || q_.numel() == 0) return std::nullopt;
    const int64_t b = q_.size(0), h = q_.size(1), s_real = q_.size(2), d = q_.size(3), s = (s_real + 7) / 8 * 8, plane = s * s * 4;
    const int64_t r = w.size(1), sk = w.size(2);
    for (const Tensor *x : {&q_, &k_, &v_})   // (what the fused kernel refuses stays refused)
        if (reinterpret_cast<uintptr_t>(ptr(*x)) % 16) return std::nullopt;
    if (plane > SCRATCH || !lower_products_supported(at::kFloat, {b, h, s, d}, true) || !mta_conv_attn_in_stages(b, h, s_real, d, (int)r, (int)sk, causal, MTA_F32)) return std::nullopt;
    Tensor q = q_, k = k_, v = v_;
    if (s != s_real) {   // (the products take rows that are whole vectors)
        RowsCopy rows(s, OptTensor());
        q = rows.add(q_, false, 1.0);
        k = rows.add(k_, false, 1.0);
        v = rows.add(v_, false, 1.0);
        rows.run();
    }
    Tensor o = at::empty(q.sizes(), q.options());
    // equal parts: of the batch, or of one batch entry's heads
    auto part = [](int64_t count, int64_t most) { const int64_t parts = (count + most - 1) / most; return (count + parts - 1) / parts; };
    const int64_t nb = h * plane <= SCRATCH ? part(b, SCRATCH / (h * plane)) : 1, nh = h * plane <= SCRATCH ? h : part(h, SCRATCH / plane);
    const Tensor raw = at::empty({nb, nh, s, s}, q.options()), conv = at::empty({nb, nh, s, s}, q.options()),
                 probs = 3 * nb * nh * plane <= 2 * SCRATCH ? at::empty({nb, nh, s, s}, q.options()) : raw;
    void *const st = stream_of(q), *const x = out_ptr(raw), *const y = out_ptr(conv), *const p = out_ptr(probs);
    const auto *qp = q.const_data_ptr<float>(), *kp = k.const_data_ptr<float>(), *vp = v.const_data_ptr<float>();
    const auto *wp = static_cast<const char *>(ptr(w));
    for (int64_t b0 = 0; b0 < b; b0 += nb)
        for (int64_t h0 = 0; h0 < h; h0 += nh) {   // (a part lies in one piece: all heads, or one batch entry)
            const int64_t bs = std::min(nb, b - b0), hs = std::min(nh, h - h0), at = (b0 * h + h0) * s * d;
            check(mta_lower_scores_f32(qp + at, kp + at, x, bs, hs, s, d, st), "mta_lower_scores_f32");
            check(mta_conv2d_scaled_fwd(x, wp + h0 * r * sk * w.element_size(), y, bs, hs, s, s, (int)r, (int)sk, causal_mode(true, false), (float)scale,
                                        MTA_F32, code(w, "W"), st),
                  "mta_conv2d_fwd");
            check(mta_headmix_softmax_band_fwd(y, nullptr, nullptr, nullptr, nullptr, p, bs, hs, s, s, 0, true, false, MTA_F32, MTA_F32, st),
                  "mta_headmix_softmax_band_fwd");
            check(mta_causal_pv_f32(p, vp + at, o.mutable_data_ptr<float>() + at, bs, hs, s, d, 1.0f, st), "mta_causal_pv_f32");
        }
    return s == s_real ? o : o.narrow(2, 0, s_real).contiguous();
}

// O = softmax(mask(conv(mask0(Q K^T))) * scale) V, without the row statistic a backward pass would keep
Tensor conv_attn(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &w_, bool causal, std::optional<double> softmax_scale)
{
    no_tangents({&q_, &k_, &v_, &w_}, "TritonConvAttention");
    const Tensor q = on_gpu(q_, "Q"), k = on_gpu(k_, "K"), v = on_gpu(v_, "V"), w = on_gpu(w_, "W");
    TORCH_CHECK_VALUE(q.dim() == 4 && q.sizes() == k.sizes() && q.sizes() == v.sizes(), "Q, K, V must share a (B,H,S,D) shape, got ", q.sizes(),
                      ", ", k.sizes(), ", ", v.sizes());
    TORCH_CHECK_TYPE(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(), "Q, K, V must share a dtype");
    TORCH_CHECK(w.dim() == 3 && w.size(0) == q.size(1), "CHANNEL_DIM == NUM_HEADS");
    const c10::OptionalDeviceGuard guard(q.device());
    const double scale = softmax_scale ? *softmax_scale : 1.0 / std::sqrt((double)q.size(3));
    try {
        if (OptTensor staged = conv_attn_stages(q, k, v, w, causal, scale)) return *staged;
    } catch (const c10::OutOfMemoryError &) {   // (the fused kernel needs none of it)
    }
    Tensor o = at::empty(q.sizes(), q.options());
    check(mta_conv_attn_fwd(ptr(q), ptr(k), ptr(v), ptr(w), out_ptr(o), q.size(0), q.size(1), q.size(2), q.size(3), (int)w.size(1), (int)w.size(2),
                            causal, (float)scale, code(q, "Q"), code(w, "W"), stream_of(q)),
          "mta_conv_attn_fwd");
    return o;
}

}  // namespace
}  // namespace mta_host

PYBIND11_MODULE(_host, m)
{
    using namespace mta_host;
    m.def("forward_inference", &forward_inference);
    m.def("forward_training", &forward_training);
    m.def("conv2d_apply", &conv2d_apply);
    m.def("headmix_apply", &headmix_apply);
    m.def("conv_attn", &conv_attn);
}
