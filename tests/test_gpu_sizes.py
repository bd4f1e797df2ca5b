"""GPU parity at the sizes where a kernel's tiling can go wrong - remainders, edges of tiles, the smallest of a range - for
kernel variants that a rule on sizes or types chooses.  Against the CPU oracle; tolerances as in test_gpu_attention.py for
module outputs (fp32 rtol 1e-4 / atol 1e-5, 16-bit atol 2e-2), derived where the test says so."""
import pytest
import torch

from oracle import mta_oracle as O

pytestmark = pytest.mark.gpu


def tol(dtype):
    return dict(rtol=1e-4, atol=1e-5) if dtype == torch.float32 else dict(rtol=0.0, atol=2e-2)


@pytest.fixture(scope="module")
def pkg():
    import multitokenatention_triton_amd as m
    return m


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype,r,sk", [(torch.bfloat16, 3, 5), (torch.float16, 7, 9), (torch.bfloat16, 11, 15),
                                        *[(torch.float32, *k) for k in ((3, 3), (3, 5), (5, 5), (5, 7), (6, 11), (7, 7), (7, 9), (11, 15))]])
def test_conv_attention_kernel_sizes(pkg, dtype, r, sk, d, causal):
    """Every compile-time kernel size of the fused kernels: one row, one key block, edges of the 118- to 128-row query
    blocks and 64-key blocks."""
    for s in (1, 63, 121, 130, 257):
        print(f"conv_attention {dtype} {r}x{sk} d={d} s={s} causal={causal}", flush=True)
        q, k, v = O.seeded_qkv(1, 2, s, d, dtype, seed=43)
        w = O.seeded_conv_weight(2, r, sk, 0.05, dtype)
        want = O.conv_attention_forward(q, k, v, w, causal, None)
        got = pkg.ops.conv_attn_fwd(q.cuda(), k.cuda(), v.cuda(), w.cuda(), causal, None).cpu()
        torch.testing.assert_close(got.float(), want.float(), **tol(dtype))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("c,group", [(32, None), (64, 32)])
@pytest.mark.parametrize("q", [4, 60, 256, 260, 508, 512, 516])
def test_headmix_fp32_32_heads_short_rows(pkg, q, c, group, causal):
    """fp32 mixing of 32 heads around the row lengths where the lanes' share changes, forward and input gradient, against 64 bits: 32 products
    and sums of values around 1, each within 2^-24 of the running sum: 32 * 2^-24 * sqrt(32) < 2e-5."""
    print(f"headmix fp32 q={q} c={c} group={group} causal={causal}", flush=True)
    torch.manual_seed(3)
    x, w = torch.randn(2, c, q, q), torch.randn(c, c)
    if group:
        block = torch.arange(c) // group
        w = w * (block[:, None] == block[None, :])
    keep = torch.ones(q, q).tril() if causal else torch.ones(q, q)
    for fn, m in ((pkg.ops.headmix, w), (pkg.ops.headmix_bwd_input, w.t())):
        want = torch.einsum("oi,nipq->nopq", m.double(), x.double()) * keep
        got = fn(x.cuda(), w.cuda(), causal, group_size=group).cpu()
        torch.testing.assert_close(got.double(), want, rtol=0, atol=2e-5)


@pytest.mark.parametrize("b,h,s,d,r,sk", [
    (1, 3, 64, 128, 6, 11), (1, 2, 65, 128, 3, 3), (2, 3, 129, 64, 11, 15), (1, 2, 200, 64, 3, 5), (2, 2, 257, 64, 5, 7),   # whole and ragged lengths
    (3, 4, 2300, 64, 7, 9),      # all at once (256 MB)
    (5, 4, 2300, 64, 7, 9),      # the batch entries in turns, three and two
    (2, 5, 4104, 128, 5, 5),     # the heads of a batch entry in turns, a last part that is smaller
])
@pytest.mark.parametrize("factor", [None, -0.3])
def test_conv_attention_fp32_stages(pkg, b, h, s, d, r, sk, factor):
    """fp32 conv-attention of sizes that take scores, conv, softmax and P V one after the other, against the fused kernel (which writes the
    row statistic), which the tests above hold against the oracle: the two orders of sums differ by a few 2^-24 of the scores, whose
    exponentials turn that into relative errors; both 2-norms are below 5e-7."""
    print(f"conv_attention stages b={b} h={h} s={s} d={d} {r}x{sk}", flush=True)
    assert pkg._lib.load().mta_conv_attn_in_stages(b, h, s, d, r, sk, 1, 0) == 1
    q, k, v = (x.cuda() for x in O.seeded_qkv(b, h, s, d, torch.float32, seed=47))
    module = pkg.TritonConvAttention(h, (r, sk), causal=True).cuda()
    with torch.no_grad():
        module.weight.copy_(O.seeded_conv_weight(h, r, sk, 0.05, torch.float32))
        got = module(q, k, v, True, factor)[0]
    want, _ = pkg.ops.conv_attn_fwd(q, k, v, module.weight.detach(), True, factor, return_lse=True)
    assert got.shape == want.shape and got.is_contiguous()
    assert ((got - want).double().norm() / want.double().norm()).item() < 2e-6
    torch.testing.assert_close(got, want, **tol(torch.float32))


@pytest.mark.parametrize("b,h,s", [(4, 16, 1024), (5, 4, 1500), (1, 4, 5792), (1, 2, 8192)])
def test_conv_attention_fp32_scratch(pkg, b, h, s):
    """What fp32 conv-attention in stages allocates beside its result: up to 512 MB in two or three tensors of scores (and padded operands where
    the length is ragged); and where that cannot be had, the fused kernel's result."""
    module = pkg.TritonConvAttention(h, (6, 11), causal=True).cuda()
    q, k, v = (x.cuda() for x in O.seeded_qkv(b, h, s, 64, torch.float32, seed=48))
    with torch.no_grad():
        torch.cuda.empty_cache()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        got = module(q, k, v, True, None)[0]
        beside = torch.cuda.max_memory_allocated() - before - (1 if s % 8 == 0 else 5) * q.numel() * 4
        assert s * s * 4 < beside <= 516 << 20
        del got
        torch.cuda.empty_cache()
        total, room, fill = torch.cuda.get_device_properties(0).total_memory, torch.cuda.memory_reserved(), []
        try:
            torch.cuda.set_per_process_memory_fraction(room / total)
            with pytest.raises(torch.OutOfMemoryError):   # (what is left free in the pool's segments)
                while len(fill) < 4096:
                    fill.append(torch.empty(16 << 20, dtype=torch.uint8, device="cuda"))
            torch.cuda.set_per_process_memory_fraction((room + 6 * q.numel() * 4 + (24 << 20)) / total)
            got = module(q, k, v, True, None)[0]
        finally:
            fill.clear()
            torch.cuda.set_per_process_memory_fraction(1.0)
    want, _ = pkg.ops.conv_attn_fwd(q, k, v, module.weight.detach(), True, None, return_lse=True)
    assert torch.equal(got, want)


@pytest.mark.parametrize("s", [512, 513])
def test_conv_attention_fp32_refuses(pkg, s):
    """fp32 conv-attention refuses the same calls where it runs in stages: operands that do not lie at whole 16-byte vectors, more than 65535
    planes."""
    module = pkg.TritonConvAttention(4, (6, 11), causal=True).cuda()
    ok = torch.zeros(1, 4, s, 64, device="cuda")
    off = torch.zeros(ok.numel() + 1, device="cuda")[1:].view_as(ok)
    many = torch.zeros(1, 65536, s, 64, device="cuda")
    with torch.no_grad():
        module(ok, ok, ok, True, None)
        for q, k, v in ((off, ok, ok), (ok, off, ok), (ok, ok, off)):
            with pytest.raises(ValueError):
                module(q, k, v, True, None)
        with pytest.raises(ValueError):
            pkg.TritonConvAttention(65536, (6, 11), causal=True).cuda()(many, many, many, True, None)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("factor", [-0.08, 0.0, 0.08])
@pytest.mark.parametrize("dtype,d,r,sk", [(torch.bfloat16, 128, 6, 11), (torch.float16, 64, 3, 3), (torch.float16, 128, 11, 15)])
def test_conv_attention_factor(pkg, dtype, d, r, sk, factor, causal):
    """Factors of either sign and 0 (the kernel's maxima are taken ahead of the factor): one row, one 64-key block and its edges, the
    edge of a query block and rows that take more than one of them.  Output and row statistic against the oracle in fp32; bounds as for
    the default factor (test_conv_attention_lse), which is no smaller: the scores are rounded to 16 bits ahead of it."""
    for s in (1, 64, 65, 130, 200):
        print(f"conv_attention {dtype} {r}x{sk} d={d} s={s} factor={factor} causal={causal}", flush=True)
        q, k, v = O.seeded_qkv(1, 2, s, d, dtype, seed=44)
        w = O.seeded_conv_weight(2, r, sk, 0.05, dtype)
        scores = O.conv_attention_scores(q.float(), k.float(), w.float(), causal, 1.0)
        scores = torch.where(torch.isinf(scores), scores, scores * factor)   # (a key above the diagonal has no weight, whatever the factor)
        o, lse = pkg.ops.conv_attn_fwd(q.cuda(), k.cuda(), v.cuda(), w.cuda(), causal, factor, return_lse=True)
        want = torch.matmul(torch.softmax(scores, -1), v.float())
        torch.testing.assert_close(o.cpu().float(), want, **tol(dtype))
        torch.testing.assert_close(lse.cpu(), torch.logsumexp(scores, -1), rtol=2.0 ** -7, atol=2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("h,d", [(1, 64), (20, 64), (1, 128), (20, 128)])
def test_conv_attention_sums_do_not_drift(pkg, h, d, dtype):
    """128 key blocks of equal logits, 772, whose product with log2(e) is rounded by a unit of 6e-5: a row's sum stays the number of its
    keys, and its first and its last block weigh the same.  Bound: the statistic's own rounding, 2^-14 at 772, and one of the logarithm.
    Eight wavefronts of 16 rows (one head) and four of 32."""
    s = 8192
    q, k, v = (torch.zeros(1, h, s, d, dtype=dtype, device="cuda") for _ in range(3))
    q[..., 0], k[..., 0], k[..., 1], q[..., 1] = 27.75, 27.75, 1.0, 1.9375   # (27.75^2 + 1.9375 = 772)
    v[:, :, :64, 0] = v[:, :, -64:, 1] = 64.0
    w = torch.zeros(h, 3, 3, dtype=dtype, device="cuda")
    w[:, -1, 1] = 1.0
    o, lse = pkg.ops.conv_attn_fwd(q, k, v, w, True, 1.0, return_lse=True)
    want = 772.0 + torch.log(torch.arange(1, s + 1, dtype=torch.float64, device="cuda"))
    assert (lse.double() - want).abs().max().item() <= 2.0 ** -13
    assert torch.equal(o[:, :, -1, 0], o[:, :, -1, 1])


@pytest.mark.parametrize("dtype,r,sk", [(torch.bfloat16, 3, 5), (torch.float16, 7, 9)])
def test_qk_conv_kernel_sizes(pkg, dtype, r, sk):
    """The scores stage at the same sizes; bound as in test_qk_conv_parity: two 16-bit roundings of scores of magnitude
    sqrt(d)*|w|, i.e. 2 ulp + atol."""
    for s, d in ((8, 64), (120, 128), (264, 64), (1032, 128)):
        print(f"qk_conv {dtype} {r}x{sk} d={d} s={s}", flush=True)
        q, k, _ = O.seeded_qkv(1, 2, s, d, dtype, seed=7)
        w = O.seeded_conv_weight(2, r, sk, 0.05, dtype)
        scale = float(torch.rsqrt(torch.tensor(float(d))))
        want = O.depthwise_conv(torch.tril(torch.matmul(q, k.transpose(2, 3)) * torch.rsqrt(torch.tensor(d))), w, True)
        got = pkg.ops.qk_conv(q.cuda(), k.cuda(), w.cuda(), True, scale).cpu()
        ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
        torch.testing.assert_close(got.float(), want.float(), rtol=2 * ulp, atol=2e-2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_narrow_products(pkg, d, dtype):
    """P V and P^T X on the narrow kernels (small grids): one row, edges of the 32-row blocks and of the steps that the four
    wavefronts share, NaN above the diagonal.  Against the fp32 product of the same 16-bit values; what differs is the order
    of at most 264 fp32 sums and one rounding of a result of magnitude at most sqrt(264)."""
    g = torch.Generator().manual_seed(11)
    for s in (8, 32, 40, 136, 264):
        print(f"narrow products {dtype} d={d} s={s}", flush=True)
        p = torch.randn(2, 3, s, s, generator=g).to(dtype)
        x = torch.randn(2, 3, s, d, generator=g).to(dtype)
        low = torch.tril(torch.ones(s, s, dtype=torch.bool))
        poisoned = p.masked_fill(~low, float("nan")).cuda()
        lower = p.float().masked_fill(~low, 0.0)
        ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
        for got, want in ((pkg.ops.causal_pv(poisoned, x.cuda(), True), lower @ x.float()),
                          (pkg.ops.causal_ptx(poisoned, x.cuda(), True), lower.transpose(2, 3) @ x.float()),
                          (pkg.ops.causal_pv(p.cuda(), x.cuda(), False), p.float() @ x.float()),
                          (pkg.ops.causal_ptx(p.cuda(), x.cuda(), False), p.float().transpose(2, 3) @ x.float())):
            torch.testing.assert_close(got.float().cpu(), want, rtol=ulp * 1.01, atol=1e-4)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c", [3, 5, 12, 17, 32])
def test_headmix_weight_gradient_head_counts(pkg, c, dtype):
    """dW on the matrix cores for head counts that do not fill the operand rows (sets of 4 or 8 heads, blocks of 16), rows of
    whole 16-byte vectors and ragged ones (whose last vectors reach the end of the tensor), NaN above the diagonal.  Against
    the double-precision sum of the same values: fp32 sums of n products are off by at most n*2^-24 of the sum of their
    magnitudes in the worst order, far less in this one; sqrt(n)*2^-22 covers it."""
    g = torch.Generator().manual_seed(5)
    for p, q, causal in ((8, 8, True), (33, 65, False), (97, 97, True), (200, 200, True), (64, 1032, False)):
        print(f"headmix dW c={c} {p}x{q} causal={causal} {dtype}", flush=True)
        x, dy = (torch.randn(2, c, p, q, generator=g).to(dtype) for _ in range(2))
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        xd, dyd = (t.double().masked_fill(~keep, 0.0) for t in (x, dy))
        want = torch.einsum("nopq,nipq->oi", dyd, xd)
        size = torch.einsum("nopq,nipq->oi", dyd.abs(), xd.abs())
        got = pkg.ops.headmix_bwd_weight(x.masked_fill(~keep, float("nan")).cuda(), dy.masked_fill(~keep, float("nan")).cuda(), causal)
        bound = (2 * p * q) ** 0.5 * 2.0 ** -22 * size
        assert ((got.cpu().double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("transposed", [False, True])
def test_headmix_twelve_heads(pkg, transposed, dtype):
    """12 heads mixed densely, alone and as two groups of 24 heads, whole vectors and ragged rows, forward and input gradient;
    one rounding of an fp32 sum of 12 products of magnitude at most 1.5 each (fp32: the order of that sum)."""
    g = torch.Generator().manual_seed(6)
    for c, group, p, q, causal in ((12, None, 40, 40, True), (12, None, 33, 1032, False), (24, 12, 72, 72, True), (12, None, 51, 51, True)):
        print(f"headmix 12 heads c={c} {p}x{q} {dtype}", flush=True)
        x = torch.randn(2, c, p, q, generator=g).to(dtype)
        w = (O.block_diag_head_weight(c, 12, 0.3, g, dtype) if group else torch.eye(c) + 0.3 * torch.randn(c, c, generator=g)).to(dtype)
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        m = w.double().t() if transposed else w.double()
        want = torch.einsum("oi,nipq->nopq", m, x.double().masked_fill(~keep, 0.0))
        xd = x.masked_fill(~keep, float("nan")).cuda()
        got = (pkg.ops.headmix_bwd_input(xd, w.cuda(), causal, group_size=group) if transposed
               else pkg.ops.headmix(xd, w.cuda(), causal, 0.0, group_size=group))
        ulp = {torch.float32: 2.0 ** -21, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
        torch.testing.assert_close(got.double().cpu(), want.masked_fill(~keep, 0.0), rtol=ulp, atol=1e-5)


def _mta(pkg, h, ks, ks2, dtype, seed, use_mask=False, structure=None):
    g = torch.Generator().manual_seed(seed)
    cfg = pkg.MTAConfig(query_kernel_size=ks[0], key_kernel_size=ks[1], after_sm_query_kernel_size=ks2[0], after_sm_key_kernel_size=ks2[1])
    mod = pkg.MTAAttentionTriton(h, cfg, dropout=0.0, causal=True, use_mask=use_mask)
    params = [O.seeded_conv_weight(h, *ks, 0.05, dtype, seed=seed), (torch.eye(h) + 0.1 * torch.randn(h, h, generator=g)).to(dtype),
              O.seeded_conv_weight(h, *ks2, 0.05, dtype, seed=seed + 1), (torch.eye(h) + 0.1 * torch.randn(h, h, generator=g)).to(dtype)]
    with torch.no_grad():
        for p, w in zip((mod.mta_conv_triton, mod.wpsm_triton, mod.mta_conv_after_sm_triton, mod.wposm_triton), params):
            p.weight.copy_(w)
    return mod.to(dtype).cuda(), params


def _ragged_mask(kind, b, s):
    rows = torch.arange(s)
    causal = rows[None, :] <= rows[:, None]
    if kind == "window":
        return (causal & (rows[None, :] > rows[:, None] - max(1, s // 3)))[None, None]
    if kind == "padding":
        lengths = torch.tensor([s - 3 * i for i in range(b)]).clamp(min=1)
        return (causal[None] & (rows[None, None, :] < lengths[:, None, None]))[:, None]
    return None


@pytest.mark.parametrize("kind", ["none", "padding", "window"])
@pytest.mark.parametrize("dtype,h,s,d", [(torch.bfloat16, 4, 33, 64), (torch.float16, 16, 129, 128), (torch.bfloat16, 12, 68, 64),
                                         (torch.float32, 8, 61, 64), (torch.bfloat16, 8, 1, 64), (torch.float16, 16, 7, 64)])
def test_mta_padded_lengths(pkg, dtype, h, s, d, kind):
    """Causal lengths that are not a multiple of 8 run padded with zero rows: output and all seven gradients, without a mask,
    under key padding and under a window, against the oracle (given the mask tensor)."""
    print(f"mta padded length {dtype} h={h} s={s} d={d} {kind}", flush=True)
    b = 2
    mod, params = _mta(pkg, h, (5, 5), (3, 3), dtype, 51, use_mask=kind != "none")
    mask = _ragged_mask(kind, b, s)
    q, k, v = O.seeded_qkv(b, h, s, d, dtype, seed=52)
    go = torch.randn(b, s, h, d, generator=torch.Generator().manual_seed(53)).to(dtype)
    leaves = [t.clone().float().requires_grad_(True) for t in (q, k, v)]
    wl = [p.clone().float().requires_grad_(True) for p in params]
    am = None if mask is None else torch.where(mask, 0.0, float("-inf"))
    want = O.mta_forward(*leaves, wl[0].unsqueeze(1), wl[1], wl[2].unsqueeze(1), wl[3], mask=am)
    want.backward(go.float())
    dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    gmask = None if mask is None else mask.cuda()
    with torch.no_grad():
        plain = mod(*dev, gmask, None)
    out = mod(*dev, gmask, None)
    out.backward(go.cuda())
    assert out.shape == (b, s, h, d) and plain.shape == out.shape
    # the forward against the oracle in the data's own dtype, which rounds where the kernels round: what is left is one ulp
    # of the 16-bit format here and there (head mixing makes |out| a little larger than the convex combinations of tol())
    want16 = O.mta_forward(q, k, v, params[0].unsqueeze(1), params[1], params[2].unsqueeze(1), params[3],
                           mask=None if am is None else am.to(dtype)).float()
    bound = tol(dtype) if dtype == torch.float32 else dict(rtol=2.0 ** (-7 if dtype == torch.bfloat16 else -10), atol=2e-2)
    torch.testing.assert_close(plain.float().cpu(), want16, **bound)
    torch.testing.assert_close(out.detach().float().cpu(), want16, **bound)
    # gradients in the norm: a chain of about eight roundings of relative size 2^-9 (bf16) / 2^-12 (fp16), times the
    # cancellation in softmax backward; fp32: sums in another order
    rel = {torch.float32: 1e-4, torch.bfloat16: 4e-2, torch.float16: 1e-2}[dtype]
    got = [t.grad for t in dev] + [m.weight.grad for m in (mod.mta_conv_triton, mod.wpsm_triton, mod.mta_conv_after_sm_triton, mod.wposm_triton)]
    for name, a, w in zip("q k v conv pre conv2 post".split(), got, [t.grad for t in leaves + wl]):
        assert torch.isfinite(a.float()).all(), name
        assert float((a.float().cpu() - w).norm()) <= rel * float(w.norm()) + 1e-5, name


@pytest.mark.parametrize("d", [64, 128])
def test_fp32_lower_products(pkg, d):
    """The three fp32 products on the lower triangle: one vector of rows, edges of the tiles (32 / 64 rows, 64 / 128 keys) and
    of the steps the wavefronts share, NaN above the diagonal.  fp32 sums of n products against double precision: at most
    sqrt(n) * 2^-22 of the sum of the products' magnitudes."""
    lib, st = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(12)
    for s in (4, 32, 36, 64, 100, 128, 196, 260, 516):
        print(f"fp32 products d={d} s={s}", flush=True)
        b, h = 2, 3
        p = torch.randn(b, h, s, s, generator=g)
        x, y = torch.randn(b, h, s, d, generator=g), torch.randn(b, h, s, d, generator=g)
        low = torch.tril(torch.ones(s, s, dtype=torch.bool))
        pd = p.masked_fill(~low, float("nan")).cuda()
        lower = p.double().masked_fill(~low, 0.0)
        xd, yd, out = x.cuda(), y.cuda(), torch.full((b, h, s, d), float("nan"), device="cuda")

        def close(got, want, size, n):
            assert ((got.double().cpu() - want).abs() <= n ** 0.5 * 2.0 ** -22 * size + 1e-30).all()

        assert lib.mta_causal_pv_f32(pd.data_ptr(), xd.data_ptr(), out.data_ptr(), b, h, s, d, 0.5, st) == 0
        close(out, 0.5 * (lower @ x.double()), 0.5 * (lower.abs() @ x.double().abs()), s)
        assert lib.mta_causal_ptx_f32(pd.data_ptr(), xd.data_ptr(), out.data_ptr(), b, h, s, d, 0.5, st) == 0
        close(out, 0.5 * (lower.transpose(2, 3) @ x.double()), 0.5 * (lower.abs().transpose(2, 3) @ x.double().abs()), s)
        scores = torch.full((b, h, s, s), 7.0, device="cuda")
        assert lib.mta_lower_scores_f32(xd.data_ptr(), yd.data_ptr(), scores.data_ptr(), b, h, s, d, st) == 0
        close(scores[..., low.cuda()], (x.double() @ y.double().transpose(2, 3))[..., low], (x.double().abs() @ y.double().abs().transpose(2, 3))[..., low], d)
        up = scores.cpu()[..., ~low]
        assert ((up == 7.0) | (up == 0.0)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_lower_scores_without_conv(pkg, d, dtype):
    """round(a b^T) on and below the diagonal: one vector of rows, edges of the 128-row and 64-key blocks, lengths cut into
    several work items.  Exact for small integers, whose products and sums fp32 and the 16-bit type (up to 2^8) hold."""
    g = torch.Generator().manual_seed(13)
    for s in (8, 64, 72, 128, 200, 264, 1160):
        print(f"lower scores d={d} s={s} {dtype}", flush=True)
        a, c = (torch.zeros(1, 2, s, d) for _ in range(2))
        a[..., :8] = torch.randint(-2, 3, (1, 2, s, 8), generator=g).float()
        c[..., :8] = torch.randint(-2, 3, (1, 2, s, 8), generator=g).float()
        got = pkg.ops.lower_scores(a.to(dtype).cuda(), c.to(dtype).cuda()).cpu()
        low = torch.tril(torch.ones(s, s, dtype=torch.bool))
        assert torch.equal(got[..., low].float(), (a @ c.transpose(2, 3))[..., low])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,h,s", [(1, 9, 3080), (3, 5, 3080), (1, 12, 4088), (1, 9, 3072), (1, 16, 3080)])
def test_lower_scores_of_ragged_rows(pkg, b, h, s, dtype):
    """Raw scores of 3072 to 4096 keys and heads that do not divide among the XCDs, whose items go out head by head where the rows are no
    whole lines: the bits of each head alone, with a band mask too; nothing missing and nothing else on and below the diagonal."""
    g = torch.Generator(device="cuda").manual_seed(77)
    a, c = (torch.randn(b, h, s, 64, generator=g, device="cuda").to(dtype) for _ in range(2))
    low = torch.ones(s, s, dtype=torch.bool, device="cuda").tril()
    first = (torch.arange(s, device="cuda") - 700).clamp(min=0).to(torch.int32).expand(b, s).contiguous()
    for band in (None, first):
        got = pkg.ops.lower_scores(a, c, band)
        for i in range(b):
            for j in range(h):
                alone = pkg.ops.lower_scores(a[i:i + 1, j:j + 1], c[i:i + 1, j:j + 1], None if band is None else band[i:i + 1])
                inside = low if band is None else low & (torch.arange(s, device="cuda")[None] >= first[0][:, None])
                assert torch.equal(got[i, j][inside], alone[0, 0][inside]), (i, j)


@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("r,sk", [(3, 3), (3, 5), (5, 5), (5, 7), (6, 11), (7, 7), (7, 9), (11, 15)])
def test_row_sliding_conv(pkg, r, sk, dtype, wdtype):
    """The row-sliding conv kernels, forward / scaled / input gradient / kernel gradient: widths below a window and with every
    remainder modulo 4, edges of the 64-key and 64- / 128-row wavefront tiles, non-square planes, NaN above the diagonal.
    Against double precision: R*S (or N*P*Q) fp32 sums, one rounding to the data type (16-bit: also of the scaled input)."""
    g = torch.Generator().manual_seed(31)
    io = {torch.float32: 2.0 ** -22, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for p, q, causal in ((4, 4, True), (5, 7, False), (65, 65, True), (66, 70, False), (131, 131, True), (140, 140, True), (33, 259, False)):
        if dtype == torch.float16 and q % 8 == 0:
            continue   # (rows of whole vectors: the matrix-core kernels)
        print(f"rows conv {r}x{sk} {p}x{q} causal={causal} {dtype}/{wdtype}", flush=True)
        x, dy = (torch.randn(2, 3, p, q, generator=g).to(dtype) for _ in range(2))
        w = (0.2 * torch.randn(3, r, sk, generator=g)).to(wdtype)
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        xd, dyd = (t.double().masked_fill(~keep, 0.0) for t in (x, dy))
        xg, dyg = (t.masked_fill(~keep, float("nan")).cuda() for t in (x, dy))

        def conv(a):
            pad = torch.nn.functional.pad(a, ((sk - 1) // 2, sk - 1 - (sk - 1) // 2, r - 1, 0))
            return torch.nn.functional.conv2d(pad, w.double().unsqueeze(1), groups=3).masked_fill(~keep, 0.0)

        xa = xd.clone().requires_grad_(True)
        conv(xa).backward(dyd)
        wa = w.double().requires_grad_(True)
        pad = torch.nn.functional.pad(xd, ((sk - 1) // 2, sk - 1 - (sk - 1) // 2, r - 1, 0))
        torch.nn.functional.conv2d(pad, wa.unsqueeze(1), groups=3).backward(dyd)
        size = float(r * sk) ** 0.5 * 0.2 * 4          # of a sum of R*S products
        for got, want in ((pkg.ops.conv2d_causal(xg, w.cuda(), causal), conv(xd)),
                          (pkg.ops.conv2d_causal(xg, w.cuda(), causal, in_scale=0.125), conv((x.float() * 0.125).to(dtype).double().masked_fill(~keep, 0.0))),
                          (pkg.ops.conv2d_bwd_input(dyg, w.cuda(), causal), xa.grad.masked_fill(~keep, 0.0))):
            torch.testing.assert_close(got.double().cpu(), want, rtol=io, atol=size * 2.0 ** -21)
        dw = pkg.ops.conv2d_bwd_weight(xg, dyg, (r, sk), causal).double().cpu()
        assert float((dw - wa.grad).abs().max()) <= (2 * p * q) ** 0.5 * 2.0 ** -19 * 16


@pytest.mark.parametrize("dtype,wdtype,h,s,d,kernel", [(torch.float32, torch.float32, 4, 65, 64, (5, 5)), (torch.float32, torch.float32, 16, 132, 128, (7, 9)),
                                                       (torch.bfloat16, torch.float32, 8, 73, 64, (3, 3)), (torch.float16, torch.float32, 12, 200, 128, (6, 11))])
@pytest.mark.parametrize("kind", ["window", "left"])
def test_mta_band_mask_two_kernel_first_stage(pkg, dtype, wdtype, h, s, d, kernel, kind):
    """Band masks where the scores and their conv are two kernels (fp32 data; weights of another dtype): no mask pass over the
    scores, output and all seven gradients against the oracle given the mask tensor (left: a batch entry whose first rows see
    nothing, forward only - the reference's gradients are NaN there)."""
    print(f"band mask two kernels {dtype} {wdtype} h={h} s={s} d={d} {kernel} {kind}", flush=True)
    b = 2
    mod, params = _mta(pkg, h, kernel, (3, 3), wdtype, 61, use_mask=True)
    rows = torch.arange(s)
    causal = rows[None, :] <= rows[:, None]
    mask = _ragged_mask("window", b, s)
    if kind == "left":
        keep = rows[None, :] >= torch.tensor([0, s // 3])[:, None]
        mask = (keep[:, None, :] & keep[:, :, None] & causal)[:, None]
    q, k, v = O.seeded_qkv(b, h, s, d, dtype, seed=62)
    go = torch.randn(b, s, h, d, generator=torch.Generator().manual_seed(63)).to(dtype)
    leaves = [t.clone().float().requires_grad_(True) for t in (q, k, v)]
    wl = [p.clone().float().requires_grad_(True) for p in params]
    want = O.mta_forward(*leaves, wl[0].unsqueeze(1), wl[1], wl[2].unsqueeze(1), wl[3], mask=torch.where(mask, 0.0, float("-inf")).expand(b, h, s, s))
    dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    stages = []
    mod._stage_hook = stages.append
    with torch.no_grad():
        plain = mod(*dev, mask.cuda(), None)
    out = mod(*dev, mask.cuda(), None)
    assert "mask" not in stages and stages.count("pv") == 2, stages
    # the oracle computes in fp32 throughout: a chain of about six roundings to the data type (2^-9 / 2^-12 each) in the norm
    rel = {torch.float32: 1e-5, torch.bfloat16: 1.5e-2, torch.float16: 2e-3}[dtype]
    for got in (plain, out.detach()):
        assert float((got.float().cpu() - want.detach()).norm()) <= rel * float(want.detach().norm())
    if kind == "left":
        assert not out[1, :s // 3].any()
        return
    want.backward(go.float())
    out.backward(go.cuda())
    rel = {torch.float32: 1e-4, torch.bfloat16: 4e-2, torch.float16: 1e-2}[dtype]   # (as in test_mta_padded_lengths)
    got = [t.grad for t in dev] + [m.weight.grad for m in (mod.mta_conv_triton, mod.wpsm_triton, mod.mta_conv_after_sm_triton, mod.wposm_triton)]
    for name, a, w in zip("q k v conv pre conv2 post".split(), got, [t.grad for t in leaves + wl]):
        assert torch.isfinite(a.float()).all(), name
        assert float((a.float().cpu() - w).norm()) <= rel * float(w.norm()) + 1e-5, name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_headmix_twelve_heads_infinity(pkg, dtype):
    """An infinite score of one head and key: the output heads hold +-inf there (w has no zeros), as the sum of 12 products
    does - not NaN, which an operand row without a head would make of it (0 * inf)."""
    g = torch.Generator().manual_seed(8)
    x, w = torch.randn(1, 12, 16, 16, generator=g).to(dtype), (torch.rand(12, 12, generator=g) + 0.5).to(dtype)
    x[0, 0, 9, 4] = float("inf")
    got = pkg.ops.headmix(x.cuda(), w.cuda(), True, 0.0).cpu()
    assert (got[0, :, 9, 4] == float("inf")).all()
    assert torch.isfinite(got[0, :, 9, [0, 3, 5]]).all() and torch.isfinite(got[0, :, 8]).all()


@pytest.mark.parametrize("masked", [None, "bias", "band"])
@pytest.mark.parametrize("h", [9, 12, 16, 32])
def test_fp32_dense_mix_softmax_mix(pkg, h, masked):
    """mix -> softmax -> mix of fp32 scores in dense groups, with either weight, both or a bf16 one: lengths around the edges of
    the 64-key passes and of every instance, non-causal rows, a key bias that hides keys, a band mask.  Against float64: a
    score's sum is off by at most h * 2^-24 * 4, which the exponential turns into a relative error of its own size (< 1e-5)."""
    g = torch.Generator().manual_seed(22)
    longest = 4096 if h <= 16 else 2048
    for p, q, causal in ((1, 4, True), (64, 64, True), (132, 132, True), (260, 260, True), (7, 516, False), (3, 1028, False), (2, longest, False)):
        if masked == "band" and not causal:
            continue
        print(f"fp32 dense softmax h={h} {p}x{q} causal={causal} {masked}", flush=True)
        n, c = (2, 2 * h) if p < 200 else (1, h)
        x = 2.0 * torch.randn(n, c, p, q, generator=g)
        keep = (torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)).expand(n, 1, p, q)
        first, bias = None, None
        if masked == "band":
            first = (torch.arange(p).expand(n, p) - torch.tensor([[5], [70]])[:n]).clamp(min=0).to(torch.int32)
            keep = keep & (torch.arange(q) >= first[:, None, :, None])
        if masked == "bias":
            bias = torch.randn(n, q, generator=g)
            bias[:, q // 2:q // 2 + 2] = float("-inf")
            bias[:, 0] = 0.5   # (every row sees a key)
        weights = [torch.block_diag(*[torch.eye(h) + 0.2 * torch.randn(h, h, generator=g) for _ in range(c // h)]) for _ in range(2)]
        below = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        xd = x.masked_fill(~below, float("nan")).cuda()
        for one, two, wdtype in ((True, False, torch.float32), (False, True, torch.float32), (True, True, torch.float32), (True, True, torch.bfloat16)):
            w1, w2 = (w.to(wdtype) if use else None for w, use in zip(weights, (one, two)))
            s = x.double().masked_fill(~keep, 0.0)
            if one:
                s = torch.einsum("oi,nipq->nopq", w1.double(), s)
            if bias is not None:
                s = s + bias.double()[:, None, None, :]
            s = torch.softmax(s.masked_fill(~keep, float("-inf")), -1)
            if two:
                s = torch.einsum("oi,nipq->nopq", w2.double(), s)
            got = pkg.ops.headmix_softmax(xd, None if w1 is None else w1.cuda(), None if w2 is None else w2.cuda(), causal, group_size=h,
                                          key_bias=None if bias is None else bias.cuda(), first_visible=None if first is None else first.cuda())
            torch.testing.assert_close(got.double().cpu(), s, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("masked", ["", "bias", "band"])
def test_softmax_of_8_heads_long_rows(pkg, masked, dtype):
    """Groups of 8 beyond 2048 keys (16 bits: one pass of 8 wavefronts, up to 4096; fp32: three passes, up to 3072, or 8 wavefronts), and what lies
    beyond; 16 bits also groups of 2 with a band.  Whole numbers in x and the first weight: their mixed scores are exact in every type.
    What is left, in halves of an ulp (2^-8 in bf16, 2^-11 in fp16): two where a probability near a tie is rounded the other way, and one for the
    result, of sum |w2| p each; fp32: exp2 of an argument of up to 64 log2(e), 92 ulp of 2^-24 of it, and the sums."""
    g = torch.Generator().manual_seed(61)
    half = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -18}[dtype]
    lengths = {torch.float32: (2052, 3072, 3076)}.get(dtype, (2056,))
    shapes = [(s, s, True) for s in lengths[:2]] + ([] if masked == "band" else [(2, s, False) for s in (*lengths, 4096, 4104)])
    for group in (8, 2) if dtype != torch.float32 and masked == "band" else (8,):
        for p, q, causal in shapes:
            print(f"softmax of {group} heads {p}x{q} causal={causal} {masked} {dtype}", flush=True)
            x = torch.randint(-2, 3, (1, group, p, q), generator=g).cuda()
            at = torch.arange(q, device="cuda")
            keep = (at <= torch.arange(p, device="cuda")[:, None] if causal else torch.ones(p, q, dtype=torch.bool, device="cuda"))[None, None]
            first = bias = None
            if masked == "band":
                first = (torch.arange(p, device="cuda") - 700).clamp(min=0)[None].to(torch.int32)
                first[0, 2050:] = 2049 - 5   # a visible stretch that starts in the last of the slices of 512 keys
                keep = keep & (at >= first[:, None, :, None])
            if masked == "bias":
                bias = torch.randint(-3, 2, (1, q), generator=g).float().cuda()
                bias[0, 1:q // 2] = float("-inf")
            w1 = torch.randint(-1, 2, (group, group), generator=g).cuda()
            w2 = (torch.eye(group) + 0.1 * torch.randn(group, group, generator=g)).to(dtype).cuda()
            below = at <= torch.arange(p, device="cuda")[:, None] if causal else torch.ones(p, q, dtype=torch.bool, device="cuda")
            xd = x.to(dtype).masked_fill(~below, float("nan"))
            for one, two in ((True, False), (False, True), (True, True)):
                s = torch.einsum("oi,nipq->nopq", w1.double(), x.double()) if one else x.double()
                if bias is not None:
                    s = s + bias.double()[:, None, None, :]
                want = torch.softmax(s.masked_fill(~keep, float("-inf")), -1).to(dtype).double()
                size = want
                if two:
                    size = torch.einsum("oi,nipq->nopq", w2.double().abs(), want)
                    want = torch.einsum("oi,nipq->nopq", w2.double(), want)
                got = pkg.ops.headmix_softmax(xd, w1.to(dtype) if one else None, w2 if two else None, causal, group_size=group, key_bias=bias, first_visible=first)
                least = 2.0 ** -23 if dtype == torch.float16 else 1e-30   # (probabilities that are subnormal in fp16)
                assert ((got.double() - want).abs() <= 3 * half * size + group * least).all(), (one, two)


def test_fp32_softmax_gradient_sizes(pkg):
    """fp32 rows in registers (up to 8192 keys of whole vectors) and in two sweeps: edges of the instances, NaN above the
    diagonal.  Against float64: the order of the row's sum of p * dp, sum of |p * dp| at most about 4."""
    g = torch.Generator().manual_seed(23)
    for p, q, causal in ((1, 4, True), (68, 68, True), (67, 67, True), (3, 1024, False), (3, 1028, False), (2, 2052, False), (2, 4100, False), (2, 8192, False), (2, 8196, False)):
        print(f"fp32 softmax gradient {p}x{q} causal={causal}", flush=True)
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        prob = torch.softmax(torch.randn(2, 3, p, q, generator=g).masked_fill(~keep, float("-inf")), -1)
        dp = torch.randn(2, 3, p, q, generator=g)
        pd, gd = prob.double(), dp.double().masked_fill(~keep, 0.0)
        want = pd * (gd - (pd * gd).sum(-1, keepdim=True))
        got = pkg.ops.softmax_bwd(prob.masked_fill(~keep, float("nan")).cuda(), dp.masked_fill(~keep, float("nan")).cuda(), causal)
        torch.testing.assert_close(got.double().cpu(), want, rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ks", [3, 5, 7])
def test_conv_mix16_one_or_two_kernels(pkg, ks, dtype):
    """Post-softmax conv and dense mixing of 16 heads: the one-kernel form and the two kernels that small grids take hold the same
    rounding points and the same products; what differs is the order of fp32 sums, i.e. one rounding of the conv result and one
    of an output of magnitude at most about 8."""
    g = torch.Generator().manual_seed(31)
    for n, c, s in ((1, 16, 8), (1, 16, 72), (2, 32, 136)):
        print(f"conv mix16 {dtype} {ks}x{ks} n={n} c={c} s={s}", flush=True)
        x = torch.rand(n, c, s, s, generator=g).to(dtype).cuda()
        wc = O.seeded_conv_weight(c, ks, ks, 0.1, dtype).cuda()
        wm = torch.block_diag(*[torch.eye(16) + 0.1 * torch.randn(16, 16, generator=g) for _ in range(c // 16)]).to(dtype).cuda()
        one = pkg.ops.conv2d_headmix(x, wc, wm, True, group_size=16)
        two = pkg.ops.headmix(pkg.ops.conv2d_causal(x, wc, True), wm, True, 0.0, group_size=16)
        ulp = 2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10
        torch.testing.assert_close(one.float(), two.float(), rtol=ulp, atol=4 * ulp)


def _unit(dtype):
    return {torch.float32: 2.0 ** -22, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,group", [(2, 0), (4, 0), (8, 0), (12, 0), (16, 0), (32, 0), (16, 2), (8, 4), (24, 12), (32, 16), (16, 8)])
def test_headmix_both_gradients(pkg, c, group, dtype):
    """The head mixing's two gradients in one pass, at edges of its tiles (vectors, 64 or 128 keys, 256 or 512) and with NaN above the
    diagonal.  Against float64: dx is one rounding of an fp32 sum of at most 32 products; dw fp32 sums of n products in an order
    whose error sqrt(n)*2^-22 of the sum of magnitudes covers."""
    g = torch.Generator().manual_seed(41)
    half_step = 2.0 ** -25 if dtype == torch.float16 else 0.0   # (rounding of a subnormal result)
    for p, q, mode in ((1, 8, "fill"), (8, 8, "lower"), (72, 72, "fill"), (65, 136, "all"), (136, 136, "lower"), (200, 520, "fill"), (33, 1032, "all"),
                       (264, 264, "lower")):
        print(f"headmix gradients c={c} group={group} {p}x{q} {mode} {dtype}", flush=True)
        causal, n = mode != "all", 3 if p == 65 else 2
        x, dy = (torch.randn(n, c, p, q, generator=g).to(dtype) for _ in range(2))
        w = (torch.eye(c) + 0.3 * torch.randn(c, c, generator=g)).to(dtype)
        block = torch.arange(c) // (group or c)
        same = block[:, None] == block[None, :]
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        xd, dyd, wd = x.double().masked_fill(~keep, 0.0), dy.double().masked_fill(~keep, 0.0), w.double() * same
        want = torch.einsum("oi,nopq->nipq", wd, dyd)
        want_w = torch.einsum("nopq,nipq->oi", dyd, xd) * same
        size_w = torch.einsum("nopq,nipq->oi", dyd.abs(), xd.abs())
        sent = torch.full(x.shape, 7.0, dtype=dtype, device="cuda")
        # (the entries of w outside its blocks are nobody's)
        dx, dw = pkg.ops.headmix_grads(dy.masked_fill(~keep, float("nan")).cuda(), x.masked_fill(~keep, float("nan")).cuda(),
                                       w.masked_fill(~same, float("inf")).cuda(), causal, group_size=group, fill_upper=mode == "fill", out=sent)
        dx, dw = dx.cpu().double(), dw.cpu().double()
        assert ((dx - want).abs() <= _unit(dtype) * 1.01 * want.abs() + 2.0 ** -19 * torch.einsum("oi,nopq->nipq", wd.abs(), dyd.abs()) + half_step)[..., keep].all()
        if mode == "fill":
            assert (dx[..., ~keep] == 0.0).all()
        assert ((dw - want_w).abs() <= _unit(dtype) * want_w.abs() + (n * p * q) ** 0.5 * 2.0 ** -22 * size_w + half_step).all()


@pytest.mark.parametrize("parts", [1, 15, 16, 17, 255, 256, 257, 1023, 1025, 2048])
def test_sums_by_number_of_partial_results(pkg, parts):
    """One gradient and three of them at once, edges of a thread's share and of a round of loads; conv kernels (entries no multiple of
    16), a dense head weight, one of groups, one masked to them.  Against float64: fp32 sums of at most 2048 values of magnitude up to
    about 5 in shares of at most 33, then 18: 51 roundings of at most 2^-24 of the sum of magnitudes, and one of the result."""
    import ctypes
    lib, st, Partials = pkg._lib.load(), torch.cuda.current_stream().cuda_stream, pkg._lib.Partials
    g = torch.Generator(device="cuda").manual_seed(parts)
    blocks = lambda t: torch.block_diag(*t)   # noqa: E731
    jobs, want, size, dws = [], [], [], []
    same = torch.block_diag(*[torch.ones(4, 4, device="cuda")] * 3).double()
    for rows, entries, side, mask, n, dtype in ((3, 66, 0, 0, parts, torch.float32), (12, 16, 4, 0, parts, torch.bfloat16), (12, 144, 12, 4, max(1, parts // 3), torch.float16)):
        count = rows if side == 0 else rows // side
        p = torch.randn(count, n, entries, generator=g, device="cuda")
        exact, most = ((t.double().sum(1) * 0.5) for t in (p, p.abs()))
        if side:
            exact, most = (blocks(list(t.view(count, side, side))) for t in (exact, most))
        if mask:
            exact, most = exact * same, most * same
        dw = torch.full(exact.shape, 7.0, dtype=dtype, device="cuda")
        jobs.append((p, Partials(p.data_ptr(), dw.data_ptr(), rows, entries, n, side, mask, {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype], 0.5)))
        want.append(exact), size.append(most), dws.append(dw)

    def check():
        for exact, most, dw in zip(want, size, dws):
            assert ((dw.double() - exact).abs() <= 51 * 2.0 ** -24 * most + _unit(dw.dtype) * 1.01 * exact.abs()).all()

    for i in range(3):
        assert lib.mta_sum_partials(1, ctypes.byref(jobs[i][1]), st) == 0
    check()
    alone = [dw.clone() for dw in dws]
    for dw in dws:
        dw.fill_(7.0)
    assert lib.mta_sum_partials(3, (Partials * 3)(*(j for _, j in jobs)), st) == 0
    check()
    if parts <= 256 or parts // 3 > 256:   # (else the three take 64 threads an entry and the last one alone 16)
        assert all(torch.equal(a, b) for a, b in zip(alone, dws))


@pytest.mark.parametrize("r,k", [(3, 3), (5, 5), (6, 11), (7, 7), (11, 15)])
@pytest.mark.parametrize("d", [64, 128])
def test_fp16_attention_by_grid(pkg, d, r, k):
    """fp16 attention of 600 workgroups, four wavefronts of 32 rows each, and, of the same heads, of 2 x 300, few enough for eight of 16: the
    same sums in the same order."""
    g = torch.Generator(device="cuda").manual_seed(59)
    q, kk, v = (torch.randn(1, 300, 136, d, generator=g, device="cuda").half() for _ in range(3))
    w = (0.1 * torch.randn(300, r, k, generator=g, device="cuda")).half()
    run = lambda lo, hi: pkg.ops.conv_attn_fwd(q[:, lo:hi].contiguous(), kk[:, lo:hi].contiguous(), v[:, lo:hi].contiguous(), w[lo:hi], True, d ** -0.5)   # noqa: E731
    first = lambda out: out[0] if isinstance(out, tuple) else out   # noqa: E731
    whole = first(run(0, 300))
    assert torch.isfinite(whole.float()).all()
    assert torch.equal(whole, torch.cat([first(run(0, 150)), first(run(150, 300))], 1))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("s", [8, 100, 396, 512])
def test_fp32_scores_by_tile(pkg, s, d):
    """fp32 scores of 8 heads on tiles of 64 x 128 (of few: 32 x 64), of 2 heads at a time on tiles of 32 x 64: the same sums in the same
    order, bit by bit, and nothing written above the diagonal beyond its vectors."""
    lib, st = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    a, b = (torch.randn(1, 8, s, d, device="cuda") for _ in range(2))
    whole, part = (torch.full((1, 8, s, s), 7.0, device="cuda") for _ in range(2))
    assert lib.mta_lower_scores_f32(a.data_ptr(), b.data_ptr(), whole.data_ptr(), 1, 8, s, d, st) == 0
    for h in range(0, 8, 2):
        assert lib.mta_lower_scores_f32(a[0, h].data_ptr(), b[0, h].data_ptr(), part[0, h].data_ptr(), 1, 2, s, d, st) == 0
    assert torch.equal(whole, part)
    want = (a.double() @ b.double().transpose(2, 3)).tril()
    size = (a.double().abs() @ b.double().abs().transpose(2, 3))
    assert ((whole.double().tril() - want).abs() <= d * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_operands_read_where_their_rows_lie(pkg, d, dtype):
    """P^T X and the lower scores with an operand laid out (B,S,H,D), a batch slice of one, and rows further apart: the bits that a
    contiguous copy gives, for every form of the product."""
    lib, code = pkg._lib.load(), {torch.bfloat16: 1, torch.float16: 2}[dtype]
    st = torch.cuda.current_stream().cuda_stream
    for b, h, s, apart in ((1, 1, 8, 0), (2, 8, 256, 0), (2, 3, 72, 8), (1, 16, 1096, 0), (2, 16, 1000, 0), (3, 16, 1024, 16), (4, 32, 784, 0)):
        print(f"rows in place {b}x{h}x{s}x{d} {apart} {dtype}", flush=True)
        x = torch.randn(b, s, h, d + apart, device="cuda").to(dtype)[..., :d].transpose(1, 2)
        other = torch.randn(b, h, s, d, device="cuda").to(dtype)
        p = torch.randn(b, h, s, s, device="cuda").to(dtype)
        got, want = ([torch.zeros(b, h, s, n, dtype=dtype, device="cuda") for n in (d, s)] for _ in range(2))
        y = x.contiguous()
        assert lib.mta_causal_ptx_rows_fwd(p.data_ptr(), x.data_ptr(), *x.stride()[:3], got[0].data_ptr(), b, h, s, d, 1, 0.5, code, st) == 0
        assert lib.mta_causal_ptx_scaled_fwd(p.data_ptr(), y.data_ptr(), want[0].data_ptr(), b, h, s, d, 1, 0.5, code, st) == 0
        assert lib.mta_lower_scores_rows_fwd(x.data_ptr(), *x.stride()[:3], other.data_ptr(), None, got[1].data_ptr(), b, h, s, d, code, st) == 0
        assert lib.mta_lower_scores_fwd(y.data_ptr(), other.data_ptr(), None, want[1].data_ptr(), b, h, s, d, code, st) == 0
        assert torch.equal(got[0], want[0]) and torch.equal(got[1].tril(), want[1].tril())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
def test_both_products_of_a_matrix(pkg, d, dtype):
    """The two products in one call: the bits of the single ones, in one launch (grids of up to 256 blocks, heads that divide over the
    XCDs and that do not, one block, a last block in part) and in two; NaN above the diagonal."""
    lib, code = pkg._lib.load(), {torch.bfloat16: 1, torch.float16: 2}[dtype]
    for b, h, s, causal in ((1, 1, 8, True), (1, 8, 256, True), (2, 3, 72, True), (1, 16, 1000, True), (3, 5, 264, False), (1, 8, 2048, True), (1, 16, 1096, True)):
        print(f"both products {b}x{h}x{s}x{d} causal={causal} {dtype}", flush=True)
        p = torch.randn(b, h, s, s, device="cuda").to(dtype)
        if causal:
            p = p.masked_fill(~torch.tril(torch.ones(s, s, dtype=torch.bool, device="cuda")), float("nan"))
        v, x = (torch.randn(b, h, s, d, device="cuda").to(dtype) for _ in range(2))
        got, want = ([torch.full_like(v, 7.0) for _ in range(2)] for _ in range(2))
        st = torch.cuda.current_stream().cuda_stream
        at = lambda t: t.data_ptr()  # noqa: E731
        assert lib.mta_causal_products(at(p), at(v), at(x), at(got[0]), at(got[1]), b, h, s, d, causal, 0.37, code, st) == 0
        assert lib.mta_causal_pv_scaled_fwd(at(p), at(v), at(want[0]), b, h, s, d, causal, 0.37, code, st) == 0
        assert lib.mta_causal_ptx_scaled_fwd(at(p), at(x), at(want[1]), b, h, s, d, causal, 0.37, code, st) == 0
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and not got[0].isnan().any()


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("r,k", [(3, 3), (6, 11), (7, 9)])
def test_conv_kernel_gradient_of_large_and_of_small_tensors(pkg, r, k, causal):
    """Beyond 32 M elements the kernel gradient takes steps of 64 keys, its batch entries one by one steps of 32: fp32 sums of the same
    exact products in another order, whose error sqrt(n)*2^-22 of the sum of magnitudes covers."""
    x, dy = (torch.randn(2, 5, 2048, 2040, device="cuda").to(torch.bfloat16) for _ in range(2))
    assert x.numel() > 32 << 20 >= x[:1].numel()
    whole = pkg.ops.conv2d_bwd_weight(x, dy, (r, k), causal)
    parts = sum(pkg.ops.conv2d_bwd_weight(x[i:i + 1], dy[i:i + 1], (r, k), causal).double() for i in range(2))
    size = pkg.ops.conv2d_bwd_weight(x.abs(), dy.abs(), (r, k), causal).double()
    assert ((whole.double() - parts).abs() <= (2 * 2048 * 2040) ** 0.5 * 2.0 ** -22 * size).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,k", [(3, 3), (5, 5), (7, 7)])
@pytest.mark.parametrize("n,c,s,group", [(4, 16, 640, 4), (2, 32, 648, 2), (1, 16, 1288, 4)])
def test_conv_and_small_groups_on_the_matrix_cores(pkg, n, c, s, group, r, k, dtype):
    """Conv and mixing of groups of 2 or 4 in one pass against the two kernels (the same roundings; sums of at most 4 products in
    another order: a neighbour of the result), NaN above the diagonal, and NaN in one head that must stay in its group."""
    g = torch.Generator().manual_seed(61)
    block = torch.arange(c) // group
    same = block[:, None] == block[None, :]
    x = torch.randn(n, c, s, s, generator=g).to(dtype).cuda()
    x = x.masked_fill(~torch.tril(torch.ones(s, s, dtype=torch.bool, device="cuda")), float("nan"))
    w = torch.randn(c, r, k, generator=g).to(dtype).cuda()
    wm = (torch.eye(c) + 0.3 * torch.randn(c, c, generator=g)).to(dtype).masked_fill(~same, float("inf")).cuda()
    ulp = 2 * _unit(dtype)
    for fill in (False, True):
        one = pkg.ops.conv2d_headmix(x, w, wm, True, group_size=group, fill_upper=fill)
        two = pkg.ops.headmix(pkg.ops.conv2d_causal(x, w, True, fill_upper=False), wm, True, 0.0, group_size=group, fill_upper=fill)
        one, two = (t if fill else t.tril() for t in (one, two))
        torch.testing.assert_close(one.float(), two.float(), rtol=ulp, atol=4 * ulp)
    x[0, 5] = float("nan")
    one = pkg.ops.conv2d_headmix(x, w, wm, True, group_size=group, fill_upper=True)
    assert one.isnan().any(-1).any(-1).nonzero().tolist() == [[0, h] for h in range(c) if h // group == 5 // group]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,group", [(9, 0), (12, 0), (24, 12), (17, 0), (24, 0), (32, 0), (64, 32)])
def test_mix_softmax_of_dense_groups(pkg, c, group, dtype):
    """16-bit groups of 9 to 32 heads in one pass: rows about a tile of 128 keys, of one and several wavefronts and passes, the longest
    row; one and two weights; a key bias; a band mask (rows that start inside a tile, behind one, behind all attended keys); NaN above
    the diagonal.  Against float64 with the stages' roundings: a mixed score that rounds to its neighbour, 2u|s| away, moves every
    probability of the row by as much, twice (numerator and sum)."""
    g = torch.Generator().manual_seed(59)
    u, hg = _unit(dtype), group or c
    half_step = 2.0 ** -25 if dtype == torch.float16 else 0.0   # (rounding of a subnormal result)
    block = torch.arange(c) // hg
    same = block[:, None] == block[None, :]
    longest = 4096 if hg <= 16 else 2048
    for n, p, q, causal, two, bias, band in ((2, 8, 8, True, False, False, False), (1, 136, 136, True, True, False, False), (2, 130, 136, True, False, True, False),
                                             (1, 264, 264, True, True, False, True), (1, 520, 520, True, False, True, True), (2, 3, 264, False, True, True, False),
                                             (1, 3, 1032, False, False, False, False), (1, 2, longest - 8, False, True, False, False), (1, 2, longest, False, False, True, False)):
        print(f"mix + softmax of dense groups c={c} group={group} {n}x{p}x{q} causal={causal} two={two} bias={bias} band={band} {dtype}", flush=True)
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        x = torch.randn(n, c, p, q, generator=g).to(dtype)
        w1, w2 = ((torch.eye(c) + 0.2 * torch.randn(c, c, generator=g)).to(dtype) for _ in range(2))
        kb = torch.where(torch.rand(n, q, generator=g) < 0.2, float("-inf"), 0.25) if bias else None
        if bias:
            kb[:, 0] = 0.0
        first = None
        if band:   # (the last row sees nothing)
            first = torch.clamp(torch.arange(p) - q // 3, min=0).int().repeat(n, 1)
            first[:, -1] = p
        s = torch.einsum("oi,nipq->nopq", w1.double() * same, x.double()).to(dtype)
        if bias:
            s = (s.float() + kb[:, None, None, :]).to(dtype)
        seen = keep[None, None].expand(n, 1, p, q)
        if band:
            seen = seen & (torch.arange(q)[None, None, None, :] >= first[:, None, :, None])
        s = s.double().masked_fill(~seen, float("-inf"))
        off = 4 * u * s.masked_fill(s.isinf(), 0.0).abs().amax(-1, keepdim=True)
        want = torch.softmax(s, -1)
        size = want
        if two:
            want = torch.einsum("oi,nipq->nopq", w2.double() * same, want.to(dtype).double())
            size = torch.einsum("oi,nipq->nopq", w2.double().abs() * same, size)
        got = pkg.ops.headmix_softmax(x.masked_fill(~keep, float("nan")).cuda(), w1.masked_fill(~same, float("inf")).cuda(),
                                      w2.masked_fill(~same, float("inf")).cuda() if two else None, causal, group_size=group or None, fill_upper=causal,
                                      key_bias=kb.cuda() if bias else None, first_visible=first.cuda() if band else None).cpu().double()
        rows = p - 1 if band else p
        assert ((got - want).abs() <= (off + 3 * u) * size + half_step * (hg + 1))[..., :rows, :].all()
        if causal:
            assert (got[..., ~keep] == 0.0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,k", [(3, 3), (6, 11), (7, 7), (7, 9), (11, 15)])
def test_conv_of_the_lower_triangle_by_strips(pkg, r, k, dtype):
    """The conv and its input gradient on the lower triangle only, at edges of the 64 x 128 strips and of the planes, NaN above the
    diagonal; and with every output written, where 11 rows take the same strips.  Against float64: an fp32 sum of at most r*k exact
    products, one rounding to the dtype."""
    import torch.nn.functional as F
    g, pad = torch.Generator().manual_seed(53), (k - 1) // 2
    half_step = 2.0 ** -25 if dtype == torch.float16 else 0.0   # (rounding of a subnormal result)
    for n, c, s in ((1, 1, 8), (2, 3, 56), (1, 2, 64), (3, 2, 72), (1, 3, 128), (2, 2, 136), (1, 2, 192), (1, 1, 264), (2, 3, 328)):
        print(f"conv of the lower triangle {r}x{k} {n}x{c}x{s} {dtype}", flush=True)
        keep = torch.tril(torch.ones(s, s, dtype=torch.bool))
        x, w = torch.randn(n, c, s, s, generator=g).to(dtype), torch.randn(c, r, k, generator=g).to(dtype)
        xd, wd = x.double().masked_fill(~keep, 0.0), w.double()[:, None]
        fwd = lambda t, u: F.conv2d(F.pad(t, (pad, pad, r - 1, 0)), u, groups=c)  # noqa: E731
        bwd = lambda t, u: F.conv2d(F.pad(t, (pad, pad, 0, r - 1)), u.flip(2, 3), groups=c)  # noqa: E731
        dirty = x.masked_fill(~keep, float("nan")).cuda()
        for op, ref in ((pkg.ops.conv2d_causal, fwd), (pkg.ops.conv2d_bwd_input, bwd)):
            want, size = ref(xd, wd), ref(xd.abs(), wd.abs())
            for fill in (False, True):
                got = op(dirty, w.cuda(), True, fill_upper=fill).cpu().double()
                bad = (got - want).abs() > _unit(dtype) * 1.01 * want.abs() + r * k * 2.0 ** -24 * size + half_step
                assert not bad[..., keep].any()
                if fill:
                    assert (got[..., ~keep] == 0.0).all()


@pytest.mark.parametrize("r,k", [(3, 3), (6, 11)])
def test_conv_strips_of_large_and_of_small_tensors_agree(pkg, r, k):
    """A tensor beyond 128 MB takes 32 x 256 strips on its lower triangle, its parts 64 x 128: the same sums in the same order."""
    x = torch.randn(2, 4, 2944, 2944, device="cuda").to(torch.bfloat16)
    w = torch.randn(4, r, k, device="cuda").to(torch.bfloat16)
    assert x.numel() * 2 > 128 << 20 >= x[:1].numel() * 2
    for op in (pkg.ops.conv2d_causal, pkg.ops.conv2d_bwd_input):
        whole = op(x, w, True, fill_upper=False).tril()
        for i in range(2):
            assert torch.equal(whole[i:i + 1], op(x[i:i + 1], w, True, fill_upper=False).tril())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("count", [1, 3, 8])
def test_sums_of_partial_results(pkg, count, dtype):
    """Several gradients' partial results in one launch: one block per channel (conv kernels), one per group on the diagonal, a whole
    matrix cut to its groups; numbers of entries and of partial results about 16 and 64.  Against float64: an fp32 sum of n values in
    any order is within n * 2^-24 of the sum of magnitudes, one rounding to the dtype."""
    lib, code = pkg._lib.load(), {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}[dtype]
    g = torch.Generator().manual_seed(47)
    kinds = [(3, 15, 1, 0, 0), (2, 66, 63, 0, 0), (8, 4, 130, 2, 0), (16, 256, 65, 16, 4), (1, 1, 64, 0, 0), (5, 17, 2, 0, 0), (6, 36, 1, 6, 0), (12, 9, 1000, 3, 0)]
    jobs, want = (pkg._lib.Partials * count)(), []
    for i, (rows, entries, parts, side, mask) in enumerate(kinds[:count]):
        blocks = rows // side if side else rows
        data = torch.randn(blocks, parts, entries, generator=g)
        scale = 0.5 if side == 0 else 1.0
        sums, sizes = data.double().sum(1) * scale, data.double().abs().sum(1) * scale
        if side:
            sums, sizes = (torch.block_diag(*t.view(blocks, side, side)) for t in (sums, sizes))
            if mask:
                sums, sizes = (t * torch.block_diag(*[torch.ones(mask, mask)] * (rows // mask)) for t in (sums, sizes))
        dw = torch.full((sums.numel() + 8,), 7.0, dtype=dtype, device="cuda")
        kept = data.cuda()
        jobs[i] = pkg._lib.Partials(kept.data_ptr(), dw.data_ptr(), rows, entries, parts, side, mask, code, scale)
        want.append((kept, dw, sums.flatten(), sizes.flatten(), parts))
    assert lib.mta_sum_partials(count, jobs, torch.cuda.current_stream().cuda_stream) == 0
    half_step = 2.0 ** -25 if dtype == torch.float16 else 0.0   # (rounding of a subnormal result)
    for _, dw, sums, sizes, parts in want:
        got = dw.cpu().double()
        assert (got[sums.numel():] == 7.0).all()
        assert ((got[:sums.numel()] - sums).abs() <= _unit(dtype) * 1.01 * sums.abs() + parts * 2.0 ** -24 * sizes + half_step).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,group,longest", [(2, 0, 4096), (4, 0, 4096), (8, 0, 4096), (12, 0, 4096), (16, 0, 4096), (32, 0, 2048), (8, 4, 4096), (32, 16, 4096)])
def test_softmax_and_headmix_gradients(pkg, c, group, longest, dtype):
    """Softmax gradient, mixing and weight gradient in one pass: rows of one wavefront and of several, of one tile per wavefront and
    of several, the longest row, NaN above the diagonal.  Against float64: the score gradient is rounded to the dtype (one unit u
    of its magnitude), dx once more, dw's sums as above; fp32: the order of a row's sum of p * dp, below 4."""
    g = torch.Generator().manual_seed(43)
    longest = longest // 2 if dtype == torch.float32 else longest
    u = _unit(dtype) if dtype != torch.float32 else 2.0 ** -20
    for n, p, q, causal in ((2, 1, 8, True), (1, 8, 8, True), (3, 72, 72, True), (1, 136, 136, True), (1, 520, 520, True), (2, 3, 264, False), (1, 2, 1032, False),
                            (1, 3, longest - 8, False), (1, 2, longest, False)):
        if q > longest:
            continue
        print(f"softmax + headmix gradients c={c} group={group} {n}x{p}x{q} causal={causal} {dtype}", flush=True)
        keep = torch.tril(torch.ones(p, q, dtype=torch.bool)) if causal else torch.ones(p, q, dtype=torch.bool)
        s = torch.softmax(torch.randn(n, c, p, q, generator=g).masked_fill(~keep, float("-inf")), -1).to(dtype)
        ds, x = (torch.randn(n, c, p, q, generator=g).to(dtype) for _ in range(2))
        w = (torch.eye(c) + 0.3 * torch.randn(c, c, generator=g)).to(dtype)
        block = torch.arange(c) // (group or c)
        same = block[:, None] == block[None, :]
        sd, dsd, xd, wd = s.double().masked_fill(~keep, 0.0), ds.double().masked_fill(~keep, 0.0), x.double().masked_fill(~keep, 0.0), w.double() * same
        dy = sd * (dsd - (sd * dsd).sum(-1, keepdim=True))
        most = sd * (dsd.abs() + (sd * dsd.abs()).sum(-1, keepdim=True))   # (what a rounding of one of its terms is relative to)
        want, size = torch.einsum("oi,nopq->nipq", wd, dy), torch.einsum("oi,nopq->nipq", wd.abs(), dy.abs() + 2.0 ** -19 / u * most)
        want_w = torch.einsum("nopq,nipq->oi", dy, xd) * same
        size_w = torch.einsum("nopq,nipq->oi", dy.abs() + 2.0 ** -19 / u * most, xd.abs())
        tiny = 2.0 ** -24 * 32 if dtype == torch.float16 else 0.0   # (fp16: subnormal score gradients)
        nan = float("nan")
        dx, dw = pkg.ops.headmix_grads(ds.masked_fill(~keep, nan).cuda(), x.masked_fill(~keep, nan).cuda(), w.cuda(), causal, group_size=group,
                                       probs=s.masked_fill(~keep, nan).cuda())
        dx, dw = dx.cpu().double(), dw.cpu().double()
        assert ((dx - want).abs() <= 2.02 * u * size + tiny)[..., keep].all()
        assert ((dw - want_w).abs() <= u * want_w.abs() + 1.01 * u * size_w + tiny * xd.abs().sum()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("c,group", [(2, 0), (4, 0), (8, 0), (12, 0), (16, 0), (32, 0), (16, 4), (16, 8)])
def test_headmix_gradients_of_many_rows(pkg, c, group, dtype):
    """The same kernels with more rows than wavefronts: a wavefront of the first takes several chunks, of rows of two batch entries
    too (an odd number of rows each), a workgroup of the one behind the softmax gradient several rows, whose wavefronts end one after
    the other.  Against float64 on the GPU, bounds as in the tests of the small sizes above."""
    g = torch.Generator(device="cuda").manual_seed(53)
    lanes = (group or c) <= 4
    half_step = 2.0 ** -25 if dtype == torch.float16 else 0.0
    block = torch.arange(c, device="cuda") // (group or c)
    same = block[:, None] == block[None, :]
    w = (torch.eye(c, device="cuda") + 0.3 * torch.randn(c, c, generator=g, device="cuda")).to(dtype)
    wd = w.double() * same
    mix = lambda t: torch.matmul(wd.t(), t.flatten(2)).view_as(t)   # noqa: E731
    size_of = lambda t: torch.matmul(wd.abs().t(), t.flatten(2)).view_as(t)   # noqa: E731
    contract = lambda a, b: torch.matmul(a.transpose(0, 1).flatten(1), b.transpose(0, 1).flatten(1).t()) * same   # noqa: E731
    nan = float("nan")
    for n, p, q, mode in ((3, 3001, 520, "lower") if lanes else (3, 1501, 264, "lower"), (2, 8193, 8, "fill"), (2, 8193, 16, "all")):
        print(f"headmix gradients c={c} group={group} {n}x{p}x{q} {mode} {dtype}", flush=True)
        causal = mode != "all"
        keep = torch.ones(p, q, dtype=torch.bool, device="cuda")
        keep = keep.tril() if causal else keep
        x, dy = (torch.randn(n, c, p, q, generator=g, device="cuda").to(dtype) for _ in range(2))
        xd, dyd = x.double().masked_fill(~keep, 0.0), dy.double().masked_fill(~keep, 0.0)
        dx, dw = pkg.ops.headmix_grads(dy.masked_fill(~keep, nan), x.masked_fill(~keep, nan), w, causal, group_size=group, fill_upper=mode == "fill")
        dx, dw, want, want_w = dx.double(), dw.double(), mix(dyd), contract(dyd, xd)
        assert ((dx - want).abs() <= _unit(dtype) * 1.01 * want.abs() + 2.0 ** -19 * size_of(dyd.abs()) + half_step)[..., keep].all()
        if mode == "fill":
            assert (dx[..., ~keep] == 0.0).all()
        assert ((dw - want_w).abs() <= _unit(dtype) * want_w.abs() + (n * p * q) ** 0.5 * 2.0 ** -22 * contract(dyd.abs(), xd.abs()) + half_step).all()
    u = _unit(dtype) if dtype != torch.float32 else 2.0 ** -20
    tiny = 2.0 ** -24 * 32 if dtype == torch.float16 else 0.0
    for n, p, q, causal in ((3, 1301, 264, True), (2, 2600, 40, True), (1, 4200, 136, False)):
        print(f"softmax + headmix gradients c={c} group={group} {n}x{p}x{q} causal={causal} {dtype}", flush=True)
        keep = torch.ones(p, q, dtype=torch.bool, device="cuda")
        keep = keep.tril() if causal else keep
        s = torch.softmax(torch.randn(n, c, p, q, generator=g, device="cuda").masked_fill(~keep, float("-inf")), -1).to(dtype)
        ds, x = (torch.randn(n, c, p, q, generator=g, device="cuda").to(dtype) for _ in range(2))
        sd, dsd, xd = (t.double().masked_fill(~keep, 0.0) for t in (s, ds, x))
        dy = sd * (dsd - (sd * dsd).sum(-1, keepdim=True))
        most = dy.abs() + 2.0 ** -19 / u * sd * (dsd.abs() + (sd * dsd.abs()).sum(-1, keepdim=True))
        dx, dw = pkg.ops.headmix_grads(ds.masked_fill(~keep, nan), x.masked_fill(~keep, nan), w, causal, group_size=group, probs=s.masked_fill(~keep, nan))
        dx, dw, want_w = dx.double(), dw.double(), contract(dy, xd)
        assert ((dx - mix(dy)).abs() <= 2.02 * u * size_of(most) + tiny)[..., keep].all()
        assert ((dw - want_w).abs() <= u * want_w.abs() + 1.01 * u * contract(most, xd.abs()) + tiny * xd.abs().sum()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,s,d", [(256, 40, 64), (130, 136, 128), (520, 8, 64), (512, 40, 64), (250, 136, 128), (1030, 40, 128), (600, 136, 128), (2100, 40, 64),
                                       (32, 1160, 128), (32, 2056, 128), (12, 2056, 64)])
def test_products_by_grid_size(pkg, heads, s, d, dtype):
    """P V and P^T X on the kernels that the number of row blocks chooses (64 or 128 rows, key blocks shared by one, two or four groups
    of wavefronts): one block, edges of the 64- and 128-row blocks and of the groups' shares, NaN above the diagonal, a band
    mask, the triangular layout.  Against the fp32 product of the same 16-bit values: one rounding of a result, and fp32 sums
    of s products below 1 * 4 in another order."""
    g = torch.Generator(device="cuda").manual_seed(47)
    print(f"products heads={heads} s={s} d={d} {dtype}", flush=True)
    p = torch.rand((1, heads, s, s), generator=g, device="cuda").to(dtype)
    x = torch.randn((1, heads, s, d), generator=g, device="cuda").to(dtype)
    low = torch.tril(torch.ones(s, s, dtype=torch.bool, device="cuda"))
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    some = [0, 1, heads // 2, heads - 1]
    close = dict(rtol=ulp * 1.01, atol=s * 2.0 ** -20)
    poisoned = p.masked_fill(~low, float("nan"))
    o, y = pkg.ops.causal_pv(poisoned, x, True), pkg.ops.causal_ptx(poisoned, x, True)
    full_o, full_y = pkg.ops.causal_pv(p, x, False), pkg.ops.causal_ptx(p, x, False)
    for h in some:
        a, b = p[0, h].float().masked_fill(~low, 0.0), x[0, h].float()
        torch.testing.assert_close(o[0, h].float(), a @ b, **close)
        torch.testing.assert_close(y[0, h].float(), a.t().contiguous() @ b, **close)
        torch.testing.assert_close(full_o[0, h].float(), p[0, h].float() @ b, **close)
        torch.testing.assert_close(full_y[0, h].float(), p[0, h].float().t().contiguous() @ b, **close)
    if heads % 2 == 0:
        assert torch.equal(pkg.ops.causal_pv_tri(pkg.ops.tri_pack(poisoned, 2), x, 2), o)
    first = (torch.arange(s, device="cuda") - s // 3).clamp(min=0).int()[None]
    keys = torch.arange(s, device="cuda")
    banded = poisoned.masked_fill(keys[None, :] < first[0][:, None], 0.0)
    assert torch.equal(pkg.ops.causal_pv(banded, x, True, first_visible=first), pkg.ops.causal_pv(banded, x, True))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,s,d", [(258, 8, 64), (258, 8, 128), (70, 200, 64), (17, 1008, 128), (9, 1800, 128), (10, 3080, 128), (79, 776, 128),
                                       (44, 1032, 128), (33, 2056, 128), (30, 2312, 64), (24, 2784, 128)])
def test_products_on_rings(pkg, heads, s, d, dtype):
    """The products of grids whose blocks come through rings of buffers: fewer blocks than a ring holds, as many as it holds and one more,
    last blocks of 8 and of all rows, 64 and 128 output rows, one and two groups, a grid of one round more than is resident at once; as
    test_products_by_grid_size compares them.  P^T X of rows that lie apart is that of the same rows side by side."""
    test_products_by_grid_size(pkg, heads, s, d, dtype)
    lib, st, code = pkg._lib.load(), torch.cuda.current_stream().cuda_stream, 1 if dtype == torch.bfloat16 else 2
    g = torch.Generator(device="cuda").manual_seed(59)
    p = torch.rand((1, heads, s, s), generator=g, device="cuda").to(dtype)
    x = torch.randn((1, s, heads, d), generator=g, device="cuda").to(dtype).transpose(1, 2)
    got, want = (torch.full((heads, s, d), float("nan"), dtype=dtype, device="cuda") for _ in range(2))
    assert lib.mta_causal_ptx_rows_fwd(p.data_ptr(), x.data_ptr(), *x.stride()[:3], got.data_ptr(), 1, heads, s, d, 1, 0.5, code, st) == 0
    y = x.contiguous()
    assert lib.mta_causal_ptx_scaled_fwd(p.data_ptr(), y.data_ptr(), want.data_ptr(), 1, heads, s, d, 1, 0.5, code, st) == 0
    assert torch.equal(got, want)


@pytest.mark.parametrize("heads,s,d", [(288, 4, 64), (160, 68, 128), (256, 36, 64), (512, 36, 64), (260, 128, 128), (768, 36, 64), (400, 100, 128)])
def test_fp32_products_by_grid_size(pkg, heads, s, d):
    """P V and P^T X in fp32 on the kernels that share V (X) in LDS, which the number of row blocks chooses: one block, edges of the
    32- and 64-row blocks and of the groups' shares, NaN above the diagonal.  Bound as in test_fp32_lower_products."""
    lib, st = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(53)
    print(f"fp32 products heads={heads} s={s} d={d}", flush=True)
    p = torch.randn((1, heads, s, s), generator=g, device="cuda")
    x = torch.randn((1, heads, s, d), generator=g, device="cuda")
    low = torch.tril(torch.ones(s, s, dtype=torch.bool, device="cuda"))
    pd, out = p.masked_fill(~low, float("nan")), torch.full_like(x, float("nan"))
    lower, xd = p.double().masked_fill(~low, 0.0).cpu(), x.double().cpu()
    for entry, left in ((lib.mta_causal_pv_f32, lower), (lib.mta_causal_ptx_f32, lower.transpose(2, 3))):
        assert entry(pd.data_ptr(), x.data_ptr(), out.data_ptr(), 1, heads, s, d, 0.5, st) == 0
        assert ((out.cpu().double() - 0.5 * (left @ xd)).abs() <= s ** 0.5 * 2.0 ** -22 * 0.5 * (left.abs() @ xd.abs()) + 1e-30).all()


def _bits(t):
    return t.view(torch.int32 if t.dtype == torch.float32 else torch.int16)


# groups of heads (0: a softmax without weights) and rows for the kernels of the softmax stage: one tile, several, several wavefronts
_SOFTMAX_GROUPS = (0, 2, 3, 4, 8, 9, 12, 16, 32)
_SOFTMAX_ROWS = (20, 24, 136, 264, 1040)


def _softmax_weights(group, dtype, g):
    c = group or 2
    w = [(torch.eye(c) + 0.2 * torch.randn(c, c, generator=g)).to(dtype).cuda() for _ in range(2)]
    return c, ((None, None),) if group == 0 else ((w[0], None), (None, w[1]), (w[0], w[1]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", _SOFTMAX_GROUPS)
def test_softmax_rows_that_are_not_finite_keep_the_fill(pkg, group, dtype):
    """A row with a NaN, or with every attended key hidden by the bias, is NaN on and below the diagonal and +0 above it (left alone
    or +0 without the fill); an infinity in the second weight stays below the diagonal; the other rows keep their bits."""
    g = torch.Generator().manual_seed(67)
    for s in _SOFTMAX_ROWS:
        c, weights = _softmax_weights(group, dtype, g)
        x = torch.randn(1, c, s, s, generator=g).to(dtype).cuda()
        upper = torch.triu(torch.ones(s, s, dtype=torch.bool, device="cuda"), 1)
        rows = torch.tensor([1, s // 3, s // 2, s - 2], device="cuda")
        others = torch.ones(s, dtype=torch.bool, device="cuda")
        others[rows] = False
        bad = x.clone()
        bad[0, 0, rows, rows // 2] = float("nan")
        bias = torch.zeros(1, s, device="cuda")
        bias[0, :s // 2] = float("-inf")
        for w1, w2 in weights:
            print(f"softmax of NaN group={group} s={s} {w1 is not None} {w2 is not None} {dtype}", flush=True)
            run = lambda t, v2=w2, **k: pkg.ops.headmix_softmax(t, w1, v2, True, group_size=group, **k)  # noqa: E731
            got, clean = run(bad), run(x)
            assert (_bits(got)[..., upper] == 0).all()
            mixed = slice(None) if w1 is not None or w2 is not None else slice(0, 1)   # (one weight mixes the NaN into every head)
            assert got[0, mixed][:, rows][..., ~upper[rows]].isnan().all()
            assert torch.equal(_bits(got)[:, :, others], _bits(clean)[:, :, others])
            above = run(bad, fill_upper=False, out=torch.full_like(x, 7.0))[..., upper]
            assert ((above == 7.0) | (_bits(above) == 0)).all()
            hidden = run(x, key_bias=bias)
            assert (_bits(hidden)[..., upper] == 0).all() and hidden[:, :, :s // 2][..., ~upper[:s // 2]].isnan().all()
            assert torch.isfinite(hidden[:, :, s // 2:]).all()
            if w2 is not None:
                w_inf = w2.clone()
                w_inf[0, c - 1] = float("inf")
                assert (_bits(run(x, w_inf))[..., upper] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", _SOFTMAX_GROUPS)
def test_softmax_rows_without_a_visible_key(pkg, group, dtype):
    """Rows whose first visible key lies behind their last one, at every place in a tile: NaN at all keys up to the diagonal, as the
    softmax of -inf is, and the fill above it; the other rows keep their bits.  In (N,C,S,S) planes and in the triangular layout."""
    g = torch.Generator().manual_seed(71)
    for s in _SOFTMAX_ROWS:
        c, weights = _softmax_weights(group, dtype, g)
        x = torch.randn(1, c, s, s, generator=g).to(dtype).cuda()
        p = torch.arange(s, device="cuda")
        upper, empty = p[None, :] > p[:, None], p % 4 != 0      # (p + 1 = 64, 128, 256, ... among the empty rows)
        first = torch.where(empty, p + 1 + 3 * (p % 4 == 2), p // 2).int()[None]
        seen = torch.where(empty, 0, p // 2).int()[None]
        for bias in (None, torch.full((1, s), 0.25, device="cuda")):
            for w1, w2 in weights:
                print(f"softmax of nothing group={group} s={s} {w1 is not None} {w2 is not None} bias={bias is not None} {dtype}", flush=True)
                run = lambda lo: pkg.ops.headmix_softmax(x, w1, w2, True, group_size=group, key_bias=bias, first_visible=lo)  # noqa: E731
                got, want = run(first), run(seen)
                assert (_bits(got)[..., upper] == 0).all()
                assert got[:, :, empty][..., ~upper[empty]].isnan().all()
                assert torch.equal(_bits(got)[:, :, ~empty], _bits(want)[:, :, ~empty])
                code = pkg.ops._code(x, "input")
                if group and pkg._lib.load().mta_headmix_softmax_tri_supported(c, s, group, 0, code, code, w1 is not None, w2 is not None, 1, bias is not None):
                    tri = pkg.ops.headmix_softmax_tri(pkg.ops.tri_pack(x, group), w1, w2, 1, c, s, group, key_bias=bias, first_visible=first)
                    tri = pkg.ops.tri_unpack(tri, 1, c, s, group)[..., ~upper]
                    assert torch.equal(tri.nan_to_num(7.0), got[..., ~upper].nan_to_num(7.0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", _SOFTMAX_GROUPS)
def test_softmax_of_a_window_wider_than_its_rows(pkg, group, dtype):
    """First visible keys below 0, by less than a tile and by several: the bits that 0 gives, row by row, beside rows that hide keys."""
    g = torch.Generator().manual_seed(73)
    for s in _SOFTMAX_ROWS:
        c, weights = _softmax_weights(group, dtype, g)
        x = torch.randn(1, c, s, s, generator=g).to(dtype).cuda()
        p = torch.arange(s, device="cuda")
        first = torch.where(p % 3 == 0, p - s - 1, torch.where(p % 3 == 1, p // 2, p - 5 * s - 700)).int()[None]
        for w1, w2 in weights:
            print(f"softmax of a wide window group={group} s={s} {w1 is not None} {w2 is not None} {dtype}", flush=True)
            run = lambda lo: _bits(pkg.ops.headmix_softmax(x, w1, w2, True, group_size=group, first_visible=lo))  # noqa: E731
            got = run(first)
            assert torch.equal(got, run(first.clamp(min=0))) and not got.view(dtype).isnan().any()


def _conv64(x, w, causal, bwd):
    """The depthwise conv (or its input gradient) in 64 bits, and the sum of the magnitudes it adds up."""
    r, k = w.shape[-2:]
    x, w = x.double(), w.double()
    low = torch.ones(x.shape[-2:], dtype=torch.bool, device=x.device).tril()
    if causal:
        x = torch.where(low, x, 0.0)
    pad, padr = (k - 1) // 2, k - 1 - (k - 1) // 2
    x = torch.nn.functional.pad(x, (padr, pad, 0, r - 1) if bwd else (pad, padr, r - 1, 0))
    w = w.flip(-1, -2) if bwd else w
    both = [torch.nn.functional.conv2d(a.cpu(), b.cpu()[:, None], groups=x.shape[1]).cuda() for a, b in ((x, w), (x.abs(), w.abs()))]
    return [torch.where(low, y, 0.0) for y in both] if causal else both


@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32),
                                          (torch.float16, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("h,w", [(1, 4), (31, 127), (33, 129), (64, 128), (40, 300), (300, 70), (389, 389)])
def test_conv_11x15_split(pkg, h, w, dtype, wdtype):
    """11x15 kernels on the parts of the values (fp32; 16-bit data with other weights or of odd widths): edges of the 32 x 128 strips,
    planes of one strip and of several (a workgroup each; several in turns: test_conv_split_strips_in_turns), wide and tall ones; forward, scaled, lower triangle only, input gradient; causal
    or not.  Bound: 165 products and sums of 32 bits in any order, (165 + 2) 2^-24 of the sum of their magnitudes, and one rounding
    of the result to its type."""
    g = torch.Generator(device="cuda").manual_seed(61)
    x = torch.randn(2, 3, h, w, generator=g, device="cuda").to(dtype)
    k = (0.1 * torch.randn(3, 11, 15, generator=g, device="cuda")).to(wdtype)
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]

    def close(got, x, causal, bwd):
        want, size = _conv64(x, k, causal, bwd)
        assert ((got.double() - want).abs() <= 167 * 2.0 ** -24 * size + ulp * want.abs() + 2.0 ** -25 * (dtype == torch.float16)).all()

    for causal in (True, False):
        close(pkg.ops.conv2d_causal(x, k, causal), x, causal, False)
        close(pkg.ops.conv2d_bwd_input(x, k, causal), x, causal, True)
    close(pkg.ops.conv2d_causal(x, k, True, in_scale=0.3), (x.float() * 0.3).to(dtype), True, False)
    out = torch.full_like(x, 7.0)
    pkg.ops.conv2d_causal(x, k, True, out=out, fill_upper=False)
    close(torch.tril(out), x, True, False)


@pytest.mark.parametrize("bwd", [False, True])
def test_conv_11x15_split_values(pkg, bwd):
    """Values that do not split into bf16 parts: infinities and NaN stay where a tap takes them, the largest numbers are not taken for
    infinite, and data or weights so small that their parts underflow keep their 32 bits."""
    g = torch.Generator(device="cuda").manual_seed(62)
    k = 0.1 * torch.randn(2, 11, 15, generator=g, device="cuda")
    run = (lambda x, k: pkg.ops.conv2d_bwd_input(x, k, True)) if bwd else (lambda x, k: pkg.ops.conv2d_causal(x, k, True))
    x = torch.randn(1, 2, 200, 200, generator=g, device="cuda")
    plain = run(x, k)
    for value in (float("inf"), float("-inf"), float("nan")):
        y = x.clone()
        y[0, 0, 120, 60] = value
        got = run(y, k)
        touched = torch.zeros(200, 200, dtype=torch.bool, device="cuda")
        touched[(slice(110, 121) if bwd else slice(120, 131)), 53:68] = True
        assert not torch.isfinite(got[0, 0][touched.tril()]).any()
        torch.testing.assert_close(got[0, 0][~touched], plain[0, 0][~touched], rtol=1e-4, atol=1e-5)
        assert torch.equal(got[0, 1], plain[0, 1])
    y = torch.zeros_like(x)
    y[0, 0, 150, 70] = 3.4e38
    want = _conv64(y, 0.01 * k, True, bwd)[0]
    torch.testing.assert_close(run(y, 0.01 * k).double(), want, rtol=2.0 ** -22, atol=0.0)
    for sx, sk in ((2.0 ** -115, 1.0), (1.0, 2.0 ** -115), (2.0 ** -60, 2.0 ** -60)):
        torch.testing.assert_close(run(x * sx, k * sk) * (1 / (sx * sk)), plain, rtol=2.0 ** -20, atol=2.0 ** -20)


@pytest.mark.parametrize("bwd", [False, True])
def test_conv_11x15_split_range(pkg, bwd):
    """The 32 bits are kept at the ends of fp32's range, whatever lies beside a value: tiny taps under huge data and the reverse (every sum finite,
    of values that a common factor of 2^100 overflows), values and taps down to the denormals beside ordinary ones, products at the
    smallest normal number, sums of 2^80 and more.  Bound: 165 products and sums of 32 bits, and the last place of a denormal for each."""
    g = torch.Generator(device="cuda").manual_seed(75)
    x, k = torch.randn(1, 2, 200, 200, generator=g, device="cuda"), 0.1 * torch.randn(2, 11, 15, generator=g, device="cuda")
    far, top, one = x.clone(), k.clone(), torch.zeros_like(x)
    far[..., 60:] *= 2.0 ** -126
    far[..., 110:] *= 2.0 ** -9
    top[:, :5] *= 2.0 ** -115
    one[..., 100, 80] = 1.7
    for a, w in ((torch.full_like(x, 2.0 ** 122), torch.full_like(k, 1.9 * 2.0 ** -101)), (torch.full_like(x, 1.9 * 2.0 ** -101), torch.full_like(k, 2.0 ** 122)),
                 (far, k), (one, top), (x * 2.0 ** -60, k * 2.0 ** -60), (x * 2.0 ** -64, k * 2.0 ** -64), (x * 2.0 ** 85, k), (x, k * 2.0 ** 100),
                 (x * 2.0 ** 110, k * 2.0 ** -110)):
        got = pkg.ops.conv2d_bwd_input(a, w, True) if bwd else pkg.ops.conv2d_causal(a, w, True)
        want, size = _conv64(a, w, True, bwd)
        assert ((got.double() - want).abs() <= 167 * (2.0 ** -24 * size + 2.0 ** -149)).all()


@pytest.mark.parametrize("n,c,h,w", [(2, 8, 1000, 1001), (1, 16, 777, 777), (3, 7, 700, 801), (1, 5, 261, 331), (1, 5, 300, 269), (2, 8, 200, 335)])
@pytest.mark.parametrize("dtype,wdtype,r,k", [(torch.float32, torch.float32, 11, 15), (torch.bfloat16, torch.float32, 6, 11), (torch.float16, torch.float16, 7, 9),
                                                (torch.bfloat16, torch.bfloat16, 6, 11), (torch.float16, torch.float32, 6, 11)])
def test_conv_split_strips_in_turns(pkg, dtype, wdtype, r, k, n, c, h, w):
    """Convs on the parts of the values where a workgroup walks several strips (two workgroups per CU with fp32 data, three with the others: 24 to 48
    per plane here), planes dealt to the XCDs and not, and planes of few strips whose rows end at all places of the eight keys that are
    stored together: forward, lower triangle only, input gradient, causal or not; in the middle of a walk an infinite value, whose results
    come from multiply-adds, and in fp32 a stretch of tiny ones.  Bounds as for planes of few strips."""
    g = torch.Generator(device="cuda").manual_seed(79)
    x, weight = torch.randn(n, c, h, w, generator=g, device="cuda").to(dtype), (0.1 * torch.randn(c, r, k, generator=g, device="cuda")).to(wdtype)
    hit = (n - 1, c // 2, h // 2, w // 4)
    if dtype == torch.float32:
        x[:, :, h // 2 + 40:h // 2 + 100, :w // 3] *= 2.0 ** -125
    low = torch.ones(h, w, dtype=torch.bool, device="cuda").tril()
    ulp = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    left = (k - 1) // 2
    for causal in (True, False):
        for bwd in (False, True):
            taps = weight.flip(-1, -2) if bwd else weight
            pads = (k - 1 - left, left, 0, r - 1) if bwd else (left, k - 1 - left, r - 1, 0)
            data = torch.nn.functional.pad(torch.where(low, x, torch.zeros_like(x)) if causal else x, pads).double()
            want, size = torch.zeros(n, c, h, w, dtype=torch.float64, device="cuda"), torch.zeros(n, c, h, w, dtype=torch.float64, device="cuda")
            for i in range(r):
                for j in range(k):
                    piece, tap = data[..., i:i + h, j:j + w], taps[:, i, j].double().view(1, c, 1, 1)
                    want.addcmul_(piece, tap)
                    size.addcmul_(piece.abs(), tap.abs())
            bound = (r * k + 2) * 2.0 ** -24 * size + ulp * want.abs() + (2.0 ** -25 if dtype == torch.float16 else r * k * 2.0 ** -149)
            keep = low if causal else torch.ones_like(low)
            rows = slice(hit[2] - r + 1, hit[2] + 1) if bwd else slice(hit[2], hit[2] + r)
            reach = slice(hit[3] - (left if bwd else k - 1 - left), hit[3] + (k - 1 - left if bwd else left) + 1)
            for fill in (True, False):
                for infinite in (False, True):
                    y = x.clone()
                    if infinite:
                        y[hit] = float("inf")
                    got = pkg.ops.conv2d_bwd_input(y, weight, causal, fill_upper=fill) if bwd else pkg.ops.conv2d_causal(y, weight, causal, fill_upper=fill)
                    off = ~((got.double() - want).abs() <= bound) & keep
                    if fill and causal:
                        assert not got[..., ~low].any()
                    if infinite:
                        seen = torch.zeros_like(off)
                        seen[hit[0], hit[1], rows, reach] = True
                        assert not torch.isfinite(got[seen & keep]).any()
                        off &= ~seen
                    assert not off.any(), (causal, bwd, fill, infinite)


@pytest.mark.parametrize("heads,s,d", [(300, 4, 64), (300, 132, 64), (37, 388, 64), (9, 1000, 64), (16, 1024, 64), (130, 60, 128), (130, 64, 128), (23, 388, 128),
                                       (5, 1036, 128)])
def test_fp32_scores_split(pkg, heads, s, d):
    """fp32 scores of the larger grids, on the parts of the operands: edges of the 128-row blocks and of the steps of 64 (32) keys, runs of two
    and more.  Bound: d products and sums of 32 bits in any order.  Nothing written above the diagonal beyond its vectors; an infinite
    operand gives what fp32 products give, and operands so small that their parts underflow keep their bits."""
    lib, st = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(63)
    a, b = (torch.randn(1, heads, s, d, generator=g, device="cuda") for _ in range(2))
    row = torch.arange(s, device="cuda")
    beyond = row[None, :] > (row[:, None] | 3)

    def run(a, b):
        out = torch.full((1, heads, s, s), 7.0, device="cuda")
        assert lib.mta_lower_scores_f32(a.data_ptr(), b.data_ptr(), out.data_ptr(), 1, heads, s, d, st) == 0
        assert (out[..., beyond] == 7.0).all() and (out[..., (row[None, :] > row[:, None]) & ~beyond] == 0.0).all()
        return out.tril()

    want = (a.double() @ b.double().transpose(2, 3)).tril()
    size = (a.double().abs() @ b.double().abs().transpose(2, 3)).tril()
    plain = run(a, b)
    assert ((plain.double() - want).abs() <= d * 2.0 ** -24 * size).all()
    for value in (float("inf"), float("nan"), 3.4e38):
        x, y = a.clone(), 0.01 * b
        x[0, 1, s - 2, 5] = value
        got, clean = run(x, y), run(a, y)
        hit = x[0, 1, s - 2] @ y[0, 1].T
        assert torch.equal(torch.isnan(got[0, 1, s - 2, :s - 1]), torch.isnan(hit[:s - 1]))
        torch.testing.assert_close(got[0, 1, s - 2, :s - 1], hit[:s - 1], rtol=2.0 ** -20, atol=0.0, equal_nan=True)
        got[0, 1, s - 2] = clean[0, 1, s - 2]
        assert torch.equal(got[0, 2:], clean[0, 2:])
        torch.testing.assert_close(got, clean, rtol=1e-4, atol=1e-5)
    for sx, sy in ((2.0 ** -115, 1.0), (1.0, 2.0 ** -115)):
        assert ((run(a * sx, b * sy).double() / (sx * sy) - want).abs() <= d * 2.0 ** -24 * size).all()


@pytest.mark.parametrize("heads,s,d", [(64, 512, 64), (64, 260, 128)])
def test_fp32_scores_split_range(pkg, heads, s, d):
    """The 32 bits are kept at the ends of fp32's range: tiny operands against huge ones, tiny rows and keys down to the denormals beside ordinary
    ones, products at the smallest normal number, sums of 2^80 and more.  Bound: d products and sums of 32 bits, and the last place of a
    denormal for each."""
    lib, st = pkg._lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(76)
    a, b = (torch.randn(1, heads, s, d, generator=g, device="cuda") for _ in range(2))
    rows, keys = a.clone(), b.clone()
    rows[:, :, ::2] *= 2.0 ** -118
    rows[:, :, ::6] *= 2.0 ** -16
    keys[:, :, 1::3] *= 2.0 ** -125
    for x, y in ((a * 2.0 ** -120, b * 2.0 ** 110), (a * 2.0 ** 120, b * 2.0 ** -126), (rows, b), (a, keys), (rows, keys), (a * 2.0 ** -60, b * 2.0 ** -60),
                 (a * 2.0 ** -64, b * 2.0 ** -64), (a * 2.0 ** 45, b * 2.0 ** 45), (a * 2.0 ** 110, b)):
        out = torch.empty(1, heads, s, s, device="cuda")
        assert lib.mta_lower_scores_f32(x.data_ptr(), y.data_ptr(), out.data_ptr(), 1, heads, s, d, st) == 0
        want, size = ((u.double() @ v.double().transpose(2, 3)).tril() for u, v in ((x, y), (x.abs(), y.abs())))
        assert ((out.tril().double() - want).abs() <= d * (2.0 ** -24 * size + 2.0 ** -149)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("group", [1, 2, 4, 8])
def test_softmax_wavefronts_per_row(pkg, group, dtype):
    """Mix + softmax + mix of short rows on one, two and four wavefronts per row: row p of a causal plane knows only its first p + 1 keys, so
    the planes cut out of a wider one, which takes more wavefronts, get the same bits - without a mask, under a key bias and
    under a band, with one weight and with both.  The wide plane against torch (two roundings of the data type)."""
    g = torch.Generator(device="cuda").manual_seed(64)
    n, h, wide = 2, 16, 1600
    x = torch.randn(n, h, wide, wide, generator=g, device="cuda").to(dtype)
    block = torch.arange(h, device="cuda") // group
    w1, w2 = ((torch.eye(h, device="cuda") + 0.1 * torch.randn(h, h, generator=g, device="cuda")) * (block[:, None] == block[None]) for _ in range(2))
    w1, w2 = w1.to(dtype), w2.to(dtype)
    bias = torch.zeros(n, wide, device="cuda")
    bias[0, 100:180] = bias[1, 7:300] = float("-inf")
    lo = (torch.arange(wide, device="cuda") - 150).clamp(min=0).to(torch.int32).expand(n, wide).contiguous()
    for a, b in ((None, None),) if group == 1 else ((None, w2), (w1, None), (w1, w2)):
        for kb, band in ((None, None), (bias, None), (None, lo)):
            run = lambda s: pkg.ops.headmix_softmax(x[..., :s, :s].contiguous(), a, b, True, group_size=group, fill_upper=False,   # noqa: E731
                                                    key_bias=None if kb is None else kb[:, :s].contiguous(),
                                                    first_visible=None if band is None else band[:, :s].contiguous()).tril()
            whole = run(wide)
            for s in (8, 248, 256, 264, 504, 512, 520, 1016, 1024, 1032):
                assert torch.equal(whole[..., :s, :s], run(s)), (s, a is None, b is None, kb is None, band is None)
    s = x.float() if group == 1 else torch.matmul(w1.float(), x.float().flatten(2)).view_as(x).to(dtype).float()
    want = torch.softmax(s.masked_fill(torch.ones(wide, wide, dtype=torch.bool, device="cuda").triu(1), float("-inf")), -1)
    got = pkg.ops.headmix_softmax(x, None if group == 1 else w1, None, True, group_size=group, fill_upper=False).tril()
    ulp = {torch.float32: 2.0 ** -18, torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}[dtype]
    torch.testing.assert_close(got.float(), want, rtol=ulp * (1.0 if group == 1 else 8.0), atol=1e-6)


@pytest.mark.parametrize("dtype,r,k", [(torch.bfloat16, 3, 3), (torch.float16, 7, 9), (torch.bfloat16, 11, 15)])
@pytest.mark.parametrize("d", [64, 128])
def test_attention_of_few_workgroups(pkg, d, dtype, r, k):
    """Attention on eight wavefronts of 16 rows (small grids) and on four of 32: the same bits for the same heads, whether they are alone or
    among so many that the larger grid takes the other form; edges of the 112- to 120-row query blocks and of the 64-key blocks."""
    g = torch.Generator(device="cuda").manual_seed(65)
    for s in (1, 17, 64, 113, 121, 250):
        q, kk, v = (torch.randn(1, 600, s, d, generator=g, device="cuda").to(dtype) for _ in range(3))
        w = (0.1 * torch.randn(600, r, k, generator=g, device="cuda")).to(dtype)
        for causal in (True, False):
            run = lambda lo, hi: pkg.ops.conv_attn_fwd(q[:, lo:hi].contiguous(), kk[:, lo:hi].contiguous(), v[:, lo:hi].contiguous(), w[lo:hi], causal,   # noqa: E731
                                                       None, return_lse=True)
            (many, many_lse), (few, few_lse) = run(0, 600), run(590, 600)
            assert torch.equal(many[:, 590:], few) and torch.equal(many_lse[:, 590:], few_lse), (s, causal)
            assert torch.isfinite(many.float()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,k", [(3, 3), (3, 5), (5, 5), (5, 7), (6, 11), (7, 7), (7, 9), (11, 15)])
def test_conv_both_gradients(pkg, r, k, dtype):
    """Both gradients of the conv in one pass over dy against the two kernels: dx bit for bit; dw, the same exact products summed in fp32 in
    another order and rounded to the weight's dtype, within sqrt(n)*2^-22 of the sum of magnitudes and half a unit.  Edges of the 64 x 128
    strips, fewer strips than workgroups, more channels than workgroups (several rounds of strips: the test below); whole rows, the lower triangle, no
    mask on planes that are not square; NaN above the diagonal of both operands."""
    g = torch.Generator(device="cuda").manual_seed(67)
    for b, c, h, w, causal, fill in ((1, 2, 8, 8, True, True), (2, 3, 64, 64, True, False), (1, 2, 136, 136, True, True), (2, 2, 200, 200, True, False),
                                     (1, 520, 72, 72, True, True), (3, 1, 1288, 1288, True, True), (1, 2, 1096, 1096, True, False),
                                     (2, 3, 65, 136, False, True), (1, 2, 200, 128, False, True), (1, 1, 3, 520, False, True)):
        x, dy = (torch.randn(b, c, h, w, generator=g, device="cuda").to(dtype) for _ in range(2))
        weight = torch.randn(c, r, k, generator=g, device="cuda").to(dtype)
        size = pkg.ops.conv2d_bwd_weight(x.abs(), dy.abs(), (r, k), causal).double()
        if causal:
            above = ~torch.tril(torch.ones(h, w, dtype=torch.bool, device="cuda"))
            x, dy = x.masked_fill(above, float("nan")), dy.masked_fill(above, float("nan"))
        dx, dw = pkg.ops.conv2d_grads(x, dy, weight, causal, fill_upper=fill)
        want = pkg.ops.conv2d_bwd_input(dy, weight, causal, fill_upper=fill)
        assert torch.equal(dx, want) if fill else torch.equal(dx.tril(), want.tril()), (b, c, h, w)
        exact = pkg.ops.conv2d_bwd_weight(x, dy, (r, k), causal).double()
        bound = (b * h * w) ** 0.5 * 2.0 ** -22 * size + exact.abs() * _unit(dtype) + (2.0 ** -25 if dtype == torch.float16 else 0.0)
        assert dw.dtype == dtype and ((dw.double() - exact).abs() <= bound).all(), (b, c, h, w)
        _, again = pkg.ops.conv2d_grads(x, dy, weight, causal, fill_upper=fill, over_x=True)   # the gradient in x's place
        assert torch.equal(again, dw) and (torch.equal(x, dx) if fill else torch.equal(x.tril(), dx.tril())), (b, c, h, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("r,k", [(3, 3), (6, 11), (7, 7), (11, 15)])
def test_conv_both_gradients_in_rounds(pkg, r, k, dtype):
    """... where a workgroup walks several strips of its channel, in uneven rounds (two workgroups per CU: 32 per channel of 16, 64 of 8, 12 of 43)
    over one plane and several: dx bit for bit, dw within the bound above, in x's place the same bits."""
    g = torch.Generator(device="cuda").manual_seed(78)
    for b, c, s, fill in ((1, 16, 1096, True), (2, 16, 520, False), (3, 16, 776, True), (1, 8, 1800, False), (2, 43, 456, True)):
        x, dy = (torch.randn(b, c, s, s, generator=g, device="cuda").to(dtype) for _ in range(2))
        weight = torch.randn(c, r, k, generator=g, device="cuda").to(dtype)
        size = pkg.ops.conv2d_bwd_weight(x.abs(), dy.abs(), (r, k), True).double()
        above = ~torch.tril(torch.ones(s, s, dtype=torch.bool, device="cuda"))
        x, dy = x.masked_fill(above, float("nan")), dy.masked_fill(above, float("nan"))
        dx, dw = pkg.ops.conv2d_grads(x, dy, weight, True, fill_upper=fill)
        want, exact = pkg.ops.conv2d_bwd_input(dy, weight, True, fill_upper=fill), pkg.ops.conv2d_bwd_weight(x, dy, (r, k), True).double()
        assert torch.equal(dx, want) if fill else torch.equal(dx.tril(), want.tril()), (b, c, s)
        bound = (b * s * s) ** 0.5 * 2.0 ** -22 * size + exact.abs() * _unit(dtype) + (2.0 ** -25 if dtype == torch.float16 else 0.0)
        assert ((dw.double() - exact).abs() <= bound).all(), (b, c, s)
        _, again = pkg.ops.conv2d_grads(x, dy, weight, True, fill_upper=fill, over_x=True)
        assert torch.equal(again, dw) and (torch.equal(x, dx) if fill else torch.equal(x.tril(), dx.tril())), (b, c, s)


def test_conv_both_gradients_refuses(pkg):
    """No kernel: causal planes that are not square on the matrix cores, and for what those do not take - other dtypes, widths and
    alignments - kernels of more than 35 taps."""
    def ask(h, w, r=7, k=7, causal=True, io=torch.bfloat16, wd=torch.bfloat16, shift=0):
        x, dy = (torch.randn(2 * h * w + shift, device="cuda").to(io)[shift:].view(1, 2, h, w) for _ in range(2))
        return pkg.ops.conv2d_grads(x, dy, torch.randn(2, r, k, device="cuda").to(wd), causal)
    assert ask(64, 64) is not None and ask(64, 72, causal=False) is not None
    for call in (dict(h=64, w=72), dict(h=68, w=68), dict(h=64, w=64, r=4, k=5), dict(h=64, w=64, io=torch.float32, wd=torch.float32),
                 dict(h=64, w=64, wd=torch.float32), dict(h=64, w=64, shift=1), dict(h=3, w=3, r=3, k=3)):
        assert ask(**call) is None, call


@pytest.mark.parametrize("dtype,wd", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32), (torch.float16, torch.float16)])
@pytest.mark.parametrize("r,k", [(3, 3), (3, 5), (5, 5), (5, 7)])
def test_conv_both_gradients_by_rows(pkg, r, k, dtype, wd):
    """Both gradients of the conv in one pass on the vector units against the two kernels: dx bit for bit in fp32; in 16 bits the same
    sums in another order (5x7), or a last multiply-add rounded to 16 bits with or without a stop at 32: 2^-24 of the magnitudes for each
    of its r k steps on either side, and the neighbour; dw, fp32 sums in another order, within sqrt(n)*2^-22 of
    the sum of magnitudes (and half a unit of a 16-bit weight).  Strips of 4 and 8 rows, one wavefront's and
    several rounds of them, the edges of their 240 to 248 keys, the narrowest rows; whole rows, the lower triangle, no mask, planes
    that are not square; NaN above the diagonal of both operands; the gradient in x's place."""
    g = torch.Generator(device="cuda").manual_seed(68)
    for b, c, h, w, causal, fill in ((1, 2, 5, 5, True, True), (2, 3, 65, 65, True, False), (1, 2, 249, 249, True, True), (2, 2, 121, 121, True, False),
                                     (2, 3, 65, 4, False, True), (1, 2, 30, 301, True, True), (1, 2, 301, 30, True, True), (1, 1100, 41, 41, True, True),
                                     (8, 16, 489, 489, True, True), (8, 16, 489, 489, True, False)):
        x, dy = (torch.randn(b, c, h, w, generator=g, device="cuda").to(dtype) for _ in range(2))
        weight = torch.randn(c, r, k, generator=g, device="cuda").to(wd)
        size = pkg.ops.conv2d_bwd_weight(x.abs(), dy.abs(), (r, k), causal).double()
        if causal:
            above = ~torch.tril(torch.ones(h, w, dtype=torch.bool, device="cuda"))
            x, dy = x.masked_fill(above, float("nan")), dy.masked_fill(above, float("nan"))
        dx, dw = pkg.ops.conv2d_grads(x, dy, weight, causal, fill_upper=fill)
        want = pkg.ops.conv2d_bwd_input(dy, weight, causal, fill_upper=fill)
        at, of = (dx, want) if fill else (dx.tril(), want.tril())
        if dtype == torch.float32:
            assert torch.equal(at, of), (b, c, h, w)
        else:
            near = pkg.ops.conv2d_bwd_input(torch.where(dy.isnan(), torch.zeros_like(dy), dy).abs(), weight.abs(), causal).double()
            near = 2 * (r * k + 2) * 2.0 ** -24 * near + 2 * _unit(dtype) * of.double().abs() + 2.0 ** -24
            assert ((at.double() - of.double()).abs() <= near).all(), (b, c, h, w)
        exact = pkg.ops.conv2d_bwd_weight(x, dy, (r, k), causal).double()
        half = 0.0 if wd == torch.float32 else exact.abs() * _unit(wd) + 2.0 ** -25
        assert dw.dtype == wd and ((dw.double() - exact).abs() <= (b * h * w) ** 0.5 * 2.0 ** -22 * size + half).all(), (b, c, h, w)
        _, again = pkg.ops.conv2d_grads(x, dy, weight, causal, fill_upper=fill, over_x=True)
        assert torch.equal(again, dw) and (torch.equal(x, dx) if fill else torch.equal(x.tril(), dx.tril())), (b, c, h, w)


@pytest.mark.parametrize("dtype,wd,r,k", [(d, w, *rk) for d, w, sizes in (
    (torch.bfloat16, torch.float32, ((5, 7), (7, 7), (6, 11), (7, 9))), (torch.bfloat16, torch.bfloat16, ((5, 7), (7, 7), (6, 11), (7, 9))),
    (torch.float16, torch.float32, ((6, 11), (7, 9))), (torch.float16, torch.float16, ((6, 11), (7, 9))), (torch.bfloat16, torch.float16, ((6, 11),))) for rk in sizes])
def test_conv_split_of_16_bit_data(pkg, dtype, wd, r, k):
    """16-bit data with other weights, or of odd widths, on the parts of the values: edges of the 32 x 128 strips; an
    infinite value stays where a tap takes it.  Bound: r k products and sums of 32 bits in any order, and one rounding to 16 bits."""
    g = torch.Generator(device="cuda").manual_seed(69)
    w = (0.1 * torch.randn(3, r, k, generator=g, device="cuda")).to(wd)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for h, wid in ((1, 5), (31, 33), (33, 129), (128, 120) if wd != dtype else (128, 121), (333, 333)):
        x = torch.randn(2, 3, h, wid, generator=g, device="cuda").to(dtype)
        for causal in (True, False):
            for bwd in (False, True):
                got = pkg.ops.conv2d_bwd_input(x, w, causal) if bwd else pkg.ops.conv2d_causal(x, w, causal)
                want, size = _conv64(x, w, causal, bwd)
                bound = (r * k + 2) * 2.0 ** -24 * size + ulp * want.abs() + 2.0 ** -25
                assert ((got.double() - want).abs() <= bound).all(), (h, wid, causal, bwd)
    x[0, 0, 200, 100] = float("inf")
    got, plain = pkg.ops.conv2d_causal(x, w, True), pkg.ops.conv2d_causal(x.masked_fill(x == float("inf"), 0.0), w, True)
    touched = torch.zeros(333, 333, dtype=torch.bool, device="cuda")
    touched[200:200 + r, 100 - (k - 1 - (k - 1) // 2):101 + (k - 1) // 2] = True
    assert not torch.isfinite(got[0, 0][touched.tril()]).any()
    torch.testing.assert_close(got[0, 0][~touched].float(), plain[0, 0][~touched].float(), rtol=2 * ulp, atol=2.0 ** -20)
    assert torch.equal(got[0, 1], plain[0, 1])


@pytest.mark.parametrize("causal", [True, False])
def test_mask_kinds_in_one_read(pkg, causal):
    """mta_mask_classify against the elementwise operations that other dtypes take: every kind of mask, booleans and additive ones, one plane or one
    per batch entry or head, strides that vectors fit and others, lengths around vectors and a wavefront's step; exact."""
    g = torch.Generator().manual_seed(71)
    mod = pkg.MTAAttentionTriton(2, pkg.MTAConfig(), dropout=0.0, causal=causal, use_mask=True).cuda()
    kinds = {}
    for s in (1, 7, 16, 17, 250, 256, 1025, 1040, 2100):
        at = torch.arange(s)
        lower = at[None, :] <= at[:, None]
        n = max(1, s // 3)
        forms = {"all": torch.ones(2, 1, s, s, dtype=torch.bool), "causal": lower.expand(2, 1, s, s),
                 "padded": (at < torch.tensor([[n], [s]])[:, None])[:, None].expand(2, 1, s, s), "first hidden": (at >= min(n, s - 1)).expand(1, 1, s, s),
                 "window": (lower & (at[None, :] > at[:, None] - n))[None, None], "nothing": torch.zeros(1, 1, s, s, dtype=torch.bool),
                 "left": (lower & (at[None, :] >= torch.tensor([n, 0])[:, None, None]))[:, None], "holes": (torch.rand(1, 1, s, s, generator=g) < 0.9) | (at == 0),
                 "upper only": lower[None, None] | (torch.rand(1, 1, s, s, generator=g) < 0.5)}
        for where in {(s - 1, 0), (s - 1, s - 1), (s // 2, s // 4), (0, 0), (0, s - 1)}:   # one position off
            off = forms["padded"].clone()
            off[-1, 0][where] ^= True
            forms[f"off {where}"] = off
        for name, m in forms.items():
            heads = m.expand(m.size(0), 2, s, s).clone()
            other = heads.clone()
            other[0, 1, s // 2, s - 1] ^= True
            for what, plane in (("one", m), ("heads", heads), ("differ", other)):
                add = torch.where(plane, 0.0, float("-inf"))
                odd, minus, nan = add.clone(), add.clone(), add.clone()
                odd[-1, -1, s // 2, 0], nan[0, 0, 0, s - 1] = -1e9, float("nan")
                minus[plane] = -0.0
                made = [("bool", plane), ("fp32", add), ("bf16", add.bfloat16()), ("fp16", add.half()), ("value", odd), ("value bf16", odd.bfloat16()),
                        ("nan", nan), ("-0", minus.half())]
                if what == "one":
                    wide = torch.zeros(*m.shape[:3], s + 3, dtype=torch.bool)
                    wide[..., 1:s + 1] = m
                    made += [("stride", wide.cuda()[..., 1:s + 1]), ("transposed", m.cuda().transpose(2, 3).contiguous().transpose(2, 3)), ("expanded", m[:1].cuda().expand(2, 1, s, s))]
                for kind, mask in made:
                    mask = mask.cuda()
                    mod._mask_cache = None
                    got, empty = mod._structured_mask(mask, 2, s), mod._band_empty_rows(mask)
                    want, want_empty = mod._structured_mask_elementwise(mask, 2, s)
                    assert got[0] == want[0], (s, name, what, kind, got[0], want[0])
                    kinds[got[0]] = kinds.get(got[0], 0) + 1
                    for a, b in ((got[1], want[1]), (empty, want_empty)):
                        assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and a.is_contiguous() and torch.equal(a, b))), (s, name, what, kind)
    assert set(kinds) == ({"keys", "band", None} if causal else {"keys", None})


@pytest.mark.parametrize("n", [65535, 65536])
def test_mask_of_many_batch_entries(pkg, n):
    """One entry per grid row: more of them than a grid has are classified by the elementwise operations, with the same answer."""
    mod = pkg.MTAAttentionTriton(2, pkg.MTAConfig(), dropout=0.0, causal=True, use_mask=True).cuda()
    mask = torch.ones(n, 1, 4, 4, dtype=torch.bool, device="cuda")
    mask[:, :, :, 3] = torch.arange(n, device="cuda")[:, None, None] % 2 == 0
    got, want = mod._structured_mask(mask, n, 4), mod._structured_mask_elementwise(mask, n, 4)[0]
    assert got[0] == want[0] == "keys" and torch.equal(got[1], want[1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [16, 32])
def test_headmix_wide_groups_with_fp32_weights(pkg, group, dtype):
    """16-bit data with fp32 weights: four keys per lane up to 1024 keys (32 heads in bf16: any length), eight beyond, and ragged lengths one.  Against
    float64: half an ulp of the result and fp32 sums of `group` terms."""
    g = torch.Generator().manual_seed(81)
    half = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for n, c, p, q in ((1, group, 3, 8), (2, 2 * group, 70, 70), (1, group, 136, 136), (1, group, 2, 1024), (1, group, 3, 1028), (1, group, 2, 1032), (1, group, 2, 2056)):
        x = torch.randn(n, c, p, q, generator=g).to(dtype).cuda()
        w = torch.block_diag(*[torch.eye(group) + 0.2 * torch.randn(group, group, generator=g) for _ in range(c // group)]).cuda()
        keep = torch.ones(p, q, dtype=torch.bool, device="cuda")
        for causal in (True, False):
            low = keep.tril() if causal else keep
            xd = x.masked_fill(~low, float("nan"))
            for name, m, fn in (("forward", w, lambda: pkg.ops.headmix(xd, w, causal, 0.0, group_size=group)),
                                ("input gradient", w.t(), lambda: pkg.ops.headmix_bwd_input(xd, w, causal, group))):
                want = torch.einsum("oi,nipq->nopq", m.double(), x.double()) * low
                size = torch.einsum("oi,nipq->nopq", m.double().abs(), x.double().abs())
                got = fn()
                assert ((got.double() - want).abs() <= half * want.abs() + group * 2.0 ** -23 * size + 2.0 ** -24).all(), (name, n, c, p, q, causal)
                assert (got[..., ~low] == 0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("kind", ["groups of 2", "groups of 4", "groups of 8", "dense", "post conv"])
def test_ragged_lengths_are_read_where_they_lie(pkg, kind, masked, dtype):
    """16-bit forwards of lengths that are not a multiple of 8 against the same rows with zero rows behind them, bit for bit: the same kernels in the
    same form, and what lies behind a head's rows - the next head's, or NaN behind the last - is not read.  All forms of P V, the triangular layout
    and planes, scores with statistics, windows; head groups of NaN beside the compared ones."""
    g = torch.Generator(device="cuda").manual_seed(91)
    group = int(kind[-1]) if "groups" in kind else 0
    for b, h, s, d in ((1, 8, 1, 64), (2, 8, 7, 128), (1, 8, 65, 64), (2, 16, 129, 128), (2, 16, 1001, 64), (1, 16, 2045, 128), (4, 16, 1531, 64), (1, 32, 4093, 64)):
        if s > 4000 and kind not in ("post conv", "groups of 4"):
            continue
        print(f"ragged {kind} masked={masked} {dtype} {(b, h, s, d)}", flush=True)
        mod = pkg.MTAAttentionTriton(h, pkg.MTAConfig(query_kernel_size=3, key_kernel_size=5), dropout=0.0, causal=True, use_mask=masked).cuda().to(dtype)
        with torch.no_grad():
            mod.mta_conv_triton.weight.copy_(0.2 * torch.randn(h, 3, 5, generator=g, device="cuda"))
            post = mod.mta_conv_after_sm_triton.weight
            post.zero_()[:, -1, 1] = 1.0
            if kind == "post conv":
                post.add_(0.1 * torch.randn(post.shape, generator=g, device="cuda"))
            block = torch.arange(h, device="cuda") // (group or h)
            for w in (mod.wpsm_triton.weight, mod.wposm_triton.weight):
                w.copy_((torch.eye(h, device="cuda") + 0.2 * torch.randn(h, h, generator=g, device="cuda")) * (block[:, None] == block[None, :]))
            if group in (2, 4):
                mod.wpsm_triton.weight.copy_(torch.eye(h))
        mod.eval().requires_grad_(False)
        mod.infer_weight_structure()
        pad = -s % 8
        at = torch.arange(s + pad, device="cuda")
        window = (at[None, :] <= at[:, None]) & (at[None, :] > at[:, None] - max(1, s // 3))
        mask = window[None, None] if masked else None
        rows = [torch.randn(b, h, s, d, generator=g, device="cuda").to(dtype) for _ in range(3)]
        clean = h
        if group and group < h:   # the last groups NaN
            clean = h - group
            for x in rows:
                x[:, clean:] = float("nan")
        ragged = []
        for x in rows:
            room = torch.full((x.numel() + 64 * d,), float("nan"), dtype=dtype, device="cuda")
            room[:x.numel()] = x.flatten()
            ragged.append(room[:x.numel()].view(x.shape))
        padded = [torch.nn.functional.pad(x, (0, 0, 0, pad)) for x in rows]
        with torch.no_grad():
            got = mod(*ragged, mask[..., :s, :s] if masked else None, None)
            want = mod(*padded, mask, None)[:, :s]
        assert got.shape == (b, s, h, d)
        assert torch.equal(got[:, :, :clean], want[:, :, :clean]) and not got[:, :, :clean].isnan().any()
