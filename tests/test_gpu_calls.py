"""Calls beyond the ordinary one (Q, K and V of one shape, whole rows, weights of the data's dtype): what the library products
take by broadcasting is the same through the kernels.  Against the CPU oracle in fp32, which sees the operands expanded."""
import pytest
import torch

from oracle import mta_oracle as O

pytestmark = pytest.mark.gpu

_WEIGHTS = ("mta_conv_triton", "wpsm_triton", "mta_conv_after_sm_triton", "wposm_triton")
# of the norm: fp32 sums in another order; 16 bits: a chain of about six roundings of 2^-9 / 2^-12 each
_REL = {torch.float32: 1e-5, torch.bfloat16: 1.5e-2, torch.float16: 2e-3}


@pytest.fixture(scope="module")
def pkg():
    import multitokenatention_triton_amd as m
    return m


def _module(pkg, h, dtype, wdtype=None, causal=True, use_mask=False, seed=11, **cfg):
    g = torch.Generator().manual_seed(seed)
    mod = pkg.MTAAttentionTriton(h, pkg.MTAConfig(**cfg), 0.0, causal, use_mask=use_mask)
    with torch.no_grad():
        for name in _WEIGHTS:
            w = getattr(mod, name).weight
            if w.dim() == 2:
                w.copy_(torch.eye(h) + 0.1 * torch.randn(h, h, generator=g))
            else:
                w.copy_(O.seeded_conv_weight(h, w.size(1), w.size(2), 0.05, torch.float32, seed=seed))
    return mod.to(wdtype or dtype).cuda()


def _oracle(mod, q, k, v, mask=None):
    """(output, leaves) of the oracle in fp32; the leaves are q, k, v as given and the four weights."""
    leaves = [t.float().cpu().clone().requires_grad_(True) for t in (q, k, v)]
    wl = [getattr(mod, n).weight.detach().float().cpu().clone().requires_grad_(True) for n in _WEIGHTS]
    b, h = (max(t.size(i) for t in leaves) for i in (0, 1))
    x = [t.expand(b, mod.n_heads if i < 2 else h, -1, -1) for i, t in enumerate(leaves)]
    return O.mta_forward(*x, wl[0].unsqueeze(1), wl[1], wl[2].unsqueeze(1), wl[3], mask=mask), leaves + wl


def _near(got, want, rel, what=""):
    got, want = got.detach().float().cpu(), want.detach().float()
    assert got.shape == want.shape, (what, got.shape, want.shape)
    assert torch.isfinite(got).all(), what
    assert float((got - want).norm()) <= rel * float(want.norm()), (what, float((got - want).norm() / want.norm()))


@pytest.mark.parametrize("s", [64, 45])
@pytest.mark.parametrize("dtype,form", [(torch.float32, "v_head"), (torch.float32, "v_batch"), (torch.float32, "k_head"), (torch.float32, "q_batch"),
                                        (torch.float32, "one_head_many_values"), (torch.float16, "v_head"), (torch.float16, "one_head_many_values")])
def test_operands_that_broadcast(pkg, dtype, form, s):
    """V, K or Q of one head or one batch entry, and V of more heads than the scores of a one-head module: the kernels that index
    the scores by V's sizes are not taken, the result is that of the expanded operands (fp32: with all gradients)."""
    print(f"broadcast {form} {dtype} s={s}", flush=True)
    h, d = (1 if form == "one_head_many_values" else 4), 64
    shapes = [[2, h, s, d] for _ in range(3)]
    if form == "one_head_many_values":
        shapes[2][1] = 3
    else:
        shapes["qkv".index(form[0])][1 if form.endswith("head") else 0] = 1
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(*sh, generator=g).to(dtype) for sh in shapes)
    mod = _module(pkg, h, dtype)
    want, leaves = _oracle(mod, q, k, v)
    dev = [t.cuda() for t in (q, k, v)]
    with torch.no_grad():
        _near(mod(*dev, None, None), want, _REL[dtype], "inference")
    if dtype != torch.float32:
        return
    dev = [t.requires_grad_(True) for t in dev]
    out = mod(*dev, None, None)
    _near(out, want, _REL[dtype], "training")
    go = torch.randn(want.shape, generator=g)
    want.backward(go)
    out.backward(go.cuda())
    for name, a, w in zip("q k v conv pre conv2 post".split(), [t.grad for t in dev] + [getattr(mod, n).weight.grad for n in _WEIGHTS],
                          [t.grad for t in leaves]):
        _near(a, w, 1e-4, name)


@pytest.mark.parametrize("kind", ["keys", "window"])
def test_masked_value_heads_that_broadcast(pkg, kind):
    """Hidden keys and a window with V of one head (fp32, a padded and a whole length): as of the expanded V."""
    for s in (45, 64):
        print(f"broadcast under a mask {kind} s={s}", flush=True)
        mod = _module(pkg, 4, torch.float32, use_mask=True)
        g = torch.Generator().manual_seed(4)
        q, k, v = torch.randn(2, 4, s, 64, generator=g), torch.randn(2, 4, s, 64, generator=g), torch.randn(2, 1, s, 64, generator=g)
        rows = torch.arange(s)
        visible = (rows[None, :] <= rows[:, None])[None, None].expand(2, 1, s, s).clone()
        if kind == "keys":
            visible[1, :, :, s - 9:] = False
            visible[1, 0, s - 9:, 0] = True
        else:
            visible &= (rows[None, :] > rows[:, None] - 17)
        want, leaves = _oracle(mod, q, k, v, mask=torch.where(visible, 0.0, float("-inf")).expand(2, 4, s, s))
        dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
        with torch.no_grad():
            _near(mod(*dev, visible.cuda(), None), want, 1e-5, "inference")
        out = mod(*dev, visible.cuda(), None)
        _near(out, want, 1e-5, "training")
        want.sum().backward()
        out.sum().backward()
        for name, a, w in zip("qkv", dev, leaves):
            _near(a.grad, w.grad, 1e-4, name)


def _misaligned(t):
    """t at an address that is not that of a 16-byte vector."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda")
    view = flat[1:].view(t.shape)
    view.copy_(t)
    assert view.is_contiguous() and view.data_ptr() % 16
    return view


@pytest.mark.parametrize("mask", [None, "keys", "window", "holes"])
@pytest.mark.parametrize("dtype,wdtype,which", [(torch.float32, torch.float32, "qkv"), (torch.float32, torch.float32, "v"), (torch.float16, torch.float32, "qk")])
def test_operands_between_vectors(pkg, dtype, wdtype, which, mask):
    """Contiguous Q, K and V in the middle of a flat buffer, where the products were the library's before the lower-triangle
    kernels took them: whole and padded lengths, inference and (fp32) training."""
    if mask == "holes" and dtype != torch.float32:
        pytest.skip("the mask passes over 16-bit scores refuse Q and K between vectors")
    for s in (64, 45):
        print(f"between vectors {dtype} {which} {mask} s={s}", flush=True)
        mod = _module(pkg, 4, dtype, wdtype, use_mask=mask is not None)
        g = torch.Generator().manual_seed(6)
        q, k, v = (torch.randn(2, 4, s, 64, generator=g).to(dtype) for _ in range(3))
        rows = torch.arange(s)
        visible = (rows[None, :] <= rows[:, None])[None, None]
        if mask == "keys":
            visible = visible & (rows < s - 7)
        elif mask == "window":
            visible = visible & (rows[None, :] > rows[:, None] - 17)
        elif mask == "holes":
            visible = visible & ((rows[None, :] + rows[:, None]) % 5 != 1)
        want, leaves = _oracle(mod, q, k, v, mask=torch.where(visible, 0.0, float("-inf")).expand(2, 4, s, s))
        dev = [_misaligned(t) if n in which else t.cuda() for n, t in zip("qkv", (q, k, v))]
        given = None if mask is None else visible.cuda()
        with torch.no_grad():
            _near(mod(*dev, given, None), want, _REL[dtype], "inference")
        if dtype != torch.float32:
            continue
        dev = [t.requires_grad_(True) for t in dev]
        out = mod(*dev, given, None)
        _near(out, want, _REL[dtype], "training")
        want.sum().backward()
        out.sum().backward()
        for name, a, w in zip("qkv", dev, leaves):
            _near(a.grad, w.grad, 1e-4, name)


@pytest.mark.parametrize("h", [12, 16, 32])
def test_head_weights_of_two_dtypes(pkg, h):
    """fp32 data, dense head weights of which one is kept in 16 bits, no conv between them: mix, softmax and mix one by one."""
    print(f"head weights of two dtypes h={h}", flush=True)
    for name in ("wpsm_triton", "wposm_triton"):
        mod = _module(pkg, h, torch.float32).requires_grad_(False)
        getattr(mod, name).to(torch.bfloat16)
        mod.mta_conv_after_sm_triton.weight.zero_()[:, -1, 1] = 1.0
        mod.declare_weight_structure(post_conv_identity=True)
        g = torch.Generator().manual_seed(8)
        q, k, v = (torch.randn(2, h, 64, 64, generator=g) for _ in range(3))
        want, _ = _oracle(mod, q, k, v)
        _near(mod(q.cuda(), k.cuda(), v.cuda(), None, None), want, 1e-5, name)


def test_more_keys_than_rows(pkg):
    """causal=False with more keys than query rows (no padding, no row copies): output and the gradients of Q, K and V."""
    print("more keys than rows", flush=True)
    mod = _module(pkg, 4, torch.float32, causal=False)
    g = torch.Generator().manual_seed(5)
    q, k, v = torch.randn(2, 4, 24, 64, generator=g), torch.randn(2, 4, 40, 64, generator=g), torch.randn(2, 4, 40, 64, generator=g)
    want, leaves = _oracle(mod, q, k, v, mask=torch.zeros(2, 4, 24, 40))
    dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    out = mod(*dev, None, None)
    _near(out, want, 1e-5)
    go = torch.randn(want.shape, generator=g)
    want.backward(go)
    out.backward(go.cuda())
    for name, a, w in zip("qkv", dev, leaves):
        _near(a.grad, w.grad, 1e-4, name)


@pytest.mark.parametrize("train", [False, True])
def test_masks_left_on_the_host(pkg, train):
    """A mask that was not moved to the GPU is refused, for each form that masks take to the kernels."""
    print(f"masks on the host train={train}", flush=True)
    mod = _module(pkg, 4, torch.float16, use_mask=True).requires_grad_(train)
    x = torch.randn(1, 4, 64, 64, dtype=torch.float16, device="cuda")
    rows = torch.arange(64)
    causal = (rows[None, :] <= rows[:, None])[None, None]
    holes = causal & ((rows[None, :] + rows[:, None]) % 5 != 1)
    for mask in (rows[None] < 50, torch.where(rows[None] < 50, 0.0, -1.0), causal & (rows < 50), causal & (rows[None, :] > rows[:, None] - 9), holes):
        with pytest.raises(RuntimeError):
            mod(x, x, x, mask, None)
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype,scores", [(torch.bfloat16, 5), (torch.float32, 6)])
def test_training_peak_memory(pkg, dtype, scores):
    """A training step holds the score tensors that backward needs (conv result, probabilities, post-softmax conv and mixing; the raw
    scores too where the first stage is two operators) and drops each where it is consumed: at the peak those and one gradient.
    Everything else is (B,H,S,D) or smaller: half a score tensor covers it (D = 64 against S = 2048, about ten tensors)."""
    print(f"training peak memory {dtype}", flush=True)
    b, h, s, d = 1, 4, 2048, 64
    mod = _module(pkg, h, dtype)
    q, k, v = (torch.randn(b, h, s, d, device="cuda", dtype=dtype).requires_grad_(True) for _ in range(3))
    go = torch.randn(b, s, h, d, device="cuda", dtype=dtype)

    def step():
        for t in (q, k, v, *mod.parameters()):
            t.grad = None
        mod(q, k, v, None, None).backward(go)

    step()
    for t in (q, k, v, *mod.parameters()):
        t.grad = None
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    step()
    one = b * h * s * s * q.element_size()
    peak = (torch.cuda.max_memory_allocated() - before) / one
    print(f"peak: {peak:.2f} score tensors", flush=True)
    assert peak <= scores + 0.5, peak


def test_backward_twice(pkg):
    """A graph that is kept gives the same gradients again; one that is not is refused the second time."""
    print("backward twice", flush=True)
    for s, use_mask in ((64, False), (45, True)):
        mod = _module(pkg, 4, torch.bfloat16, use_mask=use_mask)
        q, k, v = (torch.randn(2, 4, s, 64, device="cuda", dtype=torch.bfloat16).requires_grad_(True) for _ in range(3))
        mask = None
        if use_mask:
            rows = torch.arange(s, device="cuda")
            mask = ((rows[None, :] <= rows[:, None]) & (rows < s - 7))[None, None]
        out = mod(q, k, v, mask, None)
        leaves = (q, k, v, *mod.parameters())
        first = torch.autograd.grad(out, leaves, torch.ones_like(out), retain_graph=True)
        again = torch.autograd.grad(out, leaves, torch.ones_like(out))
        assert all(torch.equal(a, w) for a, w in zip(first, again))
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(out, leaves, torch.ones_like(out))


def test_gradients_of_some_inputs(pkg):
    """Each input alone wanting a gradient, and through saved-tensor hooks: as all together."""
    print("gradients of some inputs", flush=True)
    mod = _module(pkg, 4, torch.float16).requires_grad_(False)
    base = [torch.randn(2, 4, 61, 64, device="cuda", dtype=torch.float16) for _ in range(3)]
    params = list(mod.parameters())

    def grads(wanted):
        x = [t.clone().requires_grad_("qkv"[i] in wanted) for i, t in enumerate(base)]
        for i, p in enumerate(params):
            p.requires_grad_(str(i) in wanted)
            p.grad = None
        mod(*x, None, None).float().square().sum().backward()
        return {n: t.grad for n, t in zip("qkv0123", [*x, *params])}

    every = grads("qkv0123")
    for one in "qkv0123":
        got = grads(one)
        assert all((t is None) == (n != one) for n, t in got.items())
        assert torch.equal(got[one], every[one]), one
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.clone())[1], lambda t: t):
        got = grads("qkv0123")
    assert all(torch.equal(got[n], t) for n, t in every.items())
    assert sum(len(sh) == 4 and sh[2] == sh[3] for sh in packed) >= 4     # the score tensors went through the hooks


@pytest.mark.parametrize("kind", ["none", "keys", "window", "left"])
@pytest.mark.parametrize("dtype,s", [(torch.bfloat16, 205), (torch.float32, 208)])
def test_training_by_one_node_or_several(pkg, dtype, s, kind):
    """A step whose score tensors are small is one autograd node, a larger one a node per score tensor: a batch on one side of the
    line against its halves on the other.  The products choose their tiling by the size of the grid: sums in another order."""
    print(f"one node or several {dtype} s={s} {kind}", flush=True)
    h, d = 4, 64
    s8 = (s + 7) // 8 * 8
    one = h * s8 * s8 * (2 if dtype == torch.bfloat16 else 4)
    b = ((16 << 20) // one + 2) // 2 * 2
    assert b * one > (16 << 20) and b // 2 * one <= (16 << 20)
    mod = _module(pkg, h, dtype, use_mask=kind != "none")
    x = [torch.randn(b, h, s, d, device="cuda", dtype=dtype) for _ in range(3)]
    go = torch.randn(b, s, h, d, device="cuda", dtype=dtype)
    rows = torch.arange(s, device="cuda")
    mask = (rows[None, :] <= rows[:, None])[None, None].expand(b, 1, s, s).clone()
    if kind == "keys":
        mask[1::2, ..., s - 20:] = False
    elif kind == "window":
        mask &= rows[None, :] > rows[:, None] - 50
    elif kind == "left":
        mask[1::2, ..., :30] = False
        go[1::2, :30] = 0

    def step(at):
        leaves = [t[at].clone().requires_grad_(True) for t in x]
        for p in mod.parameters():
            p.grad = None
        out = mod(*leaves, None if kind == "none" else mask[at], None)
        out.backward(go[at])
        return [out.detach(), *(t.grad for t in leaves)], [p.grad.float() for p in mod.parameters()]

    whole, whole_w = step(slice(None))
    first, first_w = step(slice(0, b // 2))
    second, second_w = step(slice(b // 2, None))
    rel = {torch.float32: 1e-5, torch.bfloat16: 5e-3}[dtype]
    for name, a, f, t in zip("out q k v".split(), whole, first, second):
        _near(a, torch.cat([f, t]).cpu(), rel, name)
    for name, a, f, t in zip(_WEIGHTS, whole_w, first_w, second_w):
        _near(a, (f + t).cpu(), rel * 2, name)


@pytest.mark.parametrize("b", [2, 52])
def test_training_dropout(pkg, b):
    """Dropout on the last score tensor, one node (b = 2) and several: the output is linear in V, so out . go = dV . V for the mask
    that was drawn, and the same seed draws it again."""
    print(f"training dropout b={b}", flush=True)
    mod = _module(pkg, 4, torch.float32)
    mod.dropout = 0.25
    x = [torch.randn(b, 4, 205, 64, device="cuda").requires_grad_(True) for _ in range(3)]
    go = torch.randn(b, 205, 4, 64, device="cuda")
    grads = []
    for _ in range(2):
        torch.manual_seed(5)
        out = mod(*x, None, None)
        grads.append(torch.autograd.grad(out, [*x, *mod.parameters()], go))
        a, w = (out.detach().double() * go.double()).sum(), (grads[-1][2].double() * x[2].detach().double()).sum()
        assert abs(float(a - w)) <= 1e-5 * float((out.detach().double() * go.double()).norm()) * out.numel() ** 0.5
    assert all(torch.isfinite(t).all() for t in grads[0])
    assert all(torch.equal(a, w) for a, w in zip(*grads))


@pytest.mark.parametrize("s", [64, 45])
def test_tangent_of_the_values(pkg, s):
    """Inference with a dual V: the output is linear in V, and its tangent is the output for V's tangent (a whole and an odd length,
    without a mask and under key padding)."""
    import torch.autograd.forward_ad as fw
    for use_mask in (False, True):
        print(f"tangent of the values s={s} mask={use_mask}", flush=True)
        mod = _module(pkg, 4, torch.float32, use_mask=use_mask).requires_grad_(False)
        q, k, v, t = (torch.randn(2, 4, s, 64, device="cuda") for _ in range(4))
        rows = torch.arange(s, device="cuda")
        mask = ((rows[None, :] <= rows[:, None]) & (rows < s - 7))[None, None] if use_mask else None
        want, tangent = mod(q, k, v, mask, None), mod(q, k, t, mask, None)
        with fw.dual_level():
            got = fw.unpack_dual(mod(q, k, fw.make_dual(v, t), mask, None))
            _near(got.primal, want.cpu(), 1e-5)
            _near(got.tangent, tangent.cpu(), 1e-5)


@pytest.mark.parametrize("mask", [None, "keys", "window", "holes"])
@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
                                          (torch.float16, torch.float16), (torch.float16, torch.float32)])
def test_autocast(pkg, dtype, wdtype, mask):
    """Under torch.autocast the products of Q K^T and P V that the library would do come out in autocast's dtype, whichever kernel
    does them, and so does the output; the scores kernel with weights of its own dtype is no library product.  Backward runs
    inside and outside, the gradients have the inputs' dtypes."""
    amp = torch.float16
    for s in (64, 45):
        print(f"autocast {dtype} {wdtype} {mask} s={s}", flush=True)
        if mask == "holes" and s % 8:
            continue
        # (16-bit data of another dtype than autocast's: only where the scores kernel takes it, the general kernels take one dtype)
        own = dtype == wdtype and dtype != torch.float32 and s % 8 == 0 and mask != "holes"
        if mask is not None and not own and dtype == torch.bfloat16:
            continue
        mod = _module(pkg, 4, dtype, wdtype, use_mask=mask is not None)
        g = torch.Generator().manual_seed(9)
        q, k, v = (torch.randn(2, 4, s, 64, generator=g).to(dtype) for _ in range(3))
        rows = torch.arange(s)
        visible = (rows[None, :] <= rows[:, None])[None, None]
        if mask == "keys":
            visible = visible & (rows < s - 7)
        elif mask == "window":
            visible = visible & (rows[None, :] > rows[:, None] - 17)
        elif mask == "holes":
            visible = visible & ((rows[None, :] + rows[:, None]) % 5 != 1)
        want, leaves = _oracle(mod, q, k, v, mask=torch.where(visible, 0.0, float("-inf")).expand(2, 4, s, s))
        want.sum().backward()
        given = None if mask is None else visible.cuda()
        dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
        expect = dtype if own else amp
        rel = _REL[torch.bfloat16 if torch.bfloat16 in (dtype, expect) else torch.float16]
        with torch.autocast("cuda", dtype=amp), torch.no_grad():
            plain = mod(*dev, given, None)
        with torch.autocast("cuda", dtype=amp):     # (a context of its own: autocast keeps the casts it has made without a graph)
            out = mod(*dev, given, None)
            inside = torch.autograd.grad(out.float().sum(), dev, retain_graph=True)
        assert plain.dtype == out.dtype == expect
        _near(plain, want, rel, "inference")
        _near(out, want, rel, "training")
        outside = torch.autograd.grad(out.float().sum(), dev)
        for grads in (inside, outside):
            for name, a, w in zip("qkv", grads, leaves):
                assert a.dtype == dtype
                _near(a, w.grad, 4 * rel, name)


@pytest.mark.parametrize("dtype,ks", [(torch.bfloat16, (3, 5)), (torch.float16, (7, 9)), (torch.float32, (3, 5)), (torch.bfloat16, (11, 15))])
def test_left_padded_batches_of_every_kernel_size(pkg, dtype, ks):
    """A band mask whose padding rows see nothing takes the band route whatever the conv kernel: output against the oracle, gradients
    against the mask passes on the same mask (the reference's are NaN there)."""
    print(f"left padding {dtype} {ks}", flush=True)
    b, h, s, d = 2, 4, 136, 64
    mod = _module(pkg, h, dtype, use_mask=True, query_kernel_size=ks[0], key_kernel_size=ks[1])
    g = torch.Generator().manual_seed(10)
    q, k, v = (torch.randn(b, h, s, d, generator=g).to(dtype) for _ in range(3))
    keep = torch.arange(s)[None, :] >= torch.tensor([0, 37])[:, None]
    visible = keep[:, None, None, :] & torch.tril(torch.ones(s, s, dtype=torch.bool))[None, None]
    want, _ = _oracle(mod, q, k, v, mask=torch.where(visible, 0.0, float("-inf")).expand(b, h, s, s))
    dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    go = torch.randn(b, s, h, d, generator=g).to(dtype).cuda()
    go[1, :37] = 0
    seen, grads = [], []
    mod._stage_hook = seen.append
    with torch.no_grad():
        plain = mod(*dev, visible.cuda(), None)
    assert "mask" not in seen
    _near(plain, want, _REL[dtype], "inference")
    assert not plain[1, :37].any()
    for passes in (False, True):
        if passes:
            mod._band_training_supported = lambda *a: False
        seen.clear()
        out = mod(*dev, visible.cuda(), None)
        assert ("mask" in seen) == passes
        _near(out, want, _REL[dtype], "training")
        grads.append(torch.autograd.grad(out, [*dev, *mod.parameters()], go))
    for a, w in zip(*grads):
        _near(a, w.cpu(), 10 * _REL[dtype])


def test_observer_hears_the_kernels_that_run(pkg):
    """One mark per kernel: the fp32 one-pass mixing and softmax of more than 8 heads is one stage, in inference and in training, and
    conv + mixing of 16 heads is two where the grid makes it two kernels.  The figures of a stage are those of what it names."""
    print("observer", flush=True)
    for dtype, s, want in ((torch.float32, 64, ["qk", "conv_pre", "mix_softmax", "conv_post", "mix_post", "pv", "end"]),
                           (torch.float16, 64, ["qk_conv", "mix_softmax", "conv_post", "mix_post", "pv", "end"]),
                           (torch.float16, 2048, ["qk_conv", "mix_softmax", "conv_mix_post", "pv", "end"])):
        mod = _module(pkg, 16, dtype)
        x = [torch.randn(1, 16, s, 64, device="cuda", dtype=dtype) for _ in range(3)]
        seen = []
        mod._stage_hook = seen.append
        with torch.no_grad():
            mod(*x, None, None)
        assert seen == want
        if dtype == torch.float32:
            seen.clear()
            mod(*x, None, None)
            assert seen == want
            with torch.no_grad():
                mod.mta_conv_after_sm_triton.weight.zero_()[:, -1, 1] = 1.0
                mod.declare_weight_structure(post_conv_identity=True)
                seen.clear()
                mod(*x, None, None)
            assert seen == ["qk", "conv_pre", "mix_softmax_mix", "pv", "end"]


@pytest.mark.parametrize("dtype,d,dv", [(torch.float32, 64, 128), (torch.float32, 128, 32), (torch.float16, 64, 128), (torch.float16, 128, 32),
                                        (torch.float32, 32, 64)])
def test_values_of_another_head_size(pkg, dtype, d, dv):
    """V of another head size than Q and K, one the P V kernels know or not: a whole and a padded length."""
    for s in (64, 45):
        print(f"values of another head size {dtype} {d} {dv} s={s}", flush=True)
        mod = _module(pkg, 4, dtype)
        g = torch.Generator().manual_seed(12)
        q, k, v = (torch.randn(2, 4, s, n, generator=g).to(dtype) for n in (d, d, dv))
        want, leaves = _oracle(mod, q, k, v)
        dev = [t.cuda().requires_grad_(True) for t in (q, k, v)]
        with torch.inference_mode():
            _near(mod(*dev, None, None), want, _REL[dtype], "inference")
        out = mod(*dev, None, None)
        _near(out, want, _REL[dtype], "training")
        go = torch.randn(want.shape, generator=g)
        want.backward(go.to(dtype).float())
        out.backward(go.to(dtype).cuda())
        for name, a, w in zip("qkv", dev, leaves):
            _near(a.grad, w.grad, {torch.float32: 1e-4, torch.float16: 1e-2}[dtype], name)


def test_calls_that_stay_refused(pkg):
    """Empty tensors and functorch transforms: an exception, nothing launched."""
    print("refused calls", flush=True)
    for train in (False, True):
        for dtype in (torch.float32, torch.float16):
            mod = _module(pkg, 4, dtype).requires_grad_(train)
            for shape in ((0, 4, 64, 64), (2, 4, 0, 64), (0, 4, 45, 64)):
                x = torch.zeros(shape, device="cuda", dtype=dtype)
                with pytest.raises(ValueError):
                    mod(x, x, x, None, None)
            x = torch.zeros(3, 2, 4, 64, 64, device="cuda", dtype=dtype)
            for call in (lambda t: mod(t, t, t, None, None), lambda t: mod.mta_conv_triton(t), lambda t: mod.wpsm_triton(t)):
                with pytest.raises(RuntimeError):
                    torch.func.vmap(call)(x)
    torch.cuda.synchronize()


def test_anomaly_mode(pkg):
    """torch.autograd.detect_anomaly over a step whose score tensors are large: what lies above the diagonal between the stages, memory
    that nobody wrote (here: NaN), is not taken for a gradient."""
    print("anomaly mode", flush=True)
    mod = _module(pkg, 4, torch.bfloat16)
    q, k, v = (torch.randn(1, 4, 2048, 64, device="cuda", dtype=torch.bfloat16).requires_grad_(True) for _ in range(3))
    poison = [torch.full((1, 4, 2048, 2048), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(12)]
    del poison
    with torch.autograd.detect_anomaly():
        out = mod(q, k, v, None, None)
        out.sum().backward()
    assert all(torch.isfinite(t.grad).all() for t in (q, k, v, *mod.parameters()))


@pytest.mark.parametrize("name", ["mta_conv_triton", "mta_conv_after_sm_triton", "wposm_triton"])
def test_anomaly_mode_of_one_weight(pkg, name):
    """A step over large score tensors in which one weight wants a gradient: anomaly mode, whose step is one node, forms that gradient alone as
    the other nodes do - the same bits, where the kernel for both gradients of a conv adds up in another order."""
    print(f"anomaly mode of {name}", flush=True)
    mod = _module(pkg, 4, torch.float32).requires_grad_(False)
    weight = getattr(mod, name).weight.requires_grad_(True)
    q, k, v = (torch.randn(1, 4, 1280, 64, device="cuda") for _ in range(3))   # (26 MB a score tensor)
    grads = []
    for anomaly in (False, True):
        weight.grad = None
        with torch.autograd.set_detect_anomaly(anomaly):
            mod(q, k, v, None, None).square().sum().backward()
        grads.append(weight.grad)
    assert torch.equal(*grads)
