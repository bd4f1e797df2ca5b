"""CPU-only: calls of the modules that do not fit together are refused ahead of the first stage - with the exception that names
the misfit, not with the one that says there is no CPU path - so that no kernel reads an operand beyond its end."""
import pytest
import torch

import multitokenatention_triton_amd as mta


def _module(h=4, dtype=torch.float32, train=False, **kw):
    mod = mta.MTAAttentionTriton(h, mta.MTAConfig(), 0.0, True, **kw).to(dtype).requires_grad_(train)
    mod.reset_mta_parameters()
    seen = []
    mod._stage_hook = seen.append
    return mod, seen


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("q,k,v,error,match", [
    ((2, 4, 16, 64), (2, 4, 16, 64), (2, 8, 16, 64), RuntimeError, "must match"),      # V of more heads
    ((2, 4, 16, 64), (2, 4, 16, 64), (4, 4, 16, 64), RuntimeError, "must match"),      # ... of more batch entries
    ((2, 4, 16, 64), (2, 4, 16, 64), (2, 4, 24, 64), RuntimeError, "share their length"),
    ((2, 4, 13, 64), (2, 4, 13, 64), (2, 4, 16, 64), RuntimeError, "share their length"),
    ((2, 4, 16, 64), (2, 3, 16, 64), (2, 4, 16, 64), RuntimeError, "must match"),      # K of other heads
    ((2, 4, 16, 64), (2, 4, 16, 128), (2, 4, 16, 64), RuntimeError, "head size"),
    ((2, 4, 16, 64), (4, 16, 64), (2, 4, 16, 64), ValueError, "expected Q, K, V"),
])
def test_products_that_do_not_exist(q, k, v, error, match, dtype, train):
    mod, seen = _module(dtype=dtype, train=train)
    with pytest.raises(error, match=match):
        mod(*(torch.zeros(s, dtype=dtype) for s in (q, k, v)), None, None)
    assert seen == []


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads", [1, 2, 8])
def test_weights_of_other_head_counts(heads, dtype, train):
    """A module of 4 heads given tensors of more or fewer: the conv and head kernels index their weights by the data's heads.
    With the structure declared the stages that would notice later are skipped."""
    for declare in (False, True):
        mod, seen = _module(dtype=dtype, train=train)
        if declare:
            mod.declare_weight_structure(pre_head_identity=True, post_conv_identity=True, post_head_identity=True)
        x = torch.zeros(2, heads, 16, 64, dtype=dtype)
        with pytest.raises(AssertionError, match="heads of Q and K"):
            mod(x, x, x, None, None)
        assert seen == []


@pytest.mark.parametrize("name", ["mta_conv_triton", "wpsm_triton", "mta_conv_after_sm_triton", "wposm_triton"])
def test_a_weight_of_another_head_count(name):
    for train in (False, True):
        mod, seen = _module(train=train)
        part = getattr(mod, name)
        w = part.weight
        part.weight = torch.nn.Parameter(torch.zeros(8, *((8,) if w.dim() == 2 else w.shape[1:])), requires_grad=train)
        x = torch.zeros(2, 4, 16, 64)
        with pytest.raises(AssertionError, match="heads of Q and K"):
            mod(x, x, x, None, None)
        assert seen == []


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("s", [13, 16])
def test_key_masks_that_do_not_fit(s, train):
    """2-D key masks of another length (also one that pads to the same multiple of 8) and on another device: the kernels read one
    value per key from the pointer they are given."""
    mod, seen = _module(train=train, use_mask=True)
    x = torch.zeros(1, 4, s, 64)
    for n in (1, s - 1, s + 1, 8):
        for mask in (torch.ones(1, n, dtype=torch.bool), torch.zeros(1, n)):
            with pytest.raises(RuntimeError, match="does not match the"):
                mod(x, x, x, mask, None)
    with pytest.raises(RuntimeError, match="key mask lives on meta"):
        mod(x, x, x, torch.ones(1, s, dtype=torch.bool, device="meta"), None)
    assert seen == []


@pytest.mark.parametrize("train", [False, True])
def test_mask_rows_that_do_not_fit(train):
    """The same for the arrays the module hands to its native routes: batch, length, dtype and device, ahead of the first stage."""
    mod, seen = _module(train=train)
    x = torch.zeros(2, 4, 13, 64)     # (causal: 16 columns)
    good = {"key_bias": torch.zeros(2, 16), "first_visible": torch.zeros(2, 16, dtype=torch.int32), "empty_rows": torch.zeros(2, 16, dtype=torch.bool)}
    for name, t in good.items():
        for bad in (t[:1], t[:, :13], t[:, :8], t[0], t.double(), torch.zeros(3, 16, dtype=t.dtype)):
            with pytest.raises(ValueError, match="must be"):
                mod._forward_native(x, x, x, **{name: bad})
        with pytest.raises(RuntimeError, match="lives on meta"):
            mod._forward_native(x, x, x, **{name: t.to("meta")})
    with pytest.raises(RuntimeError, match="live on"):
        mod(x, x, x.to("meta"), None, None)
    assert seen == []


@pytest.mark.parametrize("train", [False, True])
def test_forward_mode_is_refused(train):
    """The kernels know no tangents: a dual tensor is refused whether or not something else wants a gradient."""
    import torch.autograd.forward_ad as fw
    x, s = torch.zeros(2, 4, 16, 64), torch.zeros(2, 4, 16, 16)
    conv = mta.Conv2dTriton(4, 3, causal=True).requires_grad_(train)
    mix = mta.TritonLinearHead(4).requires_grad_(train)
    attn = mta.TritonConvAttention(4, 3, causal=True).requires_grad_(train)
    mod, seen = _module(train=True)
    with fw.dual_level(), torch.set_grad_enabled(train):
        ds, dx = fw.make_dual(s, torch.ones_like(s)), fw.make_dual(x, torch.ones_like(x))
        for call in (lambda: conv(ds), lambda: mix(ds)):
            with pytest.raises(NotImplementedError):
                call()
        if not train:
            for operands in ((dx, x, x), (x, dx, x), (x, x, dx)):
                with pytest.raises(NotImplementedError):
                    attn(*operands, True, None)
    with fw.dual_level():
        dx = fw.make_dual(x, torch.ones_like(x))
        for operands in ((dx, x, x), (x, dx, x), (x, x, dx)):
            with pytest.raises(NotImplementedError):
                mod(*operands, None, None)
    assert seen == []
