"""The work this framework is used for, as cases that can be timed: Multi-Token-Attention modules in inference and in
training, the two operators they are made of, and the fused conv-attention module, each through its public class.

A case is a dict of plain values:

    op       "mta" (MTAAttentionTriton), "conv" (Conv2dTriton), "headmix" (TritonLinearHead), "conv_attn"
             (TritonConvAttention)
    train    forward and backward, with the gradients of every input and weight; else the forward under no_grad
    b h s d  batch, heads (channels), sequence length, head size (0 where there is none)
    dtype    of the activations; weights: "same", or "float32" (16-bit activations from autocast, fp32 master weights)
    r k      rows and keys of the (pre-softmax) conv kernel; r2, k2 of the post-softmax one, 0 = the identity tap
    group    mixing groups of that many heads, declared to the module; 0 = dense head weights, nothing declared
    mask     "none"; "padding" (a right-padded batch as a (B,1,S,S) boolean mask); "window" (a sliding window over the
             last quarter of the longest row)
"""
from __future__ import annotations

import math

import torch

import multitokenatention_triton_amd as mta

_FIELDS = ("op", "train", "b", "h", "s", "d", "dtype", "weights", "r", "k", "r2", "k2", "group", "mask")


def _case(name, *values):
    case = dict(zip(_FIELDS, values))
    return dict(case, name=name) if name else case


def listed():
    return [
        # one attention layer of a small model, a short prompt: latency and launches are all there is
        _case("mta_fwd_small_fp32", "mta", False, 1, 4, 256, 64, "float32", "same", 3, 5, 0, 0, 2, "none"),
        # a training step of such a layer, default kernel sizes, dense head weights
        _case("mta_train_small_bf16", "mta", True, 1, 8, 256, 64, "bfloat16", "same", 3, 3, 3, 3, 0, "none"),
        # ordinary prompt in fp32 with large kernels before and after the softmax
        _case("mta_fwd_1k_fp32", "mta", False, 1, 16, 1024, 64, "float32", "same", 11, 15, 11, 15, 0, "none"),
        # a batch of prompts whose lengths are whatever the text gave: an odd number of tokens
        _case("mta_fwd_ragged_bf16", "mta", False, 2, 16, 1001, 64, "bfloat16", "same", 6, 11, 3, 3, 0, "none"),
        # a batch of prompts of different lengths, padded on the right, known weight structure
        _case("mta_fwd_padded_bf16", "mta", False, 4, 16, 1024, 128, "bfloat16", "same", 6, 11, 0, 0, 4, "padding"),
        # long prefill with sparse structure: identity stages skipped, heads mixed in groups of 4 (the headline workload)
        _case("mta_fwd_4k_bf16", "mta", False, 2, 16, 4096, 128, "bfloat16", "same", 6, 11, 0, 0, 4, "none"),
        # long prefill of a trained model: all four weights dense
        _case("mta_fwd_4k_dense_fp16", "mta", False, 1, 16, 4096, 128, "float16", "same", 7, 7, 7, 7, 0, "none"),
        # training of the same kind of layer in 16 bits ...
        _case("mta_train_2k_fp16", "mta", True, 1, 16, 2048, 128, "float16", "same", 7, 7, 7, 7, 0, "none"),
        # ... and in fp32
        _case("mta_train_1k_fp32", "mta", True, 1, 32, 1024, 64, "float32", "same", 5, 5, 5, 5, 0, "none"),
        # the two operators alone, as a module of somebody else's attention uses them: forward and both gradients
        _case("conv_train_2k_bf16", "conv", True, 2, 16, 2048, 0, "bfloat16", "same", 6, 11, 0, 0, 0, "none"),
        _case("headmix_train_2k_bf16", "headmix", True, 2, 32, 2048, 0, "bfloat16", "same", 0, 0, 0, 0, 4, "none"),
        # fused conv-attention over a long sequence, no score tensor in memory
        _case("conv_attn_8k_bf16", "conv_attn", False, 1, 32, 8192, 128, "bfloat16", "same", 6, 11, 0, 0, 0, "none"),
    ]


_KERNELS = ((3, 3), (3, 5), (5, 5), (5, 7), (6, 11), (7, 7), (7, 9), (11, 15))
# elements of one score tensor that a drawn case has at most (the fp32 and training cases keep several of them)
_MOST = {False: 2 * 16 * 4096 ** 2, True: 32 * 2048 ** 2}
_MOST_FP32 = {False: 16 * 2048 ** 2, True: 16 * 2048 ** 2}


def _length(rng, low, high):
    """A sequence length, spread over its logarithm: most are multiples of 64 or 8, one in four is whatever comes."""
    s = math.exp(rng.uniform(math.log(low), math.log(high)))
    step = rng.choice((64, 64, 8, 1))
    return max(low, int(s) // step * step)


def draw(rng):
    """One more case of the ranges that the listed ones stand for."""
    top = work(listed()[-1])["flops"]
    while True:
        op = rng.choice(("mta",) * 12 + ("conv",) * 2 + ("headmix",) * 2 + ("conv_attn",) * 3)
        dtype = rng.choice(("bfloat16", "bfloat16", "bfloat16", "float16", "float16", "float32", "float32"))
        b, h, d = rng.choice((1, 1, 2, 4)), rng.choice((4, 8, 12, 16, 16, 32)), rng.choice((64, 128))
        train = rng.random() < (0.0 if op == "conv_attn" else 0.4 if op == "mta" else 0.6)
        s = _length(rng, 64, 8192 if op == "conv_attn" else 4096)
        weights = "float32" if train and dtype != "float32" and rng.random() < 0.15 else "same"
        (r, k), (r2, k2), group, mask = rng.choice(_KERNELS), (0, 0), 0, "none"
        if op == "mta":
            if train or rng.random() < 0.6:
                r2, k2 = (r, k) if rng.random() < 0.5 else (3, 3)
            if not train:
                group = rng.choice((0, 0, 2, 4, 4, h))
            mask = rng.choice(("none",) * 6 + ("padding", "padding", "window"))
        elif op == "headmix":
            r = k = d = 0
            group = rng.choice((0, 2, 4))
        elif op == "conv":
            d = 0
        case = _case(None, op, train, b, h, s, d, dtype, weights, r, k, r2, k2, group, mask)
        most = (_MOST_FP32 if dtype == "float32" else _MOST)[train]
        if (op == "conv_attn" or b * h * s * s <= most) and work(case)["flops"] <= (top / 16 if dtype == "float32" else top):
            return case


def _conv_weight(shape, g, dtype):
    """N(0, 0.05) around the pass-through tap."""
    w = 0.05 * torch.randn(shape, generator=g, device="cuda")
    w[:, -1, shape[2] // 2] += 1.0
    return w.to(dtype)


def _head_weight(h, group, g, dtype):
    """The identity plus N(0, 0.1), block diagonal where there are groups."""
    w = torch.eye(h, device="cuda") + 0.1 * torch.randn(h, h, generator=g, device="cuda")
    if group:
        block = torch.arange(h, device="cuda") // group
        w = w * (block[:, None] == block[None, :])
    return w.to(dtype)


def _mask(kind, b, s, g):
    """(B,1,S,S) or (1,1,S,S), True = attend."""
    if kind == "none":
        return None
    at = torch.arange(s, device="cuda")
    causal = at[None, :] <= at[:, None]
    if kind == "window":
        return (causal & (at[None, :] > at[:, None] - max(1, s // 4)))[None, None]
    lengths = torch.randint((s + 1) // 2, s + 1, (b,), generator=g, device="cuda")
    return (causal[None] & (at[None, None, :] < lengths[:, None, None]))[:, None]


def prepare(case, seed):
    c = dict(case)
    b, h, s, d, op, train = c["b"], c["h"], c["s"], c["d"], c["op"], c["train"]
    dtype = getattr(torch, c["dtype"])
    wdtype = dtype if c["weights"] == "same" else getattr(torch, c["weights"])
    g = torch.Generator(device="cuda").manual_seed(seed)
    normal = lambda *shape: torch.randn(shape, generator=g, device="cuda").to(dtype)  # noqa: E731
    mask = None
    if op == "mta":
        cfg = mta.MTAConfig(query_kernel_size=c["r"], key_kernel_size=c["k"], after_sm_query_kernel_size=c["r2"] or 3,
                            after_sm_key_kernel_size=c["k2"] or 3)
        mask = _mask(c["mask"], b, s, g)
        module = mta.MTAAttentionTriton(h, cfg, dropout=0.0, causal=True, use_mask=mask is not None).to("cuda", wdtype)
        with torch.no_grad():
            module.mta_conv_triton.weight.copy_(_conv_weight((h, c["r"], c["k"]), g, wdtype))
            if c["r2"]:
                module.mta_conv_after_sm_triton.weight.copy_(_conv_weight((h, c["r2"], c["k2"]), g, wdtype))
            else:
                module.mta_conv_after_sm_triton.weight.zero_()[:, -1, 1] = 1.0
            pre_identity = bool(c["group"]) and not c["r2"]
            module.wpsm_triton.weight.copy_(torch.eye(h) if pre_identity else _head_weight(h, c["group"], g, wdtype))
            module.wposm_triton.weight.copy_(_head_weight(h, c["group"], g, wdtype))
        if c["group"] and not train:
            module.infer_weight_structure()
        inputs = [normal(b, h, s, d) for _ in range(3)]
        grad = normal(b, s, h, d)
    elif op == "conv_attn":
        module = mta.TritonConvAttention(h, (c["r"], c["k"]), causal=True).to("cuda", wdtype)
        with torch.no_grad():
            module.weight.copy_(_conv_weight((h, c["r"], c["k"]), g, wdtype))
        inputs, grad = [normal(b, h, s, d) for _ in range(3)], None
    else:
        if op == "conv":      # scores, nothing above the diagonal
            module = mta.Conv2dTriton(h, (c["r"], c["k"]), causal=True).to("cuda", wdtype)
            weight = _conv_weight((h, c["r"], c["k"]), g, wdtype)
            x = torch.randn((b, h, s, s), generator=g, device="cuda").tril_()
        else:                 # rows of probabilities
            module = mta.TritonLinearHead(h, causal=True, group_size=c["group"] or None).to("cuda", wdtype)
            weight = _head_weight(h, c["group"], g, wdtype)
            x = torch.randn((b, h, s, s), generator=g, device="cuda")
            x.masked_fill_(torch.ones(s, s, dtype=torch.bool, device="cuda").triu_(1), float("-inf"))
            x = torch.softmax(x, -1)
        with torch.no_grad():
            module.weight.copy_(weight)
        inputs, grad = [x.to(dtype)], normal(b, h, s, s)
    module.train(train)
    for x in inputs:
        x.requires_grad_(train)
    return {"op": op, "train": train, "module": module, "inputs": inputs, "mask": mask, "grad": grad if train else None}


def _forward(state):
    module, inputs = state["module"], state["inputs"]
    if state["op"] == "mta":
        return module(*inputs, state["mask"], None)
    if state["op"] == "conv_attn":
        return module(*inputs, True, None)[0]
    return module(*inputs)


def run(state):
    if not state["train"]:
        with torch.no_grad():
            return _forward(state)
    leaves = [*state["inputs"], *state["module"].parameters()]
    for x in leaves:
        x.grad = None
    out = _forward(state)
    out.backward(state["grad"])
    return [out.detach(), *(x.grad for x in leaves)]


def work(case):
    """What one pass cannot do without.  Bytes: inputs, weights and outputs (a training step: the gradients too), each
    once, and of the operators' (B,H,S,S) operands that follow the causal rule the lower triangle where they are read.
    Flops: the products on and below the diagonal; a training step has two more of each, and the scores it does not keep
    are not counted again."""
    b, h, s, d, train, op = case["b"], case["h"], case["s"], case["d"], case["train"], case["op"]
    size = 4 if case["dtype"] == "float32" else 2
    wsize = size if case["weights"] == "same" else 4
    lower, passes = b * h * s * (s + 1) // 2, 3 if train else 1
    mix = case["group"] or h
    if op in ("mta", "conv_attn"):
        flops = lower * (4 * d + 2 * case["r"] * case["k"])
        tensors, weights = 4 * b * h * s * d, h * case["r"] * case["k"]
        if op == "mta":
            flops += lower * 2 * (case["r2"] * case["k2"] + 2 * mix)
            weights += h * (case["r2"] * case["k2"] + 2 * mix)
        bytes_ = (2 * tensors if train else tensors) * size + (2 if train else 1) * weights * wsize
        if case["mask"] == "padding":
            bytes_ += b * s * s
        elif case["mask"] == "window":
            bytes_ += s * s
        return {"bytes": bytes_, "flops": passes * flops}
    full = b * h * s * s
    taps = case["r"] * case["k"] if op == "conv" else mix
    weights = h * taps
    bytes_ = (lower + full) * size + weights * wsize
    if train:   # dy read once for both gradients, dx written
        bytes_ += (lower + full) * size + weights * wsize
    return {"bytes": bytes_, "flops": passes * 2 * taps * lower}


def tolerance(case):
    """One rounding to the data type is 2^-9 (bf16) or 2^-12 (fp16) of a value; a pass has a handful one after another,
    the scores' among them, which the exponential turns into relative errors of their own size.  fp32: the order of sums."""
    return {"rel": {"float32": 1e-5, "float16": 2e-3, "bfloat16": 1e-2}[case["dtype"]]}
