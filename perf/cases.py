"""Workloads that the speed of this library is judged by, run through its public Python operators.

Four kinds of pass, named by a case's ``kind``:

* ``forward``: one ``dot_product_attention`` call (prefill, cross-attention, decoding);
* ``train``: the forward call and its gradient, as a training step of an attention layer makes them;
* ``product``: ``batched_mul``, alone or with its pullback;
* ``softmax``: ``softmax`` / ``logsoftmax`` over one dimension, alone or with the gradient.

``listed()`` holds one case of each way the library is used, ``draw()`` makes others of the same ranges: head dims
and sequence lengths that are no multiple of anything among them.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "nnlib.jl_amd"))
import nnlib_amd as nn  # noqa: E402

TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def attention(kind, dtype, D, H, Lq, Lkv, B, causal=False, weights=False, mask="none", bias="none", dropout=0.0, name=None):
    """``mask``: "padding" keeps the first keys of each sequence, (Lkv, 1, 1, B); "dense" drops a tenth of the pairs,
    (Lkv, Lq).  ``bias``: "full" has an entry per score, "shared" one for all sequences of the batch, (Lkv, Lq, H)."""
    case = dict(kind=kind, dtype=dtype, D=D, H=H, Lq=Lq, Lkv=Lkv, B=B, causal=causal, weights=weights, mask=mask,
                bias=bias, dropout=dropout)
    return dict(case, name=name) if name else case


def product(dtype, m, n, k, batch, ta=False, tb=False, shared=False, pullback=False, name=None):
    """(m, k, batch) times (k, n, batch); ``ta`` / ``tb``: that operand is a lazily transposed array; ``shared``: the
    left operand is one matrix for the whole batch."""
    case = dict(kind="product", dtype=dtype, m=m, n=n, k=k, batch=batch, ta=ta, tb=tb, shared=shared, pullback=pullback)
    return dict(case, name=name) if name else case


def softmax(dtype, inner, length, outer, log, grad, name=None):
    """An array (inner, length, outer), or (length, outer) where inner is 1, reduced over ``length``."""
    case = dict(kind="softmax", dtype=dtype, inner=inner, length=length, outer=outer, log=log, grad=grad)
    return dict(case, name=name) if name else case


def listed():
    return [
        # a layer of a small encoder at inference, called as the reference is (Float32, weights returned): 32 (head,
        # batch) pairs of 128 x 128 leave most of the chip idle, so this is launches and host work
        attention("forward", "f32", 64, 8, 128, 128, 4, weights=True, name="encoder_small_f32"),
        # prompt processing of a decoder: the software-pipelined 16-bit kernel, bound by the matrix cores
        attention("forward", "bf16", 128, 32, 4096, 4096, 2, causal=True, name="prefill_causal_bf16"),
        # cross-attention with an additive bias per score and a random mask: a stream over the bias
        attention("forward", "f16", 64, 16, 256, 8192, 4, mask="dense", bias="full", name="cross_bias_mask_f16"),
        # one step of text generation against a long context: a stream over K and V
        attention("forward", "bf16", 128, 32, 1, 32768, 16, name="decode_long_context_bf16"),
        # training step of a decoder layer in 16 bits
        attention("train", "bf16", 128, 32, 4096, 4096, 2, causal=True, name="train_causal_bf16"),
        # training step in the reference's default element type, weights returned as the reference always does
        attention("train", "f32", 64, 16, 1024, 1024, 8, causal=True, weights=True, name="train_causal_weights_f32"),
        # training step of an encoder on a padded batch of sentences with dropout; the lengths are ragged
        attention("train", "bf16", 64, 12, 333, 333, 24, mask="padding", dropout=0.1, name="train_padded_dropout_bf16"),
        # training step of an encoder on image patches (14 x 14 and a class token) with a learned relative-position
        # bias per head, whose gradient is wanted too
        attention("train", "bf16", 64, 12, 197, 197, 64, bias="shared", name="train_position_bias_bf16"),
        # batched products, 16 bits, sizes the matrix cores like
        product("bf16", 2048, 2048, 2048, 16, name="batched_mul_bf16"),
        # batched products of odd sizes with a lazily transposed operand, and their pullback
        product("f32", 333, 517, 77, 96, ta=True, pullback=True, name="batched_mul_odd_pullback_f32"),
        # the last layer of a classifier: class scores along dimension 1, forward and gradient
        softmax("f32", 1, 10000, 4096, True, True, name="logsoftmax_classes_f32"),
        # softmax over the middle dimension, a strided reduction
        softmax("bf16", 256, 4096, 128, False, False, name="softmax_dims2_bf16"),
    ]


# ---- drawn cases -----------------------------------------------------------------------------------------------------

def spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm: half of them as they fall, half of them multiples of 8."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and x >= 8:
        x -= x % 8
    return max(lo, min(hi, x))


def few(case, field, most):
    """``case`` with ``field`` (then the heads) lowered until the pass moves and computes no more than ``most`` =
    (bytes, flops)."""
    for name in (field, "H"):
        while case.get(name, 1) > 1 and (work(case)["bytes"] > most[0] or work(case)["flops"] > most[1]):
            case[name] = max(1, case[name] * 3 // 4)
    return case


def draw(rng):
    kind = rng.choice(("encoder", "prefill", "cross", "decode", "train16", "train32", "padded", "bias", "product",
                       "product_odd", "softmax1", "softmax2"))
    head = rng.choice((32, 48, 64, 64, 80, 96, 128, 128))
    heads = rng.choice((4, 6, 8, 12, 16, 32))
    half = rng.choice(("bf16", "bf16", "f16"))
    if kind == "encoder":
        n = spread(rng, 16, 512)
        c = attention("forward", "f32", head, heads, n, n, spread(rng, 1, 32), causal=rng.random() < 0.3,
                      weights=rng.random() < 0.7, mask=rng.choice(("none", "none", "padding")))
        return few(c, "B", (7e8, 4e10))
    if kind == "prefill":
        n = spread(rng, 128, 8192)
        c = attention("forward", half, head, heads, n, n, spread(rng, 1, 16), causal=rng.random() < 0.7,
                      mask=rng.choice(("none", "none", "padding")))
        return few(c, "B", (2e9, 6e11))
    if kind == "cross":
        c = attention("forward", half, head, heads, spread(rng, 16, 1024), spread(rng, 64, 8192), spread(rng, 1, 16),
                      mask=rng.choice(("none", "padding", "dense")), bias=rng.choice(("none", "shared", "full")))
        return few(c, "B", (6e8, 3e11))
    if kind == "decode":
        c = attention("forward", rng.choice(("bf16", "bf16", "f16", "f32")), rng.choice((64, 128)), heads,
                      rng.choice((1, 1, 1, 1, 2, 4)), spread(rng, 512, 32768), spread(rng, 1, 32),
                      mask=rng.choice(("none", "padding")))
        return few(c, "B", (8e9, 1e12))
    if kind == "train16":
        n = spread(rng, 128, 4096)
        c = attention("train", half, head, heads, n, n, spread(rng, 1, 32), causal=rng.random() < 0.6)
        return few(c, "B", (2e9, 9.5e11))
    if kind == "train32":
        n = spread(rng, 32, 1024)
        c = attention("train", "f32", head, heads, n, n, spread(rng, 1, 32), causal=rng.random() < 0.5,
                      weights=rng.random() < 0.5)
        return few(c, "B", (1.5e9, 8e10))
    if kind == "padded":
        n = spread(rng, 32, 1024)
        c = attention("train", half, head, heads, n, n, spread(rng, 4, 64), mask="padding",
                      dropout=rng.choice((0.0, 0.1)))
        return few(c, "B", (1e9, 3e11))
    if kind == "bias":
        n = spread(rng, 49, 577)
        c = attention("train", half, head, heads, n, n, spread(rng, 4, 64), bias="shared")
        return few(c, "B", (6e8, 1e11))
    if kind == "product":
        shared = rng.random() < 0.2
        c = product(half, 8 * spread(rng, 8, 256), 8 * spread(rng, 8, 256), 8 * spread(rng, 4, 256), spread(rng, 1, 256),
                    ta=rng.random() < 0.3, tb=rng.random() < 0.3, shared=shared, pullback=not shared and rng.random() < 0.4)
        return few(c, "batch", (1.5e9, 6e11))
    if kind == "product_odd":
        dtype = rng.choice(("f32", "f32", half))
        c = product(dtype, spread(rng, 16, 1024), spread(rng, 16, 1024), spread(rng, 16, 1024), spread(rng, 1, 256),
                    ta=rng.random() < 0.3, tb=rng.random() < 0.3, shared=dtype == "f32" and rng.random() < 0.2,
                    pullback=rng.random() < 0.5)
        return few(c, "batch", (1e9, 1e11))
    if kind == "softmax1":
        c = softmax(rng.choice(("f32", "f32", half)), 1, spread(rng, 16, 131072), spread(rng, 16, 65536),
                    rng.random() < 0.5, rng.random() < 0.5)
        return few(c, "outer", (2e9, 1e12))
    c = softmax(rng.choice(("f32", half)), spread(rng, 8, 1024), spread(rng, 16, 8192), spread(rng, 1, 256),
                rng.random() < 0.5, rng.random() < 0.5)
    return few(c, "outer", (1e9, 1e12))


# ---- one case --------------------------------------------------------------------------------------------------------

class Inputs:
    """Device arrays of normal values, made from one seed."""

    def __init__(self, seed, dtype):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.dtype = dtype

    def normal(self, *dims, scale=1.0):
        t = torch.randn(math.prod(dims), generator=self.gen, device="cuda", dtype=TORCH[self.dtype])
        return nn.DeviceArray.from_torch(t if scale == 1.0 else t * scale, dims, self.dtype)

    def kept(self, share, *dims):
        t = torch.rand(math.prod(dims), generator=self.gen, device="cuda") < share
        return nn.DeviceArray.from_torch(t.to(torch.uint8), dims, "bool")

    def prefixes(self, L, B):
        """A key-padding mask: sequence b keeps its first keys, between half and all of them."""
        n = torch.randint(L // 2, L, (B, 1), generator=self.gen, device="cuda") + 1
        t = (torch.arange(L, device="cuda")[None, :] < n).to(torch.uint8)
        return nn.DeviceArray.from_torch(t.contiguous(), (L, 1, 1, B), "bool")


def prepare(case, seed):
    c, make = case, Inputs(seed, case["dtype"])
    state = {"case": c}
    if c["kind"] in ("forward", "train"):
        E, Lq, Lkv, H, B = c["D"] * c["H"], c["Lq"], c["Lkv"], c["H"], c["B"]
        state.update(q=make.normal(E, Lq, B), k=make.normal(E, Lkv, B), v=make.normal(E, Lkv, B))
        if c["kind"] == "train":
            state["dy"] = make.normal(E, Lq, B)
        state["bias"] = None if c["bias"] == "none" else make.normal(Lkv, Lq, H, B if c["bias"] == "full" else 1, scale=0.5)
        mask = None if c["mask"] == "none" else make.kept(0.9, Lkv, Lq) if c["mask"] == "dense" else make.prefixes(Lkv, B)
        if c["causal"]:
            causal = nn.make_causal_mask(state["q"])
            mask = causal if mask is None else causal & mask
        state["mask"] = mask
        state["fdrop"] = nn.Dropout(c["dropout"], seed) if c["dropout"] else nn.identity
    elif c["kind"] == "product":
        na = 1 if c["shared"] else c["batch"]
        m, n, k, b = c["m"], c["n"], c["k"], c["batch"]
        state["A"] = nn.batched_transpose(make.normal(k, m, na)) if c["ta"] else make.normal(m, k, na)
        state["B"] = nn.batched_transpose(make.normal(n, k, b)) if c["tb"] else make.normal(k, n, b)
        if c["pullback"]:
            state["dC"] = make.normal(m, n, b)
    else:
        dims = (c["length"], c["outer"]) if c["inner"] == 1 else (c["inner"], c["length"], c["outer"])
        state["x"] = make.normal(*dims, scale=2.0)
        if c["grad"]:
            state["dy"] = make.normal(*dims)
    return state


def run(state):
    """One pass.  Arrays come back as the device tensors that own their (column-major) memory."""
    c = state["case"]
    if c["kind"] in ("forward", "train"):
        s = state
        train = c["kind"] == "train"
        y, alpha = nn.dot_product_attention(s["q"], s["k"], s["v"], s["bias"], fdrop=s["fdrop"], mask=s["mask"],
                                            nheads=c["H"], return_weights=c["weights"], save_for_backward=train)
        out = {"y": y}
        if alpha is not None:
            out["alpha"] = alpha
        if train:
            grads = nn.dot_product_attention_grad(s["dy"], s["q"], s["k"], s["v"], s["bias"], y=y, mask=s["mask"],
                                                  nheads=c["H"], fdrop=s["fdrop"])
            out.update((n, g) for n, g in zip(("dq", "dk", "dv", "dbias"), grads) if g is not None)
    elif c["kind"] == "product":
        out = {"C": nn.batched_mul(state["A"], state["B"])}
        if c["pullback"]:
            out["dA"], out["dB"] = nn.batched_mul_pullback(state["A"], state["B"], state["dC"])
    else:
        dims = 1 if c["inner"] == 1 else 2
        forward, backward = (nn.logsoftmax, nn.grad_logsoftmax) if c["log"] else (nn.softmax, nn.grad_softmax)
        out = {"y": forward(state["x"], dims=dims)}
        if c["grad"]:
            out["dx"] = backward(state["dy"], out["y"], dims=dims)
    return {name: a.storage for name, a in out.items()}


def work(case):
    """Every input read once, every output written once; two operations per multiply-add of the products, which are two
    forward and five in the gradient of attention.  Pairs above a causal diagonal count for nothing."""
    c, size = case, SIZE[case["dtype"]]
    if c["kind"] in ("forward", "train"):
        E, Lq, Lkv, H, B = c["D"] * c["H"], c["Lq"], c["Lkv"], c["H"], c["B"]
        pairs = Lq * (Lq + 1) // 2 if c["causal"] else Lq * Lkv
        scores = Lq * Lkv * H
        rows = E * B * (2 * Lq + 2 * Lkv)                     # q, y, k, v
        bias = {"none": 0, "shared": scores, "full": scores * B}[c["bias"]]
        nbytes = size * (rows + bias + (scores * B if c["weights"] else 0))
        nbytes += {"none": 0, "padding": Lkv * B, "dense": Lkv * Lq}[c["mask"]]
        flops = 4 * c["D"] * H * B * pairs
        if c["kind"] == "train":
            nbytes += size * E * B * (2 * Lq + 2 * Lkv) + 4 * bias   # dy, dq, dk, dv; the bias gradient is Float32
            flops += 10 * c["D"] * H * B * pairs
        return {"bytes": nbytes, "flops": flops}
    if c["kind"] == "product":
        m, n, k, b = c["m"], c["n"], c["k"], c["batch"]
        a = m * k * (1 if c["shared"] else b)
        nbytes, flops = a + k * n * b + m * n * b, 2 * m * n * k * b
        if c["pullback"]:
            nbytes, flops = nbytes + a + k * n * b + m * n * b, 3 * flops
        return {"bytes": size * nbytes, "flops": flops}
    n = c["inner"] * c["length"] * c["outer"]
    return {"bytes": size * n * (4 if c["grad"] else 2), "flops": n * (10 if c["grad"] else 5)}


def tolerance(case):
    """About four times the largest relative error (2-norm) of any output against the same pass in 64 bits, over the
    listed cases and 60 drawn ones: 5.6e-7 in Float32, 3.6e-4 in Float16, 3.0e-3 in BFloat16."""
    return {"rel": {"f32": 2.5e-6, "f16": 1.5e-3, "bf16": 1.2e-2}[case["dtype"]]}
