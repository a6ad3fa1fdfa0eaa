"""What a program built on this package has it do, as cases that can be timed and compared.

Six kinds of work, all through the public surface (``SillyLinear``, ``SillyEmbedding``, ``RT_GPT``):

infer      a matrix-coef layer's forward under ``no_grad``: a served model, one token at a time up to a prompt
train      a matrix-coef layer's forward and backward through autograd, with or without the fused random bias
mlp        the MNIST-shaped classifier, forward, loss and backward: the smallest training step, bound by launches and the host
vector     the reference's own form, one coefficient vector per tensor (``SillyLinear``'s default): materialise, dense products,
           gradient of the coefficients
embedding  lookup in a pseudorandom table and the gradient of its coefficients
gpt        a training step of the GPT-2-shaped model, every block's linears random-backed

Sizes are those of this repository's configurations (784 -> 256 -> 10; 768 -> 3072, k = 256, 8192 tokens; 4096 -> 4096, k = 16;
4096 -> 14336, k = 1024; GPT-2 small) and of its tests, and the ranges around them.
"""
import math

import torch
import torch.nn.functional as F

from randumb_amd import SillyEmbedding, SillyLinear
from randumb_amd.gpt import RT_GPT, RT_GPTConfig

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # a served fp32 model generating one sequence: GEMV-like, latency and launches are everything
        {"name": "decode_fp32_1tok", "kind": "infer", "tokens": 1, "in_f": 4096, "out_f": 4096, "k": 16, "dtype": "fp32"},
        # a served bf16 model generating for a small batch
        {"name": "decode_bf16_16tok", "kind": "infer", "tokens": 16, "in_f": 4096, "out_f": 11008, "k": 256, "dtype": "bf16"},
        # a prompt, not a round number of tokens long, through a square layer
        {"name": "prefill_bf16_2000tok", "kind": "infer", "tokens": 2000, "in_f": 4096, "out_f": 4096, "k": 256, "dtype": "bf16"},
        # 784 -> 256 -> 10, batch 128, fp32: the smallest configuration, as a training step
        {"name": "mlp_fp32_step", "kind": "mlp", "tokens": 128, "in_f": 784, "hidden": 256, "out_f": 10, "k": 64},
        # the headline layer as a model built from layers pays for it
        {"name": "fc_bf16_train", "kind": "train", "tokens": 8192, "in_f": 768, "out_f": 3072, "k": 256, "dtype": "bf16", "rt_bias": False},
        # the layer whose stored weight would have 58.7 M elements
        {"name": "llm_bf16_train", "kind": "train", "tokens": 4096, "in_f": 4096, "out_f": 14336, "k": 1024, "dtype": "bf16", "rt_bias": False},
        # no size a multiple of anything: ragged tiles, rows that are not 16-byte aligned
        {"name": "odd_bf16_train", "kind": "train", "tokens": 4097, "in_f": 1001, "out_f": 999, "k": 100, "dtype": "bf16", "rt_bias": False},
        # torch's default dtype; a micro-batch
        {"name": "fc_fp32_train", "kind": "train", "tokens": 2048, "in_f": 768, "out_f": 3072, "k": 256, "dtype": "fp32", "rt_bias": False},
        # the reference's default initialisation trains the scale of a full-rank random bias beside the coefficients
        {"name": "rbias_bf16_train", "kind": "train", "tokens": 8192, "in_f": 768, "out_f": 3072, "k": 256, "dtype": "bf16", "rt_bias": True},
        # the reference's layer as it stands: k hashed values per weight element, dense products by the library
        {"name": "vector_fp32_train", "kind": "vector", "tokens": 1024, "in_f": 768, "out_f": 3072, "k": 256},
        # GPT-2's token table, 4 sequences of 1024
        {"name": "embedding_train", "kind": "embedding", "tokens": 4096, "vocab": 50304, "dim": 768, "k": 256},
        # GPT-2 small, 12 layers, 48 random-backed linears, 8 x 1024 tokens
        {"name": "gpt2_small_step", "kind": "gpt", "batch": 8, "seq": 1024, "layers": 12, "heads": 12, "k": 256},
    ]


# ------------------------------------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi, odd):
    """A feature count: a multiple of 8 unless ``odd``, as nearly all layers' are."""
    n = _log(rng, lo, hi)
    return n if odd else max(8, (n + 4) // 8 * 8)


def _layer_sizes(rng, k_lo, k_hi, in_hi, out_hi):
    odd = rng.random() < 0.2
    in_f, out_f = _size(rng, 256, in_hi, odd), _size(rng, 256, out_hi, odd)
    k = _size(rng, k_lo, min(k_hi, in_f // 2, out_f // 2), odd)   # the coefficients are fewer than what they stand for
    return in_f, out_f, k


def draw(rng):
    kind = rng.choices(["infer", "train", "mlp", "vector", "embedding", "gpt"], [5, 7, 2, 2, 2, 2])[0]
    if kind == "infer":
        in_f, out_f, k = _layer_sizes(rng, 16, 512, 8192, 11008)
        return {"kind": kind, "tokens": _log(rng, 1, 2048), "in_f": in_f, "out_f": out_f, "k": k, "dtype": rng.choice(["bf16", "bf16", "fp32"])}
    if kind == "train":
        in_f, out_f, k = _layer_sizes(rng, 32, 1024, 4096, 8192)
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return {"kind": kind, "tokens": _log(rng, 256, 4096 if dtype == "fp32" else 8192), "in_f": in_f, "out_f": out_f, "k": k, "dtype": dtype,
                "rt_bias": dtype == "bf16" and rng.random() < 0.25}
    if kind == "mlp":
        return {"kind": kind, "tokens": _log(rng, 32, 512), "in_f": _log(rng, 196, 3072), "hidden": _log(rng, 64, 512), "out_f": _log(rng, 10, 100),
                "k": _log(rng, 16, 128)}
    if kind == "vector":
        return {"kind": kind, "tokens": _log(rng, 64, 2048), "in_f": _log(rng, 196, 1024), "out_f": _log(rng, 196, 3072), "k": _log(rng, 16, 256)}
    if kind == "embedding":
        return {"kind": kind, "tokens": _log(rng, 64, 4096), "vocab": 50304, "dim": _size(rng, 64, 768, False), "k": _size(rng, 16, 256, False)}
    return {"kind": kind, "batch": rng.randint(1, 8), "seq": _size(rng, 64, 1024, False), "layers": rng.randint(1, 12), "heads": rng.randint(4, 12),
            "k": _size(rng, 32, 256, False)}


# ------------------------------------------------------------------------------------------------ what the program has in hand
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _coefs(layer, std, g):
    """C ~ N(0, 3*std^2/k): the weight then has standard deviation ``std``."""
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, math.sqrt(3.0 / layer.weight_coef.shape[-1]) * std, generator=g)
        if getattr(layer, "bias_coef", None) is not None:
            layer.bias_coef.normal_(0.0, math.sqrt(3.0 / layer.bias_coef.shape[-1]) * std, generator=g)


def _randn(g, dtype, *shape):
    return torch.randn(*shape, device="cuda", generator=g).to(dtype)


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("infer", "train"):
        dtype, k = _DTYPES[case["dtype"]], case["k"]
        layer = SillyLinear(case["in_f"], case["out_f"], [k, k], [seed % 1000, seed % 1000 + 1], bias=False, rt_bias=case.get("rt_bias", False),
                            device="cuda", dtype=dtype, matrix_coef=True)
        _coefs(layer, 1.0 / math.sqrt(case["in_f"]), g)
        s.update(layer=layer, x=_randn(g, dtype, case["tokens"], case["in_f"]))
        if kind == "train":
            s["x"].requires_grad_()
            s["dy"] = _randn(g, dtype, case["tokens"], case["out_f"])
            s["wanted"] = [s["x"], layer.weight_coef] + ([layer.weight_scale_bias] if case["rt_bias"] else [])
    elif kind == "mlp":
        k = case["k"]
        first = SillyLinear(case["in_f"], case["hidden"], [k, k], [1337, 1338], device="cuda", matrix_coef=True)
        second = SillyLinear(case["hidden"], case["out_f"], [k, k], [1339, 1340], device="cuda", matrix_coef=True)
        _coefs(first, 1.0 / math.sqrt(3.0 * case["in_f"]), g)
        _coefs(second, 1.0 / math.sqrt(3.0 * case["hidden"]), g)
        s.update(first=first, second=second, x=torch.rand(case["tokens"], case["in_f"], device="cuda", generator=g),
                 target=torch.randint(0, case["out_f"], (case["tokens"],), device="cuda", generator=g),
                 wanted=[first.weight_coef, first.bias_coef, second.weight_coef, second.bias_coef])
    elif kind == "vector":
        k = case["k"]
        layer = SillyLinear(case["in_f"], case["out_f"], [k, k], [seed % 1000, seed % 1000 + 1], device="cuda")
        _coefs(layer, 1.0 / math.sqrt(case["in_f"]), g)
        x = _randn(g, torch.float32, case["tokens"], case["in_f"]).requires_grad_()
        s.update(layer=layer, x=x, dy=_randn(g, torch.float32, case["tokens"], case["out_f"]), wanted=[x, layer.weight_coef, layer.bias_coef])
    elif kind == "embedding":
        table = SillyEmbedding(case["vocab"], case["dim"], [case["k"]], [seed % 1000], device="cuda")
        _coefs(table, 0.02, g)
        s.update(table=table, idx=torch.randint(0, case["vocab"], (case["tokens"],), device="cuda", generator=g),
                 dy=_randn(g, torch.float32, case["tokens"], case["dim"]), wanted=[table.weight_coef])
    else:
        n = 4 * case["layers"]
        with torch.device("cuda"):
            model = RT_GPT(RT_GPTConfig(int_dim_gen=iter([case["k"]] * n), seed_gen=iter(range(n)), n_layer=case["layers"], n_head=case["heads"],
                                        n_embd=64 * case["heads"])).to(torch.bfloat16)
        with torch.no_grad():
            for m in model.modules():
                if isinstance(m, SillyLinear):
                    _coefs(m, 0.02, g)
            model.wte.weight.normal_(0.0, 1.0, generator=g)
            model.lm_head.weight.normal_(0.0, 0.02, generator=g)
        tokens = torch.randint(0, 50304, (case["batch"], case["seq"] + 1), device="cuda", generator=g)
        s.update(model=model, idx=tokens[:, :-1].contiguous(), target=tokens[:, 1:].contiguous())
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    kind = s["kind"]
    if kind == "infer":
        with torch.no_grad():
            return s["layer"](s["x"])
    if kind in ("train", "vector"):
        y = s["layer"](s["x"])
        return [y.detach(), *torch.autograd.grad(y, s["wanted"], s["dy"])]
    if kind == "mlp":
        logits = s["second"](F.relu(s["first"](s["x"])))
        loss = F.cross_entropy(logits, s["target"])
        return [loss.detach(), logits.detach(), *torch.autograd.grad(loss, s["wanted"])]
    if kind == "embedding":
        y = s["table"](s["idx"])
        return [y.detach(), *torch.autograd.grad(y, s["wanted"], s["dy"])]
    model = s["model"]
    model.zero_grad(set_to_none=True)
    loss = model(s["idx"], s["target"])
    loss.backward()
    return [loss.detach()] + [p.grad for p in model.parameters() if p.grad is not None]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _product_flops(tokens, in_f, out_f, k):
    """y = x.W^T with W = C.N: through the k coefficients, or through a weight formed first, whichever is less."""
    return min(2.0 * tokens * k * (in_f + out_f), 2.0 * tokens * in_f * out_f + 2.0 * in_f * out_f * k)


def _train_flops(tokens, in_f, out_f, k):
    """Forward, input gradient, and the coefficients' gradient from the forward pass's x.N^T."""
    return 2.0 * _product_flops(tokens, in_f, out_f, k) + 2.0 * tokens * out_f * k


def work(case):
    """Bytes: inputs read once, outputs written once, coefficients and their gradients.  Flops: multiplications and additions of
    the products; the integer arithmetic of the hash (some 13 operations a value) comes on top and is what bounds ``vector``
    and ``embedding``: k hashed values per element and direction."""
    kind = case["kind"]
    if kind in ("infer", "train"):
        size = 2.0 if case["dtype"] == "bf16" else 4.0
        t, i, o, k = case["tokens"], case["in_f"], case["out_f"], case["k"]
        once = t * (i + o) + o * k
        if kind == "infer":
            return {"bytes": size * once, "flops": _product_flops(t, i, o, k)}
        full = 6.0 * t * i * o if case["rt_bias"] else 0.0   # the bias has full rank: one more product each way, the scale's gradient from one of them
        return {"bytes": size * 2 * once, "flops": _train_flops(t, i, o, k) + full * 2.0 / 3.0}
    if kind == "mlp":
        t, i, h, o, k = case["tokens"], case["in_f"], case["hidden"], case["out_f"], case["k"]
        first = _product_flops(t, i, h, k) + 2.0 * t * h * k   # no gradient of the images
        return {"bytes": 4.0 * (t * (i + o) + 2 * (h + o + 2) * k) + 8.0 * t, "flops": first + _train_flops(t, h, o, k)}
    if kind == "vector":
        t, i, o, k = case["tokens"], case["in_f"], case["out_f"], case["k"]
        return {"bytes": 4.0 * 2 * (t * (i + o) + 2 * k), "flops": 6.0 * t * i * o + 4.0 * i * o * k}
    if kind == "embedding":
        t, d, k = case["tokens"], case["dim"], case["k"]
        return {"bytes": 8.0 * t + 4.0 * 2 * (t * d + k), "flops": 4.0 * t * d * k}
    t, d, k, v, n = case["batch"] * case["seq"], 64 * case["heads"], case["k"], 50304, case["layers"]
    linears = _train_flops(t, d, 3 * d, k) + _train_flops(t, d, d, k) + _train_flops(t, d, 4 * d, k) + _train_flops(t, 4 * d, d, k)
    attention = 3.5 * 4.0 * t * case["seq"] * d / 2   # two products forward, five backward, half of each under the causal mask
    saved = 2.0 * t * d * 2 * 22   # bf16 activations of a block that the backward pass reads again, written and read once
    params = 2.0 * (2 * v * d + n * 12 * d * k)
    return {"bytes": n * saved + 2.0 * params + 2 * 2.0 * t * v + 16.0 * t, "flops": n * (linears + attention) + 6.0 * t * d * v}


def tolerance(case):
    kind = case["kind"]
    if kind == "gpt":
        # bf16 roundings of a whole model, forwards and back: another normalisation alone (fp32 inside, rounded once) moves the
        # first layers' gradients by 1.6e-2, another attention by 1.1e-2
        return {"rel": 2.5e-2}
    if kind in ("infer", "train") and case["dtype"] == "bf16":
        return {"rel": 1e-2}
    return {"rel": 2e-5 if kind == "mlp" else 1e-5}   # fp32 sums; the classifier's gradients pass through two layers and the loss
