"""The kernels around a block's linears (randumb_amd/csrc/rdb_block.hip, rdb_attention.hip) against the stock operators they
replace, in fp32 or fp64 on the same bf16 inputs, at sizes around their tiles' edges."""
import math

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
EPS = torch.finfo(torch.float32).eps


@pytest.fixture(scope="module")
def ext():
    from randumb_amd import _lib

    return _lib.extension()


def rel(a, b):
    a, b = a.detach().double(), b.detach().double()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


def bf16(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).bfloat16()


@pytest.mark.parametrize("rows,dim", [(1, 4), (3, 64), (5, 260), (130, 768), (7, 1024), (2, 2052), (3, 4096)])
def test_rms_norm_and_residual(ext, rows, dim):
    print(f"case rms norm {rows} x {dim}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(dim)
    x, d, dy, ds = (bf16(g, rows, dim, scale=s) for s in (1.0, 0.5, 1.0, 1.0))
    leaves = [t.clone().requires_grad_() for t in (x, d)]
    ref = [t.double().requires_grad_() for t in (x, d)]
    s, y = ext.add_rms_norm(*leaves, EPS)
    assert torch.equal(s, x + d)
    rs = (ref[0] + ref[1])
    rs = rs + (s.double() - rs).detach()   # the sum is rounded to bf16 before it is normalised
    ry = F.rms_norm(rs, (dim,), eps=EPS)
    assert rel(y, ry) < 3e-3
    got = torch.autograd.grad([s, y], leaves, [ds, dy])
    want = torch.autograd.grad([rs, ry], ref, [ds.double(), dy.double()])
    assert torch.equal(got[0], got[1]) and rel(got[0], want[0]) < 5e-3
    p, q = x.clone().requires_grad_(), x.double().requires_grad_()
    y, ry = ext.rms_norm(p, EPS), F.rms_norm(q, (dim,), eps=EPS)
    assert rel(y, ry) < 3e-3
    if dim > 4:   # with so few values the gradient is what is left of a cancellation
        assert rel(torch.autograd.grad(y, p, dy)[0], torch.autograd.grad(ry, q, dy.double())[0]) < 5e-3


@pytest.mark.parametrize("n", [1, 7, 8, 2047, 5000, 1 << 20])
def test_relu_square_is_the_stock_chain_bit_for_bit(ext, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    x, dy = bf16(g, n), bf16(g, n)
    x[0] = math.nan
    a, b = x.clone().requires_grad_(), x.clone().requires_grad_()
    ya, yb = ext.relu_square(a), F.relu(b).square()
    assert torch.equal(ya.nan_to_num(7), yb.nan_to_num(7)) and bool(ya[0].isnan())
    ga, gb = torch.autograd.grad(ya, a, dy)[0], torch.autograd.grad(yb, b, dy)[0]
    assert torch.equal(ga.nan_to_num(7), gb.nan_to_num(7))


@pytest.mark.parametrize("offset", [1, 2, 4, 6])
@pytest.mark.parametrize("op", ["rms_norm", "add_rms_norm", "relu_square", "cross_entropy", "causal_attention"])
def test_slices_that_begin_between_the_boundaries_of_wide_loads(ext, op, offset):
    """Contiguous inputs and gradients `offset` values behind a 16-byte boundary: the results of aligned ones."""
    g = torch.Generator(device="cuda").manual_seed(offset)

    def at(t, off):
        buf = torch.empty(t.numel() + 16, device="cuda", dtype=t.dtype)
        return buf[off : off + t.numel()].view(t.shape).copy_(t)

    x, d = bf16(g, 2, 9, 192), bf16(g, 2, 9, 192)
    t = torch.randint(0, 192, (18,), device="cuda", generator=g)
    inv = torch.ones(32, device="cuda")
    f = {"rms_norm": lambda a, b: ext.rms_norm(a, EPS), "add_rms_norm": lambda a, b: ext.add_rms_norm(a, b, EPS)[1], "relu_square": lambda a, b: ext.relu_square(a),
         "cross_entropy": lambda a, b: ext.cross_entropy(a.view(18, 192), t, -100), "causal_attention": lambda a, b: ext.causal_attention(a, inv, 1, EPS)}[op]
    out = []
    for off in (0, offset):
        a, b = at(x, off).requires_grad_(), at(d, off)
        y = f(a, b)
        dy = at(torch.arange(y.numel(), device="cuda").remainder(7).to(y.dtype).view(y.shape) - 3, off if y.dim() else 0)
        out.append([y.detach(), torch.autograd.grad(y, a, dy)[0]])
    assert a.data_ptr() % 16 != 0
    for p, q in zip(*out):
        assert torch.equal(p, q)


def test_relu_square_with_gradients_that_are_not_finite(ext):
    """Where x <= 0 the stock operators pass nothing on, an infinite gradient included."""
    v = torch.tensor([-2.0, -0.0, 0.0, 1.5, math.inf, -math.inf, math.nan], device="cuda").bfloat16()
    x, dy = (t.flatten() for t in torch.meshgrid(v, v, indexing="ij"))
    a, b = x.clone().requires_grad_(), x.clone().requires_grad_()
    ga, gb = torch.autograd.grad(ext.relu_square(a), a, dy)[0], torch.autograd.grad(F.relu(b).square(), b, dy)[0]
    assert torch.equal(ga.isnan(), gb.isnan()) and torch.equal(ga.nan_to_num(7), gb.nan_to_num(7))


@pytest.mark.parametrize("rows,classes", [(1, 8), (3, 64), (130, 2056), (1025, 4096), (64, 50304)])
def test_cross_entropy(ext, rows, classes):
    print(f"case cross entropy {rows} x {classes}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(classes)
    x = bf16(g, rows, classes, scale=3.0)
    t = torch.randint(0, classes, (rows,), generator=g, device="cuda")
    if rows > 2:
        t[1] = -100
        x[2, : classes // 2] = -math.inf
        t[2] = classes - 1
    a, b = x.clone().requires_grad_(), x.double().requires_grad_()
    la, lb = ext.cross_entropy(a, t, -100), F.cross_entropy(b, t)
    assert la.dtype == torch.float32 and la.shape == () and abs(float(la.detach()) - float(lb.detach())) < 1e-5 * abs(float(lb.detach()))
    ga, gb = torch.autograd.grad(la * 3, a)[0], torch.autograd.grad(lb * 3, b)[0]
    assert rel(ga, gb) < 3e-3
    if rows > 2:
        assert not bool(ga[1].any())
    assert torch.equal(torch.autograd.grad(ext.cross_entropy(a, t, -100) * 3, a)[0], ga)
    assert bool(ext.cross_entropy(x, torch.full_like(t, -100), -100).isnan())   # no row counts, as in the stock operator
    assert bool(ext.cross_entropy(x, torch.full_like(t, classes), -100).isnan())


@pytest.mark.parametrize("label", [-1, 2056, 1 << 40, -(1 << 40)])
def test_a_label_outside_the_classes_does_not_train(ext, label):
    """Its loss is NaN and so is its row of the gradient; the other rows' gradients are what they are."""
    g = torch.Generator(device="cuda").manual_seed(5)
    x = bf16(g, 9, 2056).requires_grad_()
    t = torch.randint(0, 2056, (9,), generator=g, device="cuda")
    t[3] = -100
    (ref,) = torch.autograd.grad(ext.cross_entropy(x, t, -100), x)
    t[4] = label
    loss = ext.cross_entropy(x, t, -100)
    (got,) = torch.autograd.grad(loss, x)
    assert bool(loss.isnan()) and bool(got[4].isnan().all())
    rest = [i for i in range(9) if i != 4]
    assert torch.equal(got[rest], ref[rest]) and not bool(got[3].any())


def _attention(qkv, inv_freq, H):
    """The stock operators of RT_CausalSelfAttention, in qkv's precision, with q, k rounded to bf16 as they are there."""
    from randumb_amd.gpt import Rotary

    B, T, D3 = qkv.shape
    q, k, v = qkv.view(B, T, 3, H, 64).unbind(2)

    def r16(t):   # value rounded to bf16, gradient passed on
        return t + (t.detach().bfloat16().to(t.dtype) - t.detach())

    freqs = torch.outer(torch.arange(T, device=qkv.device), inv_freq)
    cos, sin = freqs.cos().to(qkv.dtype)[None, :, None, :], freqs.sin().to(qkv.dtype)[None, :, None, :]

    def rot(x):
        x = r16(F.rms_norm(x, (64,), eps=EPS))
        x1, x2 = x.chunk(2, dim=3)
        return r16(torch.cat((x1 * cos + x2 * sin, x2 * cos - x1 * sin), 3))

    q, k = rot(q).transpose(1, 2), rot(k).transpose(1, 2)
    s = (q @ k.transpose(-1, -2).contiguous()) / 8.0
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=qkv.device).triu(1), -math.inf)
    assert Rotary is not None
    return (s.softmax(-1) @ v.transpose(1, 2).contiguous()).transpose(1, 2).reshape(B, T, H * 64)


@pytest.mark.parametrize("B,T,H,inv", [(1, 1, 1, "bf16"), (2, 31, 3, "fp32"), (1, 64, 2, "bf16"), (1, 65, 8, "bf16"), (2, 127, 1, "bf16"), (1, 129, 5, "fp32"),
                                       (2, 200, 4, "bf16"), (1, 384, 2, "bf16"), (1, 1000, 3, "bf16")])
def test_causal_attention(ext, B, T, H, inv):
    print(f"case attention B={B} T={T} H={H} {inv}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    qkv = bf16(g, B, T, 3 * H * 64, scale=0.7)
    dy = bf16(g, B, T, H * 64)
    f = (1.0 / 10000.0) ** (torch.arange(0, 64, 2, device="cuda") / 64)
    f = f.bfloat16() if inv == "bf16" else f
    a, b = qkv.clone().requires_grad_(), qkv.double().requires_grad_()
    ya, yb = ext.causal_attention(a, f, H, EPS), _attention(b, f, H)
    assert ya.shape == (B, T, H * 64) and rel(ya, yb) < 5e-3
    ga, gb = torch.autograd.grad(ya, a, dy)[0], torch.autograd.grad(yb, b, dy.double())[0]
    for part, (x, w) in enumerate(zip(ga.view(B, T, 3, -1).unbind(2), gb.view(B, T, 3, -1).unbind(2))):
        if T > 1 or part == 2:   # with one token there is no gradient in q and k but rounding
            assert rel(x, w) < 1.5e-2, part
    y2 = ext.causal_attention(a, f, H, EPS)
    assert torch.equal(y2, ya) and torch.equal(torch.autograd.grad(y2, a, dy)[0], ga)


# enough blocks for 128 rows each: forward and backward, backward alone, with two blocks to a head
@pytest.mark.parametrize("B,T,H,inv", [(8, 1100, 9, "bf16"), (5, 900, 11, "fp32"), (43, 129, 8, "bf16")])
def test_causal_attention_of_many_rows(ext, B, T, H, inv):
    test_causal_attention(ext, B, T, H, inv)


def test_model_with_and_without_the_fused_kernels(ext, monkeypatch):
    from randumb_amd import gpt

    torch.manual_seed(0)
    with torch.device("cuda"):
        model = gpt.RT_GPT(gpt.RT_GPTConfig(int_dim_gen=iter([32] * 8), seed_gen=iter(range(8)), vocab_size=512, n_layer=2, n_head=2, n_embd=128)).bfloat16()
    ids = torch.randint(0, 512, (2, 97), device="cuda")
    out = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(gpt, "_fused", lambda x: None)
        model.zero_grad(set_to_none=True)
        loss = model(ids[:, :-1].contiguous(), ids[:, 1:].contiguous())
        loss.backward()
        out.append([loss.detach()] + [p.grad for p in model.parameters() if p.grad is not None])
    assert len(out[0]) == len(out[1]) == 1 + 8 + 2
    assert abs(float(out[0][0]) - float(out[1][0])) < 1e-3 * float(out[1][0])
    for x, y in zip(out[0], out[1]):
        assert rel(x, y) < 2e-2


def test_blocks_that_share_their_normalisation():
    """Blocks with and without a hook (which sends a block through its ``forward``): the same bits in the loss and every gradient."""
    from randumb_amd import gpt

    torch.manual_seed(0)
    with torch.device("cuda"):
        model = gpt.RT_GPT(gpt.RT_GPTConfig(int_dim_gen=iter([32] * 12), seed_gen=iter(range(12)), vocab_size=512, n_layer=3, n_head=2, n_embd=128)).bfloat16()
        idx, target = torch.randint(0, 512, (2, 65)), torch.randint(0, 512, (2, 65))
    seen, results = [], []
    for hooked in ([], [1], [0, 1, 2]):
        handles = [model.h[i].register_forward_hook(lambda m, a, out: seen.append(out.shape)) for i in hooked]
        model.zero_grad(set_to_none=True)
        loss = model(idx, target)
        loss.backward()
        results.append([loss.detach()] + [p.grad for p in model.parameters() if p.grad is not None])
        for h in handles:
            h.remove()
    assert seen == [(2, 65, 128)] * 4
    for other in results[1:]:
        assert len(other) == len(results[0])
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))


def _loss_in_64_bits(model, idx, target):
    """RT_GPT.forward in fp64 on leaves that are the model's parameters: (loss, gradients in the parameters' order).  The angles of
    the rotary embedding are the bf16 ones the model has: they are what it computes, not how exactly."""
    from randumb_amd import hip

    leaves = {n: p.detach().double().requires_grad_() for n, p in model.named_parameters() if "scale_bias" not in n}

    def linear(x, name, layer):
        N = hip.sq5_fill_2d(layer.in_features, layer.weight_coef.shape[1], layer.seed[0]).double()
        return (x @ N) @ leaves[name + ".weight_coef"].t()

    def norm(x):
        return F.rms_norm(x, (x.size(-1),), eps=EPS)

    x = norm(leaves["wte.weight"][idx])
    B, T, D = x.shape
    for i, block in enumerate(model.h):
        H = block.attn.n_head
        freqs = torch.outer(torch.arange(T, device=x.device), block.attn.rotary.inv_freq)
        cos, sin = freqs.cos().double()[None, :, None, :], freqs.sin().double()[None, :, None, :]

        def rot(t):
            t1, t2 = norm(t).chunk(2, dim=3)
            return torch.cat((t1 * cos + t2 * sin, t2 * cos - t1 * sin), 3).transpose(1, 2)

        q, k, v = linear(norm(x), f"h.{i}.attn.c_qkv", block.attn.c_qkv).view(B, T, 3, H, 64).unbind(2)
        s = (rot(q) @ rot(k).transpose(-1, -2).contiguous()) / 8.0
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=x.device).triu(1), -math.inf)
        y = (s.softmax(-1) @ v.transpose(1, 2).contiguous()).transpose(1, 2).reshape(B, T, D)
        x = x + linear(y, f"h.{i}.attn.c_proj", block.attn.c_proj)
        x = x + linear(F.relu(linear(norm(x), f"h.{i}.mlp.c_fc", block.mlp.c_fc)).square(), f"h.{i}.mlp.c_proj", block.mlp.c_proj)
    loss = F.cross_entropy((norm(x) @ leaves["lm_head.weight"].t()).view(-1, leaves["lm_head.weight"].shape[0]), target.view(-1))
    return loss.detach(), dict(zip(leaves, torch.autograd.grad(loss, list(leaves.values()))))


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_the_fused_model_is_no_further_from_64_bits_than_the_stock_one(ext, monkeypatch, seed):
    """A bf16 training step with the fused kernels and with the stock operators around the same linears, each against the same
    model in fp64.  Their roundings are different ones, so single gradients may differ either way (a quarter); over all of them
    the fused step must not be further off (5 % for chance)."""
    from randumb_amd import gpt

    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = gpt.RT_GPT(gpt.RT_GPTConfig(int_dim_gen=iter([64] * 16), seed_gen=iter(range(16)), vocab_size=1024, n_layer=4, n_head=4, n_embd=256)).bfloat16()
        ids = torch.randint(0, 1024, (3, 193))
    with torch.no_grad():
        model.lm_head.weight.normal_(0.0, 0.02)
        for m in model.modules():
            if isinstance(m, gpt.RT_CastedLinear):
                m.weight_coef.mul_(2.0)
    idx, target = ids[:, :-1].contiguous(), ids[:, 1:].contiguous()
    exact_loss, exact = _loss_in_64_bits(model, idx, target)
    off = {}
    for fused in (True, False):
        if not fused:
            monkeypatch.setattr(gpt, "_fused", lambda x: None)
        model.zero_grad(set_to_none=True)
        loss = model(idx, target)
        loss.backward()
        off[fused] = {n: rel(p.grad, exact[n]) for n, p in model.named_parameters() if p.grad is not None and n in exact}
        off[fused]["loss"] = abs(float(loss.detach().double() - exact_loss) / float(exact_loss))
    grads = [n for n in off[True] if n != "loss"]
    assert len(grads) == 2 + 16
    ratios = {n: off[True][n] / off[False][n] for n in grads}
    mean = math.exp(sum(math.log(r) for r in ratios.values()) / len(ratios))
    print(f"  fused against stock, distance from 64 bits: gradients {mean:.3f} times, at most {max(ratios.values()):.3f}; "
          f"loss {off[True]['loss']:.2e} and {off[False]['loss']:.2e}; a gradient is off by {max(off[True][n] for n in grads):.1e}", flush=True)
    assert mean <= 1.05 and max(ratios.values()) <= 1.25, ratios
    # One number, so chance alone decides which loss is nearer.  A logit (0.3 typically) is off by some 1.4e-2 of itself, as the gradients
    # are; over 576 rows the mean is off by 4e-3 / 24 = 1.8e-4, 2.5e-5 of a loss of 6.9.  Four times that.
    assert off[True]["loss"] <= 1e-4 and off[False]["loss"] <= 1e-4


@pytest.mark.parametrize("dim,k,tokens", [(64, 64, 40), (192, 136, 700), (128, 264, 300), (72, 64, 520)])
@pytest.mark.parametrize("kind", ["all", "frozen coefficients", "frozen input", "saved elsewhere", "second derivative"])
def test_squared_relu_in_the_projections_node(dim, k, tokens, kind):
    """The activation in c_proj's autograd node against a c_proj with a hook, which is called for itself: bit for bit, also where dx is not stored through
    the activation's gradient (k > 256, features that are no whole lines)."""
    from randumb_amd.gpt import RT_GPTConfig, RT_MLP

    print(f"case squared ReLU in the projection's node dim={dim} k={k} {kind}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(dim)
    with torch.device("cuda"):
        mlp = RT_MLP(dim, RT_GPTConfig(int_dim_gen=iter([k, k]), seed_gen=iter([3, 4]))).bfloat16()
    with torch.no_grad():
        for m in (mlp.c_fc, mlp.c_proj):
            m.weight_coef.normal_(0.0, (3.0 / k) ** 0.5, generator=g)
    x, dy = bf16(g, 2, tokens // 2, dim).requires_grad_(), bf16(g, 2, tokens // 2, dim)
    leaves = [x, mlp.c_fc.weight_coef, mlp.c_proj.weight_coef]
    if kind == "frozen coefficients":
        leaves.pop().requires_grad_(False)
    if kind == "frozen input":
        x.requires_grad_(False), mlp.c_fc.weight_coef.requires_grad_(False)
        leaves = leaves[2:]

    def run():
        if kind == "saved elsewhere":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
                y = mlp(x)
        else:
            y = mlp(x)
        if kind == "second derivative":   # the layers have none: each of the first derivatives in what it depends on
            first = torch.autograd.grad(y, leaves, dy, create_graph=True)
            for of, leaf in ((0, 0), (0, 1), (0, 2), (1, 0), (1, 2), (2, 0), (2, 1)):
                with pytest.raises(RuntimeError, match="no second derivative"):
                    torch.autograd.grad(first[of].float().square().sum(), leaves[leaf], retain_graph=True)
            assert torch.autograd.grad(first[2].float().square().sum(), leaves[2], retain_graph=True, allow_unused=True) == (None,)   # dC = dy^T . z
            return y, [f.detach() for f in first]
        return y, torch.autograd.grad(y, leaves, dy)

    y, grads = run()
    assert "Projected" in y.grad_fn.name() or "Projected" in y.grad_fn.next_functions[0][0].name()
    seen = []
    hook = mlp.c_fc.register_forward_hook(lambda m, args, out: seen.append(out))   # the activation from its own kernel
    y1, grads1 = run()
    assert len(seen) == 1 and torch.equal(y, y1) and all(torch.equal(a, b) for a, b in zip(grads, grads1))
    hook.remove()
    mlp.c_proj.register_forward_hook(lambda m, args, out: seen.append(args[0]))
    y2, grads2 = run()
    assert len(seen) == 2 and torch.equal(y, y2) and all(torch.equal(a, b) for a, b in zip(grads, grads2))
    node = lambda t: t.grad_fn.next_functions[0][0].next_functions[0][0]
    assert not torch.is_grad_enabled() or kind == "frozen input" or "ReluSquare" not in str(node(y)) and "ReluSquare" in str([node(y2)] + [f[0] for f in node(y2).next_functions])


@pytest.mark.parametrize("dim,k,tokens", [(64, 64, 40), (192, 136, 700), (72, 64, 520)])
def test_second_derivative_of_the_squared_relu(ext, dim, k, tokens):
    """In the projection's node, whose layer has none: dx under create_graph depends on what feeds the activation as the stock operators' does, and on the
    coefficients by what raises."""
    from randumb_amd import ops

    print(f"case second derivative of the squared ReLU dim={dim} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(dim)
    h, dy, v, c = bf16(g, tokens, 4 * dim).requires_grad_(), bf16(g, tokens, dim), bf16(g, tokens, 4 * dim), bf16(g, dim, k)
    y = ext.relu_square_linear(h, c, 4 * dim, dim, 3)
    dx, = torch.autograd.grad(y, h, dy, create_graph=True)
    got, = torch.autograd.grad(dx, h, v)
    a = F.relu(h.detach()).square().requires_grad_()
    behind, = torch.autograd.grad(ops.linear(a, c, 4 * dim, dim, 4 * dim, 1, 3, None, None), a, dy)
    want_dx, want = behind.double() * 2 * F.relu(h).detach().double(), v.double() * behind.double() * 2 * (h > 0)
    for x, w in ((dx, want_dx), (got, want)):   # a few products of bf16 values, each rounded
        assert bool(((x.detach().double() - w).abs() <= 2.0**-6 * w.abs()).all()) and float(w.abs().sum()) > 0
    c.requires_grad_()
    dx, = torch.autograd.grad(ext.relu_square_linear(h, c, 4 * dim, dim, 3), h, dy, create_graph=True)
    with pytest.raises(RuntimeError, match="no second derivative"):
        torch.autograd.grad(dx, c, v)


@pytest.mark.parametrize("first_half", ["trained", "frozen", "frozen, its input not"])
@pytest.mark.parametrize("dim,k,tokens", [(64, 64, 40), (192, 136, 700)])
def test_what_the_squared_relu_keeps(dim, k, tokens, first_half):
    """From the forward to the backward pass: as many bytes as the layers and the activation keep where each is called for itself, none of them the
    activation's input where that has no gradient."""
    from randumb_amd.gpt import RT_GPTConfig, RT_MLP

    print(f"case what the squared ReLU keeps dim={dim} k={k}, first half {first_half}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(dim)
    with torch.device("cuda"):
        mlp = RT_MLP(dim, RT_GPTConfig(int_dim_gen=iter([k, k]), seed_gen=iter([3, 4]))).bfloat16()
    mlp.c_fc.weight_coef.requires_grad_(first_half == "trained")
    x, dy = bf16(g, tokens, dim).requires_grad_(first_half != "frozen"), bf16(g, tokens, dim)
    kept = []

    def run():
        kept.append([])
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (kept[-1].append(t), t)[1], lambda t: t):
            y = mlp(x)
        torch.autograd.grad(y, mlp.c_proj.weight_coef, dy)

    run()
    handles = [mlp.c_fc.register_forward_hook(lambda m, args, out: None)]
    run()
    handles.append(mlp.c_proj.register_forward_hook(lambda m, args, out: None))
    run()
    bytes_of = [sum(t.untyped_storage().nbytes() for t in run_kept) for run_kept in kept]
    assert bytes_of == bytes_of[-1:] * 3, bytes_of
    hidden = [[t.shape[-1] for t in run_kept].count(4 * dim) for run_kept in kept]
    assert hidden == [0 if first_half == "frozen" else 1] * 3, hidden
    for h in handles:
        h.remove()


# one position, one row; fewer positions than waves; a last block of one row; rows of more than a wave's share (65, all, and half of the positions); columns of one
# piece, of a part of one and of several
@pytest.mark.parametrize("positions,vocab,dim,hot", [(1, 1, 8, 0), (7, 129, 64, 0), (600, 65, 520, 0), (1000, 64, 768, 65), (8192, 5030, 768, 4096), (3000, 40, 1032, 3000),
                                                     (16384, 50304, 256, 64)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_gradient_of_a_dense_table(ext, positions, vocab, dim, hot, dtype):
    print(f"case dense table {positions} of {vocab} x {dim}, {hot} of them one row, {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(positions)
    idx = torch.randint(0, vocab, (positions,), generator=g, device="cuda")
    idx[torch.randperm(positions, generator=g, device="cuda")[:hot]] = vocab // 2
    idx, w, dy = idx.to(dtype), bf16(g, vocab, dim).requires_grad_(), bf16(g, positions, dim)
    y = ext.embedding(w, idx)
    assert torch.equal(y, F.embedding(idx, w))
    got, = torch.autograd.grad(y, w, dy)
    want = torch.zeros(vocab, dim, dtype=torch.float64, device="cuda").index_add_(0, idx.long(), dy.double())
    size = torch.zeros(vocab, dim, dtype=torch.float64, device="cuda").index_add_(0, idx.long(), dy.double().abs())
    # bf16's rounding of the result, and at most `positions` roundings to 24 bits of sums no larger than `size`
    assert bool(((got.double() - want).abs() <= 2.0**-8 * want.abs() + min(positions, 64 + positions / 8) * 2.0**-24 * size).all())
    assert torch.equal(torch.autograd.grad(ext.embedding(w, idx), w, dy)[0], got)


# tables of several rounds of blocks, the last one of one row; a row of many positions among them
@pytest.mark.parametrize("positions,vocab,dim,hot", [(1024, 65537, 8, 100), (2048, 262144, 24, 1000), (4096, 270000, 768, 0)])
def test_gradient_of_a_long_table(ext, positions, vocab, dim, hot):
    test_gradient_of_a_dense_table(ext, positions, vocab, dim, hot, torch.int64)


def test_long_tables_are_left_to_the_stock_operator(ext):
    w, idx = torch.zeros(300000, 8, device="cuda", dtype=torch.bfloat16, requires_grad=True), torch.zeros(4096, dtype=torch.int64, device="cuda")
    assert ext.embedding(w, idx) is None and ext.embedding(w[:131072], idx) is not None and ext.embedding(w[:131072], idx[:1000]) is None


def test_dense_tables_that_the_kernel_leaves(ext):
    w, many = torch.zeros(10, 64, device="cuda", dtype=torch.bfloat16, requires_grad=True), torch.zeros(16385, dtype=torch.int64, device="cuda")
    assert ext.embedding(w, many) is None and ext.embedding(w, many[:0]) is None and ext.embedding(w.detach(), many[:5]) is None
    assert ext.embedding(torch.zeros(10, 60, device="cuda", dtype=torch.bfloat16, requires_grad=True), many[:5]) is None
    y = ext.embedding(w, many[:6].view(2, 3))
    g, = torch.autograd.grad(y, w, torch.ones_like(y).requires_grad_(), create_graph=True)
    assert g.requires_grad and float(g[0, 0]) == 6.0 and float(g[1:].abs().sum()) == 0.0


# one to four groups of 64 coefficients and more, rows that are no whole lines (72), one launch and two, a last tile of tokens that is not full
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 64, 64, 8), (300, 96, 192, 72), (513, 128, 320, 128), (700, 256, 1024, 192), (1025, 768, 3072, 256), (300, 64, 72, 64), (513, 128, 256, 320)])
@pytest.mark.parametrize("one_launch", [1, 0])
def test_squared_relu_beside_a_forward_product(T, in_f, out_f, k, one_launch):
    import ctypes

    from randumb_amd import _lib, hip

    print(f"case squared ReLU beside a forward product {T} x {in_f} -> {out_f} k={k}", flush=True)
    lib, stream, g = _lib.load(), torch.cuda.current_stream().cuda_stream, torch.Generator(device="cuda").manual_seed(T)
    x, c = bf16(g, T, in_f), bf16(g, out_f, k)
    x[T // 2, 3] = float("inf")
    before = hip.set_one_launch(one_launch)
    try:
        want, state = hip.linear_project_fwd(x, c, 5, None)
        d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0)
        y, a = (torch.full((T + 1, out_f), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
        assert lib.rdb_linear_project_fwd_relu_square(y.data_ptr(), a.data_ptr(), state.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), ctypes.byref(d), None, 0, stream) == 0
        same = lambda u, v: torch.equal(torch.nan_to_num(u, nan=1234.0), torch.nan_to_num(v, nan=1234.0))
        assert same(y[:T], want) and same(a[:T], F.relu(want).square())
        assert bool((y[T] == 7.0).all()) and bool((a[T] == 7.0).all())
    finally:
        hip.set_one_launch(before)
