"""What is refused, and what goes on working, around the calls that reach kernels by address."""
import pytest
import torch

from randumb_amd import SillyEmbedding, SillyLinear, _lib, listgen

pytestmark = pytest.mark.gpu


def _layer(form):
    """(layer, input) of every way a layer's forward pass saves for its backward pass."""
    dt = torch.float32 if form.endswith("fp32") else torch.bfloat16
    sizes = {"projected_bf16": (300, 256, 192, 64), "projected_fp32": (300, 256, 192, 128), "random_bias_bf16": (300, 256, 192, 64),
             "kept_bf16": (130, 133, 99, 50), "one_call_fp32": (3, 256, 192, 16), "vector_fp32": (40, 96, 64, 16)}
    tokens, in_f, out_f, k = sizes[form]
    layer = SillyLinear(in_f, out_f, [k, k], [1, 2], device="cuda", dtype=dt, matrix_coef=not form.startswith("vector"), rt_bias=form.startswith("random"))
    with torch.no_grad():
        for p in (layer.weight_coef, layer.bias_coef):
            p.normal_(0.0, 0.05)
    return layer, torch.randn(tokens, in_f, device="cuda").to(dt).requires_grad_()


FORMS = ["projected_bf16", "projected_fp32", "random_bias_bf16", "kept_bf16", "one_call_fp32", "vector_fp32"]


@pytest.mark.parametrize("form", FORMS)
def test_saved_tensors_that_come_back_on_the_host_are_refused(form):
    """Hooks that pack saved tensors to the host and do not bring them back: an exception from the backward pass."""
    layer, x = _layer(form)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
        y = layer(x)
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        y.backward(torch.ones_like(y))


@pytest.mark.parametrize("form", FORMS)
def test_saved_tensors_may_rest_on_the_host(form):
    layer, x = _layer(form)
    wanted = [x, *layer.parameters()]
    y = layer(x)
    ref = torch.autograd.grad(y, wanted, torch.ones_like(y), allow_unused=True)
    with torch.autograd.graph.save_on_cpu():
        y = layer(x)
    got = torch.autograd.grad(y, wanted, torch.ones_like(y), allow_unused=True)
    for a, b in zip(got, ref):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


def test_saved_indices_of_the_embedding_on_the_host_are_refused():
    e = SillyEmbedding(50, 24, listgen([16]), listgen([3]), device="cuda")
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
        y = e(torch.tensor([1, 5, 49], device="cuda"))
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        y.sum().backward()


@pytest.mark.parametrize("op", ["rms_norm", "add_rms_norm", "relu_square", "cross_entropy", "causal_attention"])
def test_saved_activations_on_the_host_are_refused(op):
    ext = _lib.extension()
    x = torch.randn(2, 8, 3 * 64, device="cuda").bfloat16().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t):
        if op == "rms_norm":
            y = ext.rms_norm(x, 1e-6)
        elif op == "add_rms_norm":
            y = ext.add_rms_norm(x, x.detach(), 1e-6)[1]
        elif op == "relu_square":
            y = ext.relu_square(x)
        elif op == "cross_entropy":
            y = ext.cross_entropy(x.view(-1, 192), torch.zeros(16, dtype=torch.int64, device="cuda"), -100)
        else:
            y = ext.causal_attention(x, torch.ones(32, device="cuda"), 1, 1e-6)
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        y.backward(torch.ones_like(y))


def test_a_layer_and_an_input_on_different_devices_are_refused():
    layer = SillyLinear(768, 96, [32, 32], [1, 2], matrix_coef=True)
    with pytest.raises(NotImplementedError, match="CPU implementation"):
        layer(torch.randn(4, 768, device="cuda"))
    layer = layer.to("cuda")
    assert layer(torch.randn(4, 768, device="cuda")).shape == (4, 96)


# ------------------------------------------------------------------------------------------------ modes, transforms, tangents
@pytest.mark.parametrize("form", [f for f in FORMS if not f.startswith("vector")])
def test_fake_inputs_of_a_layer_give_fake_outputs(form):
    from torch._subclasses.fake_tensor import FakeTensor, FakeTensorMode

    layer, x = _layer(form)
    mode = FakeTensorMode(allow_non_fake_inputs=True)
    with mode:
        y = layer(mode.from_tensor(x))
    assert isinstance(y, FakeTensor) and y.shape == (x.shape[0], layer.out_features) and y.dtype == x.dtype


@pytest.mark.parametrize("which", ["x", "coef"])
@pytest.mark.parametrize("form", [f for f in FORMS if not f.startswith("vector")])
@torch.no_grad()
def test_forward_mode_is_refused_not_dropped(form, which):
    import torch.autograd.forward_ad as fwd

    layer, x = _layer(form)
    x = x.detach()
    with fwd.dual_level():
        if which == "x":
            x = fwd.make_dual(x, torch.ones_like(x))
        else:
            coef = layer.weight_coef.detach()
            del layer._parameters["weight_coef"]
            layer.weight_coef = fwd.make_dual(coef, torch.ones_like(coef))
        with pytest.raises(NotImplementedError, match="jvp"):
            layer(x)


def test_forward_mode_of_the_embedding_is_refused_not_dropped():
    import torch.autograd.forward_ad as fwd

    e = SillyEmbedding(50, 24, listgen([16]), listgen([3]), device="cuda").requires_grad_(False)
    with fwd.dual_level():
        c = e.weight_coef.detach()
        del e._parameters["weight_coef"]
        e.weight_coef = fwd.make_dual(c, torch.ones_like(c))
        with pytest.raises(NotImplementedError, match="forward-mode"):
            e(torch.tensor([1, 2], device="cuda"))


def test_vmap_over_a_layer_is_refused_and_over_the_embedding_runs():
    layer, x = _layer("one_call_fp32")
    with pytest.raises(RuntimeError, match="functorch|vmap"):
        torch.vmap(layer)(x.detach().unsqueeze(1))
    e = SillyEmbedding(50, 24, listgen([16]), listgen([3]), device="cuda").requires_grad_(False)
    idx = torch.tensor([[1, 5], [49, 0]], device="cuda")
    assert torch.equal(torch.vmap(e)(idx), e(idx))


def test_forward_mode_through_the_stock_operators_of_a_block():
    """Normalisation, squared ReLU and the residual sum have forward-mode derivatives in their stock form, which tangents take."""
    import torch.nn.functional as F

    from randumb_amd import gpt

    x, v = (torch.randn(6, 64, device="cuda").bfloat16() for _ in range(2))
    for f, stock in ((gpt.RT_norm, lambda t: F.rms_norm(t, (64,))), (lambda t: gpt._add_norm(t, v)[1], lambda t: F.rms_norm(t + v, (64,)))):
        got, want = torch.func.jvp(f, (x,), (v,)), torch.func.jvp(stock, (x,), (v,))
        assert torch.equal(got[1], want[1])


def test_a_counting_mode_sees_a_layers_products():
    """A dispatch mode over real tensors sees the operators; the values are those of the direct calls."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Names(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    for form, op in (("one_call_fp32", "rten.linear_fwd"), ("projected_bf16", "rten.linear_project_fwd"), ("vector_fp32", "aten.addmm")):
        layer, x = _layer(form)
        want = layer(x)
        with Names() as mode:
            got = layer(x)
        assert any(op in n for n in mode.seen), mode.seen
        assert torch.allclose(got.float(), want.float(), rtol=1e-5, atol=1e-5 * float(want.float().abs().max()))


# ------------------------------------------------------------------------------------------------ second derivatives
@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("op", ["rms_norm", "add_rms_norm", "relu_square", "cross_entropy"])
def test_second_derivatives_of_a_blocks_operators(op, strided):
    """First derivatives under create_graph, and the derivatives of those, are the stock operators' in bf16 (the same kernels)."""
    import torch.nn.functional as F

    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(64, 40, device="cuda", generator=g).bfloat16()
    x = (x.t() if strided else x.t().contiguous()).requires_grad_()           # 40 rows of 64
    d = torch.randn(40, 64, device="cuda", generator=g).bfloat16().requires_grad_()
    t = torch.randint(0, 64, (40,), device="cuda", generator=g)
    w = torch.randn(40, 64, device="cuda", generator=g).bfloat16().requires_grad_()   # the incoming gradient, differentiated as well
    ext, eps = _lib.extension(), torch.finfo(torch.float32).eps
    fused, stock, inputs = {
        "rms_norm": (lambda: ext.rms_norm(x, eps), lambda: F.rms_norm(x, (64,)), [x, w]),
        "add_rms_norm": (lambda: sum(ext.add_rms_norm(x, d, eps)), lambda: (x + d) + F.rms_norm(x + d, (64,)), [x, d, w]),
        "relu_square": (lambda: ext.relu_square(x), lambda: F.relu(x).square(), [x, w]),
        "cross_entropy": (lambda: ext.cross_entropy(x, t, -100), lambda: F.cross_entropy(x.float(), t), [x]),
    }[op]

    def both(f):
        y = f()
        first = torch.autograd.grad(y, [i for i in inputs if i is not w], w if y.dim() else None, create_graph=True)
        return [*first, *torch.autograd.grad(sum((p.float() ** 2).sum() for p in first), inputs)]

    for a, b in zip(both(fused), both(stock)):
        assert a.shape == b.shape and torch.linalg.vector_norm((a - b).double()) <= 1e-2 * torch.linalg.vector_norm(b.double())


@pytest.mark.parametrize("leaf", [False, True])
@pytest.mark.parametrize("op", ["rms_norm", "add_rms_norm", "relu_square", "cross_entropy"])
def test_hooks_on_an_operators_input_run_once(op, leaf):
    """Under create_graph as without it, on the whole of the input's gradient (it is used twice)."""
    ext, eps = _lib.extension(), torch.finfo(torch.float32).eps
    x = torch.randn(40, 64, device="cuda").bfloat16().requires_grad_()
    t = torch.randint(0, 64, (40,), device="cuda")

    def run(create):
        seen = []
        u = x if leaf else x * 1.0
        handle = u.register_hook(lambda g: seen.append(g.detach().clone()))
        if op == "add_rms_norm":
            s, y = ext.add_rms_norm(u, u.detach(), eps)
            s.register_hook(lambda g: seen.append(g.detach().clone()))
            y = y + s
        else:
            y = {"rms_norm": lambda: ext.rms_norm(u, eps), "relu_square": lambda: ext.relu_square(u), "cross_entropy": lambda: ext.cross_entropy(u, t, -100)}[op]()
        (g,) = torch.autograd.grad(y.float().sum() + (u.float() * 3.0).sum(), x, create_graph=create)
        handle.remove()
        return seen, g.detach()

    (plain, g0), (graph, g1) = run(False), run(True)
    assert len(plain) == len(graph) == (2 if op == "add_rms_norm" else 1)
    for a, b in zip(plain + [g0], graph + [g1]):
        assert torch.linalg.vector_norm((a - b).double()) <= 1e-2 * torch.linalg.vector_norm(a.double())


def test_second_derivatives_that_do_not_exist_raise():
    e = SillyEmbedding(50, 24, listgen([16]), listgen([3]), device="cuda")
    w = torch.randn(2, 24, device="cuda", requires_grad=True)
    y = e(torch.tensor([1, 5], device="cuda"))
    (first,) = torch.autograd.grad(y, e.weight_coef, w, create_graph=True)
    assert torch.equal(first.detach(), torch.autograd.grad(e(torch.tensor([1, 5], device="cuda")), e.weight_coef, w.detach())[0])
    with pytest.raises(RuntimeError, match="second derivative"):
        first.sum().backward()
    qkv = torch.randn(1, 8, 192, device="cuda").bfloat16().requires_grad_()
    y = _lib.extension().causal_attention(qkv, torch.ones(32, device="cuda"), 1, 1e-6)
    (first,) = torch.autograd.grad(y, qkv, torch.ones_like(y), create_graph=True)
    with pytest.raises(RuntimeError, match="second derivative"):
        first.float().sum().backward()


@pytest.mark.parametrize("python", [False, True])
@pytest.mark.parametrize("form", [f for f in FORMS if not f.startswith("vector")])
def test_second_derivatives_of_a_matrix_layer_raise(form, python, monkeypatch):
    """Its first derivatives are there under create_graph; going through them raises where they depend on something (alone, and between
    operators that have second derivatives), and is refused as for any constant where they do not.  The bias's is linear in dy."""
    from randumb_amd import ops

    if python:   # the functions in Python, which the extension module leaves some requests to
        monkeypatch.setattr(ops, "_bias_form", lambda bias, out_features: None)
    layer, x = _layer(form)
    wanted = [x, layer.weight_coef, layer.bias_coef] + ([layer.weight_scale_bias] if form.startswith("random") else [])
    dy = torch.randn(x.shape[0], layer.out_features, device="cuda").to(x.dtype)
    ref = torch.autograd.grad(layer(x), wanted, dy)
    if python and form == "one_call_fp32":   # a layer takes one call here; that function's name is the module's otherwise
        assert type(layer(x).grad_fn).__name__ == "_OneCallFunctionBackward"
    w = dy.clone().requires_grad_()
    for gradient in (dy, w):
        first = torch.autograd.grad(layer(x), wanted, gradient, create_graph=True)
        for i, (got, want) in enumerate(zip(first, ref)):
            assert torch.linalg.vector_norm((got - want).double()) <= (1e-6 if x.dtype == torch.float32 else 1e-2) * torch.linalg.vector_norm(want.double())
            if i != 2:
                with pytest.raises(RuntimeError, match="second derivative"):
                    torch.autograd.grad(got.float().square().sum(), [layer.weight_coef] if i == 0 else [x], allow_unused=True)
    if python:   # a bias's gradient goes through the materialise operators there
        with pytest.raises(RuntimeError, match="no autograd formula"):
            torch.autograd.grad(first[2].sum(), w)
    else:        # d (sum of the bias's gradient) / dy: the values of a bias with coefficients 1, for every token
        (got,) = torch.autograd.grad(first[2].double().sum(), w)
        want = layer.bias.get_noise_matrix().double().sum(1)
        assert got.shape == w.shape and torch.linalg.vector_norm(got.double() - want) <= 1e-2 * torch.linalg.vector_norm(want) * x.shape[0] ** 0.5
    # between operators with second derivatives nothing is dropped
    s = x.detach().clone().requires_grad_()
    (g,) = torch.autograd.grad((layer(s.square()).float() ** 2).sum(), s, create_graph=True)
    with pytest.raises(RuntimeError, match="second derivative"):
        torch.autograd.grad(g.float().sum(), s)
    # the gradients that a program accumulates under create_graph can be cleared in place
    for gradient in (dy, w):
        layer(x).backward(gradient, create_graph=True)
        layer.zero_grad(set_to_none=False)
        assert not bool(layer.weight_coef.grad.any()) and layer.weight_coef.grad.grad_fn is None
    layer.zero_grad(set_to_none=True)
    # nothing to come: constants, as they were
    layer.requires_grad_(False)
    (g,) = torch.autograd.grad(layer(x), x, dy, create_graph=True)
    assert not g.requires_grad and torch.equal(g, ref[0])
    layer.weight_coef.requires_grad_(True)
    (g,) = torch.autograd.grad(layer(x.detach()), layer.weight_coef, dy, create_graph=True)
    assert not g.requires_grad and torch.linalg.vector_norm((g - ref[1]).double()) <= 1e-2 * torch.linalg.vector_norm(ref[1].double())


@pytest.mark.parametrize("rt_bias", [False, True])
def test_third_derivatives_of_a_vector_layer(rt_bias):
    """The gradient of the coefficients, N^T vec(w^T x), is linear in w: the third derivatives of the sum of its fourth powers against a
    dense matrix's."""
    g = torch.Generator(device="cuda").manual_seed(5)
    layer = SillyLinear(12, 9, [8, 8], [3, 4], device="cuda", bias=False, rt_bias=rt_bias)
    x, w, u = (torch.randn(7, n, device="cuda", generator=g).requires_grad_() for n in (12, 9, 9))
    N = layer.weight.get_noise_matrix().double()

    def third(first, w, u):
        (second,) = torch.autograd.grad((first ** 4).sum(), w, create_graph=True)
        return torch.autograd.grad((second * u).square().sum(), [w, u])

    (first,) = torch.autograd.grad(layer(x), layer.weight_coef, w, create_graph=True)
    got = third(first, w, u)
    w64, u64 = w.detach().double().requires_grad_(), u.detach().double().requires_grad_()
    want = third(N.t() @ (w64.t() @ x.detach().double()).flatten(), w64, u64)
    for a, b in zip(got, want):
        assert torch.linalg.vector_norm(a.double() - b) <= 1e-4 * torch.linalg.vector_norm(b)


def test_a_missing_second_derivative_is_not_dropped_from_a_sum():
    """Asked for one input by name, beside another way to it."""
    e = SillyEmbedding(50, 24, listgen([16]), listgen([3]), device="cuda")
    w = torch.randn(2, 24, device="cuda", requires_grad=True)
    (first,) = torch.autograd.grad(e(torch.tensor([1, 5], device="cuda")), e.weight_coef, w, create_graph=True)
    with pytest.raises(RuntimeError, match="second derivative"):
        torch.autograd.grad(first.sum() + w.sum(), w)
    qkv = torch.randn(1, 8, 192, device="cuda").bfloat16().requires_grad_()
    y = _lib.extension().causal_attention(qkv, torch.ones(32, device="cuda"), 1, 1e-6)
    (first,) = torch.autograd.grad(y, qkv, torch.ones_like(y), create_graph=True)
    with pytest.raises(RuntimeError, match="second derivative"):
        torch.autograd.grad(first.float().sum() + qkv.float().square().sum(), qkv)


# ------------------------------------------------------------------------------------------------ slices of very wide matrices
@pytest.mark.parametrize("sliced", ["x", "dy"])
@pytest.mark.parametrize("form", ["projected_bf16", "projected_fp32", "random_bias_bf16", "kept_bf16"])
def test_rows_farther_apart_than_one_launch_addresses(form, sliced):
    """2^29 elements from the first row to the last: the layer runs, with the results of a contiguous input."""
    layer, x = _layer(form)
    wanted = [x, *[p for n, p in layer.named_parameters() if "scale" not in n or form.startswith("random")]]
    dy = torch.randn(x.shape[0], layer.out_features, device="cuda").to(x.dtype)
    y = layer(x)
    ref = [y.detach(), *torch.autograd.grad(y, wanted, dy)]

    def spread(t):
        wide = torch.empty(t.shape[0], (1 << 29) // t.shape[0] // 8 * 8 + 8, device="cuda", dtype=t.dtype)[:, : t.shape[1]]
        return wide.copy_(t)

    wanted[0] = x2 = spread(x.detach()).requires_grad_() if sliced == "x" else x
    assert x2.shape[0] * x2.stride(0) >= 1 << 29 or sliced == "dy"
    y = layer(x2)
    got = [y.detach(), *torch.autograd.grad(y, wanted, spread(dy) if sliced == "dy" else dy)]
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


# ------------------------------------------------------------------------------------------------ gradients of the pseudorandom tensors themselves
@pytest.mark.parametrize("how", ["retain_grad", "register_hook"])
@pytest.mark.parametrize("form,which", [("vector_fp32", "weight"), ("vector_fp32", "bias"), ("kept_bf16", "bias"), ("projected_bf16", "bias"), ("one_call_fp32", "bias")])
def test_somebody_who_waits_for_a_tensors_own_gradient_gets_it(form, which, how):
    layer, x = _layer(form)
    wanted = [x, layer.weight_coef, layer.bias_coef]
    dy = torch.randn(x.shape[0], layer.out_features, device="cuda").to(x.dtype)
    ref = torch.autograd.grad(layer(x), wanted, dy)
    t, seen = getattr(layer, which), []
    if how == "retain_grad":
        t.retain_grad()
    else:
        t.register_hook(lambda g: seen.append(g.detach().clone()))
    layer(x).backward(dy)
    grad = t.grad if how == "retain_grad" else seen[0]
    want = (dy.double().t() @ x.detach().double()) if which == "weight" else dy.double().sum(0)
    assert grad.shape == t.shape
    assert float((grad.double() - want).norm()) <= (1e-5 if x.dtype == torch.float32 else 1e-2) * float(want.norm())
    for p, r in zip(wanted, ref):
        assert float((p.grad.double() - r.double()).norm()) <= (1e-5 if x.dtype == torch.float32 else 2e-2) * float(r.double().norm())


# ------------------------------------------------------------------------------------------------ outputs that are changed in place
@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("form", FORMS + ["vector_bf16"])
def test_a_layers_output_may_be_changed_in_place(form, dims):
    """As that of F.linear: relu_(layer(x)), and its gradient."""
    layer, x = _layer(form.replace("vector_bf16", "vector_fp32"))
    if form == "vector_bf16":
        layer, x = layer.bfloat16(), x.detach().bfloat16().requires_grad_()
    if dims == 3:
        x = x.detach().unsqueeze(0).requires_grad_()
    (want,) = torch.autograd.grad(torch.relu(layer(x)).sum(), x)
    y = layer(x)
    assert not y._is_view() or dims == 3
    (got,) = torch.autograd.grad(y.relu_().sum(), x)
    assert torch.equal(got, want)
