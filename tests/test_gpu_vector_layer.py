"""The vector-coef layer and embedding as the extension module runs them: against float64, with every input's gradient, at the edges
of the bias kernels' and the products' tiles, and against the tensor subclass's own dispatch for second derivatives."""
import pytest
import torch
import torch.nn.functional as F

from randumb_amd import SillyEmbedding, SillyLinear, ops

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm().clamp_min(1e-300))


def _layer(in_f, out_f, k, rt_bias, bias=True, dtype=torch.float32):
    layer = SillyLinear(in_f, out_f, [k, max(1, k // 2)], [11, 12], bias=bias, rt_bias=rt_bias, device="cuda", dtype=dtype)
    g = torch.Generator(device="cuda").manual_seed(in_f)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.3, generator=g)
    return layer


@pytest.mark.parametrize("shape,in_f,out_f,k,rt_bias", [((33,), 67, 130, 5, False), ((2, 65), 196, 257, 16, True), ((513,), 128, 64, 130, True),
                                                        ((1, 1), 8, 8, 12, False), ((700,), 260, 1031, 33, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer(shape, in_f, out_f, k, rt_bias, dtype):
    layer = _layer(in_f, out_f, k, rt_bias, dtype=dtype)
    torch.manual_seed(out_f)
    x = torch.randn(*shape, in_f, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(*shape, out_f, device="cuda").to(dtype)
    y = layer(x)
    assert "VectorLinear" in repr(y.grad_fn)
    names = ["weight_coef", "bias_coef"] + (["weight_scale_bias", "bias_scale_bias"] if rt_bias else [])
    grads = torch.autograd.grad(y, [x] + [getattr(layer, n) for n in names], dy)
    N = ops.sq5_gen_2d(in_f * out_f, k, 11).double().cpu()
    n1, n1b = ops.sq5_gen_1d(in_f * out_f, 11).double().cpu(), ops.sq5_gen_1d(out_f, 12).double().cpu()
    Nb = ops.sq5_gen_2d(out_f, layer.bias_coef.numel(), 12).double().cpu()
    par = {n: getattr(layer, n).detach().double().cpu() for n in names}
    W, b = N @ par["weight_coef"], Nb @ par["bias_coef"]
    if rt_bias:
        W, b = W + par["weight_scale_bias"] * n1, b + par["bias_scale_bias"] * n1b
    W, X, D = W.view(out_f, in_f), x.detach().double().cpu().reshape(-1, in_f), dy.double().cpu().reshape(-1, out_f)
    dW, db = (D.t() @ X).flatten(), D.sum(0)
    want = [D @ W, N.t() @ dW, Nb.t() @ db] + ([(dW * n1).sum().view(1), (db * n1b).sum().view(1)] if rt_bias else [])
    tol = 1e-2 if dtype == torch.bfloat16 else 5e-6
    assert _rel(y.detach().reshape(-1, out_f), X @ W.t() + b) < tol
    for n, g, w in zip(["x"] + names, grads, want):
        # sums over many elements of either sign: against the size of what is added up, not of what is left of it
        size = w.norm() if "scale" not in n else (dW.abs().sum() if n == "weight_scale_bias" else db.abs().sum()) * 0.05
        assert float((g.double().cpu().reshape(w.shape) - w).norm() / size) < tol, n


@pytest.mark.parametrize("tokens,features", [(64, 256), (2000, 96)])   # W no larger than the activations (kept for backward), and larger
def test_second_derivatives_and_the_subclass(tokens, features):
    layer = _layer(features, 2 * features, 9, True)
    x = torch.randn(tokens, features, device="cuda", requires_grad=True)
    inputs = [x, layer.weight_coef, layer.bias_coef, layer.weight_scale_bias]
    seen = []
    for forward in (layer, lambda v: F.linear(v, layer.weight, layer.bias)):
        y = forward(x)
        first = torch.autograd.grad((y * y).sum(), inputs, create_graph=True)
        plain = torch.autograd.grad((forward(x) ** 2).sum(), inputs)
        for a, b in zip(first, plain):
            assert _rel(a.detach(), b.double().cpu()) < 5e-6
        second = torch.autograd.grad(first[0].square().sum(), [x, layer.weight_coef])
        seen.append([y.detach(), *[f.detach() for f in first], *second])
    for a, b in zip(*seen):
        assert _rel(a, b.double().cpu()) < 2e-5


def test_without_gradients_and_frozen_inputs():
    layer = _layer(40, 24, 6, False)
    x = torch.randn(7, 40, device="cuda")
    with torch.no_grad():
        y = layer(x)
    assert not y.requires_grad and torch.equal(y, layer(x).detach())
    layer(x).sum().backward()   # x needs no gradient: the coefficients' alone
    assert x.grad is None and layer.weight_coef.grad is not None and layer.bias_coef.grad is not None
    with pytest.raises(RuntimeError):
        layer(torch.randn(7, 41, device="cuda"))


@pytest.mark.parametrize("shape,dim,k", [((3, 5), 24, 7), ((65,), 64, 130)])
def test_embedding(shape, dim, k):
    table = SillyEmbedding(1000, dim, [k], [4], device="cuda")
    idx = torch.randint(0, 1000, shape, device="cuda")
    y = table(idx)
    assert "EmbedRows" in repr(y.grad_fn) and y.shape == (*shape, dim)
    assert torch.equal(y, ops.embed_fwd(idx, table.weight_coef, dim, 4))
    dy = torch.randn_like(y)
    got, = torch.autograd.grad(y, [table.weight_coef], dy)
    assert torch.equal(got, ops.embed_bwd(idx, dy, k, dim, 4))
