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


@pytest.mark.parametrize("tokens,in_f,out_f,k,bias_k", [(1, 1, 1, 1, 1), (33, 67, 130, 17, 0), (257, 300, 65, 40, 9), (700, 129, 1000, 256, 64), (1500, 300, 520, 100, 300),
                                                         (9000, 24, 40, 20, 5), (13001, 135, 67, 33, 0), (4100, 300, 129, 8, 70)])   # dW in more ranges than the contraction adds up
def test_backward_pass_in_one_call(tokens, in_f, out_f, k, bias_k):
    """rdb_vector_linear_bwd against fp64 and against the calls it stands for: dx or not, a bias or not, rows that are slices."""
    from randumb_amd import _lib, hip

    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(tokens + k)
    dy = torch.randn(tokens, out_f + 3, generator=g, device="cuda")[:, :out_f]
    x = torch.randn(tokens, in_f + 1, generator=g, device="cuda")[:, :in_f]
    W = torch.randn(out_f, in_f, generator=g, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    noise = hip.sq5_fill_2d(out_f * in_f, k, 3).double()
    want_dc = (dy.double().t() @ x.double()).reshape(-1) @ noise
    for with_dx in (True, False):
        need = lib.rdb_vector_linear_bwd_workspace_bytes(tokens, in_f, out_f, k, with_dx, bias_k > 0)
        assert need > 0
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        dx, dc, db = torch.full((tokens, in_f), 7.0, device="cuda"), torch.empty(k, device="cuda"), torch.empty(max(bias_k, 1), device="cuda")

        def call(bytes_given):
            return lib.rdb_vector_linear_bwd(dx.data_ptr() if with_dx else None, dc.data_ptr(), db.data_ptr() if bias_k else None, dy.data_ptr(), dy.stride(0), x.data_ptr(),
                                             x.stride(0), W.data_ptr() if with_dx else None, tokens, in_f, out_f, k, 3, bias_k, 4, ws.data_ptr(), bytes_given, stream)

        assert call(need) == 0
        first = (dx.clone(), dc.clone(), db.clone())
        assert call(need) == 0 and all(torch.equal(a, b) for a, b in zip(first[: 2 + (bias_k > 0)], (dx, dc, db)))
        # sums of products that are exact to 2^-21 or so, dW's rounded to fp32
        assert _rel(dc, want_dc.cpu()) < 3e-6
        if with_dx:
            assert _rel(dx, (dy.double() @ W.double()).cpu()) < 3e-6
        else:
            assert bool((dx == 7.0).all())
        if bias_k:
            assert _rel(db, (dy.double().sum(0) @ hip.sq5_fill_2d(out_f, bias_k, 4).double()).cpu()) < 3e-6
        assert call(need - 1) < 0


# few tiles of a large dW: one range and two beside dx, one and three alone
@pytest.mark.parametrize("tokens,in_f,out_f,k", [(1279, 1388, 1566, 6), (1280, 1388, 1566, 6)])
def test_backward_pass_of_a_dw_of_few_tiles(tokens, in_f, out_f, k):
    test_backward_pass_in_one_call(tokens, in_f, out_f, k, 0)
