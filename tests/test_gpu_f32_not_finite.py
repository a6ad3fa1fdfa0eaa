"""Infinities and NaNs in the fp32 products that run as bf16 matrix instructions on three-way splits of their operands: they come
out where a product in 64 bits has them."""
import math

import pytest
import torch

from randumb_amd import SillyLinear, hip

pytestmark = pytest.mark.gpu


def same_pattern(got, want):
    assert got.shape == want.shape
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    fin = want.isfinite()
    if fin.any():
        assert float((got.double() - want)[fin].norm()) <= 1e-5 * float(want[fin].norm())


def spoiled(g, rows, cols):
    """Ordinary values with an infinite row, infinities of one and of both signs in a row, zeros, a NaN, and the largest finite value."""
    x = torch.randn(rows, cols, device="cuda", generator=g)
    x[1, 3] = math.inf
    x[2, cols - 1] = -math.inf
    x[3, 0], x[3, cols // 2] = math.inf, -math.inf
    x[4] = 0.0
    x[4, 5] = math.inf
    x[5, cols - 2] = math.nan
    x[rows - 1] = math.inf
    return x


@pytest.mark.parametrize("tokens,in_f,out_f", [(130, 96, 200), (65, 97, 51), (1, 64, 33), (300, 1000, 257)])
def test_vector_layer(tokens, in_f, out_f):
    """Its three dense products: y (bias on top), dx = dy . W, and dW = dy^T . x, seen through the contraction with the noise."""
    print(f"case {tokens} x {in_f} -> {out_f}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    layer = SillyLinear(in_f, out_f, [8, 8], [3, 4], device="cuda")
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, 0.1, generator=g)
        layer.bias_coef.normal_(0.0, 0.1, generator=g)
    W, b, N = layer.weight.get_materialized().double(), layer.bias.get_materialized().double(), layer.weight.get_noise_matrix().double()
    x = torch.randn(tokens, in_f, device="cuda", generator=g)
    dy = torch.randn(tokens, out_f, device="cuda", generator=g)
    bad = spoiled(g, max(tokens, 7), in_f)[-tokens:].clone().requires_grad_()
    same_pattern(layer(bad).detach(), bad.detach().double() @ W.t() + b)
    bad_dy = spoiled(g, max(tokens, 7), out_f)[-tokens:]
    x.requires_grad_()
    dx, dc = torch.autograd.grad(layer(x), [x, layer.weight_coef], bad_dy)
    same_pattern(dx, bad_dy.double() @ W)
    one = dy.clone()
    one[0, 1] = math.inf            # one infinite column of dW: the sums over the elements have infinities of both signs or one
    (dc,) = torch.autograd.grad(layer(x), [layer.weight_coef], one)
    same_pattern(dc, N.t() @ (one.double().t() @ x.detach().double()).flatten())


@pytest.mark.parametrize("row_len", [2048, 2051])
def test_matrix_coefficient_gradient(row_len):
    """dcoef = dW . N^T with infinities in dW (a row each, one or both signs)."""
    g = torch.Generator(device="cuda").manual_seed(row_len)
    rows, k, seed = 64, 70, 11
    dW = spoiled(g, rows, row_len)
    N = hip.sq5_fill_2d(row_len, k, seed).double()
    same_pattern(hip.materialize_bwd(dW.contiguous().flatten(), k, seed, rows), dW.double() @ N)


@pytest.mark.parametrize("tokens,in_f,out_f,k", [(300, 256, 192, 128), (128, 784, 256, 64), (130, 133, 99, 70)])
def test_projection_and_its_products(tokens, in_f, out_f, k):
    """z = x . N^T of an fp32 layer keeps the infinities; dC = dy^T . z has them where the tokens' sums have."""
    g = torch.Generator(device="cuda").manual_seed(k)
    x, dy = spoiled(g, tokens, in_f), torch.randn(tokens, out_f, device="cuda", generator=g)
    N = hip.sq5_fill_2d(in_f, k, 5).double()
    state = hip.linear_project(x, k, out_f, 5)
    z = x.double() @ N
    same_pattern(hip.projection_unpack(state, in_f, out_f, k, torch.float32)["z"], z)
    dc, _ = hip.linear_bwd_dcoef(dy, x, k, out_f, in_f, out_f, in_f, 1, 5)
    same_pattern(dc, dy.double().t() @ z)
    x[:] = torch.randn(tokens, in_f, device="cuda", generator=g)
    x[2, 7] = math.inf              # one infinite token row of z, the signs of its noise: dC = sign(dy) inf where nothing meets it
    dc, _ = hip.linear_bwd_dcoef(dy, x, k, out_f, in_f, out_f, in_f, 1, 5)
    same_pattern(dc, dy.double().t() @ (x.double() @ N))


# tiles of 128 and 64 rows, one group of waves and several, one range of the contraction and several, pieces that are and are not aligned; the
# random bias's share is added to an output
@pytest.mark.parametrize("form", ["matrix", "random_bias", "vector"])
@pytest.mark.parametrize("tokens,in_f,out_f,k", [(600, 256, 192, 70), (2048, 768, 3072, 256), (4100, 301, 259, 83), (2000, 2001, 130, 66), (700, 2048, 2048, 512)])
def test_finite_sums_are_what_they_are_without_others_beside_them(form, tokens, in_f, out_f, k):
    """An infinity, a NaN or a product beyond the largest float in a row of x or in one value of dy: the other rows and columns keep
    their bits."""
    if form == "vector" and (k > 100 or in_f > 400):
        k = 16
    print(f"case beside {form} {tokens} x {in_f} -> {out_f}, k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    layer = SillyLinear(in_f, out_f, [k, k], [3, 4], device="cuda", bias=False, matrix_coef=form != "vector", rt_bias=form == "random_bias")
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, 0.1, generator=g)
    x, dy = torch.randn(tokens, in_f, device="cuda", generator=g), torch.randn(tokens, out_f, device="cuda", generator=g)

    def run(x, dy):
        x = x.clone().requires_grad_()
        y = layer(x)
        dx, dc = torch.autograd.grad(y, [x, layer.weight_coef], dy)
        return y.detach(), dx, dc

    y, dx, dc = run(x, dy)
    row, col = tokens - 3, out_f // 2
    rows, cols = torch.arange(tokens, device="cuda") != row, torch.arange(out_f, device="cuda") != col
    for bad in (math.inf, math.nan, 3.0e38):
        spoiled = x.clone()
        spoiled[row, in_f // 3] = bad
        got = run(spoiled, dy)
        assert torch.equal(got[0][rows], y[rows]) and torch.equal(got[1], dx)
        spoiled = dy.clone()
        spoiled[row, col] = bad
        got = run(x, spoiled)
        assert torch.equal(got[0], y) and torch.equal(got[1][rows], dx[rows])
        assert form == "vector" or torch.equal(got[2][cols], dc[cols])
        if bad != 3.0e38:   # as it has to be: no value of the row is finite
            assert not bool(got[1][row].isfinite().any())


def test_the_largest_values_do_not_become_nan():
    """Parts of one sign: a product that overflows is an infinity of its own sign, one that does not is finite."""
    layer = SillyLinear(64, 32, [8, 8], [3, 4], device="cuda", bias=False)
    with torch.no_grad():
        layer.weight_coef.fill_(1.0)
    W = layer.weight.get_materialized()
    x = torch.zeros(40, 64, device="cuda")
    x[0, 3], x[1, 3], x[2, 5] = 3.4028234663852886e38, -3.4028234663852886e38, 1e-3 * 3.4028234663852886e38
    want = (x.double() @ W.double().t()).float()   # rounds to an infinity beyond the largest float
    got = layer(x).detach()
    assert not bool(got.isnan().any())
    edge = want.double().abs() > 3.3e38            # rounding decides there
    assert torch.equal(got.isinf() | edge, want.isinf() | edge)
