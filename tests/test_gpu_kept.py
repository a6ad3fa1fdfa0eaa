"""Layers whose forward pass keeps z = x . N^T for the backward pass (bf16 with odd sizes, fp32 in the few-token regime): against
float64, at both ends of the range, with the fused random bias and with gradients that are not wanted."""
import ctypes

import pytest
import torch

from randumb_amd import _lib, hip, ops

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


@pytest.mark.parametrize("T,in_f,out_f,k,dtype", [(32, 784, 256, 64, torch.float32), (128, 256, 10, 64, torch.float32), (500, 999, 77, 33, torch.float32),
                                                  (97, 1001, 130, 100, torch.bfloat16), (1200, 260, 515, 71, torch.bfloat16)])
@pytest.mark.parametrize("rbias", [False, True])
def test_against_float64(T, in_f, out_f, k, dtype, rbias):
    g = torch.Generator().manual_seed(T)
    x, dy = torch.randn(T, in_f, generator=g).to(dtype), torch.randn(T, out_f, generator=g).to(dtype)
    c, s = (torch.randn(out_f, k, generator=g) / k ** 0.5).to(dtype), torch.tensor([0.25]).to(dtype)
    W = c.double() @ ops.sq5_gen_2d(in_f, k, 8).double().cpu().t()
    R = ops.sq5_gen_1d(in_f * out_f, 8).double().cpu().view(out_f, in_f)
    if rbias:
        W = W + 0.25 * R
    leaves = [t.cuda().requires_grad_() for t in ([x, c, s] if rbias else [x, c])]
    d = hip._desc(T, in_f, out_f, leaves[1], in_f, 1, 8, dtype, 0)
    kept = _lib.load().rdb_linear_kept_bytes(ctypes.byref(d))
    assert kept >= 4 * T * k
    y = ops.linear(leaves[0], leaves[1], in_f, out_f, in_f, 1, 8, leaves[2] if rbias else None, None)
    assert "OneCall" in repr(y.grad_fn)
    grads = torch.autograd.grad(y, leaves, dy.cuda(), retain_graph=True)
    X, D = x.double(), dy.double()
    dW = D.t() @ X
    want = [D @ W, dW @ ops.sq5_gen_2d(in_f, k, 8).double().cpu()] + ([(dW * R).sum().view(1)] if rbias else [])
    tol = 5e-6 if dtype == torch.float32 else 8e-3
    assert _rel(y.detach(), X @ W.t()) < tol
    for got, w in zip(grads, want):
        size = w.norm() if got.numel() > 1 else (dW * R).norm()
        assert got.dtype == dtype and float((got.double().cpu() - w).norm() / size) < tol
    # one at a time: the others are not formed
    for leaf, w in zip(leaves, grads):
        alone, = torch.autograd.grad(y, [leaf], dy.cuda(), retain_graph=True)
        assert float((alone.double() - w.double()).norm() / w.double().norm().clamp_min(1e-3)) < 2 * tol


def test_not_kept():
    L = _lib.load()

    def kept(T, in_f, out_f, k, dtype):
        c = torch.empty(out_f, k, dtype=dtype)
        return L.rdb_linear_kept_bytes(ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 8, dtype, 0)))

    assert kept(31, 784, 256, 64, torch.float32) == 0 and kept(128, 784, 256, 64, torch.float32) == 128 * 64 * 4
    assert kept(2000, 784, 256, 64, torch.float32) == 0          # has a projection state
    assert kept(128, 16, 256, 64, torch.float32) == 0            # z more than twice x
    assert kept(96, 1001, 999, 100, torch.bfloat16) == 0 and kept(97, 1001, 999, 100, torch.bfloat16) > 0
    assert kept(4096, 1000, 1000, 104, torch.bfloat16) == 0      # multiples of 8: the bf16 kernels
    assert kept(4096, 100, 999, 101, torch.bfloat16) == 0


@pytest.mark.parametrize("T,in_f,out_f,k", [(32, 128, 256, 64), (33, 785, 257, 33), (300, 128, 256, 32), (1024, 1000, 3000, 17), (1023, 770, 12, 64)])
def test_few_token_forward_and_dx_on_the_matrix_cores(T, in_f, out_f, k):
    """fp32, k <= 64, on either side of the rule that chooses between the few-token kernels and the matrix cores, and without a
    workspace (which leaves neither of them)."""
    g = torch.Generator().manual_seed(T + k)
    x, dy, c = torch.randn(T, in_f, generator=g), torch.randn(T, out_f, generator=g), torch.randn(out_f, k, generator=g) / k ** 0.5
    W = c.double() @ ops.sq5_gen_2d(in_f, k, 8).double().cpu().t()
    assert _rel(hip.linear_fwd(x.cuda(), c.cuda(), in_f, out_f, in_f, 1, 8), x.double() @ W.t()) < 5e-6
    assert _rel(hip.linear_bwd_dx(dy.cuda(), c.cuda(), in_f, out_f, in_f, 1, 8), dy.double() @ W) < 5e-6
    y, xc, cc = torch.empty(T, out_f, device="cuda"), x.cuda(), c.cuda()
    d = hip._desc(T, in_f, out_f, cc, in_f, 1, 8, torch.float32, 0)
    rc = _lib.load().rdb_linear_fwd(y.data_ptr(), out_f, xc.data_ptr(), in_f, cc.data_ptr(), None, None, ctypes.byref(d), None, 0,
                                    torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and _rel(y, x.double() @ W.t()) < 5e-6


# the forward of up to 512 tokens is rdb_few.hip's: the same rule above that, with products of either kind the faster ones
@pytest.mark.parametrize("T,in_f,out_f,k", [(513, 128, 256, 64), (700, 785, 257, 33), (520, 2000, 100, 16), (600, 1030, 130, 8)])
def test_forward_and_dx_of_more_than_a_few_tokens(T, in_f, out_f, k):
    test_few_token_forward_and_dx_on_the_matrix_cores(T, in_f, out_f, k)


# every kind of block the pair of products in one launch is planned for (128 rows with one group and with two, 64 rows with two), with
# one and with several ranges on either side, whole and ragged tiles, pieces of four that are and are not aligned
@pytest.mark.parametrize("T,in_f,out_f,k,dtype", [(131, 259, 129, 65, torch.float32), (131, 259, 129, 65, torch.bfloat16), (2048, 768, 3072, 256, torch.float32),
                                                  (902, 720, 886, 606, torch.float32), (1552, 484, 2592, 20, torch.float32), (1000, 2001, 4000, 150, torch.bfloat16),
                                                  (6000, 700, 3001, 333, torch.bfloat16), (3000, 130, 257, 65, torch.bfloat16), (300, 2048, 2048, 512, torch.float32)])
def test_both_products_over_dy_in_one_launch(T, in_f, out_f, k, dtype):
    """dx and dC of one backward call, where t = dy . C and dC = dy^T . z share a launch, against float64, against the calls that want only
    one of them, and bit for bit run to run."""
    print(f"case pair T={T} in={in_f} out={out_f} k={k} {dtype}", flush=True)
    g = torch.Generator().manual_seed(T + k)
    x, dy = torch.randn(T, in_f, generator=g).to(dtype), torch.randn(T, out_f, generator=g).to(dtype)
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).to(dtype)
    N = ops.sq5_gen_2d(in_f, k, 8).double().cpu()
    leaves = [x.cuda().requires_grad_(), c.cuda().requires_grad_()]
    y = ops.linear(leaves[0], leaves[1], in_f, out_f, in_f, 1, 8, None, None)
    dx, dc = torch.autograd.grad(y, leaves, dy.cuda(), retain_graph=True)
    D = dy.double()
    tol = 5e-6 if dtype == torch.float32 else 2.0**-8   # fp32 sums throughout; bf16 results are rounded once, by at most 2^-8 of a value
    assert _rel(dx, (D @ c.double()) @ N.t()) < tol and _rel(dc, D.t() @ (x.double() @ N)) < tol
    again = torch.autograd.grad(y, leaves, dy.cuda(), retain_graph=True)
    assert torch.equal(dx, again[0]) and torch.equal(dc, again[1])
    assert _rel(torch.autograd.grad(y, leaves[:1], dy.cuda(), retain_graph=True)[0], dx.double().cpu()) < 2 * tol
    assert _rel(torch.autograd.grad(y, leaves[1:], dy.cuda())[0], dc.double().cpu()) < 2 * tol


@pytest.mark.parametrize("dtype,T,in_f,out_f,k", [(torch.float32, 2048, 768, 3072, 256), (torch.float32, 3000, 520, 100, 60), (torch.float32, 5000, 33, 2100, 257),
                                                  (torch.float32, 700, 40, 3000, 300), (torch.bfloat16, 4097, 301, 2999, 200), (torch.bfloat16, 3001, 77, 129, 50)])
def test_sums_of_the_coefficients_gradient_beside_dx(dtype, T, in_f, out_f, k):
    """Both sides of the line, dx of one tile and of many, in every kind of block; against float64."""
    from randumb_amd import SillyLinear, hip

    layer = SillyLinear(in_f, out_f, [k, k], [3, 4], bias=False, device="cuda", dtype=dtype, matrix_coef=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, 1.0, generator=g)
    x = torch.randn(T, in_f, generator=g, device="cuda").to(dtype).requires_grad_()
    dy = torch.randn(T, out_f, generator=g, device="cuda").to(dtype)
    y = layer(x)
    dx, dc = torch.autograd.grad(y, [x, layer.weight_coef], dy)
    N, x64 = hip.sq5_fill_2d(in_f, k, 3).double(), x.detach().double()
    want_dx, want_dc = (dy.double() @ layer.weight_coef.detach().double()) @ N.t(), dy.double().t() @ (x64 @ N)
    # fp32 sums; bf16: rounded once at the end
    tol = 3e-6 if dtype is torch.float32 else 2.0**-8
    for got, want in ((dx, want_dx), (dc, want_dc)):
        assert float((got.double() - want).norm() / want.norm()) < tol
    again = torch.autograd.grad(layer(x), [x, layer.weight_coef], dy)
    assert torch.equal(again[0], dx) and torch.equal(again[1], dc)
