"""The extension module that issues ops.linear's calls: its rule of path against the Python restatement (CPU), and its autograd
functions against the Python ones on the GPU."""
import ctypes
import itertools

import pytest
import torch

from randumb_amd import _lib, hip


def test_the_librarys_rule_is_the_python_rule():
    L = _lib.load()
    sizes = (8, 64, 256, 768, 1000, 1536, 4096)
    for dtype in (torch.bfloat16, torch.float32):
        for T, i, o, k in itertools.product((1, 64, 96, 97, 1024, 1025, 8192), sizes, sizes, (8, 36, 64, 72, 256, 1024)):
            d = hip._proj_desc(T, i, o, k, 0, dtype, dtype)
            want = hip.linear_projection_preferred(T, i, o, k, dtype)
            assert bool(L.rdb_linear_projection_preferred(ctypes.byref(d))) == bool(want), (T, i, o, k, dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("T,in_f,out_f,k,dtype,rt_bias,bias", [
    (300, 128, 256, 32, torch.bfloat16, False, "dense"),
    (200, 136, 264, 40, torch.bfloat16, True, None),
    (130, 77, 55, 9, torch.bfloat16, False, None),
    (16, 2048, 512, 72, torch.bfloat16, False, None),
    (1100, 96, 200, 33, torch.float32, False, "dense"),
    (40, 96, 50, 16, torch.float32, True, "random"),
])
def test_extension_matches_the_python_functions(T, in_f, out_f, k, dtype, rt_bias, bias):
    import randumb_amd as ra
    from randumb_amd import ops

    g = torch.Generator().manual_seed(T)
    layer = ra.SillyLinear(in_f, out_f, [k, 12], [5, 6], bias=bias == "random", rt_bias=rt_bias, matrix_coef=True).to(dtype).cuda()
    with torch.no_grad():
        layer.weight_coef.copy_(torch.randn(out_f, k, generator=g) * 0.05)
        if bias == "random":
            layer.bias_coef.copy_(torch.randn(12, generator=g) * 0.05)
    x = torch.randn(T, in_f, generator=g).to(dtype).cuda().requires_grad_()
    dy = torch.randn(T, out_f, generator=g).to(dtype).cuda()
    b = torch.randn(out_f, generator=g).to(dtype).cuda().requires_grad_() if bias == "dense" else layer.bias
    sb = layer.weight_scale_bias if rt_bias else None
    leaves = [x, layer.weight_coef] + ([sb] if rt_bias else []) + ([b] if bias == "dense" else [layer.bias_coef] if bias else [])
    args = (x, layer.weight_coef, in_f, out_f, in_f, 1, 5, sb, b)

    def grads(y):
        return [y.detach()] + list(torch.autograd.grad(y, leaves, dy))

    got = grads(ops.linear(*args))
    if hip.linear_projection_preferred(T, in_f, out_f, k, dtype):
        want = grads(ops._ProjectedFunction.apply(x, layer.weight_coef, in_f, out_f, 5, b, sb))
    else:
        want = grads(ops._OneCallFunction.apply(*args))
    d = hip._desc(T, in_f, out_f, layer.weight_coef, in_f, 1, 5, dtype, 0)
    if _lib.load().rdb_linear_kept_bytes(ctypes.byref(d)):   # z kept from the forward pass: the same products, summed in other ranges
        tol = 1e-6 if dtype == torch.float32 else 5e-3
        for a, w in zip(got, want):
            assert a.dtype == w.dtype and a.shape == w.shape and float((a.double() - w.double()).norm() / w.double().norm()) < tol
        return
    if bias == "random":   # its coefficients' gradient: added up in another order than the column sums and their contraction
        a, w = got.pop(), want.pop()
        assert a.dtype == w.dtype and a.shape == w.shape and float((a - w).norm() / w.norm()) < 1e-6
    for a, w in zip(got, want):
        assert a.dtype == w.dtype and a.shape == w.shape and torch.equal(a, w)
    with torch.no_grad():
        assert torch.equal(ops.linear(*args), got[0])
        assert torch.equal(layer.requires_grad_(False)(x.detach().view(1, T, in_f)).view(T, out_f) if b is layer.bias else got[0], got[0])
