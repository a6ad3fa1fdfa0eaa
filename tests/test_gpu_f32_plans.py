"""fp32-accurate products in groups and ranges (f32_gemm_kernel): sizes at the edges of tiles, stages, groups and ranges, with rows
that start at any element, against float64."""
import pytest
import torch

from randumb_amd import hip, ops

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


# one group and several (few / many tiles, short / long contractions), remainders of 1 .. 3 elements along every extent
@pytest.mark.parametrize("T,in_f,out_f,k", [(129, 68, 132, 68), (257, 1392, 424, 104), (300, 515, 1501, 71), (1030, 2049, 131, 129),
                                            (2050, 770, 1030, 256), (4097, 333, 259, 100), (130, 3071, 65, 66)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_products(T, in_f, out_f, k, dtype):
    g = torch.Generator().manual_seed(T + in_f)
    x, dy = torch.randn(T, in_f, generator=g).to(dtype), torch.randn(T, out_f, generator=g).to(dtype)
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).to(dtype)
    noise = ops.sq5_gen_2d(in_f, k, 5).double().cpu()
    z = x.double() @ noise
    xs, cs = x.cuda().requires_grad_(), c.cuda().requires_grad_()
    y = ops.linear(xs, cs, in_f, out_f, in_f, 1, 5, None, None)
    dx, dc = torch.autograd.grad(y, [xs, cs], dy.cuda())
    tol = 2e-6 if dtype == torch.float32 else 6e-3
    assert _rel(y.detach(), z @ c.double().t()) < tol
    assert _rel(dx, dy.double() @ c.double() @ noise.t()) < tol
    assert _rel(dc, dy.double().t() @ z) < tol


@pytest.mark.parametrize("rows,k,row_len", [(333, 129, 1027), (70, 300, 4001)])
def test_materialise_and_adjoint(rows, k, row_len):
    g = torch.Generator().manual_seed(rows)
    c, d = torch.randn(rows, k, generator=g), torch.randn(rows, row_len, generator=g)
    noise = ops.sq5_gen_2d(row_len, k, 3).double().cpu()
    assert _rel(hip.materialize_fwd(c.cuda(), (rows, row_len), (row_len, 1), 3, None, False), c.double() @ noise.t()) < 2e-6
    assert _rel(hip.materialize_bwd(d.cuda(), k, 3, rows), d.double() @ noise) < 2e-6
