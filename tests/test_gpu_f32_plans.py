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


@pytest.mark.parametrize("tokens,in_f,out_f,k", [(51, 205, 468, 43), (137, 764, 161, 27), (66, 2253, 280, 28), (44, 226, 251, 19), (725, 246, 906, 44),
                                                 (300, 512, 1024, 64)])
def test_few_token_products_are_no_further_from_64_bits_than_fp32_ones(tokens, in_f, out_f, k):
    """Layers of few tokens and coefficients, which the vector ALU's fp32 kernels may run as well, against the same two products in
    the library's fp32.  Its sums are cut into pieces too, so neither is systematically ahead: 1.1 covers that."""
    from randumb_amd import hip

    g = torch.Generator(device="cuda").manual_seed(k)
    x, dy, c = (torch.randn(*s, device="cuda", generator=g) for s in ((tokens, in_f), (tokens, out_f), (out_f, k)))
    N = hip.sq5_fill_2d(in_f, k, 7)
    off = lambda a, b: float((a.double() - b).norm() / b.norm())
    y, dx = hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 7), hip.linear_bwd_dx(dy, c, in_f, out_f, in_f, 1, 7)
    dc, _ = hip.linear_bwd_dcoef(dy, x, k, out_f, in_f, out_f, in_f, 1, 7)
    z, t = x.double() @ N.double(), dy.double() @ c.double()
    for name, got, plain, exact in (("y", y, (x @ N) @ c.t(), z @ c.double().t()), ("dx", dx, (dy @ c) @ N.t(), t @ N.double().t()),
                                    ("dcoef", dc, dy.t() @ (x @ N), dy.double().t() @ z)):
        print(f"  {name}: {off(got, exact):.2e}, in fp32 {off(plain, exact):.2e}", flush=True)
        assert off(got, exact) <= 1.1 * off(plain, exact), name
