"""The random bias's share of layers with many tiles: R written to memory first, tiles of 192 or 256 features, R beside the projection."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles of 192 features (as many rounds of them as of 256, at 256 compute units) whose last one has 8, 40 and 8 features, and of 256 with a last one of 8;
# the last token tile of 36, 52, 1 and 8 tokens
@pytest.mark.parametrize("T,in_f,out_f", [(8100, 584, 72), (5300, 1000, 136), (16385, 200, 264), (16264, 264, 72)])
def test_input_gradient_against_float64(T, in_f, out_f):
    from randumb_amd import _lib, hip

    print(f"case rbias tiles T={T} in={in_f} out={out_f}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    ref = ctypes.byref(hip._rbias_desc(T, in_f, out_f, 9))
    s = torch.tensor([0.37]).bfloat16().cuda()
    R = hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).bfloat16().double()   # what the kernels multiply
    FULL = 10
    n = lib.rdb_linear_workspace_bytes(FULL, ref)
    assert n >= 2 * in_f * out_f   # room for R
    ws = torch.full((n + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    x, dy, dx0 = (torch.randn(T, cols + 8, generator=g).bfloat16().cuda() for cols in (in_f, out_f, in_f))
    dx, ds, dx_only = dx0.clone(), torch.full((2,), 5.0, device="cuda"), dx0.clone()
    args = (dy.data_ptr(), out_f + 8)
    assert lib.rdb_linear_rbias_bwd(dx.data_ptr(), in_f + 8, ds.data_ptr(), *args, x.data_ptr(), in_f + 8, s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    assert lib.rdb_linear_rbias_bwd(dx_only.data_ptr(), in_f + 8, None, *args, None, 0, s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    assert torch.equal(dx, dx_only) and torch.equal(dx[:, in_f:], dx0[:, in_f:]) and float(ds[1]) == 5.0 and bool((ws[n:] == 0x5A).all())
    dot = dy[:, :out_f].double() @ R
    want = dx0[:, :in_f].double() + s.double() * dot
    assert float((dx[:, :in_f].double() - want).norm() / want.norm()) < 2e-3   # one rounding to bf16: 2^-9 at most, 1.13e-3 as a norm
    xd = x[:, :in_f].double()
    assert abs(float(ds[0]) - float((dot * xd).sum())) < 1e-5 * float(dot.norm() * xd.norm())   # fp32 sums


# R beside a projection in one range of its contraction, in several, and ahead of one on 256-wide tiles (a launch of its own); sizes that are no multiple of
# a tile, fragment or k-step
@pytest.mark.parametrize("T,in_f,out_f,k", [(2040, 136, 2056, 8), (2100, 2056, 2008, 72), (8200, 264, 520, 520)])
def test_forward_against_float64(T, in_f, out_f, k):
    from randumb_amd import SillyLinear, hip

    print(f"case rbias forward T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    layer = SillyLinear(in_f, out_f, [k, k], [9, 10], bias=False, rt_bias=True, device="cuda", dtype=torch.bfloat16, matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, k**-0.5, generator=g)
        layer.weight_scale_bias.fill_(0.37)
    x = torch.randn(T, in_f, device="cuda", generator=g).bfloat16().requires_grad_()
    y = layer(x)
    N, R = hip.sq5_fill_2d(in_f, k, 9).double(), hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double()
    want = x.detach().double() @ (layer.weight_coef.detach().double() @ N.t() + layer.weight_scale_bias.detach().double() * R).t()
    assert float((y.detach().double() - want).norm() / want.norm()) < 6e-3   # N, z, R and y rounded to bf16 once each, 1.13e-3 as a norm; 2^-9 at most
