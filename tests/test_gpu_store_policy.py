"""Results written through the caches, streamed past them and with plain stores: by the size of the pass and the rows' alignment."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows of whole lines, 64 MB of activations and just above; rows of parts of lines
@pytest.mark.parametrize("T,in_f,out_f", [(8192, 192, 3904), (8200, 192, 3904), (8192, 3904, 192), (8200, 3904, 192), (8192, 200, 3880), (2048, 1544, 1032)])
@pytest.mark.parametrize("rt_bias", [False, True])
def test_layer_against_float64(T, in_f, out_f, rt_bias):
    from randumb_amd import SillyLinear, hip

    print(f"case stores T={T} in={in_f} out={out_f} rt_bias={rt_bias}", flush=True)
    k = 64
    g = torch.Generator(device="cuda").manual_seed(T + in_f)
    layer = SillyLinear(in_f, out_f, [k, k], [9, 10], bias=False, rt_bias=rt_bias, device="cuda", dtype=torch.bfloat16, matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, k**-0.5, generator=g)
        if rt_bias:
            layer.weight_scale_bias.fill_(0.37)
    x = torch.randn(T, in_f, device="cuda", generator=g).bfloat16().requires_grad_()
    dy = torch.randn(T, out_f, device="cuda", generator=g).bfloat16()
    y = layer(x)
    (dx,) = torch.autograd.grad(y, [x], dy) if not rt_bias else torch.autograd.grad(y, [x, layer.weight_coef, layer.weight_scale_bias], dy)[:1]
    W = layer.weight_coef.detach().double() @ hip.sq5_fill_2d(in_f, k, 9).double().t()
    if rt_bias:
        W += 0.37109375 * hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double()   # 0.37 in bf16
    # N, z or t, R and the result rounded to bf16 once each (without the one call both ways, dx twice), 1.13e-3 as a norm; 2^-9 at most
    for got, want in ((y, x.detach().double() @ W.t()), (dx, dy.double() @ W)):
        assert float((got.detach().double() - want).norm() / want.norm()) < 6e-3
