"""The input of a layer with a random bias, kept for the backward pass by hooks in another dtype."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# gradients in two calls and in one (many tiles), by the Python functions, and of sizes that are no multiples of 8
@pytest.mark.parametrize("T,in_f,out_f,k,python", [(300, 256, 192, 64, False), (8100, 584, 72, 40, False), (300, 256, 192, 64, True), (130, 133, 99, 50, False)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_is_read_as_what_it_is(T, in_f, out_f, k, python, dtype):
    from randumb_amd import SillyLinear, ops

    print(f"case restored input T={T} in={in_f} out={out_f} {dtype}", flush=True)
    layer = SillyLinear(in_f, out_f, [k, k], [1, 2], bias=False, rt_bias=True, device="cuda", dtype=torch.bfloat16, matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, 0.05)
    x = torch.randn(T, in_f, device="cuda").bfloat16().requires_grad_()
    dy = torch.randn(T, out_f, device="cuda").bfloat16()
    wanted = [x, layer.weight_coef, layer.weight_scale_bias]

    def grads():
        y = ops._ProjectedFunction.apply(x, layer.weight_coef, in_f, out_f, 1, None, layer.weight_scale_bias) if python else layer(x)
        return torch.autograd.grad(y, wanted, dy)

    want, restored = grads(), []

    def unpack(t):
        if t.shape != (T, in_f):
            return t
        restored.append(t)
        return t.to(dtype)   # a wider one: the same values

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        got = grads()
    assert restored
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and torch.equal(a, b)
