"""Layers with a fused random bias and many tiles through autograd: the extension module and the Python function, which ask the library the same way."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# both shares of either product in one call, in tiles of 192 and of 256 features, dx's rows whole lines or not; k too long for that backward; sums of ranges
# both ways; a forward product with R in memory only
@pytest.mark.parametrize("T,in_f,out_f,k", [(8100, 584, 72, 40), (8100, 768, 72, 72), (8190, 1024, 136, 200), (2100, 2056, 2056, 72), (8200, 584, 520, 520),
                                            (270, 2912, 632, 64), (2040, 136, 2056, 72)])
@pytest.mark.parametrize("bias", [False, True])
def test_extension_and_python_function_agree_to_the_bit(T, in_f, out_f, k, bias):
    from randumb_amd import ops

    print(f"case rbias functions T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    x, dy, C = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((T, in_f), (T, out_f), (out_f, k)))
    s, b = torch.tensor([0.37], device="cuda").bfloat16(), torch.randn(out_f, device="cuda", generator=g).bfloat16() if bias else None
    leaves = [t.requires_grad_() for t in (x, C, s)]
    results = []
    for layer in (lambda: ops._lib.extension().linear_projected(x, C, in_f, out_f, 9, b, None, -1, s), lambda: ops._ProjectedFunction.apply(x, C, in_f, out_f, 9, b, s)):
        results.append([layer().detach()])
        for wanted in (leaves, [x, C], [x, s], [C, s]):
            for t in leaves:
                t.requires_grad_(any(t is w for w in wanted))
            results[-1] += torch.autograd.grad(layer(), wanted, dy)
        for t in leaves:
            t.requires_grad_()
    for a, w in zip(*results):
        assert a.dtype == w.dtype and torch.equal(a, w)
