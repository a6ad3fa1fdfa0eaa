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


# backward in one call: tiles of 192 features with rows of dx that are no whole lines and that are, tiles of 256
@pytest.mark.parametrize("T,in_f,out_f,k", [(8100, 584, 72, 40), (8100, 768, 72, 72), (8190, 1024, 136, 200)])
def test_gradients_in_one_call_against_float64(T, in_f, out_f, k):
    from randumb_amd import _lib, hip, ops

    print(f"case rbias autograd T={T} in={in_f} out={out_f} k={k}", flush=True)
    assert hip.linear_projection_preferred(T, in_f, out_f, k)
    assert _lib.load().rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_BWD_PROJECTED_RBIAS, ctypes.byref(hip._proj_desc(T, in_f, out_f, k, 9))) > 0
    g = torch.Generator(device="cuda").manual_seed(T)
    x, dy, C = (torch.randn(*s, device="cuda", generator=g).bfloat16() for s in ((T, in_f), (T, out_f), (out_f, k)))
    C = (C.float() * k**-0.5).bfloat16()
    s = torch.tensor([0.37], device="cuda").bfloat16()

    def grads(x=x, C=C, s=s, dy=dy, frozen=()):
        leaves = [t.detach().requires_grad_(name not in frozen) for name, t in (("x", x), ("C", C), ("s", s))]
        y = ops.linear(leaves[0], leaves[1], in_f, out_f, in_f, 1, 9, leaves[2], None)
        got = iter(torch.autograd.grad(y, [t for t in leaves if t.requires_grad], dy))
        return [next(got) if t.requires_grad else None for t in leaves]

    def wide(t, columns, first=0):   # the same rows as a slice of a wider matrix
        out = torch.full((t.shape[0], t.shape[1] + columns), 5.0, device="cuda", dtype=t.dtype)[:, first:first + t.shape[1]]
        return out.copy_(t)

    dx, dC, ds = grads()
    N, R, xd, dyd, Cd = hip.sq5_fill_2d(in_f, k, 9).double(), hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double(), x.double(), dy.double(), C.double()
    want = dyd @ Cd @ N.t() + s.double() * dyd @ R
    # N, t or z, R and the result rounded to bf16 once each: 1.13e-3 as a norm, 2^-9 at most
    assert dx.dtype == torch.bfloat16 and float((dx.double() - want).norm() / want.norm()) < 6e-3
    want = dyd.t() @ (xd @ N)
    assert dC.dtype == torch.bfloat16 and float((dC.double() - want).norm() / want.norm()) < 6e-3
    dot = dyd @ R.bfloat16().double()
    exact, bound = float((dot * xd).sum()), 1e-5 * float(dot.norm() * xd.norm())   # fp32 sums
    assert ds.dtype == torch.bfloat16 and abs(float(ds) - exact) < bound + 2**-8 * abs(exact)

    def same(got, *wanted):
        for a, b in zip(got, wanted):
            assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and torch.equal(a, b)))

    same(grads(frozen=["s"]), dx, dC, None)
    same(grads(frozen=["x"]), None, dC, ds)
    got = grads(s=s.float())   # the scale as fp32: its gradient too
    same(got[:2], dx, dC)
    assert got[2].dtype == torch.float32 and torch.equal(got[2].bfloat16(), ds) and abs(float(got[2]) - exact) < bound
    same(grads(dy=wide(dy, 8)), dx, dC, ds)       # read where it is
    same(grads(dy=wide(dy, 9, 1)), dx, dC, ds)    # rows that are not 16-byte aligned: copied
    same(grads(x=wide(x, 8)), dx, dC, ds)
    with torch.autograd.graph.save_on_cpu():
        same(grads(), dx, dC, ds)
    # the coefficients frozen: both shares of dx apart, rounded once more
    got, want = grads(frozen=["C"]), dyd @ Cd @ N.t() + s.double() * dyd @ R
    assert float((got[0].double() - want).norm() / want.norm()) < 6e-3 and got[1] is None
    assert abs(float(got[2]) - exact) < bound + 2**-8 * abs(exact)
