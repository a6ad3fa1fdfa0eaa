"""Contractions over tokens whose rows lie so far apart that the 32-bit offset of a row behind the last one comes round to a row that exists."""
import pytest
import torch

pytestmark = pytest.mark.gpu

T = 7


def _far(t, ld, fill):
    assert T * ld < 2**29   # taken as it is
    far = torch.full(((T - 1) * ld + t.shape[1],), fill, device="cuda", dtype=torch.bfloat16).as_strided(t.shape, (ld, 1))
    far.copy_(t)
    return far


# dy^T . x formed and contracted with the noise (the offset of row 32 is 2^32 bytes: that of row 0), and dy^T . z on 128-wide and on 256-wide tiles, where z
# is zero behind the last token (that of row 33 lies 528 bytes ahead of row 1: between the rows)
@pytest.mark.parametrize("route", ["weight_gradient", "projected", "projected_256"])
def test_coefficient_gradient_counts_each_token_once(route):
    from randumb_amd import hip

    print(f"case far rows {route}", flush=True)
    in_f, out_f, k = (256, 192, 64) if route == "weight_gradient" else (264, 200, 320)
    g = torch.Generator(device="cuda").manual_seed(1)
    x, dy = (torch.randn(T, n, device="cuda", generator=g).bfloat16() for n in (in_f, out_f))
    C = (torch.randn(out_f, k, device="cuda", generator=g) * k**-0.5).bfloat16()
    N = hip.sq5_fill_2d(in_f, k, 9).double()
    want = dy.double().t() @ (x.double() @ N)
    if route == "weight_gradient":
        got, ds = hip.linear_bwd_dcoef(_far(dy, 2**26, 0.0), _far(x, 2**26, 0.0), k, out_f, in_f, out_f, in_f, 1, 9, want_scale_bias_grad=True)
        R = hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double()
        dw = dy.double().t() @ x.double()
        assert abs(float(ds) - float((dw * R).sum())) < 4e-3 * float(dw.norm() * R.norm())   # dW rounded to bf16: 2^-9 at most
    else:
        before = hip.set_big_tiles(2 if route == "projected_256" else 0)
        try:
            state = hip.linear_project(x, k, out_f, 9, C)
            got = hip.linear_bwd_projected(_far(dy, 2**26 - 8, float("nan")), state, C, in_f, 9)[1]
        finally:
            hip.set_big_tiles(before)
    assert float((got.double() - want).norm() / want.norm()) < 8e-3   # two operands rounded to bf16 (N and z, or dW and N): 2^-9 each at most
