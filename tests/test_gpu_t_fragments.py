"""t = dy . C with C's fragments loaded one or two stages of 128 output features ahead, by how many blocks there are, and from 2048 output
features on in ranges of 512 or more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _backward(T, in_f, out_f, k, n):
    from randumb_amd import hip

    print(f"case t fragments T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator().manual_seed(out_f)
    c = (torch.randn(out_f, k, generator=g) * 0.05).bfloat16().cuda()
    x, dy = torch.randn(n, in_f, generator=g).bfloat16().cuda()[:T], torch.randn(n, out_f, generator=g).bfloat16().cuda()[:T]
    return x, dy, c, hip.linear_bwd_projected(dy, hip.linear_project(x, k, out_f, 9, c), c, in_f, 9)


# one stage, two, three (the last of them past the end), a part of the last; 2048 features and more: four ranges, two to eight, the last one short
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 64, 8, 8), (65, 96, 136, 40), (200, 64, 384, 136), (130, 72, 1000, 256), (300, 64, 2048, 64),
                                            (1056, 72, 3080, 240), (97, 64, 8200, 24), (2050, 64, 2056, 200),
                                            (97, 64, 2568, 264), (300, 520, 8192, 512), (2800, 320, 4104, 304)])
def test_against_float64(T, in_f, out_f, k):
    from randumb_amd import hip

    x, dy, c, (dx, dc) = _backward(T, in_f, out_f, k, T)
    N = hip.sq5_fill_2d(in_f, k, 9).double()
    dc_ref, dx_ref = dy.double().t() @ (x.double() @ N), dy.double() @ c.double() @ N.t()
    # two bf16 roundings at most (z or t, then the result): 2^-9 each at most, a third of that as a norm; few values: the bound itself
    tol = 4e-3 if T * min(in_f, out_f, k) > 1000 else 2.0 ** -8
    assert float((dc.double() - dc_ref).norm() / dc_ref.norm()) < tol and float((dx.double() - dx_ref).norm() / dx_ref.norm()) < tol
    hip.sync_check()


def test_same_rows_on_either_side_of_the_line():
    # 128 blocks of 64 tokens are half of the compute units, 129 are more
    few, more = (_backward(T, 72, 1000, 104, 8256)[3][0] for T in (8192, 8256))
    assert torch.equal(few, more[:8192])
