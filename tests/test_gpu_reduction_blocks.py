"""Coefficient gradient whose partial sums are added beside the blocks of the input gradient: on the compute units that those leave free, or,
where these are fewer than half of the blocks that add, in a second round."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# units left free of 256, with 256 tokens and 64 features a unit of work: 8 (9 x 27 blocks, in groups of 8), 64 (6 x 32), 32 (7 x 32), none (8 x 32),
# more than elements to add (one block, and a part of a second)
@pytest.mark.parametrize("T,in_f,out_f,k", [(6784, 576, 264, 168), (8192, 384, 1160, 256), (8192, 448, 1160, 256), (8000, 512, 520, 72), (528, 64, 32, 64), (528, 384, 40, 64)])
def test_coefficient_gradient_against_float64(T, in_f, out_f, k):
    from randumb_amd import hip

    print(f"case reduction blocks T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator().manual_seed(in_f)
    x, dy = (torch.randn(T, n, generator=g).bfloat16().cuda() for n in (in_f, out_f))
    c = (torch.randn(out_f, k, generator=g) * 0.05).bfloat16().cuda()
    dx, dc = hip.linear_bwd_projected(dy, hip.linear_project(x, k, out_f, 9, c), c, in_f, 9)
    N = hip.sq5_fill_2d(in_f, k, 9).double()
    dc_ref, dx_ref = dy.double().t() @ (x.double() @ N), dy.double() @ c.double() @ N.t()
    # two bf16 roundings at most (z or t, then the result): 2^-9 each at most, a third of that as a norm
    assert float((dc.double() - dc_ref).norm() / dc_ref.norm()) < 4e-3 and float((dx.double() - dx_ref).norm() / dx_ref.norm()) < 4e-3
    hip.sync_check()
