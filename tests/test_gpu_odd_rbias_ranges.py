"""Input gradient of bf16 layers of odd sizes with a random bias: dy . R in ranges of the output features, as many as the workspace holds once t and
dC's partial matrices are used up, added onto dx by a kernel of its own."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# several ranges, one column, a last range of part of a stage; room for one range only (k = 3); ragged in every direction
@pytest.mark.parametrize("T,in_f,out_f,k", [(502, 527, 2918, 251), (130, 33, 4099, 30), (97, 1031, 999, 3), (942, 729, 6529, 92)])
@pytest.mark.parametrize("pad", [0, 5])
def test_against_float64(T, in_f, out_f, k, pad):
    from randumb_amd import _lib, hip

    print(f"case odd rbias ranges T={T} in={in_f} out={out_f} k={k} pad={pad}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    x, dy, c = (torch.randn(*m, generator=g).bfloat16().cuda() for m in ((T, in_f + pad), (T, out_f + pad), (out_f, k)))
    s, ref = torch.tensor([0.37]).bfloat16().cuda(), ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0))
    kept = torch.zeros(lib.rdb_linear_kept_bytes(ref), dtype=torch.uint8, device="cuda")
    y = torch.empty(T, out_f, dtype=torch.bfloat16, device="cuda")
    assert lib.rdb_linear_fwd_kept(y.data_ptr(), out_f, kept.data_ptr(), x.data_ptr(), in_f + pad, c.data_ptr(), s.data_ptr(), None, ref, stream) == 0
    n = lib.rdb_linear_workspace_bytes(7, ref)
    out = []
    for want_s in (True, True, False):
        ws = torch.full((n + 64,), 0x5A, dtype=torch.uint8, device="cuda")
        dx, dc, ds = torch.full((T + 1, in_f + pad), 7.0, dtype=torch.bfloat16, device="cuda"), torch.empty(out_f, k, device="cuda"), torch.full((2,), 5.0, device="cuda")
        assert lib.rdb_linear_bwd_kept(dx.data_ptr(), in_f + pad, dc.data_ptr(), 0, ds.data_ptr() if want_s else None, dy.data_ptr(), out_f + pad, x.data_ptr(),
                                       in_f + pad, kept.data_ptr(), c.data_ptr(), s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
        assert bool((ws[n:] == 0x5A).all()) and bool((dx[T] == 7.0).all()) and bool((dx[:, in_f:] == 7.0).all()) and float(ds[1]) == 5.0
        out.append((dx[:T, :in_f], dc, float(ds[0])))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][0], out[2][0]) and out[0][2] == out[1][2]
    xd, dyd, cd = x[:, :in_f].double(), dy[:, :out_f].double(), c.double()
    N, R = hip.sq5_fill_2d(in_f, k, 5).double(), hip.sq5_fill_1d(out_f * in_f, 5).view(out_f, in_f).double()
    dot = dyd @ R
    want = dyd @ cd @ N.t() + s.double() * dot
    # dx rounded to bf16 twice, the low-rank share and the sum: 2^-9 each at most, a third of that as a norm
    assert float((out[0][0].double() - want).norm() / want.norm()) < 4e-3
    assert abs(out[0][2] - float((dot * xd).sum())) < 1e-5 * float(dot.norm() * xd.norm())   # fp32 sums
    hip.sync_check()
