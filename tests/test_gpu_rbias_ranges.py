"""The random bias's share of layers with few tiles: the contraction in ranges, their sums added up by a kernel of its own."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# the contraction of one direction or of both is long enough for ranges: last ranges of one stage and of part of one, tiles of one token and of
# one piece of eight features, more ranges than are fetched at a time
@pytest.mark.parametrize("T,in_f,out_f", [(1, 4096, 8), (255, 1000, 72), (257, 72, 2056), (300, 264, 5896), (513, 2312, 520)])
def test_ranges_against_float64(T, in_f, out_f):
    from randumb_amd import _lib, hip

    print(f"case rbias ranges T={T} in={in_f} out={out_f}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    ref = ctypes.byref(hip._rbias_desc(T, in_f, out_f, 9))
    s = torch.tensor([0.37]).bfloat16().cuda()
    R = hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).bfloat16().double()   # what the kernels multiply
    FWD, BWD, FULL = 8, 6, 10

    def scratch(op, extra=64):
        n = lib.rdb_linear_workspace_bytes(op, ref)
        return n, torch.full((n + extra,), 0x5A, dtype=torch.uint8, device="cuda")

    def padded(rows, cols):
        return torch.randn(rows, cols + 8, generator=g).bfloat16().cuda()

    x, dy, y0, dx0 = padded(T, in_f), padded(T, out_f), padded(T, out_f), padded(T, in_f)
    sizes = [lib.rdb_linear_workspace_bytes(op, ref) for op in (FWD, FULL)]
    assert sizes[0] > 0 or sizes[1] > lib.rdb_linear_workspace_bytes(BWD, ref)   # one of the directions takes ranges
    n, ws = scratch(FWD)
    y, y_one, dx, dx_one, dx_only = y0.clone(), y0.clone(), dx0.clone(), dx0.clone(), dx0.clone()
    ds, ds_one = (torch.full((2,), 5.0, device="cuda") for _ in range(2))
    for out, size in ((y, n), (y_one, 0)):
        assert lib.rdb_linear_rbias_fwd_ws(out.data_ptr(), out_f + 8, x.data_ptr(), in_f + 8, s.data_ptr(), ref, ws.data_ptr() if size else None, size, stream) == 0
    assert bool((ws[n:] == 0x5A).all())
    n, ws = scratch(FULL)
    for out, d, size in ((dx, ds, n), (dx_one, ds_one, lib.rdb_linear_workspace_bytes(BWD, ref))):
        assert lib.rdb_linear_rbias_bwd(out.data_ptr(), in_f + 8, d.data_ptr(), dy.data_ptr(), out_f + 8, x.data_ptr(), in_f + 8, s.data_ptr(), ref,
                                        ws.data_ptr(), size, stream) == 0
    assert lib.rdb_linear_rbias_bwd(dx_only.data_ptr(), in_f + 8, None, dy.data_ptr(), out_f + 8, None, 0, s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    ds16 = torch.full((2,), 5.0, dtype=torch.bfloat16, device="cuda")   # the same sum in bf16
    assert lib.rdb_linear_rbias_bwd_to(dx0.clone().data_ptr(), in_f + 8, ds16.data_ptr(), 1, dy.data_ptr(), out_f + 8, x.data_ptr(), in_f + 8, s.data_ptr(),
                                       ref, ws.data_ptr(), n, stream) == 0
    assert torch.equal(ds16, ds.bfloat16())
    assert bool((ws[n:] == 0x5A).all()) and float(ds[1]) == 5.0 and float(ds_one[1]) == 5.0
    assert torch.equal(dx, dx_only)
    for out, old, cols in ((y, y0, out_f), (y_one, y0, out_f), (dx, dx0, in_f), (dx_one, dx0, in_f)):
        assert torch.equal(out[:, cols:], old[:, cols:])   # nothing beside the rows
    xd, dyd, sd = x[:, :in_f].double(), dy[:, :out_f].double(), s.double()
    want_y, dot = y0[:, :out_f].double() + sd * (xd @ R.t()), dyd @ R
    want_dx = dx0[:, :in_f].double() + sd * dot
    for out, want in ((y[:, :out_f], want_y), (y_one[:, :out_f], want_y), (dx[:, :in_f], want_dx), (dx_one[:, :in_f], want_dx)):
        assert float((out.double() - want).norm() / want.norm()) < 2e-3   # one rounding to bf16: 2^-9 at most, 1.13e-3 as a norm
    for d in (ds, ds_one):   # fp32 sums
        assert abs(float(d[0]) - float((dot * xd).sum())) < 1e-5 * float(dot.norm() * xd.norm())
