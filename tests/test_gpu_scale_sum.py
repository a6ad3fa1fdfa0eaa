"""Gradient of the random bias's scale, added up by the last block of the launch that forms the shares: with scratch that holds anything, again on
the same scratch, and replayed from a graph."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# 256-wide tiles (130 of them, six blocks without one; more tiles than blocks), ranges (one tile; 12 of them; 130)
@pytest.mark.parametrize("T,in_f,out_f", [(8320, 512, 264), (16500, 776, 72), (200, 64, 4096), (513, 200, 2056), (3300, 640, 1600)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scale_gradient(T, in_f, out_f, dtype):
    from randumb_amd import _lib, hip

    print(f"case scale sum T={T} in={in_f} out={out_f} {dtype}", flush=True)
    lib = _lib.load()
    g = torch.Generator().manual_seed(T)
    x, dy, dx0 = (torch.randn(T, n, generator=g).bfloat16().cuda() for n in (in_f, out_f, in_f))
    s, ref = torch.tensor([0.37]).bfloat16().cuda(), ctypes.byref(hip._rbias_desc(T, in_f, out_f, 9))
    n = lib.rdb_linear_workspace_bytes(10, ref)
    ws, dx, ds = torch.full((n + 64,), 0x5A, dtype=torch.uint8, device="cuda"), dx0.clone(), torch.full((2,), 5.0, dtype=dtype, device="cuda")

    def call():
        dx.copy_(dx0)
        assert lib.rdb_linear_rbias_bwd_to(dx.data_ptr(), in_f, ds.data_ptr(), int(dtype is torch.bfloat16), dy.data_ptr(), out_f, x.data_ptr(), in_f,
                                           s.data_ptr(), ref, ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream) == 0

    call()
    first, first_dx = ds.clone(), dx.clone()
    R = hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).bfloat16().double()
    dot = dy.double() @ R
    # fp32 sums, and one rounding to bf16
    tol = 1e-5 * float(dot.norm() * x.double().norm()) + (2.0 ** -8 * abs(float((dot * x.double()).sum())) if dtype is torch.bfloat16 else 0.0)
    assert abs(float(first[0]) - float((dot * x.double()).sum())) < tol
    assert float(ds[1]) == 5.0 and bool((ws[n:] == 0x5A).all())
    call()
    assert torch.equal(ds, first) and torch.equal(dx, first_dx)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for fill in (0xFF, 0, 0x5A):
        ws[:n].fill_(fill)
        ds[0] = 7.0
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(ds, first) and torch.equal(dx, first_dx)
    hip.sync_check()
