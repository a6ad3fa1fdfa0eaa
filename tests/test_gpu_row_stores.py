"""Row stores of the kernels that keep a token's contraction in registers: rows of y and dx that are whole 128-byte lines and rows that are
not take different kernels, which give the same bits and write nothing beside their rows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 64, 64, 64), (257, 128, 320, 40), (300, 72, 264, 128), (515, 328, 1000, 192), (70, 1032, 96, 256)])
@pytest.mark.parametrize("bias", [False, True])
def test_rows_of_whole_lines_and_others(T, in_f, out_f, k, bias):
    from randumb_amd import _lib, hip

    print(f"case row stores T={T} in={in_f} out={out_f} k={k} bias={bias}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    x, dy = torch.randn(T, in_f, generator=g).bfloat16().cuda(), torch.randn(T, out_f, generator=g).bfloat16().cuda()
    c = (torch.randn(out_f, k, generator=g) * 0.05).bfloat16().cuda()
    b = torch.randn(out_f, generator=g).bfloat16().cuda() if bias else None
    ref = ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0))
    size = lib.rdb_linear_workspace_bytes(4, ref)
    ws, kept = torch.empty(size, dtype=torch.uint8, device="cuda"), []
    # (leading dimension, offset of the first row) in elements: whole lines, a padded stride, a base inside a line, neither
    for up, start in ((64, 0), (8, 0), (64, 8), (8, 40)):
        ldy, ldx = -(-out_f // up) * up + (8 if up == 8 else 0), -(-in_f // up) * up + (8 if up == 8 else 0)
        y, dx = (torch.full((start + T * n,), 7.0, dtype=torch.bfloat16, device="cuda") for n in (ldy, ldx))
        state, dc = torch.empty(lib.rdb_linear_projection_bytes(ref), dtype=torch.uint8, device="cuda"), torch.empty_like(c)
        assert lib.rdb_linear_project_fwd(y.data_ptr() + 2 * start, ldy, state.data_ptr(), x.data_ptr(), in_f, c.data_ptr(),
                                          b.data_ptr() if bias else None, ref, stream) == 0
        assert lib.rdb_linear_bwd_projected_to(dx.data_ptr() + 2 * start, ldx, dc.data_ptr(), 1, dy.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), ref,
                                               ws.data_ptr(), size, stream) == 0
        for out, n, cols in ((y, ldy, out_f), (dx, ldx, in_f)):
            assert bool((out[:start] == 7.0).all()) and bool((out[start:].view(T, n)[:, cols:] == 7.0).all())
        kept.append((y[start:].view(T, ldy)[:, :out_f], dx[start:].view(T, ldx)[:, :in_f], dc))
    for got in kept[1:]:
        assert all(torch.equal(a, w) for a, w in zip(got, kept[0]))
    N = hip.sq5_fill_2d(in_f, k, 5).double()
    y_ref, dx_ref = x.double() @ N @ c.double().t() + (b.double() if bias else 0.0), dy.double() @ c.double() @ N.t()
    # two bf16 roundings (z or t, then the result): 2^-9 each at most, a third of that as a norm
    assert float((kept[0][0].double() - y_ref).norm() / y_ref.norm()) < 4e-3 and float((kept[0][1].double() - dx_ref).norm() / dx_ref.norm()) < 4e-3
    hip.sync_check()
