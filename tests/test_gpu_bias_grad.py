"""Gradient of a pseudorandom bias: a dy small enough for one launch, and the sizes around the line to two."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one output, one row, as many threads side by side as there are, none beside, outputs past one turn of the block, just past the line;
# as many coefficients as a block a compute unit takes, and one more
@pytest.mark.parametrize("rows,n,k", [(1, 1, 1), (128, 10, 64), (17, 64, 5), (511, 65, 33), (64, 1000, 16), (33, 1025, 7), (1, 4097, 3), (64, 1024, 8), (65, 1024, 8),
                                      (40, 70, 1020), (40, 70, 1021)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_against_float64(rows, n, k, dtype):
    from randumb_amd import _lib, hip

    print(f"case bias gradient {rows} x {n} k={k} {dtype}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(rows + n + k)
    wide = torch.randn(rows, n + 3, generator=g).to(dtype).cuda()   # rows with a leading dimension
    dy = wide[:, :n]
    need = lib.rdb_bias_bwd_workspace_bytes(rows, n)
    ws = torch.full((need + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    dc, ds = torch.full((k + 1,), 7.0, device="cuda"), torch.full((2,), 7.0, device="cuda")
    call = lambda c, s: lib.rdb_bias_bwd(c, s, dy.data_ptr(), int(dtype == torch.bfloat16), n + 3, rows, n, k, 11, ws.data_ptr(), need, stream)
    assert call(dc.data_ptr(), ds.data_ptr()) == 0
    sums = dy.double().sum(0)
    noise, line = hip.sq5_fill_2d(n, k, 11).double(), hip.sq5_fill_1d(n, 11).double()
    # fp32 sums of rows * n terms: 2^-24 sqrt(rows * n) of their root sum of squares
    bound = 1.2e-7 * (rows * n) ** 0.5 * float(dy.double().norm()) + 1e-6
    assert float((dc[:k].double() - sums @ noise).abs().max()) < bound and abs(float(ds[0]) - float(sums @ line)) < bound
    assert float(dc[k]) == 7.0 and float(ds[1]) == 7.0 and bool((ws[need:] == 0x5A).all())
    alone = [t.clone() for t in (dc, ds)]
    assert call(alone[0].data_ptr(), 0) == 0 and call(0, alone[1].data_ptr()) == 0
    assert torch.equal(alone[0], dc) and torch.equal(alone[1], ds)


@pytest.mark.parametrize("rows,n", [(128, 10), (65, 1024)])
def test_a_workspace_is_asked_for_whichever_kernels_run(rows, n):
    from randumb_amd import _lib

    print(f"case bias gradient without its workspace {rows} x {n}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    dy, dc, need = torch.randn(rows, n, device="cuda"), torch.empty(8, device="cuda"), lib.rdb_bias_bwd_workspace_bytes(rows, n)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    call = lambda w, size: lib.rdb_bias_bwd(dc.data_ptr(), 0, dy.data_ptr(), 0, n, rows, n, 8, 11, w, size, stream)
    assert call(0, need) == -6 and call(ws.data_ptr(), need - 1) == -6 and call(ws.data_ptr(), need) == 0


def test_many_coefficients():
    """512 x 128, which one launch takes with few coefficients, beside 520 x 128, which takes two: with 16384 the one took 94 us, the two 10."""
    from randumb_amd import _lib

    print("case bias gradient of many coefficients", flush=True)
    lib, k, us = _lib.load(), 16384, []
    for rows in (512, 520):
        dy, dc = torch.randn(rows, 128, device="cuda"), torch.empty(k, device="cuda")
        need = lib.rdb_bias_bwd_workspace_bytes(rows, 128)
        ws, best = torch.empty(need, dtype=torch.uint8, device="cuda"), 1e9
        for _ in range(20):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                assert lib.rdb_bias_bwd(dc.data_ptr(), 0, dy.data_ptr(), 0, 128, rows, 128, k, 11, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream) == 0
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end) * 100.0)
        us.append(best)
    assert us[0] < us[1] + 30.0, us


# beside the last launch of a layer's backward pass: one tile and many, blocks of 256, 512 and 1024 threads, more outputs than threads, a dy too large for it
@pytest.mark.parametrize("T,in_f,out_f,k,dtype", [(128, 784, 256, 64, torch.float32), (128, 256, 10, 64, torch.float32), (1, 33, 7, 16, torch.float32), (64, 4100, 1000, 100, torch.float32),
                                                  (500, 900, 120, 31, torch.float32), (33, 65, 1025, 300, torch.float32), (600, 4000, 100, 16, torch.float32),
                                                  (300, 200, 300, 64, torch.float32), (129, 301, 77, 50, torch.bfloat16), (300, 3001, 257, 30, torch.bfloat16)])
@pytest.mark.parametrize("split", [1, 0])
def test_beside_a_layers_backward_pass(T, in_f, out_f, k, dtype, split):
    import ctypes

    from randumb_amd import _lib, hip

    print(f"case bias gradient beside {T} tokens {in_f} -> {out_f} k={k} {dtype} split={split}", flush=True)
    lib, stream, b16 = _lib.load(), torch.cuda.current_stream().cuda_stream, int(dtype == torch.bfloat16)
    before = hip.set_f32_split(split)
    try:
        g = torch.Generator().manual_seed(T + out_f)
        c, dy = torch.randn(out_f, k, generator=g).to(dtype).cuda(), torch.randn(T, out_f + 3, generator=g).to(dtype).cuda()
        d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, dtype, 0)
        ref, kept = ctypes.byref(d), torch.randn(T, k, generator=g).cuda()
        if not lib.rdb_linear_kept_bytes(ref):
            pytest.skip("nothing is kept of this layer")
        room = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_BWD_KEPT, ref)
        need = max(room, lib.rdb_bias_bwd_workspace_bytes(T, out_f))
        ws = torch.randint(0, 256, (need + 64,), dtype=torch.uint8, device="cuda")
        tail = ws[need:].clone()
        noise, line = hip.sq5_fill_2d(out_f, k, 11).double(), hip.sq5_fill_1d(out_f, 11).double()
        sums = dy[:, :out_f].double().sum(0)
        bound = 1.2e-7 * (T * out_f) ** 0.5 * float(dy.double().norm()) + 1e-6   # as above
        for want_dx, want_dc in ((1, 1), (0, 1), (1, 0), (0, 0)):
            dx, dc = torch.full((T, in_f), 7.0, device="cuda", dtype=dtype), torch.full((out_f, k), 7.0, device="cuda", dtype=dtype)
            args = (dx.data_ptr() if want_dx else None, in_f, dc.data_ptr() if want_dc else None, b16, None, dy.data_ptr(), out_f + 3, None, in_f, kept.data_ptr(), c.data_ptr(),
                    None)
            assert lib.rdb_linear_bwd_kept(*args, ref, ws.data_ptr(), need, stream) == 0
            want = dx.clone(), dc.clone()
            for grads in ((1, 1), (1, 0), (0, 1)):
                db, ds = torch.full((k + 1,), 7.0, device="cuda"), torch.full((2,), 7.0, device="cuda")
                dx.fill_(7.0), dc.fill_(7.0)
                bias = _lib.PseudoBiasGrad(db.data_ptr() if grads[0] else None, ds.data_ptr() if grads[1] else None, k, 11)
                assert lib.rdb_linear_bwd_kept_pseudo_bias(*args, ctypes.byref(bias), ref, ws.data_ptr(), need, stream) == 0
                assert torch.equal(dx, want[0]) and torch.equal(dc, want[1])
                assert float((db[:k].double() - sums @ noise).abs().max()) < bound if grads[0] else bool((db == 7.0).all())
                assert abs(float(ds[0]) - float(sums @ line)) < bound if grads[1] else float(ds[0]) == 7.0
                assert float(db[k]) == 7.0 and float(ds[1]) == 7.0 and torch.equal(ws[need:], tail)
        assert lib.rdb_linear_bwd_kept_pseudo_bias(*args, ctypes.byref(bias), ref, ws.data_ptr(), need - 1, stream) != 0
    finally:
        hip.set_f32_split(before)
