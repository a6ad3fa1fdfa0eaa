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
