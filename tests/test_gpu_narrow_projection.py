"""Projection of layers whose y is too narrow for the sums of the contraction's ranges: they lie in scratch of the call's own, where nothing need be
written over their tags, so replays of a graph on other inputs have to find them cleared."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# k <= 256, one launch: one token (of the fewest stages that are cut into ranges: 1352 features are 22 of them), one range more than y would hold, sixteen
# ranges, several token tiles with a ragged last one; k > 256
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 1352, 8, 8), (97, 2048, 64, 64), (257, 8192, 1024, 32), (600, 4104, 200, 160), (640, 3400, 696, 264), (255, 1544, 72, 520)])
def test_narrow_layers(T, in_f, out_f, k):
    import ctypes

    from randumb_amd import _lib, hip

    print(f"case narrow projection T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator().manual_seed(T)
    xs = [torch.randn(T, in_f, generator=g).bfloat16().cuda() for _ in range(3)]
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).bfloat16().cuda()
    N = hip.sq5_fill_2d(in_f, k, 5).double()
    want = []
    for x in xs:
        y, state = hip.linear_project_fwd(x, c, 5)
        ref = x.double() @ N @ c.double().t()
        assert float((y.double() - ref).norm() / ref.norm()) < 8e-3   # z and y rounded to bf16: 2^-9 each at most, fewer values than a norm needs
        assert torch.equal(hip.linear_fwd_projected(hip.linear_project(x, k, out_f, 5), c, in_f, 5), y)   # the projection alone
        old = hip.set_one_launch(0)   # every block adds its tile's ranges up itself
        try:
            assert torch.equal(hip.linear_project_fwd(x, c, 5)[0], y)
        finally:
            hip.set_one_launch(old)
        want.append(y)
    # a transient state without the room: y by the one-call form, from scratch of the caller's and, what fits there, the library's
    lib, stream, y = _lib.load(), torch.cuda.current_stream().cuda_stream, torch.empty_like(want[0])
    ref = ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, _lib.RDB_ALGO_FACTORED))
    n = lib.rdb_linear_workspace_bytes(0, ref)
    less = n - (T * 8 + 255) // 256 * 256
    ws = torch.full((n,), 0x5A, dtype=torch.uint8, device="cuda")
    for size in (n, less):
        assert lib.rdb_linear_fwd(y.data_ptr(), out_f, xs[0].data_ptr(), in_f, c.data_ptr(), None, None, ref, ws.data_ptr(), size, stream) == 0
        assert torch.equal(y, want[0])
    assert lib.rdb_linear_fwd_static(y.data_ptr(), out_f, xs[0].data_ptr(), in_f, c.data_ptr(), None, None, ref, stream) == 0
    assert torch.equal(y, want[0])
    x = xs[0].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, state = hip.linear_project_fwd(x, c, 5)
        alone = hip.linear_project(x, k, out_f, 5)
    for i in (1, 2, 0, 0, 2):
        x.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[i]), i
        assert torch.equal(hip.linear_fwd_projected(alone, c, in_f, 5), want[i]), i
        assert torch.equal(hip.linear_project_fwd(xs[i], c, 5)[0], want[i])
    hip.sync_check()


# fp32 sums: odd sizes in bf16, and fp32; one token more than a tile, several ranges, y of one column
@pytest.mark.parametrize("T,in_f,out_f,k,dtype", [(492, 3184, 273, 118, torch.bfloat16), (129, 1027, 1, 20, torch.bfloat16), (433, 3320, 96, 144, torch.float32),
                                                  (65, 4000, 33, 257, torch.float32)])
@pytest.mark.parametrize("split", [1, 0])
def test_narrow_layers_in_fp32_sums(T, in_f, out_f, k, dtype, split):
    import ctypes

    from randumb_amd import _lib, hip

    print(f"case narrow kept T={T} in={in_f} out={out_f} k={k} {dtype} split={split}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    x, c = torch.randn(T, in_f, generator=g).to(dtype).cuda(), (torch.randn(out_f, k, generator=g) / k ** 0.5).to(dtype).cuda()
    ref = ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, dtype, 0))
    N = hip.sq5_fill_2d(in_f, k, 5).double()
    z = x.double() @ N
    want = z @ c.double().t()
    calls = [("kept", lib.rdb_linear_kept_bytes(ref), 0, _lib.RDB_OP_LINEAR_FWD_KEPT)]
    if dtype is torch.float32:
        calls.append(("state", lib.rdb_linear_projection_bytes(ref), 256, _lib.RDB_OP_LINEAR_PROJECT))
    rooms = [lib.rdb_linear_workspace_bytes(op, ref) for _, n, _, op in calls if n]
    assert min(rooms) >= 3 * T * k * 4   # room for ranges
    for what, n, at, op in calls:
        if n == 0:
            continue
        room = lib.rdb_linear_workspace_bytes(op, ref)
        kept, ws = (torch.full((m + 64,), 0x5A, dtype=torch.uint8, device="cuda") for m in (n, room))
        y = torch.full((T + 1, out_f), 7.0, dtype=dtype, device="cuda")
        before = lib.rdb_set_f32_split(split)   # asked for after the buffer's size
        try:
            if what == "kept":
                rc = lib.rdb_linear_fwd_kept_ws(y.data_ptr(), out_f, kept.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), None, None, None, ref, ws.data_ptr(), room, stream)
            else:
                rc = lib.rdb_linear_project_fwd_ws(y.data_ptr(), out_f, kept.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), None, ref, ws.data_ptr(), room, stream)
        finally:
            lib.rdb_set_f32_split(before)
        assert rc == 0 and bool((kept[n:] == 0x5A).all()) and bool((ws[room:] == 0x5A).all()) and bool((y[T] == 7.0).all())
        got = kept[at:at + T * k * 4].view(torch.float32).view(T, k).double()
        assert float((got - z).norm() / z.norm()) < 2e-6   # fp32 sums of products of fp32 accuracy
        # y rounded once: to bf16 2^-9 at most
        assert float((y[:T].double() - want).norm() / want.norm()) < (2.0 ** -9 if dtype is torch.bfloat16 else 4e-6)
    hip.sync_check()
