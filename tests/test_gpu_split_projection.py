"""The projection's contraction spread over blocks of their own (few tiles, long in_f): the same bits as the unspread launches, in
every piece of the state, and the right values; replayed from a graph too."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1024, 1024, 64), (97, 1032, 2048, 64), (257, 2048, 1024, 96), (300, 4096, 4096, 256), (2000, 4096, 512, 32), (200, 3000, 4096, 320), (512, 8192, 328, 40)]


@pytest.fixture(scope="module")
def hip():
    from randumb_amd import hip

    return hip


def _inputs(T, in_f, out_f, k):
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, in_f, generator=g, device="cuda").bfloat16()
    C = (torch.randn(out_f, k, generator=g, device="cuda") * 0.05).bfloat16()
    return x, C


@pytest.mark.parametrize("T,in_f,out_f,k", SHAPES)
def test_spread_projection_is_the_unspread_one(hip, T, in_f, out_f, k):
    print(f"case spread projection T={T} in={in_f} out={out_f} k={k}", flush=True)
    x, C = _inputs(T, in_f, out_f, k)
    y, state = hip.linear_project_fwd(x, C, 5)
    apart = hip.linear_project(x, k, out_f, 5, C)
    pieces, want = hip.projection_unpack(state, in_f, out_f, k), hip.projection_unpack(apart, in_f, out_f, k)
    for name in ("z", "z_t", "coef_t"):
        assert torch.equal(pieces[name], want[name]), name
    assert torch.equal(y, hip.linear_fwd_projected(apart, C, in_f, 5))
    before = hip.set_one_launch(0)
    try:
        y2, _ = hip.linear_project_fwd(x, C, 5)
    finally:
        hip.set_one_launch(before)
    assert torch.equal(y, y2)
    z = x.double() @ hip.sq5_fill_2d(in_f, k, 5).double()
    assert float((pieces["z"].double() - z).norm() / z.norm()) < 3e-3
    ref = z @ C.double().t()
    assert float((y.double() - ref).norm() / ref.norm()) < 5e-3
    hip.sync_check()


def test_spread_projection_replayed_from_a_graph(hip):
    x, C = _inputs(300, 4096, 1024, 96)
    xs = [torch.randn_like(x) for _ in range(3)]
    want = [hip.linear_project_fwd(v, C, 7)[0].clone() for v in xs]
    static = xs[0].clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        hip.linear_project_fwd(static, C, 7)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y, _state = hip.linear_project_fwd(static, C, 7)
    for i in (0, 1, 2, 0, 2):
        static.copy_(xs[i])
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[i]), i
        assert torch.equal(hip.linear_project_fwd(xs[i], C, 7)[0], want[i])
    hip.sync_check()


@pytest.mark.parametrize("T,in_f,out_f,k", [(300, 264, 2056, 72), (1178, 136, 6520, 160), (70, 64, 8200, 248), (129, 72, 3080, 256)])
@pytest.mark.parametrize("with_ct", [True, False])
def test_split_dy_product(T, in_f, out_f, k, with_ct):
    """t = dy . C in ranges of the output features (few tiles, long rows of dy): against float64, and the same bits
    twice, with a workspace that has no room for the ranges' sums, and from the input gradient's own entry point."""
    import ctypes

    from randumb_amd import _lib, hip, ops

    lib = _lib.load()
    g = torch.Generator().manual_seed(T)
    x, dy = torch.randn(T, in_f, generator=g).bfloat16().cuda(), torch.randn(T, out_f, generator=g).bfloat16().cuda()
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).bfloat16().cuda()
    ref = ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0))
    state = hip.linear_project(x, k, out_f, 5, coef=c if with_ct else None)
    full, part = lib.rdb_linear_workspace_bytes(4, ref), T * k * 4
    out = []
    for size in (full, full, full - 2 * part):
        dx, dc, ws = torch.empty_like(x), torch.empty_like(c), torch.empty(size, dtype=torch.uint8, device="cuda")
        assert lib.rdb_linear_bwd_projected_to(dx.data_ptr(), in_f, dc.data_ptr(), 1, dy.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), ref,
                                               ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream) == 0
        out.append((dx, dc))
    for dx, dc in out[1:]:
        assert torch.equal(dx, out[0][0]) and torch.equal(dc, out[0][1])
    assert torch.equal(hip.linear_bwd_dx(dy, c, in_f, out_f, in_f, 1, 5, algo=_lib.RDB_ALGO_FACTORED), out[0][0])
    N = ops.sq5_gen_2d(in_f, k, 5).double().cpu()
    want = (dy.double().cpu() @ c.double().cpu()) @ N.t()
    assert float((out[0][0].double().cpu() - want).norm() / want.norm()) < 8e-3
    assert float((out[0][1].double().cpu() - dy.double().cpu().t() @ (x.double().cpu() @ N)).norm() / (dy.double().cpu().t() @ (x.double().cpu() @ N)).norm()) < 8e-3


@pytest.mark.parametrize("T,in_f,out_f,k", [(40, 64, 8, 8), (300, 264, 2056, 72), (1178, 136, 6520, 160), (65, 3080, 40, 256), (300, 1032, 2008, 328)])
@pytest.mark.parametrize("one_launch", [True, False])
def test_transposed_coefficients_from_blocks_of_their_own(T, in_f, out_f, k, one_launch):
    """Few projecting blocks: C is transposed beside them.  The input gradient from the state's transposed coefficients and from C itself:
    the same bits, from the call that forms y too and from the projection alone."""
    from randumb_amd import hip

    g = torch.Generator().manual_seed(T)
    x, dy = torch.randn(T, in_f, generator=g).bfloat16().cuda(), torch.randn(T, out_f, generator=g).bfloat16().cuda()
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).bfloat16().cuda()
    plain = hip.linear_project(x, k, out_f, 5)
    old = hip.set_one_launch(1 if one_launch else 0)
    try:
        y, state = hip.linear_project_fwd(x, c, 5)
        alone = hip.linear_project(x, k, out_f, 5, coef=c)
        results = [hip.linear_bwd_projected(dy, s, c, in_f, 5) for s in (state, alone, plain)]
        hip.sync_check()
    finally:
        hip.set_one_launch(old)
    assert [int(s.view(-1)[:4].view(torch.int32)[0]) for s in (state, alone, plain)] == [1, 1, 0]
    assert torch.equal(y, hip.linear_fwd_projected(plain, c, in_f, 5))
    for dx, dc in results[:2]:
        assert torch.equal(dx, results[2][0]) and torch.equal(dc, results[2][1])


@pytest.mark.parametrize("T,in_f,out_f,k", [(300, 4096, 4096, 64), (97, 8192, 2048, 64), (512, 8192, 1024, 32), (2000, 4096, 4096, 256)])
def test_sums_on_the_way_do_not_stay_in_the_rows_of_a_block_that_gave_up(hip, T, in_f, out_f, k):
    """Multiplying blocks that look once and give up leave NaN; projecting blocks that are still at work then put their sums into
    the same rows, and have to take them back.  Every value of y is its own or NaN, in whole blocks of tokens."""
    from randumb_amd import _lib

    print(f"case hasty wait T={T} in={in_f} out={out_f} k={k}", flush=True)
    x, C = _inputs(T, in_f, out_f, k)
    hip.sync_check()
    want, _ = hip.linear_project_fwd(x, C, 5)
    seen = 0
    try:
        for _ in range(3):
            y = hip.selftest_hasty_wait(x, C, 5, polls=1)
            poisoned = y.isnan()
            seen += int(poisoned.any())
            assert torch.equal(y[~poisoned], want[~poisoned])
        assert seen, "no block gave up"
        with pytest.raises(_lib.RandumbHipError, match="gave up"):
            hip.sync_check()
    finally:
        hip.set_one_launch(1)
    assert torch.equal(hip.linear_project_fwd(x, C, 5)[0], want)
    hip.sync_check()
