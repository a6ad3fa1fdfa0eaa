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
