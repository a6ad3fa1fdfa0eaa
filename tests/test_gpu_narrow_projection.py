"""Projection of layers whose y is too narrow for the sums of the contraction's ranges: they lie behind the state, where nothing is written
over their tags, so replays of a graph on other inputs have to find them cleared."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# k <= 256, one launch: one token, one range more than y would hold, sixteen ranges, several token tiles with a ragged last one; k > 256
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 1032, 8, 8), (97, 2048, 64, 64), (257, 8192, 1024, 32), (600, 4104, 200, 160), (640, 3400, 696, 264), (255, 1544, 72, 520)])
def test_narrow_layers(T, in_f, out_f, k):
    from randumb_amd import hip

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
