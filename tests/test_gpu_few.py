"""Forward pass for few tokens (rdb_few.hip) against float64: sizes around its tiles (16 tokens, 16 coefficients, chunks of 128
and more input features, 64 output features), odd ones, any alignment, infinities; one launch against two; replays; a wait that gives up."""
import ctypes

import pytest
import torch

from randumb_amd import _lib, hip, ops

pytestmark = pytest.mark.gpu

# fp32: sums of up to some thousand products, each rounded at 2^-24 of a running sum; bf16: the same, then rounded once (8 bits: 2^-8 of a value at most)
TOL = {torch.float32: 2e-6, torch.bfloat16: 2.0**-8}


def _case(T, in_f, out_f, k, dtype, seed=5):
    g = torch.Generator().manual_seed(T * 1000 + k)
    x, c, b = torch.randn(T, in_f, generator=g), torch.randn(out_f, k, generator=g) / k ** 0.5, torch.randn(out_f, generator=g)
    return [t.to(dtype).cuda() for t in (x, c, b)] + [ops.sq5_gen_2d(in_f, k, seed).double()]


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 1, 1, 1), (2, 7, 3, 5), (15, 127, 63, 15), (16, 128, 64, 16), (17, 129, 65, 17), (1, 4104, 2049, 16), (32, 513, 257, 128),
                                            (31, 2056, 2120, 100), (16, 1000, 4100, 129), (13, 4096, 1000, 256), (1, 1030, 70, 257), (32, 1040, 2200, 512),
                                            (33, 300, 100, 33), (48, 264, 2112, 64), (48, 4100, 300, 250), (47, 1200, 520, 510),
                                            # one tile of tokens and two to an expanding block, the last group not full
                                            (49, 130, 65, 17), (97, 264, 5100, 40), (96, 260, 2800, 256), (81, 515, 130, 129), (90, 700, 2850, 300),
                                            (192, 2050, 1000, 131), (256, 1001, 999, 100), (240, 600, 3000, 16), (255, 264, 352, 64), (512, 512, 600, 64),
                                            (500, 1030, 200, 30), (509, 2000, 2200, 50)])
def test_against_float64(T, in_f, out_f, k, dtype):
    print(f"case few T={T} in={in_f} out={out_f} k={k} {dtype}", flush=True)
    x, c, b, N = _case(T, in_f, out_f, k, dtype)
    want = (x.double() @ N) @ c.double().t()
    y = hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5, bias=b)
    assert _rel(y, want + b.double()) < TOL[dtype]
    before = hip.set_one_launch(0)
    try:
        assert torch.equal(y, hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5, bias=b))   # the same sums in the same order
    finally:
        hip.set_one_launch(before)
    # rows that begin anywhere, NaNs around them, y in a wider matrix
    wide = torch.full((T, in_f + 3), float("nan"), device="cuda", dtype=dtype)
    wide[:, 1:1 + in_f] = x
    assert torch.equal(y, hip.linear_fwd(wide[:, 1:1 + in_f], c, in_f, out_f, in_f, 1, 5, bias=b))
    d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, dtype, 0)
    need = _lib.load().rdb_linear_workspace_bytes(0, ctypes.byref(d))
    ws, out = torch.randint(0, 256, (need,), dtype=torch.uint8, device="cuda"), torch.full((T, out_f + 5), 7.0, device="cuda", dtype=dtype)
    assert _lib.load().rdb_linear_fwd(out.data_ptr(), out_f + 5, x.data_ptr(), in_f, c.data_ptr(), None, b.data_ptr(), ctypes.byref(d), ws.data_ptr(), need,
                                      torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[:, :out_f], y) and bool((out[:, out_f:] == 7.0).all())


# four waves of a block and eight, in one launch: 8 tokens and 9, chunks of 256 and 512, k below 128 and above, odd and a multiple of 8; as many blocks as compute units and one more
@pytest.mark.parametrize("T,in_f,out_f,k", [(8, 1030, 130, 129), (8, 1030, 130, 136), (9, 1030, 130, 129), (8, 2048, 64, 255), (8, 2049, 64, 255), (8, 1030, 130, 127), (1, 8000, 64, 255), (1, 7680, 1024, 254), (1, 7680, 1025, 254), (200, 8192, 64, 32), (200, 8192, 64, 48),
                                            (2, 300, 10304, 100), (16, 200, 10304, 30), (51, 327, 2944, 32), (100, 200, 1500, 20), (100, 120, 1500, 20)])   # more than 160 expanding blocks
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_waves_of_a_block(T, in_f, out_f, k, dtype):
    test_against_float64(T, in_f, out_f, k, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [1, 2, 40])
def test_not_finite(k, dtype):
    """Infinities and NaNs come out where and as 64-bit arithmetic has them, and nowhere else; very large values stay finite."""
    T, in_f, out_f = 6, 200, 70
    x, c, _, N = _case(T, in_f, out_f, k, dtype)
    inf = float("inf")
    x[1, 3], x[2, 150], x[3, 7] = inf, -inf, float("nan")
    x[4] = 0.0
    x[4, 60] = 1.0e37
    c[5, 0], c[6, k - 1] = inf, -inf
    want = (x.double() @ N) @ c.double().t()
    y = hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5).double()
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.isinf(y), torch.isinf(want)) and torch.equal(y[torch.isinf(y)], want[torch.isinf(want)])
    # against the sum of the terms' sizes: fp32 roundings along the way, and 2^-21 where a sum beside one that is not finite is done again
    size = (x.double().abs() @ N.abs()) @ c.double().abs().t()
    bound = 2.0**-19 * size + (0.0 if dtype == torch.float32 else 2.0**-8) * want.abs()
    ok = torch.isfinite(want)
    assert bool(((y - want).abs() <= bound)[ok].all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,in_f,out_f,k", [(5, 96, 70, 2), (16, 512, 64, 16), (40, 300, 130, 33), (33, 2048, 5000, 64)])
def test_a_value_that_is_not_finite_leaves_its_neighbours_alone(T, in_f, out_f, k, dtype):
    """Other tokens of the call and other output features: bit for bit what they are without it."""
    x, c, b, _ = _case(T, in_f, out_f, k, dtype)
    call = lambda x, c: hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5, bias=b)
    want = call(x, c)
    t, o = T - 2, out_f - 3
    for bad in (float("inf"), float("nan"), 3.0e38):
        spoiled = x.clone()
        spoiled[t, in_f // 2] = bad
        got = call(spoiled, c)
        assert torch.equal(got[torch.arange(T) != t], want[torch.arange(T) != t])
        spoiled = c.clone()
        spoiled[o, k - 1] = bad
        got = call(x, spoiled)
        assert torch.equal(got[:, torch.arange(out_f) != o], want[:, torch.arange(out_f) != o])


@pytest.mark.parametrize("T,in_f,out_f,k", [(20, 1000, 520, 100), (200, 512, 512, 128), (3, 4096, 300, 16), (500, 700, 333, 40)])
def test_fp32_products_where_they_are_asked_for(T, in_f, out_f, k):
    """rdb_set_f32_split(0): a forward of few tokens in fp32 leaves the split products too, for the kernels that FACTORED names."""
    x, c, b, N = _case(T, in_f, out_f, k, torch.float32)
    call = lambda algo: hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5, bias=b, algo=algo)
    split = call(_lib.RDB_ALGO_AUTO)
    before = hip.set_f32_split(0)
    try:
        plain = call(_lib.RDB_ALGO_AUTO)
        assert torch.equal(plain, call(_lib.RDB_ALGO_FACTORED)) or k <= 64   # k <= 64: AUTO chooses between two kernels, FACTORED does not
    finally:
        hip.set_f32_split(before)
    assert not torch.equal(plain, split) and _rel(plain, (x.double() @ N) @ c.double().t() + b.double()) < 1e-5
    assert torch.equal(call(_lib.RDB_ALGO_AUTO), split)


@pytest.mark.parametrize("T,in_f,out_f,k", [(97, 2048, 512, 64), (128, 4096, 1024, 256), (300, 1024, 2048, 128), (500, 8192, 512, 16), (16, 1024, 1024, 384)])
def test_evaluation_and_training_in_bf16(T, in_f, out_f, k):
    """A forward that keeps z for a backward pass keeps it in bf16 and multiplies what it keeps; one that keeps nothing goes on with z in
    fp32.  So y differs: by z's rounding and its own, each 2^-9 of a value at most either way (1.7e-3 of a result in the 2-norm), and
    evaluation is the nearer one to 64 bits."""
    from randumb_amd import SillyLinear

    x, c, _, N = _case(T, in_f, out_f, k, torch.bfloat16)
    layer = SillyLinear(in_f, out_f, [k, k], [5, 6], bias=False, device="cuda", dtype=torch.bfloat16, matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.copy_(c)
        evaluated = layer(x)
    trained = layer(x.requires_grad_())
    assert "Projected" in repr(trained.grad_fn)
    want = (x.detach().double() @ N) @ c.double().t()
    e, t = _rel(evaluated, want), _rel(trained.detach(), want)
    assert e < t < 4e-3 and e < 2e-3 and _rel(evaluated, trained.detach().double()) < 4e-3


def test_recorded_launches():
    """Both forms recorded into one graph and replayed on changing inputs, with eager calls in between."""
    shapes = [(5, 1001, 999, 99), (100, 264, 352, 64), (16, 4096, 4096, 256), (40, 8192, 512, 512)]   # one launch (one group of tokens, four), two, three
    cases = [_case(*s, torch.bfloat16)[:2] for s in shapes]
    call = lambda: [hip.linear_fwd(x, c, s[1], s[2], s[1], 1, 5) for s, (x, c) in zip(shapes, cases)]
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for i in range(4):
        for x, _ in cases:
            x.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(i)))
        graph.replay()
        got = [o.clone() for o in out]
        assert all(torch.equal(a, b) for a, b in zip(got, call())), i
        torch.cuda.synchronize()


# 20 and 64 tokens: these kernels, one group of tokens and several; 520: the vector-ALU kernels of rdb_smallk.hip, whose wait is their own
@pytest.mark.parametrize("T", [20, 64, 520])
def test_a_wait_that_gives_up(T):
    """NaN throughout, the counter, and the host's watch, as for the other one-launch forms."""
    in_f, out_f, k = 1000, 520, 16
    x, c, _, _ = _case(T, in_f, out_f, k, torch.float32)
    want = hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5)
    d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.float32, 0)
    ws = torch.zeros(int(_lib.load().rdb_linear_workspace_bytes(0, ctypes.byref(d))), dtype=torch.uint8, device="cuda")
    y = torch.zeros(T, out_f, device="cuda")
    hip.selftest_sync_giveup(y, ws, c, in_f, 5, polls=32)
    torch.cuda.synchronize()
    assert bool(torch.isnan(y).all())
    with pytest.raises(_lib.RandumbHipError, match="gave up"):
        hip.sync_check()
    hip.set_one_launch(1)
    assert torch.equal(hip.linear_fwd(x, c, in_f, out_f, in_f, 1, 5), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,in_f,out_f,k", [(3, 3990, 12300, 40), (20, 4095, 11000, 250), (1, 2047, 11010, 63), (8, 2049, 12287, 64), (9, 2048, 12290, 64), (64, 3000, 9000, 200),
                                            (7, 1025, 4000, 300), (5, 500, 4000, 70), (2, 33, 20000, 9)])
def test_chunks_in_eight_and_sixteen_waves(T, in_f, out_f, k, dtype):
    """Four, eight or sixteen waves to a chunk, the last chunk's not all with something to add; both sides of the line to one launch."""
    test_against_float64(T, in_f, out_f, k, dtype)
