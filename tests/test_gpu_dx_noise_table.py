"""The input gradient of layers with 136 to 256 coefficients and many tokens: N written to memory beside the first launch's products."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# k padded to three and to four groups of 64; a last unit of 8 and of 40 features, a last token tile of 1 and of 6 tokens; t added up in ranges, their sums
# ahead of N in the scratch; one token range of dC stored directly; rows of dx that are whole lines (1464 + 8 and 1976 + 8 features apart), with a last unit of 56
# and a last token tile of 7 and of 8 tokens
@pytest.mark.parametrize("T,in_f,out_f,k", [(2817, 1416, 72, 136), (6000, 1000, 264, 200), (2824, 1416, 2120, 256), (16390, 264, 136, 144), (3000, 1608, 8, 256),
                                            (2823, 1464, 72, 192), (2824, 1976, 264, 256)])
def test_from_memory_is_hashed_in_place(T, in_f, out_f, k):
    from randumb_amd import _lib, hip

    print(f"case dx table T={T} in={in_f} out={out_f} k={k}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(T)
    ref = ctypes.byref(hip._proj_desc(T, in_f, out_f, k, 9))
    table = -(-in_f // 32) * 32 * -(-k // 64) * 64 * 2
    C = (torch.randn(out_f, k, device="cuda", generator=g) * k**-0.5).bfloat16()
    x, dy = (torch.randn(T, cols + 8, device="cuda", generator=g).bfloat16() for cols in (in_f, out_f))
    state = hip.linear_project(x[:, :in_f], k, out_f, 9, C)
    results = []
    for op, dtype, code in ((_lib.RDB_OP_LINEAR_BWD_PROJECTED_TO, torch.bfloat16, _lib.RDB_BF16), (_lib.RDB_OP_LINEAR_BWD_PROJECTED, torch.float32, _lib.RDB_F32)):
        n = lib.rdb_linear_workspace_bytes(op, ref)
        for room in (n, n - 1):   # the table does not fit: N is hashed where it is used
            ws = torch.full((n + 64,), 0xFF, dtype=torch.uint8, device="cuda")
            dx, dc = torch.full((T, in_f + 8), 5.0, device="cuda", dtype=torch.bfloat16), torch.empty(out_f, k, device="cuda", dtype=dtype)
            assert lib.rdb_linear_bwd_projected_to(dx.data_ptr(), in_f + 8, dc.data_ptr(), code, dy.data_ptr(), out_f + 8, state.data_ptr(), C.data_ptr(), ref,
                                                   ws.data_ptr(), room, stream) == 0
            assert bool((dx[:, in_f:] == 5.0).all()) and bool((ws[n:] == 0xFF).all())
            written = not bool((ws[n - table:n] == 0xFF).all())
            assert written == (room == n)   # each case takes the route it is meant to
            results.append((dx[:, :in_f], dc))
    for dx, dc in results[1:]:
        assert torch.equal(dx, results[0][0]) and torch.equal(dc.bfloat16(), results[0][1])
    want = dy[:, :out_f].double() @ C.double() @ hip.sq5_fill_2d(in_f, k, 9).double().t()
    assert float((results[0][0].double() - want).norm() / want.norm()) < 6e-3   # N, t and dx rounded to bf16 once each, 1.13e-3 as a norm; 2^-9 at most


# t in one to four groups of 64 coefficients, N hashed and from memory, the last tiles of tokens and features not full
@pytest.mark.parametrize("T,in_f,out_f,k", [(1, 64, 8, 8), (255, 64, 40, 64), (300, 192, 136, 72), (257, 320, 64, 128), (700, 960, 256, 136), (3300, 3072, 768, 192),
                                            (3333, 2048, 512, 256), (1000, 4096, 264, 250 // 8 * 8)])
def test_dx_through_the_gradient_of_a_squared_relu(T, in_f, out_f, k):
    """Bit for bit what the backward call and the pass over its dx give, infinities and NaNs included."""
    import ctypes

    from randumb_amd import _lib, hip

    print(f"case dx through a squared ReLU T={T} {in_f} -> {out_f} k={k}", flush=True)
    lib, stream, bf = _lib.load(), torch.cuda.current_stream().cuda_stream, torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(T + k)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(bf)
    h, c, dy = rand(T, in_f), rand(out_f, k), rand(T, out_f)
    h.view(-1)[::97], h.view(-1)[5::101], h.view(-1)[7::103], h.view(-1)[9::107] = 0.0, float("inf"), float("nan"), -float("inf")
    dy[T // 2, 0] = float("inf")
    y, state = hip.linear_project_fwd(rand(T, in_f), c, 5, None)
    d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, bf, 0)
    ref = ctypes.byref(d)
    assert lib.rdb_linear_bwd_projected_takes_relu_square(ref) == 1
    need = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_BWD_PROJECTED_TO, ref)
    ws = torch.randint(0, 256, (need + 64,), dtype=torch.uint8, device="cuda")
    tail = ws[need:].clone()
    dx, got = (torch.full((T, in_f), 7.0, dtype=bf, device="cuda") for _ in range(2))
    dc, dc2 = torch.empty_like(c), torch.empty_like(c)
    assert lib.rdb_linear_bwd_projected_to(dx.data_ptr(), in_f, dc.data_ptr(), 1, dy.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), ref, ws.data_ptr(), need, stream) == 0
    leaf = h.clone().requires_grad_()
    want, = torch.autograd.grad(_lib.extension().relu_square(leaf), leaf, dx)
    assert lib.rdb_linear_bwd_projected_relu_square(got.data_ptr(), dc2.data_ptr(), dy.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), h.data_ptr(), ref, ws.data_ptr(),
                                                    need, stream) == 0
    same = lambda a, b: torch.equal(torch.nan_to_num(a, nan=1234.0), torch.nan_to_num(b, nan=1234.0))
    assert same(got, want) and same(dc2, dc) and torch.equal(ws[need:], tail)
    assert lib.rdb_linear_bwd_projected_relu_square(got.data_ptr() + 16, dc2.data_ptr(), dy.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), h.data_ptr(), ref, ws.data_ptr(),
                                                    need, stream) != 0


@pytest.mark.parametrize("T,in_f,out_f,k", [(64, 72, 64, 64), (512, 128, 64, 264)])
def test_layers_whose_dx_has_no_such_store(T, in_f, out_f, k):
    import ctypes

    from randumb_amd import _lib, hip

    c = torch.zeros(out_f, k, dtype=torch.bfloat16, device="cuda")
    d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0)
    assert _lib.load().rdb_linear_bwd_projected_takes_relu_square(ctypes.byref(d)) == 0
