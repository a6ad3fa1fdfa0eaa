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
