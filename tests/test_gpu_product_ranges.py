"""Dense fp32 products with and without a bias, in one range of the contraction and in several: the sums, the bias's columns, nothing beside the output."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles of 64 x 128 with remainders of one, rows that are not 16-byte aligned, an output of one value, contractions just short and just past a range
@pytest.mark.parametrize("M,N,K", [(216, 198, 966), (64, 128, 127), (65, 129, 260), (1, 1, 4096), (130, 3, 701), (3, 1030, 513)])
@pytest.mark.parametrize("across", [(0, 0), (0, 1), (1, 1)])
def test_product(M, N, K, across):
    from randumb_amd import _lib

    print(f"case product {M} x {N} x {K} across={across}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(M + N + K)
    a, b, bias = (torch.randn(*s, generator=g).cuda() for s in ((K, M) if across[0] else (M, K), (K, N) if across[1] else (N, K), (N,)))
    need = lib.rdb_product_f32_workspace_bytes(M, N, K)
    ws = torch.full((need + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    want = (a.double().t() if across[0] else a.double()) @ (b.double() if across[1] else b.double().t())
    for add in (None, bias):
        ref = want if add is None else want + add.double()
        # fp32 sums of K terms in some order: 2^-24 sqrt(K) as a norm at most, and the last rounding
        bound = 6e-8 * (K**0.5 + 1.0) * float(want.norm())
        for size in (need, 0):
            out = torch.full((M * N + 4,), 7.0, device="cuda")
            call = lambda: lib.rdb_product_f32(out.data_ptr(), a.data_ptr(), a.stride(0), across[0], b.data_ptr(), b.stride(0), across[1],
                                               0 if add is None else add.data_ptr(), M, N, K, ws.data_ptr() if size else 0, size, stream)
            assert call() == 0
            first = out.clone()
            assert call() == 0 and torch.equal(out, first)
            assert bool((out[M * N:] == 7.0).all()) and float((out[: M * N].view(M, N).double() - ref).norm()) < bound
    assert bool((ws[need:] == 0x5A).all())
