"""A pseudorandom bias formed in a launch that its layer makes anyway: the values of a launch of their own, whatever the sizes."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


class _PseudoBias(ctypes.Structure):
    _fields_ = [("coef", ctypes.c_void_p), ("scale", ctypes.c_void_p), ("values", ctypes.c_void_p), ("k", ctypes.c_int64), ("seed", ctypes.c_uint32)]


def _values(hip, coef, scale, n, seed):
    return hip.materialize_fwd(coef, (n,), (1,), seed, scale, scale is not None)


# few and many elements (another number of lanes each), terms by eights and not, long weights (two launches)
@pytest.mark.parametrize("n,k,bn,bk", [(1, 1, 1, 8), (70, 9, 3, 16), (40000, 48, 257, 64), (140000, 49, 1000, 100), (600000, 300, 65, 17), (5000, 20, 33000, 9), (300, 5, 40, 3)])
@pytest.mark.parametrize("scaled", [False, True])
def test_weight_and_bias(n, k, bn, bk, scaled):
    from randumb_amd import _lib, hip

    print(f"case weight and bias n={n} k={k} bias n={bn} k={bk} scaled={scaled}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(n + bn)
    c, bc, s = (torch.randn(m, generator=g).cuda() for m in (k, bk, 1))
    w, b = torch.full((n + 4,), 7.0, device="cuda"), torch.full((bn + 4,), 7.0, device="cuda")
    ref = _PseudoBias(bc.data_ptr(), s.data_ptr() if scaled else None, b.data_ptr(), bk, 22)
    assert lib.rdb_materialize_weight_and_bias(w.data_ptr(), n, c.data_ptr(), k, 21, s.data_ptr() if scaled else None, ctypes.byref(ref), bn, stream) == 0
    sc = s if scaled else None
    assert torch.equal(w[:n], _values(hip, c, sc, n, 21)) and torch.equal(b[:bn], _values(hip, bc, sc, bn, 22))
    assert bool((w[n:] == 7.0).all()) and bool((b[bn:] == 7.0).all())


# one tile and many, one slice of the grid and many, more elements than a slice has groups of lanes, ranges of the contraction beside them; the longest sums
# and the most elements that are formed beside the projection, and one more of each
@pytest.mark.parametrize("T,in_f,out_f,k,bk", [(64, 784, 256, 64, 64), (33, 301, 1, 64, 8), (128, 256, 10, 64, 64), (32, 512, 4099, 96, 130), (64, 4096, 4099, 64, 17),
                                               (700, 264, 301, 40, 33), (64, 784, 1000, 64, 1024), (64, 784, 77, 64, 1025), (64, 784, 32768, 64, 9), (64, 784, 32769, 64, 9)])
@pytest.mark.parametrize("scaled", [False, True])
@pytest.mark.parametrize("split", [1, 0])
def test_layer(T, in_f, out_f, k, bk, scaled, split):
    from randumb_amd import _lib, hip

    print(f"case layer with a pseudorandom bias T={T} {in_f}->{out_f} k={k} bias k={bk} scaled={scaled} split={split}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T + out_f)
    x, c, bc, s = (torch.randn(*m, generator=g).cuda() for m in ((T, in_f), (out_f, k), (bk,), (1,)))
    ref = ctypes.byref(hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.float32, 0))
    size = lib.rdb_linear_kept_bytes(ref)
    assert size > 0
    before = lib.rdb_set_f32_split(split)
    try:
        sc, values = s if scaled else None, torch.full((out_f + 4,), 7.0, device="cuda")
        want_b = _values(hip, bc, sc, out_f, 9)
        y, want = (torch.empty(T, out_f, device="cuda") for _ in range(2))
        kept, want_kept = (torch.zeros(size, dtype=torch.uint8, device="cuda") for _ in range(2))
        pb = _PseudoBias(bc.data_ptr(), s.data_ptr() if scaled else None, values.data_ptr(), bk, 9)
        assert lib.rdb_linear_fwd_kept_pseudo_bias(y.data_ptr(), out_f, kept.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), None, ctypes.byref(pb), ref, stream) == 0
        assert lib.rdb_linear_fwd_kept(want.data_ptr(), out_f, want_kept.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), None, want_b.data_ptr(), ref, stream) == 0
        assert torch.equal(values[:out_f], want_b) and bool((values[out_f:] == 7.0).all())
        assert torch.equal(y, want) and torch.equal(kept, want_kept)
    finally:
        lib.rdb_set_f32_split(before)


def test_many_values_beside_few_tiles():
    """A projection of a single tile of rows beside 32768 values: one block a tile formed them all in 500 us, where the layer without a bias takes 16."""
    from randumb_amd import SillyLinear

    print("case a long bias beside few tiles", flush=True)
    x, us = torch.randn(64, 784, device="cuda").requires_grad_(), []
    for bias in (True, False):
        layer = SillyLinear(784, 32768, [64, 64], [1, 2], bias=bias, device="cuda", matrix_coef=True)
        best = 1e9
        for _ in range(20):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                layer(x)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end) * 100.0)
        us.append(best)
    assert us[0] < us[1] + 100.0, us
