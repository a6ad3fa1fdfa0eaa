"""Vector-coef materialise, its adjoint and the embedding against fp64 sums of the noise matrix:
sizes around the tiles' edges, views, magnitudes from denormal to huge, infinities and NaNs."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from randumb_amd import hip

    return hip


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-300))


@pytest.mark.parametrize("n,k,scale", [(1, 1, 1.0), (15, 3, 1e-3), (33, 16, 1e20), (127, 17, 1.0), (129, 64, 1e-30), (700, 65, 1.0), (1000, 256, 1e-3), (257, 1023, 1.0),
                                       (300, 1025, 1e-42), (70, 3000, 1.0), (70001, 40, 1.0)])
def test_sums_of_hashed_values(hip, n, k, scale):
    print(f"case hash sums n={n} k={k} scale={scale}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    noise = hip.sq5_fill_2d(n, k, 11).double()
    c = torch.randn(k, generator=g, device="cuda") * scale
    d = torch.randn(n, generator=g, device="cuda") * scale
    tol = 2e-6 if scale > 1e-38 else 0.2   # denormals have few bits themselves
    assert rel(hip.materialize_fwd(c, (n,), (1,), 11, None, False), noise @ c.double()) < tol
    got = hip.materialize_bwd(d, k, 11)
    assert rel(got, d.double() @ noise) < tol
    assert torch.equal(got, hip.materialize_bwd(d, k, 11))
    if scale == 1.0:
        sb = torch.tensor([0.7], device="cuda")
        want = (noise @ c.double()) + sb.double() * hip.sq5_fill_1d(n, 11).double()
        assert rel(hip.materialize_fwd(c, (n,), (1,), 11, sb, True), want) < tol
        cb, db = c.bfloat16(), d.bfloat16()
        assert rel(hip.materialize_fwd(cb, (n,), (1,), 11, None, False), noise @ cb.double()) < tol
        assert rel(hip.materialize_bwd(db, k, 11), db.double() @ noise) < 2e-6


def test_magnitudes_of_different_size_and_views(hip):
    g = torch.Generator(device="cuda").manual_seed(0)
    c = torch.randn(300, generator=g, device="cuda") * torch.exp(torch.randn(300, generator=g, device="cuda") * 4)
    noise = hip.sq5_fill_2d(60 * 70, 300, 3).double()
    want = (noise @ c.double()).view(60, 70)
    assert rel(hip.materialize_fwd(c, (60, 70), (70, 1), 3, None, False), want) < 2e-6
    assert torch.equal(hip.materialize_fwd(c, (70, 60), (1, 70), 3, None, False), hip.materialize_fwd(c, (60, 70), (70, 1), 3, None, False).t())
    assert torch.equal(hip.materialize_fwd(c, (20, 70), (140, 1), 3, None, False), hip.materialize_fwd(c, (60, 70), (70, 1), 3, None, False)[:40:2])
    d = torch.randn(4200, generator=g, device="cuda") * torch.exp(torch.randn(4200, generator=g, device="cuda") * 4)
    assert rel(hip.materialize_bwd(d, 300, 3), d.double() @ noise) < 2e-6
    one = torch.zeros(300, device="cuda")
    one[123] = 1.0
    assert torch.equal(hip.materialize_fwd(one, (4200,), (1,), 3, None, False), hip.sq5_fill_2d(4200, 300, 3)[:, 123])   # exact
    assert not bool(hip.materialize_fwd(torch.zeros(300, device="cuda"), (4200,), (1,), 3, None, False).any())
    assert not bool(hip.materialize_bwd(torch.zeros(4200, device="cuda"), 300, 3).any())


@pytest.mark.parametrize("bad", [math.inf, -math.inf, math.nan])
def test_infinities_and_nans_come_out(hip, bad):
    c = torch.ones(40, device="cuda")
    c[7] = bad
    noise = hip.sq5_fill_2d(500, 40, 3)
    got, want = hip.materialize_fwd(c, (500,), (1,), 3, None, False), (noise * c).sum(1)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    d = torch.ones(500, device="cuda")
    d[300] = bad
    got, want = hip.materialize_bwd(d, 40, 3), (noise * d[:, None]).sum(0)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())


@pytest.mark.parametrize("n,dim,k", [(1, 8, 5), (9, 100, 64), (65, 33, 200), (500, 64, 300)])
def test_embedding(hip, n, dim, k):
    g = torch.Generator(device="cuda").manual_seed(n)
    idx = torch.randint(0, 50304, (n,), generator=g, device="cuda")
    c = torch.randn(k, generator=g, device="cuda")
    d = torch.randn(n, dim, generator=g, device="cuda")
    table = torch.stack([_noise_rows(hip, int(i), dim, k, 9) for i in idx]).double()   # (n, dim, k)
    assert rel(hip.embed_fwd(idx, c, dim, 9), table @ c.double()) < 2e-6
    assert rel(hip.embed_bwd(idx, d, k, dim, 9), (d.double().unsqueeze(-1) * table).sum((0, 1))) < 2e-6


def _noise_rows(hip, row, dim, k, seed):
    PRIME, N1, M = 198491317, 0xD2A80A3F, 1 << 32
    # noise(PRIME * (row * dim + r) + m, seed) = the 2-D fill's element (r, m) with the first row's offset folded into the seed
    return hip.sq5_fill_2d(dim, k, (seed + PRIME * row * dim * N1) % M)


@pytest.mark.parametrize("n,k", [(1, 1), (3000, 7), (3000, 8), (70001, 9), (300, 2047), (70001, 2049), (300, 2063), (5000, 4100)])
def test_terms_with_and_without_their_common_factor(hip, n, k):
    """Coefficients from which on the factor 2^-31 is applied term by term, everywhere or first from the second chunk of 2048 on, or only in the
    first: powers of two of the same coefficients give the same bits, larger by that power (n: a lane an element, or several)."""
    print(f"case common factor n={n} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    c = torch.randn(k, generator=g, device="cuda")
    values = lambda coef: hip.materialize_fwd(coef, (n,), (1,), 11, None, False)
    want = values(c)
    for p in (70, 76, 100):
        assert torch.equal(values(c * 2.0**p), want * 2.0**p), p
    for at in sorted({0, k // 2, k - 1}):   # one large coefficient among others
        big = c * 2.0**-40
        big[at] = 3.0e37
        noise = hip.sq5_fill_2d(n, k, 11).double()[:, at] if n <= 5000 else None
        got = values(big)
        assert bool(torch.isfinite(got).all())
        if noise is not None:
            assert rel(got, noise * 3.0e37) < 1e-6
    c[k - 1] = float("inf")
    assert not bool(torch.isfinite(values(c)).any())


@pytest.mark.parametrize("n,k", [(3000, 47), (3000, 48), (70001, 48), (3000, 49), (70001, 49), (300, 49), (70001, 55)])
def test_few_terms_and_more(hip, n, k):
    """Up to 48 terms have the factor applied term by term, more do not: the same sums on either side of the line."""
    test_terms_with_and_without_their_common_factor(hip, n, k)
    g = torch.Generator(device="cuda").manual_seed(n * k)
    c = torch.randn(k, generator=g, device="cuda")
    noise = hip.sq5_fill_2d(n, k, 11).double()
    got = hip.materialize_fwd(c, (n,), (1,), 11, None, False)
    # k fp32 multiply-adds one after the other, each rounded by at most 2^-24 of the running sum
    assert float((got.double() - noise @ c.double()).abs().max()) <= k * 2.0**-24 * float((noise.abs() @ c.double().abs()).max())


@pytest.mark.parametrize("n,k", [(131073, 49), (131200, 63), (131073, 64), (140001, 67), (131100, 2047), (131073, 2065), (131073, 2115)])
def test_one_thread_an_element_whatever_is_left_of_a_turn(hip, n, k):
    """From 2^17 elements on: turns of 16 terms, then fours, then single ones, in each chunk of 2048."""
    g = torch.Generator(device="cuda").manual_seed(k)
    c, d = torch.randn(k, generator=g, device="cuda"), torch.randn(n, generator=g, device="cuda")
    rows = torch.cat([torch.arange(300), torch.arange(n - 300, n)]).cuda()
    noise = hip.sq5_fill_2d(n, k, 5)
    # fp32 chains of k terms: 2^-24 each, relative to the largest partial sum
    assert rel(hip.materialize_fwd(c, (n,), (1,), 5, None, False)[rows], noise[rows].double() @ c.double()) < 2e-6
    want = sum(d[i : i + 20000].double() @ noise[i : i + 20000].double() for i in range(0, n, 20000))
    assert rel(hip.materialize_bwd(d, k, 5), want) < 2e-6


@pytest.mark.parametrize("k", [16, 17, 40, 64, 100, 256])
@pytest.mark.parametrize("n", [31, 32, 33, 255, 257, 287, 289, 600])
def test_gradient_at_the_edges_of_a_step(hip, n, k):
    """Steps of 32 elements, one to four waves along them, and values of one sign: every byte and digit counts."""
    g = torch.Generator(device="cuda").manual_seed(n * 1000 + k)
    d = torch.rand(n, generator=g, device="cuda") + 0.5
    noise = hip.sq5_fill_2d(n, k, 6)
    want = d.double() @ noise.double()
    # integers throughout and one rounding of a sum of some sqrt(n), 6e-8 of it; the oracle's noise is rounded to fp32, 4.5e-8 a term at most, of either sign
    assert float((hip.materialize_bwd(d, k, 6).double() - want).abs().max()) < 4e-7 * float(n) ** 0.5


@pytest.mark.parametrize("n", [524288, 524289, 1200001])
@pytest.mark.parametrize("k", [5, 48, 70, 2051])
def test_blocks_of_one_turn_and_of_several(hip, n, k):
    """One thread an element, on either side of what is resident at once (eight blocks to each of 256 compute units), alone and beside a bias."""
    import ctypes

    from randumb_amd import _lib

    class PseudoBias(ctypes.Structure):
        _fields_ = [("coef", ctypes.c_void_p), ("scale", ctypes.c_void_p), ("values", ctypes.c_void_p), ("k", ctypes.c_int64), ("seed", ctypes.c_uint32)]

    g = torch.Generator(device="cuda").manual_seed(k)
    c, cb = torch.randn(k, generator=g, device="cuda"), torch.randn(30, generator=g, device="cuda")
    got = hip.materialize_fwd(c, (n,), (1,), 5, None, False)
    rows = torch.cat([torch.arange(200), torch.arange(n // 2, n // 2 + 200), torch.arange(524188, 524288), torch.arange(n - 200, n)]).cuda()
    assert rel(got[rows], hip.sq5_fill_2d(n, k, 5)[rows].double() @ c.double()) < 2e-6   # chains of k terms, 2^-24 each
    w, b = torch.empty(n, device="cuda"), torch.empty(777, device="cuda")
    pb = PseudoBias(cb.data_ptr(), None, b.data_ptr(), 30, 6)
    assert _lib.load().rdb_materialize_weight_and_bias(w.data_ptr(), n, c.data_ptr(), k, 5, None, ctypes.byref(pb), 777, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(w, got) and torch.equal(b, hip.materialize_fwd(cb, (777,), (1,), 6, None, False))
