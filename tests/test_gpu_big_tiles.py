"""The 256-wide, persistent kernels of the projected entry points (k > 256) against the 128-wide ones and the CPU oracle.

Both kinds contract in the same order (stage after stage of 64, k-step after k-step of 16, fp32 accumulators of the same matrix
instruction), so y and dx must be equal bit for bit.  dcoef is equal bit for bit where the 128-wide kernels contract all tokens
in one range too (few tokens, or many output tiles); where they add up partial sums over token ranges the two differ by fp32
rounding only (1e-6 of the norm).  The oracle comparison holds the bf16 tolerance of the path (2e-2)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BF16_TOL = 2e-2


def rel_l2(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.fixture(scope="module")
def hip():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from randumb_amd import hip as h

    return h


def _inputs(T, in_f, out_f, k, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, in_f, generator=g).bfloat16()
    dy = torch.randn(T, out_f, generator=g).bfloat16()
    coef = (torch.randn(out_f, k, generator=g) * (3.0 / k) ** 0.5 * 0.05).bfloat16()
    bias = torch.randn(out_f, generator=g).bfloat16()
    return x, dy, coef, bias


def _run(hip, mode, x, dy, coef, bias, in_f, out_f, k, seed, with_ct):
    before = hip.set_big_tiles(mode)
    try:
        z = hip.linear_project(x, k, out_f, seed, coef=coef if with_ct else None)
        y = hip.linear_fwd_projected(z, coef, in_f, seed, bias=bias)
        dx, dc = hip.linear_bwd_projected(dy, z, coef, in_f, seed)
        dc_alone = hip.linear_bwd_dcoef_projected(dy, z, k, in_f, seed)   # the coefficient gradient's own entry point
        torch.cuda.synchronize()
    finally:
        hip.set_big_tiles(before)
    # one pass over all tokens on the 256-wide tiles, fp32 atomics over token ranges on the 128-wide ones
    assert rel_l2(dc_alone.cpu().numpy(), dc.cpu().numpy()) < 1e-6
    if mode == 2:
        assert torch.equal(dc_alone, dc)
    return y, dx, dc


SHAPES = [
    # tokens, in_f, out_f, k, seed
    (300, 128, 264, 512, 2),      # one ragged tile in every direction
    (1000, 200, 520, 328, 5),     # k = 8 mod 16 (padded to 384 in the state), three output tiles, four token tiles
    (2088, 256, 4104, 1024, 7),   # many tiles: several rounds per block, a half-tile tail round, ragged edges
    (128, 64, 8, 264, 1),         # a single tile, mostly padding
]


@pytest.mark.parametrize("T,in_f,out_f,k,seed", SHAPES)
@pytest.mark.parametrize("with_ct", [True, False])
@pytest.mark.parametrize("with_bias", [True, False])
def test_big_tiles_equal_the_128_wide_kernels(hip, T, in_f, out_f, k, seed, with_ct, with_bias):
    print(f"case big tiles T={T} in={in_f} out={out_f} k={k} ct={with_ct} bias={with_bias}", flush=True)
    x, dy, coef, bias = [t.cuda() for t in _inputs(T, in_f, out_f, k, seed)]
    b = bias if with_bias else None
    want = _run(hip, 0, x, dy, coef, b, in_f, out_f, k, seed, with_ct)
    got = _run(hip, 2, x, dy, coef, b, in_f, out_f, k, seed, with_ct)
    for name, a, w in zip(("y", "dx"), got, want):
        assert a.shape == w.shape and torch.equal(a, w), f"{name} differs between the 256-wide and the 128-wide kernels"
    if T <= 256:   # a single token range in the 128-wide kernels as well
        assert torch.equal(got[2], want[2])
    assert got[2].shape == want[2].shape and rel_l2(got[2].cpu().numpy(), want[2].cpu().numpy()) < 1e-6
    # twice in a row on the same buffers: the same bits (no atomics, no state left behind by the persistent blocks)
    again = _run(hip, 2, x, dy, coef, b, in_f, out_f, k, seed, with_ct)
    for a, w in zip(again, got):
        assert torch.equal(a, w)


def test_big_tiles_against_the_oracle(hip, oracle):
    T, in_f, out_f, k, seed = 520, 136, 528, 384, 11
    print(f"case big tiles oracle T={T} in={in_f} out={out_f} k={k}", flush=True)
    x, dy, coef, bias = _inputs(T, in_f, out_f, k, seed)
    xn, dyn, cn = x.float().numpy(), dy.float().numpy(), coef.float().numpy()
    want_y = oracle.linear_fwd(xn, cn, in_f, out_f, seed, bias=bias.float().numpy())
    want_dx, want_dc, _ = oracle.linear_bwd(xn, dyn, cn, in_f, out_f, seed)
    y, dx, dc = _run(hip, 2, x.cuda(), dy.cuda(), coef.cuda(), bias.cuda(), in_f, out_f, k, seed, True)
    assert rel_l2(y.float().cpu().numpy(), want_y) < BF16_TOL
    assert rel_l2(dx.float().cpu().numpy(), want_dx) < BF16_TOL
    assert rel_l2(dc.float().cpu().numpy(), want_dc) < BF16_TOL


def test_big_tiles_run_by_default_on_a_layer_with_many_tiles(hip):
    """4096 -> 14336 with k = 1024 at 4096 tokens takes the 256-wide kernels without being asked to: same bits as with them off."""
    T, in_f, out_f, k, seed = 4096, 4096, 14336, 1024, 0
    print("case big tiles default", flush=True)
    x, dy, coef, _ = [t.cuda() for t in _inputs(T, in_f, out_f, k, seed)]
    assert hip.set_big_tiles(1) == 1   # the default mode
    got = _run(hip, 1, x, dy, coef, None, in_f, out_f, k, seed, True)
    want = _run(hip, 0, x, dy, coef, None, in_f, out_f, k, seed, True)
    for a, w in zip(got, want):
        assert torch.equal(a, w)


def test_big_tiles_random_shapes(hip):
    """Sixteen random layers with k > 256 (sizes in multiples of 8, tokens any number, ragged against every tile edge), with
    the transposed coefficients in the state or not, with the ordered-sum workspace or the smaller one."""
    rng = np.random.default_rng(31)
    for case in range(16):
        T = int(rng.integers(1, 160)) * 8 - int(rng.integers(0, 8))
        in_f, out_f = (int(rng.integers(1, 100)) * 8 for _ in range(2))
        k = int(rng.integers(33, 130)) * 8                      # 264 .. 1032
        seed = int(rng.integers(0, 2**32))
        print(f"case big tiles random {case}: T={T} in={in_f} out={out_f} k={k} seed={seed}", flush=True)
        x, dy, coef, bias = [t.cuda() for t in _inputs(T, in_f, out_f, k, case)]
        b = bias if case % 2 else None
        outs = {}
        for mode in (0, 2):
            before = hip.set_big_tiles(mode)
            try:
                z = hip.linear_project(x, k, out_f, seed, coef=coef if case % 3 else None)
                y = hip.linear_fwd_projected(z, coef, in_f, seed, bias=b)
                dx, dc = hip.linear_bwd_projected(dy, z, coef, in_f, seed, ordered_sums=case % 4 != 0)
                torch.cuda.synchronize()
            finally:
                hip.set_big_tiles(before)
            outs[mode] = (y, dx, dc)
        assert torch.equal(outs[2][0], outs[0][0]) and torch.equal(outs[2][1], outs[0][1]), case
        assert rel_l2(outs[2][2].cpu().numpy(), outs[0][2].cpu().numpy()) < 1e-5, case   # atomics / token ranges in the 128-wide kernels


def test_big_tiles_take_leading_dimensions(hip):
    """dy as a column slice of a wider matrix and y, dx written into wider matrices: same bits as on contiguous buffers."""
    import ctypes

    from randumb_amd import _lib
    from randumb_amd.hip import RDB_OP_LINEAR_BWD_PROJECTED, _p, _proj_desc, _stream

    print("case big tiles on strided activations", flush=True)
    T, in_f, out_f, k, seed = 700, 264, 520, 520, 4
    g = torch.Generator().manual_seed(8)
    x = torch.randn(T, in_f, generator=g).bfloat16().cuda()
    dyw = torch.randn(T, out_f + 24, generator=g).bfloat16().cuda()
    C = (torch.randn(out_f, k, generator=g) * 0.05).bfloat16().cuda()
    dy = dyw[:, 8:8 + out_f]
    L = _lib.load()
    before = hip.set_big_tiles(2)
    try:
        z = hip.linear_project(x, k, out_f, seed, coef=C)
        y_c = hip.linear_fwd_projected(z, C, in_f, seed)
        dx_c, dC_c = hip.linear_bwd_projected(dy.contiguous(), z, C, in_f, seed)
        d = _proj_desc(T, in_f, out_f, k, seed)
        yw = torch.full((T, out_f + 40), 7.0, dtype=torch.bfloat16, device="cuda")
        dxw = torch.full((T, in_f + 16), 7.0, dtype=torch.bfloat16, device="cuda")
        dC = torch.empty(out_f, k, dtype=torch.float32, device="cuda")
        y, dx = yw[:, 16:16 + out_f], dxw[:, 8:8 + in_f]
        n = L.rdb_linear_workspace_bytes(RDB_OP_LINEAR_BWD_PROJECTED, ctypes.byref(d))
        ws = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
        st = _stream(x.device)
        _lib.check(L.rdb_linear_fwd_projected(_p(y), y.stride(0), _p(z), _p(C), None, ctypes.byref(d), st), "rdb_linear_fwd_projected")
        _lib.check(L.rdb_linear_bwd_projected(_p(dx), dx.stride(0), _p(dC), _p(dy), dy.stride(0), _p(z), _p(C), ctypes.byref(d), _p(ws), n, st),
                   "rdb_linear_bwd_projected")
        torch.cuda.synchronize()
    finally:
        hip.set_big_tiles(before)
    assert torch.equal(y, y_c) and torch.equal(dx, dx_c) and torch.equal(dC, dC_c)
    # nothing outside the slices was written
    assert bool((yw[:, :16] == 7).all()) and bool((yw[:, 16 + out_f:] == 7).all())
    assert bool((dxw[:, :8] == 7).all()) and bool((dxw[:, 8 + in_f:] == 7).all())


def test_big_tiles_through_the_layer(hip):
    """SillyLinear in matrix-coef form with k = 512: forward, backward and the gradients of input and coefficients are the
    same with the 256-wide kernels as with the 128-wide ones (autograd function, custom ops and C ABI in between)."""
    import randumb_amd as rten

    print("case big tiles through SillyLinear", flush=True)
    torch.manual_seed(3)
    outs = {}
    for mode in (0, 2):
        before = hip.set_big_tiles(mode)
        try:
            assert hip.linear_projection_preferred(300, 1032, 2056, 512)   # the projected kernels are what the layer runs
            layer = rten.SillyLinear(1032, 2056, [512, 512], [9, 10], bias=False, matrix_coef=True).to(torch.bfloat16).cuda()
            with torch.no_grad():
                g = torch.Generator().manual_seed(5)
                layer.weight_coef.copy_((torch.randn(2056, 512, generator=g) * 0.02).bfloat16())
                layer.weight_scale_bias.zero_()
            x = torch.randn(300, 1032, generator=torch.Generator().manual_seed(6)).bfloat16().cuda().requires_grad_(True)
            y = layer(x)
            (y.float() ** 2).sum().backward()
            torch.cuda.synchronize()
            outs[mode] = (y.detach(), x.grad.detach(), layer.weight_coef.grad.detach())
        finally:
            hip.set_big_tiles(before)
    assert torch.equal(outs[2][0], outs[0][0]) and torch.equal(outs[2][1], outs[0][1])
    assert rel_l2(outs[2][2].float().cpu().numpy(), outs[0][2].float().cpu().numpy()) < 1e-2   # bf16 gradients of fp32 sums in two orders
    assert float(outs[2][2].float().abs().sum()) > 0


def test_big_tiles_on_chunked_tokens(hip):
    """40000 tokens x 14336 output features hold more elements than one launch addresses: the projected calls run the layer
    in chunks of tokens, the later chunks adding to dcoef.  Same y and dx bit for bit on both kinds of kernels, same dcoef up to
    the order of fp32 sums, and the same dcoef bit for bit on a second run."""
    T, in_f, out_f, k, seed = 40000, 256, 14336, 512, 3
    print(f"case big tiles chunked T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator().manual_seed(12)
    x = torch.randn(T, in_f, generator=g).bfloat16().cuda()
    dy = (torch.randn(T, 64, generator=g).bfloat16().cuda()).repeat(1, out_f // 64)   # cheap to make, still different per column block
    dy = dy * torch.linspace(0.5, 1.5, out_f, device="cuda").bfloat16()
    coef = (torch.randn(out_f, k, generator=g) * 0.01).bfloat16().cuda()
    outs = {}
    for mode in (0, 2, 2):
        before = hip.set_big_tiles(mode)
        try:
            z = hip.linear_project(x, k, out_f, seed, coef=coef)
            y = hip.linear_fwd_projected(z, coef, in_f, seed)
            dx, dc = hip.linear_bwd_projected(dy, z, coef, in_f, seed)
            torch.cuda.synchronize()
        finally:
            hip.set_big_tiles(before)
        if mode in outs:   # second run on the 256-wide kernels
            assert torch.equal(outs[mode][2], dc) and torch.equal(outs[mode][0], y)
        outs[mode] = (y, dx, dc)
        del z
    assert torch.equal(outs[2][0], outs[0][0]) and torch.equal(outs[2][1], outs[0][1])
    assert rel_l2(outs[2][2].cpu().numpy(), outs[0][2].cpu().numpy()) < 1e-5
    assert float(outs[2][2].abs().sum()) > 0


@pytest.mark.parametrize("T,in_f,out_f,k", [(300, 264, 512, 264), (128, 8, 264, 264), (2088, 1032, 520, 1000), (257, 520, 256, 328)])
def test_backward_with_the_noise_from_memory(T, in_f, out_f, k):
    """dx = t . N with N written once, and dC rounded to bf16 by the tiles themselves: the bits of the kernel that hashes and of the
    launch that adds fp32 sums up; also with a workspace that has no room for N."""
    import ctypes

    from randumb_amd import _lib, hip, ops

    lib = _lib.load()
    g = torch.Generator().manual_seed(k)
    x, dy = torch.randn(T, in_f, generator=g).bfloat16().cuda(), torch.randn(T, out_f, generator=g).bfloat16().cuda()
    c = (torch.randn(out_f, k, generator=g) / k ** 0.5).bfloat16().cuda()
    d = hip._desc(T, in_f, out_f, c, in_f, 1, 5, torch.bfloat16, 0)
    ref = ctypes.byref(d)
    old = lib.rdb_set_big_tiles(2)
    try:
        y, state = hip.linear_project_fwd(x, c, 5)
        full = lib.rdb_linear_workspace_bytes(4, ref)
        table = -(-in_f // 32) * 32 * -(-k // 64) * 64 * 2
        results = []
        for size, dtype in ((full, torch.bfloat16), (full - table, torch.bfloat16), (full, torch.float32)):
            dx, dc = torch.empty_like(x), torch.empty(out_f, k, dtype=dtype, device="cuda")
            ws = torch.empty(size, dtype=torch.uint8, device="cuda")
            rc = lib.rdb_linear_bwd_projected_to(dx.data_ptr(), in_f, dc.data_ptr(), 1 if dtype == torch.bfloat16 else 0, dy.data_ptr(), out_f,
                                                 state.data_ptr(), c.data_ptr(), ref, ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)
            assert rc == 0
            results.append((dx, dc))
    finally:
        lib.rdb_set_big_tiles(old)
    for dx, dc in results[1:]:
        assert torch.equal(dx, results[0][0]) and torch.equal(dc.bfloat16(), results[0][1])
    N = ops.sq5_gen_2d(in_f, k, 5).float().cpu()
    t = dy.float().cpu() @ c.float().cpu()
    want_dx, want_dc = t @ N.t(), dy.float().cpu().t() @ (x.float().cpu() @ N)
    for got, want in ((results[0][0], want_dx), (results[0][1], want_dc)):
        assert float((got.float().cpu() - want).norm() / want.norm()) < 1e-2


@pytest.mark.parametrize("T,in_f,out_f,k", [(300, 128, 264, 512), (1000, 200, 520, 328), (129, 1032, 2056, 264), (2088, 264, 4104, 1024), (32, 72, 1096, 264)])
def test_projection_with_the_noise_from_memory(hip, T, in_f, out_f, k):
    """z, z^T and C^T of the call that also forms y (256-wide tiles, N in y's rows) against those of the projection on its own (the kernel
    that hashes): the same bits in everything computed from them, and in the state's pieces where nothing is padding."""
    x, dy, coef, bias = [t.cuda() for t in _inputs(T, in_f, out_f, k, 3)]
    want = _run(hip, 0, x, dy, coef, bias, in_f, out_f, k, 3, True)
    before = hip.set_big_tiles(2)
    try:
        y, state = hip.linear_project_fwd(x, coef, 3, bias=bias)
        alone = hip.linear_project(x, k, out_f, 3, coef=coef)
        dx, dc = hip.linear_bwd_projected(dy, state, coef, in_f, 3)
        dx_alone, dc_alone = hip.linear_bwd_projected(dy, alone, coef, in_f, 3)
        torch.cuda.synchronize()
    finally:
        hip.set_big_tiles(before)
    assert torch.equal(y, want[0]) and torch.equal(dx, want[1]) and torch.equal(dx, dx_alone) and torch.equal(dc, dc_alone)


@pytest.mark.parametrize("T,in_f,out_f", [(300, 264, 520), (129, 8, 1032), (513, 1000, 72), (128, 64, 64), (2056, 520, 776)])
def test_random_bias_from_memory(T, in_f, out_f):
    """The random bias's share on 256-wide tiles against the kernels that hash it: the same bits in y and dx (the same products in the same
    order); the scale's gradient adds the same terms up in other groups (fp32)."""
    import ctypes

    from randumb_amd import _lib, hip

    lib = _lib.load()
    g = torch.Generator().manual_seed(T)
    x, dy = torch.randn(T, in_f, generator=g).bfloat16().cuda(), torch.randn(T, out_f, generator=g).bfloat16().cuda()
    y0, dx0 = torch.randn(T, out_f, generator=g).bfloat16().cuda(), torch.randn(T, in_f, generator=g).bfloat16().cuda()
    s = torch.tensor([0.375]).bfloat16().cuda()
    ref = ctypes.byref(hip._rbias_desc(T, in_f, out_f, 9))
    stream = torch.cuda.current_stream().cuda_stream
    old = lib.rdb_set_big_tiles(2)
    try:
        dots = -(-in_f // 64) * -(-T // 256) * 4
        out = []
        for table in (True, False):
            fwd, bwd = [lib.rdb_linear_workspace_bytes(op, ref) if table else n for op, n in ((8, 0), (10, dots))]
            if table:
                assert fwd >= in_f * out_f * 2 and bwd >= dots + in_f * out_f * 2
            y, dx, dx_only, ds = y0.clone(), dx0.clone(), dx0.clone(), torch.empty(1, device="cuda")
            ws = torch.empty(max(fwd, bwd, 256), dtype=torch.uint8, device="cuda")
            assert lib.rdb_linear_rbias_fwd_ws(y.data_ptr(), out_f, x.data_ptr(), in_f, s.data_ptr(), ref, ws.data_ptr(), fwd, stream) == 0
            assert lib.rdb_linear_rbias_bwd(dx.data_ptr(), in_f, ds.data_ptr(), dy.data_ptr(), out_f, x.data_ptr(), in_f, s.data_ptr(), ref, ws.data_ptr(), bwd,
                                            stream) == 0
            assert lib.rdb_linear_rbias_bwd(dx_only.data_ptr(), in_f, None, dy.data_ptr(), out_f, None, 0, s.data_ptr(), ref, ws.data_ptr(), bwd, stream) == 0
            assert torch.equal(dx, dx_only)
            out.append((y, dx, float(ds)))
    finally:
        lib.rdb_set_big_tiles(old)
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    # the sum of T * in_f terms of mean square out_f / 3: fp32 roundings of it, in two orders
    assert abs(out[0][2] - out[1][2]) < 1e-5 * (T * in_f * out_f / 3) ** 0.5


@pytest.mark.parametrize("T,in_f,out_f,k,with_bias", [(300, 264, 520, 72, True), (129, 64, 1032, 264, False), (2056, 520, 776, 256, True), (513, 1000, 72, 328, False)])
def test_forward_with_the_random_bias_in_one_product(T, in_f, out_f, k, with_bias):
    """y = z . C^T + s * x . R^T + bias with one rounding: no further from float64 than the two products that round twice, the same state,
    and the odd workspace refused."""
    import ctypes

    from randumb_amd import _lib, hip, ops

    lib = _lib.load()
    x, _, coef, bias = [t.cuda() for t in _inputs(T, in_f, out_f, k, 11)]
    b = bias if with_bias else None
    s = torch.tensor([0.0625]).bfloat16().cuda()
    d = hip._desc(T, in_f, out_f, coef, in_f, 1, 4, torch.bfloat16, 0)
    ref = ctypes.byref(d)
    stream = torch.cuda.current_stream().cuda_stream
    old = lib.rdb_set_big_tiles(2)
    try:
        y2, state = hip.linear_project_fwd(x, coef, 4, bias=b)
        assert lib.rdb_linear_rbias_fwd(y2.data_ptr(), out_f, x.data_ptr(), in_f, s.data_ptr(), ref, stream) == 0
        need = lib.rdb_linear_workspace_bytes(9, ref)
        assert need >= in_f * out_f * 2
        ws, y, state1 = torch.empty(need, dtype=torch.uint8, device="cuda"), torch.empty_like(y2), torch.zeros_like(state)

        def call(size):
            return lib.rdb_linear_project_fwd_rbias(y.data_ptr(), out_f, state1.data_ptr(), x.data_ptr(), in_f, coef.data_ptr(), s.data_ptr(),
                                                    b.data_ptr() if with_bias else None, ref, ws.data_ptr(), size, stream)

        assert call(need - 1) != 0 and call(need) == 0
        again = hip.linear_fwd_projected(state1, coef, in_f, 4, bias=b)
        first = hip.linear_fwd_projected(state, coef, in_f, 4, bias=b)
    finally:
        lib.rdb_set_big_tiles(old)
    assert torch.equal(again, first)
    N = ops.sq5_gen_2d(in_f, k, 4).double().cpu()
    R = ops.sq5_gen_1d(in_f * out_f, 4).double().cpu().view(out_f, in_f)
    W = coef.double().cpu() @ N.t() + 0.0625 * R
    want = x.double().cpu() @ W.t() + (bias.double().cpu() if with_bias else 0.0)
    err, err2 = [float((t.double().cpu() - want).norm() / want.norm()) for t in (y, y2)]
    assert err < 8e-3 and err <= 1.02 * err2
