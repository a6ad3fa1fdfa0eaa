"""The random bias's share of layers with many tiles: R written to memory first, tiles of 192 or 256 features, R beside the projection."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# tiles of 192 features (as many rounds of them as of 256, at 256 compute units) whose last one has 8, 40 and 8 features, and of 256 with a last one of 8;
# the last token tile of 36, 52, 1 and 8 tokens
@pytest.mark.parametrize("T,in_f,out_f", [(8100, 584, 72), (5300, 1000, 136), (16385, 200, 264), (16264, 264, 72)])
def test_input_gradient_against_float64(T, in_f, out_f):
    from randumb_amd import _lib, hip

    print(f"case rbias tiles T={T} in={in_f} out={out_f}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(T)
    ref = ctypes.byref(hip._rbias_desc(T, in_f, out_f, 9))
    s = torch.tensor([0.37]).bfloat16().cuda()
    R = hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).bfloat16().double()   # what the kernels multiply
    FULL = 10
    n = lib.rdb_linear_workspace_bytes(FULL, ref)
    assert n >= 2 * in_f * out_f   # room for R
    ws = torch.full((n + 64,), 0x5A, dtype=torch.uint8, device="cuda")
    x, dy, dx0 = (torch.randn(T, cols + 8, generator=g).bfloat16().cuda() for cols in (in_f, out_f, in_f))
    dx, ds, dx_only = dx0.clone(), torch.full((2,), 5.0, device="cuda"), dx0.clone()
    args = (dy.data_ptr(), out_f + 8)
    assert lib.rdb_linear_rbias_bwd(dx.data_ptr(), in_f + 8, ds.data_ptr(), *args, x.data_ptr(), in_f + 8, s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    assert lib.rdb_linear_rbias_bwd(dx_only.data_ptr(), in_f + 8, None, *args, None, 0, s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    assert torch.equal(dx, dx_only) and torch.equal(dx[:, in_f:], dx0[:, in_f:]) and float(ds[1]) == 5.0 and bool((ws[n:] == 0x5A).all())
    dot = dy[:, :out_f].double() @ R
    want = dx0[:, :in_f].double() + s.double() * dot
    assert float((dx[:, :in_f].double() - want).norm() / want.norm()) < 2e-3   # one rounding to bf16: 2^-9 at most, 1.13e-3 as a norm
    xd = x[:, :in_f].double()
    assert abs(float(ds[0]) - float((dot * xd).sum())) < 1e-5 * float(dot.norm() * xd.norm())   # fp32 sums


# R beside a projection in one range of its contraction, in several, and ahead of one on 256-wide tiles (a launch of its own); sizes that are no multiple of
# a tile, fragment or k-step
@pytest.mark.parametrize("T,in_f,out_f,k", [(2040, 136, 2056, 8), (2100, 2056, 2008, 72), (8200, 264, 520, 520)])
def test_forward_against_float64(T, in_f, out_f, k):
    from randumb_amd import SillyLinear, hip

    print(f"case rbias forward T={T} in={in_f} out={out_f} k={k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    layer = SillyLinear(in_f, out_f, [k, k], [9, 10], bias=False, rt_bias=True, device="cuda", dtype=torch.bfloat16, matrix_coef=True)
    with torch.no_grad():
        layer.weight_coef.normal_(0.0, k**-0.5, generator=g)
        layer.weight_scale_bias.fill_(0.37)
    x = torch.randn(T, in_f, device="cuda", generator=g).bfloat16().requires_grad_()
    y = layer(x)
    N, R = hip.sq5_fill_2d(in_f, k, 9).double(), hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double()
    want = x.detach().double() @ (layer.weight_coef.detach().double() @ N.t() + layer.weight_scale_bias.detach().double() * R).t()
    assert float((y.detach().double() - want).norm() / want.norm()) < 6e-3   # N, z, R and y rounded to bf16 once each, 1.13e-3 as a norm; 2^-9 at most


# both shares of dx and all gradients in one call: both kinds of tiles, k of one step, of no multiple of a step and the largest; the last case adds up dy . C
# in ranges; rows of dx that are whole lines (760 + 8 and 1016 + 8 features apart), which leave past the caches, in both kinds of tiles.  The scratch holds NaN
# beforehand; the first case's state has no transposed coefficients
@pytest.mark.parametrize("T,in_f,out_f,k", [(8100, 584, 72, 8), (5300, 1000, 136, 72), (16385, 200, 264, 200), (16264, 264, 72, 256), (2100, 2056, 2056, 72),
                                            (8100, 760, 72, 72), (8190, 1016, 136, 200)])
def test_backward_in_one_call_against_float64(T, in_f, out_f, k):
    from randumb_amd import _lib, hip

    print(f"case rbias backward T={T} in={in_f} out={out_f} k={k}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(T)
    desc = hip._proj_desc(T, in_f, out_f, k, 9)
    ref = ctypes.byref(desc)
    n = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_BWD_PROJECTED_RBIAS, ref)
    assert n >= 2 * in_f * (out_f + k)   # room for R and N
    C = (torch.randn(out_f, k, device="cuda", generator=g) * k**-0.5).bfloat16()
    x, dy = (torch.randn(T, cols + 8, device="cuda", generator=g).bfloat16() for cols in (in_f, out_f))
    s = torch.tensor([0.37], device="cuda").bfloat16()
    state = hip.linear_project(x[:, :in_f], k, out_f, 9, None if k == 8 else C)
    ws = torch.full((n + 64,), 0xFF, dtype=torch.uint8, device="cuda")

    def call(dc, ds, room=n):   # ds None: x is not read
        ws.fill_(0xFF)
        dx = torch.full((T, in_f + 8), 5.0, device="cuda", dtype=torch.bfloat16)
        code = {torch.float32: _lib.RDB_F32, torch.bfloat16: _lib.RDB_BF16}
        rc = lib.rdb_linear_bwd_projected_rbias(dx.data_ptr(), in_f + 8, dc.data_ptr(), code[dc.dtype], None if ds is None else ds.data_ptr(),
                                                0 if ds is None else code[ds.dtype], dy.data_ptr(), out_f + 8, state.data_ptr(), None if ds is None else x.data_ptr(),
                                                0 if ds is None else in_f + 8, C.data_ptr(), s.data_ptr(), ref, ws.data_ptr(), room, stream)
        assert bool((ws[n:] == 0xFF).all()) and bool((dx[:, in_f:] == 5.0).all())
        return rc, dx[:, :in_f]

    ds, ds16, dc, dc32 = torch.full((2,), 5.0, device="cuda"), torch.full((2,), 5.0, device="cuda").bfloat16(), torch.empty_like(C), C.float()
    assert call(dc, ds, n - 1)[0] != 0 and float(ds[0]) == 5.0   # refused, not run
    (rc, dx), (rc16, dx16), (rc32, dx32) = call(dc, ds), call(dc.clone(), ds16), call(dc32, None)
    assert rc == rc16 == rc32 == 0 and torch.equal(dx, dx16) and torch.equal(dx, dx32)
    assert float(ds[1]) == float(ds16[1]) == 5.0 and torch.equal(ds[:1].bfloat16(), ds16[:1])
    # the coefficients' gradient is that of the layer without the bias, to the bit
    for got in (dc, dc32):
        want = hip.linear_bwd_projected(dy[:, :out_f], state, C, in_f, 9, dcoef_dtype=got.dtype)[1]
        assert torch.equal(got, want)
    N, R, xd, dyd = hip.sq5_fill_2d(in_f, k, 9).double(), hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).double(), x[:, :in_f].double(), dy[:, :out_f].double()
    dot = dyd @ R.bfloat16().double()
    want = dyd @ C.double() @ N.t() + s.double() * dyd @ R
    assert float((dx.double() - want).norm() / want.norm()) < 6e-3   # N, t, R and dx rounded to bf16 once each, 1.13e-3 as a norm; 2^-9 at most
    assert abs(float(ds[0]) - float((dot * xd).sum())) < 1e-5 * float(dot.norm() * xd.norm())   # fp32 sums


# rows of x so far apart that the offset of a token behind the last one, taken in 32 bits, lies between two rows: what is there is no part of the sum
def test_scale_gradient_reads_no_gap_between_rows():
    from randumb_amd import _lib, hip

    T, in_f, out_f, k, ldx = 16, 32768, 16, 24, 2**25 - 8
    print(f"case rbias backward, rows of x {ldx} apart", flush=True)
    assert T * ldx < 2**29 and 65 * ldx * 2 - 2**32 < ldx * 2   # taken as it is; the 66th row of a tile of 128
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device="cuda").manual_seed(T)
    ref = ctypes.byref(hip._proj_desc(T, in_f, out_f, k, 9))
    n = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_BWD_PROJECTED_RBIAS, ref)
    assert n > 0
    far = torch.full(((T - 1) * ldx + in_f,), float("nan"), device="cuda", dtype=torch.bfloat16)
    x = far.as_strided((T, in_f), (ldx, 1))
    x.copy_(torch.randn(T, in_f, device="cuda", generator=g))
    C, dy = (torch.randn(out_f, k, device="cuda", generator=g) * k**-0.5).bfloat16(), torch.randn(T, out_f, device="cuda", generator=g).bfloat16()
    s, ws, ds = torch.tensor([0.37], device="cuda").bfloat16(), torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(1, device="cuda")
    state = hip.linear_project(x.contiguous(), k, out_f, 9, C)
    dx, dc = torch.empty(T, in_f, device="cuda", dtype=torch.bfloat16), torch.empty_like(C)
    assert lib.rdb_linear_bwd_projected_rbias(dx.data_ptr(), in_f, dc.data_ptr(), _lib.RDB_BF16, ds.data_ptr(), _lib.RDB_F32, dy.data_ptr(), out_f, state.data_ptr(),
                                              x.data_ptr(), ldx, C.data_ptr(), s.data_ptr(), ref, ws.data_ptr(), n, stream) == 0
    dot = dy.double() @ hip.sq5_fill_1d(out_f * in_f, 9).view(out_f, in_f).bfloat16().double()
    assert abs(float(ds) - float((dot * x.double()).sum())) < 1e-5 * float(dot.norm() * x.double().norm())   # fp32 sums
