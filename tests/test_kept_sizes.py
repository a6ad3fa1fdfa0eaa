"""What a layer keeps from its forward to its backward pass: z and, in bf16, the transposed coefficients; scratch of the forward pass is asked for apart."""
import ctypes
import random

import pytest

from randumb_amd import _lib


def _desc(tokens, in_f, out_f, k, dtype):
    d = _lib.LinearDesc()
    d.tokens, d.in_f, d.out_f, d.k, d.coef_rows, d.sO, d.sI, d.seed = tokens, in_f, out_f, k, out_f, in_f, 1, 5
    d.act_dtype = d.coef_dtype = dtype
    d.algo = _lib.RDB_ALGO_AUTO
    return d


def _up(n, to=256):
    return -(-n // to) * to


# narrow layers, whose projection runs in ranges that y has no room for, among layers of any shape
CASES = [(2048, 3072, 768, 256), (256, 8192, 1024, 512), (257, 8192, 1024, 32), (700, 4000, 256, 120), (492, 3184, 273, 118), (433, 3320, 96, 144)]


@pytest.mark.parametrize("tokens,in_f,out_f", [(30138, 111, 331), (13811, 135, 211), (9080, 280, 560), (9000, 24, 40)])
@pytest.mark.parametrize("dx", [0, 1])
def test_many_tokens_of_a_small_vector_coef_layer(tokens, in_f, out_f, dx):
    """The backward pass in one call has room for as many ranges of dW as the product alone, up to 16 MB: with eight at most its few tiles run on for most of the step."""
    lib = _lib.load()
    assert lib.rdb_vector_linear_bwd_workspace_bytes(tokens, in_f, out_f, 16, dx, 0) >= min(lib.rdb_product_f32_workspace_bytes(out_f, in_f, tokens), 16 << 20)


@pytest.mark.parametrize("tokens,in_f,out_f", [(8192, 768, 3072), (19876, 1288, 680)])
def test_a_long_product_of_dw_alone_has_room_for_ranges(tokens, in_f, out_f):
    """Without dx beside it there is nothing to fill its last round of tiles."""
    lib = _lib.load()
    assert lib.rdb_vector_linear_bwd_workspace_bytes(tokens, in_f, out_f, 8, 0, 0) >= min(lib.rdb_product_f32_workspace_bytes(out_f, in_f, tokens), 28 << 20)


@pytest.mark.parametrize("tokens,in_f,out_f,dx,ranges", [(1722, 1388, 1566, 0, 3), (8192, 1388, 1566, 1, 2), (8192, 1771, 1463, 1, 2), (1400, 768, 3072, 1, 2)])
def test_a_dw_of_few_tiles_has_room_for_ranges(tokens, in_f, out_f, dx, ranges):
    """Fewer tiles than two to three compute units: in one range they are the last to be done, with dx beside them too."""
    lib = _lib.load()
    assert lib.rdb_vector_linear_bwd_workspace_bytes(tokens, in_f, out_f, 8, dx, 0) >= ranges * in_f * out_f * 4


@pytest.mark.parametrize("tokens,in_f,out_f,alone", [(29, 8, 10, 0), (2, 769, 314, 0), (59, 78, 1915, 0), (13448, 1031, 73, 0), (8169, 9, 2565, 0), (333, 84, 23, 1), (443, 42, 287, 1), (8192, 768, 3072, 1)])
def test_where_a_vector_coef_gradient_alone_pays_in_one_call(tokens, in_f, out_f, alone):
    """Where it saves the launch that adds up dW's ranges; with dx or a bias it saves others."""
    lib = _lib.load()
    assert [lib.rdb_vector_linear_bwd_pays(tokens, in_f, out_f, dx, bias) for dx, bias in ((0, 0), (0, 1), (1, 0), (1, 1))] == [alone, 1, 1, 1]
    assert lib.rdb_vector_linear_bwd_pays(0, in_f, out_f, 1, 1) == 0


@pytest.mark.parametrize("dtype", [_lib.RDB_BF16, _lib.RDB_F32])
def test_nothing_but_what_the_backward_pass_reads(dtype):
    lib, rng = _lib.load(), random.Random(3)
    cases = CASES + [tuple(int(2 ** rng.uniform(*r)) for r in ((5, 13), (3, 13), (0, 12), (3, 9))) for _ in range(3000)]
    scratch = 0
    for T, in_f, out_f, k in cases:
        ref = ctypes.byref(_desc(T, in_f, out_f, k, dtype))
        state, kept = lib.rdb_linear_projection_bytes(ref), lib.rdb_linear_kept_bytes(ref)
        assert kept in (0, _up(4 * T * k)), (T, in_f, out_f, k)
        if dtype == _lib.RDB_F32:
            assert state == 256 + _up(4 * T * k), (T, in_f, out_f, k)
        elif state:
            kpad = _up(k, 64)
            z, z_t, c_t, tags = (_up(n) for n in (_up(T, 32) * kpad * 2, _up(T, 64) * kpad * 2, _up(out_f, 64) * kpad * 2, -(-T // 256) * (kpad // 32 + 1) * 8))
            assert state == 256 + z + z_t + c_t + tags, (T, in_f, out_f, k)
        for op, has in ((_lib.RDB_OP_LINEAR_PROJECT, state), (_lib.RDB_OP_LINEAR_FWD_KEPT, kept)):
            n = lib.rdb_linear_workspace_bytes(op, ref)
            assert 0 <= n <= 33 << 20 and (has or n == 0), (T, in_f, out_f, k, op)
            scratch += n > 0
    assert scratch > 20


def test_a_forward_pass_alone_runs_its_projection_in_ranges():
    """Few tiles of z with long contractions: a training step may do without the launch that adds ranges up, a forward pass waits for its kernels."""
    lib = _lib.load()
    for T, in_f, out_f, k in ((4700, 496, 32, 16), (2086, 368, 2352, 8), (470, 336, 3624, 104)):
        n = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_FWD, ctypes.byref(_desc(T, in_f, out_f, k, _lib.RDB_F32)))
        assert n >= 3 * _up(4 * T * k), (T, in_f, out_f, k)


def test_short_inputs_of_narrow_layers_take_one_range():
    lib = _lib.load()
    for in_f, ranges in ((1040, False), (1344, False), (1352, True)):   # 17, 21 and 22 stages of 64 features
        n = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_PROJECT, ctypes.byref(_desc(2304, in_f, 32, 16, _lib.RDB_BF16)))
        assert (n > 0) == ranges, (in_f, n)


@pytest.mark.parametrize("T,in_f,out_f,k", [(8192, 3072, 768, 256), (8192, 768, 768, 200), (6000, 2048, 6144, 200), (6000, 1000, 1000, 192), (4096, 8192, 1024, 136)])
def test_the_backward_pass_with_a_random_bias_has_room_for_the_noise_once(T, in_f, out_f, k):
    """Its scratch: that of the layer without the bias, which holds N^T for these, and R, the shares of the scale's gradient and a word to count in."""
    lib, RBIAS_BWD_FULL = _lib.load(), 10
    d, rbias = _desc(T, in_f, out_f, k, _lib.RDB_BF16), _desc(T, in_f, out_f, 8, _lib.RDB_BF16)
    ops = (_lib.RDB_OP_LINEAR_BWD_PROJECTED_RBIAS, _lib.RDB_OP_LINEAR_BWD_PROJECTED_TO, RBIAS_BWD_FULL)
    both, base, more = (lib.rdb_linear_workspace_bytes(op, ctypes.byref(x)) for op, x in zip(ops, (d, d, rbias)))
    assert both and more > 2 * in_f * out_f and both <= base + more + 3 * 256, (both, base, more)
