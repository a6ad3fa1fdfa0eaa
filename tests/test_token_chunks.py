"""Layers of more tokens than one launch addresses: every chunk of tokens keeps within its own part of the projection state."""
import ctypes
import random

import pytest
import torch

from randumb_amd import _lib

# tokens, in_f, out_f, k: a last chunk with fewer tokens than the others, and so with more ranges of its projection's contraction
SHORT_LAST = [(33024, 8192, 64, 64), (21672, 14336, 256, 64), (10960, 28672, 512, 128), (27884, 32408, 56, 64)]


def _desc(tokens, in_f, out_f, k):
    d = _lib.LinearDesc()
    d.tokens, d.in_f, d.out_f, d.k, d.coef_rows, d.sO, d.sI, d.seed = tokens, in_f, out_f, k, out_f, in_f, 1, 5
    d.act_dtype = d.coef_dtype = _lib.RDB_BF16
    d.algo = _lib.RDB_ALGO_AUTO
    return d


def _chunks(lib, d):
    per = ctypes.c_int64()
    return lib.rdb_linear_projection_chunks(ctypes.byref(d), ctypes.byref(per)), per.value


def test_the_last_chunk_fits_its_part_of_the_state():
    lib, rng = _lib.load(), random.Random(7)
    cases = list(SHORT_LAST)
    while len(cases) < 4000:
        in_f, out_f, k = (max(8, int(2 ** rng.uniform(*r)) // 8 * 8) for r in ((8, 15), (3, 14), (3, 9)))
        cases.append((int((1 << 28) / max(in_f, out_f, k) * rng.uniform(1.0, 4.2)), in_f, out_f, k))
    several = with_scratch = 0
    for case in cases:
        d = _desc(*case)
        n, per = _chunks(lib, d)
        if n < 2:
            continue
        several += 1
        part = lib.rdb_linear_projection_bytes(ctypes.byref(d)) // n
        last = _desc(case[0] - (n - 1) * per, *case[1:])
        assert 0 < last.tokens <= per and lib.rdb_linear_projection_bytes(ctypes.byref(last)) <= part, case
        scratch = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_PROJECT, ctypes.byref(d))
        assert lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_PROJECT, ctypes.byref(last)) <= scratch, case
        with_scratch += scratch > 0
    assert several > 3000 and with_scratch > 20


@pytest.mark.gpu
@pytest.mark.parametrize("T,in_f,out_f,k", [SHORT_LAST[0], SHORT_LAST[3]])
def test_nothing_is_written_behind_the_state_and_the_scratch(T, in_f, out_f, k):
    from randumb_amd import hip

    print(f"case token chunks T={T} in={in_f} out={out_f} k={k}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    d = _desc(T, in_f, out_f, k)
    ref, n = ctypes.byref(d), lib.rdb_linear_projection_bytes(ctypes.byref(d))
    g = torch.Generator(device="cuda").manual_seed(3)
    x = torch.randn(T, in_f, device="cuda", generator=g, dtype=torch.bfloat16)
    c = (torch.randn(out_f, k, device="cuda", generator=g) / k ** 0.5).bfloat16()
    N = hip.sq5_fill_2d(in_f, k, 5)
    want = torch.cat([p.float() @ N @ c.float().t() for p in x.split(4096)])
    state = torch.full((n + (16 << 20),), 0x5A, dtype=torch.uint8, device="cuda")
    m = lib.rdb_linear_workspace_bytes(_lib.RDB_OP_LINEAR_PROJECT, ref)
    ws = torch.full((m + (16 << 20),), 0x5A, dtype=torch.uint8, device="cuda")
    first = None
    for with_y, room in ((True, 0), (True, m), (False, m), (False, m - 256)):
        y = torch.full((T, out_f), float("nan"), device="cuda", dtype=torch.bfloat16)
        if with_y:
            rc = lib.rdb_linear_project_fwd_ws(y.data_ptr(), out_f, state.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), None, ref, ws.data_ptr(), room, stream)
        else:
            rc = lib.rdb_linear_project_ws(state.data_ptr(), x.data_ptr(), in_f, c.data_ptr(), ref, ws.data_ptr(), room, stream)
            rc = rc or lib.rdb_linear_fwd_projected(y.data_ptr(), out_f, state.data_ptr(), c.data_ptr(), None, ref, stream)
        assert rc == 0 and bool((state[n:] == 0x5A).all()) and bool((ws[m:] == 0x5A).all())
        first = y if first is None else first
        assert m > 0 and torch.equal(y, first)   # the same ranges in the same order, whoever adds them up
        assert float((y.float() - want).norm() / want.norm()) < 8e-3   # z and y rounded to bf16: 2^-9 each at most, fewer values than a norm needs
    hip.sync_check()
