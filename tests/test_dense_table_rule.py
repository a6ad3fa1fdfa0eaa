"""Which dense tables' gradients go to the kernel of one launch, on the CPU (the rule counts 256 compute units there)."""
import pytest

from randumb_amd import _lib


@pytest.mark.parametrize("positions,vocab,dim,takes", [
    (1, 1, 8, 1), (6, 10, 64, 1), (64, 50304, 768, 0), (157, 50304, 768, 0), (158, 50304, 768, 1), (341, 65536, 504, 0), (342, 65536, 504, 1), (26, 5000, 8, 0), (27, 5000, 8, 1),   # one round of blocks
    (1024, 10, 384, 1), (1024, 10, 768, 0), (2048, 31, 1600, 0), (3072, 32, 1600, 1), (3073, 30, 64, 1), (8192, 81, 768, 0), (8192, 82, 768, 1), (16384, 65, 64, 0),                    # few rows
    (1023, 65537, 64, 0), (1024, 65537, 64, 1), (1535, 150000, 64, 0), (1536, 150000, 64, 1), (2047, 262144, 8, 0), (2048, 262144, 8, 1),   # several
    (16384, 262145, 760, 0), (2560, 262145, 768, 1), (4096, 524288, 768, 1), (16384, 524289, 4096, 0), (16384, 1000000, 8, 0),
    (16384, (1 << 29) + 1, 8, 0), (16385, 100, 8, 0), (0, 100, 8, 0), (16, 100, 12, 0)])
def test_where_the_lines_lie(positions, vocab, dim, takes):
    assert _lib.load().rdb_embedding_bwd_takes(positions, vocab, dim) == takes


@pytest.mark.parametrize("positions,vocab,dim", [(16, (1 << 30) + 1, 8), (16, 1 << 31, 8), (16385, 100, 8), (16, 100, 12)])
def test_what_one_launch_cannot_do_is_refused(positions, vocab, dim):
    """Before a launch: a grid of 2^32 threads and more is one that the runtime refuses."""
    lib = _lib.load()
    assert lib.rdb_embedding_bwd(None, None, 8, None, positions, vocab, dim, None) == -5 and b"2^29 rows" in lib.rdb_last_error_string()
    assert lib.rdb_embedding_bwd_takes(positions, vocab, dim) == 0
