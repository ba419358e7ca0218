"""Which kernels the library launches, on the CPU (tests/launch_log.py): the
dispatch rules on sizes, types and alignment."""
import pytest

from prichs_amd import _lib as L
from tests import launch_log as ll

OPS = {"ab": L.MATMUL_AB, "atb": L.MATMUL_ATB, "abt": L.MATMUL_ABT}


def _matmul_launches(cases):
    """Launches of f32 products: cases of (op, M, N, R, bytes past alignment)."""
    rows = ll.run(f"""
result = []
for op, M, N, R, by in {cases!r}:
    m, k, n = {{"ab": (M, R, N), "atb": (R, M, N), "abt": (M, R, N)}}[op]
    code = {{"ab": L.MATMUL_AB, "atb": L.MATMUL_ATB, "abt": L.MATMUL_ABT}}[op]
    L.check(lib.prichs_matmul_f32(code, P + by, P + by, P + by, m, k, n, None))
    result += launches()
""")
    assert len(rows) == len(cases)
    return ll.as_launches(rows)


@pytest.mark.parametrize("op", sorted(OPS))
def test_matmul_short_reductions(op):
    # Where the pipelined tiles measured slower (up to 3.4 times) the short
    # kernel runs, and where it is the slower one they do.
    short = [(4096, 4096, 16, 0), (3000, 3001, 17, 0), (1341, 1245, 91, 0), (341, 3005, 1, 0),
             (16, 16, 16, 0), (1, 1, 1, 0), (2044, 2040, 8, 4)]
    tiles = [(2048, 1280, 1536, 0), (60, 84, 64, 0), (2000, 2000, 64, 0), (1024, 1024, 1024, 4),
             (101, 103, 151, 0), (16, 16, 512, 0)]
    got = _matmul_launches([(op, *c) for c in short + tiles])
    for c, x in zip(short + tiles, got):
        assert x.kernel.startswith("f32_matmul_short_kernel<") == (c in short), (c, x.kernel)
        if c in short:
            assert x.grid[0] == -(-c[0] // 64) * -(-c[1] // 64)


def test_matmul_largest_launches():
    # One output column (or row) of 2^27: 2^23 tiles of 16 x 16 with 512
    # threads would be 2^32 threads, more than a launch may have.
    for c, x in zip(cases := [("abt", 1 << 27, 1, 256, 0), ("abt", 1, 1 << 27, 256, 0),
                              ("abt", (1 << 27) - 64, 16, 512, 0), ("atb", 1 << 27, 4, 300, 0)],
                    _matmul_launches(cases)):
        assert x.grid[0] * x.block < 1 << 32, (c, x)
