"""Which kernels the library launches, on the CPU (tests/launch_log.py): the
dispatch rules on sizes, types and alignment."""
import re

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
             (101, 103, 151, 0), (16, 16, 512, 0), (936, 1140, 613, 0), (3645, 379, 601, 0),
             (1721, 826, 662, 0)]
    got = _matmul_launches([(op, *c) for c in short + tiles])
    for c, x in zip(short + tiles, got):
        assert x.kernel.startswith("f32_matmul_short_kernel<") == (c in short), (c, x.kernel)
        if c in short:
            assert x.grid[0] == -(-c[0] // 64) * -(-c[1] // 64)


def _matmul_kernel(x):
    """Tile shape / elements per load of an f32 product's launch, or "short"."""
    if x.kernel.startswith("f32_matmul_short_kernel<"):
        return "short"
    t = re.findall(r"Tile<(\d+), (\d+),[^>]*, (\d)>", x.kernel)
    return f"{t[0][0]}x{t[0][1]}{'+halves' if t[0] != t[1] else ''}/{t[0][2]}"


def test_cases_of_the_matmul_tiles():
    # What the GPU test of the products' kernels launches; together every
    # kernel with either kind of loads it has.
    from tests.test_gpu_matmul import MATMUL_TILES

    cases = [(op, M, N, R, by) for M, N, R, _, _ in MATMUL_TILES for by in (0, 4)
             for op in sorted(OPS)]
    want = [k for *_, k0, k1 in MATMUL_TILES for k in (k0, k1) for _ in OPS]
    got = [_matmul_kernel(x) for x in _matmul_launches(cases)]
    assert got == want, [(c, g, w) for c, g, w in zip(cases, got, want) if g != w]
    shapes = {f"{t}/{w}" for t in ("128x128", "64x64", "32x64", "32x32", "16x16") for w in (1, 4)}
    assert shapes | {"64x64+halves/4", "short"} == set(want)


def test_matmul_largest_launches():
    # One output column (or row) of 2^27: 2^23 tiles of 16 x 16 with 512
    # threads would be 2^32 threads, more than a launch may have.
    for c, x in zip(cases := [("abt", 1 << 27, 1, 256, 0), ("abt", 1, 1 << 27, 256, 0),
                              ("abt", (1 << 27) - 64, 16, 512, 0), ("atb", 1 << 27, 4, 300, 0)],
                    _matmul_launches(cases)):
        assert x.grid[0] * x.block < 1 << 32, (c, x)


def test_decode_launch_workgroups_per_cu():
    # The router's and the GEMM's LDS share one buffer: three workgroups of
    # the decode launch fit a CU's 160 KiB, or two where a third place would
    # only leave a nearly empty round behind (d = 1024, f = 2816: 792 + 1
    # workgroups on 768 places).
    cases = [(256, 4096, 32), (512, 2048, 8), (1536, 1280, 1), (1536, 1280, 32), (1024, 4096, 1),
             (1024, 2816, 1)]
    rows = ll.run(f"""
result = []
for d, f, T in {cases!r}:
    h = engine(d, f, 8, 2, L.DTYPE_BF16, 32)
    L.check(lib.prichs_moe_engine_forward(h, P, T, None, 0, P, L.DTYPE_BF16, None))
    result += launches()[:1]
    L.check(lib.prichs_moe_engine_destroy(h))
""")
    static = ll.static_lds()
    for c, x in zip(cases, ll.as_launches(rows)):
        assert x.kernel.startswith("skinny::decode_gate_up_router_kernel<"), x.kernel
        per_cu = 160 * 1024 // (x.lds + static[x.symbol])
        if c[1] == 1280:  # one round on two places per CU
            assert x.grid[0] <= 512 and per_cu >= 2, (c, x.lds, static[x.symbol])
        else:
            assert per_cu == (2 if c[1] == 2816 else 3), (c, x.lds, static[x.symbol])
        assert x.lds + static[x.symbol] <= 64 * 1024


def _tiles(x):
    """(rows, columns) of the tiles of a grouped or dense bf16 GEMM launch."""
    m = re.match(r"bf16_gemm_kernel<Bf16Cfg<(\d+), (\d+)", x.kernel)
    return (int(m[1]), int(m[2])) if m else None


def _forward_gemms(cases, **env):
    """Launches of the gate/up and down GEMMs of bf16 engine forwards: cases of
    (E, k, d, f, T)."""
    rows = ll.run(f"""
result = []
for E, k, d, f, T in {cases!r}:
    h = engine(d, f, E, k, L.DTYPE_BF16, T)
    L.check(lib.prichs_moe_engine_forward(h, P, T, None, 0, P, L.DTYPE_BF16, None))
    result += [x for x in launches() if "gemm_kernel" in x[0]]
    L.check(lib.prichs_moe_engine_destroy(h))
""", **env)
    rows = ll.as_launches(rows)
    assert len(rows) == 2 * len(cases)
    return list(zip(rows[::2], rows[1::2]))


def test_grouped_tiles_near_whole_rounds():
    # Batches whose groups sit near a multiple of a tile's rows, where the
    # faster tiles (measured with random routing) were not taken: the larger
    # ones of gate/up (first three) and down.
    cases = [(16, 2, 1536, 1280, 3800), (4, 2, 1536, 1280, 1024), (8, 2, 1536, 640, 2048),
             (8, 2, 1536, 1280, 6860)]
    for c, g in zip(cases, _forward_gemms(cases)):
        assert _tiles(g[c[-1] == 6860]) == (256, 256), (c, g)
    # Few rows keep the smaller tiles.
    cases = [(8, 2, 1536, 1280, 333), (8, 2, 1536, 1280, 128), (8, 2, 1536, 1280, 8192)]
    want = [((128, 256), (128, 256)), ((64, 128), (64, 128)), ((256, 256), (256, 256))]
    assert [tuple(map(_tiles, g)) for g in _forward_gemms(cases)] == want


def test_gemm_cu_cap():
    # PRICHS_GEMM_MAX_CUS bounds the workgroups of every persistent bf16
    # launch, of 64 x 128 tiles too, two of which fit a CU.
    cases = [(8, 2, 512, 512, T) for T in (100, 300, 1000, 4096)]
    tiles = set()
    for cap in (48, 512):
        for g in _forward_gemms(cases, PRICHS_GEMM_MAX_CUS=str(cap)):
            for x in g:
                tiles.add((cap, _tiles(x)))
                assert x.grid[0] <= (48 if cap == 48 else 512), x
    assert (48, (64, 128)) in tiles and (512, (64, 128)) in tiles, tiles


def test_lds_limits_on_every_device():
    # A kernel's limit on dynamic LDS is the device's: every launch with more
    # than 64 KiB follows a raise of its kernel's limit on that device.
    rows = ll.run("""
for dev in (0, 1, 0, 2):
    hip().hipSetDevice(dev)
    for M in (64, 1000, 20000):
        L.check(lib.prichs_gemm(P, 512, M, 512, P, 512, P, 512, L.DTYPE_BF16, None))
    for E, d in ((8, 4096), (64, 512), (8, 1024)):
        L.check(lib.prichs_router_topk(P, L.DTYPE_F32, P, P, None, 0, 5000, d, E, 2, P, P, P, P, None))
    h = engine(256, 256, 8, 2, L.DTYPE_BF16, 6000, backward=True)
    g = L.MoEGrads(P, P, P, P, 1 << 20, 0)
    for T in (100, 400, 6000):
        L.check(lib.prichs_moe_engine_forward(h, P, T, None, 0, P, L.DTYPE_BF16, None))
        L.check(lib.prichs_moe_engine_backward(h, P, P, T, P, L.DTYPE_BF16, C.byref(g), 2, None))
result = raw_events()
""")
    limit, seen = {}, set()
    for r in rows:
        if r[0] == "attribute":
            limit[r[1], r[3]] = int(r[2])
        elif int(r[7]) > 64 * 1024:
            name, lds, dev = r[1], int(r[7]), r[8]
            assert limit.get((name, dev), 0) >= lds, (name, lds, dev)
            seen.add((name, dev))
    assert {dev for _, dev in seen} == {"0", "1", "2"}
    kinds = {n.split("<")[0].split("::")[-1] for n, _ in seen}
    assert {"bf16_gemm_kernel", "wgrad_bf16_kernel", "wgrad_bf16_short_kernel",
            "router_topk_quad_kernel"} <= kinds, kinds


def _rounds(x, counts, Np):
    """(tile, whole rounds, last round in halves) of a grouped bf16 launch over
    groups of `counts` rows and Np packed columns."""
    bm, bn = _tiles(x)
    tiles = sum(-(-c // bm) for c in counts) * (Np // bn)
    whole, tail = divmod(tiles, x.grid[0])
    cfgs = re.findall(r"Bf16Cfg<[^>]*>", x.kernel)
    return (bm, bn), whole, cfgs[0] != cfgs[1] and 0 < 2 * tail <= x.grid[0]


def test_cases_of_the_smaller_tiles():
    # What the GPU tests of the 128 x 256 and 64 x 128 tiles launch, and that
    # their reference launches take 256 x 256 tiles.
    from tests.test_gpu_moe import MID_TILES, REF_ROWS

    calls = []
    for d, f, counts, _, _ in MID_TILES:
        calls += [(d, f, len(counts), sum(counts)), (d, f, len(counts) + 1, REF_ROWS[d])]
    rows = ll.as_launches(ll.run(f"""
result = []
for d, f, G, rows in {calls!r}:
    L.check(lib.prichs_grouped_gate_up_swiglu(P, P, P, G, rows, P, d, f, L.DTYPE_BF16, P, None))
    L.check(lib.prichs_grouped_down(P, P, G, rows, P, d, f, L.DTYPE_BF16, P, None))
    result += launches()
"""))
    assert len(rows) == 4 * len(MID_TILES)
    for (d, f, counts, gu, dn), (a, b, ra, rb) in zip(MID_TILES, zip(*[iter(rows)] * 4)):
        np_gu, np_dn = -(-2 * f // 256) * 256, -(-d // 256) * 256
        assert _rounds(a, counts, np_gu) == gu, (d, f, counts, a)
        assert _rounds(b, counts, np_dn) == dn, (d, f, counts, b)
        assert _tiles(ra) == _tiles(rb) == (256, 256), (d, f, counts)


def test_cases_of_the_dense_tiles():
    from tests.test_gpu_block import DENSE_TILES

    rows = ll.as_launches(ll.run(f"""
result = []
for M, N in {sorted(DENSE_TILES)!r}:
    L.check(lib.prichs_gemm(P, 1536, M, 1536, P, N, P, N, L.DTYPE_BF16, None))
    result += launches()
"""))
    got = {}
    for (M, N), x in zip(sorted(DENSE_TILES), rows):
        tile, _, halves = _rounds(x, [M], -(-N // 256) * 256)
        got[M, N] = (tile, halves)
    assert got == DENSE_TILES


def test_cases_of_the_f32_and_weight_gradient_kernels():
    # The tiles and kernels that the GPU tests of the f32 grouped GEMMs and of
    # the weight gradients say they take (gate/up and down; dW_down and
    # dW_gate/up).
    got = ll.run("""
result = []
for d, f, G, rows in [(48, 1008, 2, 1700), (2000, 48, 2, 1700), (80, 496, 2, 850), (112, 80, 6, 105)]:
    L.check(lib.prichs_grouped_gate_up_swiglu(P, P, P, G, rows, P, d, f, L.DTYPE_F32, P, None))
    L.check(lib.prichs_grouped_down(P, P, G, rows, P, d, f, L.DTYPE_F32, P, None))
    result.append([x[0] for x in launches()])
for T, d, f, E, k, dt in [(40, 1536, 1296, 3, 2, 0), (37, 656, 624, 3, 2, 0), (512, 256, 128, 8, 2, 0),
                          (130, 448, 128, 2, 1, 1), (2600, 1536, 1280, 8, 2, 1),
                          (3000, 256, 128, 4, 2, 1)]:
    h = engine(d, f, E, k, dt, T, backward=True)
    g = L.MoEGrads(P, P, P, P, d * f, 0)
    L.check(lib.prichs_moe_engine_forward(h, P, T, None, 0, P, 0, None))
    launches()
    L.check(lib.prichs_moe_engine_backward(h, P, P, T, P, 0, C.byref(g), 2, None))
    result.append([x[0] for x in launches() if x[0].startswith("wgrad_") and "reduce" not in x[0]])
    L.check(lib.prichs_moe_engine_destroy(h))
""")

    def short(name):
        t = re.search(r"Tile<(\d+), (\d+)", name)
        return f"{t[1]}x{t[2]}" if t else name.split("<")[0]

    assert [[short(n) for n in pair] for pair in got] == [
        ["128x128", "32x64"], ["32x64", "128x128"], ["64x64", "32x64"], ["32x64", "32x64"],
        ["128x128", "128x128"], ["64x64", "64x64"], ["32x64", "32x64"],
        ["wgrad_bf16_short_kernel"] * 2, ["wgrad_bf16_kernel", "wgrad_bf16_short_kernel"],
        ["wgrad_bf16_kernel"] * 2]
