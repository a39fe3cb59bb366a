"""The C-ABI libraries load on the CPU and export every symbol their headers declare."""

import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


def _declared(header: str) -> set[str]:
    text = (ROOT / "include" / header).read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = set(re.findall(r"^\s*(?:const\s+)?[A-Za-z_][A-Za-z0-9_\s\*]*?\b(ts[a-z]*_[a-z0-9_]+)\s*\(", text, flags=re.M))
    return names


def test_headers_declare_expected_entry_points():
    d = _declared("tensorsat_amd.h")
    assert {"ts_contract2", "ts_rewire", "ts_batch_run", "ts_program_count"} <= d
    assert {"tsp_greedy", "tsp_hyper", "tsp_tree_cost", "tsp_slice"} <= _declared("tensorsat_plan.h")
    assert {"tsc_compile", "tsc_sat_batch", "tsp_elim"} <= _declared("tensorsat_prog.h")


def test_planner_library_exports_everything():
    lib = ctypes.CDLL(str(ROOT / "tensorsat_amd" / "libtsplan.so"))
    for name in _declared("tensorsat_plan.h") | _declared("tensorsat_prog.h"):
        assert hasattr(lib, name), name


def test_hip_library_exports_everything():
    path = ROOT / "tensorsat_amd" / "libtensorsat_amd.so"
    if not path.exists():
        pytest.fail("libtensorsat_amd.so is not built (python -m tensorsat_amd.build)")
    from tensorsat_amd import _native as N

    lib = N.load()  # no GPU call
    declared = _declared("tensorsat_amd.h")
    for name in declared:
        assert hasattr(lib, name), name
    assert set(N.EXPORTS) == declared
    assert lib.ts_version().startswith(b"tensorsat_amd")


def test_dense_tile_table_host_side():
    """The dense tile table is host state (no GPU needed): set, read back, reset to the
    built-in rule, bad arguments."""
    import ctypes

    from tensorsat_amd import _native as N

    L = N.load()

    def tile_of(*shape):
        t = ctypes.c_int32(0)
        assert L.ts_dense_tile_of(*shape, ctypes.byref(t)) == 0
        return t.value

    assert tile_of(8, 8, 0, 8) == 4 and tile_of(5, 9, 0, 8) == 1 and tile_of(10, 12, 0, 8) == 6  # built-in rule
    assert L.ts_dense_tiles(8, 8, 0, 8, 2) == 0
    assert tile_of(8, 8, 0, 8) == 2
    assert L.ts_dense_tiles(8, 8, 0, 8, 0) == 0
    assert tile_of(8, 8, 0, 8) == 4
    assert L.ts_dense_tiles(8, 8, 0, 8, 7) == N.TS_EINVAL
    assert L.ts_dense_tiles(-1, 8, 0, 8, 1) == N.TS_EINVAL
    assert L.ts_dense_tile_of(8, 8, 0, 28, None) == N.TS_EINVAL


def test_weight_gradient_scratch_sizes():
    """Host arithmetic only: no columns or rows need no scratch, a multiple of 64 KiB per tile
    otherwise, sizes out of range refused."""
    from tensorsat_amd import _native as N

    L = N.load()
    need = N.i64(-1)
    for m, rows, blocks in ((0, 0, 0), (0, 1000, 0), (1, 0, 1), (128, 1, 1), (132, 257, 4), (32768, 10**6, 256)):
        assert L.ts_gnn_wgrad_scratch(m, rows, ctypes.byref(need)) == 0
        assert need.value == blocks * 128 * 128 * 4, (m, rows)
    for m, rows in ((-1, 5), (5, -1), (32769, 5)):
        assert L.ts_gnn_wgrad_scratch(m, rows, ctypes.byref(need)) == N.TS_EINVAL
    assert L.ts_gnn_wgrad_scratch(4, 4, None) == N.TS_EINVAL


def _contract_scratch(lhs, rhs, out):
    """Scratch bytes that ts_contract2 can use for these wires (0: it copies no operand)."""
    from tensorsat_amd import _native as N

    need = N.i64(-1)
    args = [x for ws in (lhs, rhs, out) for x in (len(ws), N.i32arr(ws))]
    assert N.load().ts_contract2_scratch(*args, ctypes.byref(need)) == 0
    return need.value


@pytest.mark.parametrize("own", [0, 1, 3])
@pytest.mark.parametrize("out_bits", [20, 22])
def test_rows_in_place_are_not_copied(out_bits, own):
    """Contractions whose summed wires are innermost in both operands: rows of 16 bytes or more,
    and shorter ones whose two last out wires are each operand's last kept ones."""
    shared = out_bits - 2 * own
    kept_l, kept_r = [*range(shared)], [*range(shared)]
    kept_l[shared // 2 : shared // 2] = range(100, 100 + own)
    kept_r[shared // 3 : shared // 3] = range(200, 200 + own)
    out = [*range(100, 100 + own), *range(200, 200 + own), *range(shared)]
    for k in range(8):
        if max(len(kept_l), len(kept_r)) + k > 27 or (k >= 6 and own >= 4):
            continue
        summed = [*range(300, 300 + k)]
        for swap in (False, True):  # the wires above the two last ones in any order
            a, b = list(kept_l), list(kept_r)
            if swap:
                a[0], a[3], b[1], b[4] = a[3], a[0], b[4], b[1]
            assert _contract_scratch(a + summed, b + summed, out) == 0, (k, swap)
        if 4 <= k:  # any order of the kept wires
            assert _contract_scratch(kept_l[::-1] + summed, kept_r + summed, out) == 0, k
        elif own == 0:  # reversed: copied where that costs at most 4 bytes per output
            size = 2 ** (out_bits + k)
            assert _contract_scratch(kept_l[::-1] + summed, kept_r[::-1] + summed, out) == (2 * size if k < 2 else 0)


def test_small_products_keep_their_gather():
    """Summed wires outermost in both operands: which products copy them innermost first."""
    def bytes_for(batch, m, n, k):
        b, s = [*range(batch)], [*range(300, 300 + k)]
        l, r = [*range(100, 100 + m)], [*range(200, 200 + n)]
        return _contract_scratch(s + b + l, s + b + r, b + l + r)

    moved = lambda batch, m, n, k: 2 ** (batch + m + k) + 2 ** (batch + n + k)
    # matrix cores: not for 2^10 or fewer outputs of 256 or more terms, 2^11 of less than 2^16
    for shape, copies in (((0, 4, 4, 12), False), ((0, 5, 5, 10), False), ((2, 4, 4, 8), False), ((0, 5, 6, 12), False),
                          ((0, 5, 6, 16), True), ((0, 6, 6, 8), True), ((4, 4, 4, 6), True), ((0, 6, 6, 6), True)):
        assert bytes_for(*shape) == (moved(*shape) if copies else 0), shape
    # a workgroup per output: long sums, or half a byte to copy per product and 2^23 of them
    for shape, copies in (((4, 3, 3, 12), False), ((8, 0, 1, 13), False), ((12, 0, 0, 11), False), ((2, 2, 5, 14), True),
                          ((0, 2, 2, 16), False), ((1, 2, 3, 16), True), ((2, 0, 2, 18), True)):
        assert bytes_for(*shape) == (moved(*shape) if copies else 0), shape
    # rows of the step engine
    for shape, copies in (((18, 0, 0, 4), False), ((14, 3, 1, 4), False), ((8, 3, 8, 4), True), ((16, 1, 0, 5), False),
                          ((16, 2, 1, 5), True), ((18, 0, 0, 7), False), ((16, 1, 1, 7), True), ((10, 0, 3, 11), True)):
        assert bytes_for(*shape) == (moved(*shape) if copies else 0), shape


def test_no_scratch_below_the_lines_that_callers_ask_from():
    """The native rule and the bits from which it is asked agree: random wires just below."""
    import random

    from tensorsat_amd import _native as N

    rng, asked = random.Random(1), 0
    for _ in range(4000):
        batch, m, n, k = rng.randint(0, 19), rng.randint(0, 10), rng.randint(0, 10), rng.randint(0, 16)
        out, products = batch + m + n, batch + m + n + k
        if batch + max(m, n) + k > 27 or not 14 <= products <= 24:
            continue
        lhs = [*range(batch), *range(100, 100 + m), *range(300, 300 + k)]
        rhs = [*range(batch), *range(200, 200 + n), *range(300, 300 + k)]
        res = [*range(batch), *range(100, 100 + m), *range(200, 200 + n)]
        for ws in (lhs, rhs, res):
            rng.shuffle(ws)
        ask = products >= N.SCRATCH_BITS or out >= N.SCRATCH_OUT_BITS or (products >= N.SCRATCH_DENSE_BITS and k >= 6)
        asked += ask
        assert ask or _contract_scratch(lhs, rhs, res) == 0, (lhs, rhs, res)
    assert 200 < asked < 3000
