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
