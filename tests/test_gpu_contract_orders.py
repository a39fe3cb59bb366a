"""
GPU parity of contractions whose wires come in any order (operands permuted into scratch
memory first, products summed outside, the dense route) against plain numpy products, exact.
Ranks lie around the thresholds of the route rule (20 out bits, 18 and 22 bits of terms, 6 and
8 summed wires).
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(rng, batch, m, n, k, shuffle_out):
    b, lo, ro, s = range(batch), range(100, 100 + m), range(200, 200 + n), range(300, 300 + k)
    lw = [int(w) for w in rng.permutation([*b, *lo, *s])]
    rw = [int(w) for w in rng.permutation([*b, *ro, *s])]
    ow = [w for w in lw if w < 300] + [w for w in rw if 200 <= w < 300]
    if shuffle_out:
        ow = [int(w) for w in rng.permutation(ow)]
    return lw, rw, ow


def _expected(lhs, lw, rhs, rw, ow, mode):
    """Counts as a batched float32 product (at most 2^13 terms: exact)."""
    summed = [w for w in lw if w not in ow]
    both = [w for w in lw if w in rw and w in ow]
    lo, ro = [w for w in lw if w not in rw], [w for w in rw if w not in lw]
    a = lhs.transpose([lw.index(w) for w in both + lo + summed]).reshape(1 << len(both), 1 << len(lo), -1)
    b = rhs.transpose([rw.index(w) for w in both + summed + ro]).reshape(1 << len(both), 1 << len(summed), -1)
    c = np.matmul(a.astype(np.float32), b.astype(np.float32)).reshape((2,) * len(ow))
    have = both + lo + ro
    c = c.transpose([have.index(w) for w in ow])
    return ((c.astype(np.int64) % 256 != 0) if mode == "MOD256" else c > 0).astype(np.uint8)


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
@pytest.mark.parametrize(
    "batch,m,n,k",
    [
        (19, 0, 0, 0), (20, 0, 0, 0), (18, 1, 1, 0), (0, 10, 10, 0),  # products: below and at the threshold
        (15, 2, 3, 1), (15, 0, 5, 2), (21, 0, 0, 3), (4, 12, 4, 1), (0, 1, 19, 1),
        (14, 3, 3, 4), (11, 5, 4, 5), (14, 3, 4, 6), (15, 2, 3, 7),  # at most 128 terms outside
        (11, 2, 2, 8), (13, 1, 0, 9), (0, 3, 5, 14), (3, 2, 1, 13),  # popcount rows
        (2, 4, 5, 6), (0, 6, 6, 6), (4, 5, 5, 6), (2, 6, 7, 8), (0, 8, 7, 9), (1, 4, 9, 8), (0, 7, 7, 13),  # matrix cores
    ],
)
def test_wire_orders(batch, m, n, k, mode):
    from tensorsat_amd.rel import DeviceRel

    rng = np.random.default_rng([batch, m, n, k])
    for trial in range(3):
        lw, rw, ow = _case(rng, batch, m, n, k, trial == 2)
        dens = 0.5 if k < 8 or trial == 0 else 2.0 ** (-k / 2)  # a zero count is frequent, 256 is met at 0.5
        lhs = (rng.random((2,) * len(lw)) < dens).astype(np.uint8)
        rhs = (rng.random((2,) * len(rw)) < dens).astype(np.uint8)
        print(f"lhs {lw} rhs {rw} out {ow} {mode}", flush=True)
        with DeviceRel.mode_scope(mode):
            got = DeviceRel.contract2(DeviceRel(lhs), lw, DeviceRel(rhs), rw, ow).tensor
        np.testing.assert_array_equal(got, _expected(lhs, lw, rhs, rw, ow, mode))


@pytest.mark.parametrize("mode", ["GT0", "MOD256"])
def test_composition_of_ragged_extents(mode):
    from tensorsat_amd.rel import DeviceRel

    rng = np.random.default_rng(5)
    for r, i, c in ((1000, 700, 513), (61, 4097, 67), (3000, 65, 100)):
        a = (rng.random((r, i)) < i**-0.5).astype(np.uint8)
        b = (rng.random((i, c)) < i**-0.5).astype(np.uint8)
        cnt = (a.astype(np.float32) @ b.astype(np.float32)).astype(np.int64)
        print(f"{r} x {i} x {c} {mode}", flush=True)
        with DeviceRel.mode_scope(mode):
            got = DeviceRel.contract2(DeviceRel(a), [0, 1], DeviceRel(b), [1, 2], [0, 2]).tensor
        np.testing.assert_array_equal(got, (cnt % 256 != 0 if mode == "MOD256" else cnt > 0).astype(np.uint8))


def test_all_ones_rows_of_256_terms():
    """Exactly 256 terms everywhere: the count is 0 mod 256."""
    from tensorsat_amd.rel import DeviceRel

    for m, n in ((8, 8), (3, 11)):  # matrix cores, popcount rows
        a, b = np.ones((2,) * (m + 8), np.uint8), np.ones((2,) * (8 + n), np.uint8)
        lw, rw = [*range(300, 308), *range(m)], [*range(100, 100 + n), *range(300, 308)]
        ow = [*range(m), *range(100, 100 + n)]
        for mode, want in (("GT0", 1), ("MOD256", 0)):
            with DeviceRel.mode_scope(mode):
                got = DeviceRel.contract2(DeviceRel(a), lw, DeviceRel(b), rw, ow).tensor
            assert (got == want).all(), (m, n, mode)
