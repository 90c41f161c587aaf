"""Single permanents of bunched rows and columns (perm_one.hip) against the
double-double oracle within the call's own bound: lanes that hold a few
digits' states in one set of 64 or in several, the last one short; one to
eight waves, and several blocks; binomials in a byte and beyond; both sides
as the digits, both types of the products, and the allocation-free entry's
bits."""

import numpy as np
import pytest

from piquasso_amd import _capi

pytestmark = pytest.mark.gpu

CASES = [
    ([64], [64]),
    ([32, 32], [32, 32]),            # 1056 states of the lanes, binomials past a byte
    ([20, 20], [20, 20]),
    ([10, 11], [7, 7, 7]),           # radices 10 and 12
    ([8, 8, 8], [8, 8, 8]),
    ([8, 3, 11, 2, 1], [2, 1, 1, 1, 1, 1, 3, 1, 2, 3, 3, 1, 2, 2, 1]),
    ([21, 10, 6, 1], [2] * 19),
    ([5, 5, 4], [2] * 7),
    ([4, 4, 4, 1], [1] * 13),        # 125 states: two sets
    ([2] * 7, [7, 7]),               # five digits of three states, one of two
    ([12, 12], [1] * 24),
    ([3] * 8, [1] * 24),             # radix 4: 64 lanes of three digits, blocks
    ([2] * 9, [1] * 18),             # radix 3
    ([5] * 6, [3] * 10),             # sets of lanes in several blocks
    ([7] * 4, [4] * 7),
    ([1, 1, 1, 1, 1, 1, 1, 3, 4], [2] * 7),   # six binary lanes, mixed others
    ([1, 1, 1, 2, 4], [3, 3, 3]),    # two binary lanes
    ([1, 2, 3, 4, 5, 6], [1] * 21),
    ([4] * 9, [2] * 18),             # 1.6 million terms
]


def _call(entry, a, rows, cols, flags):
    out, dd = np.zeros(2), np.zeros(4)
    assert entry(a.ctypes.data_as(_capi._dp), len(rows), len(cols), len(cols), rows.ctypes.data_as(_capi._i32p),
                 cols.ctypes.data_as(_capi._i32p), flags, out.ctypes.data_as(_capi._dp),
                 dd.ctypes.data_as(_capi._dp)) == 0
    return complex(*out), dd, _capi.lib().pqp_last_error_bound()


@pytest.mark.parametrize("flags", [0, _capi.PQP_FLAG_AS_GIVEN, _capi.PQP_FLAG_FP32])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_oracle(gpu, oracle, case, flags):
    L = _capi.lib()
    for rows, cols in (CASES[case], CASES[case][::-1]):
        if flags == _capi.PQP_FLAG_AS_GIVEN and np.prod([float(r) + 1 for r in rows]) > 1e6:
            continue
        rng = np.random.default_rng(case)
        rows, cols = np.array(rows, dtype=np.int32), np.array(cols, dtype=np.int32)
        a = rng.standard_normal((len(rows), len(cols))) + 1j * rng.standard_normal((len(rows), len(cols)))
        a /= np.sqrt(2 * rows.sum())
        if flags == _capi.PQP_FLAG_FP32 and max(_largest(a, rows, cols), _largest(a.T, cols, rows)) > 3e38:
            continue  # terms beyond single precision
        print(f"bunched single {rows.tolist()} x {cols.tolist()} flags {flags}", flush=True)
        got, dd, bound = _call(L.pqp_permanent_c128, a, rows, cols, flags)
        # the oracle by the side with fewer terms
        if np.prod(rows + 1.0) <= np.prod(cols + 1.0):
            ref = oracle.perm_dd(a, rows, cols)
        else:
            ref = oracle.perm_dd(np.ascontiguousarray(a.T), cols, rows)
        if flags == _capi.PQP_FLAG_FP32:
            # the entries rounded to single precision: n of them in a product
            bound += rows.sum() * 2.0 ** -24 * _magnitude(oracle, a, rows, cols)
        assert np.isfinite(bound) and abs(got - ref) <= bound
        assert got == complex(dd[0] + dd[1], dd[2] + dd[3])
        again = _call(L.pqp_permanent_c128_noalloc, a, rows, cols, flags)
        assert again[0] == got and np.array_equal(again[1], dd)


def _largest(a, rows, cols):
    """A bound on the magnitude of every term with `rows` as the digits."""
    return float(np.prod((np.abs(a).T @ rows) ** cols))


def _magnitude(oracle, a, rows, cols):
    """The sum of the expanded permanent's products in magnitude."""
    b = np.abs(a).astype(complex)
    if np.prod(rows + 1.0) <= np.prod(cols + 1.0):
        return oracle.perm_dd(b, rows, cols).real
    return oracle.perm_dd(np.ascontiguousarray(b.T), cols, rows).real
