"""Single permanents without tables (perm_one.hip) against the double-double
oracle: the edges of the lane, inner and other digits (binary and larger
radices, fewer than 64 states, one block and several), of the widths, and
both types of the products.  The tolerance is the call's own bound,
4 (n + 2) u times the sum of the terms' magnitudes."""

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd import _capi

pytestmark = pytest.mark.gpu

# rows, columns (multiplicities)
CASES = [
    ([1], [1]),
    ([3], [1, 2]),
    ([1, 1], [2]),
    ([1] * 6, [1] * 6),              # five binary digits: 32 lanes
    ([1] * 7, [1] * 7),              # six: one state of the others
    ([1] * 8, [1] * 8),
    ([0, 2, 1, 0, 2, 2], [1, 0, 3, 1, 2]),
    ([2] * 5, [1] * 10),             # 54 lanes
    ([3] * 4, [4, 4, 4]),            # 48 lanes
    ([7, 7], [2] * 7),               # 56 lanes, the other digits none
    ([12, 9], [3] * 7),              # larger than 64 states a digit pair
    ([1] * 12, [1] * 12),            # 2048 terms: one block
    ([1] * 13, [1] * 13),            # several blocks
    ([2] * 8, [1] * 16),             # radices 3, inner ones too
    ([1, 1, 2, 2, 3, 3, 4], [1] * 16),
    ([4, 4, 4, 4], [1, 1, 2, 3, 4, 5]),
    ([1] * 16 + [2], [1] * 18),      # binary lanes and inner digits, four waves a block
    ([1, 2, 3, 4, 5, 1], [16]),      # one column
    ([1] * 20, [1] * 16 + [4]),
]


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_against_oracle(gpu, oracle, case, dtype):
    rows, cols = CASES[case]
    rng = np.random.default_rng(case)
    a = rng.standard_normal((len(rows), len(cols))) + 1j * rng.standard_normal((len(rows), len(cols)))
    a = (a / np.sqrt(2 * sum(rows))).astype(dtype)
    print(f"single {rows} x {cols} {dtype.__name__}", flush=True)
    got = complex(pa.permanent(a, rows, cols))
    bound = _capi.lib().pqp_last_error_bound()
    ref = oracle.perm_dd(a.astype(np.complex128), rows, cols)
    assert np.isfinite(bound) and abs(got - ref) <= bound


@pytest.mark.parametrize("flag", ["PQP_FLAG_EXPAND_COLS", "PQP_FLAG_KEEP_COLS", "PQP_FLAG_AS_GIVEN"])
def test_flags_and_repeats(gpu, oracle, flag):
    """The columns' form and the orientation change the sum, not its value;
    calls with other occupations in between do not change its bits."""
    rng = np.random.default_rng(5)
    a = rng.standard_normal((4, 9)) + 1j * rng.standard_normal((4, 9))
    rows = np.array([4, 1, 3, 4], dtype=np.int32)
    cols = np.array([1, 1, 2, 0, 2, 1, 3, 1, 1], dtype=np.int32)
    L = _capi.lib()

    def call(f):
        out, dd = np.zeros(2), np.zeros(4)
        assert L.pqp_permanent_c128(a.ctypes.data_as(_capi._dp), 4, 9, 9, rows.ctypes.data_as(_capi._i32p),
                                    cols.ctypes.data_as(_capi._i32p), f, out.ctypes.data_as(_capi._dp),
                                    dd.ctypes.data_as(_capi._dp)) == 0
        return complex(*out), dd, L.pqp_last_error_bound()

    got, dd, bound = call(getattr(_capi, flag))
    assert abs(got - oracle.perm_dd(a, rows, cols)) <= bound
    assert got == complex(dd[0] + dd[1], dd[2] + dd[3])
    pa.permanent(np.ones((15, 15)) * 0.5j, np.ones(15, int), np.ones(15, int))
    assert np.array_equal(call(getattr(_capi, flag))[1], dd)
