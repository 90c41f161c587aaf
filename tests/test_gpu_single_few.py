"""Single permanents of up to 12 particles in distinct modes, whose kernels
take fewer arguments, and the first that do not, against the oracle within
the call's own bound; and the allocation-free entry's bits."""

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd import _capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", range(1, 15))
def test_few_particles(gpu, oracle, n, dtype):
    rng = np.random.default_rng(n)
    m = n + 3
    a = ((rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))) / np.sqrt(2 * n)).astype(dtype)
    rows, cols = np.zeros(m, dtype=np.int32), np.zeros(m, dtype=np.int32)
    rows[rng.permutation(m)[:n]] = 1
    cols[rng.permutation(m)[:n]] = 1
    print(f"few {n} {dtype.__name__}", flush=True)
    got = complex(pa.permanent(a, rows, cols))
    bound = _capi.lib().pqp_last_error_bound()
    assert abs(got - oracle.perm_dd(a.astype(np.complex128), rows, cols)) <= bound
    if dtype is np.complex128:
        out = np.zeros(2)
        assert _capi.lib().pqp_permanent_c128_noalloc(
            a.ctypes.data_as(_capi._dp), m, m, m, rows.ctypes.data_as(_capi._i32p),
            cols.ctypes.data_as(_capi._i32p), 0, out.ctypes.data_as(_capi._dp), None) == 0
        assert complex(*out) == got
