"""The matrix-polynomial permanent on both sides of the rule that leaves a few
outputs of 6 and 7 particles to the subset sum, and the orders beside them,
one call after another."""

import numpy as np
import pytest

import piquasso_amd as pa
from test_gpu_lossy_pd import _tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, m", [(5, 3), (6, 1), (6, 4), (7, 2), (7, 10), (8, 3)])
def test_few_outputs_match_oracle(gpu, oracle, n, m):
    rng = np.random.default_rng(10 * n + m)
    b0 = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(n)
    bm = (rng.standard_normal((m, n, n)) + 1j * rng.standard_normal((m, n, n))) / np.sqrt(n)
    for count in (1, 4, 5, 64, 65, 2, 0, 65):
        e = np.array([np.bincount(rng.integers(0, m, rng.integers(0, n + 1)), minlength=m) for _ in range(count)],
                     dtype=np.int32).reshape(count, m)
        print(f"poly few n={n} vars={m} outputs={count}", flush=True)
        got = pa.perm_poly_coefficients(b0, bm, e)
        ref, scale = oracle.perm_poly_dd(b0, bm, e)
        assert np.all(np.abs(got - ref) <= _tol(n, scale))
    none = np.full((3, m), n, dtype=np.int32)  # degrees above n (at m = 1: the one output)
    assert np.all(np.isfinite(pa.perm_poly_coefficients(b0, bm, none)))
