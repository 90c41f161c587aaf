"""The last row of the layer path folds the links of a coefficient in
double-double: with diagonal matrices that are 1 but for the last row, every
link's sum is exact, and so is their sum, whatever cancels in whatever order."""

import itertools
import math

import numpy as np
import pytest

import piquasso_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("last", [(1.0, 2.0 ** -60, -1.0), (1.0, 2.0 ** -60, -1.0, 2.0 ** -59)])
def test_links_cancel_exactly(gpu, last):
    n = len(last)
    print(f"poly fold n={n}", flush=True)
    for order in itertools.permutations(last):
        bm = np.array([np.diag([1.0] * (n - 1) + [v]) for v in order], dtype=complex)
        got = pa.perm_poly_coefficients(np.zeros((n, n), complex), bm, np.ones((1, n), dtype=np.int32))
        # the other rows take the other variables in any order
        assert got[0] == math.factorial(n - 1) * math.fsum(last)
