"""The row-by-row layer path of the matrix-polynomial permanent
(poly_layer_kernel, poly_last_kernel) where it can go wrong: the smallest
orders, groups narrower and wider than a wave, the widest order (several
column blocks per layer), degrees capped below n, the first sizes that stay
on the subset sum, and a plan tried for a call whose rows turn out to be
others."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _case(n, m, top, count, seed):
    rng = np.random.default_rng(seed)
    b0 = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(n)
    bm = (rng.standard_normal((m, n, n)) + 1j * rng.standard_normal((m, n, n))) / np.sqrt(n)
    exps = np.zeros((count, m), dtype=np.int32)
    for e in exps[1:]:
        for v in rng.integers(0, m, size=rng.integers(0, top + 1)) if m else ():
            e[v] += 1
    return b0, bm, exps


def _check(pa, oracle, b0, bm, exps):
    n, m = len(b0), len(bm)
    got = pa.perm_poly_coefficients(b0, bm, exps)
    ref, _ = oracle.perm_poly_dd(b0, bm, exps)
    # the same sums of magnitudes; layer i adds (m + 1) i products per value
    mag, _ = oracle.perm_poly_dd(np.abs(b0).astype(complex), np.abs(bm).astype(complex), exps)
    steps = sum((m + 1) * i + 4 for i in range(1, n + 1))
    assert np.all(np.abs(got - ref) <= steps * EPS * np.abs(mag) + 1e-300)


# (order, variables, largest total degree)
@pytest.mark.parametrize("n, m, top", [
    (1, 1, 1), (1, 0, 0), (2, 3, 2), (3, 2, 2), (4, 6, 4),
    (7, 3, 7), (8, 2, 3), (9, 3, 9), (10, 4, 6), (11, 2, 11),
    (12, 2, 12), (12, 3, 4), (12, 84, 2),   # the widest layers; the most coefficients kept in LDS
    (12, 85, 2), (13, 2, 6),                # past the layer path: the subset sum
])
def test_layers_match_oracle(gpu, oracle, n, m, top):
    import piquasso_amd as pa

    print(f"poly layers n={n} vars={m} degree<={top}", flush=True)
    _check(pa, oracle, *_case(n, m, top, 9, 1000 * n + m))


def test_other_rows_of_the_same_sizes(gpu, oracle):
    """Calls of equal sizes with other exponent rows: the kept plan is tried
    first and must not leave its answer."""
    import piquasso_amd as pa

    b0, bm, e1 = _case(6, 3, 6, 9, 5)
    e2 = np.ascontiguousarray(e1[:, ::-1])
    e3 = e1.copy()
    e3[4] = (0, 0, 7)  # degree above n: coefficient 0
    for e in (e1, e2, e1, e3, e3, e1):
        _check(pa, oracle, b0, bm, e)
    bad = e1.copy()
    bad[2, 1] = -1
    with pytest.raises(ValueError):
        pa.perm_poly_coefficients(b0, bm, bad)
    _check(pa, oracle, b0, bm, e1)
