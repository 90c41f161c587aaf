"""The wave-planned exact integer sweep (perm_int.hip) over its dispatch:
every column group (12, 8, 4, 2, 1, from the entries' size), one to eight
moduli, each padded width with full and ragged columns, rows that leave no
binary digit, and sweeps of one wave up to several states and chunks a lane;
exact against the integer oracle or closed forms."""

import math

import numpy as np
import pytest

import piquasso_amd as pa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 12, 15, 16, 17, 20])
@pytest.mark.parametrize("entry", [1, 3, 2**7, 2**19, 2**30, 2**43])
def test_groups_and_moduli_match_the_oracle(gpu, oracle, n, entry):
    """Column sums of n entries: 1 gives groups of 12, 2^43 single columns;
    the permanent's bound (20 x 2^47 = 2^940 at most) ends the range."""
    rng = np.random.default_rng(1000 * n + entry.bit_length())
    a = rng.integers(-entry, entry + 1, size=(n, n), dtype=np.int64)
    one = np.ones(n, dtype=int)
    print(f"exact n={n} entries to {entry}", flush=True)
    rows = np.abs(a).sum(axis=1)
    cols = np.abs(a).sum(axis=0)
    log2_perm = sum(math.log2(r) if r else 0 for r in rows.tolist())
    if cols.max() > 2**48 or math.ceil((log2_perm + 2.0) / 48.99) > 8:
        with pytest.raises(ValueError):
            pa.permanent_exact(a, one, one)
        return
    assert pa.permanent_exact(a, one, one) == oracle.perm_int_exact(a, one, one)


@pytest.mark.parametrize("rows, cols", [
    ([2, 2, 2], [3, 3]), ([3, 3, 3, 3], [12]), ([5], [1, 1, 1, 1, 1]), ([2] * 8, [1] * 16),
    ([4, 4, 4, 4], [2] * 8), ([0, 7, 0, 1], [0, 2, 6]), ([1, 3, 2, 1, 5], [4, 4, 4]),
    ([13, 1], [2] * 7), ([6, 6, 6], [9, 9]),
])
def test_multiplicities_match_the_oracle(gpu, oracle, rows, cols):
    rng = np.random.default_rng(sum(rows) + len(cols))
    a = rng.integers(-4, 5, size=(len(rows), len(cols)), dtype=np.int64)
    print(f"exact rows {rows} cols {cols}", flush=True)
    assert pa.permanent_exact(a, rows, cols) == oracle.perm_int_exact(a, rows, cols)


@pytest.mark.parametrize("n, k", [(25, 3), (26, 5), (31, 2), (33, 40), (40, 50), (41, 41), (56, 56), (64, 64)])
def test_wide_matrices_of_repeated_rows(gpu, n, k):
    """k copies of one all-ones row and n - k of another row x: the permanent
    is n! prod over choices, sum over which columns the x rows take."""
    # x = (2, .., 2) gives n! 2^(n - k); rows of multiplicity keep the sweep short
    rows = [min(k, n), n - min(k, n)] if k < n else [n]
    a = np.ones((len(rows), n), dtype=np.int64)
    if len(rows) == 2:
        a[1] = 2
    print(f"exact wide n={n}", flush=True)
    log2_perm = n * math.log2(n) + (n - min(k, n))
    weight = math.log2(math.comb(rows[0], rows[0] // 2)) + \
        (math.log2(math.comb(rows[1], rows[1] // 2)) if len(rows) == 2 else 0)
    if weight > 52 or math.ceil((log2_perm + 2) / 48.99) > 8:
        with pytest.raises(ValueError):
            pa.permanent_exact(a, rows, [1] * n)
    else:
        assert pa.permanent_exact(a, rows, [1] * n) == math.factorial(n) * 2 ** (n - min(k, n))
