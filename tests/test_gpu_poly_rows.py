"""Calls of the matrix-polynomial permanent with other exponent rows of the
sizes of the call before: no evaluation is spent on the kept plan where its
rows differ at once, and lists that differ late get their own answer."""

import time

import numpy as np
import pytest

import piquasso_amd as pa

pytestmark = pytest.mark.gpu


def _case(n, m, seed):
    rng = np.random.default_rng(seed)
    b0 = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(n)
    bm = (rng.standard_normal((m, n, n)) + 1j * rng.standard_normal((m, n, n))) / np.sqrt(n)
    return b0, bm


def test_other_rows_cost_no_evaluation_of_the_kept_plan(gpu):
    # 65535 subsets of 16 columns: milliseconds of kernels, planning next to nothing
    b0, bm = _case(16, 2, 1)
    rows = [np.array([[8, 8], [3, 4]], dtype=np.int32), np.array([[7, 9], [2, 2]], dtype=np.int32)]

    def fastest(alternate):
        times = []
        for k in range(12):
            t0 = time.perf_counter()
            pa.perm_poly_coefficients(b0, bm, rows[k % 2 if alternate else 0])
            times.append(time.perf_counter() - t0)
        return min(times[2:])

    print("poly rows alternating", flush=True)
    same, other = fastest(False), fastest(True)
    print(same, other, flush=True)
    assert other < 1.5 * same


def test_lists_that_differ_past_the_first_bytes(gpu, oracle):
    """40 000 rows of 2 variables: 320 kB, of which only the end differs."""
    b0, bm = _case(6, 2, 2)
    base = np.array([[i, j] for i in range(7) for j in range(7 - i)], dtype=np.int32)
    e1 = np.resize(base, (40000, 2))
    e2 = e1.copy()
    e2[-28:] = base[::-1]
    ref, _ = oracle.perm_poly_dd(b0, bm, base)
    mag, _ = oracle.perm_poly_dd(np.abs(b0).astype(complex), np.abs(bm).astype(complex), base)
    place = {tuple(e): k for k, e in enumerate(base.tolist())}
    print("poly rows late difference", flush=True)
    for e in (e1, e2, e1, e1, e2):
        got = pa.perm_poly_coefficients(b0, bm, e)
        at = np.array([place[tuple(r)] for r in e.tolist()])
        # layer i adds (m + 1) i products per value
        steps = sum(3 * i + 4 for i in range(1, 7))
        assert np.all(np.abs(got - ref[at]) <= steps * np.finfo(float).eps * np.abs(mag[at]))
