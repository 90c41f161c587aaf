"""The tensor-permanent sweep with precomputed sign rows (tensor_perm.hip) and
the overlap tables on it: every small order, the first orders of more than
one lane block and of longer walks, repeated input modes, outputs of other
particle numbers, and tables of one row and of more rows than a pass."""

import math

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd import workloads as W
from piquasso_amd.distinguishability import uniform_input_norm

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _expected(oracle, u, s, t, x):
    """(probability, tolerance) from the double-double tensor permanent of
    the expanded matrix; the kernels' sum of magnitudes bounds the error as
    8 (n + 2) eps sum|term|."""
    ri, ci = np.repeat(np.arange(len(t)), t), np.repeat(np.arange(len(s)), s)
    a = np.ascontiguousarray(np.asarray(u)[np.ix_(ri, ci)])
    (got,), (mag,) = pa.tensor_permanent_batch([a], [x], with_abs_sum=True)
    ref, _ = oracle.tensor_perm_dd(a, x)
    tol = 8 * (len(ri) + 2) * EPS * mag
    assert abs(got - ref) <= tol
    norm = uniform_input_norm(s, x) * math.prod(math.factorial(int(k)) for k in t)
    return ref / norm, tol / norm + 4 * EPS * abs(ref / norm)


@pytest.mark.parametrize("n, m", [(1, 1), (1, 4), (2, 2), (3, 5), (4, 4), (5, 7), (6, 6), (7, 9), (8, 5), (9, 9),
                                  (10, 12), (11, 11)])
@pytest.mark.parametrize("x", [0.0, 0.37, 1.0])
def test_tables_match_oracle(gpu, oracle, n, m, x):
    rng = np.random.default_rng(10 * n + m)
    u = W.haar_unitary(m, rng)
    s = np.bincount(np.arange(n) % m, minlength=m)
    outs = [np.bincount(rng.integers(0, m, n), minlength=m) for _ in range(3)]
    outs.append(np.eye(m, dtype=int)[m // 2] * n)
    outs.insert(1, np.zeros(m, dtype=int))
    print(f"overlap table n={n} modes={m} x={x}", flush=True)
    got = pa.detection_probabilities(outs, u, s, x)
    assert got[1] == 0.0
    for t, g in zip(outs, got):
        if sum(t) == n:
            ref, tol = _expected(oracle, u, s, t, x)
            assert abs(g - ref) <= tol, (t, g, ref)


@pytest.mark.parametrize("n", [12, 13, 15])
def test_longer_walks_against_glynn(gpu, n):
    """x = 1: |perm|^2; x = 0: perm(|A|^2), from the permanent kernels."""
    rng = np.random.default_rng(n)
    u = W.haar_unitary(n, rng)
    one = np.ones(n, dtype=int)
    t = np.bincount(rng.integers(0, n, n), minlength=n)
    fact = math.prod(math.factorial(int(k)) for k in t)
    print(f"overlap walk n={n}", flush=True)
    for x, want in ((1.0, abs(complex(pa.permanent(u, t, one))) ** 2),
                    (0.0, complex(pa.permanent(np.abs(u) ** 2 + 0j, t, one)).real)):
        a = np.repeat(u, t, axis=0)
        (got,), (mag,) = pa.tensor_permanent_batch([a], [x], with_abs_sum=True)
        assert abs(got - want) <= 16 * (n + 2) * EPS * mag
        p = pa.detection_probabilities([t], u, one, x)[0]
        assert abs(p - got / fact) <= 4 * EPS * abs(p)


def test_more_rows_than_a_pass(gpu):
    """A row's value does not depend on its company: 32768 items are a pass."""
    rng = np.random.default_rng(3)
    u = W.haar_unitary(4, rng)
    s = np.array([1, 1, 0, 0])
    outs = np.array([np.bincount(rng.integers(0, 4, 2), minlength=4) for _ in range(32770)])
    outs[7] = [300, 0, 0, 0]
    got = pa.detection_probabilities(outs, u, s, 0.6)
    assert got[7] == 0.0
    for k in (0, 1, 32766, 32767, 32768, 32769):
        assert got[k] == pa.detection_probabilities([outs[k]], u, s, 0.6)[0]
    patterns = np.unique(np.delete(outs, 7, axis=0), axis=0)
    assert abs(pa.detection_probabilities(patterns, u, s, 0.6).sum() - 1.0) < 1e-13


def test_errors(gpu):
    u = np.eye(3, dtype=complex)
    with pytest.raises(ValueError, match="non-negative"):
        pa.detection_probabilities([[1, 1, 0], [3, -1, 0]], u, [1, 1, 0], 0.5)
    with pytest.raises(ValueError, match="finite"):
        pa.detection_probabilities([[1, 1, 0]], u, [1, 1, 0], float("nan"))
    with pytest.raises(ValueError, match="20"):
        pa.detection_probabilities([[21, 0, 0]], u, [21, 0, 0], 0.5)
    assert pa.detection_probabilities([[0, 0, 0], [1, 0, 0]], u, [0, 0, 0], 0.5).tolist() == [1.0, 0.0]
