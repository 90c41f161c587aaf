"""The probability-table kernel (perm_table.hip) at its edges: 1 to 16
particles across the 1-, 4- and 16-wave forms, repeated input modes, 64
modes, outputs from one mode holding everything to all distinct, rows of
other particle numbers, and row counts around a chunk."""

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd import workloads as W

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _norm(occ):
    f = 1.0
    for k in occ:
        for q in range(2, int(k) + 1):
            f *= q
    return f


def _check(oracle, u, s, outs):
    """Against the double-double oracle within the forward-error bound of the
    sweep as given, 4 (n + 2) u sum|terms| / 2^(n-1), from the batch kernels."""
    s, outs = np.asarray(s), np.asarray(outs)
    got = pa.output_amplitudes(u, s, outs)
    prob = pa.output_probabilities(u, s, outs)
    with pa.PermanentBatch([u] * len(outs), list(outs), [s] * len(outs), as_given=True) as b:
        bound = b.run("eager").error_bounds()
    for t, g, p, e in zip(outs, got, prob, bound):
        scale = np.sqrt(_norm(t) * _norm(s))
        ref = oracle.perm_dd(u, t, s) / scale
        tol = e / scale + 4 * EPS * abs(ref)
        assert abs(g - ref) <= tol, (t, g, ref)
        assert abs(p - abs(ref) ** 2) <= 3 * abs(ref) * tol + tol ** 2, (t, p, ref)


def _outputs(rng, m, n, count):
    outs = [np.bincount(rng.integers(0, m, n), minlength=m) for _ in range(count)]
    heap = np.zeros(m, dtype=int)
    heap[m // 2] = n  # every particle in one mode
    outs.append(heap)
    if n <= m:
        outs.append((np.arange(m) < n).astype(int)[::-1])  # one in each of the last modes
    return np.array(outs)


@pytest.mark.parametrize("n, m", [
    (1, 1), (1, 5), (2, 2), (3, 64), (5, 4), (7, 14), (8, 8), (9, 11), (10, 12), (12, 12),
    (12, 64), (13, 16), (15, 20), (16, 16), (16, 40),
])
def test_unit_input(gpu, oracle, n, m):
    rng = np.random.default_rng(100 * n + m)
    s = np.bincount(np.arange(n) % m, minlength=m)
    print(f"table n={n} modes={m}", flush=True)
    _check(oracle, W.haar_unitary(m, rng), s, _outputs(rng, m, n, 5))


@pytest.mark.parametrize("s", [[2], [0, 3, 0, 1], [4, 4], [1, 2, 0, 3, 1], [16], [5, 0, 4, 3, 0, 1, 1, 1],
                               [2, 2, 2, 2, 2, 2, 2, 2]])
def test_repeated_input_modes(gpu, oracle, s):
    rng = np.random.default_rng(len(s) + sum(s))
    print(f"table input {s}", flush=True)
    _check(oracle, W.haar_unitary(len(s), rng), s, _outputs(rng, len(s), sum(s), 5))


@pytest.mark.parametrize("count", [1, 3, 4, 5, 16383, 16384, 16385])
def test_row_counts_and_other_particle_numbers(gpu, count):
    """Every row equals the same row asked alone; other particle numbers,
    also ones a byte cannot hold, give exactly 0."""
    rng = np.random.default_rng(count)
    u = W.haar_unitary(6, rng)
    s = [1, 1, 0, 2, 0, 0]
    outs = np.array([np.bincount(rng.integers(0, 6, 4), minlength=6) for _ in range(count)])
    outs[count // 2] = 1                    # 6 particles
    outs[-1] = [4 + 256, 0, 0, 0, 0, 0]
    print(f"table of {count} rows", flush=True)
    got = pa.output_amplitudes(u, s, outs)
    sums = outs.sum(axis=1)
    assert np.all(got[sums != 4] == 0)
    pick = rng.integers(0, count, 8)
    for k in pick:
        assert got[k] == pa.output_amplitudes(u, s, outs[k])[0]
    assert abs(pa.output_probabilities(u, s, outs)[0] - abs(got[0]) ** 2) <= 2 * EPS * abs(got[0]) ** 2


def test_errors(gpu):
    u = np.eye(3, dtype=complex)
    with pytest.raises(ValueError, match="non-negative"):
        pa.output_probabilities(u, [1, 1, 0], [[1, 1, 0], [2, -1, 1]])
    with pytest.raises(ValueError, match="non-negative"):
        pa.output_probabilities(u, [1, -1, 2], [[1, 1, 0]])
    assert pa.output_probabilities(u, [1, 1, 0], np.zeros((0, 3), dtype=int)).shape == (0,)
    # vacuum, and more particles than the kernel takes: the planned batch
    assert pa.output_probabilities(u, [0, 0, 0], [[0, 0, 0], [1, 0, 0]]).tolist() == [1.0, 0.0]
    assert abs(pa.output_probabilities(u, [17, 0, 0], [[17, 0, 0]])[0] - 1.0) < 1e-12
