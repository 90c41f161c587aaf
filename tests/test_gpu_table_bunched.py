"""Probability tables of inputs with several particles in a mode: each output
is summed over the digits, the output's or the input's, that the planner
takes.  The rows of the matrix differ by powers of ten (a lossy circuit's),
so the other sweep cancels and leaves the planned one's error bound."""

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd import workloads as W
from conftest import glynn_abs_sum
from test_gpu_table import EPS, _norm, _outputs

pytestmark = pytest.mark.gpu


def _perm(oracle, u, t, s):
    """The oracle's sum by the digits that cancel less: in double-double the
    other one may keep fewer digits than the result has."""
    by_input = glynn_abs_sum(u.T, s, t) < glynn_abs_sum(u, t, s)
    return oracle.perm_dd(np.ascontiguousarray(u.T), s, t) if by_input else oracle.perm_dd(u, t, s)


@pytest.mark.parametrize("s", [
    [2, 0], [4, 0, 0], [2, 1, 0, 0], [5, 1, 1, 0], [3, 3, 0, 0], [0, 2, 2, 2, 0, 0],
    [2, 2, 2, 2, 2, 0, 0, 0], [12, 0, 0, 0, 0, 0], [6, 0, 6, 0, 0], [4, 4, 4, 4, 0, 0],
    [16, 0, 0, 0], [8, 8, 0, 0, 0, 0], [2] * 8, [3, 2, 2, 2, 2, 2, 2, 1], [2] + [1] * 14 + [0] * 49,
])
def test_sums_by_the_cheaper_digits(gpu, oracle, s):
    rng = np.random.default_rng(100 * sum(s) + len(s))
    m, n = len(s), sum(s)
    u = W.haar_unitary(m, rng) * 10.0 ** -(np.arange(m) % 4)[:, None]
    outs = _outputs(rng, m, n, 12)
    print(f"bunched table input {s}", flush=True)
    got = pa.output_amplitudes(u, s, outs)
    prob = pa.output_probabilities(u, s, outs)
    with pa.PermanentBatch([u] * len(outs), list(outs), [np.array(s)] * len(outs)) as b:
        bound = b.run("eager").error_bounds()
    for t, g, p, e in zip(outs, got, prob, bound):
        scale = np.sqrt(_norm(t) * _norm(s))
        ref = _perm(oracle, u, t, s) / scale
        tol = e / scale + 4 * EPS * abs(ref)
        assert abs(g - ref) <= tol, (t, g, ref)
        assert abs(p - abs(ref) ** 2) <= 3 * abs(ref) * tol + tol ** 2, (t, p, ref)


def test_other_inputs_in_between(gpu):
    """The input's states are laid out for each call."""
    rng = np.random.default_rng(5)
    u = W.haar_unitary(6, rng)
    inputs = [[4, 2, 0, 0, 0, 0], [1] * 6, [2, 2, 2, 0, 0, 0], [0, 0, 6, 0, 0, 0]]
    outs = _outputs(rng, 6, 6, 30)
    want = [pa.output_amplitudes(u, s, outs) for s in inputs]
    for k in (3, 0, 2, 1, 0, 3, 3, 1):
        assert np.array_equal(pa.output_amplitudes(u, inputs[k], outs), want[k])
