"""The device-planned column minors (perm_minors_wave.hip) at their edges:
every width through permanent_laplace from one digit to the widest, rows
that leave no binary digit, rows of one mode; and the device sampler against
the lockstep one, whose steps come from the planned minors."""

import numpy as np
import pytest

import piquasso_amd as pa
import piquasso_amd.sampling as P
from piquasso_amd import workloads as W

pytestmark = pytest.mark.gpu

EPS = np.finfo(float).eps


def _rows(kind, n, rng):
    if kind == "ones":
        return [1] * n
    if kind == "one mode":
        return [0, n, 0]
    if kind == "pairs":  # the prepend leaves one binary digit
        return [2] * (n // 2) + [1] * (n % 2)
    if kind == "triples":  # none where n is a multiple of 3
        return [3] * (n // 3) + ([n % 3] if n % 3 else [])
    return np.bincount(rng.integers(0, n, n), minlength=n).tolist()


@pytest.mark.parametrize("kind", ["ones", "one mode", "pairs", "triples", "random"])
@pytest.mark.parametrize("width", [2, 3, 4, 7, 8, 9, 13, 16, 17, 20])
def test_minors_match_oracle(gpu, oracle, width, kind):
    n = width - 1
    rng = np.random.default_rng(width * 10 + len(kind))
    rows = _rows(kind, n, rng)
    u = W.haar_unitary(max(len(rows), width), rng)[: len(rows), :width]
    print(f"wave minors width={width} rows {kind}", flush=True)
    got = pa.permanent_laplace(u, rows, [1] * width)
    ref = oracle.laplace_dd(u, rows, [1] * width)
    # Glynn terms are at most prod_j sum_i r_i |a_ij| over the kept columns,
    # n + 1 rounded factors each, averaged over the terms
    col = np.abs(u).T @ np.asarray(rows, dtype=float)
    tol = [4 * (n + 2) * EPS * np.prod(np.delete(col, l)) for l in range(width)]
    assert got.shape == (width,) and np.all(np.abs(got - ref) <= tol)


@pytest.mark.parametrize("width", [21, 22, 23, 24])
def test_widest_minors_expand_the_permanent(gpu, width):
    """perm(A) = sum_l a_l M_l for the row a added to the minors' rows."""
    rng = np.random.default_rng(width)
    u = W.haar_unitary(width, rng)
    rows = [1] * (width - 1)
    print(f"wave minors width={width}", flush=True)
    got = pa.permanent_laplace(u[1:], rows, [1] * width)
    perm = complex(pa.permanent(u, [1] * width, [1] * width))
    col = np.abs(u).sum(axis=0)
    assert abs(u[0] @ got - perm) <= 8 * (width + 2) * EPS * np.prod(col)


def test_planned_path_and_errors_stay(gpu, oracle):
    """Columns of other multiplicities keep the planned kernels; sums that do
    not fit stay refused."""
    u = W.haar_unitary(5, np.random.default_rng(1))
    for rows, cols in (([1, 1, 0, 1, 0], [1, 0, 2, 1, 0]), ([2, 0, 0, 0, 1], [1, 1, 1, 1, 0])):
        got, ref = pa.permanent_laplace(u, rows, cols), oracle.laplace_dd(u, rows, cols)
        assert np.all(np.abs(got - ref) <= 1e-13)
    with pytest.raises(RuntimeError):
        pa.permanent_laplace(u, [1, 1, 1, 1, 1], [1, 1, 1, 1, 1])
    with pytest.raises(ValueError):
        pa.permanent_laplace(u, [1, -1, 2, 1, 1], [1, 1, 1, 1, 1])


@pytest.mark.parametrize("occ, shots, loss, overlap", [
    ([1] * 12 + [0] * 12, 65, 0.0, None),
    ([1, 2, 0, 1, 1, 0, 0, 1], 33, 0.0, None),
    ([5], 3, 0.0, None),
    ([1] * 9, 40, 0.3, None),
    ([2, 1, 0, 1], 50, 0.9, None),          # shots that keep no photon
    ([1, 1, 2, 0, 1], 40, 0.2, 0.4),
    ([1] * 5 + [0] * 59, 2049, 0.0, None),  # 64 modes, one shot past a pass of the buffers
    ([1] * 24 + [0] * 8, 4, 0.0, None),     # the most photons
])
def test_device_sampler_equals_lockstep(gpu, monkeypatch, occ, shots, loss, overlap):
    u = W.haar_unitary(len(occ), np.random.default_rng(len(occ) + shots))

    def samples():
        lost = np.random.default_rng(11)
        reject = (lambda: lost.uniform() < loss) if loss else None
        return pa.generate_samples(occ, shots, u, reject, uniform_particle_overlap=overlap, seed_sequence=321)

    print(f"sampler {len(occ)} modes {sum(occ)} photons {shots} shots", flush=True)
    got = samples()
    run = dict(pa.sampling.last_run)
    monkeypatch.setattr(P._MinorsBatch, "device_photons", -1)
    assert got == samples()
    assert [run[k] for k in ("rounds", "problems")] == [pa.sampling.last_run[k] for k in ("rounds", "problems")]
    assert got[: shots // 2] == got[: len(got) // 2] and len(got) == shots


def test_sampler_rejects_bad_distributions(gpu):
    with pytest.raises(ValueError, match="NaN"):
        pa.generate_samples([1, 1], 4, np.zeros((2, 2)), seed_sequence=1)
    with pytest.raises(ValueError, match="NaN"):
        pa.generate_samples([1, 1], 4, np.full((2, 2), np.nan), seed_sequence=1)
