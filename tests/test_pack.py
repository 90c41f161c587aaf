"""The CPython binding's argument lists of batched calls (fastcall.c: pack):
what it packs, what it leaves to the general path, and one-shot batches
against a kept handle."""

import ctypes

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd._math.permanent import _fast_module
from piquasso_amd.engine import _packed, permanent_batch
from piquasso_amd.tune import mean_log2_terms


def _items(seed, count=7):
    rng = np.random.default_rng(seed)
    mats, rows, cols = [], [], []
    for k in range(count):
        m_r, m_c = int(rng.integers(1, 5)), int(rng.integers(1, 5))
        mats.append(rng.standard_normal((m_r, m_c)) + 1j * rng.standard_normal((m_r, m_c)))
        r, c = rng.integers(0, 3, m_r), rng.integers(0, 3, m_c)
        d = int(r.sum() - c.sum())
        (c if d > 0 else r)[0] += abs(d)
        rows.append(r.astype(np.int32 if k % 2 else np.int64))
        cols.append(c.astype(np.int64 if k % 3 else np.int32))
    return mats, rows, cols


def _read(address, shape, dtype):
    size = int(np.prod(shape)) * np.dtype(dtype).itemsize
    return np.frombuffer(ctypes.string_at(int(address), size), dtype=dtype).reshape(shape)


@pytest.fixture(autouse=True)
def binding():
    if not _fast_module():
        pytest.skip("the CPython binding is not built")


@pytest.mark.parametrize("narrow", [(), (0,), (2, 5), tuple(range(7))])
def test_packs_what_the_arrays_hold(narrow):
    mats, rows, cols = _items(3)
    for k in narrow:
        mats[k] = mats[k].astype(np.complex64)
    (mp, rp, cp), m_r, m_c, _keep, log2_terms = _packed(mats, rows, cols, True)
    mp, rp, cp = (np.frombuffer(p, dtype=np.uint64) for p in (mp, rp, cp))
    for k, (m, r, c) in enumerate(zip(mats, rows, cols)):
        assert (m_r[k], m_c[k]) == m.shape
        assert np.array_equal(_read(mp[k], m.shape, np.complex128), m.astype(np.complex128))
        assert np.array_equal(_read(rp[k], r.shape, np.int32), r)
        assert np.array_equal(_read(cp[k], c.shape, np.int32), c)
    assert abs(log2_terms - mean_log2_terms(rows)) < 1e-12


def _other_forms():
    mats, rows, cols = _items(4)
    # (an array of one entry is contiguous whatever its stride)
    mats[3], rows[3], cols[3] = np.ones((2, 3), dtype=complex), np.array([2, 1]), np.array([1, 1, 1])

    def with_(which, k, value):
        lists = [list(mats), list(rows), list(cols)]
        lists[which][k] = value
        return lists

    return {
        "float matrix": with_(0, 1, mats[1].real.copy()),
        "transposed matrix": with_(0, 1, np.asfortranarray(np.ones((2, 3)) * (1 + 0j))),
        "list matrix": with_(0, 1, mats[1].tolist()),
        "vector matrix": with_(0, 1, np.ones(3, dtype=complex)),
        "list rows": with_(1, 2, rows[2].tolist()),
        "float rows": with_(1, 2, rows[2].astype(float)),
        "short rows": with_(1, 2, rows[2][:-1]),
        "strided columns": with_(2, 3, np.repeat(cols[3], 2)[::2]),
        "wide columns": with_(2, 3, cols[3].astype(np.int64) + 2**33),
        "two-dimensional columns": with_(2, 3, cols[3][None, :]),
        "an array of matrices": [np.ones((2, 2, 2), dtype=complex), [np.ones(2, int)] * 2, [np.ones(2, int)] * 2],
        "no items": [[], [], []],
    }


@pytest.mark.parametrize("form", sorted(_other_forms()))
def test_leaves_other_forms_to_the_general_path(form):
    assert _packed(*_other_forms()[form], True) is None


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_shot_equals_a_kept_batch(gpu, precision):
    """The same plan on the library's own buffers: bit for bit, also for the
    forms the general path takes, and after a batch of another size."""
    for seed in (5, 6):
        mats, rows, cols = _items(seed, 40 if seed == 5 else 9)
        with pa.PermanentBatch(mats, rows, cols, precision=precision) as b:
            want = b.run("eager").results()
        assert np.array_equal(permanent_batch(mats, rows, cols, precision=precision), want)
        lists = [r.tolist() for r in rows], [c.tolist() for c in cols]
        assert np.array_equal(permanent_batch(mats, *lists, precision=precision), want)
    with pytest.raises(RuntimeError):
        permanent_batch([np.ones((2, 2), dtype=complex)], [np.array([1, 1])], [np.array([1, 0])])
    with pytest.raises(ValueError):
        permanent_batch([np.ones((2, 2), dtype=complex)], [np.array([1, -1])], [np.array([0, 0])])
    with pytest.raises(ValueError):
        permanent_batch([np.ones((2, 2), dtype=complex)], [np.array([1, 1])], [])
    assert len(permanent_batch([], [], [])) == 0


@pytest.mark.gpu
def test_gradients_of_packed_and_listed_items(gpu):
    mats, rows, cols = _items(8)
    p1, g1 = pa.permanent_grad_batch(mats, rows, cols)
    p2, g2 = pa.permanent_grad_batch(mats, [r.tolist() for r in rows], [c.tolist() for c in cols])
    assert np.array_equal(p1, p2) and all(np.array_equal(a, b) for a, b in zip(g1, g2))
    assert [g.shape for g in g1] == [m.shape for m in mats]
