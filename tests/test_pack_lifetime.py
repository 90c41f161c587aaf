"""What a packed batch points to lives as long as the packed arguments, also
when another thread takes an item out of the caller's list meanwhile."""

import ctypes
import gc
import weakref

import numpy as np
import pytest

from piquasso_amd._math.permanent import _fast_module
from piquasso_amd.engine import _packed


@pytest.fixture(autouse=True)
def binding():
    if not _fast_module():
        pytest.skip("the CPython binding is not built")


def test_matrices_outlive_the_list_that_held_them():
    mats = [np.full((2, 2), k + 1j) for k in range(3)]
    alive = [weakref.ref(m) for m in mats]
    mult = [np.ones(2, dtype=np.int32)] * 3
    packed = _packed(mats, mult, mult, True)
    mats[1] = None
    mats.clear()
    gc.collect()
    assert all(r() is not None for r in alive)
    at = np.frombuffer(packed[0][0], dtype=np.uint64)
    for k in range(3):
        held = np.frombuffer(ctypes.string_at(int(at[k]), 64), dtype=np.complex128)
        assert np.array_equal(held, np.full(4, k + 1j))
    del packed
    gc.collect()
    assert all(r() is None for r in alive)


def test_refused_batches_hold_nothing():
    mats = [np.ones((2, 2), dtype=complex), np.ones((2, 2))]
    alive = [weakref.ref(m) for m in mats]
    mult = [np.ones(2, dtype=np.int32)] * 2
    assert _packed(mats, mult, mult, True) is None
    mats.clear()
    gc.collect()
    assert all(r() is None for r in alive)
