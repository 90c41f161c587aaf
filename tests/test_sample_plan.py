"""The device sampler's buffer of partial minors (pqp_sample_plan_info)
against what its kernels write in every pass, the short last one included:
component c of wave w of shot s at doubles 2 ((s waves + w) 2 W + c) + {0, 1}."""

import ctypes

import numpy as np
import pytest

from piquasso_amd import _capi


def _plan(shots, photons, first):
    info = np.zeros(2 + 2 * photons, dtype=np.int64)
    st = _capi.lib().pqp_sample_plan_info(shots, photons, first, info.ctypes.data_as(_capi._i64p))
    assert st == 0
    return int(info[0]), int(info[1]), info[2::2], info[3::2]


@pytest.mark.parametrize("photons", range(1, 25))
def test_every_pass_stays_inside_its_partials(photons):
    steps = np.arange(1, photons)
    for shots in [*range(1, 4100), 6143, 6145, 8191, 10000, 100000]:
        first = 0
        while first < shots:
            n, held, digits, waves = _plan(shots, photons, first)
            assert 1 <= n <= min(2048, shots - first)
            if len(steps):
                k, w, width = digits[1:], waves[1:], steps + 1
                assert k.min() >= 0 and k.max() <= 7 and w.min() >= 1
                last = 2 * (((n - 1) * w + w - 1) * (2 * width) + 2 * width - 1) + 1
                assert 8 * (int(last.max()) + 1) <= held
            first += n
        assert first == shots


def test_arguments():
    info = np.zeros(64, dtype=np.int64)
    call = _capi.lib().pqp_sample_plan_info
    p = info.ctypes.data_as(_capi._i64p)
    assert call(10, 25, 0, p) == _capi.PQP_ERR_RANGE
    for args in ((10, -1, 0), (10, 3, 10), (0, 3, 0), (10, 3, -1)):
        assert call(*args, p) == _capi.PQP_ERR_INVALID
    assert call(10, 3, 0, ctypes.cast(None, _capi._i64p)) == _capi.PQP_ERR_INVALID
