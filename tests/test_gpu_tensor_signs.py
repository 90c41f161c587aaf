"""Sign rows of items of several orders, written by one launch: orders whose
items take one block and several (256 entries a block: 6 particles 192, 7 448),
and more passes than one launch holds, each the same bits as alone."""

import numpy as np
import pytest

import piquasso_amd as pa
from test_tensor_permanent import _rand

pytestmark = pytest.mark.gpu


def _same_alone(mats, x, which):
    got, asum = pa.tensor_permanent_batch(mats, x, with_abs_sum=True)
    for k in which:
        (one,), (s,) = pa.tensor_permanent_batch([mats[k]], [x[k]], with_abs_sum=True)
        assert got[k] == one and asum[k] == s
    return got


@pytest.mark.parametrize("orders", [
    [6, 7], [7, 6], [1, 8, 1], [10, 6, 7, 6, 7, 2], list(range(1, 14)), [13, 1], [12] * 3 + [11] * 2 + [1] * 5,
])
def test_orders_of_one_and_several_blocks(gpu, orders):
    mats = [_rand(n, 11 * k + n) for k, n in enumerate(orders)]
    x = [0.05 * (k % 20) for k in range(len(orders))]
    print(f"tensor sign rows {orders}", flush=True)
    _same_alone(mats, x, range(len(orders)))


def test_more_passes_than_one_launch_holds(gpu):
    """21 passes of one particle (32 768 items each, the last one short) and
    one of two: |a|^2 whatever the overlap."""
    few = [_rand(1, k) for k in range(5)]
    count = 20 * 32768 + 3
    mats = (few * (count // 5 + 1))[:count] + [_rand(2, 9)]
    x = [0.3] * len(mats)
    print(f"tensor passes, {len(mats)} items", flush=True)
    got = np.asarray(_same_alone(mats, x, [0, 32767, 32768, count - 1, count]))
    want = np.array([abs(a[0, 0]) ** 2 for a in few])
    ref = np.tile(want, count // 5 + 1)[:count]
    assert np.all(np.abs(got[:count] - ref) <= 8 * 2.0 ** -52 * ref)
