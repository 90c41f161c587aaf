"""Tensor permanents of few and of many items: results written to host memory
up to 4096 items and copied beyond, each the same bits as alone; short walks
(up to 10 particles) for several items of every order."""

import numpy as np
import pytest

import piquasso_amd as pa
from test_gpu_tensor import _tol
from test_tensor_permanent import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 4095, 4096, 4097, 9000])
def test_items_are_the_same_alone(gpu, count):
    mats = [_rand(2 + (k % 2), k % 7) for k in range(count)]
    x = [0.1 * (k % 10) for k in range(count)]
    print(f"tensor items {count}", flush=True)
    got, asum = pa.tensor_permanent_batch(mats, x, with_abs_sum=True)
    for k in {0, count // 2, count - 1}:
        (one,), (s,) = pa.tensor_permanent_batch([mats[k]], [x[k]], with_abs_sum=True)
        assert got[k] == one and asum[k] == s


@pytest.mark.parametrize("n", range(1, 11))
def test_short_walks_match_oracle(gpu, oracle, n):
    mats = [_rand(n, 40 * n + k) for k in range(3)]
    x = [0.25, 0.9, 0.6]
    print(f"short tensor walks n={n}", flush=True)
    got = pa.tensor_permanent_batch(mats, x)
    for a, v, g in zip(mats, x, got):
        ref, asum = oracle.tensor_perm_dd(a, v)
        assert abs(g - ref.real) <= _tol(n, asum, ref.real)


@pytest.mark.parametrize("orders", [
    [2, 3], [9, 2, 5, 5, 1, 0, 7, 3, 3, 4], [17] * 20 + [18] * 6,  # the last: more than one flight of buffers
])
def test_mixed_orders_are_the_same_alone(gpu, orders):
    mats = [_rand(n, 7 * k + n) if n else np.zeros((0, 0), dtype=complex) for k, n in enumerate(orders)]
    x = [0.05 * (k % 20) for k in range(len(orders))]
    print(f"tensor orders {orders[:4]}..", flush=True)
    got, asum = pa.tensor_permanent_batch(mats, x, with_abs_sum=True)
    for k in sorted({0, 1, len(orders) // 2, len(orders) - 1}):
        (one,), (s,) = pa.tensor_permanent_batch([mats[k]], [x[k]], with_abs_sum=True)
        assert got[k] == one and asum[k] == s
