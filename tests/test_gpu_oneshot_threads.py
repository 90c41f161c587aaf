"""One-shot batches of several threads: a short call does not wait for a long
one, and every call has its own results."""

import threading
import time

import numpy as np
import pytest

import piquasso_amd as pa
from piquasso_amd.engine import permanent_batch

pytestmark = pytest.mark.gpu


def _batch(n, count, seed):
    rng = np.random.default_rng(seed)
    mats = [(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2 * n) for _ in range(count)]
    return mats, [np.ones(n, dtype=np.int32)] * count, [np.ones(n, dtype=np.int32)] * count


def test_a_short_call_does_not_wait_for_a_long_one(gpu):
    long_one, short = _batch(31, 60, 1), _batch(6, 5, 2)
    permanent_batch(*short)
    permanent_batch(*_batch(31, 1, 3))
    pa.permanent(short[0][0], short[1][0], short[2][0])
    done = {}

    def run():
        permanent_batch(*long_one)
        done["long"] = time.perf_counter()

    print("one-shot threads", flush=True)
    t = threading.Thread(target=run)
    start = time.perf_counter()
    t.start()
    time.sleep(0.05)
    for _ in range(3):
        permanent_batch(*short)
        pa.permanent(short[0][0], short[1][0], short[2][0])
    done["short"] = time.perf_counter()
    t.join()
    print({k: v - start for k, v in done.items()}, flush=True)
    assert done["long"] - start > 0.1
    assert done["short"] < done["long"]


def test_threads_have_their_own_results(gpu):
    items = [_batch(5 + k, 40 + 7 * k, k) for k in range(6)]
    want = [permanent_batch(*a) for a in items]
    wrong = []

    def run(k):
        for _ in range(20):
            if not np.array_equal(permanent_batch(*items[k]), want[k]):
                wrong.append(k)

    print("six one-shot threads", flush=True)
    threads = [threading.Thread(target=run, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
