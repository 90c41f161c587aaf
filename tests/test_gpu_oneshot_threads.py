"""One-shot batches of several threads at once: every call has its own results."""

import threading

import numpy as np
import pytest

from piquasso_amd.engine import permanent_batch

pytestmark = pytest.mark.gpu


def _batch(n, count, seed):
    rng = np.random.default_rng(seed)
    mats = [(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))) / np.sqrt(2 * n) for _ in range(count)]
    return mats, [np.ones(n, dtype=np.int32)] * count, [np.ones(n, dtype=np.int32)] * count


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
