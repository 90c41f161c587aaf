"""The first use of an entry point under host-forced allocation failures: each
allocation of the call fails in turn in a fresh process, as MemoryError, and
the call after the last is right.  The failures are decided on the host before
any launch."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_CHILD = """
import sys
import numpy as np
sys.path.insert(0, {root!r})
import piquasso_amd as pa
from oracle import oracle as O
from piquasso_amd import _capi
rng = np.random.default_rng(2)
a = (rng.standard_normal((5, 5)) + 1j * rng.standard_normal((5, 5))) / 3
ones = [1] * 5
call, want = {{
    "laplace": (lambda: pa.permanent_laplace(a[1:], ones[1:], ones), lambda: O.laplace_dd(a[1:], ones[1:], ones)),
    "single": (lambda: complex(pa.permanent(a, ones, ones)), lambda: O.perm_dd(a, ones, ones)),
}}[{what!r}]
L = _capi.lib()
for k in range(20):
    L.pqp_debug_fail_allocation(k)
    try:
        got = call()
    except MemoryError as e:
        assert "forced failure" in str(e)
        continue
    finally:
        L.pqp_debug_fail_allocation(-1)
    break
else:
    raise SystemExit("never succeeded")
assert k >= 2 and np.all(np.abs(got - want()) <= 1e-13)
assert np.all(np.abs(call() - want()) <= 1e-13)
print("failures", k)
"""


@pytest.mark.parametrize("what", ["laplace", "single"])
def test_each_first_allocation_failure_is_clean(gpu, what):
    print(f"first use of {what}", flush=True)
    res = subprocess.run([sys.executable, "-c", _CHILD.format(root=ROOT, what=what)], cwd=ROOT,
                         capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    assert res.stdout.startswith("failures")
