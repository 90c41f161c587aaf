"""The device sampler over more than one pass of its buffers, where the last
pass is short and its steps take several waves a shot: the lockstep sampler's
samples."""

import numpy as np
import pytest

import piquasso_amd as pa
import piquasso_amd.sampling as P
from piquasso_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("photons, shots", [(14, 4000), (15, 3000), (16, 2500), (16, 4097)])
def test_short_last_pass_equals_lockstep(gpu, monkeypatch, photons, shots):
    u = W.haar_unitary(20, np.random.default_rng(photons))
    occ = [1] * photons + [0] * (20 - photons)
    print(f"sampler passes {photons} photons {shots} shots", flush=True)
    got = pa.generate_samples(occ, shots, u, seed_sequence=77)
    monkeypatch.setattr(P._MinorsBatch, "device_photons", -1)
    assert got == pa.generate_samples(occ, shots, u, seed_sequence=77)
