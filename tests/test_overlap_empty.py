"""Detection probabilities of a circuit without modes: checked like any other."""

import numpy as np
import pytest

from piquasso_amd.distinguishability import detection_probabilities


@pytest.mark.parametrize("overlap", [float("nan"), float("inf")])
def test_overlap_is_checked_without_modes(overlap):
    with pytest.raises(ValueError, match="overlap"):
        detection_probabilities(np.zeros((2, 0), dtype=int), np.zeros((0, 0)), [], overlap)


def test_no_outputs_without_modes():
    assert detection_probabilities(np.zeros((0, 0), dtype=int), np.zeros((0, 0)), [], 0.5).shape == (0,)


@pytest.mark.gpu
def test_empty_products_are_one(gpu):
    got = detection_probabilities(np.zeros((3, 0), dtype=int), np.zeros((0, 0)), [], 0.5)
    assert np.array_equal(got, np.ones(3))
