"""Sensitivities without a GPU are refused as every projector call is."""
import pytest

import pytomography_amd
from pytomography_amd import _lib
from tests.helpers import problem_arrays, product_system_matrix


@pytest.mark.parametrize("att", [False, True])
def test_sensitivity_on_the_host_is_refused(att):
    before = pytomography_amd.device
    try:
        sm = product_system_matrix(problem_arrays(16, 4, att=att, psf=True), device="cpu")
        with pytest.raises(_lib.SpectLibraryError, match="need a ROCm/HIP device tensor"):
            sm.compute_normalization_factor()
    finally:
        pytomography_amd.set_device(before)
