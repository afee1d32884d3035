"""Sensitivity images (spect_sensitivity) against the float64 back projection of
ones that blurs every plane.

Tolerance: the same terms in another order, sums of at most 41 x 41 taps and of
the planes in float64: 1e-13."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pytomography_amd import _lib
from tests.helpers import problem_arrays, product_system_matrix, rel_l2

pytestmark = pytest.mark.gpu

CASES = {
    "no_attenuation": dict(n=32, n_angles=6),
    "table": dict(n=33, n_angles=7, nz=64, att=True),
    "ragged_slices": dict(n=24, n_angles=5, nz=13, att=True),
    "two_z_blocks": dict(n=20, n_angles=5, nz=132, att=True),
    "one_slice": dict(n=24, n_angles=5, nz=1, att=True),
    "field": dict(n=32, n_angles=6, nz=20, att=True, field=True),
    "wide": dict(n=66, n_angles=6, nz=9, att=True, radius=75.0),
    "transaxial": dict(n=32, n_angles=6, att=True, psf_dims="1D"),
}


@pytest.mark.parametrize("name", CASES)
def test_sensitivity_matches_back_projected_ones(name):
    c = dict(CASES[name])
    field, dims, radius = c.pop("field", None), c.pop("psf_dims", "2D"), c.pop("radius", 25.0)
    pa = problem_arrays(c.pop("n"), c.pop("n_angles"), seed=6, psf=True, **c)
    pa["radii"] = radius + 2.0 * np.cos(2 * np.deg2rad(pa["angles"]))
    sm = product_system_matrix(pa, attenuation_field=field, psf_dims=dims)
    sm.set_n_subsets(2)
    for k in (0, 1):
        idx = sm.subset_indices_array[k]
        ones = torch.ones((len(idx), pa["n"], pa["nz"]), dtype=torch.float64, device="cuda")
        err = rel_l2(sm._sensitivity(k), sm._backward(ones, k, _lib.BP_REFERENCE))
        print(f"[{name}] {err:.1e}")
        assert err <= 1e-13
