"""Calls that blur combined images (csrc/lowrank_launch.hpp) against the same
calls with every plane blurred by its own PSF (_lib.PLANES).

Tolerance: the images represent the planes' PSFs to 2^-22 = 2.4e-7; either side
sums up to 400 terms in float32, sqrt(400) 2^-23 = 2.4e-6 each: 5e-6."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from pytomography_amd import _lib
from tests.helpers import problem_arrays, product_system_matrix, rel_l2

pytestmark = pytest.mark.gpu

TOL = 5e-6

CASES = {
    # the back projection's rule: just below and above 39000 samples of a call
    "below_line": dict(n=32, n_angles=20, att=True),
    "above_line": dict(n=32, n_angles=32, att=True),
    "aligned_slices": dict(n=64, n_angles=9, att=True),
    "ragged_slices": dict(n=47, n_angles=24, nz=35, att=True),
    "ragged_quads": dict(n=52, n_angles=30, nz=28, att=True),
    "slices_by_four": dict(n=100, n_angles=5, att=True),
    "one_slice": dict(n=40, n_angles=7, nz=1),
    "no_attenuation": dict(n=48, n_angles=20),
    "table": dict(n=48, n_angles=20, att=True, field=False),
    "contour": dict(n=72, n_angles=10, att=True, contour=True),
    "wide": dict(n=66, n_angles=12, att=True, radius=75.0),
    "square": dict(n=48, n_angles=20, att=True, psf_shape="square"),
    "transaxial": dict(n=48, n_angles=20, att=True, psf_dims="1D"),
}


@pytest.mark.parametrize("name", CASES)
def test_combined_images_match_planes(name):
    c = dict(CASES[name])
    field, shape, dims = c.pop("field", None), c.pop("psf_shape", "gaussian"), c.pop("psf_dims", "2D")
    contour, radius = c.pop("contour", False), c.pop("radius", None)
    pa = problem_arrays(c.pop("n"), c.pop("n_angles"), seed=4, psf=True, **c)
    if radius:
        pa["radii"] = np.full(len(pa["radii"]), radius)
    if contour:
        pa["radii"] = 22.0 + 3.0 * np.cos(2 * np.deg2rad(pa["angles"]))
    sm = product_system_matrix(pa, attenuation_field=field, psf_shape=shape, psf_dims=dims)
    f = torch.from_numpy(pa["f"]).cuda()
    rng = np.random.default_rng(2)
    p = torch.from_numpy((0.5 + rng.random((len(pa["radii"]), pa["n"], pa["nz"]))).astype(np.float32)).cuda()
    sign = torch.from_numpy(rng.choice([-1.0, 1.0], p.shape).astype(np.float32)).cuda()
    for x in (f, -f):
        a, b = sm.forward(x), sm._project(x, None, "spect_forward", planes=True)
        errs = [rel_l2(a[k], b[k]) for k in range(a.shape[0])]
        print(f"[{name}] forward {max(errs):.1e}")
        assert max(errs) <= TOL
    for y in (p, p * sign):
        for mode in (_lib.BP_REFERENCE, _lib.BP_ADJOINT):
            err = rel_l2(sm._backward(y, None, mode), sm._backward(y, None, mode, planes=True))
            print(f"[{name}] back projection, mode {mode}: {err:.1e}")
            assert err <= TOL


def test_not_a_number_is_kept():
    pa = problem_arrays(32, 32, seed=4, psf=True, att=True)
    sm = product_system_matrix(pa)
    f = torch.from_numpy(pa["f"]).cuda()
    p = sm.forward(f)
    f[16, 15, 9] = p[3, 10, 12] = float("nan")
    for a, b in ((sm.forward(f), sm._project(f, None, "spect_forward", planes=True)),
                 (sm.backward(p), sm._backward(p, None, _lib.BP_REFERENCE, planes=True))):
        assert bool(b.isnan().any()) and not bool((b.isnan() & ~a.isnan()).any())
