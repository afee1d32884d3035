"""Float32 projections of a default system matrix blur every plane with its own
PSF: values are accurate relative to themselves however bright a source beside
them is, and an infinity or a NaN reaches as far as the PSF and no further."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import pytomography_amd
from pytomography_amd import _lib
from tests.helpers import problem_arrays, product_system_matrix

pytestmark = pytest.mark.gpu

CASES = {
    "attenuation_field": dict(n=64, n_angles=9, att=True),
    "no_attenuation": dict(n=48, n_angles=20),
    "ragged_slices": dict(n=47, n_angles=24, nz=35, att=True),
    "one_slice": dict(n=40, n_angles=7, nz=1),
}


@pytest.mark.parametrize("name", CASES)
def test_default_calls_blur_every_plane(name):
    """The bits of the calls that ask for it."""
    c = dict(CASES[name])
    pa = problem_arrays(c.pop("n"), c.pop("n_angles"), seed=4, psf=True, **c)
    sm = product_system_matrix(pa)
    f = torch.from_numpy(pa["f"]).cuda()
    p = sm.forward(f)
    assert torch.equal(p, sm._project(f, None, "spect_forward", planes=True))
    for mode in (_lib.BP_REFERENCE, _lib.BP_ADJOINT):
        assert torch.equal(sm._backward(p, None, mode), sm._backward(p, None, mode, planes=True))


def _near_source(n=64, n_angles=16):
    """A small ball at the object's edge, 0.5 cm from the detector at 270
    degrees: there its PSF is a third of a pixel wide."""
    pa = problem_arrays(n, n_angles, psf=True)
    pa["radii"] = np.full(n_angles, 14.0)
    x = np.arange(n, dtype=np.float32)
    c = (n - 5.0, n / 2, n / 2)
    pa["f"] = np.ascontiguousarray(((x[:, None, None] - c[0]) ** 2 + (x[:, None] - c[1]) ** 2
                                    + (x - c[2]) ** 2 <= 4.0).astype(np.float32))
    return pa, n_angles * 270 // 360


def test_count_beside_a_masked_start():
    """OSEM without an additive term, from an object that is zero outside a
    ball: one count on a pixel that sees nothing of it gives a ratio of 1e11,
    which must not reach the ball through the tails of other planes' PSFs.

    Tolerance: the composed update rounds each step alike except the last four
    operations, 4 x 2^-24 of the value or of the start: 1e-6."""
    pa, a = _near_source()
    sm = product_system_matrix(pa)
    f = torch.from_numpy(pa["f"]).cuda()
    p = sm._project(f, None, "spect_forward", planes=True)
    g = p.clone()
    lit = (p[a] > 0).nonzero()
    mid = pa["nz"] // 2
    j = int(lit[lit[:, 1] == mid][:, 0].max()) + 1
    assert float(p[a, j, mid]) == 0.0
    g[a, j, mid] = 5.0
    norm = sm.compute_normalization_factor(None)
    delta = float(pytomography_amd.delta)
    b = sm._backward(g / (p + delta), None, _lib.BP_REFERENCE, planes=True)
    want = (f + f * (1 / (norm + delta)) * (b - norm)).clamp(min=0)
    got = f.clone()
    sm.osem_step(got, g, None, norm, None)
    err = ((got - want).abs() / (want.abs() + f + 1e-30))[f > 0].max()
    print(f"largest error of a voxel of the ball: {float(err):.1e}")
    assert float(err) <= 1e-6


@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
def test_values_that_are_not_finite_reach_as_far_as_the_psf(value):
    n, z = 64, 8
    pa = problem_arrays(n, 16, psf=True, att=True, seed=2)
    sm = product_system_matrix(pa)
    far = z + sm._plan(torch.device("cuda", torch.cuda.current_device())).psf_half + 1
    f = torch.from_numpy(pa["f"]).cuda()
    p = sm.forward(f)
    f[n // 2, n // 2, z] = value
    q = sm.forward(f)
    assert not bool(torch.isfinite(q[:, :, z]).all())
    assert torch.equal(q[:, :, far:], p[:, :, far:])
    b = sm.backward(p)
    p[3, n // 2, z] = value
    d = sm.backward(p)
    assert not bool(torch.isfinite(d[:, :, z]).all())
    assert torch.equal(d[:, :, far:], b[:, :, far:])
