"""The projector on combined images (csrc/lowrank.hpp, lowrank_body.hpp) on the
CPU: the host fit of the planes' PSFs, and the wave bodies built with g++ under
AddressSanitizer and UBSan with the matrix product emulated lane by lane,
against the oracle.

Tolerances: the fit stops at a remainder of 2^-22 = 2.4e-7 of each plane's
kernel; the bodies are held to the 1e-5 per projection of the GPU parity
tests."""
from __future__ import annotations

import os
import shutil
import subprocess

import numpy as np
import pytest
import torch

from oracle import spect_oracle as so
from tests.helpers import oracle_geometry, problem_arrays, rel_l2
from tests.test_kernel_cpu_build import ROOT, _exec, _write_problem


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("lowrank_cpu") / "lowrank_cpu")
    cmd = [gxx, "-std=c++20", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
           "-fno-omit-frame-pointer", "-pthread", "-Wno-attributes", "-Wno-unknown-pragmas",
           "-I", os.path.join(ROOT, "tests", "cpu_build"), "-I", os.path.join(ROOT, "pytomography_amd", "csrc"),
           os.path.join(ROOT, "tests", "cpu_build", "lowrank_cpu.cpp"), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0 and "barrier" in r.stderr:
        pytest.skip("the host compiler lacks C++20 <barrier>")
    assert r.returncode == 0, r.stderr[-4000:]
    return out


CASES = [
    # name, problem, angles, attenuation mode (0 none, 1 field), row tiles of a forward wave
    # (with four, the back projection takes five)
    ("one_segment", dict(n=16, n_angles=8, psf=True), [0, 3], 0, 4),
    ("field_odd_ragged", dict(n=21, n_angles=9, psf=True, att=True, nz=13), [1, 4, 8], 1, 2),
    ("field_two_z_blocks", dict(n=17, n_angles=7, psf=True, att=True, nz=68), [2], 1, 1),
    ("two_row_ranges", dict(n=66, n_angles=12, psf=True, att=True, nz=5), [2], 1, 2),
    ("several_segments", dict(n=52, n_angles=12, psf=True, att=True, nz=8), [2, 7], 1, 4),
    ("single_slice", dict(n=12, n_angles=5, psf=True, nz=1), [0, 2], 0, 1),
    # 37 taps: the blur matrices reach two tiles to either side
    ("wide_psf", dict(n=24, n_angles=7, psf=True, nz=20, radius=75.0), [3], 0, 2),
    ("wide_psf_tall", dict(n=70, n_angles=7, psf=True, nz=3, radius=75.0), [3], 0, 4),
]


@pytest.mark.parametrize("name,spec,sel,att_mode,row_tiles", CASES, ids=[c[0] for c in CASES])
def test_lowrank_bodies_match_oracle(exe, tmp_path, name, spec, sel, att_mode, row_tiles):
    spec = dict(spec)
    radius = spec.pop("radius", 25.0)
    pa = problem_arrays(spec.pop("n"), spec.pop("n_angles"), seed=5, **spec)
    # a body-contour orbit: every angle has a radius, and so an image basis, of its own
    pa["radii"] = radius + 2.0 * np.cos(2 * np.deg2rad(pa["angles"]))
    _write_problem(tmp_path, pa, sel, att_mode=att_mode)
    np.ascontiguousarray(pa["f"], dtype=np.float32).tofile(tmp_path / "f.bin")
    rng = np.random.default_rng(3)
    p = (0.5 + rng.random((len(sel), pa["n"], pa["nz"]))).astype(np.float32)
    p.tofile(tmp_path / "p.bin")
    stats = _exec(exe, tmp_path, [str(row_tiles)])
    proj = torch.from_numpy(np.fromfile(tmp_path / "proj.bin", dtype=np.float32).reshape(p.shape))
    bp = torch.from_numpy(np.fromfile(tmp_path / "bp.bin", dtype=np.float32).reshape(pa["f"].shape))
    g = oracle_geometry(pa, torch.float64)
    ref = so.forward(g, torch.from_numpy(pa["f"]).double(), torch.tensor(sel))
    ref_b = so.backward(g, torch.from_numpy(p).double(), torch.tensor(sel))
    errs = [rel_l2(proj[k], ref[k]) for k in range(len(sel))]
    print(f"{name}: {stats}, forward {max(errs):.1e}, back projection {rel_l2(bp, ref_b):.1e}")
    assert stats["uncovered"] == 0
    assert bool(torch.isfinite(proj).all()) and bool(torch.isfinite(bp).all())
    assert bool((proj >= 0).all()) and bool((bp >= 0).all())
    assert max(errs) <= 1e-5 and rel_l2(bp, ref_b) <= 1e-5
