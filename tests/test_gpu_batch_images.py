"""Batched OSEM against one-at-a-time OSEM, by planes and on combined images, on
both sides of the size from which a back projection runs on images (41000
samples of the extended detector: of one call, or of a whole batch launch).

The system matrices use uniform plane chunks, as a batch does, so a batch whose
calls choose as the single ones do has their bits.  Otherwise the two differ by
the images' error of one back projection per sub-iteration, 5e-6 as in
test_gpu_combined_images.py: 8 x 5e-6 in relative L2."""
from __future__ import annotations

import pytest
import torch

from pytomography_amd import synthetic
from tests.helpers import problem_arrays, product_system_matrix, rel_l2

pytestmark = pytest.mark.gpu

SUBSETS, ITERS = 4, 2
# side, angles, members, images, does a single call's back projection run them, does the batch's
CASES = {
    "planes": (32, 16, 2, False, False, False),
    "few_samples": (32, 16, 2, True, False, False),
    "few_alone_many_together": (48, 32, 2, True, False, True),
    "many_samples": (64, 32, 1, True, True, True),
}


@pytest.mark.parametrize("name", CASES)
def test_batch_matches_single_calls(name):
    from pytomography_amd.algorithms import OSEM
    from pytomography_amd.batch import BatchedOSEM
    from pytomography_amd.likelihoods import PoissonLogLikelihood
    n, n_angles, members, images, single, batched = CASES[name]

    def likelihoods():
        out = []
        for k in range(members):
            pa = problem_arrays(n, n_angles, seed=k, att=True, psf=True)
            sm = product_system_matrix(pa, sched_rounds=-1)
            sm.combined_images = images  # as the constructor's argument, before the first plan
            sm.set_n_subsets(SUBSETS)
            f = torch.from_numpy(pa["f"]).cuda()
            exp = sm._project(f, None, "spect_forward", planes=True) * 100
            s = torch.full_like(exp, 0.05 * float(exp.mean()))
            want = {"forward": "images" if images else "uniform", "field": "images" if single else "uniform"}
            assert sm.schedule(0) == want
            out.append(PoissonLogLikelihood(sm, synthetic.poisson_data(exp + s, k), additive_term=s))
        return out

    ref = [OSEM(lk)(ITERS, SUBSETS).clone() for lk in likelihoods()]
    got = BatchedOSEM(likelihoods(), SUBSETS, use_graph=False).run(ITERS)
    torch.cuda.synchronize()
    for a, b in zip(got, ref):
        print(f"[{name}] rel-L2 {rel_l2(a, b):.1e}")
        if single == batched:
            assert torch.equal(a, b)
        else:
            assert not torch.equal(a, b) and rel_l2(a, b) <= SUBSETS * ITERS * 5e-6
