"""spect_forward_noalloc on combined images, where the images of all angles do
not fit its scratch and the angles run in groups: the bits of spect_forward."""
from __future__ import annotations

import pytest
import torch

from pytomography_amd import _lib
from tests.helpers import problem_arrays, product_system_matrix

pytestmark = pytest.mark.gpu


# 128^3: two segments of 16 images of 12 x 8 tiles of 1 KB an angle, 3.1 MB, so 42
# angles fit the 128 MiB; 43 and 65 angles run in two groups, 60 in equal ones
@pytest.mark.parametrize("n_angles,att", [(43, False), (60, True), (65, False)])
def test_groups_of_angles_equal_one_call(n_angles, att):
    pa = problem_arrays(128, n_angles, seed=1, att=att, psf=True)
    sm = product_system_matrix(pa)
    sm.combined_images = True  # as the constructor's argument, before the first plan
    assert sm.schedule()["forward"] == "images"
    assert 32 * 12 * 8 * 1024 * n_angles > _lib.NOALLOC_SCRATCH_BYTES
    dev = torch.device("cuda", torch.cuda.current_device())
    f = torch.from_numpy(pa["f"]).to(dev)
    want = sm.forward(f)
    plan, idx = sm._plan(dev), sm._angle_index(None, dev)
    mu, tab = sm._mu(dev, torch.float32), sm._att_table(dev, torch.float32)
    got = torch.full_like(want, float("nan"))
    print(f"{n_angles} angles", flush=True)
    _lib.check(plan.lib.spect_forward_noalloc(
        plan.handle, sm._code(torch.float32, tab), f.data_ptr(), _lib.ptr(mu), _lib.ptr(tab),
        idx.data_ptr(), n_angles, got.data_ptr(), _lib.stream_ptr(dev)))
    torch.cuda.synchronize()
    assert torch.equal(got, want)
