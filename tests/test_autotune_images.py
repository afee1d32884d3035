"""The autotuners where the tuned calls blur combined images: the library's own
choice, without timing; and what a cached answer stands for."""
import json

import pytest
import torch

import pytomography_amd
from pytomography_amd import batch


class _Matrix:
    def __init__(self, images, forward="images", field="images"):
        self.combined_images, self._schedule = images, {"forward": forward, "field": field}

    def set_n_subsets(self, n):
        self.n_subsets = n

    def schedule(self, subset):
        assert self.n_subsets == 4 and subset == 0
        return self._schedule


@pytest.fixture()
def timed(tmp_path, monkeypatch):
    """Candidates that were timed: the last one is the fastest."""
    out = []
    monkeypatch.setattr(batch, "_CACHE_PATH", str(tmp_path / "autotune.json"))
    monkeypatch.setattr(batch, "_cache", None)
    monkeypatch.setattr(batch.torch.cuda, "get_device_name", lambda device=None: "test device")

    def seconds(sm, *args):
        out.append(sm)
        return -len(out)

    monkeypatch.setattr(batch, "_osem_step_seconds", seconds)
    monkeypatch.setattr(batch, "_batch_iteration_seconds", seconds)
    return out


def test_images_are_not_timed(timed, tmp_path):
    args = (32, 16, 4)
    assert batch.autotune_chunk_planes(lambda c: _Matrix(True), *args, key="k", device="cpu") == 16
    assert batch.autotune_schedule(lambda c, r: _Matrix(True), *args, key="k", device="cpu") == (0, 0)
    assert batch.autotune_chunk_planes(lambda c: _Matrix(True), *args, key="k", device="cpu", candidates=(8, 24)) == 8
    assert not timed and not (tmp_path / "autotune.json").exists()


def test_planes_are_timed(timed):
    args = (32, 16, 4)
    assert batch.autotune_chunk_planes(lambda c: _Matrix(False), *args, key="k", device="cpu") == 32
    assert batch.autotune_schedule(lambda c, r: _Matrix(False), *args, key="k", device="cpu") == (32, -1)
    n = len(timed)
    # forward on images, back projection by planes: its schedule is still a choice
    part = lambda c: _Matrix(True, field="uniform")
    assert batch.autotune_chunk_planes(part, *args, key="j", device="cpu") == 32
    n = len(timed)
    partly = batch.autotune_schedule(lambda c, r: _Matrix(True, field="uniform"), *args, key="j", device="cpu")
    assert partly == (32, -1) and len(timed) == n + len(batch.SCHEDULE_CANDIDATES)


def test_cached_answers_are_kept_apart_by_dtype(timed, tmp_path, monkeypatch):
    tune = lambda: batch.autotune_chunk_planes(lambda c: _Matrix(False), 32, 16, 4, key="k", device="cpu")
    tune()
    n = len(timed)
    tune()
    assert len(timed) == n
    monkeypatch.setattr(pytomography_amd, "dtype", torch.float64)
    tune()
    assert len(timed) == 2 * n and len(json.loads((tmp_path / "autotune.json").read_text())) == 2
