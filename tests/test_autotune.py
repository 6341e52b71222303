"""The autotuner's walk over launch shapes, with a stand-in for the batch and
its timing (no device)."""
import pytest
import torch

from pysph_amd import autotune
from pysph_amd.batch import TUNE_FIELDS


class _Batch:
    dim, precision, nsims, n, device, steps_done = 2, "double", 3, 5000, "cuda:0", 0

    def __init__(self):
        self.shape = {k: 0 for k in TUNE_FIELDS}

    def tuning(self):
        return dict(self.shape)

    def set_tuning(self, tune):
        self.shape.update(tune)

    def snapshot(self):
        return None

    def restore(self, snap):
        pass

    check = synchronize = lambda self: None


@pytest.fixture
def batch(monkeypatch, tmp_path):
    monkeypatch.setenv("PYSPH_AMD_CACHE", str(tmp_path))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda device: "stand in")
    return _Batch()


def test_walk_starts_from_what_an_untuned_batch_runs(batch, monkeypatch):
    """The library picks the block size by the batch's size: a walk over
    another field leaves that choice to it."""
    untuned = batch.tuning()
    monkeypatch.setattr(autotune, "time_steps",
                        lambda sim, steps, dt: 2.0 if sim.shape["nbr_tile"] == 2 else 3.0)
    res = autotune.autotune(batch, space={"nbr_tile": (1, 2, 4)})
    assert res["trials"][0][0] == untuned
    assert res["tuning"] == dict(untuned, nbr_tile=2) == batch.tuning()


def test_shapes_tuned_for_other_kernels_are_not_used(batch, monkeypatch, tmp_path):
    monkeypatch.setattr(autotune, "time_steps", lambda sim, steps, dt: 1.0)
    space = {"nbr_tile": (1, 2)}
    assert not autotune.autotune(batch, space=space)["cached"]
    assert autotune.autotune(_Batch(), space=space)["cached"]
    (tmp_path / "csrc").mkdir()
    (tmp_path / "csrc" / "other.hip").write_text("// other kernels")
    monkeypatch.setattr(autotune, "CSRC", str(tmp_path / "csrc"), raising=False)
    assert not autotune.autotune(_Batch(), space=space)["cached"]
