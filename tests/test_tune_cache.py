"""Launch shapes cached on disk belong to the kernels that were timed: another build of the library
tunes again.  The batch is a stand-in that stops where tuning would begin."""
import json

import pytest
import torch

from fanbeamctrecon_tensorflowop_amd import _lib
from fanbeamctrecon_tensorflowop_amd import batch as B

SHAPE = dict(fp_rays=64, fp_wgs_per_cu=8, adj_tile_x=16, adj_wgs_per_cu=8, adj_stage_views=0)


class Tuning(Exception):
    pass


class Batch:
    shape = None

    def signature(self):
        return "geometry"

    def set_shape(self, **kw):
        self.shape = kw

    def upload(self):
        raise Tuning


def _tune(b):
    return B.autotune(b, torch.zeros(1), torch.zeros(1, dtype=torch.bfloat16))


@pytest.fixture
def cache(tmp_path, monkeypatch):
    path = tmp_path / "shapes.json"
    monkeypatch.setenv("FBCT_TUNE_CACHE", str(path))
    monkeypatch.setattr(torch.cuda, "get_device_name", lambda dev=None: "device")
    return path


def test_shapes_of_unknown_kernels_are_not_used(cache):
    # entries as they were before they named the library
    cache.write_text(json.dumps({"device|geometry|torch.float32|torch.bfloat16":
                                 {"shape": SHAPE, "fp_ms": 1.0, "adj_ms": 1.0}}))
    with pytest.raises(Tuning):
        _tune(Batch())


def test_shapes_of_another_build_are_not_used(cache, tmp_path, monkeypatch):
    other = tmp_path / "libfbct.so"
    other.write_bytes(b"another build")
    args = (Batch(), torch.zeros(1), torch.zeros(1, dtype=torch.bfloat16))
    B._store_cache(str(cache), B._tune_key(*args), {"shape": SHAPE, "fp_ms": 1.0, "adj_ms": 1.0})
    b = Batch()
    assert _tune(b)["cached"] and b.shape == SHAPE
    monkeypatch.setattr(_lib, "LIB_PATH", str(other))
    with pytest.raises(Tuning):
        _tune(Batch())
