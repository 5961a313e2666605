"""The arrays of a scene on a device (here the CPU): their types, values and
shapes, in one copy and in one copy each."""
import numpy as np
import pytest
import torch

from distance3d_amd import scene as sc
from distance3d_amd.scene import SceneBuilder

TYPES = {"shape_f64": torch.float64, "shape_i32": torch.int32, "vx": torch.float32, "vy": torch.float32,
         "vz": torch.float32, "v64": torch.float64}


@pytest.mark.parametrize("packed", (True, False))
@pytest.mark.parametrize("hulls", (True, False))
def test_arrays_of_other_types_are_converted(monkeypatch, packed, hulls):
    if not packed:
        monkeypatch.setattr(sc, "PACKED_UPLOAD_MAX", 0)
    b = SceneBuilder()
    b.add_sphere(np.array([1.0, 2.0, 3.0]), 0.5)
    if hulls:
        b.add_hull(np.random.RandomState(0).randint(-9, 9, (70, 3)).astype(float))
    host = b.build()
    want = {name: getattr(host, name).copy() for name in TYPES}
    host.shape_i32 = host.shape_i32.astype(np.int64)
    host.shape_f64 = np.asfortranarray(host.shape_f64)
    host.vx = host.vx.astype(np.float64)
    host.vy = np.repeat(host.vy, 2)[::2]
    dev = sc.DeviceScene(host, "cpu", cluster_min=0)
    for name, dtype in TYPES.items():
        got = getattr(dev, name)
        assert got.dtype == dtype and got.is_contiguous()
        expected = want[name] if len(want[name]) else np.zeros((1,) + want[name].shape[1:])
        assert np.array_equal(got.numpy(), expected)
    assert dev.vorig is None and dev.clusters is None
