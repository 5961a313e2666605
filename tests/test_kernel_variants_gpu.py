"""Kernel variants chosen by size, at the sizes where they change: edges of
tiles and groups, remainders, the smallest and the largest of each range,
against the oracle.  Every compared value is exact (a selection, a comparison
or the oracle's own operations in its order), so equality is bitwise."""
import numpy as np
import pytest

from distance3d_amd import kernels
from distance3d_amd.scene import SceneBuilder
from oracle import oracle
from tests import geometry_brute as gb

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def box_scene(gpu):
    """Hulls around the lane-serial limit, the wavefront width and several
    sweeps long, in FP32 and FP64, with and without margin, between analytic
    colliders."""
    rs = np.random.RandomState(31)
    b = SceneBuilder()
    for k, nv in enumerate((1, 4, 15, 16, 17, 63, 64, 65, 129, 256, 1000, 4096)):
        T = gb.random_pose(rs)
        v = rs.randn(nv, 3)
        b.add_hull(v.astype(np.float32), T[:3, :3], T[:3, 3], margin=0.1 * (k % 2))
        b.add_hull(v, T[:3, :3], T[:3, 3])
        b.add_box(T, rs.uniform(0.1, 1.0, 3))
        b.add_capsule(T, 0.2, 0.7, margin=0.05)
    return b.build()


@pytest.mark.parametrize("n", (1, 3, 4, 5, 17, 48, 65535, 65536, 65555, 524287, 524289))
def test_aabbs_of_mixed_hulls(box_scene, n):
    ids = (np.arange(n) * 7 % box_scene.n_shapes).astype(np.int32)
    ids[-1] = 4 * 11  # the largest hull, in the last tile
    got = kernels.aabb_batch(box_scene.to_device(), ids).cpu().numpy()
    want = oracle.aabbs(box_scene, np.arange(box_scene.n_shapes, dtype=np.int32))
    assert np.array_equal(got, want[ids])
