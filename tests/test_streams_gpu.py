"""Batch calls that take turns on several streams, with no wait between them,
against the oracle: no call's scratch, copies or counts are another stream's."""
import numpy as np
import pytest
import torch

from distance3d_amd import kernels, workloads
from distance3d_amd.scene import collider_centers
from oracle import oracle

pytestmark = pytest.mark.gpu

SIZES = (5000, 37, 12001, 300, 4096, 2)


@pytest.fixture(scope="module")
def streams(gpu):
    return [None, torch.cuda.Stream(), torch.cuda.Stream()]


@pytest.fixture(scope="module")
def batches(gpu):
    """A resident scene, and pair lists of several sizes with their centres."""
    host = workloads.mixed_pairs(seed=21, n_pairs=400).scene
    host.shape_f64[:, 9:12] *= 0.6
    rs = np.random.RandomState(0)
    lists = [rs.randint(0, host.n_shapes, (2, n)).astype(np.int32) for n in SIZES]
    return host, host.to_device(), lists, collider_centers(host)


def _in_turn(streams, lists, call):
    """call(pair_a, pair_b, stream) for every list on every stream, twice over,
    waited for at the end alone."""
    dev = [tuple(torch.from_numpy(x).cuda() for x in ab) for ab in lists]
    torch.cuda.synchronize()
    got = [(k, call(a, b, streams[(k + r) % len(streams)]))
           for r in range(2 * len(streams)) for k, (a, b) in enumerate(dev)]
    torch.cuda.synchronize()
    return got


def test_intersections(streams, batches):
    host, dev, lists, _ = batches
    want = [oracle.gjk_intersection(host, a, b)[0] for a, b in lists]
    for k, (hit, _) in _in_turn(streams, lists,
                                lambda a, b, s: kernels.gjk_intersection_batch(dev, a, b, stream=s)):
        assert np.array_equal(hit.cpu().numpy(), want[k])


def test_mpr(streams, batches):
    host, dev, lists, centers = batches
    c = torch.from_numpy(centers).cuda()
    want = [oracle.mpr(host, a, b, centers) for a, b in lists]
    for k, got in _in_turn(streams, lists, lambda a, b, s: kernels.mpr_batch(dev, a, b, c, stream=s)):
        for g, w in zip(got, want[k]):
            assert np.array_equal(g.cpu().numpy(), w, equal_nan=True)


def test_gjk_and_epa(streams, batches):
    host, dev, lists, _ = batches
    want = [oracle.gjk_distance(host, a, b)["dist"] for a, b in lists]
    for k, out in _in_turn(streams, lists, lambda a, b, s: kernels.gjk_epa_batch(dev, a, b, stream=s)):
        assert np.array_equal(out.dist.cpu().numpy(), want[k])
