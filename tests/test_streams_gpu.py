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


def _boxes(rs, n, size):
    lo = rs.uniform(0.0, 10.0, (n, 3))
    return np.stack([lo, lo + rs.uniform(0.1, size, (n, 3))], axis=2)


@pytest.mark.parametrize("call", ("dense", "sorted", "unsorted", "long lists"))
@pytest.mark.parametrize("cap", (None, 1))
def test_box_overlaps(streams, call, cap):
    """Counts read back from a stream that is behind the caller's: with room for
    all pairs and for one at first."""
    rs = np.random.RandomState(3)
    boxes = [_boxes(rs, n, 0.7) for n in (900, 3000)]
    queries = [_boxes(rs, n, 3.0 if call != "long lists" else 12.0) for n in (40, 200)]
    for q, b in zip(queries, boxes):
        q[0] = b[0]
    ahead = torch.zeros(1 << 24, device="cuda")
    for s in streams:
        for q, b in zip(queries, boxes):
            want, _ = oracle.all_aabbs_overlap(q, b)
            want = want[np.lexsort((want[:, 1], want[:, 0]))]
            db, dq = torch.from_numpy(b).cuda(), torch.from_numpy(q).cuda()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                for _ in range(20):
                    ahead.add_(1.0)
            if call == "dense":
                got = kernels.overlap_dense(dq, db, cap=cap, stream=s)
            else:
                bvh = kernels.bvh_build(db, stream=s)
                got = kernels.bvh_query(bvh, dq, cap=cap, sort=call != "unsorted", stream=s)
            torch.cuda.synchronize()
            got = got.cpu().numpy()
            if call == "unsorted":
                got = got[np.lexsort((got[:, 1], got[:, 0]))]
            assert np.array_equal(got, want)


@pytest.mark.parametrize("n", (20, 300, 9000))
def test_captured_batches(batches, n):
    """Intersection and MPR in a captured graph, scratch and all: replays with new
    pairs, and eager calls of another size between them."""
    host, dev, _, centers = batches
    c = torch.from_numpy(centers).cuda()
    rs = np.random.RandomState(n)
    a, b = (torch.from_numpy(rs.randint(0, host.n_shapes, n).astype(np.int32)).cuda() for _ in range(2))
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        kernels.gjk_intersection_batch(dev, a, b)
        kernels.mpr_batch(dev, a, b, c)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        hit, _ = kernels.gjk_intersection_batch(dev, a, b)
        status, out = kernels.mpr_batch(dev, a, b, c)
    for _ in range(4):
        pa, pb = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
        a.copy_(torch.from_numpy(pa))
        b.copy_(torch.from_numpy(pb))
        graph.replay()
        kernels.gjk_intersection_batch(dev, np.repeat(pa, 2), np.repeat(pb, 2))
        torch.cuda.synchronize()
        assert np.array_equal(hit.cpu().numpy(), oracle.gjk_intersection(host, pa, pb)[0])
        want = oracle.mpr(host, pa, pb, centers)
        assert np.array_equal(status.cpu().numpy(), want[0])
        assert np.array_equal(out.cpu().numpy(), want[1], equal_nan=True)
