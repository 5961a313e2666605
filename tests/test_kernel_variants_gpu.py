"""Kernel variants chosen by size, at the sizes where they change: edges of
tiles and groups, remainders, the smallest and the largest of each range,
against the oracle.  Every compared value is exact (a selection, a comparison
or the oracle's own operations in its order), so equality is bitwise."""
import numpy as np
import pytest
import torch

from distance3d_amd import kernels, workloads
from distance3d_amd.scene import SceneBuilder, collider_centers
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


def _boxes(rs, n, extent, wmax):
    lo = rs.uniform(0.0, extent, (n, 3))
    return np.stack([lo, lo + rs.uniform(0.01, wmax, (n, 3))], axis=2)


def _overlaps(boxes, queries):
    p, _ = oracle.all_aabbs_overlap(queries, boxes)
    return p[np.lexsort((p[:, 1], p[:, 0]))]


@pytest.mark.parametrize("n", (1, 7, 8, 9, 64, 65, 511, 513, 4095, 4097, 32769, 393215, 393217))
def test_box_tree_levels(gpu, n):
    """Trees around every level's edge and both sort tiles, with empty, NaN and
    infinite boxes among them; again after a refit with new boxes."""
    rs = np.random.RandomState(n)
    extent = max(1.0, n ** (1.0 / 3.0))
    boxes = _boxes(rs, n, extent, 0.8)
    boxes[n // 2, 1, 1] = np.inf
    boxes[n // 3, 0, 0] = np.nan
    boxes[n // 5] = boxes[n // 5][:, ::-1]
    queries = _boxes(rs, 67, extent, 1.5)
    queries[3] = [[-np.inf, np.inf]] * 3 if n <= 513 else queries[3]
    bvh = kernels.bvh_build(boxes)
    assert np.array_equal(kernels.bvh_query(bvh, queries).cpu().numpy(), _overlaps(boxes, queries))
    moved = boxes + rs.uniform(-1.0, 1.0, (n, 3, 1))
    kernels.bvh_refit(bvh, moved)
    assert np.array_equal(kernels.bvh_query(bvh, queries).cpu().numpy(), _overlaps(moved, queries))


@pytest.mark.parametrize("m", (1, 3, 4, 5, 8191, 8192, 8203, 49151, 49152, 49183))
def test_box_queries_by_lane_count(gpu, m):
    """Every query width at its edges; lists shorter and longer than a query's
    rows, sorted, unsorted and with too little room at first."""
    rs = np.random.RandomState(m)
    boxes = _boxes(rs, 600, 10.0, 0.5)
    boxes[:40] = [[4.0, 4.5]] * 3  # lists of forty and more
    queries = _boxes(rs, m, 10.0, 0.4)
    queries[m // 2] = [[4.2, 4.3]] * 3
    want = _overlaps(boxes, queries)
    bvh = kernels.bvh_build(boxes)
    assert np.array_equal(kernels.bvh_query(bvh, queries).cpu().numpy(), want)
    assert np.array_equal(kernels.bvh_query(bvh, queries, cap=1).cpu().numpy(), want)
    got = kernels.bvh_query(bvh, queries, sort=False).cpu().numpy()
    assert np.array_equal(got[np.lexsort((got[:, 1], got[:, 0]))], want)


@pytest.mark.parametrize("k", (15, 16, 17, 1023, 1024, 1025, 3000))
def test_box_query_list_lengths(gpu, k):
    """One query's list at the row limit and around the longest list that is
    ordered by counting."""
    boxes = np.zeros((k, 3, 2))
    boxes[:, :, 1] = 1.0 + np.arange(k)[:, None]
    queries = np.array([[[0.5, 0.6]] * 3, [[-2.0, -1.0]] * 3])
    got = kernels.bvh_query(kernels.bvh_build(boxes), queries).cpu().numpy()
    assert np.array_equal(got, np.stack([np.zeros(k, int), np.arange(k)], 1))


@pytest.mark.parametrize("n", (1, 15, 16, 17, 300, 5000))
@pytest.mark.parametrize("kind", ("mixed", "near", "analytic"))
def test_intersection_by_batch_size(gpu, kind, n):
    """Both intersection kernels at the line between them, over every work
    class, an invalid pair, a collider against itself and an iteration cap: hits
    against the oracle, statuses against the lane-per-pair kernel's."""
    if kind == "analytic":
        host = workloads.broad_phase_scene(n_boxes=600, n_capsules=100, extent=4.0).scene
    else:
        host = workloads.mixed_pairs(seed=5, n_pairs=350).scene
        if kind == "near":
            host.shape_f64[:, 9:12] *= 0.4
    rs = np.random.RandomState(n)
    a, b = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
    dev = host.to_device()
    for cap in (128, 2):
        hit, status = kernels.gjk_intersection_batch(dev, a, b, max_iterations=cap, want_status=True)
        want = oracle.gjk_intersection(host, a, b, max_iterations=cap)[0]  # -1 at the cap
        assert np.array_equal(hit.cpu().numpy(), want == 1)
        assert np.array_equal(status.cpu().numpy() == 4, want == -1)
        da, db = (torch.as_tensor(x, device="cuda") for x in (a, b))
        lane_hit, lane_status = torch.empty_like(hit), torch.empty_like(status)
        kernels.check(kernels.lib().d3d_gjk_intersection_batch(
            dev.c, kernels.ptr(da), kernels.ptr(db), n, 1e-10, cap, kernels.ptr(lane_hit),
            kernels.ptr(lane_status), kernels.stream_ptr()), "d3d_gjk_intersection_batch")
        assert torch.equal(hit, lane_hit) and torch.equal(status, lane_status)
    a[-1] = host.n_shapes
    hit, status = kernels.gjk_intersection_batch(dev, a, b, want_status=True)
    assert int(hit[-1]) == 0 and int(status[-1]) == 0x200


@pytest.mark.parametrize("n", (1, 1023, 1025, 4095, 4096, 4097, 65535, 65537, 196607, 196609, 786431,
                               786433))
def test_pair_sort_by_batch_size(gpu, n):
    """GJK distance and intersection on both sides of the one-block sort and of
    the tile sizes, with invalid pairs: every pair is taken exactly once."""
    host = workloads.mixed_pairs(seed=9, n_pairs=200).scene
    rs = np.random.RandomState(n)
    a, b = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
    bad = rs.rand(n) < 0.01
    a[bad] = host.n_shapes + 3
    dev = host.to_device()
    out = kernels.gjk_distance_batch(dev, a, b)
    hit, _ = kernels.gjk_intersection_batch(dev, a, b)
    ok = ~bad
    want = oracle.gjk_distance(host, a[ok], b[ok])
    assert np.array_equal(out.dist.cpu().numpy()[ok], want["dist"])
    assert np.array_equal(out.status.cpu().numpy()[bad], np.full(bad.sum(), 0x200))
    assert np.array_equal(hit.cpu().numpy()[ok], oracle.gjk_intersection(host, a[ok], b[ok])[0])
    assert not hit.cpu().numpy()[bad].any()


@pytest.mark.parametrize("m", (1, 63, 64, 65, 200, 131072 + 65))
def test_tet_pairs_by_batch_size(gpu, m):
    """Pairs that wait to be clipped: a single tile, several tiles per block, a
    last partial queue; coinciding tetrahedra and pairs the plane misses among
    them, with and without planes and polygons."""
    rs = np.random.RandomState(m)
    n = 50
    bodies = []
    for _ in range(2):
        T = rs.uniform(-0.6, 0.6, (n, 1, 3)) + 0.5 * rs.randn(n, 4, 3)
        e = rs.uniform(0.0, 1.0, (n, 4))
        bodies.append([T, e])
    bodies[1][0][:10], bodies[1][1][:10] = bodies[0][0][:10], bodies[0][1][:10]
    X = [oracle.tet_mesh_prep(T)[1] for T, _ in bodies]
    pairs = rs.randint(0, n, (m, 2)).astype(np.int32)
    pairs[::7, 1] = pairs[::7, 0]
    (T1, e1), (T2, e2) = bodies
    used, inverse = np.unique(pairs, axis=0, return_inverse=True)
    want = [x[inverse.reshape(-1)] for x in oracle.tet_pairs(T1, e1, X[0], T2, e2, X[1], used)]
    for geometry in (True, False):
        got = kernels.tet_pairs_batch(T1, e1, X[0], T2, e2, X[1], pairs, geometry=geometry)
        for g, w in zip(got, want):
            if g is not None:
                assert np.array_equal(g.cpu().numpy(), w, equal_nan=True)


@pytest.mark.parametrize("n", (1, 31, 32, 33, 300, 5000))
@pytest.mark.parametrize("kind", ("mixed", "near", "same"))
def test_mpr_by_batch_size(gpu, kind, n):
    """Both MPR kernels at the line between them, over every work class, with
    coinciding centres, a refinement cap and an invalid pair, with and without
    penetration."""
    host = workloads.mixed_pairs(seed=6, n_pairs=350).scene
    host.shape_f64[:, 9:12] *= {"mixed": 1.0, "near": 0.4, "same": 0.0}[kind]
    rs = np.random.RandomState(n)
    a, b = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
    centers = collider_centers(host)
    dev = host.to_device()
    for cap in (100, 1):
        want = oracle.mpr(host, a, b, centers, max_iterations=cap)
        got = kernels.mpr_batch(dev, a, b, centers, max_iterations=cap)
        for g, w in zip(got, want):
            assert np.array_equal(g.cpu().numpy(), w, equal_nan=True)
        status, out = kernels.mpr_batch(dev, a, b, centers, max_iterations=cap, penetration=False)
        want = oracle.mpr(host, a, b, centers, max_iterations=cap, penetration=False)
        assert out is None and np.array_equal(status.cpu().numpy(), want[0])
    a[-1] = host.n_shapes
    status, out = kernels.mpr_batch(dev, a, b, centers)
    assert int(status[-1]) == 0x200 and bool(torch.isnan(out[-1]).all())


@pytest.mark.parametrize("n", (65535, 65536, 65537))
def test_intersection_large_batches(gpu, n):
    """The intersection's two occupancies at the line between them."""
    host = workloads.mixed_pairs(seed=11, n_pairs=100).scene
    rs = np.random.RandomState(n)
    a, b = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
    hit, _ = kernels.gjk_intersection_batch(host.to_device(), a, b)
    assert np.array_equal(hit.cpu().numpy(), oracle.gjk_intersection(host, a, b)[0])


@pytest.mark.parametrize("boxes, queries, spread", [(1, 1, 0.0), (40, 300, 0.1), (600, 9, 0.1), (20000, 9001, 3.0),
                                                    (3000, 50001, 8.0)])
def test_unordered_query_is_the_ordered_set(boxes, queries, spread):
    """A block's hits below, at and far above what it gathers at once, for each
    number of lanes per query, with room for all pairs and for few at first."""
    rng = np.random.default_rng(boxes)
    lo = rng.uniform(-spread, spread, (boxes + queries, 3))
    ab = np.stack([lo, lo + rng.uniform(0.05, 0.5, lo.shape)], axis=2)
    bvh = kernels.bvh_build(torch.from_numpy(ab[:boxes]).cuda())
    q = torch.from_numpy(ab[boxes:]).cuda()
    want = kernels.bvh_query(bvh, q).cpu().numpy()
    for cap in (None, 5):
        got = kernels.bvh_query(bvh, q, cap=cap, sort=False).cpu().numpy()
        np.testing.assert_array_equal(got[np.lexsort((got[:, 1], got[:, 0]))], want)


@pytest.mark.parametrize("n", (1, 63, 64, 65, 255, 257, 65535, 65537, 524289))
def test_aabbs_without_hulls(gpu, n):
    """A scene without hull vertices, on both sides of the sizes at which one
    with hulls changes its colliders per wavefront."""
    host = workloads.broad_phase_scene(n_boxes=50, n_capsules=20, extent=4.0).scene
    ids = (np.arange(n) * 7 % host.n_shapes).astype(np.int32)
    got = kernels.aabb_batch(host.to_device(), ids).cpu().numpy()
    want = oracle.aabbs(host, np.arange(host.n_shapes, dtype=np.int32))
    assert np.array_equal(got, want[ids])


def test_query_of_more_than_one_launch(gpu):
    """More unordered queries than one launch has threads for (8 lanes each):
    the last ones, far away from the empty rest, are found."""
    m = (1 << 29) + 5
    q = torch.full((m, 3, 2), 100.0, dtype=torch.float64, device="cuda")
    at = torch.tensor([0, 7, (1 << 29) - 33, (1 << 29) - 32, 1 << 29, m - 1], device="cuda")
    q[at] = torch.tensor([[0.5, 0.6]] * 3, dtype=torch.float64, device="cuda")
    boxes = np.array([[[0.0, 1.0]] * 3, [[2.0, 3.0]] * 3])
    got = kernels.bvh_query(kernels.bvh_build(boxes), q, cap=64, sort=False)
    del q
    assert torch.equal(got[torch.argsort(got[:, 0])].long(), torch.stack([at, torch.zeros_like(at)], 1))


@pytest.mark.parametrize("n", (300, 4096, 4097))
@pytest.mark.parametrize("blocks", (1, 2, 3))
def test_distance_by_blocks_per_cu(gpu, n, blocks):
    """A caller's blocks per compute unit, on both sides of the size at which the
    default changes."""
    host = workloads.mixed_pairs(seed=12, n_pairs=200).scene
    a, b = np.random.RandomState(n).randint(0, host.n_shapes, (2, n)).astype(np.int32)
    out = kernels.gjk_distance_batch(host.to_device(), a, b, launch={"blocks_per_cu": blocks})
    want = oracle.gjk_distance(host, a, b)
    assert np.array_equal(out.dist.cpu().numpy(), want["dist"])


@pytest.mark.parametrize("hits", (0, 1, 5, 40, 550, 1050, 2000))
def test_ordered_pairs_hold_little_spare_room(gpu, hits):
    """What a caller keeps of an ordered query is at most 8 times its pairs or 64
    KiB, for short, long and sorted lists."""
    boxes = np.zeros((max(hits, 1), 3, 2))
    boxes[:, :, 1] = 1.0
    queries = np.full((3000, 3, 2), 50.0)
    if hits:
        queries[7] = [0.5, 0.6]
    pairs = kernels.bvh_query(kernels.bvh_build(boxes), queries)
    assert np.array_equal(pairs.cpu().numpy(), np.stack([np.full(hits, 7), np.arange(hits)], 1))
    assert pairs.untyped_storage().nbytes() <= max(64 * hits, 1 << 16)


def test_ordered_pairs_of_a_large_batch(gpu):
    """Enough queries for the smaller room per query, with short and long lists."""
    m = 400003
    rs = np.random.RandomState(4)
    boxes = _boxes(rs, 500, 30.0, 0.8)
    boxes[:30] = [[4.0, 4.5]] * 3
    queries = _boxes(rs, m, 30.0, 0.8)
    queries[::50000] = [[4.2, 4.3]] * 3
    bvh = kernels.bvh_build(boxes)
    pairs = kernels.bvh_query(bvh, queries)
    assert np.array_equal(pairs.cpu().numpy(), kernels.overlap_dense(queries, boxes).cpu().numpy())
    assert pairs.untyped_storage().nbytes() <= 8 * len(pairs) + (1 << 20)


@pytest.mark.parametrize("dense", (40, 61, 62, 63, 64))
@pytest.mark.parametrize("tiles", (1, 2, 9, 4097))
def test_tet_status_of_dense_and_sparse_tiles(gpu, dense, tiles):
    """Status-only pairs in tiles of 64 of which ``dense`` are cut, on both sides
    of the line for clipping a tile at once, each with a sparse tile after it
    whose pairs wait, coinciding tetrahedra among both."""
    rs = np.random.RandomState(5)
    n = 40
    bodies = []
    for _ in range(2):
        T = rs.uniform(-0.6, 0.6, (n, 1, 3)) + 0.5 * rs.randn(n, 4, 3)
        e = rs.uniform(0.0, 1.0, (n, 4))
        bodies.append([T, e])
    bodies[1][0][:10], bodies[1][1][:10] = bodies[0][0][:10], bodies[0][1][:10]
    (T1, e1), (T2, e2) = bodies
    X = [oracle.tet_mesh_prep(T)[1] for T, _ in bodies]
    every = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 2).astype(np.int32)
    every = every[rs.permutation(len(every))]
    status, _, nv, _ = oracle.tet_pairs(T1, e1, X[0], T2, e2, X[1], every)
    cut, missed = np.nonzero(status)[0], np.nonzero(status == 0)[0]
    assert len(cut) > 100 and len(missed) > 100
    rows = []
    for t in range(tiles):
        k = dense if t % 2 == 0 else 5
        tile = np.concatenate([rs.choice(cut, k), rs.choice(missed, 64 - k)])
        rows.append(tile[rs.permutation(64)])
    rows = np.concatenate(rows)[:64 * tiles - 3]
    got = kernels.tet_pairs_batch(T1, e1, X[0], T2, e2, X[1], every[rows], geometry=False)
    assert np.array_equal(got[0].cpu().numpy(), status[rows])
    assert np.array_equal(got[2].cpu().numpy(), nv[rows])


@pytest.mark.parametrize("n", (1, 129, 5000))
def test_instances_written_over_their_pair_lists(gpu, n):
    """Pair lists that are their own output: every instance is made from the list
    as it was."""
    host = workloads.mixed_pairs(seed=3, n_pairs=60).scene
    dev = host.to_device()
    rs = np.random.RandomState(n)
    a, b = rs.randint(0, host.n_shapes, (2, n)).astype(np.int32)
    poses = rs.uniform(-1.0, 1.0, (50, 12))
    rows = rs.randint(0, 50, (2, n)).astype(np.int32)
    cuda = lambda x: torch.from_numpy(x).cuda()
    ia, ib, pa, pb = cuda(a), cuda(b), cuda(rows[0]), cuda(rows[1])
    out = (torch.empty((2 * n, 16), dtype=torch.float64, device="cuda"),
           torch.empty((2 * n, 4), dtype=torch.int32, device="cuda"), ia, ib)
    view, va, vb = kernels.instance_pairs(dev, ia, ib, cuda(poses), cuda(poses), pa, pb, 50, out=out)
    ids = np.stack([a, b], 1).reshape(-1)
    want = host.shape_f64[ids].copy()
    want[:, :12] = poses[rows.T.reshape(-1)]
    assert np.array_equal(view.shape_i32[:, 0].cpu().numpy(), host.shape_i32[ids, 0])
    assert np.array_equal(view.shape_f64[:, :12].cpu().numpy(), want[:, :12])
    assert np.array_equal(va.cpu().numpy(), 2 * np.arange(n))
    assert np.array_equal(vb.cpu().numpy(), 2 * np.arange(n) + 1)
