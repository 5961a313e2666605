"""Timed cases of the collision path: what programs built on this framework
call, through its public entry points, from one pair to a million.

``listed()`` names the cases, ``draw(rng)`` makes further ones over the same
ranges, ``prepare``/``run`` set one up and make one pass, ``work`` states the
bytes and floating-point operations a pass cannot do without and ``exact``
gives the outputs in 64-bit numpy/torch where they have a closed value.

A case is a dict with a ``kind`` and that kind's sizes:

pair_call    gjk.gjk on two collider objects (the drop-in call)
hull_gjk     GJK distance of small hull pairs on a resident scene
request      one serving request: pairs with their own poses, GJK + EPA
mixed        GJK + EPA over a pair list on a scene of mixed colliders
penetration  GJK + EPA of overlapping hull pairs (nearly all reach EPA)
intersect    GJK intersection test over a pair list on a mixed scene
mpr          MPR penetration over a pair list on a mixed scene
scene_step   AABBs, tree, all overlaps and the intersection test of a scene
broad_build  AABBs, tree build and queries of a box scene
broad_refit  new poses, AABBs, tree refit and queries of a box scene
tet_pairs    contact planes, polygons and forces of tetrahedron pairs
contact      hydroelastic contact wrenches of two rigid bodies
"""
import itertools
import math

import numpy as np
import torch

from distance3d_amd import autotune, colliders, gjk, kernels, workloads
from distance3d_amd import hydroelastic_contact as hydro


def listed():
    return [
        # a program written against single collider objects, one query at a time
        {"name": "pair_call", "kind": "pair_call", "vertices": 64},
        # link hulls of a few robots against each other: a small resident batch
        {"name": "hull_gjk", "kind": "hull_gjk", "pairs": 4096, "vertices": 32},
        # a planner's edge check sent to a resident scene, odd count, latency lanes
        {"name": "request", "kind": "request", "pairs": 301, "colliders": 512},
        # the offline batch: every collider type, hulls of 8 to 4096 vertices
        {"name": "mixed", "kind": "mixed", "pairs": 1048576, "colliders": 131072},
        # contact resolution: overlapping hulls, depth and contact points wanted
        {"name": "penetration", "kind": "penetration", "pairs": 32768},
        # validity checks of sampled configurations: yes or no only, ragged count
        {"name": "intersect", "kind": "intersect", "pairs": 262147, "colliders": 32768},
        # penetration of the same scenes by portal refinement
        {"name": "mpr", "kind": "mpr", "pairs": 262144, "colliders": 32768},
        # one step of a simulated scene: broad phase, then the narrow test
        {"name": "scene_step", "kind": "scene_step", "colliders": 5003},
        # a static map loaded and queried by many bodies: the largest tree
        {"name": "broad_build", "kind": "broad_build", "boxes": 1048576, "queries": 65536},
        # a dynamic world's time step: all poses new, tree kept
        {"name": "broad_refit", "kind": "broad_refit", "boxes": 100003, "queries": 6001},
        # soft contact of two finely meshed bodies, polygons and forces kept
        {"name": "tet_pairs", "kind": "tet_pairs", "pairs": 524289, "tetrahedra": 100000},
        # the drop-in hydroelastic call on two spheres in deep contact
        {"name": "contact", "kind": "contact", "order": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pair_call", "hull_gjk", "request", "mixed", "penetration", "intersect",
                       "mpr", "scene_step", "broad_build", "broad_refit", "tet_pairs", "contact"])
    case = {"kind": kind}
    if kind == "pair_call":
        case["vertices"] = _log(rng, 8, 512)
    elif kind == "hull_gjk":
        case["vertices"] = _log(rng, 8, 64)
        case["pairs"] = _log(rng, 64, 16384)
    elif kind == "request":
        case["pairs"] = _log(rng, 1, 4096)
        case["colliders"] = _log(rng, 64, 1024)
    elif kind == "mixed":
        case["pairs"] = _log(rng, 4096, 1000000)
        case["colliders"] = _log(rng, 1024, 100000)
    elif kind == "penetration":
        case["pairs"] = _log(rng, 512, 32768)
    elif kind in ("intersect", "mpr"):
        case["pairs"] = _log(rng, 1024, 262144)
        case["colliders"] = _log(rng, 256, 32768)
    elif kind == "scene_step":
        case["colliders"] = _log(rng, 64, 16384)
    elif kind == "broad_build":
        case["boxes"] = _log(rng, 512, 1000000)
        case["queries"] = _log(rng, 256, 65536)
    elif kind == "broad_refit":
        case["boxes"] = _log(rng, 512, 500000)
        case["queries"] = _log(rng, 256, 32768)
    elif kind == "tet_pairs":
        case["pairs"] = _log(rng, 1000, 524288)
        case["tetrahedra"] = _log(rng, 200, 100000)
    else:
        case["order"] = rng.choice([2, 3, 4])
    return case


# ---------------------------------------------------------------- inputs


def _cuda(a, dtype):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype).cuda()


def _ids(a):
    return _cuda(a, torch.int32)


def _mixed_host(colliders, seed):
    """Mixed colliders (spheres, capsules, cylinders, boxes, ellipsoids and
    hulls of log-uniform 8..4096 vertices), centres in [-3, 3]^3."""
    return workloads.mixed_pairs(seed=seed, n_pairs=(colliders + 1) // 2).scene


def _random_pairs(rng, n, colliders):
    a = rng.integers(0, colliders, n)
    return a, (a + rng.integers(1, colliders, n)) % colliders


def _hull_and_box(case, seed):
    """World vertices of the hull and pose and size of the box of a pair_call."""
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((case["vertices"], 3))
    v = 0.5 * v / np.linalg.norm(v, axis=1, keepdims=True) + rng.uniform(-1.0, 1.0, 3)
    pose = np.eye(4)
    pose[:3, :3] = workloads.uniform_rotations(rng, 1)[0]
    pose[:3, 3] = rng.uniform(-1.0, 1.0, 3) + np.array([2.5, 0.0, 0.0])
    return v, pose, rng.uniform(0.1, 1.0, 3)


def _box_world(case, seed):
    """The box scene of a broad-phase case at constant density."""
    boxes, queries = case["boxes"], case["queries"]
    extent = 100.0 * (boxes / 1048576.0) ** (1.0 / 3.0)
    return workloads.broad_phase_scene(seed=seed, n_boxes=boxes, n_capsules=queries,
                                       extent=extent).scene


def _moved(case, host, seed):
    """Box poses one time step later: small drift, new orientations."""
    rng = np.random.default_rng(seed + 1000003)
    n = case["boxes"]
    return (workloads.uniform_rotations(rng, n),
            host.shape_f64[:n, 9:12] + rng.normal(0.0, 0.05, (n, 3)))


def _tet_body(rng, n):
    T = rng.uniform(-0.6, 0.6, (n, 1, 3)) + 0.5 * rng.standard_normal((n, 4, 3))
    return T, rng.uniform(0.0, 1.0, (n, 4))


def _tet_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n = case["tetrahedra"]
    bodies = [_tet_body(rng, n) for _ in range(2)]
    return bodies, rng.integers(0, n, (case["pairs"], 2))


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 7])
    if kind == "pair_call":
        v, pose, size = _hull_and_box(case, seed)
        return {"kind": kind, "a": colliders.ConvexHullVertices(v), "b": colliders.Box(pose, size)}
    if kind == "hull_gjk":
        w = workloads.hull_pairs(seed=seed, n_pairs=case["pairs"], n_vertices=case["vertices"])
        return {"kind": kind, "scene": w.scene.to_device(), "a": _ids(w.pair_a), "b": _ids(w.pair_b)}
    if kind == "request":
        n, c = case["pairs"], case["colliders"]
        host, poses, _ = workloads.serving_workload(seed=seed, n_colliders=c, n_requests=1,
                                                    n_poses=16384)
        a, b = _random_pairs(rng, n, c)
        poses_d = _cuda(poses, torch.float64)
        return {"kind": kind, "scene": host.to_device(), "a": _ids(a), "b": _ids(b),
                "poses": poses_d, "pose_a": _ids(rng.integers(0, len(poses), n)),
                "pose_b": _ids(rng.integers(0, len(poses), n)),
                "out": kernels.GjkEpaResult.empty(n, poses_d.device),
                "workspace": torch.empty(kernels.gjk_epa_workspace_bytes(n), dtype=torch.uint8,
                                         device=poses_d.device),
                "lanes": autotune.tuned_lanes(kind="latency"),
                "launch": autotune.tuned_launch(kind="latency")}
    if kind in ("mixed", "intersect", "mpr"):
        host = _mixed_host(case["colliders"], seed)
        a, b = _random_pairs(rng, case["pairs"], case["colliders"])
        state = {"kind": kind, "scene": host.to_device(), "a": _ids(a), "b": _ids(b)}
        if kind == "mpr":
            from distance3d_amd.scene import collider_centers
            state["centers"] = _cuda(collider_centers(host), torch.float64)
        return state
    if kind == "penetration":
        w = workloads.epa_pairs(seed=seed, n_pairs=case["pairs"])
        return {"kind": kind, "scene": w.scene.to_device(), "a": _ids(w.pair_a), "b": _ids(w.pair_b)}
    if kind == "scene_step":
        host = _mixed_host(case["colliders"], seed)
        # about eight box overlaps per collider
        host.shape_f64[:, 9:12] *= 0.25 * host.n_shapes ** (1.0 / 3.0)
        return {"kind": kind, "scene": host.to_device(), "ids": _ids(np.arange(host.n_shapes))}
    if kind in ("broad_build", "broad_refit"):
        host = _box_world(case, seed)
        nb = case["boxes"]
        state = {"kind": kind, "scene": host.to_device(), "boxes": _ids(np.arange(nb)),
                 "queries": _ids(np.arange(nb, host.n_shapes))}
        if kind == "broad_refit":
            R, t = _moved(case, host, seed)
            state["bvh"] = kernels.bvh_build(kernels.aabb_batch(state["scene"], state["boxes"]))
            state["R"], state["t"] = _cuda(R, torch.float64), _cuda(t, torch.float64)
        return state
    if kind == "tet_pairs":
        (b1, b2), pairs = _tet_inputs(case, seed)
        state = {"kind": kind, "pairs": _ids(pairs)}
        for k, (T, e) in ((1, b1), (2, b2)):
            state["T%d" % k], state["e%d" % k] = _cuda(T, torch.float64), _cuda(e, torch.float64)
            state["X%d" % k] = kernels.tet_mesh_prep(state["T%d" % k], aabbs=False)[1]
        return state
    bodies = []
    for offset in (np.zeros(3), rng.uniform(0.06, 0.1, 3)):
        bodies.append(hydro.RigidBody.make_sphere(offset, rng.uniform(0.14, 0.16), case["order"]))
    return {"kind": kind, "bodies": bodies}


# ---------------------------------------------------------------- one pass


def _gjk_epa_out(r):
    return [r.dist, r.cp_a, r.cp_b, r.status, r.epa_out, r.epa_status]


def _table(rows, size, fill=-1):
    """A list of data-dependent length in a table of fixed size, as a program
    that hands it to the next stage keeps it."""
    out = rows.new_full((size,) + tuple(rows.shape[1:]), fill)
    n = min(len(rows), size)
    out[:n] = rows[:n]
    return out


def _posed(body):
    """A body at its pose, as a simulation hands it over at every step
    (find_contact_surface re-expresses the first body it is given)."""
    return hydro.RigidBody(body.body2origin_, body.vertices_, body.tetrahedra_, body.potentials_,
                           body.youngs_modulus)


def run(state):
    kind = state["kind"]
    s = state
    if kind == "pair_call":
        return list(gjk.gjk(s["a"], s["b"]))
    if kind == "hull_gjk":
        r = kernels.gjk_distance_batch(s["scene"], s["a"], s["b"])
        return [r.dist, r.cp_a, r.cp_b, r.status, r.iterations]
    if kind == "request":
        view, a, b = kernels.instance_pairs(s["scene"], s["a"], s["b"], s["poses"], s["poses"],
                                            s["pose_a"], s["pose_b"], len(s["poses"]))
        return _gjk_epa_out(kernels.gjk_epa_batch(view, a, b, out=s["out"],
                                                  workspace=s["workspace"],
                                                  lanes_per_pair=s["lanes"], launch=s["launch"]))
    if kind in ("mixed", "penetration"):
        return _gjk_epa_out(kernels.gjk_epa_batch(s["scene"], s["a"], s["b"]))
    if kind == "intersect":
        return list(kernels.gjk_intersection_batch(s["scene"], s["a"], s["b"], want_status=True))
    if kind == "mpr":
        return list(kernels.mpr_batch(s["scene"], s["a"], s["b"], s["centers"]))
    if kind == "scene_step":
        boxes = kernels.aabb_batch(s["scene"], s["ids"])
        pairs = kernels.bvh_query(kernels.bvh_build(boxes), boxes)
        pairs = pairs[pairs[:, 0] < pairs[:, 1]]
        hit, _ = kernels.gjk_intersection_batch(s["scene"], pairs[:, 0], pairs[:, 1])
        size = 12 * len(boxes) + 64
        return [boxes, len(pairs), _table(pairs, size), _table(hit, size, 255)]
    if kind == "broad_build":
        boxes = kernels.aabb_batch(s["scene"], s["boxes"])
        queries = kernels.aabb_batch(s["scene"], s["queries"])
        pairs = kernels.bvh_query(kernels.bvh_build(boxes), queries)
        return [boxes, queries, len(pairs), _table(pairs, 8 * len(queries) + 1024)]
    if kind == "broad_refit":
        s["scene"].update_poses(s["boxes"], s["R"], s["t"])
        boxes = kernels.aabb_batch(s["scene"], s["boxes"])
        queries = kernels.aabb_batch(s["scene"], s["queries"])
        pairs = kernels.bvh_query(kernels.bvh_refit(s["bvh"], boxes), queries)
        return [boxes, queries, len(pairs), _table(pairs, 8 * len(queries) + 1024)]
    if kind == "tet_pairs":
        st, planes, nv, polys = kernels.tet_pairs_batch(s["T1"], s["e1"], s["X1"], s["T2"], s["e2"],
                                                        s["X2"], s["pairs"], checked=False)
        forces = kernels.tet_contact_forces(s["T1"], s["e1"], s["pairs"], st, planes, nv, polys,
                                            checked=False)
        return [st, planes, nv, polys, forces]
    hit, wrench12, wrench21 = hydro.contact_forces(_posed(s["bodies"][0]), _posed(s["bodies"][1]))
    return [hit, wrench12, wrench21]


# ---------------------------------------------------------------- work

RECORD = 16 * 8 + 4 * 4  # one collider record
MEAN_VERTICES = (4096 - 8) / math.log(4096 / 8)  # of a log-uniform 8..4096 hull
STEP_FLOPS = 150  # one GJK/MPR step: two supports, the closest feature, tests
GJK_OUT = 8 + 24 + 24 + 4
EPA_OUT = 13 * 8 + 4


def work(case):
    """Bytes: inputs once, outputs once.  Operations: the steps an iterative
    query takes on average, with hulls counted at one score per vertex (a
    support cannot know the extreme vertex before it looked at the hull)."""
    kind = case["kind"]
    if kind == "pair_call":
        return {"bytes": 2 * RECORD + 24 * case["vertices"] + GJK_OUT + 96,
                "flops": 5 * case["vertices"] + 6 * STEP_FLOPS}
    if kind == "hull_gjk":
        n, v = case["pairs"], case["vertices"]
        return {"bytes": n * (2 * RECORD + 24 * v + 8 + GJK_OUT + 4),
                "flops": n * (10 * v + 5 * STEP_FLOPS)}
    if kind == "request":
        n, c = case["pairs"], case["colliders"]
        hull = min(n, c // 3) * 12 * 544
        return {"bytes": min(2 * n, c) * RECORD + hull + n * (16 + 2 * 96 + GJK_OUT + EPA_OUT),
                "flops": n * (2 * 5 * 544 / 3 + 8 * STEP_FLOPS)}
    if kind in ("mixed", "intersect", "mpr"):
        n, c = case["pairs"], case["colliders"]
        used = min(2 * n, c)
        out = {"mixed": GJK_OUT + EPA_OUT, "intersect": 5, "mpr": 4 + 56 + 24}[kind]
        steps = {"mixed": 16, "intersect": 4, "mpr": 6}[kind]
        return {"bytes": used * (RECORD + 12 * MEAN_VERTICES / 6) + n * (8 + out),
                "flops": n * (2 * 5 * MEAN_VERTICES / 6 + steps * STEP_FLOPS)}
    if kind == "penetration":
        n = case["pairs"]
        return {"bytes": n * (2 * RECORD + 2 * 160 * 12 + 8 + GJK_OUT + EPA_OUT),
                "flops": n * (2 * 5 * 160 + 20 * STEP_FLOPS)}
    if kind == "scene_step":
        c = case["colliders"]
        return {"bytes": c * (RECORD + 12 * MEAN_VERTICES / 6 + 48 + 4 * (8 + 1)),
                "flops": c * (18 * MEAN_VERTICES / 6 + 60 + 4 * 4 * STEP_FLOPS)}
    if kind in ("broad_build", "broad_refit"):
        n, q = case["boxes"], case["queries"]
        pose = 96 if kind == "broad_refit" else 0
        return {"bytes": (n + q) * (RECORD + 48) + n * pose + 20 * q, "flops": 150 * n + 300 * q}
    if kind == "tet_pairs":
        n, t = case["pairs"], case["tetrahedra"]
        return {"bytes": min(n, t) * 2 * (96 + 32 + 128) + n * (8 + 4 + 32 + 4 + 576 + 56),
                "flops": 150 * n}
    t = 20 * 4 ** case["order"]
    return {"bytes": 2 * t * (96 + 32) + 96, "flops": 2 * t * 150 + 4 * t * 600}


# ---------------------------------------------------------------- 64-bit values


def _posed_vertices(host):
    """(n, v, 3) world vertices of equal-sized hulls."""
    n = host.n_shapes
    v = np.stack([host.vx, host.vy, host.vz], 1).astype(np.float64).reshape(n, -1, 3)
    f = host.shape_f64
    return f[:, None, 9:12] + np.einsum("nij,nvj->nvi", f[:, :9].reshape(n, 3, 3), v)


def _hull_distances(A, B):
    """Distances of convex hulls A (n, a, 3) and B (n, b, 3): the closest point
    of the Minkowski difference by growing a simplex of its support points;
    the closest feature comes from all faces of the simplex."""
    A, B = torch.as_tensor(A), torch.as_tensor(B)
    n = A.shape[0]
    rows = torch.arange(n)

    def support(d):
        i = (A * d[:, None]).sum(2).argmax(1)
        j = (B * d[:, None]).sum(2).argmin(1)
        return A[rows, i] - B[rows, j]

    v = support(torch.tensor([1.0, 0.0, 0.0], dtype=torch.float64).expand(n, 3))
    Y = torch.zeros((n, 4, 3), dtype=torch.float64)
    Y[:, 0] = v
    used = torch.zeros((n, 4), dtype=torch.bool)
    used[:, 0] = True
    live = torch.ones(n, dtype=torch.bool)
    for _ in range(64):
        w = support(-v)
        vv = (v * v).sum(1)
        live &= ((vv - (v * w).sum(1)) > 1e-14 * vv) & ~used.all(1)
        if not bool(live.any()):
            break
        free = (~used).int().argmax(1)
        Y[rows[live], free[live]] = w[live]
        used[rows[live], free[live]] = True
        best = torch.full((n,), math.inf, dtype=torch.float64)
        point, keep = v.clone(), used.clone()
        for size in (1, 2, 3, 4):
            for face in itertools.combinations(range(4), size):
                f = list(face)
                P = Y[:, f]
                E = P[:, 1:] - P[:, :1]
                G = E @ E.transpose(1, 2)
                det = torch.linalg.det(G) if size > 1 else torch.ones(n, dtype=torch.float64)
                scale = torch.diagonal(G, dim1=1, dim2=2).prod(1) if size > 1 else det
                sound = used[:, f].all(1) & (det > 1e-13 * scale)
                eye = torch.eye(size - 1, dtype=torch.float64).expand_as(G)
                rhs = -(E @ P[:, 0, :, None])
                lam = torch.linalg.solve(torch.where(sound[:, None, None], G, eye), rhs)[..., 0]
                lam = torch.cat([1.0 - lam.sum(1, keepdim=True), lam], 1)
                q = (lam[..., None] * P).sum(1)
                d2 = (q * q).sum(1)
                take = live & sound & (lam >= 0.0).all(1) & (d2 < best)
                best = torch.where(take, d2, best)
                point = torch.where(take[:, None], q, point)
                mask = torch.zeros(4, dtype=torch.bool)
                mask[f] = True
                keep = torch.where(take[:, None], mask, keep)
        v, used = point, keep
    d = torch.sqrt((v * v).sum(1))
    d[used.all(1) | (d < 1e-12)] = 0.0
    return d.numpy()


def _box_aabbs(f):
    h = 0.5 * (np.abs(f[:, :9].reshape(-1, 3, 3)) * f[:, None, 12:15]).sum(2)
    return np.stack([f[:, 9:12] - h, f[:, 9:12] + h], 2)


def _capsule_aabbs(f):
    h = 0.5 * f[:, 13:14] * np.abs(f[:, [2, 5, 8]]) + f[:, 12:13]
    return np.stack([f[:, 9:12] - h, f[:, 9:12] + h], 2)


def _tet_planes(case, seed):
    (b1, b2), pairs = _tet_inputs(case, seed)
    field = []
    for T, e in (b1, b2):
        M = np.concatenate([T.transpose(0, 2, 1), np.ones((len(T), 1, 4))], 1)
        field.append((e[:, None] @ np.linalg.inv(M))[:, 0])
    h = field[0][pairs[:, 0]] - field[1][pairs[:, 1]]
    h /= np.linalg.norm(h[:, :3], axis=1, keepdims=True)
    h[:, 3] *= -1.0
    return h


def exact(case, seed):
    """Outputs with a value of their own.  Those an iteration stops short of by
    its tolerance or face cap (EPA, MPR), closest points (not unique) and the
    whole mixed scenes (tens of full sweeps per pair) have none here."""
    kind = case["kind"]
    if kind == "pair_call":
        v, pose, size = _hull_and_box(case, seed)
        corners = np.array(list(itertools.product((-0.5, 0.5), repeat=3))) * size
        box = pose[:3, 3] + corners @ pose[:3, :3].T
        return [float(_hull_distances(v[None], box[None])[0]), None, None, None]
    if kind == "hull_gjk":
        w = workloads.hull_pairs(seed=seed, n_pairs=case["pairs"], n_vertices=case["vertices"])
        V = _posed_vertices(w.scene)
        return [_hull_distances(V[0::2], V[1::2]), None, None, None, None]
    if kind == "scene_step":
        return None
    if kind in ("broad_build", "broad_refit"):
        host = _box_world(case, seed)
        f = host.shape_f64.copy()
        nb = case["boxes"]
        if kind == "broad_refit":
            R, t = _moved(case, host, seed)
            f[:nb, :9], f[:nb, 9:12] = R.reshape(nb, 9), t
        return [_box_aabbs(f[:nb]), _capsule_aabbs(f[nb:]), None, None]
    if kind == "tet_pairs":
        return [None, _tet_planes(case, seed), None, None, None]
    return None
