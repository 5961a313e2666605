"""Packed collider scenes: the HBM layout every kernel reads.

A scene is a collider table plus vertex pools (layout in include/d3d.h):

* ``shape_f64`` (n, 16) float64: rotation R (row major), translation t,
  three type parameters, margin;
* ``shape_i32`` (n, 4) int32: type, vertex count, offset into the FP32 pool,
  offset into the FP64 pool (-1 when the FP32 values are exact);
* ``vx, vy, vz``: FP32 structure-of-arrays pool of hull vertices in the
  collider's local frame (coalesced rows for the wavefront sweeps);
* ``v64`` (m, 3) float64: exact values of hulls that FP32 cannot represent.

Hull vertices generated by this package are canonical FP32 values in the local
frame with an FP64 pose; vertex sets handed in by users (world frame, FP64,
like the reference's ``ConvexHullVertices``) get an identity pose and, if any
coordinate is not an FP32 value, an exact FP64 copy.

The host scene keeps every hull's vertices in their original order.  The copy
uploaded to the device (:class:`DeviceScene`) reorders hulls of at least
``CLUSTER_MIN_VERTICES`` vertices into spatial clusters with bounding spheres
(``d3d_cluster_scene``) so the support sweep can skip clusters; the original
index of each vertex travels along for tie-breaking, so supports are those of
the original order.
"""
import ctypes

import numpy as np

from . import _native

F64_COLS = 16
I32_COLS = 4
_ULP_MARGIN = 1.0 + 2.0 ** -20
CLUSTER_MIN_VERTICES = 64
# a scene of at most this many bytes is uploaded in one copy, staged in one host
# array; a large one array by array, without a second host copy of it
PACKED_UPLOAD_MAX = 1 << 20


def plane_basis_from_normal(plane_normal):
    """Two unit vectors spanning the plane of ``plane_normal``.

    Same construction as the reference's ``utils.plane_basis_from_normal``
    (utils.py:76-122), used to lay out Disk colliders.
    """
    n = np.asarray(plane_normal, dtype=np.float64)
    if abs(n[0]) >= abs(n[1]):
        length = np.sqrt(n[0] * n[0] + n[2] * n[2])
        x = np.array([-n[2] / length, 0.0, n[0] / length])
        y = np.array([n[1] * x[2], n[2] * x[0] - n[0] * x[2], -n[1] * x[0]])
    else:
        length = np.sqrt(n[1] * n[1] + n[2] * n[2])
        x = np.array([0.0, n[2] / length, -n[1] / length])
        y = np.array([n[1] * x[2] - n[2] * x[1], -n[0] * x[2], n[0] * x[1]])
    return x, y


def hull_bound(vertices):
    """max_i(|x_i| + |y_i| + |z_i|), rounded up: the scale of the FP32 sweep
    error bound (see hull_argmax in csrc/d3d_device.hpp)."""
    v = np.asarray(vertices, dtype=np.float64)
    if len(v) == 0:
        return 0.0
    return float(np.max(np.abs(v).sum(axis=1))) * _ULP_MARGIN


class HostScene:
    """Packed scene in host memory (numpy)."""

    def __init__(self, shape_f64, shape_i32, vx, vy, vz, v64=None):
        self.shape_f64 = np.ascontiguousarray(shape_f64, dtype=np.float64)
        self.shape_i32 = np.ascontiguousarray(shape_i32, dtype=np.int32)
        self.vx = np.ascontiguousarray(vx, dtype=np.float32)
        self.vy = np.ascontiguousarray(vy, dtype=np.float32)
        self.vz = np.ascontiguousarray(vz, dtype=np.float32)
        if v64 is None:
            v64 = np.zeros((0, 3))
        self.v64 = np.ascontiguousarray(v64, dtype=np.float64).reshape(-1, 3)
        assert self.shape_f64.shape == (len(self.shape_i32), F64_COLS)
        assert self.shape_i32.shape[1] == I32_COLS

    @property
    def n_shapes(self):
        return len(self.shape_i32)

    @property
    def n_vertices(self):
        return len(self.vx)

    @property
    def n_vertices64(self):
        return len(self.v64)

    def validate(self):
        """Checks that every hull's vertex range lies inside the pools."""
        t = self.shape_i32[:, 0]
        if np.any((t < 0) | (t > _native.ELLIPSE)):
            raise ValueError("unknown collider type in scene")
        hull = t == _native.HULL
        nv = self.shape_i32[hull, 1].astype(np.int64)
        off = self.shape_i32[hull, 2].astype(np.int64)
        off64 = self.shape_i32[hull, 3].astype(np.int64)
        if np.any(nv < 1):
            raise ValueError("a hull has no vertices")
        if np.any(off < 0) or np.any(off + nv > self.n_vertices):
            raise ValueError("hull vertex range outside the FP32 pool")
        has64 = off64 >= 0
        if np.any(off64[has64] + nv[has64] > self.n_vertices64):
            raise ValueError("hull vertex range outside the FP64 pool")
        if not (len(self.vx) == len(self.vy) == len(self.vz)):
            raise ValueError("FP32 pool arrays differ in length")
        return self

    def oracle_args(self):
        """(shape_f64, shape_i32, vx, vy, vz, v64) with non-empty pools."""
        vx, vy, vz = self.vx, self.vy, self.vz
        if len(vx) == 0:
            vx = vy = vz = np.zeros(1, dtype=np.float32)
        v64 = self.v64 if len(self.v64) else np.zeros((1, 3))
        return self.shape_f64, self.shape_i32, vx, vy, vz, v64

    def to_device(self, device=None):
        return DeviceScene(self, device)


def cluster_layout(host, min_vertices=CLUSTER_MIN_VERTICES, threads=0):
    """The clustered layout of ``host`` as host arrays (``d3d_cluster_scene``,
    a host-only routine of the library): dict with shape_f64, shape_i32, vx,
    vy, vz, v64, vorig and clusters (n_clusters, 4)."""
    lib = _native.load_library()
    n = host.n_shapes
    nv, nv64, nc = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_int64()
    _native.check(lib.d3d_cluster_plan(host.shape_i32.ctypes.data, n, int(min_vertices),
                                       ctypes.byref(nv), ctypes.byref(nv64), ctypes.byref(nc)),
                  "d3d_cluster_plan")
    out = {"shape_f64": np.empty_like(host.shape_f64), "shape_i32": np.empty_like(host.shape_i32),
           "vx": np.empty(nv.value, np.float32), "vy": np.empty(nv.value, np.float32),
           "vz": np.empty(nv.value, np.float32), "v64": np.empty((nv64.value, 3)),
           "vorig": np.empty(nv.value, np.int32), "clusters": np.empty((nc.value, 4), np.float32)}
    v64 = host.v64 if len(host.v64) else np.zeros((1, 3))
    _native.check(lib.d3d_cluster_scene(
        host.shape_f64.ctypes.data, host.shape_i32.ctypes.data, n, host.vx.ctypes.data,
        host.vy.ctypes.data, host.vz.ctypes.data, v64.ctypes.data, host.n_vertices,
        host.n_vertices64, int(min_vertices), int(threads), out["shape_f64"].ctypes.data,
        out["shape_i32"].ctypes.data, out["vx"].ctypes.data, out["vy"].ctypes.data,
        out["vz"].ctypes.data, out["v64"].ctypes.data, out["vorig"].ctypes.data,
        out["clusters"].ctypes.data), "d3d_cluster_scene")
    return out


# what the kernels read, whatever a caller has put in a HostScene's arrays
_DTYPES = {"shape_f64": np.float64, "shape_i32": np.int32, "vx": np.float32, "vy": np.float32,
           "vz": np.float32, "v64": np.float64, "vorig": np.int32, "clusters": np.float32}


def _upload(layout, device):
    """The arrays of a scene layout as device tensors (None stays None, an empty
    array becomes one zero row).  The eight arrays of a small scene are views of
    one tensor, each at a multiple of 256 bytes, so that one copy brings all."""
    import torch
    arrays = {}
    for name, a in layout.items():
        if a is not None:
            a = np.ascontiguousarray(a if len(a) else np.zeros((1,) + a.shape[1:]), _DTYPES[name])
        arrays[name] = a
    total = sum((a.nbytes + 255) // 256 * 256 for a in arrays.values() if a is not None)
    if total > PACKED_UPLOAD_MAX:
        return {name: None if a is None else torch.from_numpy(a).to(device)
                for name, a in arrays.items()}
    host = np.zeros(total, np.uint8)
    at = {}
    end = 0
    for name, a in arrays.items():
        if a is not None:
            at[name] = end
            host[end:end + a.nbytes] = a.reshape(-1).view(np.uint8)
            end += (a.nbytes + 255) // 256 * 256
    packed = torch.from_numpy(host).to(device)
    return {name: None if a is None else
            packed[at[name]:at[name] + a.nbytes].view(getattr(torch, a.dtype.name)).view(a.shape)
            for name, a in arrays.items()}


class DeviceScene:
    """A scene resident in HBM (torch tensors) plus its C descriptor.

    ``cluster_min``: hulls with at least this many vertices are uploaded in
    the clustered layout (0 disables it; results are the same either way)."""

    def __init__(self, host, device=None, cluster_min=CLUSTER_MIN_VERTICES):
        import torch
        host.validate()
        dev = torch.device("cuda") if device is None else torch.device(device)
        self.device = dev
        self.host = host

        if cluster_min and cluster_min > 0:
            lay = cluster_layout(host, cluster_min)
        else:
            lay = {"shape_f64": host.shape_f64, "shape_i32": host.shape_i32, "vx": host.vx,
                   "vy": host.vy, "vz": host.vz, "v64": host.v64, "vorig": None, "clusters": None}
        for name, tensor in _upload(lay, dev).items():
            setattr(self, name, tensor)
        self.n_shapes = host.n_shapes
        self.n_vertices = len(lay["vx"])
        self.n_vertices64 = len(lay["v64"])
        self.n_clusters = 0 if lay["clusters"] is None else len(lay["clusters"])
        self._c = scene_descriptor(self, self.shape_f64, self.shape_i32, self.n_shapes)

    @property
    def c(self):
        return ctypes.byref(self._c)

    def update_poses(self, shape_ids, R, t):
        """Overwrite the poses of ``shape_ids`` (device-side, no re-upload of
        the vertex pools).  R: (k,3,3), t: (k,3) tensors or arrays."""
        import torch
        ids = torch.as_tensor(shape_ids, device=self.device, dtype=torch.int64)
        R = torch.as_tensor(R, device=self.device, dtype=torch.float64).reshape(-1, 9)
        t = torch.as_tensor(t, device=self.device, dtype=torch.float64).reshape(-1, 3)
        self.shape_f64[ids, 0:9] = R
        self.shape_f64[ids, 9:12] = t


def collider_centers(host, only=None):
    """(n_shapes, 3) centres of the packed colliders, as collider.center()
    gives them (colliders.py): the mean vertex for hulls (posed), the cone's
    mid-height point, the pose origin otherwise.  With ``only`` (collider
    indices) hull means are computed for those colliders alone; the other
    hull rows keep the pose origin."""
    f = host.shape_f64
    i = host.shape_i32
    out = f[:, 9:12].copy()
    hulls = np.nonzero(i[:, 0] == _native.HULL)[0]
    if only is not None:
        hulls = np.intersect1d(hulls, np.asarray(only))
    for k in hulls:
        nv, voff, voff64 = int(i[k, 1]), int(i[k, 2]), int(i[k, 3])
        if voff64 >= 0:
            v = host.v64[voff64:voff64 + nv]
        else:
            v = np.stack([host.vx[voff:voff + nv], host.vy[voff:voff + nv],
                          host.vz[voff:voff + nv]], axis=1).astype(np.float64)
        out[k] = f[k, 9:12] + np.dot(f[k, 0:9].reshape(3, 3), np.mean(v, axis=0))
    cone = np.nonzero(i[:, 0] == _native.CONE)[0]
    out[cone] = f[cone, 9:12] + (0.5 * f[cone, 13])[:, None] * f[cone][:, [2, 5, 8]]
    return out


def scene_descriptor(pools, shape_f64, shape_i32, n_shapes):
    """d3d_scene over the collider table (shape_f64, shape_i32) and the vertex
    pools of ``pools`` (a DeviceScene)."""
    return _native.d3d_scene(
        shape_f64.data_ptr(), shape_i32.data_ptr(), pools.vx.data_ptr(), pools.vy.data_ptr(),
        pools.vz.data_ptr(), pools.v64.data_ptr(), n_shapes, pools.n_vertices,
        pools.n_vertices64, None if pools.vorig is None else pools.vorig.data_ptr(),
        None if pools.clusters is None else pools.clusters.data_ptr(), pools.n_clusters)


class SceneBuilder:
    """Incremental packer for individual colliders."""

    def __init__(self):
        self._f = []
        self._i = []
        self._v32 = []
        self._v64 = []
        self._n32 = 0
        self._n64 = 0

    def _add(self, type_, R, t, params, margin, nv=0, voff=0, voff64=-1):
        row = np.zeros(F64_COLS)
        row[0:9] = np.asarray(R, dtype=np.float64).reshape(9)
        row[9:12] = np.asarray(t, dtype=np.float64).reshape(3)
        p = np.asarray(params, dtype=np.float64).reshape(-1)
        row[12:12 + len(p)] = p
        row[15] = margin
        self._f.append(row)
        self._i.append((type_, nv, voff, voff64))
        return len(self._i) - 1

    def add_hull(self, vertices, R=None, t=None, margin=0.0):
        v = np.ascontiguousarray(vertices, dtype=np.float64).reshape(-1, 3)
        if len(v) == 0:
            raise ValueError("a convex hull needs at least one vertex")
        R = np.eye(3) if R is None else R
        t = np.zeros(3) if t is None else t
        v32 = v.astype(np.float32)
        voff = self._n32
        self._v32.append(v32)
        self._n32 += len(v)
        voff64 = -1
        if not np.array_equal(v32.astype(np.float64), v):
            voff64 = self._n64
            self._v64.append(v)
            self._n64 += len(v)
        return self._add(_native.HULL, R, t, [hull_bound(v)], margin, len(v), voff, voff64)

    def add_sphere(self, center, radius, margin=0.0):
        return self._add(_native.SPHERE, np.eye(3), center, [radius], margin)

    def add_capsule(self, pose, radius, height, margin=0.0):
        pose = np.asarray(pose, dtype=np.float64)
        return self._add(_native.CAPSULE, pose[:3, :3], pose[:3, 3], [radius, height], margin)

    def add_cylinder(self, pose, radius, length, margin=0.0):
        pose = np.asarray(pose, dtype=np.float64)
        return self._add(_native.CYLINDER, pose[:3, :3], pose[:3, 3], [radius, length], margin)

    def add_ellipsoid(self, pose, radii, margin=0.0):
        pose = np.asarray(pose, dtype=np.float64)
        return self._add(_native.ELLIPSOID, pose[:3, :3], pose[:3, 3], radii, margin)

    def add_box(self, pose, size, margin=0.0):
        pose = np.asarray(pose, dtype=np.float64)
        return self._add(_native.BOX, pose[:3, :3], pose[:3, 3], size, margin)

    def add_cone(self, pose, radius, height, margin=0.0):
        pose = np.asarray(pose, dtype=np.float64)
        return self._add(_native.CONE, pose[:3, :3], pose[:3, 3], [radius, height], margin)

    def add_disk(self, center, radius, normal, margin=0.0):
        normal = np.asarray(normal, dtype=np.float64)
        x, y = plane_basis_from_normal(normal)
        R = np.column_stack((x, y, normal))
        return self._add(_native.DISK, R, center, [radius], margin)

    def add_ellipse(self, center, axes, radii, margin=0.0):
        axes = np.asarray(axes, dtype=np.float64)
        R = np.column_stack((axes[0], axes[1], np.cross(axes[0], axes[1])))
        return self._add(_native.ELLIPSE, R, center, radii, margin)

    def build(self):
        f = np.array(self._f).reshape(-1, F64_COLS)
        i = np.array(self._i, dtype=np.int32).reshape(-1, I32_COLS)
        if self._v32:
            v32 = np.concatenate(self._v32)
        else:
            v32 = np.zeros((0, 3), dtype=np.float32)
        v64 = np.concatenate(self._v64) if self._v64 else np.zeros((0, 3))
        return HostScene(f, i, v32[:, 0], v32[:, 1], v32[:, 2], v64).validate()
