// d3d_gjk.hip -- GJK intersection of small batches, support points and AABBs
// for gfx950.
//
// (GJK distance, and the intersection of larger batches, run through the sorted
// pair queue in d3d_gjk_queue.hip.)
//
// Shape of the intersection kernel: one lane per pair, 64 pairs per wavefront.  The FP64 simplex
// (Y, P, Q of up to four points) lives in VGPRs of its lane; support points of
// analytic colliders and of small hulls are computed by the lane itself, while
// large hulls are swept by the whole wavefront (coalesced FP32 SoA rows, see
// hull_argmax), one requesting lane at a time.  The loop runs until every
// lane of the wavefront has terminated; finished lanes keep helping with the
// sweeps of the others.
#include "d3d_device.hpp"
#include "d3d_runtime.hpp"

namespace d3d {

constexpr int kBlock = 256;
constexpr int kStatusBadInput = 0x200;

// gjk_intersection_jolt (_gjk_jolt.py:29-80) and _intersection_loop (:83-135).
__global__ __launch_bounds__(kBlock) void gjk_intersection_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb, int64_t n,
    double tolerance, int max_iterations, int serial_max, uint8_t *__restrict__ hit,
    int32_t *__restrict__ status) {
    const int64_t pid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = pid < n;
    Shape A = empty_shape(), B = empty_shape();
    bool ok = false;
    if (valid) {
        const bool okA = load_checked(s, pa[pid], A);
        const bool okB = load_checked(s, pb[pid], B);
        ok = okA && okB;
    }
    Simplex S;
    simplex_zero(S);
    v3 d = mk(1.0, 0.0, 0.0);
    double prev = kMaxFloat;
    const double tol2 = tolerance * tolerance;
    int state = -1, it = 0;
    bool active = ok;

    while (__ballot(active) != 0ull) {
        if (active && it >= max_iterations) {
            state = D3D_ITER_CAP;
            active = false;
        }
        const v3 p = support_wave(s, A, d, active, serial_max);
        const v3 q = support_wave(s, B, -d, active, serial_max);
        if (!active) continue;
        ++it;
        const v3 w = p - q;
        if (dot(d, w) < -kEps) {
            state = D3D_SEPARATED;
            active = false;
            continue;
        }
        simplex_append(S, w);
        v3 v;
        double vv;
        int set;
        if (!closest_to_origin(S, prev, v, vv, set)) {
            state = D3D_SEPARATED;
            active = false;
            continue;
        }
        if (set == 15 || vv <= tol2 || vv <= kEps * max_y_len_sq(S)) {
            state = D3D_INTERSECT;
            active = false;
            continue;
        }
        d = -v;
        if (prev - vv <= kEps * prev) {
            state = D3D_SEPARATED;
            active = false;
            continue;
        }
        prev = vv;
        simplex_compact(S, set);
    }
    if (!valid) return;
    if (!ok) {
        hit[pid] = 0;
        if (status) status[pid] = kStatusBadInput;
        return;
    }
    hit[pid] = state == D3D_INTERSECT ? 1 : 0;
    if (status) status[pid] = state;
}

// collider.support_function(d) for a batch of (collider, direction) queries.
__global__ __launch_bounds__(kBlock) void support_kernel(d3d_scene s,
                                                         const int32_t *__restrict__ shape,
                                                         const double *__restrict__ dirs, int64_t n,
                                                         int serial_max, double *__restrict__ out) {
    const int64_t pid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = pid < n;
    Shape h = empty_shape();
    bool ok = false;
    v3 d = mk(0.0, 0.0, 0.0);
    if (valid) {
        ok = load_checked(s, shape[pid], h);
        d = mk(dirs[3 * pid], dirs[3 * pid + 1], dirs[3 * pid + 2]);
    }
    const v3 p = support_wave(s, h, d, ok, serial_max);
    if (!valid) return;
    out[3 * pid] = ok ? p.x : NAN;
    out[3 * pid + 1] = ok ? p.y : NAN;
    out[3 * pid + 2] = ok ? p.z : NAN;
}

// Box of the posed hull of lane `src` of the wavefront, by its 64 lanes: the
// running minimum and maximum of the world vertices, lanes striding over the
// hull, then butterfly merges (min and max are exact, so the box does not
// depend on the order).  Every lane returns the box.
__device__ __forceinline__ void hull_box_wave(const d3d_scene &s, const Shape &mine, int src,
                                              double (&mn)[3], double (&mx)[3]) {
    Shape h;
#pragma unroll
    for (int j = 0; j < 9; ++j) h.R[j] = readlane_f64(mine.R[j], src);
#pragma unroll
    for (int j = 0; j < 3; ++j) h.t[j] = readlane_f64(mine.t[j], src);
    const int nv = readlane_i32(mine.nv, src);
    const int voff = readlane_i32(mine.voff, src), voff64 = readlane_i32(mine.voff64, src);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        mn[a] = INFINITY;
        mx[a] = -INFINITY;
    }
#pragma unroll 4
    for (int j = lane_id(); j < nv; j += kWave) {
        const v3 w = to_world(h, hull_vertex(s, voff, voff64, j));
        mn[0] = w.x < mn[0] ? w.x : mn[0];
        mx[0] = w.x > mx[0] ? w.x : mx[0];
        mn[1] = w.y < mn[1] ? w.y : mn[1];
        mx[1] = w.y > mx[1] ? w.y : mx[1];
        mn[2] = w.z < mn[2] ? w.z : mn[2];
        mx[2] = w.z > mx[2] ? w.z : mx[2];
    }
    for_butterfly<kWave>([&](auto o) {
        constexpr int OFF = decltype(o)::value;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            double p, q;
            xpair<OFF>(mn[a], p, q);
            mn[a] = q < p ? q : p;
            xpair<OFF>(mx[a], p, q);
            mx[a] = q > p ? q : p;
        }
    });
}

// collider.aabb() (containment.py:6-229): a wavefront takes S colliders, one
// per lane; analytic boxes and hulls of at most serial_max vertices are the
// lane's own work, the larger hulls are swept by the whole wavefront, one
// after the other.
// Bound: memory for large batches of analytic colliders (1,048,576 boxes: 200
// MB in and out in 32 us); with hulls, the longest chain of hull sweeps a
// wavefront holds (a lane that walks its own hull takes one load round per
// vertex: 5,003 mixed colliders with hulls of up to 4,096 vertices took 1,280
// us that way, 42 us swept by the wavefront).
template <int S>
__global__ __launch_bounds__(kBlock) void aabb_kernel(d3d_scene s, const int32_t *__restrict__ shape,
                                                      int64_t n, int serial_max,
                                                      double *__restrict__ out) {
    const int lane = lane_id();
    const int64_t wave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) / kWave;
    const int64_t pid = wave * S + lane;
    const bool valid = lane < S && pid < n;
    Shape h = empty_shape();
    const bool ok = valid && load_checked(s, shape[pid], h);
    double mn[3], mx[3];
    const bool coop = ok && h.type == D3D_HULL && h.nv > serial_max;
    unsigned long long m = __ballot(coop);
    while (m) {
        const int src = __ffsll((long long)m) - 1;
        m &= m - 1;
        double bmn[3], bmx[3];
        hull_box_wave(s, h, src, bmn, bmx);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            mn[a] = lane == src ? bmn[a] : mn[a];
            mx[a] = lane == src ? bmx[a] : mx[a];
        }
    }
    if (!valid) return;
    if (!ok) {
#pragma unroll
        for (int a = 0; a < 6; ++a) out[6 * pid + a] = NAN;
        return;
    }
    const double *R = h.R, *t = h.t;
    switch (h.type) {
    case D3D_HULL: {
        if (coop) break;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            mn[a] = INFINITY;
            mx[a] = -INFINITY;
        }
        for (int j = 0; j < h.nv; ++j) {
            const v3 w = to_world(h, hull_vertex(s, h.voff, h.voff64, j));
            mn[0] = w.x < mn[0] ? w.x : mn[0];
            mx[0] = w.x > mx[0] ? w.x : mx[0];
            mn[1] = w.y < mn[1] ? w.y : mn[1];
            mx[1] = w.y > mx[1] ? w.y : mx[1];
            mn[2] = w.z < mn[2] ? w.z : mn[2];
            mx[2] = w.z > mx[2] ? w.z : mx[2];
        }
        break;
    }
    case D3D_BOX: {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            mn[a] = INFINITY;
            mx[a] = -INFINITY;
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const double l0 = (((c >> 2) & 1) ? 0.5 : -0.5) * h.p[0];
            const double l1 = (((c >> 1) & 1) ? 0.5 : -0.5) * h.p[1];
            const double l2 = ((c & 1) ? 0.5 : -0.5) * h.p[2];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double v = t[a] + (l0 * R[3 * a] + l1 * R[3 * a + 1] + l2 * R[3 * a + 2]);
                mn[a] = v < mn[a] ? v : mn[a];
                mx[a] = v > mx[a] ? v : mx[a];
            }
        }
        break;
    }
    case D3D_SPHERE:
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            mn[a] = t[a] - h.p[0];
            mx[a] = t[a] + h.p[0];
        }
        break;
    case D3D_CAPSULE:
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double e = 0.5 * h.p[1] * fabs(R[3 * a + 2]) + h.p[0];
            mn[a] = t[a] - e;
            mx[a] = t[a] + e;
        }
        break;
    case D3D_CYLINDER:
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double ax = R[3 * a + 2];
            const double e = 0.5 * h.p[1] * fabs(ax) + h.p[0] * sqrt(1.0 - ax * ax);
            mn[a] = t[a] - e;
            mx[a] = t[a] + e;
        }
        break;
    case D3D_ELLIPSOID: {
        double E[3][3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) E[i][j] = R[3 * i + j] * h.p[j];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double cn = sqrt(E[0][j] * E[0][j] + E[1][j] * E[1][j] + E[2][j] * E[2][j]);
#pragma unroll
            for (int i = 0; i < 3; ++i) E[i][j] = E[i][j] / cn;
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) E[i][j] = E[i][j] * h.p[j];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            double m = -INFINITY;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double v = R[3 * i] * E[k][0] + R[3 * i + 1] * E[k][1] + R[3 * i + 2] * E[k][2];
                m = v > m ? v : m;
            }
            mn[k] = t[k] - m;
            mx[k] = t[k] + m;
        }
        break;
    }
    case D3D_CONE:
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double ht = h.p[1], r = h.p[0];
            const double pa_ = t[a], pb_ = t[a] + ht * R[3 * a + 2];
            const double ad = pb_ - pa_;
            const double e = sqrt(1.0 - ad * ad / (ht * ht));
            const double lo = pa_ - e * r, hi = pa_ + e * r;
            mn[a] = lo < pb_ ? lo : pb_;
            mx[a] = hi > pb_ ? hi : pb_;
        }
        break;
    case D3D_DISK:
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double nr = R[3 * a + 2];
            const double e = h.p[0] * sqrt(1.0 - nr * nr);
            mn[a] = t[a] - e;
            mx[a] = t[a] + e;
        }
        break;
    default:  // D3D_ELLIPSE
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double u = h.p[0] * R[3 * a], v = h.p[1] * R[3 * a + 1];
            const double e = sqrt(u * u + v * v);
            mn[a] = t[a] - e;
            mx[a] = t[a] + e;
        }
        break;
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (h.margin != 0.0) {
            mn[a] = mn[a] - h.margin;
            mx[a] = mx[a] + h.margin;
        }
        out[6 * pid + 2 * a] = mn[a];
        out[6 * pid + 2 * a + 1] = mx[a];
    }
}

}  // namespace d3d

using namespace d3d;

extern "C" int d3d_support_batch(const d3d_scene *scene, const int32_t *shape, const double *dirs,
                                 int64_t n, double *out, void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(shape && dirs && out, "NULL buffer");
    hipLaunchKernelGGL(support_kernel, dim3(grid_for(n, kBlock)), dim3(kBlock), 0,
                       (hipStream_t)stream, *scene, shape, dirs, n, default_params().hull_serial_max,
                       out);
    D3D_CHECK_LAUNCH("support_kernel");
    return D3D_OK;
}

extern "C" int d3d_aabb_batch(const d3d_scene *scene, const int32_t *shape, int64_t n, double *out,
                              void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(shape && out, "NULL buffer");
    // Few colliders per wavefront keep its chain of hull sweeps short, many keep
    // its lanes busy on analytic boxes; the line moves with the batch because a
    // large one has wavefronts to spare.  4 / 16 / 64 colliders per wavefront:
    // 16,384 mixed 37 / 67 / 89 us, 131,072 mixed 146 / 125 / 165 us, 262,144
    // mixed 272 / 250 / 241 us; boxes alone 20,000 10.5 / 10.4 / 10.3 us, 200,000
    // 36 / 14 / 11 us, 1,048,576 165 / 52 / 32 us: a scene without hull vertices has
    // no sweeps, and always takes 64.
    const int serial_max = default_params().hull_serial_max;
    auto launch = [&](auto kernel, int per_wave) {
        hipLaunchKernelGGL(kernel, dim3(grid_for(n, kBlock / kWave * per_wave)), dim3(kBlock), 0,
                           (hipStream_t)stream, *scene, shape, n, serial_max, out);
    };
    if (n >= 524288 || scene->n_vertices == 0) launch(aabb_kernel<64>, 64);
    else if (n >= 65536) launch(aabb_kernel<16>, 16);
    else launch(aabb_kernel<4>, 4);
    D3D_CHECK_LAUNCH("aabb_kernel");
    return D3D_OK;
}

extern "C" int d3d_gjk_intersection_batch(const d3d_scene *scene, const int32_t *pair_a,
                                          const int32_t *pair_b, int64_t n, double tolerance,
                                          int32_t max_iterations, uint8_t *hit, int32_t *status,
                                          void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(pair_a && pair_b && hit, "NULL buffer");
    D3D_CHECK_ARG(max_iterations > 0, "max_iterations must be > 0");
    hipLaunchKernelGGL(gjk_intersection_kernel, dim3(grid_for(n, kBlock)), dim3(kBlock), 0,
                       (hipStream_t)stream, *scene, pair_a, pair_b, n, tolerance, max_iterations,
                       default_params().hull_serial_max, hit, status);
    D3D_CHECK_LAUNCH("gjk_intersection_kernel");
    return D3D_OK;
}
