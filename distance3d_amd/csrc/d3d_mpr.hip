// Minkowski portal refinement (mpr.py:20-393, after libccd): intersection
// and penetration depth, direction and contact position for a batch of pairs.
//
// One lane per pair, FP64 throughout, the oracle's expressions in its order.
// The algorithm calls the pair's support function from several places
// (portal discovery, refinement, penetration search); each lane runs it as a
// state machine whose phases end at a support call, and every loop round all
// lanes of the wavefront evaluate their supports together (support_wave
// sweeps large hulls with the whole wavefront).  The portal (4 rows of the
// Minkowski point and both support points) stays in registers: rows are only
// addressed with compile-time indices, runtime row choices become selects.
//
// Batches with hulls go through the sorted pair queue instead (MprMode): the
// same state machine with the support points of the portal rows in LDS.
#include "d3d_queue.hpp"

namespace d3d {

constexpr int kMprBlock = 256;
// hulls with more vertices than this are swept by the whole wavefront (the
// value the other lane-per-pair kernels use)
constexpr int kMprSerialMax = 16;

struct MprPortal {
    v3 v[4], a[4], b[4];
};

// row r (runtime) = (v, a, b)
__device__ __forceinline__ void mpr_set(MprPortal &P, int r, v3 v, v3 a, v3 b) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        P.v[k] = vsel(k == r, v, P.v[k]);
        P.a[k] = vsel(k == r, a, P.a[k]);
        P.b[k] = vsel(k == r, b, P.b[k]);
    }
}

// _portal_direction (mpr.py:286-293)
__device__ __forceinline__ v3 mpr_portal_dir(const MprPortal &P) {
    return norm_vector(cross(P.v[2] - P.v[1], P.v[3] - P.v[1]));
}

// _encapsulates_origin (mpr.py:296-299)
__device__ __forceinline__ bool mpr_encapsulates(v3 v, v3 d) { return dot(v, d) > -10.0 * kEps; }

// _portal_reach_tolerance (mpr.py:302-311)
__device__ __forceinline__ bool mpr_reach_tol(const MprPortal &P, v3 v4, v3 d, double tol) {
    const double p = dot(v4, d);
    double m = p - dot(P.v[1], d);
    const double t2 = p - dot(P.v[2], d);
    if (t2 < m) m = t2;
    const double t3 = p - dot(P.v[3], d);
    if (t3 < m) m = t3;
    return m < tol + kEps;
}

// _expand_portal (mpr.py:314-329)
__device__ __forceinline__ void mpr_expand(MprPortal &P, v3 v4, v3 a4, v3 b4) {
    const v3 x = cross(v4, P.v[0]);
    int r;
    if (dot(P.v[1], x) > 0.0) r = dot(P.v[2], x) > 0.0 ? 1 : 3;
    else r = dot(P.v[3], x) > 0.0 ? 2 : 1;
    mpr_set(P, r, v4, a4, b4);
}

__device__ __forceinline__ double vnorm(v3 v) { return sqrt(dot(v, v)); }

// point_to_triangle(zeros, (A, B, C)) (distance/_triangle.py:12-89)
__device__ __forceinline__ double origin_to_triangle(v3 A, v3 B, v3 C, v3 &cp) {
    const v3 o = mk(0.0, 0.0, 0.0);
    const v3 ab = B - A, ac = C - A;
    const v3 ap = o - A;
    const double d1 = dot(ab, ap), d2 = dot(ac, ap);
    if (d1 <= 0.0 && d2 <= 0.0) {
        cp = A;
        return vnorm(o - cp);
    }
    const v3 bp = o - B;
    const double d3 = dot(ab, bp), d4 = dot(ac, bp);
    if (d3 >= 0.0 && d4 <= d3) {
        cp = B;
        return vnorm(o - cp);
    }
    const double vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0 && 0.0 <= d1 && d3 <= 0.0) {
        const double v = d1 / (d1 - d3);
        cp = A + ab * v;
        return vnorm(o - cp);
    }
    const v3 cpt = o - C;
    const double d5 = dot(ab, cpt), d6 = dot(ac, cpt);
    if (d6 >= 0.0 && d5 <= d6) {
        cp = C;
        return vnorm(o - cp);
    }
    const double vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0 && 0.0 <= d2 && d6 <= 0.0) {
        const double w = d2 / (d2 - d6);
        cp = A + ac * w;
        return vnorm(o - cp);
    }
    const double va = d3 * d6 - d5 * d4;
    if (va <= 0.0 && 0.0 <= d4 - d3 && d5 - d6 >= 0.0) {
        const double w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
        cp = B + (C - B) * w;
        return vnorm(o - cp);
    }
    const double denom = 1.0 / (va + vb + vc);
    const double v = vb * denom, w = vc * denom;
    cp = (A + ab * v) + ac * w;
    return vnorm(o - cp);
}

// _contact_position (mpr.py:378-393)
__device__ __forceinline__ v3 mpr_contact(const MprPortal &P, v3 d) {
    double b0 = dot(cross(P.v[1], P.v[2]), P.v[3]);
    double b1 = dot(cross(P.v[3], P.v[2]), P.v[0]);
    double b2 = dot(cross(P.v[0], P.v[1]), P.v[3]);
    double b3 = dot(cross(P.v[2], P.v[1]), P.v[0]);
    double sum = ((b0 + b1) + b2) + b3;
    if (sum < kEps) {
        b0 = 0.0;
        b1 = dot(cross(P.v[2], P.v[3]), d);
        b2 = dot(cross(P.v[3], P.v[1]), d);
        b3 = dot(cross(P.v[1], P.v[2]), d);
        sum = ((b0 + b1) + b2) + b3;
    }
    b0 = b0 / sum;
    b1 = b1 / sum;
    b2 = b2 / sum;
    b3 = b3 / sum;
    const v3 p1 = ((P.a[0] * b0 + P.a[1] * b1) + P.a[2] * b2) + P.a[3] * b3;
    const v3 p2 = ((P.b[0] * b0 + P.b[1] * b1) + P.b[2] * b2) + P.b[3] * b3;
    return (p1 + p2) * 0.5;
}

// phases: each ends at a support call along d
enum : int {
    kMprDone = 0,
    kMprV1 = 1,      // _find_support_in_direction_of_origin_ray (mpr.py:180-188)
    kMprV2 = 2,      // _find_support_perpendicular_to_plane_containing_origin_v01 (:191-205)
    kMprV3 = 3,      // the discovery loop of _discover_portal (:140-160, 217-235)
    kMprRefine = 4,  // _refine_portal (:253-283)
    kMprPen = 5,     // _find_penetration_info (:332-346)
};
constexpr int kMprRefineCap = 0x100;
constexpr int kMprBadInput = 0x200;

__global__ __launch_bounds__(kMprBlock) void mpr_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const double *__restrict__ centers, int64_t n, double tol, int max_iter, int penetration,
    int serial_max, int32_t *__restrict__ status_out, double *__restrict__ out) {
    const int64_t pid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = pid < n;
    Shape A = empty_shape(), B = empty_shape();
    bool ok = false;
    int ia = 0, ib = 0;
    if (valid) {
        ia = pa[pid];
        ib = pb[pid];
        const bool okA = load_checked(s, ia, A);
        const bool okB = load_checked(s, ib, B);
        ok = okA && okB;
    }
    MprPortal P;
#pragma unroll
    for (int k = 0; k < 4; ++k) P.v[k] = P.a[k] = P.b[k] = mk(0.0, 0.0, 0.0);
    double res[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) res[k] = NAN;
    int status = 0, phase = kMprDone, it = 0;
    v3 d = mk(0.0, 0.0, 0.0);
    if (ok) {
        // _find_origin_ray (mpr.py:163-177)
        const v3 ca = mk(centers[3 * (int64_t)ia], centers[3 * (int64_t)ia + 1], centers[3 * (int64_t)ia + 2]);
        const v3 cb = mk(centers[3 * (int64_t)ib], centers[3 * (int64_t)ib + 1], centers[3 * (int64_t)ib + 2]);
        P.v[0] = ca - cb;
        P.a[0] = ca;
        P.b[0] = cb;
        if (P.v[0].x == 0.0 && P.v[0].y == 0.0 && P.v[0].z == 0.0) P.v[0].x += kEps * 10.0;
        d = norm_vector(-P.v[0]);
        phase = kMprV1;
    }
    // the refinement has succeeded: penetration info, or done
    auto intersecting = [&]() {
        if (penetration) {
            phase = kMprPen;
            it = 0;
            d = mpr_portal_dir(P);
        } else {
            status = 1;
            phase = kMprDone;
        }
    };
    // set up a refinement round along the current portal
    auto refine_round = [&]() {
        d = mpr_portal_dir(P);
        if (mpr_encapsulates(P.v[1], d)) {
            intersecting();
        } else if (it >= max_iter) {
            // the reference refines without bound; here it gives up
            status = kMprRefineCap;
            phase = kMprDone;
        } else {
            phase = kMprRefine;
        }
    };
    while (__ballot(phase != kMprDone) != 0ull) {
        const bool want = phase != kMprDone;
        const v3 sa = support_wave(s, A, d, want, serial_max);
        const v3 sb = support_wave(s, B, -d, want, serial_max);
        if (!want) continue;
        const v3 w = sa - sb;
        if (phase == kMprV1) {
            mpr_set(P, 1, w, sa, sb);
            const bool v1_zero = w.x == 0.0 && w.y == 0.0 && w.z == 0.0;
            if (!v1_zero && dot(w, d) < kEps) {
                phase = kMprDone;  // origin outside
                continue;
            }
            d = cross(P.v[0], P.v[1]);
            if (dot(d, d) < kEps) {
                status = 1;
                phase = kMprDone;
                const v3 pos = (P.a[1] + P.b[1]) * 0.5;
                if (v1_zero) {
                    // _find_penetration_touch (mpr.py:361-367)
                    res[0] = 0.0;
                    res[1] = 0.0; res[2] = 0.0; res[3] = 0.0;
                } else {
                    // _find_penetration_segment (mpr.py:370-378)
                    const v3 dir = norm_vector(P.v[1]);
                    res[0] = vnorm(P.v[1]);
                    res[1] = dir.x; res[2] = dir.y; res[3] = dir.z;
                }
                res[4] = pos.x; res[5] = pos.y; res[6] = pos.z;
                continue;
            }
            d = norm_vector(d);
            phase = kMprV2;
        } else if (phase == kMprV2) {
            mpr_set(P, 2, w, sa, sb);
            if (dot(w, d) < kEps) {
                phase = kMprDone;
                continue;
            }
            // _search_direction_perpendicular_to_plane_containing_v012 (mpr.py:208-214)
            d = norm_vector(cross(P.v[1] - P.v[0], P.v[2] - P.v[0]));
            if (dot(d, P.v[0]) > 0.0) {
                const v3 tv = P.v[1], ta = P.a[1], tb = P.b[1];
                P.v[1] = P.v[2]; P.a[1] = P.a[2]; P.b[1] = P.b[2];
                P.v[2] = tv; P.a[2] = ta; P.b[2] = tb;
                d = d * -1.0;
            }
            it = 0;
            phase = kMprV3;
        } else if (phase == kMprV3) {
            mpr_set(P, 3, w, sa, sb);
            if (dot(w, d) < kEps) {
                phase = kMprDone;
                continue;
            }
            // _iterate_discover_portal (mpr.py:217-235)
            bool cont = false;
            if (dot(cross(P.v[1], P.v[3]), P.v[0]) < kEps) {
                P.v[2] = P.v[3]; P.a[2] = P.a[3]; P.b[2] = P.b[3];
                cont = true;
            }
            if (!cont && dot(cross(P.v[3], P.v[2]), P.v[0]) < kEps) {
                P.v[1] = P.v[3]; P.a[1] = P.a[3]; P.b[1] = P.b[3];
                cont = true;
            }
            if (cont) d = norm_vector(cross(P.v[1] - P.v[0], P.v[2] - P.v[0]));
            ++it;
            if (!cont || it >= max_iter) {
                it = 0;
                refine_round();
            }
        } else if (phase == kMprRefine) {
            if (!mpr_encapsulates(w, d) || mpr_reach_tol(P, w, d, tol)) {
                phase = kMprDone;  // separated
                continue;
            }
            mpr_expand(P, w, sa, sb);
            ++it;
            refine_round();
        } else {  // kMprPen
            if (mpr_reach_tol(P, w, d, tol) || it > max_iter) {
                // _penetration_info (mpr.py:349-358)
                v3 cp;
                const double depth = origin_to_triangle(P.v[1], P.v[2], P.v[3], cp);
                v3 dir = vsel(fabs(depth) < kEps, mk(0.0, 0.0, 0.0), cp);
                dir = norm_vector(dir);
                const v3 pos = mpr_contact(P, mpr_portal_dir(P));
                res[0] = depth;
                res[1] = dir.x; res[2] = dir.y; res[3] = dir.z;
                res[4] = pos.x; res[5] = pos.y; res[6] = pos.z;
                status = 1;
                phase = kMprDone;
                continue;
            }
            mpr_expand(P, w, sa, sb);
            ++it;
            d = mpr_portal_dir(P);
        }
    }
    if (!valid) return;
    if (!ok) status = kMprBadInput;
    status_out[pid] = status;
    if (out) {
        double *o = out + 7 * pid;
#pragma unroll
        for (int k = 0; k < 7; ++k) o[k] = res[k];
    }
}

// ------------------------------------------------------ the queued machine

// The portal's support points are the pair's LDS rows (a: P, b: Q); its points
// v are their differences, except v0, which may have been moved off zero.
struct MprState {
    v3 d, v0;
    int phase, it, status, found;
};

// what the result comes from
enum : int { kMprNone = 0, kMprTouch = 1, kMprSegment = 2, kMprPortal = 3 };

struct MprOut {
    const double *centers;
    double tol;
    int max_iter, penetration;
    int32_t *status;
    double *out;
};

__device__ __forceinline__ v3 mpr_row(const PQ &pq, int r) { return pq.P(r) - pq.Q(r); }

__device__ __forceinline__ v3 portal_dir(v3 v1, v3 v2, v3 v3_) {
    return norm_vector(cross(v2 - v1, v3_ - v1));
}

__device__ __forceinline__ bool portal_reach_tol(v3 v1, v3 v2, v3 v3_, v3 v4, v3 d, double tol) {
    const double p = dot(v4, d);
    double m = p - dot(v1, d);
    const double t2 = p - dot(v2, d);
    if (t2 < m) m = t2;
    const double t3 = p - dot(v3_, d);
    if (t3 < m) m = t3;
    return m < tol + kEps;
}

struct MprMode {
    using State = MprState;
    using Out = MprOut;
    static __device__ __forceinline__ void clear(State &g, const PQ &) {
        g.d = g.v0 = mk(0.0, 0.0, 0.0);
        g.phase = kMprDone;
        g.it = g.status = 0;
        g.found = kMprNone;
    }
    // _find_origin_ray (mpr.py:163-177)
    static __device__ __forceinline__ bool start(State &g, const PQ &pq, int ia, int ib,
                                                 const d3d_gjk_params &, const Out &o) {
        const double *ca = o.centers + 3 * (int64_t)ia, *cb = o.centers + 3 * (int64_t)ib;
        const v3 a = mk(ca[0], ca[1], ca[2]), b = mk(cb[0], cb[1], cb[2]);
        pq.put(0, a, b);
        g.v0 = a - b;
        if (g.v0.x == 0.0 && g.v0.y == 0.0 && g.v0.z == 0.0) g.v0.x += kEps * 10.0;
        g.d = norm_vector(-g.v0);
        g.phase = kMprV1;
        g.it = g.status = 0;
        g.found = kMprNone;
        return true;
    }
    static __device__ __forceinline__ bool more(State &, const d3d_gjk_params &) { return true; }

    // a refinement round along the portal v1 v2 v3, or what follows the last one
    static __device__ __forceinline__ bool refine_round(State &g, const Out &o, v3 v1, v3 v2, v3 v3_) {
        g.d = portal_dir(v1, v2, v3_);
        if (mpr_encapsulates(v1, g.d)) {
            g.it = 0;
            if (o.penetration) {
                g.phase = kMprPen;
                return true;
            }
            g.status = 1;
            return false;
        }
        if (g.it >= o.max_iter) {
            // the reference refines without bound; here it gives up
            g.status = kMprRefineCap;
            return false;
        }
        g.phase = kMprRefine;
        return true;
    }

    template <int G>
    static __device__ __forceinline__ bool step(State &g, const PQ &pq, v3 p, v3 q,
                                                const d3d_gjk_params &, const Out &o) {
        // all lanes of the group read the rows its first lane wrote in earlier rounds
        row_fence();
        const v3 w = p - q;
        if (g.phase == kMprV1) {
            pq.put(1, p, q);
            const bool v1_zero = w.x == 0.0 && w.y == 0.0 && w.z == 0.0;
            if (!v1_zero && dot(w, g.d) < kEps) return false;  // origin outside
            g.d = cross(g.v0, w);
            if (dot(g.d, g.d) < kEps) {
                g.status = 1;
                g.found = v1_zero ? kMprTouch : kMprSegment;
                return false;
            }
            g.d = norm_vector(g.d);
            g.phase = kMprV2;
            return true;
        }
        const v3 r1 = mpr_row(pq, 1);
        if (g.phase == kMprV2) {
            if (dot(w, g.d) < kEps) return false;
            // _search_direction_perpendicular_to_plane_containing_v012 (mpr.py:208-214)
            g.d = norm_vector(cross(r1 - g.v0, w - g.v0));
            const bool swap = dot(g.d, g.v0) > 0.0;
            if (swap) g.d = g.d * -1.0;
            // rows 1 and 2, exchanged when the direction points away
            if (swap) pq.move(1, 2);
            pq.put(swap ? 1 : 2, p, q);
            g.it = 0;
            g.phase = kMprV3;
            return true;
        }
        const v3 r2 = mpr_row(pq, 2);
        v3 v1 = r1, v2 = r2, v3_ = w;
        if (g.phase == kMprV3) {
            if (dot(w, g.d) < kEps) return false;
            // _iterate_discover_portal (mpr.py:217-235): the new row is row 3 and,
            // where the portal misses the origin ray, takes row 2's or row 1's place
            pq.put(3, p, q);
            const bool c2 = dot(cross(v1, w), g.v0) < kEps;
            const bool c1 = !c2 && dot(cross(w, v2), g.v0) < kEps;
            if (c1 || c2) {
                pq.put(c2 ? 2 : 1, p, q);
                v1 = vsel(c1, w, v1);
                v2 = vsel(c2, w, v2);
                g.d = norm_vector(cross(v1 - g.v0, v2 - g.v0));
            }
            ++g.it;
            if ((c1 || c2) && g.it < o.max_iter) return true;
            g.it = 0;
            return refine_round(g, o, v1, v2, v3_);
        }
        v3_ = mpr_row(pq, 3);
        const bool reached = portal_reach_tol(v1, v2, v3_, w, g.d, o.tol);
        if (g.phase == kMprRefine) {
            if (!mpr_encapsulates(w, g.d) || reached) return false;  // separated
        } else if (reached || g.it > o.max_iter) {
            g.status = 1;
            g.found = kMprPortal;
            return false;
        }
        // _expand_portal (mpr.py:314-329)
        const v3 x = cross(w, g.v0);
        const int r = dot(v1, x) > 0.0 ? (dot(v2, x) > 0.0 ? 1 : 3) : (dot(v3_, x) > 0.0 ? 2 : 1);
        pq.put(r, p, q);
        v1 = vsel(r == 1, w, v1);
        v2 = vsel(r == 2, w, v2);
        v3_ = vsel(r == 3, w, v3_);
        ++g.it;
        if (g.phase == kMprRefine) return refine_round(g, o, v1, v2, v3_);
        g.d = portal_dir(v1, v2, v3_);
        return true;
    }

    static __device__ __forceinline__ void write(const State &g, const PQ &pq, int64_t pid,
                                                 const d3d_gjk_params &, const Out &o) {
        o.status[pid] = g.status;
        if (!o.out) return;
        double *r = o.out + 7 * pid;
        if (g.found == kMprNone) {
#pragma unroll
            for (int k = 0; k < 7; ++k) r[k] = NAN;
            return;
        }
        double depth = 0.0;
        v3 dir = mk(0.0, 0.0, 0.0), pos;
        if (g.found == kMprPortal) {
            // _penetration_info (mpr.py:349-358)
            MprPortal P;
            P.v[0] = g.v0;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                P.a[k] = pq.P(k);
                P.b[k] = pq.Q(k);
                if (k > 0) P.v[k] = P.a[k] - P.b[k];
            }
            v3 cp;
            depth = origin_to_triangle(P.v[1], P.v[2], P.v[3], cp);
            dir = norm_vector(vsel(fabs(depth) < kEps, mk(0.0, 0.0, 0.0), cp));
            pos = mpr_contact(P, mpr_portal_dir(P));
        } else {
            pos = (pq.P(1) + pq.Q(1)) * 0.5;
            if (g.found == kMprSegment) {
                // _find_penetration_segment (mpr.py:370-378)
                const v3 v1 = mpr_row(pq, 1);
                dir = norm_vector(v1);
                depth = vnorm(v1);
            }
        }
        r[0] = depth;
        r[1] = dir.x; r[2] = dir.y; r[3] = dir.z;
        r[4] = pos.x; r[5] = pos.y; r[6] = pos.z;
    }
    static __device__ __forceinline__ void bad(int64_t pid, const Out &o) {
        o.status[pid] = kMprBadInput;
        if (!o.out) return;
#pragma unroll
        for (int k = 0; k < 7; ++k) o.out[7 * pid + k] = NAN;
    }
};

// Bound like the other queue kernels: latency of the hull sweeps and of the FP64
// chains.  Occupancy 2 keeps the portal machine free of spills: 262,144 mixed
// pairs 672 us, 734 us at occupancy 3 with 196 spilled VGPRs, and 1,068 us one
// lane per pair in list order (mpr_kernel); 262,144 pairs of 32-vertex hulls 497,
// 515 and 1,077 us.
constexpr int kMprBlocksPerCu = 2;
__global__ __launch_bounds__(kQBlock) __attribute__((amdgpu_waves_per_eu(2))) void mpr_all_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const int32_t *__restrict__ order, const int32_t *__restrict__ cls_begin,
    const int32_t *__restrict__ cls_count, int32_t *__restrict__ cls_cursor, d3d_gjk_params prm,
    MprOut o) {
    __shared__ double pq_lds[24 * kQBlock];
    run_all<MprMode>(s, pa, pb, order, cls_begin, cls_count, cls_cursor, prm, o, pq_lds);
}

}  // namespace d3d

using namespace d3d;

extern "C" int d3d_mpr_batch(const d3d_scene *scene, const int32_t *pair_a, const int32_t *pair_b,
                             const double *centers, int64_t n, double tolerance,
                             int32_t max_iterations, int32_t penetration, int32_t *status,
                             double *out, void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(pair_a && pair_b && centers && status, "NULL buffer");
    D3D_CHECK_ARG(penetration == 0 || out, "out is NULL but penetration was requested");
    D3D_CHECK_ARG(max_iterations > 0, "max_iterations must be > 0");
    hipLaunchKernelGGL(mpr_kernel, dim3(grid_for(n, kMprBlock)), dim3(kMprBlock), 0,
                       (hipStream_t)stream, *scene, pair_a, pair_b, centers, n, tolerance,
                       max_iterations, penetration, kMprSerialMax, status, out);
    D3D_CHECK_LAUNCH("mpr_kernel");
    return D3D_OK;
}

// Pairs below which the sort costs more than it saves: lane per pair and queue
// take 13.7 and 19.0 us for 8 mixed pairs, 19.7 and 21.1 for 16, 35.8 and 23.7
// for 32.  A scene without hulls has nothing to sort for (262,144 pairs of boxes
// 56 and 77 us).
constexpr int64_t kMprQueueMin = D3D_MPR_QUEUE_MIN;

extern "C" int d3d_mpr_batch_ws(const d3d_scene *scene, const int32_t *pair_a, const int32_t *pair_b,
                                const double *centers, int64_t n, double tolerance,
                                int32_t max_iterations, int32_t penetration, int32_t *status,
                                double *out, void *workspace, int64_t workspace_bytes,
                                void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(pair_a && pair_b && centers && status, "NULL buffer");
    D3D_CHECK_ARG(penetration == 0 || out, "out is NULL but penetration was requested");
    D3D_CHECK_ARG(max_iterations > 0, "max_iterations must be > 0");
    if (n < kMprQueueMin || n >= (int64_t)0x7fffffff || scene->n_vertices == 0)
        return d3d_mpr_batch(scene, pair_a, pair_b, centers, n, tolerance, max_iterations, penetration,
                             status, out, stream);
    D3D_CHECK_ARG(workspace, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= d3d_gjk_workspace_bytes(n), "workspace too small");
    d3d_gjk_params prm = default_params();
    prm.blocks_per_cu = kMprBlocksPerCu;
    const d3d_gjk_params rp = queue_params(prm, n, 0);
    const QueueWs w = ws_view(workspace, n);
    if (int rc = queue_sort(*scene, pair_a, pair_b, n, w, (hipStream_t)stream)) return rc;
    hipLaunchKernelGGL(mpr_all_kernel, dim3(queue_grid(rp)), dim3(kQBlock), 0, (hipStream_t)stream,
                       *scene, pair_a, pair_b, w.order, w.cls_begin, w.cls_count, w.cls_cursor, rp,
                       MprOut{centers, tolerance, max_iterations, penetration, status, out});
    D3D_CHECK_LAUNCH("mpr_all_kernel");
    return D3D_OK;
}
