// d3d_gjk_queue.hip -- batched GJK distance and intersection as a sorted,
// queue-fed pipeline (d3d_queue.hpp).
//
// 1. classify + counting sort (device): every pair gets a key
//        work class (8 size classes of the pair's hull vertices, for pairs of
//        at most one hull and for pairs of two)
//        x collider type of A x collider type of B
//    and the pair indices are scattered into `order`, grouped by key.  Pairs
//    of one class have similar support-sweep cost and, within a class, run
//    next to pairs of the same type combination, so the type switch of the
//    analytic supports stays wave-uniform.
// 2. one persistent kernel over all classes, G lanes per pair (G from the tuning
//    table; 1 for analytic pairs, more for big hulls).  The G lanes of a pair
//    hold identical FP64 simplex state; hull sweeps stride over the vertices by
//    G and reduce inside the group.  Each group takes its next pair from its
//    wavefront's claim on the class as soon as its current pair terminates, so
//    lanes do not idle on the slowest pair of a wave.
// Counts and offsets stay on the device: no host synchronisation inside a
// batch.
#include <array>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "d3d_queue.hpp"

namespace d3d {

// Clears the header with a fill kernel (no memset node, so the sequence can
// be captured in a graph and replayed).
__global__ void queue_clear_kernel(int32_t *hdr, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) hdr[i] = 0;
}

// Counting and scattering go over tiles of kSortThreads * kItems pairs, a tile
// per block: every block adds its counts of the keys it met to a few hundred
// global counters, so a large batch takes large tiles (see queue_sort).
constexpr int kSortThreads = 512;

// The keys of a thread's pairs of a tile (-1 past the end), with the loads of
// all of them out together.
template <int kItems>
__device__ __forceinline__ void tile_keys(const d3d_scene &s, const int32_t *__restrict__ pa,
                                          const int32_t *__restrict__ pb, int64_t n, int64_t base,
                                          int (&key)[kItems]) {
    int a[kItems], b[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const int64_t i = base + j * kSortThreads + threadIdx.x;
        a[j] = i < n ? pa[i] : -1;
        b[j] = i < n ? pb[i] : -1;
    }
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const int64_t i = base + j * kSortThreads + threadIdx.x;
        const int k = pair_key(s, a[j], b[j]);
        key[j] = i < n ? k : -1;
    }
}

template <int kItems>
__global__ __launch_bounds__(kSortThreads) void queue_hist_kernel(d3d_scene s,
                                                                  const int32_t *__restrict__ pa,
                                                                  const int32_t *__restrict__ pb,
                                                                  int64_t n,
                                                                  int32_t *__restrict__ hist) {
    __shared__ int32_t h[kNumKeys];
    for (int i = threadIdx.x; i < kNumKeys; i += kSortThreads) h[i] = 0;
    int key[kItems];
    tile_keys<kItems>(s, pa, pb, n, (int64_t)blockIdx.x * kSortThreads * kItems, key);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j)
        if (key[j] >= 0) atomicAdd(&h[key[j]], 1);
    __syncthreads();
    for (int i = threadIdx.x; i < kNumKeys; i += kSortThreads)
        if (h[i]) atomicAdd(&hist[i], h[i]);
}

// Single-block exclusive scan over keys; class ranges follow from the key
// order (class-major).
__global__ __launch_bounds__(kQBlock) void queue_scan_kernel(int32_t *__restrict__ hist,
                                                             int32_t *__restrict__ key_off,
                                                             int32_t *__restrict__ cls_begin,
                                                             int32_t *__restrict__ cls_count) {
    __shared__ int32_t part[kQBlock];
    constexpr int per = (kNumKeys + kQBlock - 1) / kQBlock;
    const int t = threadIdx.x;
    int local = 0;
    for (int j = 0; j < per; ++j) {
        const int k = t * per + j;
        if (k < kNumKeys) local += hist[k];
    }
    part[t] = local;
    __syncthreads();
    for (int off = 1; off < kQBlock; off <<= 1) {
        const int v = (t >= off) ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = part[t] - local;
    for (int j = 0; j < per; ++j) {
        const int k = t * per + j;
        if (k < kNumKeys) {
            key_off[k] = run;
            run += hist[k];
        }
    }
    __syncthreads();
    if (t < kNumClasses) {
        const int k0 = t * kNumTypes * kNumTypes;
        const int k1 = k0 + kNumTypes * kNumTypes;
        int c = 0;
        for (int k = k0; k < k1; ++k) c += hist[k];
        cls_begin[t] = key_off[k0];
        cls_count[t] = c;
    }
}

template <int kItems>
__global__ __launch_bounds__(kSortThreads) void queue_scatter_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb, int64_t n,
    const int32_t *__restrict__ key_off, int32_t *__restrict__ key_cur,
    int32_t *__restrict__ order) {
    __shared__ int32_t h[kNumKeys];
    for (int i = threadIdx.x; i < kNumKeys; i += kSortThreads) h[i] = 0;
    const int64_t base = (int64_t)blockIdx.x * kSortThreads * kItems;
    int key[kItems], rank[kItems];
    tile_keys<kItems>(s, pa, pb, n, base, key);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) rank[j] = key[j] >= 0 ? atomicAdd(&h[key[j]], 1) : 0;
    __syncthreads();
    // the tile's place among the pairs of each key it met
    for (int k = threadIdx.x; k < kNumKeys; k += kSortThreads)
        if (h[k]) h[k] = key_off[k] + atomicAdd(&key_cur[k], h[k]);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j)
        if (key[j] >= 0)
            order[h[key[j]] + rank[j]] = (int32_t)(base + j * kSortThreads + threadIdx.x);
}

// the EPA list counter and the EPA claim cursor
__global__ void zero_u64_kernel(unsigned long long *c) {
    c[0] = 0ull;
    c[1] = 0ull;
}

// The whole sort of a small batch by one block: counts, scan and ranks in LDS,
// with the class cursors and the optional EPA counters cleared on the way.
// A whole GJK + EPA call with the four-launch sort and with this one: 1 pair 51
// and 42 us, 64 mixed pairs 294 and 282 us, 2,048 hull pairs 142 and 135 us,
// 4,096 mixed pairs 739 and 728 us; from 8,192 pairs on one block's chain of
// loads is the longer one (hull pairs 176 and 181 us, 16,384 pairs 221 and 240).
constexpr int kSmallSort = 4096;
constexpr int kSmallBlock = 1024;

__global__ __launch_bounds__(kSmallBlock) void queue_small_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb, int n, QueueWs w,
    unsigned long long *__restrict__ epa_count) {
    __shared__ int32_t h[kNumKeys];
    __shared__ uint16_t key[kSmallSort], rank[kSmallSort];
    __shared__ int32_t wsum[kSmallBlock / kWave];
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    for (int k = t; k < kNumKeys; k += kSmallBlock) h[k] = 0;
    if (t < kNumClasses) w.cls_cursor[t] = 0;
    if (epa_count && t < 2) epa_count[t] = 0ull;
    __syncthreads();
    // the keys of four pairs at a time, so that their loads go out together
    for (int b = 0; b < n; b += 4 * kSmallBlock) {
        int a4[4], b4[4], k4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = b + j * kSmallBlock + t;
            a4[j] = i < n ? pa[i] : -1;
            b4[j] = i < n ? pb[i] : -1;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) k4[j] = pair_key(s, a4[j], b4[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = b + j * kSmallBlock + t;
            if (i < n) {
                key[i] = (uint16_t)k4[j];
                rank[i] = (uint16_t)atomicAdd(&h[k4[j]], 1);
            }
        }
    }
    __syncthreads();
    // exclusive scan of the counts, two keys per thread
    static_assert(kNumKeys <= 2 * kSmallBlock && kNumKeys % 2 == 0, "two keys per thread");
    const bool in = 2 * t < kNumKeys;
    const int c0 = in ? h[2 * t] : 0, c1 = in ? h[2 * t + 1] : 0;
    int incl = c0 + c1;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
    }
    if (lane == kWave - 1) wsum[wave] = incl;
    __syncthreads();
    int first = incl - c0 - c1;
    for (int k = 0; k < wave; ++k) first += wsum[k];
    if (in) {
        h[2 * t] = first;
        h[2 * t + 1] = first + c0;
    }
    __syncthreads();
    if (t < kNumClasses) {
        constexpr int per = kNumTypes * kNumTypes;
        const int b = h[t * per], e = t + 1 < kNumClasses ? h[(t + 1) * per] : n;
        w.cls_begin[t] = b;
        w.cls_count[t] = e - b;
    }
    for (int i = t; i < n; i += kSmallBlock) w.order[h[key[i]] + rank[i]] = i;
}

// ------------------------------------------------------------- GJK state

struct GjkState {
    Simplex S;
    v3 d;
    double vv, prev;
    int it, state;
};

__device__ __forceinline__ void gjk_init(GjkState &g, const PQ &pq) {
    simplex_zero(g.S);
    pq.zero();
    g.d = mk(1.0, 0.0, 0.0);
    g.vv = dot(g.d, g.d);
    g.prev = kMaxFloat;
    g.it = 0;
    g.state = -1;
}

// Y rows are P - Q rows (w = p - q when a row is appended; compaction moves
// Y, P, Q rows alike; zero rows stay zero), so Y is rebuilt from the LDS rows
// at the start of each step instead of being held in registers across the
// supports.  Row for row the values are the ones the reference keeps in Y.
__device__ __forceinline__ void load_y(Simplex &S, const PQ &pq) {
    S.Y0 = pq.P(0) - pq.Q(0);
    S.Y1 = pq.P(1) - pq.Q(1);
    S.Y2 = pq.P(2) - pq.Q(2);
    S.Y3 = pq.P(3) - pq.Q(3);
}

// One pass of _distance_loop (_gjk_jolt.py:224-288) given the supports p, q.
// Returns false once the pair has terminated (g.state set).
__device__ __forceinline__ bool gjk_distance_step(GjkState &g, const PQ &pq, v3 p, v3 q,
                                                  double maxd2, double tol2) {
    ++g.it;
    const v3 w = p - q;
    const double dw = dot(g.d, w);
    if (dw < 0.0 && dw * dw > g.vv * maxd2) {
        g.state = D3D_CLIPPED;
        return false;
    }
    // the new row is read back from LDS with the others (selecting it into place
    // in registers took two dozen selects per step: 1,048,576 mixed pairs 5,240 us,
    // 5,131 us this way); the group's lanes see what its first lane wrote
    pq.put(g.S.n < 3 ? g.S.n : 3, p, q);
    row_fence();
    load_y(g.S, pq);
    g.S.n += 1;
    v3 nvec;
    double nvv;
    int set;
    if (closest_to_origin(g.S, g.prev, nvec, nvv, set)) {
        g.d = nvec;
        g.vv = nvv;
    } else {
        g.S.n -= 1;
        set = (1 << g.S.n) - 1;
    }
    if (set == 15) {
        g.vv = 0.0;
        g.state = D3D_INTERSECT;
        return false;
    }
    // compaction moves the P/Q rows only: the next step rebuilds Y from them,
    // and the test below reads the kept rows of Y where they are
    const double ymax = max_y_len_sq_kept(g.S, set);
    const CompactMap cm = compact_map(g.S.n, set);
    pq.compact(cm);
    g.S.n = cm.m;
    if (g.vv <= tol2 || g.vv <= kEps * ymax) {
        g.vv = 0.0;
        g.state = D3D_INTERSECT;
        return false;
    }
    g.d = -g.d;
    if (g.prev - g.vv <= kEps * g.prev) {
        g.state = D3D_SEPARATED;
        return false;
    }
    g.prev = g.vv;
    return true;
}

struct GjkOut {
    double *dist, *cpa, *cpb;
    int32_t *status, *iters;
    double *simplex;
    int32_t *npts;
    bool simplex_hits_only;  // write simplex / npts only for intersecting pairs
    // GJK -> EPA (all null without EPA): intersecting pairs are appended to
    // epa_work (epa_count counts them); the others get EPA status -1 and a
    // zero output row
    int32_t *epa_work;
    unsigned long long *epa_count;
    double *epa_out;
    int32_t *epa_status;
};

__device__ __forceinline__ void epa_route(int64_t pid, bool intersecting, const GjkOut &o) {
    if (!o.epa_work) return;
    if (intersecting) {
        o.epa_work[atomicAdd(o.epa_count, 1ull)] = (int32_t)pid;
    } else {
#pragma unroll
        for (int k = 0; k < 13; ++k) o.epa_out[13 * pid + k] = 0.0;
        o.epa_status[pid] = -1;
    }
}

// calculate_closest_points (_gjk_jolt.py:667-687)
__device__ __forceinline__ void closest_points(const Simplex &S, const PQ &pq, v3 &a, v3 &b) {
    if (S.n == 1) {
        a = pq.P(0);
        b = pq.Q(0);
    } else if (S.n == 2) {
        double u, v;
        bary_line(S.Y0, S.Y1, u, v);
        a = pq.P(0) * u + pq.P(1) * v;
        b = pq.Q(0) * u + pq.Q(1) * v;
    } else if (S.n == 3) {
        double u, v, w;
        bary_plane(S.Y0, S.Y1, S.Y2, u, v, w);
        a = (pq.P(0) * u + pq.P(1) * v) + pq.P(2) * w;
        b = (pq.Q(0) * u + pq.Q(1) * v) + pq.Q(2) * w;
    } else {
        double u, v, w, x;
        bary_tetra(S.Y0, S.Y1, S.Y2, S.Y3, u, v, w, x);
        a = ((pq.P(0) * u + pq.P(1) * v) + pq.P(2) * w) + pq.P(3) * x;
        b = ((pq.Q(0) * u + pq.Q(1) * v) + pq.Q(2) * w) + pq.Q(3) * x;
    }
}

// End of gjk_distance_jolt (_gjk_jolt.py:207-221).
__device__ __forceinline__ void gjk_write(const GjkState &g, const PQ &pq, int64_t pid,
                                          double sanity, const GjkOut &o) {
    if (o.iters) o.iters[pid] = g.it;
    epa_route(pid, g.state == D3D_INTERSECT, o);
    Simplex S = g.S;
    load_y(S, pq);
    const bool want_s = !o.simplex_hits_only || g.state == D3D_INTERSECT;
    if (o.npts && want_s) o.npts[pid] = g.S.n;
    if (o.simplex && want_s) {
        double *w = o.simplex + 36 * pid;
        const v3 y[4] = {S.Y0, S.Y1, S.Y2, S.Y3};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const v3 P = pq.P(k), Q = pq.Q(k);
            w[3 * k] = y[k].x;
            w[3 * k + 1] = y[k].y;
            w[3 * k + 2] = y[k].z;
            w[12 + 3 * k] = P.x;
            w[13 + 3 * k] = P.y;
            w[14 + 3 * k] = P.z;
            w[24 + 3 * k] = Q.x;
            w[25 + 3 * k] = Q.y;
            w[26 + 3 * k] = Q.z;
        }
    }
    if (g.state == D3D_CLIPPED) {
        o.dist[pid] = kMaxFloat;
        o.cpa[3 * pid] = o.cpa[3 * pid + 1] = o.cpa[3 * pid + 2] = NAN;
        o.cpb[3 * pid] = o.cpb[3 * pid + 1] = o.cpb[3 * pid + 2] = NAN;
        o.status[pid] = D3D_CLIPPED;
        return;
    }
    v3 a, b;
    closest_points(S, pq, a, b);
    int st = g.state;
    if (!(fabs(dot(g.d, g.d) - g.vv) < sanity)) st |= D3D_SANITY_FAILED;
    const double dd = sqrt(g.vv);
    if (dd < kEps) {
        const v3 m = (a + b) * 0.5;
        a = m;
        b = m;
    }
    o.dist[pid] = dd;
    o.cpa[3 * pid] = a.x;
    o.cpa[3 * pid + 1] = a.y;
    o.cpa[3 * pid + 2] = a.z;
    o.cpb[3 * pid] = b.x;
    o.cpb[3 * pid + 1] = b.y;
    o.cpb[3 * pid + 2] = b.z;
    o.status[pid] = st;
}

__device__ __forceinline__ void gjk_write_bad(int64_t pid, const GjkOut &o) {
    o.dist[pid] = NAN;
    o.cpa[3 * pid] = o.cpa[3 * pid + 1] = o.cpa[3 * pid + 2] = NAN;
    o.cpb[3 * pid] = o.cpb[3 * pid + 1] = o.cpb[3 * pid + 2] = NAN;
    o.status[pid] = kBadInput;
    if (o.iters) o.iters[pid] = 0;
    if (o.npts) o.npts[pid] = 0;
    epa_route(pid, false, o);
}

// GJK distance as a queue Mode.
struct DistanceMode {
    using State = GjkState;
    using Out = GjkOut;
    static __device__ __forceinline__ void clear(State &g, const PQ &pq) { gjk_init(g, pq); }
    static __device__ __forceinline__ bool start(State &g, const PQ &pq, int, int,
                                                 const d3d_gjk_params &, const Out &) {
        gjk_init(g, pq);
        return true;
    }
    static __device__ __forceinline__ bool more(State &g, const d3d_gjk_params &prm) {
        if (g.it < prm.max_iterations) return true;
        g.state = D3D_ITER_CAP;
        return false;
    }
    template <int G>
    static __device__ __forceinline__ bool step(State &g, const PQ &pq, v3 p, v3 q,
                                                const d3d_gjk_params &prm, const Out &) {
        return gjk_distance_step(g, pq, p, q, prm.max_distance_squared,
                                 prm.tolerance * prm.tolerance);
    }
    static __device__ __forceinline__ void write(const State &g, const PQ &pq, int64_t pid,
                                                 const d3d_gjk_params &prm, const Out &o) {
        gjk_write(g, pq, pid, prm.sanity_check, o);
    }
    static __device__ __forceinline__ void bad(int64_t pid, const Out &o) { gjk_write_bad(pid, o); }
};

// Occupancy 3 (<= 168 VGPRs, a hundred of them spilled) hides more latency when
// the chip is full; occupancy 2 spills nothing and is the faster one for a batch
// that does not fill it.  3 and 2: 64 mixed pairs 242 and 127 us, 1,024 mixed 279
// and 248, 4,096 mixed 418 and 424, 8,192 mixed 474 and 515, 1,048,576 mixed 5,318
// and 5,778; pairs of 32-vertex hulls, 64 41 and 36 us, 4,096 71 and 65.
constexpr int64_t kLooseMax = 4096;

__global__ __launch_bounds__(kQBlock) __attribute__((amdgpu_waves_per_eu(3))) void gjk_all_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const int32_t *__restrict__ order, const int32_t *__restrict__ cls_begin,
    const int32_t *__restrict__ cls_count, int32_t *__restrict__ cls_cursor, d3d_gjk_params prm,
    GjkOut o) {
    __shared__ double pq_lds[24 * kQBlock];
    run_all<DistanceMode>(s, pa, pb, order, cls_begin, cls_count, cls_cursor, prm, o, pq_lds);
}

__global__ __launch_bounds__(kQBlock) __attribute__((amdgpu_waves_per_eu(2))) void gjk_small_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const int32_t *__restrict__ order, const int32_t *__restrict__ cls_begin,
    const int32_t *__restrict__ cls_count, int32_t *__restrict__ cls_cursor, d3d_gjk_params prm,
    GjkOut o) {
    __shared__ double pq_lds[24 * kQBlock];
    run_all<DistanceMode>(s, pa, pb, order, cls_begin, cls_count, cls_cursor, prm, o, pq_lds);
}

// ------------------------------------------------------- GJK intersection

// The simplex of the intersection test holds Y alone: its rows go to the P half
// of the pair's LDS rows.
struct HitState {
    v3 d;
    double prev;
    int it, state, n;
};

struct HitOut {
    uint8_t *hit;
    int32_t *status;
};

// gjk_intersection_jolt (_gjk_jolt.py:29-80) and _intersection_loop (:83-135)
// as a queue Mode.
struct IntersectMode {
    using State = HitState;
    using Out = HitOut;
    static __device__ __forceinline__ void clear(State &g, const PQ &) {
        g.d = mk(1.0, 0.0, 0.0);
        g.prev = kMaxFloat;
        g.it = 0;
        g.state = -1;
        g.n = 0;
    }
    static __device__ __forceinline__ bool start(State &g, const PQ &pq, int, int,
                                                 const d3d_gjk_params &, const Out &) {
        clear(g, pq);
        return true;
    }
    static __device__ __forceinline__ bool more(State &g, const d3d_gjk_params &prm) {
        if (g.it < prm.max_iterations) return true;
        g.state = D3D_ITER_CAP;
        return false;
    }
    template <int G>
    static __device__ __forceinline__ bool step(State &g, const PQ &pq, v3 p, v3 q,
                                                const d3d_gjk_params &prm, const Out &) {
        ++g.it;
        const v3 w = p - q;
        g.state = D3D_SEPARATED;
        if (dot(g.d, w) < -kEps) return false;
        pq.put_p(g.n < 3 ? g.n : 3, w);
        row_fence();
        // rows past the new one are not used
        Simplex S;
        S.n = g.n + 1;
        S.Y0 = pq.P(0);
        S.Y1 = pq.P(1);
        S.Y2 = pq.P(2);
        S.Y3 = pq.P(3);
        v3 v;
        double vv;
        int set;
        if (!closest_to_origin(S, g.prev, v, vv, set)) return false;
        if (set == 15 || vv <= prm.tolerance * prm.tolerance || vv <= kEps * max_y_len_sq(S)) {
            g.state = D3D_INTERSECT;
            return false;
        }
        g.d = -v;
        if (g.prev - vv <= kEps * g.prev) return false;
        g.prev = vv;
        const CompactMap cm = compact_map(S.n, set);
        pq.compact<3>(cm);
        g.n = cm.m;
        return true;
    }
    static __device__ __forceinline__ void write(const State &g, const PQ &, int64_t pid,
                                                 const d3d_gjk_params &, const Out &o) {
        o.hit[pid] = g.state == D3D_INTERSECT ? 1 : 0;
        if (o.status) o.status[pid] = g.state;
    }
    static __device__ __forceinline__ void bad(int64_t pid, const Out &o) {
        o.hit[pid] = 0;
        if (o.status) o.status[pid] = kBadInput;
    }
};

// Bound like gjk_all_kernel (latency of the hull sweeps and of the FP64 chains),
// with about a quarter of its rounds.  262,144 mixed pairs: 401 us with the
// sort, against 740 us one lane per pair in list order, where a wavefront sweeps
// the hulls of its lanes one after the other in every round.  Occupancy 3 and 2
// as for the distance, with a later line since the rounds are few: 1,024 mixed
// pairs 71 and 56 us, 16,384 near ones 181 and 175, 65,536 302 and 302, 262,144
// 557 and 593.
constexpr int64_t kIntersectLooseMax = 65536;

__global__ __launch_bounds__(kQBlock) __attribute__((amdgpu_waves_per_eu(3))) void gjk_intersect_all_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const int32_t *__restrict__ order, const int32_t *__restrict__ cls_begin,
    const int32_t *__restrict__ cls_count, int32_t *__restrict__ cls_cursor, d3d_gjk_params prm,
    HitOut o) {
    __shared__ double pq_lds[24 * kQBlock];
    run_all<IntersectMode>(s, pa, pb, order, cls_begin, cls_count, cls_cursor, prm, o, pq_lds);
}

__global__ __launch_bounds__(kQBlock) __attribute__((amdgpu_waves_per_eu(2))) void gjk_intersect_small_kernel(
    d3d_scene s, const int32_t *__restrict__ pa, const int32_t *__restrict__ pb,
    const int32_t *__restrict__ order, const int32_t *__restrict__ cls_begin,
    const int32_t *__restrict__ cls_count, int32_t *__restrict__ cls_cursor, d3d_gjk_params prm,
    HitOut o) {
    __shared__ double pq_lds[24 * kQBlock];
    run_all<IntersectMode>(s, pa, pb, order, cls_begin, cls_count, cls_cursor, prm, o, pq_lds);
}

// ---------------------------------------------------------------- host

// the tuned table (distance3d_amd/tuning.json): lanes per class for the
// 1,048,576-pair mixed workload on one MI355X, class 11 from the EPA pairs
static const int kDefaultLanes[kNumClasses] = {1, 4, 16, 8, 16, 16, 32, 64,
                                               1, 8, 16, 8, 64, 16, 64, 64};

struct WsCache {
    std::mutex mu;
    std::map<std::pair<int, void *>, std::pair<void *, size_t>> bufs;
};
static WsCache g_ws;

static int workspace_for(void *stream, int64_t n, void **out) {
    int dev = 0;
    D3D_CHECK_HIP(hipGetDevice(&dev));
    const size_t need = (size_t)(ws_header_ints() + n) * sizeof(int32_t);
    std::lock_guard<std::mutex> lk(g_ws.mu);
    auto &e = g_ws.bufs[std::make_pair(dev, stream)];
    if (e.second < need) {
        if (e.first) {
            D3D_CHECK_HIP(hipStreamSynchronize((hipStream_t)stream));
            D3D_CHECK_HIP(hipFree(e.first));
            e.first = nullptr;
            e.second = 0;
        }
        const size_t grow = need + need / 4;
        D3D_CHECK_HIP(hipMalloc(&e.first, grow));
        e.second = grow;
    }
    *out = e.first;
    return D3D_OK;
}

static int cu_count() {
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            cus = 256;
    }
    return cus;
}

// EPA behind the GJK classes (after the join, on the caller's stream): the
// intersecting pairs are compacted into `work` and EPA runs over them.
struct EpaHook {
    int32_t *work;
    unsigned long long *count;
    int max_iter, max_faces;
    double eps;
    double *out;
    int32_t *status;
};

// ---------------------------------------------------------- stage timing

// Events of the calls recorded while stage timing is enabled: before the sort,
// before the GJK kernel, after it, after EPA.  Spent event sets are reused.
struct StageTiming {
    std::mutex mu;
    bool on = false;
    std::vector<std::array<hipEvent_t, 4>> rec, pool;
};
static StageTiming g_timing;

static bool stage_events(std::array<hipEvent_t, 4> &ev) {
    std::lock_guard<std::mutex> lk(g_timing.mu);
    if (!g_timing.on) return false;
    if (!g_timing.pool.empty()) {
        ev = g_timing.pool.back();
        g_timing.pool.pop_back();
    } else {
        for (auto &e : ev)
            if (hipEventCreate(&e) != hipSuccess) return false;
    }
    g_timing.rec.push_back(ev);
    return true;
}

int queue_sort(const d3d_scene &s, const int32_t *pa, const int32_t *pb, int64_t n, const QueueWs &w,
               hipStream_t stream, unsigned long long *epa_count) {
    if (n <= kSmallSort) {
        hipLaunchKernelGGL(queue_small_kernel, dim3(1), dim3(kSmallBlock), 0, stream, s, pa, pb, (int)n,
                           w, epa_count);
        D3D_CHECK_LAUNCH("queue_small_kernel");
        return D3D_OK;
    }
    if (epa_count) {
        hipLaunchKernelGGL(zero_u64_kernel, dim3(1), dim3(1), 0, stream, epa_count);
        D3D_CHECK_LAUNCH("zero_u64_kernel");
    }
    hipLaunchKernelGGL(queue_clear_kernel, dim3(4), dim3(kQBlock), 0, stream, w.hist,
                       (int)ws_header_ints());
    D3D_CHECK_LAUNCH("queue_clear_kernel");
    auto sort = [&](auto hist, auto scatter, int items) {
        const int64_t tile = (int64_t)kSortThreads * items;
        const unsigned blocks = (unsigned)((n + tile - 1) / tile);
        hipLaunchKernelGGL(hist, dim3(blocks), dim3(kSortThreads), 0, stream, s, pa, pb, n, w.hist);
        hipLaunchKernelGGL(queue_scan_kernel, dim3(1), dim3(kQBlock), 0, stream, w.hist, w.key_off,
                           w.cls_begin, w.cls_count);
        hipLaunchKernelGGL(scatter, dim3(blocks), dim3(kSortThreads), 0, stream, s, pa, pb, n, w.key_off,
                           w.key_cur, w.order);
    };
    // the whole sort with 1 / 2 / 4 / 8 pairs per thread: 16,384 mixed pairs 19 / 21
    // / 25 / 33 us, 131,072 pairs 28 / 25 / 26 / 33, 262,144 pairs 40 / 31 / 29 / 34,
    // 1,048,576 pairs 98 / 65 / 53 / 47 (129 us with 256-pair tiles)
    if (n < 65536) sort(queue_hist_kernel<1>, queue_scatter_kernel<1>, 1);
    else if (n < 196608) sort(queue_hist_kernel<2>, queue_scatter_kernel<2>, 2);
    else if (n < 786432) sort(queue_hist_kernel<4>, queue_scatter_kernel<4>, 4);
    else sort(queue_hist_kernel<8>, queue_scatter_kernel<8>, 8);
    D3D_CHECK_LAUNCH("queue sort");
    return D3D_OK;
}

d3d_gjk_params queue_params(const d3d_gjk_params &prm, int64_t n, int64_t loose_max) {
    d3d_gjk_params rp = prm;
    for (int c = 0; c < kNumClasses; ++c) {
        int G = prm.lanes_per_pair[c] > 0 ? prm.lanes_per_pair[c] : -kDefaultLanes[c];
        if (c == 0 && G > 4) G = 4;
        rp.lanes_per_pair[c] = G;
    }
    rp.blocks_per_cu = batch_blocks(n, loose_max, prm.blocks_per_cu);
    rp.claim_factor = prm.claim_factor > 0 ? prm.claim_factor : 2;
    rp.epa_blocks_per_cu = prm.epa_blocks_per_cu > 0 ? prm.epa_blocks_per_cu : 8;
    return rp;
}

unsigned queue_grid(const d3d_gjk_params &resolved) {
    return (unsigned)(cu_count() * resolved.blocks_per_cu);
}

static int launch_all(const d3d_scene &s, const int32_t *pa, const int32_t *pb, int64_t n,
                      const d3d_gjk_params &prm, const GjkOut &o, void *ws, hipStream_t stream,
                      const EpaHook *epa) {
    const QueueWs w = ws_view(ws, n);
    std::array<hipEvent_t, 4> ev;
    const bool timed = stage_events(ev);
    if (timed) D3D_CHECK_HIP(hipEventRecord(ev[0], stream));
    if (int rc = queue_sort(s, pa, pb, n, w, stream, epa ? epa->count : nullptr)) return rc;
    const d3d_gjk_params rp = queue_params(prm, n, kLooseMax);
    if (timed) D3D_CHECK_HIP(hipEventRecord(ev[1], stream));
    const bool loose = batch_is_loose(n, kLooseMax, prm.blocks_per_cu);
    hipLaunchKernelGGL(loose ? gjk_small_kernel : gjk_all_kernel, dim3(queue_grid(rp)), dim3(kQBlock), 0,
                       stream, s, pa, pb, w.order, w.cls_begin, w.cls_count, w.cls_cursor, rp, o);
    D3D_CHECK_LAUNCH("gjk_all_kernel");
    if (timed) D3D_CHECK_HIP(hipEventRecord(ev[2], stream));
    if (epa) {
        if (int rc = launch_epa(s, pa, pb, n, (const int64_t *)epa->count, epa->work, nullptr,
                                o.simplex, o.npts, epa->max_iter, epa->max_faces, epa->eps,
                                epa->out, epa->status, nullptr, epa->count + 1, stream, nullptr,
                                nullptr, rp.epa_blocks_per_cu))
            return rc;
    }
    if (timed) D3D_CHECK_HIP(hipEventRecord(ev[3], stream));
    return D3D_OK;
}

// ------------------------------------------------- GJK -> EPA pipeline

// Per-pair collider instances: record 2i is scene record a[i] posed by
// pose_a[i] (R row-major, t: 12 doubles), record 2i+1 is b[i] posed by
// pose_b[i]; NULL poses keep the scene's.  Vertex offsets are copied, so the
// instances share the scene's resident vertex pools.
__global__ __launch_bounds__(kQBlock) void instance_kernel(
    d3d_scene s, const int32_t *a, const int32_t *b, const double *__restrict__ pose_a,
    const double *__restrict__ pose_b, const int32_t *pidx_a, const int32_t *pidx_b, int64_t n_poses,
    int64_t n, double *__restrict__ f64, int32_t *__restrict__ i32, int32_t *inst_a, int32_t *inst_b) {
    const int64_t t = (int64_t)blockIdx.x * kQBlock + threadIdx.x;
    if (t >= 2 * n) return;
    const int64_t pair = t >> 1;
    const int side = (int)(t & 1);
    const int k = side ? b[pair] : a[pair];
    const double *pose = side ? pose_b : pose_a;
    const int32_t *pidx = side ? pidx_b : pidx_a;
    int64_t prow = pair;
    if (pidx) prow = pidx[pair];
    // after the reads: the lists written may be the ones read
    if (inst_a && inst_b) (side ? inst_b : inst_a)[pair] = (int32_t)t;
    double *dst = f64 + 16 * t;
    int32_t *di = i32 + 4 * t;
    if (k < 0 || (int64_t)k >= s.n_shapes || (pose && pidx && (prow < 0 || prow >= n_poses))) {
        for (int j = 0; j < 16; ++j) dst[j] = 0.0;
        di[0] = -1;  // rejected as bad input downstream
        di[1] = di[2] = 0;
        di[3] = -1;
        return;
    }
    const double *src = s.shape_f64 + 16 * (int64_t)k;
#pragma unroll
    for (int j = 0; j < 16; ++j) dst[j] = src[j];
    if (pose) {
#pragma unroll
        for (int j = 0; j < 12; ++j) dst[j] = pose[12 * prow + j];
    }
    const int32_t *si = s.shape_i32 + 4 * (int64_t)k;
#pragma unroll
    for (int j = 0; j < 4; ++j) di[j] = si[j];
}

}  // namespace d3d

using namespace d3d;

extern "C" int d3d_stage_timing(int enable) {
    clear_error();
    std::lock_guard<std::mutex> lk(g_timing.mu);
    g_timing.on = enable != 0;
    // events of calls not yet read are dropped unread (they may still be in
    // flight: destroyed only once they have completed)
    for (auto &ev : g_timing.rec) {
        (void)hipEventSynchronize(ev[3]);
        g_timing.pool.push_back(ev);
    }
    g_timing.rec.clear();
    return D3D_OK;
}

extern "C" int d3d_stage_timing_read(double *ms_out, int64_t *calls_out) {
    clear_error();
    D3D_CHECK_ARG(ms_out && calls_out, "NULL buffer");
    std::lock_guard<std::mutex> lk(g_timing.mu);
    double sum[3] = {0.0, 0.0, 0.0};
    int64_t calls = 0;
    for (auto &ev : g_timing.rec) {
        D3D_CHECK_HIP(hipEventSynchronize(ev[3]));
        for (int k = 0; k < 3; ++k) {
            float ms = 0.0f;
            D3D_CHECK_HIP(hipEventElapsedTime(&ms, ev[k], ev[k + 1]));
            sum[k] += ms;
        }
        ++calls;
        g_timing.pool.push_back(ev);
    }
    g_timing.rec.clear();
    for (int k = 0; k < 3; ++k) ms_out[k] = sum[k];
    *calls_out = calls;
    return D3D_OK;
}

extern "C" int64_t d3d_gjk_workspace_bytes(int64_t n) {
    if (n < 0) return -1;
    return (ws_header_ints() + n) * (int64_t)sizeof(int32_t);
}

static int gjk_distance_impl(const d3d_scene *scene, const int32_t *pair_a, const int32_t *pair_b,
                             int64_t n, const d3d_gjk_params *params, double *dist, double *cp_a,
                             double *cp_b, int32_t *status, int32_t *iterations, double *simplex,
                             int32_t *n_points, void *workspace, int64_t workspace_bytes,
                             const EpaHook *epa,
                             void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(n < (int64_t)0x7fffffff, "n must fit in int32");
    D3D_CHECK_ARG(pair_a && pair_b && dist && cp_a && cp_b && status, "NULL buffer");
    d3d_gjk_params prm;
    if (params) {
        prm = *params;
    } else {
        prm = default_params();
    }
    D3D_CHECK_ARG(prm.max_iterations > 0, "max_iterations must be > 0");
    D3D_CHECK_ARG(prm.blocks_per_cu >= 0 && prm.blocks_per_cu <= 3, "blocks_per_cu must be in [0, 3]");
    D3D_CHECK_ARG(prm.claim_factor >= 0 && prm.claim_factor <= 8, "claim_factor must be in [0, 8]");
    D3D_CHECK_ARG(prm.epa_blocks_per_cu >= 0 && prm.epa_blocks_per_cu <= 16,
                  "epa_blocks_per_cu must be in [0, 16]");
    for (int c = 0; c < kNumClasses; ++c) {
        const int G = prm.lanes_per_pair[c];
        D3D_CHECK_ARG(G == 0 || (G <= 64 && (G & (G - 1)) == 0),
                      "lanes_per_pair entries must be 0 or a power of two <= 64");
    }
    void *ws = workspace;
    if (ws) {
        D3D_CHECK_ARG(workspace_bytes >= d3d_gjk_workspace_bytes(n), "workspace too small");
    } else {
        if (int rc = workspace_for(stream, n, &ws)) return rc;
    }
    GjkOut o{dist,
             cp_a,
             cp_b,
             status,
             iterations,
             simplex,
             n_points,
             epa != nullptr,
             epa ? epa->work : nullptr,
             epa ? epa->count : nullptr,
             epa ? epa->out : nullptr,
             epa ? epa->status : nullptr};
    return launch_all(*scene, pair_a, pair_b, n, prm, o, ws, (hipStream_t)stream, epa);
}

extern "C" int d3d_gjk_distance_batch(const d3d_scene *scene, const int32_t *pair_a,
                                      const int32_t *pair_b, int64_t n,
                                      const d3d_gjk_params *params, double *dist, double *cp_a,
                                      double *cp_b, int32_t *status, int32_t *iterations,
                                      double *simplex, int32_t *n_points, void *stream) {
    return gjk_distance_impl(scene, pair_a, pair_b, n, params, dist, cp_a, cp_b, status, iterations,
                             simplex, n_points, nullptr, 0, nullptr, stream);
}

extern "C" int d3d_gjk_distance_batch_ws(const d3d_scene *scene, const int32_t *pair_a,
                                         const int32_t *pair_b, int64_t n,
                                         const d3d_gjk_params *params, double *dist, double *cp_a,
                                         double *cp_b, int32_t *status, int32_t *iterations,
                                         double *simplex, int32_t *n_points, void *workspace,
                                         int64_t workspace_bytes, void *stream) {
    clear_error();
    D3D_CHECK_ARG(workspace != nullptr, "workspace is NULL");
    return gjk_distance_impl(scene, pair_a, pair_b, n, params, dist, cp_a, cp_b, status, iterations,
                             simplex, n_points, workspace, workspace_bytes, nullptr, stream);
}

// Pairs below which the sort costs more than it saves: with hulls in the scene 1
// mixed pair takes 9 us in the lane-per-pair kernel and 14 us here; 16 pairs take
// 15 to 33 there, as their largest hull is, and 17 to 20 here, 24 pairs 29 and 20,
// 64 pairs 90 and 25, 262,144 pairs 747 and 409 us.  A scene without hulls has nothing to sort for (262,144 pairs of
// boxes 49 and 75 us).
constexpr int64_t kIntersectQueueMin = D3D_INTERSECTION_QUEUE_MIN;

extern "C" int d3d_gjk_intersection_batch_ws(const d3d_scene *scene, const int32_t *pair_a,
                                             const int32_t *pair_b, int64_t n, double tolerance,
                                             int32_t max_iterations, uint8_t *hit, int32_t *status,
                                             void *workspace, int64_t workspace_bytes,
                                             void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(pair_a && pair_b && hit, "NULL buffer");
    D3D_CHECK_ARG(max_iterations > 0, "max_iterations must be > 0");
    // (the queue holds pair indices as int32)
    if (n < kIntersectQueueMin || n >= (int64_t)0x7fffffff || scene->n_vertices == 0)
        return d3d_gjk_intersection_batch(scene, pair_a, pair_b, n, tolerance, max_iterations, hit,
                                          status, stream);
    D3D_CHECK_ARG(workspace, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= d3d_gjk_workspace_bytes(n), "workspace too small");
    d3d_gjk_params prm = default_params();
    prm.tolerance = tolerance;
    prm.max_iterations = max_iterations;
    const bool loose = batch_is_loose(n, kIntersectLooseMax, 0);
    const d3d_gjk_params rp = queue_params(prm, n, kIntersectLooseMax);
    const QueueWs w = ws_view(workspace, n);
    if (int rc = queue_sort(*scene, pair_a, pair_b, n, w, (hipStream_t)stream, nullptr)) return rc;
    hipLaunchKernelGGL(loose ? gjk_intersect_small_kernel : gjk_intersect_all_kernel,
                       dim3(queue_grid(rp)), dim3(kQBlock), 0, (hipStream_t)stream, *scene, pair_a, pair_b, w.order, w.cls_begin, w.cls_count,
                       w.cls_cursor, rp, HitOut{hit, status});
    D3D_CHECK_LAUNCH("gjk_intersect_all_kernel");
    return D3D_OK;
}

// Workspace of the fused pipeline: GJK queue | simplex (n*36 f64) |
// n_points (n) | EPA work list (n) | count (u64)
static constexpr int64_t a256(int64_t b) { return (b + 255) / 256 * 256; }
static constexpr int64_t gjk_ws_bytes(int64_t n) {
    return (ws_header_ints() + n) * (int64_t)sizeof(int32_t);
}
static constexpr int64_t gjk_epa_ws_bytes(int64_t n) {
    return a256(gjk_ws_bytes(n)) + a256(n * 36 * 8) + a256(n * 4) + a256(n * 4) + 256;
}

extern "C" int64_t d3d_gjk_epa_workspace_bytes(int64_t n) {
    if (n < 0) return -1;
    return gjk_epa_ws_bytes(n);
}

extern "C" int d3d_gjk_epa_batch_ws(const d3d_scene *scene, const int32_t *pair_a,
                                    const int32_t *pair_b, int64_t n, const d3d_gjk_params *params,
                                    int32_t epa_max_iterations, int32_t epa_max_faces,
                                    double epa_epsilon, double *dist, double *cp_a, double *cp_b,
                                    int32_t *status, int32_t *iterations, double *epa_out,
                                    int32_t *epa_status, void *workspace, int64_t workspace_bytes,
                                    void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(workspace && epa_out && epa_status, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= d3d_gjk_epa_workspace_bytes(n), "workspace too small");
    D3D_CHECK_ARG(epa_max_iterations >= 1, "epa_max_iterations must be >= 1");
    D3D_CHECK_ARG(epa_max_faces >= 4 && epa_max_faces <= 128, "epa_max_faces must be in [4, 128]");
    char *w = (char *)workspace;
    const int64_t gq = a256(d3d_gjk_workspace_bytes(n));
    double *simplex = (double *)(w + gq);
    int32_t *npts = (int32_t *)(w + gq + a256(n * 36 * 8));
    int32_t *work = (int32_t *)(w + gq + a256(n * 36 * 8) + a256(n * 4));
    unsigned long long *count =
        (unsigned long long *)(w + gq + a256(n * 36 * 8) + a256(n * 4) + a256(n * 4));
    const EpaHook hook{work, count, (int)epa_max_iterations, (int)epa_max_faces, epa_epsilon,
                       epa_out, epa_status};
    return gjk_distance_impl(scene, pair_a, pair_b, n, params, dist, cp_a, cp_b, status, iterations,
                             simplex, npts, workspace, gq, &hook, stream);
}

extern "C" int d3d_instance_pairs(const d3d_scene *scene, const int32_t *pair_a,
                                  const int32_t *pair_b, const double *pose_a,
                                  const double *pose_b, const int32_t *pose_idx_a,
                                  const int32_t *pose_idx_b, int64_t n_poses, int64_t n,
                                  double *inst_f64, int32_t *inst_i32, int32_t *inst_a,
                                  int32_t *inst_b, void *stream) {
    clear_error();
    if (int rc = check_scene(scene)) return rc;
    D3D_CHECK_ARG(n >= 0 && n < (int64_t)0x3fffffff, "n must be in [0, 2^30)");
    if (n == 0) return D3D_OK;
    D3D_CHECK_ARG(pair_a && pair_b && inst_f64 && inst_i32, "NULL buffer");
    hipStream_t st = (hipStream_t)stream;
    D3D_CHECK_ARG(!(pose_idx_a || pose_idx_b) || n_poses > 0, "pose indices need n_poses > 0");
    hipLaunchKernelGGL(instance_kernel, dim3(grid_for(2 * n, kQBlock)), dim3(kQBlock), 0, st, *scene,
                       pair_a, pair_b, pose_a, pose_b, pose_idx_a, pose_idx_b, n_poses, n, inst_f64,
                       inst_i32, inst_a, inst_b);
    D3D_CHECK_LAUNCH("instance_kernel");
    return D3D_OK;
}

// ------------------------------------ fused pipeline without allocation

// The fused pipeline's workspace for at most D3D_NOALLOC_MAX_PAIRS pairs, as
// a device array of the library: each GPU holds its own copy from module load
// until the process ends, and every call of d3d_gjk_epa_batch_noalloc on that
// GPU works in it (the queue header and the EPA counters are cleared by fill
// kernels at the start of each call; the other regions are written before
// they are read).  In host code `scratch` names a host-side stand-in: kernels
// get the device address that hipGetSymbolAddress returns for the current
// device, kept per device in g_scratch.
static constexpr int64_t kNoallocBytes = gjk_epa_ws_bytes(D3D_NOALLOC_MAX_PAIRS);
static __device__ __align__(256) unsigned char scratch[kNoallocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch[kMaxDevices];
}  // namespace

namespace d3d {

// Looks up the device address of `scratch` on the current device once (the
// device must be current); d3d_init calls it, and so does the first
// d3d_gjk_epa_batch_noalloc call on a device d3d_init was not called for.
int noalloc_scratch(void **out) {
    int dev = 0;
    D3D_CHECK_HIP(hipGetDevice(&dev));
    D3D_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device index beyond the 64 the library tracks");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        D3D_CHECK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        D3D_CHECK_ARG(p != nullptr, "hipGetSymbolAddress returned NULL for the scratch array");
        g_scratch[dev] = p;
    }
    if (out) *out = g_scratch[dev];
    return D3D_OK;
}

}  // namespace d3d

extern "C" int d3d_gjk_epa_batch_noalloc(const d3d_scene *scene, const int32_t *pair_a,
                                         const int32_t *pair_b, int64_t n,
                                         const d3d_gjk_params *params, int32_t epa_max_iterations,
                                         int32_t epa_max_faces, double epa_epsilon, double *dist,
                                         double *cp_a, double *cp_b, int32_t *status,
                                         int32_t *iterations, double *epa_out,
                                         int32_t *epa_status, void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 0, "n must be >= 0");
    D3D_CHECK_ARG(n <= D3D_NOALLOC_MAX_PAIRS,
                  "n exceeds D3D_NOALLOC_MAX_PAIRS (16384 pairs per call of "
                  "d3d_gjk_epa_batch_noalloc); split the batch or use d3d_gjk_epa_batch_ws");
    if (n == 0) return D3D_OK;
    void *ws = nullptr;
    if (int rc = noalloc_scratch(&ws)) return rc;
    return d3d_gjk_epa_batch_ws(scene, pair_a, pair_b, n, params, epa_max_iterations,
                                epa_max_faces, epa_epsilon, dist, cp_a, cp_b, status, iterations,
                                epa_out, epa_status, ws, kNoallocBytes, stream);
}
