// d3d_queue.hpp -- the sorted pair queue: work classes, the persistent walk over
// them, and the group supports.  An algorithm over pairs whose rounds each end
// in one pair of support points (GJK distance, GJK intersection, MPR) is a Mode
// run by it:
//   State           the pair's registers; State::d is the support direction
//   start(...)      a new pair (its collider indices are validated); false when
//                   it needs no round
//   more(...)       false ends the pair before the next support (round cap)
//   step<G>(...)    one round with the supports on A along d and on B along -d;
//                   false once the pair has terminated
//   write / bad     the pair's outputs, by one lane; those of an invalid pair
// A pair's rows of support points live in LDS (PQ): the group's first lane
// writes them and all its lanes read them, so a step puts a row_fence between
// the last write (its own or an earlier step's) and its reads.
#pragma once

#include "d3d_device.hpp"
#include "d3d_runtime.hpp"

namespace d3d {

constexpr int kQBlock = 256;
constexpr int kSizeClasses = 8;
constexpr int kNumClasses = D3D_NUM_CLASSES;  // size class, + 8 when both are hulls
static_assert(kNumClasses == 2 * kSizeClasses, "work classes: size x one or two hulls");
constexpr int kNumTypes = 9;
constexpr int kNumKeys = kNumClasses * kNumTypes * kNumTypes;
constexpr int kBadInput = 0x200;

// size class from the total hull vertex count of a pair
__device__ __forceinline__ int work_class(int nverts) {
    if (nverts == 0) return 0;
    if (nverts <= 32) return 1;
    if (nverts <= 128) return 2;
    if (nverts <= 512) return 3;
    if (nverts <= 1024) return 4;
    if (nverts <= 2048) return 5;
    if (nverts <= 4096) return 6;
    return 7;
}

__device__ __forceinline__ int pair_key(const d3d_scene &s, int a, int b) {
    if (a < 0 || b < 0 || (int64_t)a >= s.n_shapes || (int64_t)b >= s.n_shapes) return 0;
    const int4 A = *reinterpret_cast<const int4 *>(s.shape_i32 + 4 * (int64_t)a);
    const int4 B = *reinterpret_cast<const int4 *>(s.shape_i32 + 4 * (int64_t)b);
    const int ta = (A.x >= 0 && A.x < kNumTypes) ? A.x : 0;
    const int tb = (B.x >= 0 && B.x < kNumTypes) ? B.x : 0;
    const int na = (ta == D3D_HULL) ? (A.y > 0 ? A.y : 0) : 0;
    const int nb = (tb == D3D_HULL) ? (B.y > 0 ? B.y : 0) : 0;
    const int cls = work_class(na + nb) + (na > 0 && nb > 0 ? kSizeClasses : 0);
    return (cls * kNumTypes + ta) * kNumTypes + tb;
}

// Workspace layout (int32): hist[K] key_off[K] key_cur[K] cls_begin[C]
// cls_count[C] cls_cursor[C] pad order[n]
struct QueueWs {
    int32_t *hist, *key_off, *key_cur, *cls_begin, *cls_count, *cls_cursor, *order;
};

__host__ __device__ constexpr int64_t ws_header_ints() {
    return ((3 * kNumKeys + 3 * kNumClasses) + 63) / 64 * 64;
}

inline QueueWs ws_view(void *base, int64_t n) {
    (void)n;
    int32_t *p = (int32_t *)base;
    QueueWs w;
    w.hist = p;
    w.key_off = p + kNumKeys;
    w.key_cur = p + 2 * kNumKeys;
    w.cls_begin = p + 3 * kNumKeys;
    w.cls_count = w.cls_begin + kNumClasses;
    w.cls_cursor = w.cls_count + kNumClasses;
    w.order = p + ws_header_ints();
    return w;
}

// Support points on A (P) and B (Q) of the simplex rows, in LDS: they are
// touched only on append, compaction and at the end, so keeping them out of
// VGPRs leaves the registers to the simplex solve.  Structure of arrays over
// the block's threads: component c (slot * 6 + {Px,Py,Pz,Qx,Qy,Qz}) of thread
// t at base[c * kQBlock + t], conflict-free.
// P, Q rows of the simplex in LDS, structure of arrays with stride `st`
// doubles: one slot per pair, shared by the G lanes of a group (all lanes
// read it; the group's first lane, `wr`, writes it; LDS operations of a
// wavefront complete in order, so the other lanes see the writes).
struct PQ {
    double *base;
    int st;
    bool wr;
    __device__ __forceinline__ void put(int slot, v3 p, v3 q) const {
        if (!wr) return;
        double *b = base + slot * 6 * st;
        b[0] = p.x;
        b[st] = p.y;
        b[2 * st] = p.z;
        b[3 * st] = q.x;
        b[4 * st] = q.y;
        b[5 * st] = q.z;
    }
    // the P half of a row alone
    __device__ __forceinline__ void put_p(int slot, v3 p) const {
        if (!wr) return;
        double *b = base + slot * 6 * st;
        b[0] = p.x;
        b[st] = p.y;
        b[2 * st] = p.z;
    }
    __device__ __forceinline__ v3 P(int slot) const {
        const double *b = base + slot * 6 * st;
        return mk(b[0], b[st], b[2 * st]);
    }
    __device__ __forceinline__ v3 Q(int slot) const {
        const double *b = base + slot * 6 * st;
        return mk(b[3 * st], b[4 * st], b[5 * st]);
    }
    __device__ __forceinline__ void zero() const {
        if (!wr) return;
#pragma unroll
        for (int c = 0; c < 24; ++c) base[c * st] = 0.0;
    }
    // kParts: 6 for P and Q, 3 for the P half alone
    template <int kParts = 6>
    __device__ __forceinline__ void move(int from, int to) const {
        if (from == to || !wr) return;
        const double *a = base + from * 6 * st;
        double *b = base + to * 6 * st;
#pragma unroll
        for (int c = 0; c < kParts; ++c) b[c * st] = a[c * st];
    }
    // applies a compaction map (sources are >= destinations, so moving
    // rows in increasing order reads every row before it is overwritten)
    template <int kParts = 6>
    __device__ __forceinline__ void compact(const CompactMap &c) const {
        if (!c.moved) return;
        move<kParts>(c.k0, 0);
        if (c.m > 1) move<kParts>(c.k1, 1);
        if (c.m > 2) move<kParts>(c.k2, 2);
    }
};

// Orders a group's LDS writes (rows, slots) before its lanes' reads for the compiler, which
// may otherwise keep the old value on the lanes that did not write; the
// hardware runs a wavefront's LDS operations in order.
__device__ __forceinline__ void row_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ------------------------------------------------------- group supports

__device__ __forceinline__ unsigned long long lanemask_lt(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (kWave - lane));
}

// ---------------------------------------------- LDS-resident hull vertices
//
// A wavefront's 12 KB LDS region holds the P/Q rows of its 64/G pair slots
// (24 doubles each, interleaved) and, for hull classes with G >= 4, one vertex
// cache per slot in the rest: the FP32 vertices of the pair's hulls in their
// original order (A's at 0, B's after them; x, y and z arrays of
// cache_verts<G>() entries), loaded once when the group takes the pair.  Every
// support sweep of the pair then reads LDS instead of the pools.  Slot
// strides are congruent to G modulo 64 words, so the 64/G groups sweeping at
// the same time hit distinct banks.  Pairs whose hulls do not fit, or whose
// vertices are not exact in FP32, sweep the pools as before.
template <int G>
__host__ __device__ constexpr int cache_stride_words() {
    // (12288 bytes - P/Q rows) / slots, rounded down to G modulo 64 words
    constexpr int room = (3072 - 48 * (kWave / G)) / (kWave / G);
    return G >= kWave ? room : ((room - G) / 64) * 64 + G;
}
// With 8 to 32 lanes per pair the last kRecWords words of a slot hold the
// pair's two collider records (the FP64 blocks of A and B, then their int32
// parts), staged once when the group takes the pair, so the supports read
// them from LDS instead of reloading them from memory at every iteration
// (a wavefront-wide group loads them into scalar registers instead).
constexpr int kRecWords = 2 * 16 * 2 + 2 * 4;
template <int G>
__host__ __device__ constexpr bool slot_recs() {
    return G >= 8 && G < kWave;
}
// words of a slot for vertices or cluster records
template <int G>
__host__ __device__ constexpr int cache_words() {
    return cache_stride_words<G>() - (slot_recs<G>() ? kRecWords : 0);
}
template <int G>
__host__ __device__ constexpr int cache_verts() {
    return cache_words<G>() / 3;
}
static_assert(cache_verts<4>() >= 32, "class 1 pairs fit a 4-lane slot");
static_assert(cache_verts<64>() >= 1000, "one slot per wavefront holds 1000 vertices");
static_assert(cache_words<8>() % 2 == 0 && cache_stride_words<8>() % 2 == 0 &&
                  cache_words<16>() % 2 == 0 && cache_stride_words<16>() % 2 == 0,
              "slot records are 8-byte aligned");

// Collider record k (0: A, 1: B) of the pair in a slot (see slot_recs).
__device__ __forceinline__ Shape slot_shape(const float *recs, int k) {
    const double *f = reinterpret_cast<const double *>(recs) + 16 * k;
    const int32_t *i = reinterpret_cast<const int32_t *>(recs + 64) + 4 * k;
    Shape h;
#pragma unroll
    for (int j = 0; j < 9; ++j) h.R[j] = f[j];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        h.t[j] = f[9 + j];
        h.p[j] = f[12 + j];
    }
    h.margin = f[15];
    h.type = i[0];
    h.nv = i[1];
    h.voff = i[2];
    h.voff64 = i[3];
    return h;
}

// The collider record k of a pair: from the slot when it holds them, else
// from the scene by index (kUniform: the same record for the whole
// wavefront, so a wavefront-wide group loads it into scalar registers).
template <int G, bool kUniform>
__device__ __forceinline__ Shape pair_shape(const d3d_scene &s, const float *recs, int k, int idx) {
    if constexpr (slot_recs<G>()) {
        (void)s;
        (void)idx;
        return slot_shape(recs, k);
    } else {
        (void)recs;
        (void)k;
        return load_shape(s, (kUniform && G == kWave) ? wave_uniform(idx) : opaque(idx));
    }
}

// Copies the FP32 vertices of hull record h (validated) into the cache at
// `at`, in original order (vorig), by the G lanes of a group.
template <int G>
__device__ __forceinline__ void cache_fill(const d3d_scene &s, const Shape &h, float *cache,
                                           int at, int sub) {
    constexpr int C = cache_verts<G>();
    fill_orig<G>(s, h.voff, h.nv, cache, cache + C, cache + 2 * C, at, sub);
}

// Supports of records ia along d and ib along -d (see support_pair) for a
// pair whose hull vertices are in the group's cache (A's first, nA of them).
// Two hulls: the lower half of the group sweeps A while the upper half sweeps
// B; one hull: the whole group sweeps it.  Same results as support_pair.
template <int G>
__device__ __forceinline__ SupportPair support_pair_cached(const d3d_scene &s, int ia, int ib, v3 d,
                                                           int sub, const float *cache, int nA,
                                                           bool two) {
    constexpr int C = cache_verts<G>();
    const float *cx = cache, *cy = cache + C, *cz = cache + 2 * C;
    const float *recs = cache + cache_words<G>();
    if (two) {
        constexpr int H = G / 2;
        const bool upper = sub >= H;
        const Shape h = pair_shape<G, false>(s, recs, upper ? 1 : 0, upper ? ib : ia);
        const v3 dir = vsel(upper, -d, d);
        const int off = upper ? nA : 0;
        const int j = lds_orig_argmax<H>(cx, cy, cz, off, h.nv, h.p[0], to_local(h, dir), sub & (H - 1));
        const v3 v = mk((double)cx[off + j], (double)cy[off + j], (double)cz[off + j]);
        const v3 out = apply_margin(h, to_world(h, v), dir);
        SupportPair r;
        halves<H>(out.x, r.a.x, r.b.x);
        halves<H>(out.y, r.a.y, r.b.y);
        halves<H>(out.z, r.a.z, r.b.z);
        return r;
    }
    v3 a = mk(0.0, 0.0, 0.0), b = a;
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
        const Shape h = pair_shape<G, false>(s, recs, k, k == 0 ? ia : ib);
        const v3 dir = vsel(k == 0, d, -d);
        v3 out;
        if (h.type == D3D_HULL) {
            const int j = lds_orig_argmax<G>(cx, cy, cz, 0, h.nv, h.p[0], to_local(h, dir), sub);
            out = to_world(h, mk((double)cx[j], (double)cy[j], (double)cz[j]));
        } else {
            out = support_analytic(h, dir);
        }
        out = apply_margin(h, out, dir);
        a = vsel(k == 0, out, a);
        b = vsel(k == 0, b, out);
    }
    return SupportPair{a, b};
}

// Copies the cluster records of hull record h (validated, clustered) into
// the slot at record `at`, by the G lanes of a group.
template <int G>
__device__ __forceinline__ void bounds_fill(const d3d_scene &s, const Shape &h, float4 *slot, int at,
                                            int sub) {
    const float4 *__restrict__ cl = reinterpret_cast<const float4 *>(s.clusters) + (int64_t)h.p[1];
    const int nc = (int)h.p[2];
#pragma unroll 4
    for (int k = sub; k < nc; k += G) slot[at + k] = cl[k];
}

// Supports of records ia along d and ib along -d (see support_pair) for a pair
// whose clustered hulls have their cluster records in the group's slot (A's
// first, ncA of them): the sweeps read the bounds from LDS and the vertices
// from the pools.  Same results as support_pair.
template <int G>
__device__ __forceinline__ SupportPair support_pair_bounds(const d3d_scene &s, int ia, int ib, v3 d,
                                                           int sub, const float4 *slot, int ncA,
                                                           int nrec) {
    v3 a = mk(0.0, 0.0, 0.0), b = a;
    if (G == kWave) d = mk(wave_uniform(d.x), wave_uniform(d.y), wave_uniform(d.z));
    const float *recs = reinterpret_cast<const float *>(slot) + cache_words<G>();
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
        const Shape h = pair_shape<G, true>(s, recs, k, k == 0 ? ia : ib);
        const v3 dir = vsel(k == 0, d, -d);
        v3 out;
        if (h.type == D3D_HULL) {
            const v3 l = to_local(h, dir);
            const HullRef H = hull_ref(h);
            // the slot's words past the cluster records hold the survivor list
            int *list = const_cast<int *>(reinterpret_cast<const int *>(slot + nrec));
            const int hi = H.nc > 0 ? hull_argmax<G, true>(s, H, l, sub, slot + (k == 0 ? 0 : ncA),
                                                           list, cache_words<G>() - 4 * nrec)
                                    : hull_argmax<G>(s, H, l, sub);
            out = to_world(h, hull_vertex(s, h.voff, h.voff64, hi));
        } else {
            out = support_analytic(h, dir);
        }
        out = apply_margin(h, out, dir);
        a = vsel(k == 0, out, a);
        b = vsel(k == 0, b, out);
    }
    return SupportPair{a, b};
}

// Items of a class of `count` pairs that a wavefront claims at a time: `full`, or
// the class's fair share per wavefront when that is smaller; and the chunks the
// class has.  A class may have up to 2^31 - 2 pairs: the sums are unsigned.
__host__ __device__ constexpr uint32_t chunks_of(int count, int chunk) {
    return ((uint32_t)count + (uint32_t)chunk - 1u) / (uint32_t)chunk;
}
__host__ __device__ constexpr int claim_chunk(int count, int n_waves, int full) {
    const uint32_t fair = chunks_of(count, n_waves);
    return fair < (uint32_t)full ? (int)fair : full;
}

// One work class, G lanes per pair, by one wavefront: groups of G lanes take
// pairs of the class (chunked claims from the class cursor) until the class is
// exhausted and every group of the wavefront has finished its pair.  The
// wavefront's P/Q slots are `pq_wave` (24 x 64 doubles, slot stride 64 / G);
// with kCache (hull classes, G >= 4) the rest of the region holds each slot's
// vertex cache.
template <class M, int G, bool kHull, bool kCache = (kHull && G >= 4)>
__device__ __forceinline__ void run_class(const d3d_scene &s, const int32_t *__restrict__ pa,
                                          const int32_t *__restrict__ pb,
                                          const int32_t *__restrict__ order, int begin, int count,
                                          int32_t *__restrict__ cursor, const d3d_gjk_params &prm,
                                          const typename M::Out &o, double *pq_wave, int chunk,
                                          int rot) {
    const int lane = lane_id();
    const int sub = lane & (G - 1);
    const int leader = lane - sub;
    const PQ pq{pq_wave + lane / G, kWave / G, sub == 0};
    float *const cache = reinterpret_cast<float *>(pq_wave + 24 * (kWave / G)) +
                         (lane / G) * cache_stride_words<G>();
    typename M::State g;
    M::clear(g, pq);
    int ia = 0, ib = 0;
    int pid = 0;
    // pairs with their hull vertices in the group's cache: hull vertices of
    // A (the offset of B's), both records hulls
    bool cached = false, two = false;
    int nA = 0;
    // otherwise, pairs with their hulls' cluster records in the slot (ncA: A's
    // record count, the offset of B's)
    bool bounded = false;
    int ncA = 0, nrec = 0;
    // analytic classes: the two record types, read once per pair
    int ta = 0, tb = 0;
    bool have = false, exhausted = false;
    // The first chunk of every wavefront is fixed by its rank (wavefront index
    // minus `rot`, modulo the wavefront count): no atomic, so thousands of
    // wavefronts do not queue on one cursor when a launch starts, and the
    // rotation hands each class's fixed chunks to the wavefronts the earlier
    // classes left without one.  Later chunks come from the cursor, past all
    // fixed chunks; when the fixed chunks cover the class there are none.
    const int n_waves = (int)gridDim.x * (kQBlock / kWave);
    const int wv = (int)blockIdx.x * (kQBlock / kWave) + (int)threadIdx.x / kWave;
    const int64_t r = (wv - rot + n_waves) % n_waves;
    const int64_t fixed_end = (int64_t)n_waves * chunk;
    const bool dynamic = fixed_end < count;
    // the wavefront's unclaimed items are [cb, ce) of the class; past its end every
    // wavefront claims one more chunk, which goes beyond 2^31 in a class close to it
    uint32_t cb = (uint32_t)min(r * chunk, (int64_t)count), ce = cb + (uint32_t)chunk;
    while (true) {
        const bool need = !have && !exhausted;
        const unsigned long long m = __ballot(need && sub == 0);
        if (m != 0ull) {
            // groups take items from the wavefront's chunk of the class range;
            // one atomic fetches the next chunk when it runs out.  Groups
            // ranked past the items at hand wait for the next round.
            const int c = __popcll(m);
            const int rank = __popcll(m & lanemask_lt(leader));
            const int avail = (int)(ce - cb);
            uint32_t nb = 0;
            if (avail < c) {
                const int first = __ffsll((long long)m) - 1;
                if (dynamic) {
                    if (lane == first) nb = (uint32_t)fixed_end + (uint32_t)atomicAdd(cursor, chunk);
                    nb = (uint32_t)readlane_i32((int)nb, first);
                } else {
                    nb = (uint32_t)count;  // nothing past the fixed chunks
                }
            }
            const uint32_t base = rank < avail ? cb : nb - (uint32_t)avail;
            const bool served = rank < avail + (avail < c ? chunk : 0);
            if (avail < c) {
                const int taken = c - avail < chunk ? c - avail : chunk;
                cb = nb + (uint32_t)taken;
                ce = nb + (uint32_t)chunk;
            } else {
                cb += (uint32_t)c;
            }
            if (need && served) {
                const uint32_t idx = base + (uint32_t)rank;
                if (idx < (uint32_t)count) {
                    pid = order[begin + (int)idx];
                    ia = pa[pid];
                    ib = pb[pid];
                    Shape A, B;
                    const bool okA = load_checked(s, ia, A);
                    const bool okB = load_checked(s, ib, B);
                    const bool ok =
                        okA && okB && (kHull || (A.type != D3D_HULL && B.type != D3D_HULL));
                    if (ok) {
                        have = M::start(g, pq, ia, ib, prm, o);
                        ta = A.type;
                        tb = B.type;
                        if constexpr (kCache) {
                            const bool ha = A.type == D3D_HULL, hb = B.type == D3D_HULL;
                            nA = ha ? A.nv : 0;
                            const int nB = hb ? B.nv : 0;
                            cached = nA + nB <= cache_verts<G>() && (!ha || A.voff64 < 0) &&
                                     (!hb || B.voff64 < 0);
                            two = ha && hb;
                            ncA = ha ? (int)A.p[2] : 0;
                            const int ncB = hb ? (int)B.p[2] : 0;
                            bounded = !cached && ncA + ncB > 0 &&
                                      4 * (ncA + ncB) <= cache_words<G>();
                            nrec = ncA + ncB;
                            if (cached) {
                                if (ha) cache_fill<G>(s, A, cache, 0, sub);
                                if (hb) cache_fill<G>(s, B, cache, nA, sub);
                            } else if (bounded) {
                                float4 *slot = reinterpret_cast<float4 *>(cache);
                                if (ncA > 0) bounds_fill<G>(s, A, slot, 0, sub);
                                if (ncB > 0) bounds_fill<G>(s, B, slot, ncA, sub);
                            }
                            if constexpr (slot_recs<G>()) {
                                double *rf = reinterpret_cast<double *>(cache + cache_words<G>());
                                int32_t *ri = reinterpret_cast<int32_t *>(rf + 32);
                                for (int k = sub; k < 40; k += G) {
                                    if (k < 32)
                                        rf[k] = s.shape_f64[16 * (int64_t)(k < 16 ? ia : ib) + (k & 15)];
                                    else
                                        ri[k - 32] = s.shape_i32[4 * (int64_t)(k < 36 ? ia : ib) + (k & 3)];
                                }
                            }
                            // the group's lanes read what the others wrote
                            row_fence();
                        }
                    } else if (sub == 0) {
                        M::bad(pid, o);
                    }
                } else {
                    exhausted = true;
                }
            }
            // the cursor only grows: once any group sees an item past the end
            // the class is empty for every group of the wavefront
            if (__ballot(exhausted) != 0ull) exhausted = true;
        }
        if (__ballot(have) == 0ull) {
            if (__ballot(!exhausted) == 0ull) break;
            continue;
        }
        if (have) {
            bool running = true;
            if (!M::more(g, prm)) {
                running = false;
            } else {
                // the records were validated when the pair was taken
                SupportPair w;
                // a wavefront in its support sweep (memory rounds) issues ahead of
                // those in their FP64 simplex step, so its loads go out sooner;
                // priority only orders issue between the SIMD's wavefronts
                __builtin_amdgcn_s_setprio(2);
                if constexpr (kCache) {
                    if (cached)
                        w = support_pair_cached<G>(s, ia, ib, g.d, sub, cache, nA, two);
                    else if (bounded)
                        w = support_pair_bounds<G>(s, ia, ib, g.d, sub,
                                                   reinterpret_cast<const float4 *>(cache), ncA, nrec);
                    else
                        w = support_pair<G, kHull>(s, ia, ib, g.d, sub);
                } else if constexpr (!kHull) {
                    w = support_pair_analytic(s, ia, ib, ta, tb, g.d);
                } else {
                    w = support_pair<G, kHull>(s, ia, ib, g.d, sub);
                }
                __builtin_amdgcn_s_setprio(0);
                running = M::template step<G>(g, pq, w.a, w.b, prm, o);
            }
            if (!running) {
                if (sub == 0) M::write(g, pq, pid, prm, o);
                have = false;
            }
        }
    }
}

// All work classes in one persistent launch: every wavefront walks the classes
// from the largest hulls to the analytic pairs (size classes 7 .. 0, the pairs
// of two hulls before those of one at each size), switching its lanes per pair
// at each class, so classes overlap without a launch per class.
// lanes_per_pair holds resolved values (see queue_params; class 0: 1, 2 or 4).
template <class M>
__device__ __forceinline__ void run_all(const d3d_scene &s, const int32_t *__restrict__ pa,
                                        const int32_t *__restrict__ pb,
                                        const int32_t *__restrict__ order,
                                        const int32_t *__restrict__ cls_begin,
                                        const int32_t *__restrict__ cls_count,
                                        int32_t *__restrict__ cls_cursor, const d3d_gjk_params &prm,
                                        const typename M::Out &o, double *pq_lds) {
    double *pq_wave = pq_lds + 24 * kWave * (threadIdx.x / kWave);
    const int n_waves = (int)gridDim.x * (kQBlock / kWave);
    // A batch that leaves wavefronts idle widens the groups of the classes whose
    // lanes are the table's (negative entries): all by the largest factor that
    // still gives every pair a group at once.  More lanes shorten a pair's hull
    // sweeps and its longest chain; once the chip is full they only add FP64 work,
    // which every lane of a group repeats.  Distance batches with the table's lanes
    // and widened: 300 mixed pairs 401 and 281 us, 4,096 mixed 477 and 413, 16,384
    // mixed 691 and 659; overlapping hulls of 64 to 256 vertices, 64 pairs 155 and
    // 72 us, 2,048 pairs 158 and 82, 8,192 pairs 205 and 190.  Stopping at half the
    // chip leaves 2,048 of those pairs at 140 us.
    int64_t lanes = 0;
    for (int c = 0; c < kNumClasses; ++c) lanes += (int64_t)cls_count[c] * abs(prm.lanes_per_pair[c]);
    int widen = 1;
    while (widen < kWave && 2 * widen * lanes <= (int64_t)n_waves * kWave) widen *= 2;
    int rot = 0;  // wavefronts given a fixed chunk by the classes walked so far
    for (int step = 0; step < kNumClasses; ++step) {
        const int cls = (step & 1) ? kSizeClasses - 1 - step / 2 : kNumClasses - 1 - step / 2;
        const int count = cls_count[cls];
        if (count == 0) continue;
        const int begin = cls_begin[cls];
        int32_t *cur = cls_cursor + cls;
        const int table = prm.lanes_per_pair[cls];
        int G = abs(table);
        if (table < 0 && cls != 0) {
            // pairs of at most 128 vertices have no use for the widths between: two
            // 32-vertex hulls, 4,096 pairs 72 us with 16 lanes and 73 with 32, 2,048
            // pairs 66 with 16, 67 with 32 and 62 with 64
            const int wide = min(G * widen, kWave);
            G = (cls & (kSizeClasses - 1)) <= 2 && wide < kWave ? G : wide;
        }
        // items per claim: claim_factor * (64 / G), or the class's fair share per
        // wavefront when that is smaller, so a small batch spreads its pairs
        // over all wavefronts instead of a few wavefronts holding all of them
        const int full = prm.claim_factor * (kWave / G);
        const int chunk = claim_chunk(count, n_waves, full);
        if (cls == 0) {
            if (G <= 1) run_class<M, 1, false>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot);
            else if (G == 2) run_class<M, 2, false>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot);
            else run_class<M, 4, false>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot);
        } else {
            switch (G) {
            case 1: run_class<M, 1, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            case 2: run_class<M, 2, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            case 4: run_class<M, 4, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            case 8: run_class<M, 8, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            case 16: run_class<M, 16, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            case 32: run_class<M, 32, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            default: run_class<M, 64, true>(s, pa, pb, order, begin, count, cur, prm, o, pq_wave, chunk, rot); break;
            }
        }
        const uint32_t used = chunks_of(count, chunk);
        rot = (int)(((int64_t)rot + (used < (uint32_t)n_waves ? (int)used : n_waves)) % n_waves);
    }
}

// Sorts the pairs of a batch into `w` (work class, type of A, type of B) on
// `stream`: w.order, the class ranges and cleared class cursors; epa_count
// (optional, two counters) is cleared too.
int queue_sort(const d3d_scene &s, const int32_t *pa, const int32_t *pb, int64_t n, const QueueWs &w,
               hipStream_t stream, unsigned long long *epa_count = nullptr);

// Persistent blocks per compute unit for n pairs: the caller's where given, else
// what is resident at the occupancy that suits the batch, 2 up to loose_max pairs
// and 3 above.  A batch within loose_max runs the occupancy-2 kernel unless the
// caller asks for more blocks than that holds.
constexpr int batch_blocks(int64_t n, int64_t loose_max, int asked) {
    return asked > 0 ? asked : n <= loose_max ? 2 : 3;
}
constexpr bool batch_is_loose(int64_t n, int64_t loose_max, int asked) {
    return n <= loose_max && batch_blocks(n, loose_max, asked) <= 2;
}

// prm with the lanes per class (negative: the table's, which the kernel may
// widen; positive: the caller's) and the launch shape resolved for n pairs; the
// grid of a persistent launch (kQBlock threads per block).
d3d_gjk_params queue_params(const d3d_gjk_params &prm, int64_t n, int64_t loose_max);
unsigned queue_grid(const d3d_gjk_params &resolved);

}  // namespace d3d
