// d3d_bvh.hip -- AABB broad phase on gfx950: a packed 8-wide tree over boxes
// sorted along a Hilbert curve, its refit and its overlap queries.
//
// Build (all on the caller's stream, inside a caller-owned buffer):
//   1. bounds of the AABB centres (block partials)
//   2. 30-bit Hilbert codes of the centres
//   3. radix sort of (code, index), 3 stable passes of 10 bits
//   4. levels: level 0 holds the boxes in curve order (FP32, rounded outward),
//      a record of level k + 1 the union of 8 consecutive records of level k
// The tree has no pointers: its shape follows from n alone, so a refit is step
// 4 again, and a level-k record is found by its index.
// Query: 8 lanes test the 8 children of a node in one coalesced load and push
// the overlapping ones on an LDS stack; FP32 tests are conservative, and each
// leaf hit is confirmed with the reference's closed-interval FP64 test
// (aabb_tree.py:503-527), so the pair set equals the brute-force set of
// all_aabbs_overlap exactly.
#include "d3d_bvh_core.hpp"
#include "d3d_device.hpp"
#include "d3d_runtime.hpp"

namespace d3d {

constexpr int kBvhBlock = 256;
constexpr int kDigitBits = 10;
constexpr int kDigits = 1 << kDigitBits;
constexpr int kSortPasses = 3;  // 30-bit codes

// A box of the tree: level 0 carries the original box index.  Rows that pad a
// level to a multiple of 8 are NaN: no comparison with them holds.
struct BvhNode {
    float lo[3];
    int32_t id;
    float hi[3];
    int32_t pad;
};
static_assert(sizeof(BvhNode) == 32, "a node's 8 children are 256 consecutive bytes");

struct BvhView {
    BvhNode *nodes;
    uint64_t *items, *items_alt;  // code << 32 | index
    int32_t *order;               // sorted position -> original index
    int32_t *hist;                // tiles x kDigits
    int32_t *dtot;                // kDigits
    double *bpart;                // bound partials 6 * kBoundBlocks
};

constexpr int kBoundBlocks = 256;

// Items of a sort tile per thread: a tile per block, so a small set takes
// small tiles to have blocks for more than a few compute units, a large one
// fewer columns to scan.  The whole build with 4 / 8 / 16 items: 5,003 boxes
// 41 / 50 / 66 us, 262,144 boxes 66 / 69 / 86 us, 524,288 boxes 93 / 89 / 100
// us, 1,048,576 boxes 152 / 138 / 137 us.
__host__ __device__ inline int sort_items(int64_t n) { return n < 393216 ? 4 : 8; }
__host__ __device__ inline int64_t sort_tiles(int64_t n) {
    const int64_t tile = (int64_t)kBvhBlock * sort_items(n);
    return (n + tile - 1) / tile;
}

__host__ __device__ inline int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

// One walk over the buffer's parts, for its size and for its pointers.
inline int64_t bvh_layout(int64_t n, char *base, BvhView *v) {
    const int64_t m = n > 0 ? n : 1;
    int64_t b = 0;
    auto part = [&](int64_t bytes) {
        char *p = base ? base + b : nullptr;
        b += align256(bytes);
        return p;
    };
    BvhView w;
    w.nodes = (BvhNode *)part(bvh_levels(m).nodes * (int64_t)sizeof(BvhNode));
    w.items = (uint64_t *)part(m * 8);
    w.items_alt = (uint64_t *)part(m * 8);
    w.order = (int32_t *)part(m * 4);
    w.hist = (int32_t *)part(sort_tiles(m) * kDigits * 4);
    w.dtot = (int32_t *)part(kDigits * 4);
    w.bpart = (double *)part(6 * kBoundBlocks * 8);
    if (v) *v = w;
    return b;
}

inline int64_t bvh_bytes(int64_t n) { return bvh_layout(n, nullptr, nullptr); }

inline BvhView bvh_view(void *base, int64_t n) {
    BvhView v;
    bvh_layout(n, (char *)base, &v);
    return v;
}

// ------------------------------------------------------------- bounds

__global__ __launch_bounds__(kBvhBlock) void bvh_bounds_partial(const double *__restrict__ aabbs,
                                                                int64_t n, double *__restrict__ part) {
    __shared__ double red[6][kBvhBlock];
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * kBvhBlock + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * kBvhBlock) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double c = (aabbs[6 * i + 2 * a] + aabbs[6 * i + 2 * a + 1]) * 0.5;
            lo[a] = fmin(lo[a], c);
            hi[a] = fmax(hi[a], c);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        red[a][threadIdx.x] = lo[a];
        red[3 + a][threadIdx.x] = hi[a];
    }
    __syncthreads();
    for (int off = kBvhBlock / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                red[a][threadIdx.x] = fmin(red[a][threadIdx.x], red[a][threadIdx.x + off]);
                red[3 + a][threadIdx.x] = fmax(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + off]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) part[6 * blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__device__ __forceinline__ int item_digit(uint64_t item, int pass) {
    return (int)(item >> (32 + kDigitBits * pass)) & (kDigits - 1);
}

// Hilbert codes of a sort tile, and the tile's counts of the first digit.  The
// at most kBoundBlocks bound partials are merged again by every block (one per
// thread, butterflies, then the wavefronts'): a launch of its own for that took
// 5 us, and 51 us where one thread walked the partials.
__global__ __launch_bounds__(kBvhBlock) void bvh_code_kernel(const double *__restrict__ aabbs,
                                                               int64_t n, int items,
                                                               const double *__restrict__ part,
                                                               int nparts, uint64_t *__restrict__ out,
                                                               int32_t *__restrict__ hist) {
    static_assert(kBoundBlocks == kBvhBlock, "one partial per thread");
    constexpr int kWaves = kBvhBlock / kWave;
    __shared__ double wred[kWaves][6];
    __shared__ int32_t h[kDigits];
    const int t = threadIdx.x;
    for (int d = t; d < kDigits; d += kBvhBlock) h[d] = 0;
    double b[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) b[k] = t < nparts ? part[6 * t + k] : (k < 3 ? INFINITY : -INFINITY);
    for_butterfly<kWave>([&](auto o) {
        constexpr int OFF = decltype(o)::value;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            double p, q;
            xpair<OFF>(b[k], p, q);
            b[k] = k < 3 ? fmin(p, q) : fmax(p, q);
        }
    });
    if ((t & (kWave - 1)) == 0)
#pragma unroll
        for (int k = 0; k < 6; ++k) wred[t / kWave][k] = b[k];
    __syncthreads();
    double lo[3], ext[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double mn = wred[0][a], mx = wred[0][3 + a];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) {
            mn = fmin(mn, wred[w][a]);
            mx = fmax(mx, wred[w][3 + a]);
        }
        lo[a] = mn;
        ext[a] = mx - mn;
    }
    const int64_t base = (int64_t)blockIdx.x * kBvhBlock * items;
    for (int j = 0; j < items; ++j) {
        const int64_t i = base + (int64_t)j * kBvhBlock + t;
        if (i >= n) break;
        uint32_t q[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double c = (aabbs[6 * i + 2 * a] + aabbs[6 * i + 2 * a + 1]) * 0.5;
            double u = ext[a] > 0.0 ? (c - lo[a]) / ext[a] : 0.0;
            u = fmin(fmax(u, 0.0), 1.0);
            q[a] = (uint32_t)fmin(u * 1024.0, 1023.0);
        }
        const uint32_t key = hilbert30(q[0], q[1], q[2]);
        const uint64_t item = ((uint64_t)key << 32) | (uint32_t)i;
        out[i] = item;
        atomicAdd(&h[item_digit(item, 0)], 1);
    }
    __syncthreads();
    for (int d = t; d < kDigits; d += kBvhBlock) hist[(int64_t)blockIdx.x * kDigits + d] = h[d];
}

// --------------------------------------------------------- radix sort
//
// Three passes over (code, index) items of 8 bytes, each: counts per tile
// (rows of kDigits, tile-major, so both the count and the scatter read and
// write whole rows), an exclusive scan of every digit's column, the scatter.

__global__ __launch_bounds__(kBvhBlock) void rs_hist_kernel(const uint64_t *__restrict__ in, int64_t n,
                                                            int items, int pass,
                                                            int32_t *__restrict__ hist) {
    __shared__ int32_t h[kDigits];
    for (int d = threadIdx.x; d < kDigits; d += kBvhBlock) h[d] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kBvhBlock * items;
    for (int j = 0; j < items; ++j) {
        const int64_t i = base + (int64_t)j * kBvhBlock + threadIdx.x;
        if (i < n) atomicAdd(&h[item_digit(in[i], pass)], 1);
    }
    __syncthreads();
    for (int d = threadIdx.x; d < kDigits; d += kBvhBlock) hist[(int64_t)blockIdx.x * kDigits + d] = h[d];
}

// Exclusive scan of every digit's column over the tiles, in place, and the
// column sums: a block takes 64 digits, its 16 wavefronts a sixteenth of the
// tiles each, so a wavefront's loads are whole 256-byte rows and independent of
// each other.  (One block walking all columns in order took 112 us for 256
// tiles of 256 digits; this takes 5 us for 256 tiles of 1,024.)
constexpr int kScanSegs = 16;
__global__ __launch_bounds__(kWave * kScanSegs) void rs_scan_kernel(int32_t *__restrict__ hist,
                                                                    int64_t tiles,
                                                                    int32_t *__restrict__ dtot) {
    __shared__ int32_t seg[kScanSegs][kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int d = blockIdx.x * kWave + lane;
    const int64_t per = (tiles + kScanSegs - 1) / kScanSegs;
    const int64_t t0 = min(per * w, tiles), t1 = min(t0 + per, tiles);
    int32_t sum = 0;
#pragma unroll 8
    for (int64_t k = t0; k < t1; ++k) sum += hist[k * kDigits + d];
    seg[w][lane] = sum;
    __syncthreads();
    int32_t run = 0;
    for (int k = 0; k < w; ++k) run += seg[k][lane];
    if (w == kScanSegs - 1) dtot[d] = run + sum;
#pragma unroll 8
    for (int64_t k = t0; k < t1; ++k) {
        const int32_t c = hist[k * kDigits + d];
        hist[k * kDigits + d] = run;
        run += c;
    }
}

// Stable scatter of a tile (an LSD sort needs every pass to be stable).  A
// wavefront owns a run of kItems * 64 consecutive items; it finds the lanes
// holding the same digit by matching the digit bits with ballots, and its rank
// is its own running count of the digit plus the earlier lanes' matches, with
// no barrier between chunks.  Then the wavefronts' counts become positions:
// digits before (the scan of the column sums, redone by every block), tiles
// before (hist) and wavefronts before.  The last pass keeps the index only.
template <int kItems, bool kLast>
__global__ __launch_bounds__(kBvhBlock) void rs_scatter_kernel(const uint64_t *__restrict__ in,
                                                               int64_t n, int pass,
                                                               const int32_t *__restrict__ hist,
                                                               const int32_t *__restrict__ dtot,
                                                               uint64_t *__restrict__ out,
                                                               int32_t *__restrict__ order) {
    constexpr int kWaves = kBvhBlock / kWave;
    constexpr int kPer = kDigits / kBvhBlock;  // digits per thread
    __shared__ int32_t wcnt[kWaves][kDigits];
    __shared__ int32_t wsum[kWaves];
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t / kWave;
    const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
        for (int d = t; d < kDigits; d += kBvhBlock) wcnt[w][d] = 0;
    const int64_t base = ((int64_t)blockIdx.x * kWaves + wave) * kItems * kWave + lane;
    uint64_t item[kItems];
    int rank[kItems];
#pragma unroll
    for (int j = 0; j < kItems; ++j) item[j] = base + j * kWave < n ? in[base + j * kWave] : 0ull;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const bool valid = base + j * kWave < n;
        const int dig = item_digit(item[j], pass);
        unsigned long long same = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            const unsigned long long m = __ballot((dig >> b) & 1);
            same &= ((dig >> b) & 1) ? m : ~m;
        }
        const int before = __popcll(same & lt);
        rank[j] = wcnt[wave][dig] + before;
        // the digit's lanes have read the count before its first lane raises it
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        if (valid && before == 0) wcnt[wave][dig] += __popcll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // digits [kPer t, kPer t + kPer): start of the digit over all tiles
    int32_t start[kPer];
    int32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        start[k] = sum;
        sum += dtot[kPer * t + k];
    }
    int32_t incl = sum;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t v = __shfl_up(incl, off);
        if (lane >= off) incl += v;
    }
    if (lane == kWave - 1) wsum[wave] = incl;
    __syncthreads();
    int32_t first = incl - sum;
    for (int w = 0; w < wave; ++w) first += wsum[w];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const int d = kPer * t + k;
        int32_t pos = first + start[k] + hist[(int64_t)blockIdx.x * kDigits + d];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int32_t c = wcnt[w][d];
            wcnt[w][d] = pos;
            pos += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        if (base + j * kWave >= n) break;
        const int32_t pos = wcnt[wave][item_digit(item[j], pass)] + rank[j];
        if (kLast) order[pos] = (int32_t)(uint32_t)item[j];
        else out[pos] = item[j];
    }
}

// -------------------------------------------------------------- levels

// Up to four consecutive levels in one launch: a thread makes one record of
// level `base` (base 0: the outward-rounded FP32 box of its leaf; otherwise it
// reads the record an earlier launch made), then 8 lanes, the 64 of the
// wavefront and the block's 8 wavefronts merge theirs into records of the next
// three.  Lanes past a level's count write the rows that pad it to a multiple
// of 8.  Bound: the gather of the boxes in curve order (1,048,576 boxes: 32
// us, 48 bytes at random per box; the refit of the pointer tree this replaced
// took 62 launches and 595 us).
__device__ __forceinline__ void put_node(BvhNode *nd, const float (&lo)[3], const float (&hi)[3], int id) {
    float4 *p = reinterpret_cast<float4 *>(nd);
    p[0] = make_float4(lo[0], lo[1], lo[2], __int_as_float(id));
    p[1] = make_float4(hi[0], hi[1], hi[2], 0.0f);
}

template <bool kLeaf>
__global__ __launch_bounds__(kLevelBlock) void bvh_level_kernel(BvhLevels lv, int base,
                                                                const double *__restrict__ aabbs,
                                                                const int32_t *__restrict__ order,
                                                                BvhNode *__restrict__ nodes) {
    __shared__ float wlo[kLevelBlock / kWave][3], whi[kLevelBlock / kWave][3];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    int64_t i = (int64_t)blockIdx.x * kLevelBlock + threadIdx.x;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    const float nan3[3] = {NAN, NAN, NAN};
    const bool in = i < lv.count[base];
    if (kLeaf) {
        if (in) {
            // a refit finds the order in the leaf records
            const int32_t id = order ? order[i] : nodes[i].id;
            const double *A = aabbs + 6 * (int64_t)id;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                lo[a] = __double2float_rd(A[2 * a]);
                hi[a] = __double2float_ru(A[2 * a + 1]);
            }
            put_node(&nodes[i], lo, hi, id);
        } else if (i < round8(lv.count[0])) {
            put_node(&nodes[i], nan3, nan3, 0);
        }
    } else if (in) {
        const BvhNode nd = nodes[lv.off[base] + i];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = nd.lo[a];
            hi[a] = nd.hi[a];
        }
    }
    auto merge = [&](auto o) {
        constexpr int OFF = decltype(o)::value;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float p, q;
            xpair<OFF>(lo[a], p, q);
            lo[a] = fminf(p, q);
            xpair<OFF>(hi[a], p, q);
            hi[a] = fmaxf(p, q);
        }
    };
    auto put_level = [&](int level, bool mine) {
        i >>= 3;
        if (level > lv.top || !mine) return;
        if (i < lv.count[level]) put_node(&nodes[lv.off[level] + i], lo, hi, -1);
        else if (i < round8(lv.count[level])) put_node(&nodes[lv.off[level] + i], nan3, nan3, -1);
    };
    merge(IntC<1>{});
    merge(IntC<2>{});
    merge(IntC<4>{});
    put_level(base + 1, (lane & 7) == 0);
    merge(IntC<8>{});
    merge(IntC<16>{});
    merge(IntC<32>{});
    put_level(base + 2, lane == 0);
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            wlo[wave][a] = lo[a];
            whi[wave][a] = hi[a];
        }
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int w = 1; w < kLevelBlock / kWave; ++w)
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                lo[a] = fminf(lo[a], wlo[w][a]);
                hi[a] = fmaxf(hi[a], whi[w][a]);
            }
    put_level(base + 3, threadIdx.x == 0);
}

// Every level from the boxes: order from the sort, or NULL for a refit.
static void level_launches(const BvhView &v, const double *aabbs, int64_t n, const int32_t *order,
                           hipStream_t st) {
    const BvhLevels lv = bvh_levels(n);
    for (int base = 0; base == 0 || base < lv.top; base += kLevelStep) {
        const int64_t blocks = level_blocks(lv, base);
        if (base == 0)
            hipLaunchKernelGGL(bvh_level_kernel<true>, dim3((unsigned)blocks), dim3(kLevelBlock), 0, st, lv, base,
                               aabbs, order, v.nodes);
        else
            hipLaunchKernelGGL(bvh_level_kernel<false>, dim3((unsigned)blocks), dim3(kLevelBlock), 0, st, lv, base,
                               aabbs, order, v.nodes);
    }
}

// ------------------------------------------------------------- query

// Rows of a query's own hit list; hits past it go to the overflow list.
constexpr int kHitRows = 16;

// Scratch of a sorted query (device pointers into the caller's workspace).
struct QueryWs {
    unsigned long long *base;  // per block: its queries' hits, then their start
    int32_t *most;             // per block: most hits of one query
    int32_t *count;            // per query
    unsigned long long *off;   // per query: start of its pairs
    int32_t *rows;             // per query kHitRows box indices, as found
    int32_t *ovf;              // (query, rank, box) of the hits past the rows
    int32_t *stage;            // per pair: box indices of long lists, as found
};

// Overlaps of the queries with the tree by groups of QL lanes: each round a
// group pops QL / 8 nodes of its stack, 8 lanes each, one child per lane; the
// overlapping children are pushed, or on level 0 tested exactly and reported.
// A round costs one dependent load (a second one on level 0), so it is the
// number of rounds in a row that bounds a query; many queries fill the chip
// with 8 lanes each, a few take more nodes per round instead.  (One lane per
// query on a pointer tree, a load per node: 65,536 queries of 1,048,576 boxes
// 825 us; this kernel 80 us.)
// kSorted: hits go to the query's rows (or the overflow list) with their
// count; otherwise a block gathers its first kBlockHits hits in LDS and takes
// their place in `pairs` with one atomic, later ones are appended as they are
// found.  With an atomic per find 65,536 queries of 1,048,576 boxes (160,306
// pairs) took 844 us, the atomics on the one counter; now 89 us.
constexpr int kBlockHits = 512;

template <int QL, bool kSorted>
__global__ __launch_bounds__(kBvhBlock) void bvh_query_kernel(
    BvhLevels lv, const BvhNode *__restrict__ nodes, const double *__restrict__ aabbs,
    const double *__restrict__ q, int64_t first, int64_t m, int32_t *__restrict__ pairs, int64_t cap,
    unsigned long long *__restrict__ counter, QueryWs ws) {
    constexpr int kGroups = kBvhBlock / QL;
    constexpr int W = QL / 8;
    constexpr int kStack = query_stack(W);
    __shared__ int32_t stack[kGroups][kStack];
    __shared__ int64_t off[kBvhMaxLevels];
    __shared__ int32_t found[kGroups];
    __shared__ int2 hits[kSorted ? 1 : kBlockHits];
    __shared__ int32_t n_hits;
    __shared__ unsigned long long hits_at;
    const int t = threadIdx.x, g = t / QL, sub = t & (QL - 1);
    const int slot = sub >> 3, child = sub & 7;
    const int lane = lane_id();
    if (t < kBvhMaxLevels) off[t] = lv.off[t];
    const int64_t qi = first + (int64_t)blockIdx.x * kGroups + g;
    const bool valid = qi < m;
    double Q[6];
    float qlo[3], qhi[3];
#pragma unroll
    for (int k = 0; k < 6; ++k) Q[k] = valid ? q[6 * qi + k] : 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        qlo[a] = __double2float_rd(Q[2 * a]);
        qhi[a] = __double2float_ru(Q[2 * a + 1]);
    }
    if (sub == 0) stack[g][0] = lv.top << kNodeBits;
    if (t == 0) n_hits = 0;
    __syncthreads();
    const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    int *const st = stack[g];
    int sp = valid ? 1 : 0;
    int cnt = 0;
    while (sp > 0) {
        const int take = query_take(sp, W);
        const int e = slot < take ? st[sp - 1 - slot] : -1;
        sp -= take;
        bool push = false, hit = false;
        int level = 0, rec = 0, orig = 0;
        if (e >= 0) {
            level = e >> kNodeBits;
            rec = 8 * (e & ((1 << kNodeBits) - 1)) + child;
            const float4 *p = reinterpret_cast<const float4 *>(nodes + off[level] + rec);
            const float4 lo = p[0], hi = p[1];
            const bool ov = lo.x <= qhi[0] && hi.x >= qlo[0] && lo.y <= qhi[1] && hi.y >= qlo[1] &&
                            lo.z <= qhi[2] && hi.z >= qlo[2];
            push = ov && level > 0;
            if (ov && level == 0) {
                orig = __float_as_int(lo.w);
                const double *A = aabbs + 6 * (int64_t)orig;
                // aabb_overlap(tree_aabb, test_aabb), aabb_tree.py:520-527
                hit = A[0] <= Q[1] && A[1] >= Q[0] && A[2] <= Q[3] && A[3] >= Q[2] && A[4] <= Q[5] &&
                      A[5] >= Q[4];
            }
        }
        const unsigned long long pm = group_bits<QL>(__ballot(push), lane);
        const unsigned long long below = group_bits<QL>(lt, lane);
        if (push) st[sp + __popcll(pm & below)] = ((level - 1) << kNodeBits) | rec;
        sp += __popcll(pm);
        const unsigned long long all = __ballot(hit);
        if (all != 0ull) {
            const unsigned long long hm = group_bits<QL>(all, lane);
            if constexpr (kSorted) {
                if (hit) {
                    const int r = cnt + __popcll(hm & below);
                    if (r < kHitRows) {
                        ws.rows[kHitRows * qi + r] = orig;
                    } else {
                        const unsigned long long pos = atomicAdd(counter, 1ull);
                        if (pos < (unsigned long long)cap) {
                            ws.ovf[3 * pos] = (int32_t)qi;
                            ws.ovf[3 * pos + 1] = r;
                            ws.ovf[3 * pos + 2] = orig;
                        }
                    }
                }
                cnt += __popcll(hm);
            } else if (hit) {
                const int r = atomicAdd(&n_hits, 1);
                if (r < kBlockHits) {
                    hits[r] = make_int2((int32_t)qi, orig);
                } else {
                    const unsigned long long pos = atomicAdd(counter, 1ull);
                    if (pos < (unsigned long long)cap) {
                        pairs[2 * pos] = (int32_t)qi;
                        pairs[2 * pos + 1] = orig;
                    }
                }
            }
        }
        // the group's lanes read what the others pushed
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if constexpr (!kSorted) {
        __syncthreads();
        const int k = min(n_hits, kBlockHits);
        if (t == 0 && k > 0) hits_at = atomicAdd(counter, (unsigned long long)k);
        __syncthreads();
        for (int r = t; r < k; r += kBvhBlock) {
            const unsigned long long pos = hits_at + (unsigned long long)r;
            if (pos < (unsigned long long)cap) {
                pairs[2 * pos] = hits[r].x;
                pairs[2 * pos + 1] = hits[r].y;
            }
        }
    }
    if constexpr (kSorted) {
        if (sub == 0) {
            found[g] = cnt;
            if (valid) ws.count[qi] = cnt;
        }
        __syncthreads();
        if (t == 0) {
            unsigned long long sum = 0;
            int most = 0;
            for (int k = 0; k < kGroups; ++k) {
                sum += (unsigned long long)found[k];
                most = max(most, found[k]);
            }
            ws.base[blockIdx.x] = sum;
            ws.most[blockIdx.x] = most;
        }
    }
}

// Starts of the query blocks' pairs (exclusive scan of base in place) by one
// block; result[0] the number of pairs, result[1] the most of one query.
__global__ __launch_bounds__(1024) void query_scan_kernel(unsigned long long *__restrict__ base,
                                                          const int32_t *__restrict__ most,
                                                          int64_t blocks,
                                                          unsigned long long *__restrict__ result) {
    __shared__ unsigned long long part[1024];
    __shared__ int32_t big[1024];
    const int t = threadIdx.x;
    const int64_t per = (blocks + 1023) / 1024;
    const int64_t b0 = min((int64_t)t * per, blocks), b1 = min(b0 + per, blocks);
    unsigned long long sum = 0;
    int mx = 0;
    for (int64_t k = b0; k < b1; ++k) {
        sum += base[k];
        mx = max(mx, most[k]);
    }
    part[t] = sum;
    big[t] = mx;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned long long v = t >= d ? part[t - d] : 0ull;
        const int o = t >= d ? big[t - d] : 0;
        __syncthreads();
        part[t] += v;
        big[t] = max(big[t], o);
        __syncthreads();
    }
    unsigned long long run = part[t] - sum;
    for (int64_t k = b0; k < b1; ++k) {
        const unsigned long long c = base[k];
        base[k] = run;
        run += c;
    }
    if (t == 1023) {
        result[0] = part[1023];
        result[1] = (unsigned long long)big[1023];
    }
}

// The pairs of kQueries queries (a block of the query kernel), 16 lanes each:
// a list that fits the query's rows is ranked by counting the smaller indices
// and written in order, to at most `room` rows; of a longer one the rows are
// copied to its place in `stage`, where query_spill_kernel adds the rest.
template <int kQueries>
__global__ __launch_bounds__(kQueries * kHitRows) void query_write_kernel(int64_t m, int64_t room,
                                                                          int64_t cap, QueryWs ws,
                                                                          int32_t *__restrict__ pairs) {
    static_assert(kHitRows == 16 && kQueries >= 2 && kQueries <= 32, "16 lanes read at most two counts each");
    __shared__ int32_t cnt[32];
    __shared__ int32_t vals[kQueries][kHitRows];
    const int t = threadIdx.x, g = t / kHitRows, sub = t & (kHitRows - 1);
    const int64_t q0 = (int64_t)blockIdx.x * kQueries;
    if (t < 32) cnt[t] = t < kQueries && q0 + t < m ? ws.count[q0 + t] : 0;
    __syncthreads();
    // hits of the block's earlier queries
    int before = (sub < g ? cnt[sub] : 0) + (sub + 16 < g ? cnt[sub + 16] : 0);
    for_butterfly<16>([&](auto o) {
        int a, b;
        xpair<decltype(o)::value>(before, a, b);
        before = a + b;
    });
    const int64_t q = q0 + g;
    const int k = cnt[g];
    const unsigned long long off = ws.base[blockIdx.x] + (unsigned long long)before;
    if (q < m && sub == 0) ws.off[q] = off;
    const int b = sub < k ? ws.rows[kHitRows * q + sub] : 0x7fffffff;
    vals[g][sub] = b;
    __syncthreads();
    if (sub >= k) return;
    if (k > kHitRows) {
        if (off + sub < (unsigned long long)cap) ws.stage[off + sub] = b;
        return;
    }
    int rank = 0;
#pragma unroll
    for (int j = 0; j < kHitRows; ++j) rank += vals[g][j] < b ? 1 : 0;
    const unsigned long long pos = off + (unsigned long long)rank;
    if (pos < (unsigned long long)room) {
        pairs[2 * pos] = (int32_t)q;
        pairs[2 * pos + 1] = b;
    }
}

// The overflow list's hits to their places in `stage`.
__global__ __launch_bounds__(kBvhBlock) void query_spill_kernel(
    const unsigned long long *__restrict__ n_ovf, int64_t cap, QueryWs ws) {
    const unsigned long long n = min(*n_ovf, (unsigned long long)cap);
    for (unsigned long long i = (unsigned long long)blockIdx.x * kBvhBlock + threadIdx.x; i < n;
         i += (unsigned long long)gridDim.x * kBvhBlock) {
        const unsigned long long pos = ws.off[ws.ovf[3 * i]] + (unsigned long long)ws.ovf[3 * i + 1];
        if (pos < (unsigned long long)cap) ws.stage[pos] = ws.ovf[3 * i + 2];
    }
}

// Lists longer than a query's rows, ranked by counting in `stage` by one
// wavefront each.
__global__ __launch_bounds__(kBvhBlock) void query_long_kernel(int64_t m, int64_t cap, QueryWs ws,
                                                               int32_t *__restrict__ pairs) {
    const int lane = lane_id();
    const int64_t waves = (int64_t)gridDim.x * (kBvhBlock / kWave);
    for (int64_t q = ((int64_t)blockIdx.x * kBvhBlock + threadIdx.x) / kWave; q < m; q += waves) {
        const int k = ws.count[q];
        if (k <= kHitRows) continue;
        const unsigned long long off = ws.off[q];
        if (off + (unsigned long long)k > (unsigned long long)cap) continue;
        const int32_t *list = ws.stage + off;
        for (int i = lane; i < k; i += kWave) {
            const int b = list[i];
            int rank = 0;
            for (int j = 0; j < k; ++j) rank += list[j] < b ? 1 : 0;
            pairs[2 * (off + rank)] = (int32_t)q;
            pairs[2 * (off + rank) + 1] = b;
        }
    }
}

__global__ void bvh_zero_counter(unsigned long long *c) { *c = 0ull; }

// ------------------------------------------------------------ dense overlap
//
// all_aabbs_overlap (aabb_tree.py:465-500) by brute force, for box sets
// whose product n * m is small enough that testing every pair beats a tree
// walk (dense overlaps: a tree query with ~1000 hits is a long serial walk).
// One wavefront takes kDenseRows rows of `a` (the boxes stay in scalar
// registers) and sweeps `b` 64 boxes at a time, one per lane; a count pass,
// an exclusive scan, and a write pass that places each row's hits at the
// row's offset in b order (ballot ranks), so the pairs come out row-major
// (i outer, j inner), the reference's order, with no sort.
constexpr int kDenseRows = 4;
constexpr int kDenseBlock = 256;

__device__ __forceinline__ bool box_overlap(const double (&q)[6], const double *__restrict__ B) {
    // aabb_overlap(a_i, b_j), aabb_tree.py:520-527 (closed intervals)
    return q[0] <= B[1] && q[1] >= B[0] && q[2] <= B[3] && q[3] >= B[2] && q[4] <= B[5] &&
           q[5] >= B[4];
}

template <bool kWrite>
__global__ __launch_bounds__(kDenseBlock) void dense_overlap_kernel(
    const double *__restrict__ a, int64_t n, const double *__restrict__ b, int64_t m,
    unsigned long long *__restrict__ counts, const unsigned long long *__restrict__ total,
    int32_t *__restrict__ pairs, int64_t cap) {
    const int lane = lane_id();
    const int64_t wave = ((int64_t)blockIdx.x * kDenseBlock + threadIdx.x) / kWave;
    const int64_t row0 = wave * kDenseRows;
    if (row0 >= n) return;
    if (kWrite) {
        // nothing to write: no hits in these rows, or their place is past the room
        const unsigned long long first = counts[row0];
        const unsigned long long end = row0 + kDenseRows < n ? counts[row0 + kDenseRows] : *total;
        if (first == end || first >= (unsigned long long)cap) return;
    }
    double q[kDenseRows][6];
    unsigned long long off[kDenseRows];
#pragma unroll
    for (int r = 0; r < kDenseRows; ++r) {
        const int64_t row = min(row0 + r, n - 1);
#pragma unroll
        for (int c = 0; c < 6; ++c) q[r][c] = wave_uniform(a[6 * row + c]);
        off[r] = kWrite ? counts[row] : 0ull;
    }
    const unsigned long long lt = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    for (int64_t j0 = 0; j0 < m; j0 += kWave) {
        const int64_t j = j0 + lane;
        double B[6];
        const bool in = j < m;
#pragma unroll
        for (int c = 0; c < 6; ++c) B[c] = in ? b[6 * j + c] : 0.0;
#pragma unroll
        for (int r = 0; r < kDenseRows; ++r) {
            const bool hit = in && row0 + r < n && box_overlap(q[r], B);
            const unsigned long long msk = __ballot(hit);
            if (kWrite && hit) {
                const unsigned long long pos = off[r] + (unsigned long long)__popcll(msk & lt);
                if (pos < (unsigned long long)cap) {
                    pairs[2 * pos] = (int32_t)(row0 + r);
                    pairs[2 * pos + 1] = (int32_t)j;
                }
            }
            off[r] += (unsigned long long)__popcll(msk);
        }
    }
    if (!kWrite && lane < kDenseRows && row0 + lane < n) {
        unsigned long long mine = off[0];
#pragma unroll
        for (int r = 1; r < kDenseRows; ++r) mine = lane == r ? off[r] : mine;
        counts[row0 + lane] = mine;
    }
}

// Exclusive scan of counts[0..n) in place by one block; the sum to *total.
__global__ __launch_bounds__(1024) void dense_scan_kernel(unsigned long long *__restrict__ counts,
                                                          int64_t n,
                                                          unsigned long long *__restrict__ total) {
    __shared__ unsigned long long part[1024];
    const int t = threadIdx.x;
    const int64_t per = (n + 1023) / 1024;
    const int64_t lo = min((int64_t)t * per, n), hi = min(lo + per, n);
    unsigned long long sum = 0;
    for (int64_t k = lo; k < hi; ++k) sum += counts[k];
    part[t] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned long long v = t >= d ? part[t - d] : 0ull;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    unsigned long long run = part[t] - sum;
    for (int64_t k = lo; k < hi; ++k) {
        const unsigned long long c = counts[k];
        counts[k] = run;
        run += c;
    }
    if (t == 1023) *total = part[1023];
}

}  // namespace d3d

using namespace d3d;

extern "C" int64_t d3d_bvh_bytes(int64_t n) {
    if (n < 0) return -1;
    return bvh_bytes(n);
}

template <int kItems>
static void sort_launches(const BvhView &v, int64_t n, hipStream_t st) {
    const int64_t tiles = sort_tiles(n);
    uint64_t *in = v.items, *out = v.items_alt;
    for (int pass = 0; pass < kSortPasses; ++pass) {
        if (pass > 0)  // the code kernel counted the first digit
            hipLaunchKernelGGL(rs_hist_kernel, dim3((unsigned)tiles), dim3(kBvhBlock), 0, st, in, n,
                               kItems, pass, v.hist);
        hipLaunchKernelGGL(rs_scan_kernel, dim3(kDigits / kWave), dim3(kWave * kScanSegs), 0, st, v.hist,
                           tiles, v.dtot);
        if (pass + 1 < kSortPasses)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(rs_scatter_kernel<kItems, false>), dim3((unsigned)tiles),
                               dim3(kBvhBlock), 0, st, in, n, pass, v.hist, v.dtot, out, v.order);
        else
            hipLaunchKernelGGL(HIP_KERNEL_NAME(rs_scatter_kernel<kItems, true>), dim3((unsigned)tiles),
                               dim3(kBvhBlock), 0, st, in, n, pass, v.hist, v.dtot, out, v.order);
        uint64_t *x = in;
        in = out;
        out = x;
    }
}

extern "C" int d3d_bvh_build(const double *aabbs, int64_t n, void *bvh, int64_t bvh_bytes_avail,
                             void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 1 && n < (int64_t)0x40000000, "n must be in [1, 2^30)");
    D3D_CHECK_ARG(aabbs && bvh, "NULL buffer");
    D3D_CHECK_ARG(bvh_bytes_avail >= bvh_bytes(n), "bvh buffer smaller than d3d_bvh_bytes(n)");
    hipStream_t st = (hipStream_t)stream;
    BvhView v = bvh_view(bvh, n);
    const int64_t nb = (n + kBvhBlock - 1) / kBvhBlock;
    const int nparts = (int)(nb < kBoundBlocks ? nb : kBoundBlocks);
    hipLaunchKernelGGL(bvh_bounds_partial, dim3(nparts), dim3(kBvhBlock), 0, st, aabbs, n, v.bpart);
    D3D_CHECK_LAUNCH("bvh_bounds_partial");
    const int items = sort_items(n);
    hipLaunchKernelGGL(bvh_code_kernel, dim3((unsigned)sort_tiles(n)), dim3(kBvhBlock), 0, st, aabbs, n,
                       items, v.bpart, nparts, v.items, v.hist);
    D3D_CHECK_LAUNCH("bvh_code_kernel");
    if (items == 4) sort_launches<4>(v, n, st);
    else sort_launches<8>(v, n, st);
    D3D_CHECK_LAUNCH("bvh_sort");
    level_launches(v, aabbs, n, v.order, st);
    D3D_CHECK_LAUNCH("bvh_level_kernel");
    return D3D_OK;
}

extern "C" int d3d_bvh_refit(const double *aabbs, int64_t n, void *bvh, int64_t bvh_bytes_avail,
                             void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 1 && n < (int64_t)0x40000000, "n must be in [1, 2^30)");
    D3D_CHECK_ARG(aabbs && bvh, "NULL buffer");
    D3D_CHECK_ARG(bvh_bytes_avail >= bvh_bytes(n), "bvh buffer smaller than d3d_bvh_bytes(n)");
    level_launches(bvh_view(bvh, n), aabbs, n, nullptr, (hipStream_t)stream);
    D3D_CHECK_LAUNCH("bvh_level_kernel");
    return D3D_OK;
}

// Lanes per query: few queries take wide groups (fewer rounds in a row each),
// many fill the chip with narrow ones.  A sorted query of a tree of 1,048,576
// boxes with 8 / 16 / 32 / 64 lanes: 300 queries 34 / 23 / 19 / 17 us, 5,003
// queries 38 / 27 / 21 / 20, 8,192 queries 40 / 29 / 23 / 24, 16,384 queries 55 /
// 39 / 33 / 39, 32,768 queries 65 / 50 / 53 / 71, 49,152 queries 75 / 73 / 73 /
// 98, 65,536 queries 84 / 93 / 97 / 139, 131,072 queries 148 / 155 / 185 / 264
// (the same order on trees of 5,003 and 100,003 boxes).
static int query_lanes(int64_t m) { return m < 8192 ? 64 : m < 49152 ? 32 : 8; }

template <bool kSorted>
static void query_launch(const BvhView &v, int64_t n, const double *aabbs, const double *queries,
                         int64_t m, int32_t *pairs, int64_t cap, unsigned long long *counter,
                         const QueryWs &ws, hipStream_t st) {
    const BvhLevels lv = bvh_levels(n);
    auto go = [&](auto kernel, int lanes) {
        const int per = kBvhBlock / lanes;
        // a launch has less than 2^32 threads; more queries (of an unordered call)
        // take several
        const int64_t slice = query_slice(kBvhBlock, per);
        for (int64_t first = 0; first < m; first += slice) {
            const int64_t k = min(slice, m - first);
            hipLaunchKernelGGL(kernel, dim3((unsigned)((k + per - 1) / per)), dim3(kBvhBlock), 0, st, lv,
                               v.nodes, aabbs, queries, first, m, pairs, cap, counter, ws);
        }
    };
    switch (query_lanes(m)) {
    case 8: go(bvh_query_kernel<8, kSorted>, 8); break;
    case 32: go(bvh_query_kernel<32, kSorted>, 32); break;
    default: go(bvh_query_kernel<64, kSorted>, 64); break;
    }
}

extern "C" int d3d_bvh_query(const void *bvh, int64_t n, const double *aabbs, const double *queries,
                             int64_t m, int32_t *pairs, int64_t cap, uint64_t *n_pairs,
                             void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 1 && n < (int64_t)0x40000000, "n must be in [1, 2^30)");
    D3D_CHECK_ARG(m >= 0 && m < (int64_t)0x7fffffff, "m must fit in int32");
    D3D_CHECK_ARG(bvh && aabbs && n_pairs && (m == 0 || queries), "NULL buffer");
    D3D_CHECK_ARG(cap >= 0 && (cap == 0 || pairs), "pairs buffer is NULL");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(bvh_zero_counter, dim3(1), dim3(1), 0, st, (unsigned long long *)n_pairs);
    D3D_CHECK_LAUNCH("bvh_zero_counter");
    if (m == 0) return D3D_OK;
    query_launch<false>(bvh_view((void *)bvh, n), n, aabbs, queries, m, pairs, cap,
                        (unsigned long long *)n_pairs, QueryWs{}, st);
    D3D_CHECK_LAUNCH("bvh_query_kernel");
    return D3D_OK;
}

// Parts of a sorted query's workspace, for its size and for its pointers.
static int64_t query_layout(int64_t m, int64_t cap, char *base, QueryWs *ws) {
    int64_t b = 0;
    auto part = [&](int64_t bytes) {
        char *p = base ? base + b : nullptr;
        b += align256(bytes);
        return p;
    };
    const int64_t per = m > 0 ? kBvhBlock / query_lanes(m) : 1;
    const int64_t blocks = (m + per - 1) / per;
    QueryWs w;
    w.base = (unsigned long long *)part(blocks * 8);
    w.most = (int32_t *)part(blocks * 4);
    w.count = (int32_t *)part(m * 4);
    w.off = (unsigned long long *)part(m * 8);
    w.rows = (int32_t *)part(m * kHitRows * 4);
    w.ovf = (int32_t *)part(cap * 12);
    w.stage = (int32_t *)part(cap * 4);
    if (ws) *ws = w;
    return b;
}

static int query_write(int64_t m, int32_t *pairs, int64_t room, int64_t cap, const QueryWs &ws,
                       hipStream_t st) {
    const int per = kBvhBlock / query_lanes(m);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((m + per - 1) / per)), dim3(per * kHitRows), 0, st, m,
                           room, cap, ws, pairs);
    };
    if (per == 32) go(query_write_kernel<32>);
    else if (per == 8) go(query_write_kernel<8>);
    else go(query_write_kernel<4>);
    D3D_CHECK_LAUNCH("query_write_kernel");
    return D3D_OK;
}

extern "C" int64_t d3d_bvh_query_sorted_workspace_bytes(int64_t m, int64_t cap) {
    if (m < 0 || cap < 0) return -1;
    return query_layout(m, cap, nullptr, nullptr);
}

extern "C" int d3d_bvh_query_sorted(const void *bvh, int64_t n, const double *aabbs,
                                    const double *queries, int64_t m, int32_t *pairs, int64_t cap,
                                    uint64_t *result, void *workspace, int64_t workspace_bytes,
                                    void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 1 && n < (int64_t)0x40000000, "n must be in [1, 2^30)");
    D3D_CHECK_ARG(m >= 1 && m < (int64_t)0x10000000, "m must be in [1, 2^28)");
    D3D_CHECK_ARG(cap >= 1, "cap must be >= 1");
    D3D_CHECK_ARG(bvh && aabbs && queries && result && workspace, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= query_layout(m, cap, nullptr, nullptr), "workspace too small");
    hipStream_t st = (hipStream_t)stream;
    unsigned long long *res = (unsigned long long *)result;
    QueryWs ws;
    query_layout(m, cap, (char *)workspace, &ws);
    hipLaunchKernelGGL(bvh_zero_counter, dim3(1), dim3(1), 0, st, res + 2);
    D3D_CHECK_LAUNCH("bvh_zero_counter");
    query_launch<true>(bvh_view((void *)bvh, n), n, aabbs, queries, m, nullptr, cap, res + 2, ws, st);
    D3D_CHECK_LAUNCH("bvh_query_kernel");
    const int per = kBvhBlock / query_lanes(m);
    hipLaunchKernelGGL(query_scan_kernel, dim3(1), dim3(1024), 0, st, ws.base, ws.most, (m + per - 1) / per,
                       res);
    D3D_CHECK_LAUNCH("query_scan_kernel");
    return pairs ? query_write(m, pairs, cap, cap, ws, st) : D3D_OK;
}

extern "C" int d3d_bvh_query_sorted_write(int64_t m, int32_t *pairs, int64_t room, int64_t cap,
                                          void *workspace, int64_t workspace_bytes, void *stream) {
    clear_error();
    D3D_CHECK_ARG(m >= 1 && m < (int64_t)0x10000000, "m must be in [1, 2^28)");
    D3D_CHECK_ARG(cap >= 1 && room >= 1, "cap and room must be >= 1");
    D3D_CHECK_ARG(pairs && workspace, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= query_layout(m, cap, nullptr, nullptr), "workspace too small");
    QueryWs ws;
    query_layout(m, cap, (char *)workspace, &ws);
    return query_write(m, pairs, room, cap, ws, (hipStream_t)stream);
}

extern "C" int d3d_bvh_query_sorted_finish(int64_t m, int32_t *pairs, int64_t cap,
                                           const uint64_t *result, void *workspace,
                                           int64_t workspace_bytes, void *stream) {
    clear_error();
    D3D_CHECK_ARG(m >= 1 && m < (int64_t)0x10000000, "m must be in [1, 2^28)");
    D3D_CHECK_ARG(cap >= 1, "cap must be >= 1");
    D3D_CHECK_ARG(pairs && result && workspace, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= query_layout(m, cap, nullptr, nullptr), "workspace too small");
    hipStream_t st = (hipStream_t)stream;
    QueryWs ws;
    query_layout(m, cap, (char *)workspace, &ws);
    hipLaunchKernelGGL(query_spill_kernel, dim3(1024), dim3(kBvhBlock), 0, st,
                       (const unsigned long long *)result + 2, cap, ws);
    D3D_CHECK_LAUNCH("query_spill_kernel");
    const int64_t blocks = (m * kWave + kBvhBlock - 1) / kBvhBlock;
    hipLaunchKernelGGL(query_long_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)),
                       dim3(kBvhBlock), 0, st, m, cap, ws, pairs);
    D3D_CHECK_LAUNCH("query_long_kernel");
    return D3D_OK;
}

extern "C" int64_t d3d_overlap_dense_workspace_bytes(int64_t n) {
    if (n < 0) return -1;
    return (n + 1) * (int64_t)sizeof(unsigned long long);
}

extern "C" int d3d_overlap_dense(const double *a, int64_t n, const double *b, int64_t m,
                                 int32_t *pairs, int64_t cap, uint64_t *n_pairs, void *workspace,
                                 int64_t workspace_bytes, void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 0 && n < (int64_t)0x7fffffff && m >= 0 && m < (int64_t)0x7fffffff,
                  "n and m must fit in int32");
    D3D_CHECK_ARG(n_pairs && (n == 0 || (a && workspace)) && (m == 0 || b), "NULL buffer");
    D3D_CHECK_ARG(cap >= 0 && (cap == 0 || pairs), "pairs buffer is NULL");
    D3D_CHECK_ARG(workspace_bytes >= d3d_overlap_dense_workspace_bytes(n), "workspace too small");
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(bvh_zero_counter, dim3(1), dim3(1), 0, st, (unsigned long long *)n_pairs);
    D3D_CHECK_LAUNCH("bvh_zero_counter");
    if (n == 0 || m == 0) return D3D_OK;
    unsigned long long *counts = (unsigned long long *)workspace;
    const int64_t waves = (n + kDenseRows - 1) / kDenseRows;
    const unsigned blocks = (unsigned)((waves * kWave + kDenseBlock - 1) / kDenseBlock);
    hipLaunchKernelGGL(dense_overlap_kernel<false>, dim3(blocks), dim3(kDenseBlock), 0, st, a, n, b,
                       m, counts, nullptr, pairs, cap);
    D3D_CHECK_LAUNCH("dense_overlap_kernel<count>");
    hipLaunchKernelGGL(dense_scan_kernel, dim3(1), dim3(1024), 0, st, counts, n,
                       (unsigned long long *)n_pairs);
    D3D_CHECK_LAUNCH("dense_scan_kernel");
    if (cap > 0)
        return d3d_overlap_dense_write(a, n, b, m, pairs, cap, n_pairs, workspace, workspace_bytes,
                                       stream);
    return D3D_OK;
}

extern "C" int d3d_overlap_dense_write(const double *a, int64_t n, const double *b, int64_t m,
                                       int32_t *pairs, int64_t cap, const uint64_t *n_pairs,
                                       void *workspace, int64_t workspace_bytes, void *stream) {
    clear_error();
    D3D_CHECK_ARG(n >= 1 && n < (int64_t)0x7fffffff && m >= 1 && m < (int64_t)0x7fffffff,
                  "n and m must be in [1, 2^31)");
    D3D_CHECK_ARG(a && b && n_pairs && workspace && cap >= 1 && pairs, "NULL buffer");
    D3D_CHECK_ARG(workspace_bytes >= d3d_overlap_dense_workspace_bytes(n), "workspace too small");
    const int64_t waves = (n + kDenseRows - 1) / kDenseRows;
    const unsigned blocks = (unsigned)((waves * kWave + kDenseBlock - 1) / kDenseBlock);
    hipLaunchKernelGGL(dense_overlap_kernel<true>, dim3(blocks), dim3(kDenseBlock), 0,
                       (hipStream_t)stream, a, n, b, m, (unsigned long long *)workspace,
                       (const unsigned long long *)n_pairs, pairs, cap);
    D3D_CHECK_LAUNCH("dense_overlap_kernel<write>");
    return D3D_OK;
}
