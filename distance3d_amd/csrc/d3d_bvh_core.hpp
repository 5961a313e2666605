// d3d_bvh_core.hpp -- shapes of the box trees as plain __host__ __device__
// functions: the levels of the packed 8-wide tree the kernels use, and the
// binary radix hierarchy over sorted keys with its ropes, which the host-side
// structural check (tests/bvh_host_check.hip) covers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace d3d {

// Packed tree over n sorted boxes: level 0 has n rows, level k + 1 one row per
// 8 rows of level k, the top level at most 8.  Every level starts at a multiple
// of 8 rows (nodes: rows in all).  An entry of a query's stack is
// level << kNodeBits | index of the group of 8 rows: n < 2^30 leaves 27 bits
// for the group and 10 levels.
constexpr int kBvhMaxLevels = 10;
constexpr int kNodeBits = 27;

struct BvhLevels {
    int64_t count[kBvhMaxLevels], off[kBvhMaxLevels];
    int64_t nodes;
    int top;
};

__host__ __device__ inline int64_t round8(int64_t n) { return (n + 7) / 8 * 8; }

__host__ __device__ inline BvhLevels bvh_levels(int64_t n) {
    BvhLevels lv;
    lv.nodes = 0;
    lv.top = -1;
    for (int k = 0; k < kBvhMaxLevels; ++k) {
        const bool more = k == 0 || lv.count[k - 1] > 8;
        lv.count[k] = !more ? 0 : k == 0 ? n : (lv.count[k - 1] + 7) / 8;
        lv.off[k] = lv.nodes;
        lv.nodes += round8(lv.count[k]);
        if (more) lv.top = k;
    }
    return lv;
}

// Queries of one launch of blocks of `block` threads with `per` queries each,
// whole blocks: fewer than 2^32 threads.
constexpr int64_t query_slice(int block, int per) { return (((int64_t)1 << 32) / block - 1) * per; }

__host__ __device__ inline int clz32(uint32_t v) { return v ? __builtin_clz(v) : 32; }

// Length of the common prefix of sorted keys i and j; equal keys compare
// their positions so every pair of leaves differs (Karras 2012, section 4).
__host__ __device__ inline int delta(const uint32_t *k, int64_t n, int i, int j) {
    if (j < 0 || (int64_t)j >= n) return -1;
    const uint32_t a = k[i], b = k[j];
    if (a == b) return 32 + clz32((uint32_t)(i ^ j));
    return clz32(a ^ b);
}

// Children of internal node i (0 <= i < n-1) over n sorted keys.  Internal
// nodes are 0..n-2, leaves are n-1 .. 2n-2 (leaf of sorted position p is
// n-1+p).  Internal node i covers the sorted range between i and j and splits
// it at the highest bit in which its keys differ.
__host__ __device__ inline void karras_children(const uint32_t *keys, int64_t n, int i, int *left,
                                                int *right) {
    const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + (d < 0 ? -1 : 0);
    const int lo = i < j ? i : j, hi = i < j ? j : i;
    const int leaf0 = (int)(n - 1);
    *left = (lo == gamma) ? leaf0 + gamma : gamma;
    *right = (hi == gamma + 1) ? leaf0 + gamma + 1 : gamma + 1;
}

// Rope of node k: the node a depth-first walk visits after k's subtree (the
// right sibling of the nearest ancestor-or-self that is a left child), -1
// after the last subtree.  The walk is capped at n steps so a malformed tree
// cannot loop.
__host__ __device__ inline int rope_of(int k, int64_t n, const int32_t *parent, const int32_t *left,
                                       const int32_t *right) {
    int cur = k;
    for (int64_t steps = 0; cur != 0 && steps < n; ++steps) {
        const int p = parent[cur];
        if (p < 0) return -1;
        if (left[p] == cur) return right[p];
        cur = p;
    }
    return -1;
}

}  // namespace d3d
