// d3d_bvh_core.hpp -- shapes of the box trees as plain __host__ __device__
// functions: what the kernels use of the packed 8-wide tree (its levels, their
// launches, a query's stack, the curve its boxes are sorted along), and the
// binary radix hierarchy over sorted keys with its ropes, which no kernel uses.
// Checked on the host by tests/bvh_levels_check.hip and tests/bvh_host_check.hip.
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

// A level launch makes kLevelStep levels above level `base` (and level 0 itself
// for base 0), a block kLevelBlock, 64, 8 and 1 rows of the four: whole groups of
// 8 rows (with their padding) of the last one take a multiple of 8 blocks.
constexpr int kLevelBlock = 512;
constexpr int kLevelStep = 3;

__host__ __device__ inline int64_t level_blocks(const BvhLevels &lv, int base) {
    const int64_t blocks = (round8(lv.count[base]) + kLevelBlock - 1) / kLevelBlock;
    return base + kLevelStep <= lv.top ? round8(blocks) : blocks;
}

// A query's stack of nodes, for groups that take up to W nodes a round.  Popping
// one node of level k at a time never leaves more than 7 k + 1 entries above its
// own place (each of its 8 children is finished before the next is taken), so
// W = 1 needs 7 kBvhMaxLevels + 1 rows.  Wider groups take more than one node
// only while what they could push stays within query_wide(W) rows, and one at a
// time above that.
__host__ __device__ constexpr int query_wide(int W) { return W == 1 ? 0 : 20 * W; }
__host__ __device__ constexpr int query_stack(int W) { return query_wide(W) + 7 * kBvhMaxLevels + 1; }
__host__ __device__ constexpr int query_take(int sp, int W) {
    return sp + 7 * W <= query_wide(W) ? (sp < W ? sp : W) : 1;
}

// Queries of one launch of blocks of `block` threads with `per` queries each,
// whole blocks: fewer than 2^32 threads.
constexpr int64_t query_slice(int block, int per) { return (((int64_t)1 << 32) / block - 1) * per; }

__host__ __device__ inline uint32_t spread10(uint32_t v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Position along a Hilbert curve of 10 bits per axis (J. Skilling, "Programming
// the Hilbert curve", AIP Conf. Proc. 707, 2004: undo the excess rotations from
// the top bit down, Gray-encode, interleave).  Consecutive positions are
// neighbouring cells, so 8 rows in a row make tighter boxes than along a Morton
// curve with its jumps: 65,536 queries of 1,048,576 boxes 130 us in Morton order
// and 84 us in this one, 5,003 queries 24 and 19 us; the build 2 us longer.
__host__ __device__ inline uint32_t hilbert30(uint32_t x, uint32_t y, uint32_t z) {
    auto turn = [&](uint32_t &v, uint32_t q) {
        const uint32_t p = q - 1;
        const uint32_t t = (v & q) ? 0u : (x ^ v) & p;
        x ^= (v & q) ? p : t;
        v ^= t;
    };
#pragma unroll
    for (uint32_t q = 512; q > 1; q >>= 1) {
        x ^= (x & q) ? q - 1 : 0u;
        turn(y, q);
        turn(z, q);
    }
    y ^= x;
    z ^= y;
    uint32_t t = 0;
#pragma unroll
    for (uint32_t q = 512; q > 1; q >>= 1) t ^= (z & q) ? q - 1 : 0u;
    x ^= t;
    y ^= t;
    z ^= t;
    return (spread10(x) << 2) | (spread10(y) << 1) | spread10(z);
}

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
