// Host-side check of the packed tree's shape (d3d_bvh_core.hpp), run on the CPU
// by tests/test_bvh_levels_host.py: the levels of a tree, the rows its level
// launches write, the rows a query can read, the depth of a query's stack, the
// queries of a launch, and the curve the boxes are sorted along.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <utility>
#include <vector>

#include "d3d_bvh_core.hpp"

using namespace d3d;

static int bad = 0;
#define CHECK(cond, ...)                                          \
    do {                                                          \
        if (!(cond)) {                                            \
            if (bad++ < 20) std::printf("FAIL %s: ", #cond), std::printf(__VA_ARGS__), std::printf("\n"); \
        }                                                         \
    } while (0)

static void check_levels(int64_t n) {
    const long long N = n;
    const BvhLevels lv = bvh_levels(n);
    CHECK(lv.top >= 0 && lv.top < kBvhMaxLevels && lv.count[0] == n && lv.count[lv.top] <= 8, "n %lld", N);
    int64_t at = 0;
    for (int k = 0; k <= lv.top; ++k) {
        CHECK(lv.off[k] == at && at % 8 == 0, "n %lld level %d", N, k);
        at += round8(lv.count[k]);
        // 8 children per row, all within the padded level below; a stack entry's
        // group index and level fit their bits
        if (k > 0) {
            CHECK(8 * lv.count[k] == round8(lv.count[k - 1]), "n %lld level %d", N, k);
            CHECK(lv.count[k] <= (int64_t)1 << kNodeBits, "n %lld level %d", N, k);
        }
    }
    CHECK(at == lv.nodes && ((int64_t)lv.top << kNodeBits) + ((int64_t)1 << kNodeBits) <= 0x80000000ll, "n %lld", N);
    // every level is written by one launch, with all its padding
    std::vector<int> written(kBvhMaxLevels, 0);
    for (int base = 0; base == 0 || base < lv.top; base += kLevelStep) {
        const int64_t blocks = level_blocks(lv, base);
        CHECK(blocks >= 1 && blocks * kLevelBlock < (int64_t)1 << 32, "n %lld base %d", N, base);
        for (int k = base == 0 ? 0 : base + 1; k <= std::min(base + kLevelStep, lv.top); ++k) {
            ++written[k];
            CHECK(blocks * (kLevelBlock >> (3 * (k - base))) >= round8(lv.count[k]), "n %lld level %d", N, k);
        }
    }
    for (int k = 0; k <= lv.top; ++k) CHECK(written[k] == 1, "n %lld level %d", N, k);
}

// A query's walk as the kernel makes it, over a tree whose rows overlap it at
// random; the deepest stack.
static int walk(const BvhLevels &lv, int W, double chance, std::mt19937 &rng, int64_t rounds) {
    std::uniform_real_distribution<double> u(0.0, 1.0);
    std::vector<std::pair<int, int64_t>> st{{lv.top, 0}};
    int deepest = 1;
    for (; !st.empty() && rounds > 0; --rounds) {
        const int take = query_take((int)st.size(), W);
        CHECK(take >= 1 && take <= W && take <= (int)st.size(), "take %d of %d", take, (int)st.size());
        std::vector<std::pair<int, int64_t>> now(st.rbegin(), st.rbegin() + take);
        st.resize(st.size() - take);
        for (const auto &e : now)
            for (int c = 0; c < 8; ++c) {
                const int64_t rec = 8 * e.second + c;
                CHECK(lv.off[e.first] + rec < lv.nodes, "level %d", e.first);
                if (rec < lv.count[e.first] && e.first > 0 && u(rng) < chance) st.push_back({e.first - 1, rec});
            }
        deepest = std::max(deepest, (int)st.size());
    }
    return deepest;
}

int main() {
    std::mt19937 rng(3);
    for (int64_t n = 1; n <= 5000; ++n) check_levels(n);
    for (int64_t p = 8; p < (int64_t)1 << 30; p *= 8)
        for (int64_t f = 1; f <= 8; ++f)
            for (int64_t d = -70; d <= 70; ++d)
                if (p * f + d >= 1 && p * f + d < (int64_t)1 << 30) check_levels(p * f + d);
    for (int k = 0; k < 200000; ++k) check_levels(1 + (int64_t)(rng() & 0x3ffffffeu));
    check_levels(((int64_t)1 << 30) - 1);

    for (int64_t n : {9ll, 513ll, 4097ll, 32769ll, 262145ll, 1000003ll, (1ll << 30) - 1}) {
        const BvhLevels lv = bvh_levels(n);
        for (int W : {1, 4, 8})
            for (double chance : {1.0, 0.9, 0.5, 0.2}) {
                const int deepest = walk(lv, W, chance, rng, 300000);
                CHECK(deepest <= query_stack(W), "n %lld W %d: %d", (long long)n, W, deepest);
            }
    }
    for (int per : {4, 8, 32})
        CHECK(query_slice(256, per) % per == 0 && query_slice(256, per) / per * 256 < (int64_t)1 << 32, "per %d", per);

    // cells of an aligned block of the curve: a run of positions without gaps, each
    // next to the one before
    for (uint32_t origin : {0u, 1u, 5u, 17u, 31u}) {
        const uint32_t x0 = 32 * origin, y0 = 32 * ((7 * origin) & 31), z0 = 32 * ((13 * origin + 3) & 31);
        std::vector<std::pair<uint32_t, uint32_t>> cells;
        for (uint32_t c = 0; c < 32768; ++c)
            cells.push_back({hilbert30(x0 + (c & 31), y0 + ((c >> 5) & 31), z0 + (c >> 10)), c});
        std::sort(cells.begin(), cells.end());
        CHECK(cells[0].first % 32768 == 0, "origin %u", origin);
        for (size_t k = 1; k < cells.size(); ++k) {
            const int a = (int)cells[k - 1].second, b = (int)cells[k].second;
            const int step = std::abs((a & 31) - (b & 31)) + std::abs(((a >> 5) & 31) - ((b >> 5) & 31)) +
                             std::abs((a >> 10) - (b >> 10));
            CHECK(cells[k].first == cells[k - 1].first + 1 && step == 1, "origin %u position %d", origin, (int)k);
        }
    }
    // and the blocks themselves along the whole curve, by their first positions
    std::vector<std::pair<uint32_t, uint32_t>> blocks;
    for (uint32_t c = 0; c < 32768; ++c)
        blocks.push_back({hilbert30(32 * (c & 31), 32 * ((c >> 5) & 31), 32 * (c >> 10)) >> 15, c});
    std::sort(blocks.begin(), blocks.end());
    for (size_t k = 0; k < blocks.size(); ++k) CHECK(blocks[k].first == k, "block %d", (int)k);

    std::printf(bad ? "FAILED %d\n" : "OK\n", bad);
    return bad ? 1 : 0;
}
