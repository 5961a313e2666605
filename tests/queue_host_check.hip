// Host-side check of the pair queue's claims (d3d_queue.hpp), run on the CPU by
// tests/test_queue_modes_host.py: for classes up to the largest, every chunk is
// positive, the chunks cover the class, and no position a wavefront can claim
// past the end leaves the 32 bits it is held in; and a caller's blocks per
// compute unit are taken as given at every batch size.
#include <cstdio>

#include "d3d_queue.hpp"

using namespace d3d;

int main() {
    int bad = 0;
    const int64_t most = 0x7ffffffe;
    for (int64_t count : {(int64_t)1, (int64_t)63, (int64_t)4097, (int64_t)1 << 20, (int64_t)1 << 30,
                          most - (1 << 21), most - 3072, most - 1, most})
        for (int n_waves : {4, 1024, 2048, 3072, 3648})
            for (int full : {1, 2, 64, 128, 512}) {
                const int chunk = claim_chunk((int)count, n_waves, full);
                const int64_t chunks = chunks_of((int)count, chunk);
                // the last claims: one more chunk per wavefront past the end, and the
                // items a wavefront adds to its claim
                const int64_t last = count + (int64_t)(n_waves + 1) * chunk + 64;
                if (chunk < 1 || chunk > full || chunks * chunk < count || (chunks - 1) * chunk >= count ||
                    last > 0xffffffffll) {
                    std::printf("FAIL count %lld, %d wavefronts, full %d: chunk %d\n", (long long)count,
                                n_waves, full, chunk);
                    ++bad;
                }
            }
    for (int64_t n : {(int64_t)1, (int64_t)4096, (int64_t)4097, (int64_t)1 << 20})
        for (int asked : {0, 1, 2, 3}) {
            const int blocks = batch_blocks(n, 4096, asked);
            // the occupancy-2 kernel holds two blocks per compute unit
            if ((asked > 0 && blocks != asked) || blocks < 1 || blocks > 3 ||
                (batch_is_loose(n, 4096, asked) && (blocks > 2 || n > 4096))) {
                std::printf("FAIL %lld pairs, %d blocks asked: %d\n", (long long)n, asked, blocks);
                ++bad;
            }
        }
    std::printf(bad ? "FAILED %d\n" : "OK\n", bad);
    return bad ? 1 : 0;
}
