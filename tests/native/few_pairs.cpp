// Which thread of a few-token product converts which tokens (csrc/few_pairs.h), for each instance: every pair of every tile of a chunk
// is taken, none outside it, and one that is taken twice is taken by threads that hold the same bytes.
#include <cstdio>
#include <vector>

#include "few_pairs.h"

int main() {
    int instances = 0;
    for (bool mins : {true, false})
        for (uint32_t t = 1; t <= 3; ++t, ++instances) {
            const uint32_t tiles = few_chunk(mins, t) * t;
            std::vector<int> taken(tiles * FEW_TILE_PAIRS);
            for (uint32_t i = 0; i < few_rounds(tiles); ++i)
                for (uint32_t thread = 0; thread < FEW_WAVES * 64; ++thread) {
                    const uint32_t tile = few_tile(tiles, i, thread / 64);
                    if (tile >= tiles) {
                        std::printf("mins %d, %u tiles of tokens: pair %u of thread %u is in tile %u of %u\n", mins, t, i, thread, tile, tiles);
                        return 1;
                    }
                    ++taken[tile * FEW_TILE_PAIRS + thread % FEW_TILE_PAIRS];
                }
            for (uint32_t p = 0; p < taken.size(); ++p)
                if (!taken[p]) {
                    std::printf("mins %d, %u tiles of tokens: nobody takes pair %u\n", mins, t, p);
                    return 1;
                }
        }
    std::printf("%d instances\n", instances);
}
