// Which of a chunk's tokens a thread of the few-token products (gemm_few.hip) converts.  Plain arithmetic, without the device's headers.
#pragma once
#include <cstdint>

constexpr uint32_t FEW_WAVES = 8, FEW_TILE_PAIRS = 128;   // pairs (token, block of 32 quants) of 16 tokens and a super-block
// Super-blocks of a chunk, for `t` tiles of 16 tokens: up to four tiles, and two chunks fill at most half the LDS (Q6_K, which has no
// mins, with one tile two: 32000 x 4096 with 5 tokens 33.3 us by four, 32.0 by two, 4096 x 14336 in eight slices 17.6 and 16.8).
constexpr uint32_t few_chunk(bool mins, uint32_t t) { return t == 1 ? (mins ? 4 : 2) : t == 2 ? 2 : 1; }
// A chunk of `tiles` tiles: how many pairs a thread takes, and the tile of its i-th, of which it takes the pair of its index modulo
// FEW_TILE_PAIRS.  Wavefronts beyond the last tile take that one again: the same bytes to the same place.
constexpr uint32_t few_rounds(uint32_t tiles) { return (tiles * FEW_TILE_PAIRS + FEW_WAVES * 64 - 1) / (FEW_WAVES * 64); }
constexpr uint32_t few_tile(uint32_t tiles, uint32_t i, uint32_t wave) {
    const uint32_t t = (i * FEW_WAVES + wave) * 64 / FEW_TILE_PAIRS;
    return t < tiles ? t : tiles - 1;
}
