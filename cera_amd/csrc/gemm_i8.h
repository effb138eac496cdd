// Products of Q8_0 and Q4_0 matrices with tokens (gemm_i8.hip).
#pragma once
#include "host_common.h"

constexpr uint32_t I8_ROWS = 128;
static inline uint32_t i8_tokens(uint32_t n) { return n <= 64 ? 64 : 128; }   // of a workgroup

struct I8Args {
    const uint8_t *w, *w2;   // native blocks; w2 (nullable): a second matrix of the same type and k, or the up matrix
    const int8_t* xq;        // [n][k] the tokens' quants
    const float* xs;         // [n][k / 32] their block scales
    float *out, *out2;
    uint32_t m, m2, n, k, row_bytes, tiles1, k_chunk;   // tiles1: row tiles of the first matrix
    uint64_t ld_m, ld_n, ld_n2;                         // out[i * ld_m + j * ld_n], out2[i * ld_m + j * ld_n2]
    uint64_t part_stride;                               // floats from one slice's sums to the next one's
    const float* resid;                                 // nullable, not with more than one slice
    float resid_scale;
    // silu(gate) * up, quantized: [n][m], [n][m / 32], [n][m / 32] scale times sum of the quants
    int8_t* hq;
    float *hs, *hbsum;
};

// What the kernel takes: rows that 128 of a lane's 32-bit offsets reach, in whole 16-byte pieces at a base aligned to them (as every
// matrix here has them).
static inline bool i8_takes(const cera_hip_dtensor* w, const int8_t* xq) {
    return (w->dtype == CERA_HIP_Q8_0 || w->dtype == CERA_HIP_Q4_0) && w->k % 256 == 0 && w->row_bytes % 16 == 0 && w->row_bytes < (1u << 24) &&
           w->k < (1u << 24) && ((reinterpret_cast<uintptr_t>(w->dev) | reinterpret_cast<uintptr_t>(xq)) & 15) == 0;
}
// Slices of K: a CU holds two workgroups; K is cut into as many slices of at least two super-blocks as leave no second round.
static inline uint32_t i8_slices(uint64_t m, uint64_t m2, uint32_t n, uint64_t k, uint32_t n_cu) {
    const uint64_t tiles = (n + i8_tokens(n) - 1) / i8_tokens(n) * ((m + I8_ROWS - 1) / I8_ROWS + (m2 + I8_ROWS - 1) / I8_ROWS);
    const uint32_t nsb = static_cast<uint32_t>(k / 256);
    uint32_t split = 1;
    for (uint32_t d = 2; d <= 8; ++d)
        if (nsb % d == 0 && nsb / d >= 2 && tiles * d <= 2 * n_cu) split = d;
    return split;
}

// grid (token tiles, row tiles, slices of k_chunk)
cera_hip_status cera_launch_i8(cera_hip_ctx* ctx, uint32_t dtype, const I8Args& a, uint32_t split);
// w gate, w2 up: the quantized product of silu(gate) and up
cera_hip_status cera_launch_i8_swiglu(cera_hip_ctx* ctx, uint32_t dtype, const I8Args& a);
