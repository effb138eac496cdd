// Products of Q6_K matrices with many tokens (gemm_kq.hip): the tokens' operand and the launcher.
#pragma once
#include "host_common.h"

// The tokens' operand: one record per 16 tokens and super-block of 256, per block 64 lanes x 16 bytes of f16 quants; as many bytes
// as the row-major form where the tokens are a multiple of 16.  Tokens up to a whole tile repeat the last.
constexpr uint32_t KQ_HALF = 4 * 1024, KQ_REC = 2 * KQ_HALF, KQ_TOKENS = 128, KQ_ROWS = 256;
static inline uint32_t kq_act_records(uint32_t n, uint32_t k) { return (n + 15) / 16 * (k / 256); }
static inline uint64_t kq_act_bytes(uint64_t n, uint64_t k) { return (n + 15) / 16 * (k / 256) * KQ_REC; }

// Of the eight dwords of a block's 32 quants, lane group g holds this one and the next: groups with an even number the first
// sixteen quants, with an odd one the others.
__device__ __forceinline__ constexpr uint32_t kq_dword(uint32_t g) { return 4 * (g & 1) + 2 * (g >> 1); }
// One workgroup of 256 per record: a thread takes 8 of the 16 x 128 quants of each half.
__device__ __forceinline__ void kq_act_record(uint32_t index, const int8_t* __restrict__ bq, uint8_t* __restrict__ act, uint32_t n, uint32_t k) {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    const uint32_t nsb = k / 256, tile = index / nsb, sb = index - tile * nsb;
    uint8_t* const rec = act + static_cast<uint64_t>(index) * KQ_REC;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tok = min(tile * 16 + (lane & 15), n - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint2 q = *reinterpret_cast<const uint2*>(bq + static_cast<uint64_t>(tok) * k + sb * 256 + (h * 4 + wave) * 32 + kq_dword(lane >> 4) * 4);
        // bytes 0 and 2, then 1 and 3, as the mantissa of 1024 + 128 + quant, less that: exact
        const v2 off = {static_cast<_Float16>(-1152.f), static_cast<_Float16>(-1152.f)};
        const uint32_t a = q.x ^ 0x80808080u, b = q.y ^ 0x80808080u, w[4] = {a & 0x00FF00FFu, (a >> 8) & 0x00FF00FFu, b & 0x00FF00FFu, (b >> 8) & 0x00FF00FFu};
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2, w[i] | 0x64006400u) + off);
        *reinterpret_cast<uint4*>(rec + h * KQ_HALF + wave * 1024 + lane * 16) = make_uint4(o[0], o[1], o[2], o[3]);
    }
}

// K slices of the product of m (and m2) rows with n tokens on this kernel, or 0 where the one for fewer tokens is the better.
// A CU holds one workgroup: K is cut into as many slices as leave no second round (a slice is at least one super-block, at
// most sixteen slices).  Where that leaves half of the chip idle with slices of a few super-blocks only, the 64-token tiles
// of the other kernel are faster: 24.1 against 27.6 us for 1024 x 4096 with 160 tokens (128 workgroups of one super-block),
// but 54.7 against 48.0 us for 1024 x 14336 with 128 (56 of four), 34.6 against 29.3 us for 1024 x 4096 with 512 (256 of
// one), 64.9 against 52.6 us for 2048 x 14336 with 160, 26.3 against 22.9 us for 512 x 4096 with 128.
static inline uint32_t kq_slices(uint32_t dtype, uint64_t m, uint64_t m2, uint32_t n, uint64_t k, uint32_t n_cu) {
    if (dtype != CERA_HIP_Q6_K || n <= 64) return 0;
    const uint64_t tiles = (n + KQ_TOKENS - 1) / KQ_TOKENS * ((m + KQ_ROWS - 1) / KQ_ROWS + (m2 + KQ_ROWS - 1) / KQ_ROWS);
    const uint32_t nsb = static_cast<uint32_t>(k / 256);
    uint32_t split = 1;
    for (uint32_t d = 2; d <= 16; ++d)
        if (nsb % d == 0 && tiles * d <= n_cu) split = d;
    return tiles * split * 2 > n_cu || nsb / split >= 4 ? split : 0;
}

struct KqArgs {
    const uint8_t *w, *w2;   // native blocks; w2 (nullable): a second matrix of the same type and k
    const uint8_t* act;      // records
    const float* bs;         // [n][k / 32] the tokens' block scales
    float *out, *out2;
    uint32_t m, m2, n, k, row_bytes, tiles1, k_chunk;   // tiles1: row tiles of the first matrix
    uint64_t ld_m, ld_n, ld_n2;                         // out[i * ld_m + j * ld_n], out2[i * ld_m + j * ld_n2]
    uint64_t part_stride;                               // floats from one slice's sums to the next one's
    const float* resid;                                 // nullable, not with more than one slice
    float resid_scale;
};

cera_hip_status cera_launch_kq_act(cera_hip_ctx* ctx, const int8_t* bq, uint32_t n, uint32_t k, void* act);
// grid (token tiles, row tiles, slices of k_chunk)
cera_hip_status cera_launch_kq(cera_hip_ctx* ctx, const KqArgs& a, uint32_t split);
