// Launcher of the products of K-quant matrices with a few tokens (gemm_few.hip).
#pragma once
#include "host_common.h"

constexpr uint32_t FEW_MAX_TOKENS = 48, FEW_MIN_K = 2048;

// One matrix as the kernel sees it: its rows in up to three segments, each with an output [n][ld] of its own.
struct FewMat {
    const uint8_t* w = nullptr;
    uint32_t m = 0, row_bytes = 0;
    uint32_t cut[2] = {}, ld[3] = {};
    float* out[3] = {};
};
// One matrix as a caller names it: rows [0, len[0]) go to out[0] [n][len[0]], the next len[1] to out[1], the rest to out[2]
// (len 0: all that is left).  The lengths are multiples of four.
struct FewOut {
    const cera_hip_dtensor* w = nullptr;
    uint32_t len[2] = {};
    float* out[3] = {};
};
// What a split K left: n_split slices `stride` floats apart, in each of them the outputs of all segments of both matrices
// one behind the other.  n_split = 1: the outputs are complete.
struct FewParts {
    float* part = nullptr;
    uint32_t n_split = 1;
    uint64_t stride = 0;
};

// whether a matrix takes the kernel for n tokens: Q4_K or Q6_K, rows and k in whole fours and super-blocks, and
// rows long enough (FEW_MIN_K) for a wavefront's loads to run ahead
bool cera_gemm_few_supports(const cera_hip_dtensor* w, uint32_t n);
// y[t][row] = W . x_t (+ resid, of oa's first segment and unless K is split) for n tokens quantized to xs / xq / bsum; ob
// (nullable): a second matrix of the same k in the same launch, of the same type or Q6_K beside Q4_K.
cera_hip_status cera_launch_gemm_few(cera_hip_ctx* ctx, const FewOut& oa, const FewOut* ob, const float* xs, const int8_t* xq, const float* bsum, uint32_t n,
                                     const float* resid, float resid_scale, int part_slot, FewParts* parts);
// hq / hs / hbsum [n][m] = Q8_0(silu(gate . x) * (up . x)) in one launch.  *fused = false (nothing launched) where the two are not of one type and
// shape in whole blocks of rows, or where a pair with K in slices is faster.
cera_hip_status cera_launch_gemm_few_swiglu(cera_hip_ctx* ctx, const cera_hip_dtensor* gate, const cera_hip_dtensor* up, const float* xs, const int8_t* xq, const float* bsum,
                                            uint32_t n, int8_t* hq, float* hs, float* hbsum, bool* fused);
