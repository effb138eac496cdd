// Products of Q8_0 and Q4_0 matrices with a batch of tokens on the int8 matrix cores: exact integer dots of 32-weight blocks,
// each folded into the f32 sums with its weight's and its token's scale, in the order of the blocks.
//
// 128 rows x 128 tokens (64 for up to 64 tokens), four wavefronts of 32 rows each over all tokens, two workgroups a CU.  A
// wavefront's rows come by direct loads into LDS of its own, whole 16-byte pieces of a row side by side, half a super-block
// ahead; the tokens, 64 of k at a time, straight from their quants, row by row, with one barrier.  Nothing is staged through
// registers and a Q8_0 code needs no unpacking.  The sums start from 1.5 * 2^23 as an integer, so that the matrix core's result,
// read as a float, is that number plus the dot: a subtraction in place of the conversion, which the vector ALU issues at half
// the rate.  The product of the two scales, f16 numbers both, is an outer product on the matrix core, two blocks an instruction, exact in
// f32.  It is an f16 instruction with one of its four products in use: while one of f32 runs, no vector instruction of the SIMD does
// (32 vector instructions of another wavefront beside them: 201 clocks with f32, 138 with f16, 134 alone).  Q8_0, hidden 3072, two layers: 300 tokens 524 -> 510 us, 1001
// 992 -> 968, 2000 1714 -> 1676.  A slice of K adds its
// blocks in the order of the kernel before it; the number of slices is i8_slices' own, so that sums in parts have another order.
//
// What bounds it: one subtraction and one FMA per output and block.  In 16384 x 3072 Q8_0 (gate | up) times 1001 tokens the vector
// ALU is busy for 0.76 of the time and the matrix cores for 0.30; 28672 x 4096 times 2048 tokens with SwiGLU 655 us, 734 TOP/s.  The kernel
// before it (gemm.hip.h, which keeps Q4_1, rows of about 2^24 columns and more, the block dots and the code object's export)
// unpacks into LDS, converts, and reads both operands through LDS.  Passes of two layers, before and now:
//   hidden 3072, Q8_0:  9 tokens 263 -> 234 us, 64: 341 -> 294, 128: 453 -> 376, 512: 838 -> 605, 1001: 1320 -> 1039 (986 with the folds in order, 968 with the scales in f16)
//   hidden 4096, Q4_0:  9 tokens 331 -> 300 us, 64: 440 -> 374, 128: 591 -> 477, 512: 1181 -> 947, 1001: 2055 -> 1673
#include "f16_codes.hip.h"
#include "gemm_i8.h"
#include "lds_dma.hip.h"
#include "quantize.hip.h"

namespace {

typedef float f16x __attribute__((ext_vector_type(16)));
typedef float f32x __attribute__((ext_vector_type(32)));
typedef int i16x __attribute__((ext_vector_type(16)));
typedef _Float16 h4x __attribute__((ext_vector_type(4)));
typedef int i4x __attribute__((ext_vector_type(4)));

constexpr int I8_WAVES = 4;

// A half super-block of a row is four blocks; SB its super-block's bytes.  It is brought in as PIECES of 16 bytes, the second
// half from the piece that it begins in the middle of.  Blocks with an even number begin two bytes behind a multiple of four.
__device__ __forceinline__ i4x dwords(const uint8_t* row, uint32_t at, bool odd_block) {
    const uint32_t* const p = reinterpret_cast<const uint32_t*>(row + at);
    if (odd_block) return i4x{static_cast<int>(p[0]), static_cast<int>(p[1]), static_cast<int>(p[2]), static_cast<int>(p[3])};
    const uint32_t a = p[0], b = p[1], c = p[2], d = p[3], e = p[4];
    return i4x{static_cast<int>(__builtin_amdgcn_alignbit(b, a, 16)), static_cast<int>(__builtin_amdgcn_alignbit(c, b, 16)),
               static_cast<int>(__builtin_amdgcn_alignbit(d, c, 16)), static_cast<int>(__builtin_amdgcn_alignbit(e, d, 16))};
}
struct I8Q8_0 {
    static constexpr uint32_t SB = 272, PIECES = 9, START = 8;   // START: where the second half begins in its first piece
    // sixteen codes of block z, the first ones in the lower half of the lanes
    static __device__ __forceinline__ i4x codes(const uint8_t* row, uint32_t z, uint32_t half) {
        return dwords(row, ((34 * z + 2) & ~3u) + 16 * half, z & 1);
    }
    static __device__ __forceinline__ _Float16 scale(const uint8_t* row, uint32_t z) { return *reinterpret_cast<const _Float16*>(row + 34 * z); }
    static __device__ __forceinline__ float dot(float f, float start) { return f - start; }
};
struct I8Q4_0 {
    static constexpr uint32_t SB = 144, PIECES = 5, START = 8;
    // a nibble less 8 is, with its highest bit turned, its own two's complement: in a byte's upper half it is sixteen times it
    static __device__ __forceinline__ i4x codes(const uint8_t* row, uint32_t z, uint32_t half) {
        i4x q = dwords(row, (18 * z + 2) & ~3u, z & 1);
        const uint32_t up = half ? 0 : 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = static_cast<int>(((static_cast<uint32_t>(q[i]) ^ 0x88888888u) << up) & 0xF0F0F0F0u);
        return q;
    }
    static __device__ __forceinline__ _Float16 scale(const uint8_t* row, uint32_t z) { return *reinterpret_cast<const _Float16*>(row + 18 * z); }
    static __device__ __forceinline__ float dot(float f, float start) { return fmaf(f, 0.0625f, -0.0625f * start); }   // the codes are sixteen times theirs; exact
};

// T: tiles of 32 tokens (4; 2 for up to 64).  SWIGLU: a wavefront's rows are sixteen of the gate matrix and the same sixteen of the up matrix
template <typename W, bool SWIGLU, int T>
__global__ __launch_bounds__(64 * I8_WAVES, 2) void gemm_i8_kernel(I8Args p) {
    constexpr int LOADS = (16 * W::PIECES + 63) / 64, TOKENS = T * 32;
    constexpr uint32_t HALF16 = LOADS * 1024, BUF = 2 * HALF16, STRIDE = W::PIECES * 16;   // sixteen rows of a half super-block; both
    __shared__ __align__(16) uint8_t act[2][T * 2048];   // [token][64 bytes], its pieces turned round by the token
    __shared__ __align__(16) uint8_t acs[2][T * 256];    // [tile][block][token]
    __shared__ __align__(16) uint8_t wts[I8_WAVES][2][BUF];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), col = lane & 31, half = lane >> 5;
    const bool second = !SWIGLU && p.w2 != nullptr && blockIdx.y >= p.tiles1;
    const uint32_t rows = second ? p.m2 : p.m, m0 = SWIGLU ? blockIdx.y * (I8_ROWS / 2) : (second ? blockIdx.y - p.tiles1 : blockIdx.y) * I8_ROWS;
    const uint32_t n0 = blockIdx.x * TOKENS, sb0 = blockIdx.z * (p.k_chunk / 256), sb1 = sb0 + p.k_chunk / 256;
    // the weights' sixteen rows s: lane's share of its loads, from row m0 (rows past the end are the last one again)
    const uint8_t* const base0 = (second ? p.w2 : p.w) + static_cast<uint64_t>(m0) * p.row_bytes;
    const uint8_t* const base1 = SWIGLU ? p.w2 + static_cast<uint64_t>(m0) * p.row_bytes : base0;
    uint32_t woff[2][LOADS];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < LOADS; ++j) {
            const uint32_t q = min(64u * j + lane, 16 * W::PIECES - 1), r = q / W::PIECES, part = q - r * W::PIECES;
            const uint32_t row = SWIGLU ? m0 + wave * 16 + r : m0 + wave * 32 + s * 16 + r;
            woff[s][j] = (min(row, rows - 1) - m0) * p.row_bytes + part * 16;
        }
    const uint32_t wts_lds = lds_addr(&wts[0][0][0]) + wave * 2 * BUF;
    const uint8_t* const my_row = &wts[0][0][0] + wave * 2 * BUF + (col >> 4) * HALF16 + (col & 15) * STRIDE;
    // the tokens: a wavefront brings in a quarter of them (those past the end are the last one again: their products are not stored)
    const uint32_t last = p.n - 1 - n0;
    const int8_t* const xq = p.xq + static_cast<uint64_t>(n0) * p.k;
    const float* const xs = p.xs + static_cast<uint64_t>(n0) * (p.k / 32);
    uint32_t xoff[T / 2];
#pragma unroll
    for (int j = 0; j < T / 2; ++j) {
        const uint32_t t = wave * (T * 8) + j * 16 + (lane >> 2);
        xoff[j] = min(t, last) * p.k + ((lane & 3) ^ ((t >> 2) & 3)) * 16;
    }
    // their scales by tiles (of two tiles, two wavefronts bring in the same)
    const uint32_t xs_off = (min(wave % T * 32 + col, last) * (p.k / 32) + half) * 4;
    const uint32_t act_lds = lds_addr(&act[0][0]) + wave * (T * 512), acs_lds = lds_addr(&acs[0][0]) + wave % T * 256;
    auto tokens = [&](uint32_t part, uint32_t buf) {
#pragma unroll
        for (int j = 0; j < T / 2; ++j) lds_dma_1k(xq + part * 64, xoff[j], act_lds + buf * (T * 2048) + j * 1024);
        lds_dma_256(xs + part * 2, xs_off, acs_lds + buf * (T * 256));
    };
    auto weights = [&](uint32_t h, uint32_t to, int s) {   // half super-block h
        const uint8_t* const b = (s ? base1 : base0) + (h >> 1) * W::SB + (h & 1) * (W::SB / 2 - W::START);
#pragma unroll
        for (int j = 0; j < LOADS; ++j) lds_dma_1k(b, woff[s][j], wts_lds + to * BUF + s * HALF16 + j * 1024);
    };
    float acc[T][16];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
    i16x start;
#pragma unroll
    for (int e = 0; e < 16; ++e) start[e] = 0x4B400000;
    float start_f = 12582912.0f;
    asm volatile("" : "+v"(start), "+v"(start_f));   // in registers, once
    f32x zero;
#pragma unroll
    for (int e = 0; e < 32; ++e) zero[e] = 0.0f;
    weights(2 * sb0, 0, 0);
    weights(2 * sb0, 0, 1);
    tokens(4 * sb0, 0);
    uint32_t buf = 0;
    auto part = [&](uint32_t sb, auto q_) {   // a quarter of a super-block: two blocks
        constexpr uint32_t q = decltype(q_)::value, odd = q >> 1, z = 2 * (q & 1);
        // this part's tokens and rows are in, and no wavefront reads the other buffers any more
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        // into the buffers that nobody reads now.  Behind the last ones these are the last ones once more: no branch
        const uint32_t next = min(sb * 4 + q + 1, sb1 * 4 - 1), next_half = min(sb * 2 + odd + 1, sb1 * 2 - 1);
        const uint8_t *const xl = act[buf] + col * 64, *const sl = acs[buf] + lane * 4, *const wr = my_row + odd * (BUF + W::START);
        i4x a[2], x[2][2];
        float ts[2];
        auto read = [&](int t) {   // a tile's two fragments; lanes of the upper half the second block's scales
#pragma unroll
            for (int b = 0; b < 2; ++b) x[t & 1][b] = *reinterpret_cast<const i4x*>(xl + t * 2048 + ((2 * b + half) ^ ((col >> 2) & 3)) * 16);
            ts[t & 1] = *reinterpret_cast<const float*>(sl + t * 256);
        };
        read(0);
#pragma unroll
        for (int b = 0; b < 2; ++b) a[b] = W::codes(wr, z + b, half);
        const h4x rs{W::scale(wr, z + half), 0, 0, 0};
        i16x r[2];
        f32x scale[2];
        auto scales = [&](int t) { return __builtin_amdgcn_mfma_f32_32x32x4f16(rs, h4x{static_cast<_Float16>(ts[t & 1]), 0, 0, 0}, zero, 0, 0, 0); };
        __builtin_amdgcn_sched_barrier(0);
        scale[0] = scales(0);
        r[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0], x[0][0], start, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 2 * T; ++i) {   // block i & 1 of tile i >> 1; the products of the step behind it first
            const int t = i >> 1;
            if (i + 1 < 2 * T) {
                if (i & 1) scale[(t + 1) & 1] = scales(t + 1);
                r[(i + 1) & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[(i + 1) & 1], x[((i + 1) >> 1) & 1][(i + 1) & 1], start, 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (!(i & 1) && t + 1 < T) read(t + 1);
            if (i == 1) tokens(next, buf ^ 1);
            if ((q & 1) == 0 && i == 2) weights(next_half, odd ^ 1, 0);
            if ((q & 1) == 0 && i == 3) weights(next_half, odd ^ 1, 1);
            __builtin_amdgcn_sched_barrier(0);
            f16x f = __builtin_bit_cast(f16x, r[i & 1]);
            // Sixteen subtractions, then sixteen FMAs: an instruction that waits for the one before it costs its wavefront eight clocks, one that does
            // not five.  Q8_0, hidden 3072, two layers, 1001 tokens 1023 -> 986 us; 16384 x 3072 times 2048 tokens by itself 336 -> 310.
#pragma unroll
            for (int e = 0; e < 16; ++e) f[e] = W::dot(f[e], start_f);
            asm volatile("" : "+v"(f));
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][e] = fmaf(f[e], scale[t & 1][16 * (i & 1) + e], acc[t][e]);
            __builtin_amdgcn_sched_barrier(0);
        }
        buf ^= 1;
    };
    for (uint32_t sb = sb0; sb < sb1; ++sb) {
        part(sb, std::integral_constant<uint32_t, 0>{});
        part(sb, std::integral_constant<uint32_t, 1>{});
        part(sb, std::integral_constant<uint32_t, 2>{});
        part(sb, std::integral_constant<uint32_t, 3>{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last loads ran once more: nothing may land behind the kernel's end, or on what follows
    // a lane holds rows 8 b + 4 half .. + 3 of the wavefront's 32, b = 0 .. 3, of one token per tile
    if constexpr (SWIGLU) {
        __syncthreads();
        float* const xch = reinterpret_cast<float*>(act[0]);                          // [wave][token] largest magnitude of its sixteen rows
        int* const xsum = reinterpret_cast<int*>(act[0]) + I8_WAVES * TOKENS;      // [wave][token] sum of its quants
        float h[T][8], amax[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            amax[t] = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) {   // silu(gate) * up (cera/src/backend/cpu.rs:2570-2575)
                const float g = acc[t][e];
                h[t][e] = __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, cera_expf(-g))), acc[t][8 + e]);
                amax[t] = fmaxf(amax[t], fabsf(h[t][e]));   // fmaxf drops a NaN operand, as f32::max does
            }
            amax[t] = fmaxf(amax[t], __shfl_xor(amax[t], 32, 64));
            if (half == 0) xch[wave * TOKENS + t * 32 + col] = amax[t];
        }
        __syncthreads();
        // the Q8_0 block of a token is this wavefront's sixteen rows and its neighbour's (cpu.rs:942-958)
        const uint32_t row0 = m0 + wave * 16;
        float scale[T];
        int sum[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const uint32_t tok = n0 + t * 32 + col;
            const float d = __fdiv_rn(fmaxf(amax[t], xch[(wave ^ 1) * TOKENS + t * 32 + col]), 127.0f), r = __fdiv_rn(1.0f, d);
            const float id = (d != 0.0f && fabsf(r) != __builtin_inff() && r == r) ? r : 0.0f;
            scale[t] = h2f(f2h(d));
            uint32_t packed[2] = {0, 0};
            sum[t] = 0;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int v = q8_round(h[t][e], id);
                sum[t] += v;
                packed[e >> 2] |= (static_cast<uint32_t>(v) & 0xFF) << (8 * (e & 3));
            }
            sum[t] += __shfl_xor(sum[t], 32, 64);
            if (half == 0) xsum[wave * TOKENS + t * 32 + col] = sum[t];
            if (tok < p.n && row0 < rows)   // m % 32 == 0: the block is whole or absent
#pragma unroll
                for (int b = 0; b < 2; ++b) *reinterpret_cast<uint32_t*>(p.hq + static_cast<uint64_t>(tok) * rows + row0 + 8 * b + 4 * half) = packed[b];
        }
        __syncthreads();
        if (half == 0 && (wave & 1) == 0 && row0 < rows)
#pragma unroll
            for (int t = 0; t < T; ++t) {
                const uint32_t tok = n0 + t * 32 + col;
                if (tok >= p.n) continue;
                const uint64_t at = static_cast<uint64_t>(tok) * (rows / 32) + row0 / 32;
                p.hs[at] = scale[t];
                p.hbsum[at] = scale[t] * static_cast<float>(sum[t] + xsum[(wave + 1) * TOKENS + t * 32 + col]);
            }
        return;
    }
    float* const out = second ? p.out2 : p.out;
    const uint64_t ldn = second ? p.ld_n2 : p.ld_n;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t tok = n0 + t * 32 + col;
        if (tok >= p.n) continue;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint32_t row = m0 + wave * 32 + 8 * b + 4 * half;
            if (p.ld_m == 1 && row + 4 <= rows && (ldn & 3) == 0) {
                const uint64_t at = row + tok * ldn;
                f4v v{acc[t][4 * b], acc[t][4 * b + 1], acc[t][4 * b + 2], acc[t][4 * b + 3]};
                if (p.resid) {
                    const f4v r = *reinterpret_cast<const f4v*>(p.resid + at);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = r[e] + (p.resid_scale != 1.0f ? v[e] * p.resid_scale : v[e]);
                }
                *reinterpret_cast<f4v*>(out + at + blockIdx.z * p.part_stride) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (row + e >= rows) continue;
                    const uint64_t at = (row + e) * p.ld_m + tok * ldn;
                    float v = acc[t][4 * b + e];
                    if (p.resid) v = p.resid[at] + (p.resid_scale != 1.0f ? v * p.resid_scale : v);
                    out[at + blockIdx.z * p.part_stride] = v;
                }
            }
        }
    }
}

bool bad(const I8Args& a, uint32_t split) {
    return a.n == 0 || a.m == 0 || a.k == 0 || a.k % 256 || a.k_chunk % 256 || static_cast<uint64_t>(a.k_chunk) * split != a.k || a.row_bytes % 16;
}

}  // namespace

template <bool SWIGLU>
static void go(cera_hip_ctx* ctx, uint32_t dtype, const I8Args& a, dim3 grid) {
    const dim3 block(64 * I8_WAVES);
    const bool q8 = dtype == CERA_HIP_Q8_0;
    if (i8_tokens(a.n) == 64) {
        if (q8) hipLaunchKernelGGL((gemm_i8_kernel<I8Q8_0, SWIGLU, 2>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((gemm_i8_kernel<I8Q4_0, SWIGLU, 2>), grid, block, 0, ctx->stream, a);
    } else {
        if (q8) hipLaunchKernelGGL((gemm_i8_kernel<I8Q8_0, SWIGLU, 4>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((gemm_i8_kernel<I8Q4_0, SWIGLU, 4>), grid, block, 0, ctx->stream, a);
    }
}

cera_hip_status cera_launch_i8(cera_hip_ctx* ctx, uint32_t dtype, const I8Args& a, uint32_t split) {
    if (bad(a, split)) return cera_fail(ctx, CERA_HIP_ERR_SHAPE, "gemm_i8: bad shape");
    go<false>(ctx, dtype, a, dim3((a.n + i8_tokens(a.n) - 1) / i8_tokens(a.n), a.tiles1 + (a.w2 ? (a.m2 + I8_ROWS - 1) / I8_ROWS : 0), split));
    HIP_TRY(ctx, hipGetLastError());
    return CERA_HIP_OK;
}

cera_hip_status cera_launch_i8_swiglu(cera_hip_ctx* ctx, uint32_t dtype, const I8Args& a) {
    if (bad(a, 1) || a.m % 32 || !a.w2) return cera_fail(ctx, CERA_HIP_ERR_SHAPE, "gemm_i8: bad shape");
    go<true>(ctx, dtype, a, dim3((a.n + i8_tokens(a.n) - 1) / i8_tokens(a.n), (a.m + I8_ROWS / 2 - 1) / (I8_ROWS / 2)));
    HIP_TRY(ctx, hipGetLastError());
    return CERA_HIP_OK;
}
