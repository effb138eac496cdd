// Products of Q6_K matrices with many tokens (a prompt's pass) on the f16 matrix cores, whole numbers exact per block.
//
// A weight enters as scale * (code - 32), up to 13 bits, in two f16 parts whose sum it is, and a quant as f16, so two
// v_mfma_f32_16x16x32_f16 are one 32-weight block of a 16 x 16 tile, its result the exact whole number below 2^24: one FMA
// with the token's block scale per output and block, one with the row's d per super-block.  The kernel for fewer tokens
// multiplies codes by quants alone, one matrix instruction per group of 16, and pays two FMAs per output and block and a
// 64-clock outer product for the scales.
//
// 256 rows x 128 tokens, eight wavefronts of 32 rows each over all tokens: a wavefront unpacks its own rows, once for 128
// tokens.  Half a super-block is a stage: the tokens' fragments come by direct loads from records laid out for it, the rows'
// bytes through registers (they are 2-byte aligned), both a stage ahead, one load a step (all of them behind the barrier cost
// 3 % at 2048 tokens), with one barrier.  A step -- one block, 16 tokens -- issues its four matrix instructions, folds the
// step before and unpacks a piece of the next block while they run.
//
// 4096 x 14336 (with the tokens' operand and the sum of the slices): 512 tokens 172 -> 139 us, 2048 tokens 617 -> 440 us;
// 4096 x 4096 with 512 tokens 66 -> 56 us, 128 tokens 33 -> 29 us.  What bounds it: the products of both parts, 193 us of the
// 440 at the nominal rate, and the folds and the unpacking; the matrix cores are busy for 44 % of the time and the vector ALU
// for 55 %, and the two take turns.
#include "f16_codes.hip.h"
#include "gemm_kq.h"
#include "gemv.hip.h"
#include "lds_dma.hip.h"

namespace {

__global__ __launch_bounds__(256) void kq_act_kernel(const int8_t* __restrict__ bq, uint8_t* __restrict__ act, uint32_t n, uint32_t k) {
    kq_act_record(blockIdx.x, bq, act, n, k);
}

// ---- Q6_K: half h of a super-block is two runs j of 16 codes of each of its four blocks --------------------------
struct KqQ6 {
    // a row's bytes of a stage in LDS: two 16-byte runs of ql, of ql + 32 and of qh; eight scales; d as f32
    static constexpr uint32_t A = 0, B = KQ_ROWS * 32, Q = 2 * KQ_ROWS * 32, SC = 3 * KQ_ROWS * 32, D = SC + KQ_ROWS * 8, BYTES = D + KQ_ROWS * 4;
    struct Stage { uint4 a, b, q; uint2 sc; uint32_t d; };   // what a thread brings in: run j of its row
    static constexpr int LOADS = 5;
    template <int P> static __device__ __forceinline__ void load(Stage& s, const uint8_t* row, uint32_t stage, uint32_t j) {
        const uint8_t* const blk = row + (stage >> 1) * 210;
        const uint32_t h = stage & 1;
        if constexpr (P == 0) s.a = ld_u128_a2(blk + h * 64 + j * 16);
        if constexpr (P == 1) s.b = ld_u128_a2(blk + h * 64 + 32 + j * 16);
        if constexpr (P == 2) s.q = ld_u128_a2(blk + 128 + h * 32 + j * 16);
        if constexpr (P == 3) s.sc = ld_u64_a2(blk + 192 + h * 8);
        if constexpr (P == 4) s.d = ld_u16(blk + 208);
    }
    static __device__ __forceinline__ void store(const Stage& s, uint8_t* lds, uint32_t r, uint32_t j) {
        *reinterpret_cast<uint4*>(lds + A + r * 32 + j * 16) = s.a;
        *reinterpret_cast<uint4*>(lds + B + r * 32 + j * 16) = s.b;
        *reinterpret_cast<uint4*>(lds + Q + r * 32 + j * 16) = s.q;
        // the scales by run 0's thread, d by run 1's: no branch, which would let the compiler move a stage's folds behind it
        const uint32_t d = __builtin_bit_cast(uint32_t, h2f(s.d)), at = j ? D + r * 4 : SC + r * 8;
        *reinterpret_cast<uint32_t*>(lds + at) = j ? d : s.sc.x ^ 0x80808080u;
        *reinterpret_cast<uint32_t*>(lds + (j ? at : at + 4)) = j ? d : s.sc.y ^ 0x80808080u;
    }
    struct Raw { uint32_t a[2], b[2], q[2], sc[2]; };
    static __device__ __forceinline__ void read(Raw& w, const uint8_t* lds, uint32_t r, uint32_t g) {
        const uint32_t at = r * 32 + kq_dword(g) * 4;
        const uint2 a = *reinterpret_cast<const uint2*>(lds + A + at), b = *reinterpret_cast<const uint2*>(lds + B + at),
                    q = *reinterpret_cast<const uint2*>(lds + Q + at), s = *reinterpret_cast<const uint2*>(lds + SC + r * 8);
        w.a[0] = a.x; w.a[1] = a.y; w.b[0] = b.x; w.b[1] = b.y; w.q[0] = q.x; w.q[1] = q.y;
        w.sc[0] = s.x >> (8 * (g & 1)); w.sc[1] = s.y >> (8 * (g & 1));
    }
    // codes 4e .. 4e + 3 of this lane's eight of block z
    template <int z, int e> static __device__ __forceinline__ void unpack(const Raw& w, h8v& hi, h8v& lo) {
        const h2v sc = byte_twice<2 * (z & 1)>(w.sc[z >> 1]) - both(1152.f);
        const uint32_t ql = z & 1 ? w.b[e] : w.a[e], qh = w.q[e];
        const uint32_t top = (z == 0 ? qh << 4 : z == 1 ? qh << 2 : z == 2 ? qh : qh >> 2) & 0x30303030u;
        const uint32_t c = ((z < 2 ? ql : ql >> 4) & 0x0F0F0F0Fu) | top;
        // code - 32, times the scale: rounded to f16, and the remainder
        const h2v u = bytes02(c) - both(1056.f), v = bytes13(c) - both(1056.f);
        const h2v uh = u * sc, vh = v * sc, ul = fma2(u, sc, -uh), vl = fma2(v, sc, -vh);
        hi[4 * e] = uh[0]; hi[4 * e + 1] = uh[1]; hi[4 * e + 2] = vh[0]; hi[4 * e + 3] = vh[1];
        lo[4 * e] = ul[0]; lo[4 * e + 1] = ul[1]; lo[4 * e + 2] = vl[0]; lo[4 * e + 3] = vl[1];
    }
};

template <typename W>
__global__ __launch_bounds__(512, 2) void gemm_kq_kernel(KqArgs p) {
    constexpr int RT = 2, T = KQ_TOKENS / 16;   // 16-row and 16-token tiles of a wavefront
    constexpr uint32_t TILE = KQ_HALF + 256;    // a tile's half record, and behind it the four blocks' 16 scales each
    __shared__ __align__(16) uint8_t act[2][T * TILE];
    __shared__ __align__(16) uint8_t wts[2][W::BYTES];
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, col = lane & 15;
    const bool second = p.w2 != nullptr && blockIdx.y >= p.tiles1;
    const uint8_t* const wmat = second ? p.w2 : p.w;
    const uint32_t rows = second ? p.m2 : p.m, m0 = (second ? blockIdx.y - p.tiles1 : blockIdx.y) * KQ_ROWS, n0 = blockIdx.x * KQ_TOKENS;
    const uint32_t nsb = p.k / 256, s0 = blockIdx.z * (p.k_chunk / 128), s1 = s0 + p.k_chunk / 128;   // stages: half super-blocks
    // this thread's share of a stage's rows: one run of one row; rows past the end are the last one again
    const uint32_t wr = threadIdx.x >> 1, wj = threadIdx.x & 1;
    const uint8_t* const wrow = wmat + static_cast<uint64_t>(min(m0 + wr, rows - 1)) * p.row_bytes;
    // this wavefront's share of a stage's tokens: one tile of 16
    // (tiles past the end are the last one again: their products are not stored)
    const uint32_t tile = min(blockIdx.x * T + wave, (p.n - 1) / 16);
    const uint8_t* const rec = p.act + static_cast<uint64_t>(tile) * nsb * KQ_REC;
    const float* const bs = p.bs + static_cast<uint64_t>(tile) * 16 * (p.k / 32);
    const uint32_t bs_lane = (min(col, p.n - 1 - tile * 16) * (p.k / 32) + g) * 4;
    const uint32_t act_lds = lds_addr(&act[0][0]) + wave * TILE;
    // piece p of a stage's loads: the rows' first, then the tokens'
    typename W::Stage st;
    auto load = [&](auto p_, uint32_t stage, uint32_t buf) {
        constexpr int p = decltype(p_)::value;
        if constexpr (p < W::LOADS) W::template load<p>(st, wrow, stage, wj);
        else if constexpr (p < W::LOADS + 5) {
            const uint32_t l = act_lds + buf * (T * TILE) + (p - W::LOADS) * 1024;
            if constexpr (p < W::LOADS + 4) lds_dma_1k(rec + static_cast<uint64_t>(stage) * KQ_HALF + (p - W::LOADS) * 1024, lane * 16, l);
            else lds_dma_256(bs + stage * 4, bs_lane, l);
        }
    };
    f4v acc[RT][T], sum[RT][T];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int t = 0; t < T; ++t) acc[rt][t] = f4v{0.f, 0.f, 0.f, 0.f};
#define KQ_LOAD(p) load(std::integral_constant<int, p>{}, s0, 0)
    KQ_LOAD(0); KQ_LOAD(1); KQ_LOAD(2); KQ_LOAD(3); KQ_LOAD(4); KQ_LOAD(5); KQ_LOAD(6); KQ_LOAD(7); KQ_LOAD(8); KQ_LOAD(9);
#undef KQ_LOAD
    W::store(st, wts[0], wr, wj);
    uint32_t buf = 0;
    const f4v zero{0.f, 0.f, 0.f, 0.f};
    auto stage = [&](uint32_t s, auto odd_) {
        constexpr int odd = decltype(odd_)::value;
        // this stage's tokens and rows are in, and no wavefront reads the other buffers any more
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        const uint32_t next = min(s + 1, s1 - 1);
        const uint8_t* const wl = wts[buf];
        const uint8_t* const al = act[buf];
        typename W::Raw raw[RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) W::read(raw[rt], wl, wave * 32 + rt * 16 + col, g);
        h8v x[3];        // tokens' fragments and scales, two steps ahead
        float xs[4];
        auto read = [&](int i) {
            const uint8_t* const a = al + (i & 7) * TILE;
            x[i % 3] = *reinterpret_cast<const h8v*>(a + (i >> 3) * 1024 + lane * 16);
            xs[i & 3] = *reinterpret_cast<const float*>(a + 4096 + (i >> 3) * 64 + col * 4);
        };
        read(0);
        read(1);
        h8v hi[2][RT], lo[2][RT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            W::template unpack<0, 0>(raw[rt], hi[0][rt], lo[0][rt]);
            W::template unpack<0, 1>(raw[rt], hi[0][rt], lo[0][rt]);
        }
        f4v r[2][RT];
        auto fold = [&](int i) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    sum[rt][i & 7][e] = odd || i >= T ? fmaf(r[i & 1][rt][e], xs[i & 3], sum[rt][i & 7][e]) : r[i & 1][rt][e] * xs[i & 3];
        };
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](auto i_) {
            constexpr int i = decltype(i_)::value, z = i >> 3, t = i & 7;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) r[i & 1][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[z & 1][rt], x[i % 3], zero, 0, 0, 0);
            if (i + 2 < 4 * T) read(i + 2);
            load(std::integral_constant<int, i>{}, next, buf ^ 1);   // one a step: all at once, they would hold every wavefront up behind the barrier
            if (i) fold(i - 1);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) r[i & 1][rt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[z & 1][rt], x[i % 3], r[i & 1][rt], 0, 0, 0);
            if constexpr (z < 3 && t < 2 * RT) W::template unpack<z + 1, t & 1>(raw[t >> 1], hi[(z + 1) & 1][t >> 1], lo[(z + 1) & 1][t >> 1]);
            __builtin_amdgcn_sched_barrier(0);
        };
#define KQ_STEP4(b) step(std::integral_constant<int, b>{}); step(std::integral_constant<int, b + 1>{}); step(std::integral_constant<int, b + 2>{}); step(std::integral_constant<int, b + 3>{})
        KQ_STEP4(0); KQ_STEP4(4); KQ_STEP4(8); KQ_STEP4(12); KQ_STEP4(16); KQ_STEP4(20); KQ_STEP4(24); KQ_STEP4(28);
#undef KQ_STEP4
        fold(4 * T - 1);
        if (odd) {
            f4v d[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) d[rt] = *reinterpret_cast<const f4v*>(wl + W::D + (wave * 32 + rt * 16 + g * 4) * 4);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int t = 0; t < T; ++t)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[rt][t][e] = fmaf(d[rt][e], sum[rt][t][e], acc[rt][t][e]);
        }
        buf ^= 1;
        W::store(st, wts[buf], wr, wj);
    };
    for (uint32_t s = s0; s < s1; s += 2) {   // whole super-blocks
        stage(s, std::integral_constant<int, 0>{});
        stage(s + 1, std::integral_constant<int, 1>{});
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last stage's loads ran once more: nothing may land behind the kernel's end
    float* const out = second ? p.out2 : p.out;
    const uint64_t ldn = second ? p.ld_n2 : p.ld_n;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t tok = n0 + t * 16 + col;
        if (tok >= p.n) continue;
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const uint32_t row = m0 + wave * 32 + rt * 16 + g * 4;
            if (row >= rows) continue;
            if (p.ld_m == 1 && row + 4 <= rows && (ldn & 3) == 0) {
                const uint64_t at = row + tok * ldn;
                f4v v = acc[rt][t];
                if (p.resid) {
                    const f4v b = *reinterpret_cast<const f4v*>(p.resid + at);
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = b[e] + (p.resid_scale != 1.0f ? v[e] * p.resid_scale : v[e]);
                }
                *reinterpret_cast<f4v*>(out + at + blockIdx.z * p.part_stride) = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (row + e >= rows) continue;
                    const uint64_t at = (row + e) * p.ld_m + tok * ldn;
                    float v = acc[rt][t][e];
                    if (p.resid) v = p.resid[at] + (p.resid_scale != 1.0f ? v * p.resid_scale : v);
                    out[at + blockIdx.z * p.part_stride] = v;
                }
            }
        }
    }
}

}  // namespace

cera_hip_status cera_launch_kq_act(cera_hip_ctx* ctx, const int8_t* bq, uint32_t n, uint32_t k, void* act) {
    hipLaunchKernelGGL(kq_act_kernel, dim3(kq_act_records(n, k)), dim3(256), 0, ctx->stream, bq, static_cast<uint8_t*>(act), n, k);
    HIP_TRY(ctx, hipGetLastError());
    return CERA_HIP_OK;
}

cera_hip_status cera_launch_kq(cera_hip_ctx* ctx, const KqArgs& a, uint32_t split) {
    if (a.n == 0 || a.k % 256 || a.k_chunk % 256 || static_cast<uint64_t>(a.k_chunk) * split != a.k) return cera_fail(ctx, CERA_HIP_ERR_SHAPE, "gemm_kq: bad shape");
    const dim3 grid((a.n + KQ_TOKENS - 1) / KQ_TOKENS, a.tiles1 + (a.w2 ? (a.m2 + KQ_ROWS - 1) / KQ_ROWS : 0), split);
    hipLaunchKernelGGL(gemm_kq_kernel<KqQ6>, grid, dim3(512), 0, ctx->stream, a);
    HIP_TRY(ctx, hipGetLastError());
    return CERA_HIP_OK;
}
