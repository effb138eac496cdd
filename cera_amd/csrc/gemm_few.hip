// Products of Q4_K and Q6_K matrices with a few tokens at once (2 to 48: drafted tokens to verify, a chat turn), read from
// their decode copies or, with the same bits, from the native blocks.
//
// A wavefront owns 16 weight rows and streams their super-blocks straight into registers, two of them ahead; the tokens, in
// tiles of 16, come from LDS, where the workgroup's eight wavefronts put them as f16 (the Q8_0 codes are whole numbers, exact
// in f16), a chunk of super-blocks ahead.  One v_mfma_f32_16x16x32_f16 is one 32-weight block: Q4_K weights enter as
// scale * code, at most 945 and exact in f16; Q6_K weights, up to 4096 (-128 times -32), as scale * lower four bits and scale * (16 * upper two - 32), exact both.
// So a block's result is the exact whole number sum(scale * code * quant): quants are at most 127 (the quantizer's scale is the
// largest magnitude over 127), and 32 * 4096 * 127 is 1 % below 2^24.  What the vector ALU adds is one FMA with the token's
// block scale per output and block, one with the row's d per super-block, and for Q4_K one with dmin on the mins' own product
// (mins times the tokens' block sums in three bf16 parts).  Sums over K go in order within a slice.
//
// What bounds it: the instructions, about 140 (Q4_K) and 200 (Q6_K) per 16 rows x 256 weights to unpack and 40 per tile of 16 tokens.
// A SIMD that has matrix instructions among them issues one in four clocks, whichever it is and however many wavefronts it
// has: gate | up with 5 tokens takes 17 us without its loads, the loads alone 12, both 21.5 (3.1 TB/s).  In a pass, gate | up of 14336 x 4096 Q4_K
// with SwiGLU takes 21.9 us at 5 tokens and 36.5 at 45 (the pair 21.5 and 35.6, SwiGLU 4.6 and 5.1, with codes in the mantissa of 1024, code
// and scale of a Q6_K weight put together and then rounded and split, and up to four super-blocks ahead); Q | K | V 11.0 and 16.9 (14.0, 17.2), down, 4096
// x 14336 Q6_K, 16.8 and 23.4 (19.0, 23.7).  At 45 tokens the vector ALU is busy for half of gate | up, the matrix cores for 16 %.  The 64-token
// tiles before it took 36 us for a down product and 50 for a pair, with a launch for the tokens' copy before and one for the sums
// behind them; passes of the two-layer 8B shapes: 5 tokens 406 -> 262 us, 45 tokens 466 -> 294 (267 and 299 with SwiGLU in a launch of its own).
#include <algorithm>

#include "f16_codes.hip.h"
#include "few_pairs.h"
#include "gemv.hip.h"
#include "gemm_few.h"
#include "quantize.hip.h"

namespace {

typedef __bf16 b8v __attribute__((ext_vector_type(8)));

struct FewArgs {
    FewMat a, b;               // b: a second matrix of the same k, or m = 0
    uint32_t tiles_a;          // workgroups of a
    const int8_t* xq;
    const float *xs, *bsum;
    uint32_t n, k, sb_per;
    uint64_t part_stride;      // floats between the slices of a split K; 0: no split
    const float* resid;        // added to segment 0 of a (unsplit)
    float resid_scale;
    int8_t* hq;                // SwiGLU: the product's Q8_0 quants [n][m], scales and scale * sum of quants [n][m / 32]
    float *hs, *hbsum;
};

constexpr uint32_t FEW_ROWS = 16 * FEW_WAVES;
// LDS of one tile of 16 tokens and one super-block: a block's operand fragments (64 lanes x 16 bytes, the blocks 16 bytes
// further apart than that, so that the eight blocks of a token do not share their banks when they are written), the block
// scales, the mins' operand
constexpr uint32_t FEW_BLOCK = 1040, FEW_XS = 8 * FEW_BLOCK, FEW_MIN = FEW_XS + 512, FEW_TILE = FEW_MIN + 1024;

__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {   // a's upper 32 lanes with b's lower 32
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {   // a's odd rows of 16 lanes with b's even ones
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0]; b = r[1];
}

// Bits of a code where they are, cut out with their neighbours' cleared, are a subnormal f16, code * 2^-24 times a power of two: what a
// product by its scale leaves is exact, a whole number times 2^-19 (Q4_K) or 2^-20, and the tokens' scales make up for it.  Byte j of v,
// twice, as 2^e + byte * 2^(e - 10) with the upper byte TOP of 2^e (0x64: e = 10, 0x68: 11, 0x74: 14, 0x78: 15).
template <uint32_t TOP, int J> __device__ __forceinline__ h2v byte_above(uint32_t v) { return as_h2(__builtin_amdgcn_perm(TOP * 0x01010101u, v, 0x04000400u | J | J << 16)); }

// ---- Q4_K -----------------------------------------------------------------------------------------
// Lane group g (of 16 lanes, one per row) loads unit g of the super-block, the blocks 2g and 2g + 1, in two 16-byte halves,
// and after the exchange holds dword g of both halves of every unit: codes 4g .. 4g + 3 and 16 + 4g .. 16 + 4g + 3 of a block.
struct FewQ4 {
    static constexpr bool MINS = true;
    static constexpr float XS = 524288.0f;   // 2^19
    struct W { uint4 h, f, s; };
    static __device__ __forceinline__ uint32_t dword(int g, int e) { return 4 * e + g; }   // e-th dword of a block's quants in lane group g
    // a lane's offsets from the matrix's first byte, and the super-block's three loads at them: the base that moves is scalar
    struct At { uint32_t h, f, s; };
    template <bool COPY> static __device__ __forceinline__ At at(uint32_t row, uint32_t g, uint32_t nsb) {
        if (COPY) return At{row, row + Q4K::stream_q0(4 * nsb) + g * 16, row + Q4K::stream_q1(4 * nsb) + g * 16};
        return At{row, row + 16 + g * 32, row + 32 + g * 32};
    }
    template <bool COPY> static __device__ __forceinline__ void load(W& w, const uint8_t* m, uint32_t sb, const At& o) {
        const uint8_t *const h = m + sb * (COPY ? 16u : 144u), *const q = m + sb * (COPY ? 64u : 144u);
        w.h = ld_u128(h + o.h);
        w.f = ld_u128(q + o.f);
        w.s = ld_u128(q + o.s);
    }
    template <int T>
    static __device__ __forceinline__ void multiply(const W& w, const unsigned char* st, uint32_t lane, f4v (&acc)[T]) {
        // the tokens' fragments and scales of a unit's two blocks, read a unit ahead
        h8v x[2][T][2];
        float xs[2][T][2];
        auto read = [&](int u) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int z = 0; z < 2; ++z) {
                    const unsigned char* const p = st + t * FEW_TILE;
                    x[u & 1][t][z] = *reinterpret_cast<const h8v*>(p + (2 * u + z) * FEW_BLOCK + lane * 16);
                    xs[u & 1][t][z] = *reinterpret_cast<const float*>(p + FEW_XS + (2 * u + z) * 64 + (lane & 15) * 4);
                }
        };
        read(0);
        uint32_t dd[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) dd[i] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(((lane >> 4) * 4 + i) * 4, static_cast<int>(w.h.x)));
        uint32_t f[4] = {w.f.x, w.f.y, w.f.z, w.f.w}, s[4] = {w.s.x, w.s.y, w.s.z, w.s.w};
        swap32(f[0], f[2]); swap32(f[1], f[3]); swap32(s[0], s[2]); swap32(s[1], s[3]);
        swap16(f[0], f[1]); swap16(f[2], f[3]); swap16(s[0], s[1]); swap16(s[2], s[3]);   // now by unit
        const uint32_t sc[2] = {w.h.y & 0x3F3F3F3Fu, (w.h.w & 0x0F0F0F0Fu) | ((w.h.y >> 2) & 0x30303030u)};
        const uint32_t mn[2] = {w.h.z & 0x3F3F3F3Fu, ((w.h.w >> 4) & 0x0F0F0F0Fu) | ((w.h.z >> 2) & 0x30303030u)};
        const f4v zero{0.f, 0.f, 0.f, 0.f};
        f4v sum[T];
        b8v xm[T];
        f4v r[T][2];
        auto fold = [&](int u) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int z = 0; z < 2; ++z)
#pragma unroll
                    for (int i = 0; i < 4; ++i) sum[t][i] = u + z ? fmaf(r[t][z][i], xs[u & 1][t][z], sum[t][i]) : r[t][z][i] * xs[u & 1][t][z];
        };
        // a unit's weights are unpacked while the matrix cores are at the unit before
        auto unit = [&](auto u_) {
            constexpr int u = decltype(u_)::value;
            // 32 times the scale, and for the upper nibbles, whose codes stand sixteen times as high, twice the scale
            const h2v s0 = byte_above<0x78, 2 * (u & 1)>(sc[u >> 1]) - both(32768.f), s1 = byte_above<0x68, 2 * (u & 1) + 1>(sc[u >> 1]) - both(2048.f);
            h8v wt[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t q = e ? s[u] : f[u], q8 = q >> 8;
                const h2v a = as_h2(q & 0x000F000Fu) * s0, b = as_h2(q8 & 0x000F000Fu) * s0, c = as_h2(q & 0x00F000F0u) * s1, d = as_h2(q8 & 0x00F000F0u) * s1;
                wt[0][4 * e] = a[0]; wt[0][4 * e + 1] = a[1]; wt[0][4 * e + 2] = b[0]; wt[0][4 * e + 3] = b[1];
                wt[1][4 * e] = c[0]; wt[1][4 * e + 1] = c[1]; wt[1][4 * e + 2] = d[0]; wt[1][4 * e + 3] = d[1];
            }
            if (u) fold(u - 1);
            __builtin_amdgcn_sched_barrier(0);
            if (u < 3) read(u + 1);
            else
#pragma unroll
                for (int t = 0; t < T; ++t) xm[t] = *reinterpret_cast<const b8v*>(st + t * FEW_TILE + FEW_MIN + lane * 16);
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int z = 0; z < 2; ++z) r[t][z] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wt[z], x[u & 1][t][z], zero, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        unit(std::integral_constant<int, 0>{}); unit(std::integral_constant<int, 1>{});
        unit(std::integral_constant<int, 2>{}); unit(std::integral_constant<int, 3>{});
        b8v am;
#pragma unroll
        for (int b = 0; b < 8; ++b) am[b] = static_cast<__bf16>(static_cast<float>((mn[b >> 2] >> (8 * (b & 3))) & 0xFF));
        fold(3);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const f4v m = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, xm[t], zero, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][i] = fmaf(-h2f(dd[i] >> 16), m[i], fmaf(h2f(dd[i] & 0xFFFF), sum[t][i], acc[t][i]));
        }
    }
};

// ---- Q6_K -----------------------------------------------------------------------------------------
// Unit (h, j): run j of 16 codes of the four blocks of half h.  Lane group 2h + j loads it and after the exchange holds, as
// group 2a + j, dwords 2a and 2a + 1 of the runs j of both halves: codes 16j + 8a .. 16j + 8a + 7 of a block.
struct FewQ6 {
    static constexpr bool MINS = false;
    static constexpr float XS = 1048576.0f;   // 2^20
    struct W { uint4 a, b, q, sc; uint32_t d; };
    static __device__ __forceinline__ uint32_t dword(int g, int e) { return 4 * (g & 1) + 2 * (g >> 1) + e; }
    struct At { uint32_t a, b, q, sc, d; };
    template <bool COPY> static __device__ __forceinline__ At at(uint32_t row, uint32_t g, uint32_t nsb) {
        const uint32_t plane = Q6K::up128(64 * nsb), h = g >> 1, j = (g & 1) * 16;
        if (COPY) return At{row + g * 16, row + plane + g * 16, row + 2 * plane + g * 16, row + Q6K::stream_sc(4 * nsb), row + Q6K::stream_d(4 * nsb)};
        return At{row + h * 64 + j, row + h * 64 + 32 + j, row + 128 + h * 32 + j, row + 192, row + 208};
    }
    template <bool COPY> static __device__ __forceinline__ void load(W& w, const uint8_t* m, uint32_t sb, const At& o) {
        const uint8_t* const q = m + sb * (COPY ? 64u : 210u);
        if (COPY) {
            w.a = ld_u128(q + o.a);
            w.b = ld_u128(q + o.b);
            w.q = ld_u128(q + o.q);
            w.sc = ld_u128(m + sb * 16u + o.sc);
            w.d = ld_u16(m + sb * 2u + o.d);
        } else {
            w.a = ld_u128_a2(q + o.a);
            w.b = ld_u128_a2(q + o.b);
            w.q = ld_u128_a2(q + o.q);
            w.sc = ld_u128_a2(q + o.sc);
            w.d = ld_u16(q + o.d);
        }
    }
    template <int T>
    static __device__ __forceinline__ void multiply(const W& w, const unsigned char* st, uint32_t lane, f4v (&acc)[T]) {
        h8v x[2][T];   // a block ahead
        float xs[2][T];
        auto read = [&](int b) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                x[b & 1][t] = *reinterpret_cast<const h8v*>(st + t * FEW_TILE + b * FEW_BLOCK + lane * 16);
                xs[b & 1][t] = *reinterpret_cast<const float*>(st + t * FEW_TILE + FEW_XS + b * 64 + (lane & 15) * 4);
            }
        };
        read(0);
        uint32_t dd[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) dd[i] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(((lane >> 4) * 4 + i) * 4, static_cast<int>(w.d)));
        uint32_t a[4] = {w.a.x, w.a.y, w.a.z, w.a.w}, b[4] = {w.b.x, w.b.y, w.b.z, w.b.w}, q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
        swap32(a[0], a[2]); swap32(a[1], a[3]); swap32(b[0], b[2]); swap32(b[1], b[3]); swap32(q[0], q[2]); swap32(q[1], q[3]);   // now [half][dword]
        const uint32_t sh = 8 * ((lane >> 4) & 1);
        const f4v zero{0.f, 0.f, 0.f, 0.f};
        f4v sum[T];
        f4v r[T];
        auto fold = [&](int blk) {
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) sum[t][i] = blk ? fmaf(r[t][i], xs[blk & 1][t], sum[t][i]) : r[t][i] * xs[blk & 1][t];
        };
        auto block = [&](auto b_) {
            constexpr int blk = decltype(b_)::value, h = blk >> 2, z = blk & 3;
            const uint32_t sv = ((z < 2 ? (h ? w.sc.z : w.sc.x) : (h ? w.sc.w : w.sc.y)) ^ 0x80808080u) >> sh;
            // sixteen times the scale for the lower nibbles; what makes the two upper bits, where they stand, 16 * scale * bits; 32 * scale
            const h2v sl = z < 2 ? byte_above<0x74, 2 * (z & 1)>(sv) - both(18432.f) : byte_above<0x64, 2 * (z & 1)>(sv) - both(1152.f);
            const h2v su = sl * both(z & 1 ? 4.f : 16.f), off = sl * both(z < 2 ? -0x1p-19f : -0x1p-15f);
            constexpr uint32_t lower = z < 2 ? 0x000F000Fu : 0x00F000F0u, upper = 0x00030003u << (2 * z);
            h8v hi, lo;
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t ql = z & 1 ? b[2 * h + e] : a[2 * h + e], qh = q[2 * h + e];
                const h2v ul = as_h2(ql & lower) * sl, vl = as_h2((ql >> 8) & lower) * sl, uh = fma2(as_h2(qh & upper), su, off), vh = fma2(as_h2((qh >> 8) & upper), su, off);
                hi[4 * e] = uh[0]; hi[4 * e + 1] = uh[1]; hi[4 * e + 2] = vh[0]; hi[4 * e + 3] = vh[1];
                lo[4 * e] = ul[0]; lo[4 * e + 1] = ul[1]; lo[4 * e + 2] = vl[0]; lo[4 * e + 3] = vl[1];
            }
            if (blk) fold(blk - 1);
            __builtin_amdgcn_sched_barrier(0);
            if (blk < 7) read(blk + 1);
#pragma unroll
            for (int t = 0; t < T; ++t) r[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, x[blk & 1][t], zero, 0, 0, 0);
#pragma unroll
            for (int t = 0; t < T; ++t) r[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, x[blk & 1][t], r[t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        block(std::integral_constant<int, 0>{}); block(std::integral_constant<int, 1>{});
        block(std::integral_constant<int, 2>{}); block(std::integral_constant<int, 3>{});
        block(std::integral_constant<int, 4>{}); block(std::integral_constant<int, 5>{});
        block(std::integral_constant<int, 6>{}); block(std::integral_constant<int, 7>{});
        fold(7);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][i] = fmaf(h2f(dd[i] & 0xFFFF), sum[t][i], acc[t][i]);
    }
};

// T tiles of 16 tokens (four would spill registers)
template <typename W, int T> constexpr int FEW_CHUNK = few_chunk(W::MINS, T);
// Two super-blocks are on their way.  With four a slice of a few loads its last one up to four times again: 6144 x 4096 Q4_K in six
// slices with 5 tokens 10.8 -> 8.6 us, 4096 x 14336 Q6_K in eight 19.6 -> 17.8, 28672 x 4096 in one 21.4 -> 21.6.
constexpr int FEW_AHEAD = 2;
// The end of a SwiGLU launch.  A gate wavefront has from its up wavefront, in the same lanes, what goes with its sixteen rows; a Q8_0
// block of a token is its rows and its neighbour's (cera/src/backend/cpu.rs:2570-2575, 942-958).
template <int T>
__device__ __forceinline__ void few_swiglu(const FewArgs& a, const f4v (&acc)[T], bool second, uint32_t row0, unsigned char* lds) {
    constexpr uint32_t HALF = FEW_WAVES / 2, TOKENS = T * 16;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) % HALF, col = lane & 15, g = lane >> 4, m = a.a.m;
    f4v* const ups = reinterpret_cast<f4v*>(lds);                                      // [wave][tile][lane]
    float* const largest = reinterpret_cast<float*>(lds + HALF * T * 1024);            // [wave][token] largest magnitude of its sixteen rows
    int* const sums = reinterpret_cast<int*>(largest + HALF * TOKENS);                 // [wave][token] sum of its quants
    lds_barrier();   // nobody reads the tokens any more
    if (second)
#pragma unroll
        for (int t = 0; t < T; ++t) ups[(wave * T + t) * 64 + lane] = acc[t];
    lds_barrier();
    f4v h[T];
    float amax[T];
    if (!second)
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const f4v up = ups[(wave * T + t) * 64 + lane];
            amax[t] = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float gate = acc[t][i];
                h[t][i] = __fmul_rn(__fdiv_rn(gate, __fadd_rn(1.0f, cera_expf(-gate))), up[i]);
                amax[t] = fmaxf(amax[t], fabsf(h[t][i]));   // fmaxf drops a NaN operand, as f32::max does
            }
            amax[t] = fmaxf(amax[t], __shfl_xor(amax[t], 16, 64));
            amax[t] = fmaxf(amax[t], __shfl_xor(amax[t], 32, 64));
            if (g == 0) largest[wave * TOKENS + t * 16 + col] = amax[t];
        }
    lds_barrier();
    float scale[T];
    int sum[T];
    if (!second)
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const uint32_t tok = t * 16 + col;
            const float d = __fdiv_rn(fmaxf(amax[t], largest[(wave ^ 1) * TOKENS + tok]), 127.0f), r = __fdiv_rn(1.0f, d);
            const float id = (d != 0.0f && fabsf(r) != __builtin_inff() && r == r) ? r : 0.0f;
            scale[t] = h2f(f2h(d));
            uint32_t packed = 0;
            sum[t] = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int v = q8_round(h[t][i], id);
                sum[t] += v;
                packed |= (static_cast<uint32_t>(v) & 0xFF) << (8 * i);
            }
            sum[t] += __shfl_xor(sum[t], 16, 64);
            sum[t] += __shfl_xor(sum[t], 32, 64);
            if (g == 0) sums[wave * TOKENS + tok] = sum[t];
            if (tok < a.n && row0 < m) *reinterpret_cast<uint32_t*>(a.hq + static_cast<uint64_t>(tok) * m + row0 + 4 * g) = packed;   // m % 32 == 0
        }
    lds_barrier();
    if (second || g || wave % 2 || row0 >= m) return;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t tok = t * 16 + col;
        if (tok >= a.n) continue;
        const uint64_t at = static_cast<uint64_t>(tok) * (m / 32) + row0 / 32;
        a.hs[at] = scale[t];
        a.hbsum[at] = scale[t] * static_cast<float>(sum[t] + sums[(wave + 1) * TOKENS + tok]);
    }
}

// SWIGLU: the lower half of the wavefronts has rows of matrix a, the gate's, the upper half the same rows of b, the up matrix, and
// the workgroup leaves silu(gate) * up as quants
template <typename W, int T, bool COPY, bool SWIGLU = false>
__device__ __forceinline__ void few_body(const FewArgs& a, bool second, unsigned char* lds) {
    constexpr int S = FEW_CHUNK<W, T>, AHEAD = FEW_AHEAD, NP = few_rounds(S * T);
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nsb = a.k / 256;
    if (SWIGLU) second = wave >= FEW_WAVES / 2;
    const FewMat& M = second ? a.b : a.a;
    const uint32_t row0 = SWIGLU ? blockIdx.x * (FEW_ROWS / 2) + wave % (FEW_WAVES / 2) * 16 : (blockIdx.x - (second ? a.tiles_a : 0)) * FEW_ROWS + wave * 16;
    const uint32_t sb0 = blockIdx.y * a.sb_per, sb1 = min(nsb, sb0 + a.sb_per);
    const uint8_t* const m0 = M.w;
    const typename W::At at = W::template at<COPY>(min(row0 + (lane & 15), M.m - 1) * M.row_bytes, lane >> 4, nsb);   // rows past the end: the last one again
    // the tokens of a chunk: a thread takes the 32 quants of one block of one token, block_of of token_of of the tile
    auto tile = [&](int i) { return few_tile(S * T, i, wave); };
    const uint32_t token_of = (threadIdx.x % FEW_TILE_PAIRS) >> 3, block_of = threadIdx.x & 7;
    uint4 q0[NP], q1[NP];
    float xs[NP], bs[NP];
    uint32_t oq[NP], os[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        const uint32_t tok = min(tile(i) % T * 16 + token_of, a.n - 1);
        oq[i] = tok * a.k + block_of * 32;
        os[i] = (tok * (a.k / 32) + block_of) * 4;
    }
    auto act_load = [&](uint32_t sb) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const uint32_t s = min(sb + tile(i) / T, sb1 - 1);
            const int8_t* const x = a.xq + s * 256;
            q0[i] = *reinterpret_cast<const uint4*>(x + oq[i]);
            q1[i] = *reinterpret_cast<const uint4*>(x + oq[i] + 16);
            xs[i] = *reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.xs + s * 8) + os[i]);
            if (W::MINS) bs[i] = *reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.bsum + s * 8) + os[i]);
        }
    };
    auto act_store = [&](uint32_t buf) {
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            const uint32_t tok = token_of, b = block_of;
            unsigned char* const t = lds + (buf * S * T + tile(i)) * FEW_TILE;
            const uint32_t q[8] = {q0[i].x, q0[i].y, q0[i].z, q0[i].w, q1[i].x, q1[i].y, q1[i].z, q1[i].w};
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                h2v v[4];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const uint32_t u = q[W::dword(g, e)] ^ 0x80808080u;
                    v[2 * e] = bytes02(u) - both(1152.f);
                    v[2 * e + 1] = bytes13(u) - both(1152.f);
                }
                *reinterpret_cast<h8v*>(t + b * FEW_BLOCK + (g * 16 + tok) * 16) = h8v{v[0][0], v[0][1], v[1][0], v[1][1], v[2][0], v[2][1], v[3][0], v[3][1]};
            }
            *reinterpret_cast<float*>(t + FEW_XS + b * 64 + tok * 4) = xs[i] * W::XS;
            if (W::MINS) {   // three bf16 parts that add up to the block sum, and a zero
                float rest = bs[i];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const uint32_t top = g < 3 ? __builtin_bit_cast(uint32_t, rest) & 0xFFFF0000u : 0u;
                    rest -= __builtin_bit_cast(float, top);
                    *reinterpret_cast<uint16_t*>(t + FEW_MIN + (g * 16 + tok) * 16 + b * 2) = static_cast<uint16_t>(top >> 16);
                }
            }
        }
    };
    // The loads stand outside every condition, past the end the last super-block again: where paths with and without a load
    // meet, the compiler's wait for an older one is a wait for all.
    typename W::W w[AHEAD];
    act_load(sb0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) W::template load<COPY>(w[i], m0, min(sb0 + i, sb1 - 1), at);
    f4v acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = f4v{0.f, 0.f, 0.f, 0.f};
    act_store(0);
    uint32_t buf = 0, sb = sb0;
    auto step = [&](auto i_) {   // one super-block; whether it was the last
        constexpr int i = decltype(i_)::value;
        if (i % S == 0) {
            // this chunk is written, and no wavefront reads the other buffer any more
            lds_barrier();
            act_load(min(sb + S, sb1 - 1));
        }
        W::template multiply<T>(w[i % AHEAD], lds + (buf * S + i % S) * T * FEW_TILE, lane, acc);
        __builtin_amdgcn_sched_barrier(0);   // the next load into the registers it has left, not into others and then copied, with a wait
        W::template load<COPY>(w[i % AHEAD], m0, min(sb + AHEAD, sb1 - 1), at);
        if (++sb == sb1) return true;
        if (i % S == S - 1) {
            buf ^= 1;
            act_store(buf);
        }
        return false;
    };
    while (true) {
        if (step(std::integral_constant<int, 0>{})) break;
        if (step(std::integral_constant<int, 1>{})) break;
        if constexpr (S > 2) {
            if (step(std::integral_constant<int, 2>{})) break;
            if (step(std::integral_constant<int, 3>{})) break;
        }
    }
    if constexpr (SWIGLU) {
        few_swiglu<T>(a, acc, second, row0, lds);
        return;
    }
    // four consecutive rows of one token per lane and tile
    const uint32_t r0 = row0 + (lane >> 4) * 4;
    if (r0 >= M.m) return;
    const int seg = r0 < M.cut[0] ? 0 : r0 < M.cut[1] ? 1 : 2;   // the cuts are multiples of four
    float* const out = M.out[seg] + blockIdx.y * a.part_stride + (r0 - (seg ? M.cut[seg - 1] : 0));
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t tok = t * 16 + (lane & 15);
        if (tok >= a.n) continue;
        const uint64_t at = static_cast<uint64_t>(tok) * M.ld[seg];
        f4v v = acc[t];
        if (a.resid && !second && seg == 0) {
            const f4v r = *reinterpret_cast<const f4v*>(a.resid + at + r0);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = r[i] + (a.resid_scale != 1.0f ? v[i] * a.resid_scale : v[i]);
        }
        *reinterpret_cast<f4v*>(out + at) = v;
    }
}
// WA, WB: the types of the two matrices
template <typename WA, typename WB, int T, bool COPY>
__global__ __launch_bounds__(FEW_WAVES * 64, 2) void gemm_few_kernel(FewArgs a) {
    __shared__ __align__(16) unsigned char lds[2 * std::max(FEW_CHUNK<WA, T>, FEW_CHUNK<WB, T>) * T * FEW_TILE];
    const bool second = blockIdx.x >= a.tiles_a;
    if (std::is_same<WA, WB>::value || !second) few_body<WA, T, COPY>(a, second, lds);
    else few_body<WB, T, COPY>(a, second, lds);
}

template <typename W, int T, bool COPY>
__global__ __launch_bounds__(FEW_WAVES * 64, 2) void gemm_few_swiglu_kernel(FewArgs a) {
    __shared__ __align__(16) unsigned char lds[2 * FEW_CHUNK<W, T> * T * FEW_TILE];
    few_body<W, T, COPY, true>(a, false, lds);
}

}  // namespace

// Super-blocks of a slice of K.  It is split where the rows leave more than a quarter of one workgroup per CU idle, down to two
// super-blocks a slice.
static uint32_t few_slice(uint32_t wgs, uint32_t nsb, uint32_t n_cu) {
    const uint32_t split = wgs * 4 >= n_cu * 3 ? 1 : std::min({(n_cu + wgs - 1) / wgs, std::max(nsb / 2, 1u), 8u});
    return (nsb + split - 1) / split;
}

bool cera_gemm_few_supports(const cera_hip_dtensor* w, uint32_t n) {
    return w && (w->dtype == CERA_HIP_Q6_K || (reinterpret_cast<uintptr_t>(w->dev) & 15) == 0) && (w->dtype == CERA_HIP_Q4_K || w->dtype == CERA_HIP_Q6_K) && w->k >= FEW_MIN_K && w->k % 256 == 0 && w->m % 4 == 0 &&
           w->m * std::max(w->row_bytes, w->stream_row_bytes) < (1ull << 32) && n >= 2 &&
           n <= FEW_MAX_TOKENS;
}

cera_hip_status cera_launch_gemm_few(cera_hip_ctx* ctx, const FewOut& oa, const FewOut* ob, const float* xs, const int8_t* xq, const float* bsum, uint32_t n,
                                     const float* resid, float resid_scale, int part_slot, FewParts* parts) {
    const cera_hip_dtensor* w = oa.w;
    if (!cera_gemm_few_supports(w, n) || (ob && (!cera_gemm_few_supports(ob->w, n) || ob->w->k != w->k || (ob->w->dtype != w->dtype && w->dtype != CERA_HIP_Q4_K))))
        return cera_fail(ctx, CERA_HIP_ERR_SHAPE, "gemm_few: bad shape");
    FewArgs a{};
    const bool copy = w->dev_stream && (!ob || ob->w->dev_stream);
    a.xq = xq; a.xs = xs; a.bsum = bsum; a.n = n; a.k = static_cast<uint32_t>(w->k);
    auto tiles = [](const cera_hip_dtensor* t) { return static_cast<uint32_t>((t->m + FEW_ROWS - 1) / FEW_ROWS); };
    a.tiles_a = tiles(w);
    const uint32_t wgs = a.tiles_a + (ob ? tiles(ob->w) : 0), nsb = a.k / 256;
    a.sb_per = few_slice(wgs, nsb, ctx->n_cu);
    uint32_t split = (nsb + a.sb_per - 1) / a.sb_per;
    uint64_t rows = 0;
    void* part_room = nullptr;
    if (split > 1) CERA_TRY(cera_scratch_if_room(ctx, part_slot, split * (w->m + (ob ? ob->w->m : 0)) * static_cast<uint64_t>(n) * 4, &part_room));
    if (!part_room) {   // the whole of K in one workgroup
        split = 1;
        a.sb_per = nsb;
    }
    float* const part = static_cast<float*>(part_room);
    auto set = [&](FewMat& m, const FewOut& o) {
        m.w = copy ? o.w->dev_stream : o.w->dev;
        m.row_bytes = static_cast<uint32_t>(copy ? o.w->stream_row_bytes : o.w->row_bytes);
        m.m = static_cast<uint32_t>(o.w->m);
        uint32_t at = 0;
        for (int s = 0; s < 3; ++s) {   // segments lie side by side in a slice, as outputs of their own would
            const uint32_t len = std::min(s < 2 && o.len[s] ? o.len[s] : m.m - at, m.m - at);
            m.out[s] = split > 1 ? part + (rows + at) * n : o.out[s];
            m.ld[s] = len;
            at += len;
            if (s < 2) m.cut[s] = at;
        }
        rows += m.m;
    };
    if (split == 1) {
        a.resid = resid; a.resid_scale = resid_scale;
    }
    set(a.a, oa);
    if (ob) set(a.b, *ob);
    a.part_stride = split > 1 ? rows * n : 0;
    *parts = FewParts{part, split, a.part_stride};
    const dim3 grid(wgs, split), block(FEW_WAVES * 64);
    auto go = [&](auto type_a, auto type_b, auto from_copy) {
        using WA = decltype(type_a);
        using WB = decltype(type_b);
        constexpr bool COPY = decltype(from_copy)::value;
        if (n <= 16) hipLaunchKernelGGL((gemm_few_kernel<WA, WB, 1, COPY>), grid, block, 0, ctx->stream, a);
        else if (n <= 32) hipLaunchKernelGGL((gemm_few_kernel<WA, WB, 2, COPY>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((gemm_few_kernel<WA, WB, 3, COPY>), grid, block, 0, ctx->stream, a);
    };
    auto of_type = [&](auto from_copy) {
        if (w->dtype == CERA_HIP_Q6_K) go(FewQ6{}, FewQ6{}, from_copy);
        else if (ob && ob->w->dtype == CERA_HIP_Q6_K) go(FewQ4{}, FewQ6{}, from_copy);
        else go(FewQ4{}, FewQ4{}, from_copy);
    };
    if (copy) of_type(std::true_type{});
    else of_type(std::false_type{});
    HIP_TRY(ctx, hipGetLastError());
    return CERA_HIP_OK;
}

cera_hip_status cera_launch_gemm_few_swiglu(cera_hip_ctx* ctx, const cera_hip_dtensor* gate, const cera_hip_dtensor* up, const float* xs, const int8_t* xq, const float* bsum,
                                            uint32_t n, int8_t* hq, float* hs, float* hbsum, bool* fused) {
    *fused = false;
    if (!cera_gemm_few_supports(gate, n) || !cera_gemm_few_supports(up, n) || up->dtype != gate->dtype || up->k != gate->k || up->m != gate->m || gate->m % 32) return CERA_HIP_OK;
    const uint32_t wgs = static_cast<uint32_t>((gate->m + FEW_ROWS / 2 - 1) / (FEW_ROWS / 2)), nsb = static_cast<uint32_t>(gate->k / 256);
    // One launch with the whole of K, or a pair that may have it in slices, with their sums and SwiGLU in launches of their own, which
    // take as long as 8, 5 or 4 super-blocks of one, two or three tiles.  Passes of two layers of hidden x ffn, one launch against a pair, in us:
    // 4096 x 14336 (whole either way) 5 tokens 262 / 267, 45 tokens 294 / 299; 4096 x 10240 (two slices, 320 workgroups on 256 CUs) 182 / 193 and 263 / 282;
    // 3072 x 8192 (two slices, 256) 156 / 157 and 223 / 218; 2304 x 6144 (three, 288) 150 / 154 and 204 / 213; 2048 x 4096 (four, 256) 136 / 137 and 188 / 180
    const uint32_t pair = 2 * static_cast<uint32_t>((gate->m + FEW_ROWS - 1) / FEW_ROWS), slice = few_slice(pair, nsb, ctx->n_cu), slices = (nsb + slice - 1) / slice, cus = ctx->n_cu;
    if ((wgs + cus - 1) / cus * nsb > (pair * slices + cus - 1) / cus * slice + (n <= 16 ? 8u : n <= 32 ? 5u : 4u)) return CERA_HIP_OK;
    FewArgs a{};
    const bool copy = gate->dev_stream && up->dev_stream;
    a.xq = xq; a.xs = xs; a.bsum = bsum; a.n = n; a.k = static_cast<uint32_t>(gate->k); a.sb_per = a.k / 256;
    a.hq = hq; a.hs = hs; a.hbsum = hbsum;
    auto set = [&](FewMat& m, const cera_hip_dtensor* w) {
        m.w = copy ? w->dev_stream : w->dev;
        m.row_bytes = static_cast<uint32_t>(copy ? w->stream_row_bytes : w->row_bytes);
        m.m = static_cast<uint32_t>(w->m);
    };
    set(a.a, gate);
    set(a.b, up);
    auto go = [&](auto type, auto from_copy) {
        using W = decltype(type);
        constexpr bool COPY = decltype(from_copy)::value;
        const dim3 grid(wgs), block(FEW_WAVES * 64);
        if (n <= 16) hipLaunchKernelGGL((gemm_few_swiglu_kernel<W, 1, COPY>), grid, block, 0, ctx->stream, a);
        else if (n <= 32) hipLaunchKernelGGL((gemm_few_swiglu_kernel<W, 2, COPY>), grid, block, 0, ctx->stream, a);
        else hipLaunchKernelGGL((gemm_few_swiglu_kernel<W, 3, COPY>), grid, block, 0, ctx->stream, a);
    };
    if (gate->dtype == CERA_HIP_Q6_K) copy ? go(FewQ6{}, std::true_type{}) : go(FewQ6{}, std::false_type{});
    else copy ? go(FewQ4{}, std::true_type{}) : go(FewQ4{}, std::false_type{});
    HIP_TRY(ctx, hipGetLastError());
    *fused = true;
    return CERA_HIP_OK;
}
