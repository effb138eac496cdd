// How attention's keys are cut into parts, whose results a merge adds up.  Plain arithmetic on the host, without the device's headers.
#pragma once
#include <algorithm>
#include <cstdint>

#include "attn_types.h"

struct AttnCut {
    uint32_t n_parts = 0;
    uint32_t part_keys = 0;         // a batch of queries: keys of a part
    uint32_t chunks_per_part = 0;   // fewer queries: chunks of 8 S keys of a part
    uint32_t S = 1;
    uint32_t Gw = 0;                // and query heads of a wavefront
};
inline bool attn_is_batch(uint32_t n_queries) { return n_queries >= 16; }

// last_len: keys that the last query sees.  n_splits: parts that the caller asks for, or 0.  room(n) says whether the context has room for
// the results of n parts; it is asked only where more parts than a call needs make it faster.
template <class Room>
inline AttnCut attn_cut(uint32_t n_heads, uint32_t n_kv_heads, uint64_t last_len, uint32_t n_queries, uint32_t n_splits, bool kv_f16, uint32_t n_cu, Room room) {
    AttnCut c;
    const uint32_t G = n_heads / n_kv_heads;
    c.Gw = G;
    if (attn_is_batch(n_queries)) {
        // Parts of at most 128 keys while the context is short, about eight (four) parts per query block beyond that.
        const uint64_t want = n_queries >= 1024 ? 4 : 8;   // many query blocks fill the chip with fewer parts
        c.part_keys = last_len <= 1024 ? 128u : static_cast<uint32_t>(((last_len + want - 1) / want + 31) / 32 * 32);
        c.n_parts = static_cast<uint32_t>((last_len + c.part_keys - 1) / c.part_keys);
        // Few query blocks: as many parts as leave every CU at most one workgroup, down to a tile of 32 keys.  A part's tiles are a chain of
        // loads, splits and products of about 3 us each, and a second workgroup a CU gains less than its sums cost the merge.
        // Two layers, 32 / 8 heads of 128: 45 queries behind 700 keys (128 keys a part before, 64 now) 294 -> 289 us, behind 12000
        // 490 -> 433, 30 behind 3000 294 -> 264; by two workgroups a CU 286, 427 and 275.  A few workgroups more than CUs are a second round of
        // them: 160 queries behind 12000 keys, 32 / 4 heads of 128, 132 us a layer by the eight parts, 145 by 13 (260 workgroups), 111 by 12; 200
        // queries 186 by ten, 139 by nine.  Over eight shapes, 16 to 257 queries behind 100 to 12000 keys, both caches, no slower than by the eight
        // beyond noise, and 23 % less in the mean.  At most 64 parts: the merge adds them in order.
        const uint64_t blocks = (n_queries + 31ull) / 32 * n_kv_heads, parts = std::min<uint64_t>(std::max<uint64_t>(n_cu / blocks, 1), 64);
        const uint32_t keys = std::min(c.part_keys, static_cast<uint32_t>(((last_len + parts - 1) / parts + 31) / 32 * 32));
        const uint32_t n = static_cast<uint32_t>((last_len + keys - 1) / keys);
        if (n > c.n_parts && room(n)) {
            c.part_keys = keys;
            c.n_parts = n;
        }
        return c;
    }
    // positions per chunk (8 S): one 8-key chunk per wavefront while the context is short (a single
    // memory round trip, many wavefronts), longer chunks once there is plenty of work.  Measured on
    // the 32/8/128 shape over rotating caches; with a kv head's query heads split over two
    // wavefronts (attn_launch_partials) 32-key chunks are best from 1024 keys up to where the split
    // ends: 64-key chunks take one wavefront per SIMD (registers) and lose 2-3 us from 8k to 16k keys.
    // heads per wavefront: attn_launch_partials has the reasons
    if (G == 8 || (G == 4 && last_len < (kv_f16 ? 32768u : 16384u))) c.Gw = G / 2;
    else if (G == 6) c.Gw = 2;
    else if (G == 3 || G == 5 || G == 7) c.Gw = 1;
    const bool split_heads = c.Gw != G;
    if (split_heads) c.S = last_len >= ATTN_FUSED_NEW_KV_MAX_KEYS ? 4 : 1;
    else c.S = last_len >= 8192 ? 8 : (last_len >= 2048 ? 4 : (last_len >= ATTN_FUSED_NEW_KV_MAX_KEYS ? 2 : 1));
    if (c.Gw == 8 && c.S == 8) c.S = 4;   // eight heads x 64 positions per chunk does not fit the register file
    const uint32_t n_chunks = static_cast<uint32_t>((last_len + 8 * c.S - 1) / (8 * c.S));
    // workgroups, of four wavefronts, where a part has so many chunks
    auto workgroups = [&](uint64_t cpp) { return ((n_chunks + cpp - 1) / cpp + 3) / 4 * n_kv_heads * (G / c.Gw) * n_queries; };
    // chunks per part where a CU's share is waves_per_cu wavefronts, and a round takes per_round workgroups a CU
    auto chunks = [&](uint32_t waves_per_cu, uint32_t per_round) {
        // parts (wavefronts) per (query, kv head): enough to fill the chip ~4 waves per CU deep
        // (more parts make the partial kernel shorter but the merge longer: measured best from 2k
        // to 128k keys with an f32 cache), but at least one chunk each and at most ATTN_MAX_PARTS
        const uint32_t want_parts = std::min<uint32_t>(n_splits ? n_splits : std::max(1u, n_cu * waves_per_cu / (n_kv_heads * n_queries)), ATTN_MAX_PARTS);
        uint32_t chosen = std::max(1u, (n_chunks + want_parts - 1) / want_parts);
        if (n_splits) return chosen;
        // Between the lengths where that divides evenly the chip runs a ragged last round.  A
        // wavefront's time goes with its chunks, the launch's with the rounds of workgroups a CU
        // runs (one workgroup per CU and round with an f32 cache, which is bound by bytes; two with
        // an f16 cache or eight heads per kv head): from the nominal count down to a quarter of it, take the parts that
        // minimise chunks x rounds.  Of equals an f32 cache takes the one with more parts, an f16
        // cache the one with fewer -- either way the one nearer two workgroups per CU.
        // 9216 keys, f32: 31.2 -> 21.9 us together with the kernel's launch-index mapping, 13824:
        // 37.2 -> 27.9; f16: 8192 keys 16.3 -> 13.9.  Within 4 % of the best (chunk, parts) pair
        // of a sweep at every length from 1k to 16k keys (f32) and of a parts sweep (f16).
        uint64_t best = ~0ull;
        const uint32_t first = chosen;
        for (uint32_t cpp = first; cpp <= n_chunks; ++cpp) {
            if (cpp > first && static_cast<uint64_t>((n_chunks + cpp - 1) / cpp) * 4 < want_parts) break;
            const uint64_t round = static_cast<uint64_t>(n_cu) * per_round, cost = cpp * ((workgroups(cpp) + round - 1) / round);
            if (cost < best || (kv_f16 && cost == best)) { best = cost; chosen = cpp; }
        }
        return chosen;
    };
    // a half cache is nearer VALU-bound: more wavefronts help.  Two workgroups a round where the kernel is bound by its own
    // instructions (an f16 cache, eight heads per kv head), one where it is bound by bytes
    c.chunks_per_part = chunks(kv_f16 ? 8 : 4, kv_f16 || G == 8 ? 2 : 1);
    c.n_parts = (n_chunks + c.chunks_per_part - 1) / c.chunks_per_part;
    if (n_queries >= 8 && !n_splits) {
        // From eight queries on all but the first find the rows in the L2, and the launch is a chain of loads: three workgroups a CU,
        // where that is far faster by an estimate, in keys: a part's, once for the launch's start and its end each and once for each
        // workgroup of a CU, and 32.  The line is five thirds: 32 / 8 heads of 128, 12 queries behind 900 keys, f32, 35.2 -> 21.9 us a layer (the
        // pass of two layers 275 -> 240); of 32 / 4 heads, 8 behind 3000, where it would be 22.8 -> 28.9, the cut stays.  Thirteen shapes of 1 to 32
        // key heads, 8 to 15 queries behind 60 to 12000 keys, both caches: 5 % less time in the mean, up to 63 %, and none slower beyond noise; with
        // three workgroups everywhere 7 % less, but up to 32 % more, and more than 3 % in a sixth of 660 calls.  Five queries are level.
        const uint32_t more = chunks(12, 3), n = (n_chunks + more - 1) / more;
        auto cost = [&](uint32_t cpp) { return 32 + 8ull * c.S * cpp * (2 + (workgroups(cpp) + n_cu - 1) / n_cu); };
        if (n > c.n_parts && cost(c.chunks_per_part) * 3 > cost(more) * 5 && room(n)) {
            c.chunks_per_part = more;
            c.n_parts = n;
        }
    }
    return c;
}
