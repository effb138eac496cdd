// How a float-weight product is cut: its tile, the parts of K, and what there is room for.  Plain arithmetic on the host, without the
// device's headers.
#pragma once
#include <algorithm>
#include <cstdint>

constexpr uint32_t DENSE_PAD = 64;   // K is padded with zeros to whole 128-byte lines of bf16
static inline uint64_t dense_pad(uint64_t k) { return (k + DENSE_PAD - 1) / DENSE_PAD * DENSE_PAD; }

// the bf16 tiles, and which one a product of `groups` times m rows with n tokens takes
constexpr uint32_t DENSE_BM[] = {128, 64, 64, 256}, DENSE_BN[] = {128, 64, 32, 256};
inline int dense_shape(uint64_t m, uint64_t kp, uint64_t n, uint64_t groups, uint32_t n_cu) {
    // 256 x 256 where the outputs are at least 55 % of the rounds of one workgroup per CU: 5120 x 3072 times 2048 tokens
    // (62 %) 77 us against 86 on 128 x 128 tiles, 6176 x 4096 times 1900 (70 %) 98 / 119; below, 4096 x 18432 times 1900 (46 %)
    // 337 / 268, 3072 x 3072 times 2048 (38 %) 75 / 51.  An XCD takes whole weight tiles (dense_tile), so the rounds are those
    // of the XCD with the most: 21504 rows times 640 tokens are 252 tiles, but 33 of them on most of the XCDs' 32 CUs.
    const uint64_t per_xcd = std::max<uint64_t>(n_cu / 8, 1), most = ((m + 255) / 256 * groups + 7) / 8 * ((n + 255) / 256);
    const uint64_t rounds = (most + per_xcd - 1) / per_xcd, large = (m + 127) / 128 * ((n + 127) / 128) * groups;
    if (n > 128 && m * groups * n * 20 >= rounds * per_xcd * 8 * 65536 * 11) return 3;
    if (n > 64 && (large >= n_cu || (kp >= 8192 && large * 4 >= n_cu))) return 0;
    return n > 32 ? 1 : 2;
}
// Parts of K in which 256 x 256 tiles take a product whose sums go through the reduction anyway in place of 128 x 128 tiles with
// `split` parts, or 0: the fewest, up to four of at least eight steps of 64, whose tiles are at least 55 % of their rounds on the
// fullest XCD, as above, if those rounds cost less.  A round of the larger tiles, one a CU, is twice the work of one of the smaller, two
// a CU and counted over the chip, at about 1.3 times the rate: by that, they are 1.3 / 2 * parts * rounds128 / (split * rounds) times as
// fast, and have to be 1.07 times so.  At 1792 to 4096 rows and 200 to 2048 tokens that comes to 1.3, 1.7 or 1.95, or to 0.98, which
// stays.  Passes of two layers on the smaller tiles and by the rule: 1.3, 4096 wide, 1409 tokens (384 workgroups whole; 96 x 2) 1492 /
// 1448 us, 3328 wide, 1459 (312 x 2; 78 x 2) 1276 / 1174, 4096 wide, 617 (160 x 4; 48 x 4) 909 / 872; 1.7, 3584 wide, 796 (196 x 3; 56 x 4)
// 982 / 890; 1.95, 3584 wide, 1224 (280 x 2; 70 x 3) 1293 / 1100; 24 sizes in all, 2.3 to 15 % faster each.  2048 wide times 2048 tokens
// (256 x 2; 64 x 3: 0.98) takes 1.5 % longer on the larger tiles.  Product and reduction alone: 3072 x 8192 times 2048 tokens
// 140 + 47 -> 105 + 52 us, 3072 x 3072 62 + 47 -> 50 + 52.
inline uint32_t dense_wide_parts(uint64_t m, uint64_t n, uint32_t steps, uint64_t wgs, uint32_t split, uint32_t n_cu) {
    const uint64_t per_xcd = std::max<uint64_t>(n_cu / 8, 1), most = ((m + 255) / 256 + 7) / 8 * ((n + 255) / 256);
    const uint64_t rounds128 = (wgs * split + 2 * n_cu - 1) / (2 * n_cu);
    for (uint32_t parts = 2; n > 128 && parts <= 4 && steps / parts >= 8; ++parts) {
        const uint64_t rounds = (most * parts + per_xcd - 1) / per_xcd;
        if (m * n * parts * 20 >= rounds * per_xcd * 8 * 65536 * 11) return parts * rounds128 * 20 >= split * rounds * 33 ? parts : 0;
    }
    return 0;
}
// The same by an estimate, from 2048 columns on, the shortest measured: for products whose sums need no reduction, and for those whose
// sums go through it anyway (`apart`) where the rule above has no parts.  The number of parts, from K whole to eight of at least eight
// steps, whose estimate is least, if that is below 0.92 of the one of 128 x 128 tiles with `split` parts, else 0.  In us, from 48 products
// of 1024 to 6144 rows, 2048 to 18432 columns and 200 to 2048 tokens, most within 15 %: 256 x 256 tiles 1.1 a step and round and, as power
// is what they run out of, up to 1.65 with how full the rounds are; 128 x 128 ones 1.0, in rounds of two a CU; partial sums 3.5 TB/s and 2
// for their launch, and 2 more for parts of the larger tiles, which have to earn their workspace.  K whole on the larger tiles counts no
// sums, also where they go through the reduction: with them the choice would be another at 96 of 1.5 million sizes, five parts in place of
// one at 8224 to 8800 rows, 14912 columns and 1029 to 1110 tokens, and two-layer passes there 0 to 1.6 % slower (8256 wide, 1040 tokens
// 2058 -> 2086 us, 8704, 1050 2155 -> 2165, 8448, 1090 2154 -> 2147).  On 128 x 128 tiles and by the rule: 4096 x 18432
// times 1900 / 2048 tokens (2 parts) 342 -> 259 and 344 -> 265 us, 3072 x 11264 times 1900 / 1024 / 700 (2, 4, 5) 196 -> 152, 135 -> 89
// and 98 -> 74, 6144 x 8192 times 700 (3) 139 -> 85, 6144 x 4096 times 1400 (1) 104 -> 89; of 80 sizes the worst 1 % behind.  Refused: 5120 x
// 8192 times 1400 130 (153 in 3), 4096 x 4096 times 1900 68 (77 in 2), 3072 x 2048 times 1568 46.5 (49 in 2).  64 x 64 tiles, where they
// are taken, are ahead at all of 36 sizes.  With streams, two-layer passes of 14 sizes, before and by the rule: 3072 wide, 8192 inside, 690
// tokens (5 parts) 676 -> 636 us, 1450 (2) 993 -> 924; 4096 / 14336, 520 (5) 895 -> 822, 380 (8) 691 -> 639; 2048 / 8192, 850 (8) 502 -> 490.
inline uint32_t dense_wide_split(uint64_t m, uint64_t n, uint32_t steps, uint64_t wgs, uint32_t split, bool apart, uint32_t n_cu) {
    const uint64_t per_xcd = std::max<uint64_t>(n_cu / 8, 1), most = ((m + 255) / 256 + 7) / 8 * ((n + 255) / 256), tiles = (m + 255) / 256 * ((n + 255) / 256);
    auto sums = [&](uint32_t parts) { return parts > 1 || apart ? 2.0 + parts * m * n * 4 / 3.5e6 : 0.0; };
    const uint64_t rounds128 = (wgs * split + 2 * n_cu - 1) / (2 * n_cu);
    double best = 0.92 * (4.0 + rounds128 * ((steps + split - 1) / split) * 1.0 + sums(split));
    uint32_t take = 0;
    for (uint32_t parts = 1; n > 128 && steps >= 32 && parts <= 8; ++parts) {
        const uint32_t per = (steps + parts - 1) / parts;
        if (per < 8 || (steps + per - 1) / per != parts) continue;
        const uint64_t rounds = (most * parts + per_xcd - 1) / per_xcd;
        const double fill = static_cast<double>(tiles * parts) / (rounds * per_xcd * 8), t = 8.0 + rounds * per * (1.1 + 0.55 * fill) + (parts > 1 ? 2.0 + sums(parts) : 0.0);
        if (t < best) { best = t; take = parts; }
    }
    return take;
}
// How a product is cut: its tile, the parts of K, and whether its sums go through the reduction.
struct DensePlan {
    int shape;
    uint32_t split;
    bool apart;   // even if K is whole
    bool wide;    // 256 x 256 tiles by dense_wide_parts or dense_wide_split
    uint64_t sums(uint64_t m, uint64_t n) const { return split > 1 || apart ? split * n * m * sizeof(float) : 0; }   // bytes of partial sums
};
// streams: of DENSE_STREAMS, else 0.  wide: 256 x 256 tiles may take in parts of K what 128 x 128 ones would
inline DensePlan dense_plan(uint64_t m, uint64_t kp, uint64_t n, uint64_t groups, uint32_t streams, bool f32, bool wide, uint32_t n_cu) {
    DensePlan p{f32 ? 2 : dense_shape(m, kp, n, groups, n_cu), 1, false, false};
    const uint64_t bm = f32 ? 64 : DENSE_BM[p.shape], bn = f32 ? 64 : DENSE_BN[p.shape], wgs = (m + bm - 1) / bm * ((n + bn - 1) / bn) * groups;
    const uint32_t steps = static_cast<uint32_t>(kp / DENSE_PAD);
    // two workgroups per CU; three quarters of that are left alone on large tiles, whose partial sums cost more than the idle
    // quarter: 3072 x 3072 times 2048 tokens (384) 51 us whole, 50 + 24 in two parts
    const uint32_t want_wgs = 2 * n_cu;
    if (p.shape != 3 && wgs * 4 < want_wgs * (p.shape == 0 ? 3ull : 4ull) && groups == 1) p.split = static_cast<uint32_t>(std::min<uint64_t>({(want_wgs + wgs - 1) / wgs, steps / 4, 16}));
    if (p.split < 1) p.split = 1;
    // streams on large tiles, and any number of them but four: through the reduction, whose threads hold little else and walk
    // along the rows.  3072 x 8192 times 2048 tokens, four streams: 118 + 45 us, as the tiles' own epilogue 230
    p.apart = streams && (streams != 4 || p.shape == 0 || p.shape == 3);
    uint32_t parts = 0;
    if (wide && p.shape == 0 && groups == 1) {
        if (p.apart) parts = dense_wide_parts(m, n, steps, wgs, p.split, n_cu);
        if (!parts) parts = dense_wide_split(m, n, steps, wgs, p.split, p.apart, n_cu);
    }
    if (parts) {
        p.shape = 3;
        p.split = parts;
        p.wide = true;
    }
    const uint32_t per = (steps + p.split - 1) / p.split;
    p.split = (steps + per - 1) / per;
    return p;
}
// The same for what there is room for, room(bytes) saying so; a plan without sums does not ask.  Where the larger tiles' parts do not fit,
// the smaller tiles', which may be fewer; without room for those either, the whole of K in one workgroup, four streams by small tiles'
// own lanes.
template <class Room> inline DensePlan dense_plan_in(uint64_t m, uint64_t kp, uint64_t n, uint64_t groups, uint32_t streams, bool f32, uint32_t n_cu, Room&& room) {
    DensePlan p = dense_plan(m, kp, n, groups, streams, f32, true, n_cu);
    if (!p.sums(m, n) || room(p.sums(m, n))) return p;
    if (p.wide) {
        p = dense_plan(m, kp, n, groups, streams, f32, false, n_cu);
        if (!p.sums(m, n) || room(p.sums(m, n))) return p;
    }
    p.split = 1;
    if (p.apart && streams == 4) { p.shape = 1; p.apart = false; }
    return p;
}
