// What the cuts of attention's keys (csrc/attn_plan.h) do to the chip, over shapes, lengths and batches: a batch that takes more parts than it
// needs still has at most a workgroup a CU, and 8 to 15 queries take more where that was measured to be far faster, and not where it was slower.
#include <cstdio>
#include <initializer_list>

#include "attn_plan.h"

int main() {
    struct Shape { uint32_t heads, kv; };
    constexpr uint32_t CUS = 256;
    uint64_t more = 0;
    for (const Shape s : {Shape{32, 8}, Shape{8, 1}, Shape{16, 16}, Shape{24, 8}, Shape{28, 4}, Shape{12, 2}, Shape{24, 6}, Shape{24, 12}, Shape{40, 20}})
        for (uint64_t first : {1, 30, 128, 700, 901, 3000, 12345, 100000})
            for (uint32_t n : {16, 33, 45, 65, 100, 129, 160, 200, 257, 400})
                for (bool f16 : {false, true}) {
                    auto cut = [&](bool room) { return attn_cut(s.heads, s.kv, first + n - 1, n, 0, f16, CUS, [=](uint32_t) { return room; }); };
                    const uint32_t few = cut(false).n_parts, parts = cut(true).n_parts;
                    if (parts == few) continue;
                    ++more;
                    if ((n + 31) / 32 * s.kv * parts > CUS) {
                        std::printf("%u / %u heads, %u queries behind %llu keys: %u parts of %u blocks on %u CUs\n", s.heads, s.kv, n, (unsigned long long)first, parts,
                                    (n + 31) / 32 * s.kv, CUS);
                        return 1;
                    }
                }
    struct Measured { uint32_t heads, kv; uint64_t first; uint32_t n; bool f16, more; };   // us a layer by the parts of before and by three workgroups a CU
    for (const Measured m : {Measured{32, 8, 901, 12, false, true},      // 35.2, 21.9
                             Measured{16, 16, 3001, 10, false, true},    // 51.3, 29.4
                             Measured{32, 16, 901, 12, false, true},     // 35.5, 20.3
                             Measured{32, 4, 3001, 8, false, false},     // 22.8, 28.9
                             Measured{8, 1, 12001, 8, false, false},     // 22.6, 31.2
                             Measured{28, 4, 301, 13, false, false},     // 32 % slower
                             Measured{32, 4, 901, 10, true, false},      // 19.6, 24.0
                             Measured{32, 16, 12001, 10, true, false},   // 85.3, 106.6
                             Measured{32, 8, 301, 15, false, false}}) {  // 13.4, 15.3
        auto cut = [&](bool room) { return attn_cut(m.heads, m.kv, m.first + m.n - 1, m.n, 0, m.f16, CUS, [=](uint32_t) { return room; }); };
        if ((cut(true).n_parts > cut(false).n_parts) != m.more) {
            std::printf("%u / %u heads, %u queries behind %llu keys: %u parts, %u without room\n", m.heads, m.kv, m.n, (unsigned long long)m.first, cut(true).n_parts, cut(false).n_parts);
            return 1;
        }
    }
    std::printf("%llu batches with more parts\n", (unsigned long long)more);
    return more == 0;
}
