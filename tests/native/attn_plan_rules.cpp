// What the cuts of attention's keys (csrc/attn_plan.h) do to the chip, over shapes, lengths and batches: a batch that takes more parts than it
// needs still has at most a workgroup a CU.
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
    std::printf("%llu batches with more parts\n", (unsigned long long)more);
    return more == 0;
}
