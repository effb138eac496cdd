// How attention's keys are cut (csrc/attn_plan.h), over shapes, lengths and batches, with room for more parts than a call needs and without:
// the parts cover the keys, room is asked for only where there are more, and a refusal leaves the parts of a context without any.
#include <cstdio>
#include <initializer_list>

#include "attn_plan.h"

int main() {
    struct Shape { uint32_t heads, kv; };
    uint64_t calls = 0, asked = 0;
    for (const Shape s : {Shape{32, 8}, Shape{8, 1}, Shape{16, 16}, Shape{24, 8}, Shape{28, 4}, Shape{12, 2}, Shape{20, 4}, Shape{32, 16}, Shape{64, 8}})
        for (uint64_t first : {1, 30, 128, 700, 901, 3000, 12345, 100000})
            for (uint32_t n : {1, 2, 7, 8, 12, 15, 16, 33, 45, 64, 100, 160, 257, 1024, 2048})
                for (uint32_t splits : {0u, 6u})
                    for (bool f16 : {false, true}) {
                        const uint64_t last = first + n - 1;
                        uint32_t wanted = 0, questions = 0;
                        const AttnCut with = attn_cut(s.heads, s.kv, last, n, splits, f16, 256, [&](uint32_t parts) { wanted = parts; ++questions; return true; });
                        const AttnCut without = attn_cut(s.heads, s.kv, last, n, splits, f16, 256, [](uint32_t) { return false; });
                        ++calls;
                        asked += questions;
                        const char* bad = nullptr;
                        for (const AttnCut& c : {with, without}) {
                            const uint64_t keys = attn_is_batch(n) ? c.part_keys : 8ull * c.S * c.chunks_per_part;
                            if (c.n_parts == 0 || c.n_parts > ATTN_MAX_PARTS || c.n_parts * keys < last || (c.n_parts - 1) * keys >= last) bad = "parts that are not the keys";
                            if (attn_is_batch(n) && (c.part_keys == 0 || c.part_keys % 32)) bad = "a part that is not whole tiles";
                        }
                        if (questions > 1 || (questions && (wanted <= without.n_parts || wanted != with.n_parts))) bad = "a question that is not about more parts";
                        if (!questions && (with.n_parts != without.n_parts || with.part_keys != without.part_keys || with.chunks_per_part != without.chunks_per_part)) bad = "another cut without a question";
                        if (questions && (n < 8 || (splits && n < 16))) bad = "a question of a call that has the parts it asks for";
                        if (attn_is_batch(n) && without.part_keys != (last <= 1024 ? 128 : (last + (n >= 1024 ? 3 : 7)) / (n >= 1024 ? 4 : 8) / 32 * 32 + ((last + (n >= 1024 ? 3 : 7)) / (n >= 1024 ? 4 : 8) % 32 ? 32 : 0)))
                            bad = "without room, other parts than 128 keys or the eighth (fourth) of them";
                        if (bad) {
                            std::printf("%u / %u heads, %u queries behind %llu keys, f16 %d, splits %u: %s (%u parts with room, %u without, asked for %u)\n", s.heads, s.kv, n,
                                        (unsigned long long)first, f16, splits, bad, with.n_parts, without.n_parts, wanted);
                            return 1;
                        }
                    }
    std::printf("%llu calls, %llu questions\n", (unsigned long long)calls, (unsigned long long)asked);
    return asked == 0;
}
