// What a dense product asks of its workspace (csrc/dense_plan.h), over sizes, epilogues that need the reduction and rooms: a plan
// without partial sums asks for nothing, and one with them has been given all of them.
#include <cstdio>
#include <initializer_list>

#include "dense_plan.h"

int main() {
    uint64_t plans = 0, whole = 0;
    for (uint64_t m : {50, 130, 1100, 1792, 2304, 3001, 3072, 4096, 6176, 16400})
        for (uint64_t k : {64, 1030, 2060, 4096, 8264, 18432})
            for (uint64_t n : {1, 40, 129, 200, 616, 700, 1290, 1537, 1900, 2048})
                for (uint32_t streams : {0, 1, 3, 4})
                    for (int f32 : {0, 1}) {
                        const uint64_t one = m * n * 4;
                        for (uint64_t room : {uint64_t(0), uint64_t(1), one - 1, one, 2 * one - 1, 2 * one, 5 * one - 1, uint64_t(1) << 62}) {
                            uint64_t given = 0;
                            const char* bad = nullptr;
                            const DensePlan p = dense_plan_in(m, dense_pad(k), n, 1, streams, f32, 256, [&](uint64_t bytes) {
                                if (bytes == 0) bad = "asks for no bytes";
                                given = bytes <= room ? bytes : 0;
                                return bytes <= room;
                            });
                            const uint64_t sums = p.sums(m, n);
                            if (!bad && given != sums && !(given == 0 && p.apart)) bad = "is given something else than its sums";   // (apart: it cannot do without)
                            if (bad) {
                                std::printf("%llu x %llu times %llu, streams %u, f32 %d, room %llu: the plan (shape %d, %u parts, sums %llu) %s\n", (unsigned long long)m,
                                            (unsigned long long)k, (unsigned long long)n, streams, f32, (unsigned long long)room, p.shape, p.split, (unsigned long long)sums, bad);
                                return 1;
                            }
                            ++plans;
                            whole += room < (uint64_t(1) << 62) && !sums && dense_plan(m, dense_pad(k), n, 1, streams, f32, true, 256).sums(m, n);
                        }
                    }
    std::printf("%llu plans, %llu of them whole for want of room\n", (unsigned long long)plans, (unsigned long long)whole);
}
