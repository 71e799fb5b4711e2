// The paths of an adjoint's generation: its memory within the bound at every depth, and its growth within a quarter of
// what is free, whatever the context's queues hold already.
#include "adjoint_plan.hpp"

#include <cstdio>

using namespace eleven;

int main() {
    int bad = 0;
    const uint64_t slack = 524288 + 8 * 257;
    for (uint64_t depth = 1; depth <= 16; depth++)
        for (uint64_t total : {64ull, 65536ull, 4194304ull, 10485760ull, 1ull << 30})
            for (uint64_t held : {0ull, 1000000ull, 1ull << 27})
                for (uint64_t heldHits : {0ull, 1ull << 28})
                    for (int recorded = 0; recorded < 2; recorded++)
                        for (uint64_t freeB : {100ull << 20, 1ull << 30, 280ull << 30}) {
                            AdjointMemory m{176, 64, slack, recorded ? 0 : 16 * depth + 4, held, held ? held + slack : 0, heldHits};
                            int asked = 0;
                            const uint64_t paths = adjointPaths(m, total, [&] { asked++; return freeB; });
                            const uint64_t least = total < kAdjointMinPaths ? total : kAdjointMinPaths;
                            if (paths < least || paths > total) bad++, printf("%llu paths\n", (unsigned long long)paths);
                            if (m.bytes(paths) > kAdjointBytes) bad++, printf("depth %d: %llu bytes\n", (int)depth, (unsigned long long)m.bytes(paths));
                            if (m.growth(paths) > freeB / 4 && paths > least) bad++, printf("grows by %llu of %llu\n", (unsigned long long)m.growth(paths), (unsigned long long)freeB);
                            if (asked != (asked != 0) || (asked && m.growth(total < 64 ? total : paths) == 0 && paths == total)) bad++;
                            // no less than it could be: the next 128 paths pass a bound
                            if (paths + 128 <= total && m.bytes(paths + 128) <= kAdjointBytes && m.growth(paths + 128) <= freeB / 4)
                                bad++, printf("%llu paths are too few\n", (unsigned long long)paths);
                        }
    printf("bad=%d\n", bad);
    return bad != 0;
}
