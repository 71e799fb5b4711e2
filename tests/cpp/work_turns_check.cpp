// Every chunk goes to one wave, once, and a wave that has had its last chunk gets none however often it asks again.
#include "work_turns.hpp"

#include <cstdio>
#include <vector>

using namespace eleven;

static int cover(uint32_t waves, uint32_t chunks) {
    std::vector<uint8_t> taken(chunks, 0);
    int bad = 0;
    for (uint32_t w = 0; w < waves && w < chunks; w++) {
        WorkTurns t(w);
        for (uint32_t c; (c = t.next(waves, chunks, w)) < chunks;) bad += taken[c]++ != 0;
    }
    for (uint8_t k : taken) bad += k != 1;
    if (bad) printf("%u waves, %u chunks: %d chunks not taken once\n", waves, chunks, bad);
    return bad != 0;
}

int main() {
    int bad = 0;
    for (uint32_t waves : {1u, 2u, 3u, 5u, 7u, 8u, 9u, 64u, 100u, 8191u, 8192u})
        for (uint32_t chunks : {1u, 2u, 7u, 8u, 9u, 63u, 64u, 65u, 8191u, 8192u, 8193u, 16384u, 40961u, 262144u})
            bad += cover(waves, chunks);
    for (uint32_t waves : {512u, 8191u, 8192u}) {
        WorkTurns t(3);
        for (uint64_t k = 0, given = 0; k < 3 * ((1ull << 32) / waves); k++) {
            given += t.next(waves, 5 * waves + 4, 3) < 5 * waves + 4;
            if (k > 5 && given != 6) {
                bad++;
                printf("%u waves: a chunk more at call %llu\n", waves, (unsigned long long)k);
                break;
            }
        }
    }
    printf("bad=%d\n", bad);
    return bad != 0;
}
