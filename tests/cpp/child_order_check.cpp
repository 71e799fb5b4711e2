// The order of a BVH4 visit's children on the stack: whatever signs the zeros among the slab distances have, the four
// children get four different rows, the hit ones the lowest, far to near.  By lanes (childRows) and by quads
// (nearerKey), over distances from -inf to +inf with both zeros and denormals.
#include "child_order.hpp"

#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

using namespace eleven;

static uint32_t bits(float f) {
    uint32_t u;
    std::memcpy(&u, &f, 4);
    return u;
}

int main() {
    const float inf = INFINITY;
    const float set[] = {-inf, -1.f, -1e-45f, -0.f, 0.f, 1e-45f, 1e-38f, 0.5f, 1.f, 3e38f, inf};
    const int N = sizeof set / sizeof *set;
    std::mt19937 g(1);
    int bad = 0;
    for (int it = 0; it < 2000000 && bad < 10; it++) {
        float tn[4];
        uint32_t miss[4], key[4], above[4];
        for (int i = 0; i < 4; i++) {
            const float tz = set[3 + g() % (N - 3)];   // clamped from below: -0 and up
            const bool zeros = g() % 2;
            tn[i] = entryDistance(zeros ? -0.f : set[g() % N], zeros ? -0.f : set[g() % N], zeros ? -0.f : tz);
            if (bits(tn[i]) >> 31) bad++, printf("entry distance %g has its sign set\n", tn[i]);
            miss[i] = g() % 3 ? 0u : ~0u;
            key[i] = childKey(bits(tn[i]), miss[i]);
        }
        childRows(key, above);
        uint32_t hits = 0, seen = 0;
        for (int i = 0; i < 4; i++) hits += !miss[i];
        int at[4] = {0, 0, 0, 0};
        for (int i = 0; i < 4; i++) {
            seen |= 1u << above[i];
            if (above[i] < 4) at[above[i]] = i;
            if (!miss[i] && above[i] >= hits) bad++, printf("hit child in row %u of %u\n", above[i], hits);
        }
        if (seen != 15) bad++, printf("rows %u %u %u %u\n", above[0], above[1], above[2], above[3]);
        for (uint32_t r = 1; r < hits && seen == 15; r++)
            if (tn[at[r]] > tn[at[r - 1]]) bad++, printf("rows not far to near\n");
        // quads: as visitQuad
        uint32_t rows = 0;
        for (uint32_t j = 0; j < 4; j++) {
            if (miss[j]) continue;
            uint32_t nearer = 0;
            for (uint32_t k = 1; k < 4; k++)
                nearer += nearerKey(childKeyOfLane(bits(tn[j ^ k]), j ^ k, !miss[j ^ k]), childKeyOfLane(bits(tn[j]), j, true));
            rows |= 1u << (hits - 1 - nearer);
        }
        if (rows != (1u << hits) - 1) bad++, printf("quad rows %x of %u\n", rows, hits);
        // whatever sign a distance has: by quads
        for (uint32_t j = 0; j < 4; j++)
            if (childKeyOfLane(bits(-0.f), j, true) < 0) bad++, printf("quad key of -0 below 0\n");
    }
    printf("bad=%d\n", bad);
    return bad != 0;
}
