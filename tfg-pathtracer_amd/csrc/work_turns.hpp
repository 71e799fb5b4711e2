// Chunks of a queue handed to the waves of a launch in turn, shared by the
// device traversal and its host check.
#pragma once

#include <stdint.h>

#ifndef EL_HD
#ifdef __HIPCC__
#define EL_HD __host__ __device__
#else
#define EL_HD
#endif
#endif

namespace eleven {

// One wave's chunks: in every turn each of `waves` waves takes one, and moves
// on by 5/8 of the waves for the next (WorkSource, pt_device.hpp), except in
// a last turn that is not full, which the waves that start last miss.
struct WorkTurns {
    uint32_t turn = 0;   // first chunk of the next turn
    uint32_t place;      // this wave's place in it
    EL_HD explicit WorkTurns(uint32_t first) : place(first) {}
    // The wave's next chunk, or one past the last.  Asked again after that it
    // stays where it is: counting on, 32 bits come back to the first chunk after
    // 2^32 / waves calls, which a ray that visits millions of leaves can take.
    EL_HD uint32_t next(uint32_t waves, uint32_t chunks, uint32_t first) {
        const uint32_t c = turn + place;
        if (c >= chunks) return chunks;
        turn += waves;
        place += (waves * 5) >> 3;
        place -= place >= waves ? waves : 0u;
        if (chunks - turn < waves) place = first;
        return c;
    }
};

}  // namespace eleven
