// How many paths a generation of el_adjoint holds.
#pragma once

#include <algorithm>
#include <cstdint>

namespace eleven {

// Device memory for a generation of paths (queues, path state and, unless the
// paths are recorded, their hits and shadow answers), so that the adjoint's memory
// does not grow with the pixels and samples: 5.8 M paths at depth 6, enough to
// fill the GPU.
constexpr uint64_t kAdjointBytes = 2ull << 30;
constexpr uint64_t kAdjointMinPaths = 1u << 16;

struct AdjointMemory {
    uint64_t entryBytes, slotBytes;   // of a queue entry and a path slot (WfBuffers)
    uint64_t slackEntries;            // queue entries beyond one a path
    uint64_t hitBytes;                // a path's hits and shadow answers, 0 if recorded
    uint64_t heldSlots, heldEntries;  // what the queues hold already
    uint64_t heldHits;                // bytes of the hits' buffers

    uint64_t bytes(uint64_t paths) const {
        return paths * (slotBytes + entryBytes + hitBytes) + slackEntries * entryBytes;
    }
    // What a generation of `paths` needs beyond the buffers there are.
    uint64_t growth(uint64_t paths) const {
        auto over = [](uint64_t need, uint64_t held) { return need > held ? need - held : 0; };
        const bool fits = paths <= heldSlots && paths + slackEntries <= heldEntries;
        return (fits ? 0
                     : over(paths * slotBytes, heldSlots * slotBytes) +
                           over((paths + slackEntries) * entryBytes, heldEntries * entryBytes)) +
               over(paths * hitBytes, heldHits);
    }
};

// Paths of a generation: of `total`, what kAdjointBytes hold, or what grows the
// buffers by a quarter of the free memory (as a render's queues) if that is
// less; kAdjointMinPaths at least.  free() is asked only if something has to grow.
template <class Free>
uint64_t adjointPaths(const AdjointMemory& m, uint64_t total, Free&& free) {
    const uint64_t fixed = m.bytes(0);
    uint64_t paths = (kAdjointBytes - std::min(kAdjointBytes, fixed)) / (m.slotBytes + m.entryBytes + m.hitBytes);
    paths = std::min(total, std::max(kAdjointMinPaths, paths));
    if (m.growth(paths) == 0) return paths;
    const uint64_t room = free() / 4;
    if (m.growth(paths) <= room) return paths;
    uint64_t lo = std::min(total, kAdjointMinPaths), hi = paths;   // growth(hi) > room
    while (lo + 64 < hi) {
        const uint64_t mid = lo + (hi - lo) / 2;
        (m.growth(mid) <= room ? lo : hi) = mid;
    }
    return lo;
}

}  // namespace eleven
