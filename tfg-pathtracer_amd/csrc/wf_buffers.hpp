// The queues and path state of wavefront renders (kernels.hpp, WfState).
#pragma once

#include <algorithm>

#include "dev_buf.hpp"

namespace eleven {

struct WfBuffers {
    static constexpr size_t kEntryBytes = 176, kSlotBytes = 64;   // of a queue entry and a path slot (aov apart)
    DevBuf ray0, ray1, hits, shadowH, shadowP;              // per queue entry
    DevBuf pathT, pathL, pix, sample, quiet, pend, aov;     // per path slot
    DevBuf counters;
    size_t cap = 0, qcap = 0;   // path slots and queue entries that every buffer holds (aov apart)

    // Room for `slots` path slots and `entries` queue entries, max(slots, kXcds * segSize): the camera queue is
    // indexed by slot, the compacted queues by XCD segment.  Every buffer keeps the
    // largest size asked of it; the per-path AOV buffer is sized by this call's
    // slots whatever the others hold, since renders without AOV may have grown
    // them past its size.  What a failed call leaves is asked for again by the
    // next one, whatever its size.
    hipError_t ensure(size_t slots, size_t entries, bool withAov, size_t counterBytes) {
        if (withAov)
            if (hipError_t e = aov.ensure(slots * 48); e != hipSuccess) return e;
        if (slots <= cap && entries <= qcap) return hipSuccess;
        const size_t newCap = std::max(cap, slots), newQcap = std::max(qcap, entries);
        cap = qcap = 0;
        const struct {
            DevBuf& b;
            size_t bytes;
        } all[] = {{ray0, entries * 32},    {ray1, entries * 32}, {hits, entries * 16},
                   {shadowH, entries * 48}, {shadowP, entries * 48}, {pathT, slots * 16},
                   {pathL, slots * 16},     {pix, slots * 4},        {sample, slots * 4},
                   {quiet, slots * 8},      {pend, slots * 16},      {counters, counterBytes}};
        for (auto& x : all)
            if (hipError_t e = x.b.ensure(x.bytes); e != hipSuccess) return e;
        cap = newCap;
        qcap = newQcap;
        return hipSuccess;
    }
    // The launches index `slots` path slots and `entries` queue entries in every buffer.
    bool holds(size_t slots, size_t entries, bool withAov) const {
        return ray0.n >= entries * 32 && ray1.n >= entries * 32 && hits.n >= entries * 16 && shadowH.n >= entries * 48 &&
               shadowP.n >= entries * 48 && pathT.n >= slots * 16 && pathL.n >= slots * 16 && pix.n >= slots * 4 &&
               sample.n >= slots * 4 && quiet.n >= slots * 8 && pend.n >= slots * 16 && (!withAov || aov.n >= slots * 48);
    }
    uint64_t allocations() const {
        return allocationsOf(ray0, ray1, hits, shadowH, shadowP, pathT, pathL, pix, sample, quiet, pend, aov, counters);
    }
};

}  // namespace eleven
