// The wavefront buffers when the device runs out of memory on their way to a larger size: the call fails, and a call
// for the size they had before finds or makes every one of them.  (No device: hipMalloc and hipFree are here.)
#include "wf_buffers.hpp"

#include <cstdio>
#include <cstdlib>

static int failAt = -1, calls = 0;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
    if (calls++ == failAt) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    *p = std::malloc(n);
    return hipSuccess;
}
extern "C" hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}

using namespace eleven;

int main() {
    int bad = 0;
    for (int k = 0; k < 14; k++) {
        WfBuffers w;
        bad += w.ensure(100, 150, true, 64) != hipSuccess || !w.holds(100, 150, true);
        calls = 0;
        failAt = k;
        const hipError_t e = w.ensure(1000, 1100, true, 64);
        const bool failed = e != hipSuccess;
        failAt = -1;
        // the counters do not grow: 12 buffers do
        if (failed != (k < 12)) bad++, printf("allocation %d: failed %d\n", k, failed);
        if (w.ensure(100, 150, true, 64) != hipSuccess || !w.holds(100, 150, true))
            bad++, printf("allocation %d fails: the former size is gone\n", k);
        if (w.ensure(1000, 1100, false, 64) != hipSuccess || !w.holds(1000, 1100, false))
            bad++, printf("allocation %d fails: no larger size afterwards\n", k);
        const uint64_t held = w.allocations();
        if (w.ensure(700, 1100, false, 64) != hipSuccess || w.allocations() != held) bad++, printf("held sizes moved\n");
    }
    printf("bad=%d\n", bad);
    return bad != 0;
}
