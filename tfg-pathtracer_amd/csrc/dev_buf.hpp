// A device buffer that keeps the largest size asked of it.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

namespace eleven {

struct DevBuf {
    void* p = nullptr;
    size_t n = 0;
    uint64_t allocations = 0;   // how often p was allocated: tells a new allocation from an old one at its address
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    hipError_t ensure(size_t bytes) {
        if (bytes <= n && p) return hipSuccess;
        release();
        if (bytes == 0) bytes = 16;
        hipError_t e = hipMalloc(&p, bytes);
        if (e == hipSuccess) {
            n = bytes;
            allocations++;
        }
        return e;
    }
    template <class T>
    T* as() const {
        return (T*)p;
    }
};

// Changes whenever one of the buffers is allocated anew: what a captured
// launch sequence, which holds their addresses, has to be compared by.  The
// addresses themselves can come back with a new allocation of one buffer while
// another's does not.
template <class... Bufs>
uint64_t allocationsOf(const Bufs&... b) {
    return (b.allocations + ... + 0);
}

}  // namespace eleven
