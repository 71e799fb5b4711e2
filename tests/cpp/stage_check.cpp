// The pool of pinned stages and the copy through them, over a stand-in for the runtime: who gets which memory, what is
// pinned and given back, what an error leaves, and what the host threads do meanwhile.  Modes: pool, copy, wait, contexts.
#include "stage.hpp"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <string>

using namespace eleven;

static std::atomic<int> pins{0}, frees{0}, syncs{0};
static std::atomic<int> failSync{-1};   // which event wait fails
static std::atomic<int> busyMs{0};      // how long the GPU works before the next event
extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    pins++;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    frees++;
    std::free(p);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = (hipEvent_t)1;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) {
    std::this_thread::sleep_for(std::chrono::milliseconds(busyMs.exchange(0)));
    return failSync-- == 0 ? hipErrorUnknown : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    syncs++;
    return hipSuccess;
}
}

static int bad = 0;
static void check(bool ok, const char* what) {
    if (!ok) bad++, printf("not so: %s\n", what);
}

static void pool() {
    StagePool pool;
    {
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess && a->ensure(100000) == hipSuccess, "a stage");
    }
    const int first = pins;
    for (int k = 0; k < 5; k++) {   // other contexts' first calls
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess && a->ensure(50000 + 10000 * k) == hipSuccess, "a stage again");
    }
    check(pins == first, "a second context pins nothing");
    {
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess && a->ensure(20u << 20) == hipSuccess, "a large stage");
    }
    const int grown = pins;
    {
        StageLease a(0, nullptr, pool), b(0, nullptr, pool), c(0, nullptr, pool), other(1, nullptr, pool);
        check(a.take() == hipSuccess && b.take() == hipSuccess && c.take() == hipSuccess && other.take() == hipSuccess, "leases");
        check(&*a != &*b && &*b != &*c && &*a != &*c && &*other != &*a, "calls at the same time have stages of their own");
        check(a->bytes() == 8u << 20, "the largest idle stage first");
        check(a->ensure(3u << 20) == hipSuccess && a->bytes() == 8u << 20, "it is not pinned again for less");
        check(b->ensure(1000) == hipSuccess && c->ensure(1000) == hipSuccess && other->ensure(1000) == hipSuccess, "memory");
    }
    check(pool.idleCount() == StagePool::kIdle + 1, "the pool keeps kIdle stages of a device");
    check(frees > 0 && pins == grown + 6, "and gives the others back");
    {
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess && a->bytes() == 8u << 20, "the large one among them");
        const int before = syncs;
        a.inFlight(true);
        check(before == syncs, "no wait yet");
    }
    check(syncs == 1, "a call that ends early waits for what it enqueued");
    std::atomic<int> shared{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; t++)
        threads.emplace_back([&, t] {
            for (int k = 0; k < 2000; k++) {
                StageLease a(t & 1, nullptr, pool);
                if (a.take() != hipSuccess || a->ensure(1000 + 1000 * (k % 90)) != hipSuccess) shared++;
                std::memset(a->p, t, 1000);
                std::this_thread::yield();
                for (int i = 0; i < 1000; i++) shared += a->p[i] != t;
            }
        });
    for (auto& t : threads) t.join();
    check(shared == 0, "no thread writes another's stage");
    check(pool.idleCount() <= 2 * StagePool::kIdle, "the pool is bounded");
}

static void copy() {
    StagePool pool;
    for (size_t items : {1ul, 1000ul, 209715ul, 209716ul, 1048576ul, 2000003ul}) {
        std::vector<unsigned char> out(items * 20, 0xff);
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess, "a stage");
        const hipError_t e = stageOut(
            a, items, 20,
            [&](size_t first, size_t n, unsigned char* chunk) {
                for (size_t i = 0; i < n; i++) std::memset(chunk + 20 * i, (int)((first + i) % 251), 20);
                return hipSuccess;
            },
            [&](size_t first, size_t, const unsigned char* chunk, size_t i0, size_t i1) {
                std::memcpy(&out[20 * (first + i0)], chunk + 20 * i0, 20 * (i1 - i0));
            });
        size_t wrong = 0;
        for (size_t i = 0; i < items; i++)
            for (int k = 0; k < 20; k += 19) wrong += out[20 * i + k] != i % 251;
        check(e == hipSuccess && wrong == 0, "every item, once");
    }
    check(syncs == 0, "no wait beyond the chunks'");
    for (int at = 0; at < 4; at++) {   // a wait that fails
        failSync = at;
        {
            StageLease a(0, nullptr, pool);
            check(a.take() == hipSuccess, "a stage");
            check(stageOut(
                      a, 2000003, 20, [](size_t, size_t, unsigned char*) { return hipSuccess; },
                      [](size_t, size_t, const unsigned char*, size_t, size_t) {}) == hipErrorUnknown, "the error comes back");
        }
        check(syncs == at + 1, "an error leaves nothing in flight");
    }
}

// A thread for each of eight contexts: their calls at the same time pin once each, and what the contexts leave is freed.
static void contexts() {
    StagePool pool;
    for (int k = 0; k < 8; k++) pool.contexts(1, 1);
    for (int round = 0; round < 3; round++) {
        std::vector<std::unique_ptr<StageLease>> at;
        for (int k = 0; k < 8; k++) {
            at.push_back(std::make_unique<StageLease>(1, nullptr, pool));
            check(at.back()->take() == hipSuccess && (*at.back())->ensure(100000) == hipSuccess, "a stage");
        }
    }
    check(pins == 16, "eight stages, and the memory of each pinned once");
    check(pool.idleCount() == 8, "one stays for each context");
    for (int k = 0; k < 8; k++) pool.contexts(1, -1);
    check(pool.idleCount() == StagePool::kIdle && frees == 12, "what the contexts leave is given back");
}

// Host threads' time while the GPU works for 400 ms before the first chunk is there.
static void wait() {
    StagePool pool;
    for (int fails : {-1, 0}) {
        StageLease a(0, nullptr, pool);
        check(a.take() == hipSuccess, "a stage");
        busyMs = 400;
        failSync = fails;
        std::vector<unsigned char> out(12 << 20);
        const std::clock_t from = std::clock();
        const hipError_t e = stageOut(
            a, out.size(), 1, [](size_t, size_t, unsigned char*) { return hipSuccess; },
            [&](size_t first, size_t, const unsigned char* chunk, size_t i0, size_t i1) {
                std::memcpy(&out[first + i0], chunk + i0, i1 - i0);
            });
        const double ms = 1e3 * (double)(std::clock() - from) / CLOCKS_PER_SEC;
        check(e == (fails ? hipSuccess : hipErrorUnknown), "the wait's result");
        printf("processor time %.0f ms\n", ms);
        check(ms < 200, "the helpers sleep while the GPU works");
    }
}

int main(int, char** argv) {
    const std::string mode = argv[1];
    if (mode == "pool") pool();
    if (mode == "copy") copy();
    if (mode == "wait") wait();
    if (mode == "contexts") contexts();
    printf("bad=%d\n", bad);
    return bad != 0;
}
