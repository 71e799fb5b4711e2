// Pinned host memory between the GPU and a caller's arrays, which are
// pageable: lent by a pool to one call at a time.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <utility>
#include <vector>

#include "host_parallel.hpp"

namespace eleven {

// Two chunks in turn, one filled by the GPU while the other is copied out, and
// the words that a call's tallies are read back to.
struct Stage {
    static constexpr size_t kChunk = 4u << 20;
    static constexpr size_t kTallyWords = 64;
    unsigned char* p = nullptr;
    size_t n = 0;   // bytes of a chunk
    bool two = false;
    hipEvent_t filled[2] = {nullptr, nullptr};
    unsigned long long* tallies = nullptr;
    Stage() = default;
    Stage(const Stage&) = delete;
    Stage& operator=(const Stage&) = delete;
    ~Stage() {
        if (p) (void)hipHostFree(p);
        if (tallies) (void)hipHostFree(tallies);
        for (auto e : filled)
            if (e) (void)hipEventDestroy(e);
    }
    hipError_t ensureTallies() {
        if (tallies) return hipSuccess;
        return hipHostMalloc((void**)&tallies, sizeof(unsigned long long) * kTallyWords, hipHostMallocDefault);
    }
    // Memory for an output of `bytes`, taken chunk by chunk: one chunk, or two.
    // Whole chunks at once: pinning takes as long for 64 KB (0.05 to 0.4 ms), pages
    // cost when they are touched, and a larger output finds it pinned.
    hipError_t ensure(size_t bytes) {
        const bool both = bytes > kChunk;
        for (auto& e : filled)
            if (!e)
                if (hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming); r != hipSuccess) return r;
        if (p && both <= two) return hipSuccess;
        if (p) (void)hipHostFree(p);
        p = nullptr;
        n = 0;
        const hipError_t r = hipHostMalloc((void**)&p, kChunk * (both ? 2 : 1), hipHostMallocDefault);
        if (r != hipSuccess) return r;
        n = kChunk;
        two = both;
        return hipSuccess;
    }
    size_t bytes() const { return n * (two ? 2 : 1); }
};

// The stages that no call uses.  Pinning memory and touching it for the first
// time take 0.3 to 0.8 ms, which a stage for each context put into every
// context's first call (1000 rays on a new context took 556 us, 200 by
// pageable copies, and take 115 with a pooled stage; the first adjoint of a 128 x
// 128 frame with 256 x 256 texels 1822, 1610 and 1074).  As many stages of a
// device (of 8 MiB at most, the largest) stay pinned for the next call as it
// has contexts, so that a thread for each finds one, and kIdle where there are
// fewer, until the process ends; the others are given back at once.
class StagePool {
public:
    static constexpr size_t kIdle = 2;
    // The largest idle stage of the device, which is current, or a new one; null without host memory.
    std::unique_ptr<Stage> take(int device) noexcept {
        {
            std::lock_guard<std::mutex> lock(mu);
            size_t best = idle.size();
            for (size_t i = 0; i < idle.size(); i++)
                if (idle[i].first == device && (best == idle.size() || idle[i].second->bytes() > idle[best].second->bytes()))
                    best = i;
            if (best < idle.size()) {
                std::unique_ptr<Stage> s = std::move(idle[best].second);
                idle[best] = std::move(idle.back());
                idle.pop_back();
                return s;
            }
        }
        return std::unique_ptr<Stage>(new (std::nothrow) Stage());
    }
    void give(int device, std::unique_ptr<Stage> s) noexcept {
        std::vector<std::unique_ptr<Stage>> surplus;   // freed after the lock
        std::lock_guard<std::mutex> lock(mu);
        try {
            idle.emplace_back(device, std::move(s));
            trim(device, surplus);
        } catch (...) {
        }
    }
    // A context of the device was made (1) or is gone (-1).
    void contexts(int device, int change) noexcept {
        std::vector<std::unique_ptr<Stage>> surplus;
        std::lock_guard<std::mutex> lock(mu);
        try {
            if (users.size() <= (size_t)device) users.resize(device + 1, 0);
            users[device] += change;
            trim(device, surplus);
        } catch (...) {
        }
    }
    size_t idleCount() {
        std::lock_guard<std::mutex> lock(mu);
        return idle.size();
    }

private:
    // Moves the smallest of the device's idle stages to `surplus` until it has no more than it may.
    void trim(int device, std::vector<std::unique_ptr<Stage>>& surplus) {
        const size_t most = std::max(kIdle, (size_t)device < users.size() ? (size_t)std::max(0, users[device]) : 0);
        for (;;) {
            size_t held = 0, least = idle.size();
            for (size_t i = 0; i < idle.size(); i++) {
                if (idle[i].first != device) continue;
                held++;
                if (least == idle.size() || idle[i].second->bytes() < idle[least].second->bytes()) least = i;
            }
            if (held <= most) return;
            surplus.push_back(std::move(idle[least].second));
            idle[least] = std::move(idle.back());
            idle.pop_back();
        }
    }
    std::mutex mu;
    std::vector<std::pair<int, std::unique_ptr<Stage>>> idle;
    std::vector<int> users;   // contexts by device
};

// The process's pool, made by the first call that takes a stage (the runtime
// is up by then, and goes down after it).
inline StagePool& stagePool() {
    static StagePool pool;
    return pool;
}

// A stage for the duration of one call on one stream.  It goes back once
// nothing that the call enqueued can still write it.
class StageLease {
public:
    StageLease(int device, hipStream_t stream, StagePool& pool = stagePool()) : pool_(pool), device_(device), stream_(stream) {}
    StageLease(const StageLease&) = delete;
    StageLease& operator=(const StageLease&) = delete;
    ~StageLease() {
        if (!stage_) return;
        if (inFlight_) (void)hipStreamSynchronize(stream_);
        pool_.give(device_, std::move(stage_));
    }
    hipError_t take() {   // first of all
        stage_ = pool_.take(device_);
        return stage_ ? stage_->ensureTallies() : hipErrorOutOfMemory;
    }
    Stage& operator*() const { return *stage_; }
    Stage* operator->() const { return stage_.get(); }
    hipStream_t stream() const { return stream_; }
    void inFlight(bool f) { inFlight_ = f; }   // device work that uses the stage is enqueued / has ended

private:
    StagePool& pool_;
    int device_;
    hipStream_t stream_;
    std::unique_ptr<Stage> stage_;
    bool inFlight_ = false;
};

// Takes `items` items of `itemBytes` through the stage: fill(first, n, chunk)
// enqueues on the lease's stream what writes the items [first, first + n) to a chunk,
// copy(first, n, chunk, i0, i1) copies the chunk's items [i0, i1) out, on up
// to 8 host threads (a thread per MB: a frame's copy is bound by the page
// faults of the caller's fresh arrays, which one thread takes one at a time).
// They look for the first chunk for kSpin, which a read-back of a finished image
// takes, then sleep until it is there: the GPU may have a whole adjoint to
// finish first.  (Asleep at once, a wake-up of ~40 us each came on top of a
// read-back of 1 MB and more: twelve images 1.79 -> 1.89 ms.)
template <class Fill, class Copy>
hipError_t stageOut(StageLease& lease, size_t items, size_t itemBytes, Fill&& fill, Copy&& copy) {
    if (!items) return hipSuccess;
    Stage& st = *lease;
    const hipStream_t stream = lease.stream();
    hipError_t e = st.ensure(items * itemBytes);
    if (e != hipSuccess) return e;
    lease.inFlight(true);
    const size_t per = st.n / itemBytes, chunks = (items + per - 1) / per;
    auto count = [&](size_t k) { return std::min(per, items - k * per); };
    auto chunk = [&](size_t k) { return st.p + (k & 1) * st.n; };
    auto issue = [&](size_t k) -> hipError_t {
        hipError_t r = fill(k * per, count(k), chunk(k));
        return r == hipSuccess ? hipEventRecord(st.filled[k & 1], stream) : r;
    };
    std::atomic<size_t> ready{0}, done{0};   // chunks filled; thread-chunks copied
    std::atomic<bool> failed{false};         // no further chunk gets ready
    std::mutex mu;
    std::condition_variable begun;
    std::atomic<size_t> team{0};             // threads that share a chunk: known with the first one ready
    constexpr auto kSpin = std::chrono::microseconds(200);
    auto part = [&](size_t k, size_t t) {
        const size_t n = count(k), T = team.load(std::memory_order_relaxed);
        copy(k * per, n, chunk(k), n * t / T, n * (t + 1) / T);
    };
    auto work = [&](size_t t) {
        auto known = [&] { return team.load(std::memory_order_acquire) != 0; };
        for (const auto from = std::chrono::steady_clock::now(); !known();) {
            std::this_thread::yield();
            if (std::chrono::steady_clock::now() - from < kSpin) continue;
            std::unique_lock<std::mutex> lock(mu);
            begun.wait(lock, known);
        }
        for (size_t k = 0; k < chunks; k++) {
            while (ready.load(std::memory_order_acquire) <= k) {
                if (failed.load(std::memory_order_acquire)) return;
                std::this_thread::yield();
            }
            part(k, t);
            done.fetch_add(1, std::memory_order_release);
        }
    };
    const size_t wantThreads = std::min<size_t>({(size_t)hostThreads(), 8, items * itemBytes >> 20});
    std::vector<std::thread> threads;
    for (size_t k = 0; k < std::min<size_t>(chunks, 2) && e == hipSuccess; k++) e = issue(k);
    if (e == hipSuccess) {
        try {
            threads.reserve(wantThreads);
            for (size_t t = 1; t < wantThreads; t++) threads.emplace_back(work, t);
        } catch (...) {   // fewer threads share the work
        }
    }
    const size_t T = threads.size() + 1;
    auto begin = [&] {
        {
            std::lock_guard<std::mutex> lock(mu);
            team.store(T, std::memory_order_release);
        }
        begun.notify_all();
    };
    for (size_t k = 0; k < chunks && e == hipSuccess; k++) {
        e = hipEventSynchronize(st.filled[k & 1]);
        if (e != hipSuccess) break;
        ready.store(k + 1, std::memory_order_release);
        if (k == 0) begin();
        part(k, 0);
        if (k + 2 < chunks) {   // the chunk is filled again once every thread has copied its share
            while (done.load(std::memory_order_acquire) < (k + 1) * (T - 1)) std::this_thread::yield();
            e = issue(k + 2);
        }
    }
    if (e != hipSuccess) {
        failed.store(true, std::memory_order_release);
        begin();
    }
    for (auto& t : threads) t.join();
    if (e == hipSuccess) lease.inFlight(false);   // every chunk was waited for
    return e;
}

}  // namespace eleven
