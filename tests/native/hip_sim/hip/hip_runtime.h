// A simulated HIP runtime for copy_selftest.cpp: streams are host threads that
// run their copies in order and later than they were queued (device memory is
// host memory), so what a caller may and may not rely on shows on the CPU, and
// the sanitizers see every access.  Only what pmp_copy.hip calls.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <deque>
#include <functional>
#include <map>
#include <mutex>
#include <thread>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorNotReady = 600, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
struct hipPointerAttribute_t {
    hipMemoryType type;
};

namespace hip_sim {

struct Stats {
    std::atomic<int> pinned_allocs{0}, pinned_held{0}, copies_1d{0}, copies_2d{0}, from_pageable{0}, events{0};
    std::atomic<int> fail_copy_in{-1};      // the n-th copy from now fails
    std::atomic<bool> fail_pinned{false};
    std::atomic<int> delay_us{0};           // of each copy
};
inline Stats& stats() { static Stats s; return s; }

struct Ranges {
    std::mutex mu;
    std::map<uintptr_t, size_t> pinned;
    bool holds(const void* p) {
        std::lock_guard<std::mutex> lk(mu);
        auto it = pinned.upper_bound((uintptr_t)p);
        if (it == pinned.begin()) return false;
        --it;
        return (uintptr_t)p < it->first + it->second;
    }
};
inline Ranges& ranges() { static Ranges r; return r; }

class Stream {
public:
    Stream() : t_([this] { loop(); }) {}
    ~Stream() {
        push([this] { stop_ = true; });
        t_.join();
    }
    uint64_t push(std::function<void()> f) {
        std::lock_guard<std::mutex> lk(mu_);
        q_.push_back(std::move(f));
        cv_.notify_all();
        return ++queued_;
    }
    void wait(uint64_t n) {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return done_ >= n; });
    }
    void sync() {
        uint64_t n;
        {
            std::lock_guard<std::mutex> lk(mu_);
            n = queued_;
        }
        wait(n);
    }
    bool reached(uint64_t n) {
        std::lock_guard<std::mutex> lk(mu_);
        return done_ >= n;
    }
    bool idle() {
        std::lock_guard<std::mutex> lk(mu_);
        return done_ == queued_;
    }

private:
    void loop() {
        while (!stop_) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [this] { return !q_.empty(); });
                f = std::move(q_.front());
                q_.pop_front();
            }
            f();
            std::lock_guard<std::mutex> lk(mu_);
            ++done_;
            cv_.notify_all();
        }
    }
    std::mutex mu_;
    std::condition_variable cv_;
    std::deque<std::function<void()>> q_;
    uint64_t queued_ = 0, done_ = 0;
    bool stop_ = false;                  // the stream's thread only
    std::thread t_;
};

struct Event {
    std::mutex mu;
    Stream* s = nullptr;
    uint64_t at = 0;
};

}  // namespace hip_sim

using hipStream_t = hip_sim::Stream*;
using hipEvent_t = hip_sim::Event*;

inline const char* hipGetErrorString(hipError_t) { return "simulated"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    if (hip_sim::stats().fail_pinned) return hipErrorOutOfMemory;
    *p = malloc(bytes);
    std::lock_guard<std::mutex> lk(hip_sim::ranges().mu);
    hip_sim::ranges().pinned[(uintptr_t)*p] = bytes;
    hip_sim::stats().pinned_allocs++;
    hip_sim::stats().pinned_held++;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    {
        std::lock_guard<std::mutex> lk(hip_sim::ranges().mu);
        hip_sim::ranges().pinned.erase((uintptr_t)p);
    }
    free(p);
    hip_sim::stats().pinned_held--;
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    if (!hip_sim::ranges().holds(p)) return hipErrorInvalidValue;
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new hip_sim::Event;
    hip_sim::stats().events++;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    hip_sim::stats().events--;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    const uint64_t at = s->push([] {});
    std::lock_guard<std::mutex> lk(e->mu);
    e->s = s;
    e->at = at;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    hip_sim::Stream* s;
    uint64_t at;
    {
        std::lock_guard<std::mutex> lk(e->mu);
        s = e->s;
        at = e->at;
    }
    if (s) s->wait(at);
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
    std::lock_guard<std::mutex> lk(e->mu);
    return !e->s || e->s->reached(e->at) ? hipSuccess : hipErrorNotReady;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->sync();
    return hipSuccess;
}
inline hipError_t hip_sim_queue(void* d, const void* h, hipMemcpyKind kind, hipStream_t s, std::function<void()> f) {
    auto& st = hip_sim::stats();
    if (st.fail_copy_in >= 0 && st.fail_copy_in-- == 0) return hipErrorUnknown;
    if (!hip_sim::ranges().holds(kind == hipMemcpyHostToDevice ? h : d)) st.from_pageable++;
    const int us = st.delay_us;
    s->push([f, us] {
        if (us) std::this_thread::sleep_for(std::chrono::microseconds(us));
        f();
    });
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t st) {
    hip_sim::stats().copies_1d++;
    return hip_sim_queue(d, s, kind, st, [=] { memcpy(d, s, n); });
}
inline hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t row, size_t rows,
                                   hipMemcpyKind kind, hipStream_t st) {
    hip_sim::stats().copies_2d++;
    return hip_sim_queue(d, s, kind, st, [=] {
        for (size_t r = 0; r < rows; ++r) memcpy((char*)d + r * dp, (const char*)s + r * sp, row);
    });
}
