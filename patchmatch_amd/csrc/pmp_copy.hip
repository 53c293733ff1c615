// pmp_copy.hip -- staged host copies (pmp_copy.h).
#include "pmp_copy.h"

#include <sched.h>
#include <string.h>

#include <algorithm>
#include <exception>

namespace pmp {

Copier::~Copier() {
    {
        std::lock_guard<std::mutex> lk(sleep_mu_);
        stop_ = true;
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
    for (Slot& s : slot_) {
        if (s.dma) (void)hipEventSynchronize(s.ev);
        if (s.ev) (void)hipEventDestroy(s.ev);
    }
    if (pin_) (void)hipHostFree(pin_);
}

// The pinned chunks, at the first transfer; without memory for them transfers
// are the runtime's own.
bool Copier::start_ring() {
    if (ring_tried_) return ring_ok_;
    ring_tried_ = true;
    if (hipHostMalloc((void**)&pin_, kSlots * kChunk, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        pin_ = nullptr;
        return false;
    }
    for (Slot& s : slot_)
        if (hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            s.ev = nullptr;
            return false;
        }
    return ring_ok_ = true;
}

// The threads, at the first large transfer; false: the process has no CPU
// beside the caller's.
bool Copier::start_threads() {
    if (threads_tried_) return !threads_.empty();
    threads_tried_ = true;
    cpu_set_t set;
    CPU_ZERO(&set);
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    const int n = std::min(kThreads, cpus - 1);
    try {
        threads_.reserve(std::max(n, 0));
        for (int k = 0; k < n; ++k) threads_.emplace_back([this] { worker(); });
    } catch (const std::exception&) {   // as many as there could be
    }
    return !threads_.empty();
}

void Copier::run(const Span& p) {
    size_t off = p.off, len = p.len;
    uint8_t* lin = p.lin;
    while (len > 0) {
        const size_t r = off / p.c.row, x = off - r * p.c.row;
        const size_t m = p.c.row == p.c.pitch ? len : std::min(len, p.c.row - x);
        uint8_t* h = (uint8_t*)p.c.host + r * p.c.pitch + x;
        if (p.out) memcpy(h, lin, m);
        else memcpy(lin, h, m);
        off += m;
        lin += m;
        len -= m;
    }
}

// Takes and copies the oldest piece that nobody has taken.
bool Copier::run_one() {
    uint64_t t = taken_.load();
    do {
        if (t >= pushed_.load()) return false;
    } while (!taken_.compare_exchange_weak(t, t + 1));
    Task& k = task_[t % kTasks];
    run(k.p);
    k.done.store(t + 1, std::memory_order_release);
    return true;
}

void Copier::worker() {
    for (;;) {
        // the chunks of a transfer come some 50 us apart
        for (int spin = 0; spin < 4000; ++spin) {
            if (run_one()) spin = 0;
            else __builtin_ia32_pause();
        }
        std::unique_lock<std::mutex> lk(sleep_mu_);
        asleep_.fetch_add(1);
        cv_.wait(lk, [this] { return stop_ || taken_.load() < pushed_.load(); });
        asleep_.fetch_sub(1);
        if (stop_) return;
    }
}

// Hands the pieces of p to the threads, or copies it here and now.
void Copier::push(const Span& p, bool alone) {
    if (alone) {
        run(p);
        return;
    }
    for (size_t o = 0; o < p.len; o += kPiece) {
        if (next_ >= kTasks) wait(next_ - kTasks, next_ - kTasks + 1);
        task_[next_ % kTasks].p = Span{p.c, p.off + o, std::min(kPiece, p.len - o), p.lin + o, p.out};
        pushed_.store(++next_);
    }
    if (asleep_.load() > 0) {
        { std::lock_guard<std::mutex> lk(sleep_mu_); }
        cv_.notify_all();
    }
}

// Until pieces [begin, end) are copied; copies pieces meanwhile.
void Copier::wait(uint64_t begin, uint64_t end) {
    int spin = 0;
    for (uint64_t t = begin; t < end; ++t) {
        const Task& k = task_[t % kTasks];   // since reused for a later piece: done all the same
        while (k.done.load(std::memory_order_acquire) <= t) {
            if (run_one()) continue;
            if (++spin < 4000) __builtin_ia32_pause();
            else std::this_thread::yield();
        }
    }
}

hipError_t Copier::dma_done(Slot& s) {
    if (!s.dma) return hipSuccess;
    s.dma = false;
    return hipEventSynchronize(s.ev);
}

struct Copier::Walk {
    const HostCopy* c;
    int n, k = 0;
    size_t off = 0;
    bool end() {
        while (k < n && off >= c[k].row * c[k].rows) { ++k; off = 0; }
        return k == n;
    }
    bool next(Span& p) {
        if (end()) return false;
        p.c = c[k];
        p.off = off;
        p.len = std::min(kChunk, c[k].row * c[k].rows - off);
        off += p.len;
        return true;
    }
};

// Whether the host side of every copy is pageable memory, which the runtime
// does not know.
static bool pageable(const HostCopy* c, int n) {
    for (int k = 0; k < n; ++k) {
        hipPointerAttribute_t a;
        memset(&a, 0, sizeof(a));
        if (hipPointerGetAttributes(&a, c[k].host) != hipSuccess) {
            (void)hipGetLastError();
            continue;
        }
        if (a.type != hipMemoryTypeUnregistered) return false;
    }
    return true;
}

static size_t total(const HostCopy* c, int n) {
    size_t b = 0;
    for (int k = 0; k < n; ++k) b += c[k].row * c[k].rows;
    return b;
}

// Whether the rows of every copy follow each other in host memory.  The runtime
// moves other rows of pageable memory one by one, about 9 us each (a 1920x960
// image with a pitch of 2048: 8.8 ms, through the ring 0.06).
static bool contiguous(const HostCopy* c, int n) {
    for (int k = 0; k < n; ++k)
        if (c[k].row != c[k].pitch && c[k].rows > 1) return false;
    return true;
}

static hipError_t plain(hipStream_t s, const HostCopy* c, int n, hipMemcpyKind kind, bool wait) {
    const bool in = kind == hipMemcpyHostToDevice;
    for (int k = 0; k < n; ++k) {
        if (c[k].row * c[k].rows == 0) continue;
        const hipError_t e =
            c[k].row == c[k].pitch || c[k].rows == 1
                ? hipMemcpyAsync(in ? c[k].dev : c[k].host, in ? c[k].host : c[k].dev, c[k].row * c[k].rows, kind, s)
                : hipMemcpy2DAsync(in ? c[k].dev : c[k].host, in ? c[k].row : c[k].pitch, in ? c[k].host : c[k].dev,
                                   in ? c[k].pitch : c[k].row, c[k].row, c[k].rows, kind, s);
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(s);   // nothing reads or writes the host memory any more
            return e;
        }
    }
    return wait ? hipStreamSynchronize(s) : hipSuccess;
}

hipError_t Copier::small(hipStream_t s, const HostCopy* c, int n, bool out) {
    hipError_t e = dma_done(slot_[0]);
    size_t at = 0;
    for (int k = 0; k < n && e == hipSuccess; ++k) {
        const size_t bytes = c[k].row * c[k].rows;
        if (bytes == 0) continue;
        if (!out) run(Span{c[k], 0, bytes, pin_ + at, false});
        e = out ? hipMemcpyAsync(pin_ + at, c[k].dev, bytes, hipMemcpyDeviceToHost, s)
                : hipMemcpyAsync(c[k].dev, pin_ + at, bytes, hipMemcpyHostToDevice, s);
        at += bytes;
    }
    // an event for the next transfer to wait for would cost as much as the wait
    const hipError_t w = hipStreamSynchronize(s);
    if (e == hipSuccess) e = w;
    if (!out || e != hipSuccess) return e;
    at = 0;
    for (int k = 0; k < n; ++k) {
        const size_t bytes = c[k].row * c[k].rows;
        if (bytes) run(Span{c[k], 0, bytes, pin_ + at, true});
        at += bytes;
    }
    return e;
}

// Chunk k (of this transfer) uses slot k % kSlots; the slots' earlier pieces
// are done (every transfer ends so), their DMAs perhaps not.
hipError_t Copier::to_host(hipStream_t s, const HostCopy* c, int n, bool fresh) {
    std::lock_guard<std::mutex> lk(mu_);
    const size_t bytes = total(c, n);
    if (!pageable(c, n) || !start_ring() || (fresh && bytes < kFresh))
        return plain(s, c, n, hipMemcpyDeviceToHost, true);
    if (bytes < kAloneDown) return small(s, c, n, true);
    const bool alone = !start_threads();
    Walk w{c, n};
    bool more = true;
    uint64_t issued = 0, copied = 0;
    hipError_t e = hipSuccess;
    for (;;) {
        while (more && issued < copied + kSlots) {
            Slot& sl = slot_[issued % kSlots];
            if ((e = dma_done(sl)) != hipSuccess || !w.next(sl.p)) break;
            sl.p.lin = pin_ + (issued % kSlots) * kChunk;
            sl.p.out = true;
            wait(sl.begin, sl.end);
            e = hipMemcpyAsync(sl.p.lin, (const uint8_t*)sl.p.c.dev + sl.p.off, sl.p.len, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) break;
            ++issued;
            // the last chunk is waited for by the stream itself, without an
            // event, after which the caller's next wait for it would cost 30 us
            if ((more = !w.end()) && (e = hipEventRecord(sl.ev, s)) != hipSuccess) break;
            sl.dma = more;
        }
        if (e != hipSuccess || copied == issued) break;
        Slot& sl = slot_[copied % kSlots];
        if ((e = sl.dma ? dma_done(sl) : hipStreamSynchronize(s)) != hipSuccess) break;
        sl.begin = next_;
        push(sl.p, alone);
        sl.end = next_;
        ++copied;
    }
    for (const Slot& sl : slot_) wait(sl.begin, sl.end);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e;
}

hipError_t Copier::to_device(hipStream_t s, const HostCopy* c, int n, Until until) {
    std::lock_guard<std::mutex> lk(mu_);
    const bool wait_plain = until != Until::kQueued;   // the runtime may still read the host memory
    if (!pageable(c, n) || !start_ring()) return plain(s, c, n, hipMemcpyHostToDevice, wait_plain);
    const size_t bytes = total(c, n);
    if (bytes < kAloneUp) return small(s, c, n, false);
    if (bytes < kPinned && contiguous(c, n)) return plain(s, c, n, hipMemcpyHostToDevice, wait_plain);
    const bool alone = !start_threads();
    Walk w{c, n};
    bool more = true;
    uint64_t pushed = 0, sent = 0;
    hipError_t e = hipSuccess;
    while (e == hipSuccess) {
        while (more && pushed < sent + kSlots) {
            Slot& sl = slot_[pushed % kSlots];
            if ((e = dma_done(sl)) != hipSuccess || !(more = w.next(sl.p))) break;
            sl.p.lin = pin_ + (pushed % kSlots) * kChunk;
            sl.p.out = false;
            sl.begin = next_;
            push(sl.p, alone);
            sl.end = next_;
            ++pushed;
        }
        if (e != hipSuccess || sent == pushed) break;
        Slot& sl = slot_[sent % kSlots];
        wait(sl.begin, sl.end);
        e = hipMemcpyAsync((uint8_t*)sl.p.c.dev + sl.p.off, sl.p.lin, sl.p.len, hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(sl.ev, s);
        if (e == hipSuccess) sl.dma = true;
        ++sent;
    }
    for (const Slot& sl : slot_) wait(sl.begin, sl.end);   // no thread reads the caller's memory any more
    if (e == hipSuccess && until != Until::kDone) return e;
    const hipError_t d = hipStreamSynchronize(s);
    for (Slot& sl : slot_) sl.dma = false;
    return e == hipSuccess ? d : e;
}

void Copier::copy(void* dst, const void* src, size_t bytes) {
    std::unique_lock<std::mutex> lk(mu_, std::try_to_lock);
    if (bytes < kAloneUp || !lk.owns_lock() || !start_threads()) {
        memcpy(dst, src, bytes);
        return;
    }
    const uint64_t begin = next_;
    push(Span{flat_copy(dst, nullptr, bytes), 0, bytes, (uint8_t*)const_cast<void*>(src), true}, false);
    wait(begin, next_);
}

}  // namespace pmp
