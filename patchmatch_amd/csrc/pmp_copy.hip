// pmp_copy.hip -- staged host copies (pmp_copy.h).
#include "pmp_copy.h"

#include <pthread.h>
#include <sched.h>
#include <signal.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <exception>
#include <new>
#include <thread>
#include <vector>

namespace pmp {

// A chunk is one DMA, with 14 us of fixed costs: 48 MiB in chunks of 1 MiB
// ran at 31 GB/s, of 2 at 40, of 4 at 46.  Its pieces are what a thread
// copies at a time.  More than two chunks in flight gained nothing, and
// their pinned pages cost 0.38 ms per MiB when first touched.
static constexpr size_t kChunk = size_t(4) << 20, kPiece = size_t(256) << 10;
static constexpr int kSlots = 2;
static constexpr int kTasks = 256;       // a power of two above kSlots * kChunk / kPiece
// The process's threads, and its rings for one device: transfers beyond these
// that run at the same time are the runtime's own.
static constexpr int kThreads = 8, kRings = 4, kAllRings = 64;
// Transfers below these are copied by the caller alone, in one chunk: waking
// the threads costs more (normals of 328x182, 716 KB down: 66 us alone, 52
// with them; a 614 KB image up: 75 and 76).  Three copies and more, each of
// which is a chunk, are worth it later (the three maps of 240x120, 691 KB: 60
// us alone, 74 with them, of 300x150 77 and 73).
static constexpr size_t kAloneDown = size_t(512) << 10, kAloneDownMaps = size_t(1) << 20, kAloneUp = size_t(768) << 10;
// Uploads of contiguous rows from kAloneUp to these are the runtime's own, on
// the caller's thread: several copies in a call (five 640x320 maps to the
// cleaner and back: 222 us, with the threads 290; of 800x400: 342 and 345; of
// 1363x677: 863 and 638), or one (a 1300x650 image 41 and 43, a 1920x960 one
// 75 and 62).
static constexpr size_t kPinned = size_t(6) << 20, kPinnedOne = size_t(3) << 19;
// So are downloads to fresh memory below this: pinning takes the page
// faults at once, which the threads would fight over (the pruner's points
// and map: of 320x160 views 189 us, with the threads 225; of 640x320 366
// and 375; of 1098x494 885 and 785).
static constexpr size_t kFresh = size_t(12) << 20;

namespace {

struct Span {               // bytes [off, off + len) of c, contiguous at lin
    HostCopy c;
    size_t off, len;
    uint8_t* lin;
    bool out;               // from lin to c.host
};

void copy_span(const Span& p) {
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

// What one transfer at a time uses: pinned chunks and the pieces that the
// threads copy.
struct Ring {
    struct Task {
        Span p;
        std::atomic<uint64_t> done{0};   // 1 + the last ticket done
    };
    struct Slot {                        // a chunk's pinned memory
        Span p;
        uint64_t begin = 0, end = 0;     // its pieces' tickets: [begin, end)
        hipEvent_t ev = nullptr;         // after its last DMA
        bool dma = false;                // ev is recorded
    };
    explicit Ring(int dev) : device(dev) {}
    ~Ring() {
        for (Slot& s : slot) {
            if (s.dma) (void)hipEventSynchronize(s.ev);
            if (s.ev) (void)hipEventDestroy(s.ev);
        }
        if (pin) (void)hipHostFree(pin);
    }

    // The pinned chunks, at the first DMA; on the ring's device.
    bool start() {
        if (!pin && hipHostMalloc((void**)&pin, kSlots * kChunk, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            pin = nullptr;
            return false;
        }
        for (Slot& s : slot)
            if (!s.ev && hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                s.ev = nullptr;
                return false;
            }
        return true;
    }

    // Whether a transfer on s need not wait for another stream's DMA.
    bool ready(hipStream_t s) {
        if (last == s) return true;
        for (Slot& k : slot) {
            if (!k.dma) continue;
            if (hipEventQuery(k.ev) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
            k.dma = false;
        }
        return true;
    }

    hipError_t dma_done(Slot& s) {
        if (!s.dma) return hipSuccess;
        s.dma = false;
        return hipEventSynchronize(s.ev);
    }

    // Takes and copies the oldest piece that nobody has taken.
    bool run_one() {
        uint64_t t = taken.load();
        do {
            if (t >= pushed.load()) return false;
        } while (!taken.compare_exchange_weak(t, t + 1));
        Task& k = task[t % kTasks];
        copy_span(k.p);
        k.done.store(t + 1, std::memory_order_release);
        return true;
    }

    // Until pieces [begin, end) are copied; copies pieces meanwhile.
    void wait(uint64_t begin, uint64_t end) {
        int spin = 0;
        for (uint64_t t = begin; t < end; ++t) {
            const Task& k = task[t % kTasks];   // since reused for a later piece: done all the same
            while (k.done.load(std::memory_order_acquire) <= t) {
                if (run_one()) continue;
                if (++spin < 4000) __builtin_ia32_pause();
                else std::this_thread::yield();
            }
        }
    }

    const int device;
    bool lent = false;                   // under the pool's mutex
    hipStream_t last = nullptr;          // of the last transfer
    uint8_t* pin = nullptr;
    Slot slot[kSlots];
    Task task[kTasks];
    uint64_t next = 0;                   // the next piece's ticket; its task is ticket % kTasks
    std::atomic<uint64_t> pushed{0}, taken{0};
};

// The chunks of a list of copies.
struct Walk {
    const HostCopy* c;
    int n, k = 0;
    size_t off = 0;
    bool end() {
        while (k < n && off >= c[k].row * c[k].rows) { ++k; off = 0; }
        return k == n;
    }
    void next(Span& p) {   // where there is one
        (void)end();
        p.c = c[k];
        p.off = off;
        p.len = std::min(kChunk, c[k].row * c[k].rows - off);
        off += p.len;
    }
};

}  // namespace

class CopyPool {
public:
    static std::shared_ptr<CopyPool> get() {
        static std::mutex* mu = new std::mutex;                               // outlive every context
        static std::weak_ptr<CopyPool>* the = new std::weak_ptr<CopyPool>;
        std::lock_guard<std::mutex> lk(*mu);
        std::shared_ptr<CopyPool> p = the->lock();
        if (!p) *the = p = std::make_shared<CopyPool>();
        return p;
    }
    CopyPool() { threads_.reserve(kThreads); }
    ~CopyPool() {
        {
            std::lock_guard<std::mutex> lk(sleep_mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto& t : threads_) t.join();
        for (int k = 0; k < n_rings_; ++k) delete rings_[k];
    }

    // A ring for a transfer on the current device, nullptr where all are in use.
    // s: the stream of its DMAs; none: it copies from host to host.
    Ring* lend(hipStream_t s) {
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess) return nullptr;
        std::lock_guard<std::mutex> lk(mu_);
        const int n = n_rings_.load();
        Ring* r = nullptr;
        int mine = 0;
        for (int k = 0; k < n && !r; ++k) {
            if (rings_[k]->device != device) continue;
            ++mine;
            if (!rings_[k]->lent && (!s || rings_[k]->ready(s))) r = rings_[k];
        }
        if (!r) {
            if (mine >= kRings || n >= kAllRings || !(r = new (std::nothrow) Ring(device))) return nullptr;
            rings_[n] = r;
            n_rings_.store(n + 1);
        }
        if (s) {
            if (!r->start()) return nullptr;
            r->last = s;
        }
        r->lent = true;
        return r;
    }
    void give_back(Ring* r) {
        std::lock_guard<std::mutex> lk(mu_);
        r->lent = false;
    }

    // At least one thread beside the caller's, for a transfer of `bytes`: as many
    // as have a piece to copy, and a CPU.
    bool start_threads(size_t bytes) {
        std::lock_guard<std::mutex> lk(mu_);
        size_t want = std::min<size_t>(kThreads, bytes / kPiece);
        if (threads_.size() < want) {
            cpu_set_t set;
            CPU_ZERO(&set);
            const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
            want = std::min<size_t>(want, std::max(cpus - 1, 0));
            // the process's signals are not theirs
            sigset_t all, old;
            sigfillset(&all);
            pthread_sigmask(SIG_SETMASK, &all, &old);
            try {
                while (threads_.size() < want) threads_.emplace_back([this] { worker(); });
            } catch (const std::exception&) {   // as many as there could be
            }
            pthread_sigmask(SIG_SETMASK, &old, nullptr);
        }
        return !threads_.empty();
    }

    // Hands the pieces of p to the threads, or copies it here and now.
    void push(Ring& r, const Span& p, bool alone) {
        if (alone) {
            copy_span(p);
            return;
        }
        for (size_t o = 0; o < p.len; o += kPiece) {
            if (r.next >= kTasks) r.wait(r.next - kTasks, r.next - kTasks + 1);
            r.task[r.next % kTasks].p = Span{p.c, p.off + o, std::min(kPiece, p.len - o), p.lin + o, p.out};
            r.pushed.store(++r.next);
        }
        if (asleep_.load() > 0) {
            { std::lock_guard<std::mutex> lk(sleep_mu_); }
            cv_.notify_all();
        }
    }

private:
    bool run_any() {
        for (int k = 0, n = n_rings_.load(); k < n; ++k)
            if (rings_[k]->run_one()) return true;
        return false;
    }
    bool any() {
        for (int k = 0, n = n_rings_.load(); k < n; ++k)
            if (rings_[k]->taken.load() < rings_[k]->pushed.load()) return true;
        return false;
    }
    void worker() {
        for (;;) {
            // the chunks of a transfer come some 50 us apart
            for (int spin = 0; spin < 4000; ++spin) {
                if (run_any()) spin = 0;
                else __builtin_ia32_pause();
            }
            std::unique_lock<std::mutex> lk(sleep_mu_);
            asleep_.fetch_add(1);
            cv_.wait(lk, [this] { return stop_ || any(); });
            asleep_.fetch_sub(1);
            if (stop_) return;
        }
    }

    std::mutex mu_;                      // rings_ and threads_
    Ring* rings_[kAllRings] = {};       // the first n_rings_ never change
    std::atomic<int> n_rings_{0};
    std::vector<std::thread> threads_;
    std::atomic<int> asleep_{0};
    std::mutex sleep_mu_;
    std::condition_variable cv_;
    bool stop_ = false;
};

namespace {

// A ring for the length of a transfer.
struct Lent {
    CopyPool* pool;
    Ring* r;
    Lent(CopyPool* p, hipStream_t s) : pool(p), r(p ? p->lend(s) : nullptr) {}
    ~Lent() {
        if (r) pool->give_back(r);
    }
};

// Whether the host side of every copy is pageable memory, which the runtime
// does not know.
bool pageable(const HostCopy* c, int n) {
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

size_t total(const HostCopy* c, int n) {
    size_t b = 0;
    for (int k = 0; k < n; ++k) b += c[k].row * c[k].rows;
    return b;
}

// Whether the rows of every copy follow each other in host memory.  The runtime
// moves other rows of pageable memory one by one, about 9 us each (a 1920x960
// image with a pitch of 2048: 8.8 ms, through the ring 0.06).
bool contiguous(const HostCopy* c, int n) {
    for (int k = 0; k < n; ++k)
        if (c[k].row != c[k].pitch && c[k].rows > 1) return false;
    return true;
}

hipError_t plain(hipStream_t s, const HostCopy* c, int n, hipMemcpyKind kind, bool wait) {
    const bool in = kind == hipMemcpyHostToDevice;
    for (int k = 0; k < n; ++k) {
        if (c[k].row * c[k].rows == 0) continue;
        const hipError_t e =
            contiguous(c + k, 1)
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

// Uploads without a ring: pitched rows are packed first.
hipError_t plain_up(hipStream_t s, const HostCopy* c, int n, bool wait) {
    if (contiguous(c, n)) return plain(s, c, n, hipMemcpyHostToDevice, wait);
    hipError_t e = hipSuccess;
    for (int k = 0; k < n && e == hipSuccess; ++k) {
        const size_t bytes = c[k].row * c[k].rows;
        uint8_t* p = contiguous(c + k, 1) ? nullptr : (uint8_t*)malloc(bytes);
        if (p) copy_span(Span{c[k], 0, bytes, p, false});
        const HostCopy flat = p ? flat_copy(p, c[k].dev, bytes) : c[k];
        e = plain(s, &flat, 1, hipMemcpyHostToDevice, true);
        free(p);
    }
    return e;
}

hipError_t small(Ring& r, hipStream_t s, const HostCopy* c, int n, bool out) {
    hipError_t e = r.dma_done(r.slot[0]);
    size_t at = 0;
    for (int k = 0; k < n && e == hipSuccess; ++k) {
        const size_t bytes = c[k].row * c[k].rows;
        if (bytes == 0) continue;
        if (!out) copy_span(Span{c[k], 0, bytes, r.pin + at, false});
        e = out ? hipMemcpyAsync(r.pin + at, c[k].dev, bytes, hipMemcpyDeviceToHost, s)
                : hipMemcpyAsync(c[k].dev, r.pin + at, bytes, hipMemcpyHostToDevice, s);
        at += bytes;
    }
    // an event for the next transfer to wait for would cost as much as the wait
    const hipError_t w = hipStreamSynchronize(s);
    if (e == hipSuccess) e = w;
    if (!out || e != hipSuccess) return e;
    at = 0;
    for (int k = 0; k < n; ++k) {
        const size_t bytes = c[k].row * c[k].rows;
        if (bytes) copy_span(Span{c[k], 0, bytes, r.pin + at, true});
        at += bytes;
    }
    return e;
}

}  // namespace

CopyPool* Copier::pool() {
    std::lock_guard<std::mutex> lk(mu_);
    if (!pool_) {
        try {
            pool_ = CopyPool::get();
        } catch (const std::exception&) {   // no memory: the runtime's copies
        }
    }
    return pool_.get();
}

// Chunk k (of this transfer) uses slot k % kSlots; the slots' earlier pieces
// are done (every transfer ends so), their DMAs perhaps not.
hipError_t Copier::to_host(hipStream_t s, const HostCopy* c, int n, bool fresh) {
    const size_t bytes = total(c, n);
    if (!pageable(c, n) || (fresh && bytes < kFresh)) return plain(s, c, n, hipMemcpyDeviceToHost, true);
    CopyPool* const pool = this->pool();
    const Lent lent(pool, s);
    if (!lent.r) return plain(s, c, n, hipMemcpyDeviceToHost, true);
    Ring& r = *lent.r;
    if (bytes < (n > 2 ? kAloneDownMaps : kAloneDown)) return small(r, s, c, n, true);
    const bool alone = !pool->start_threads(bytes);
    Walk w{c, n};
    uint64_t issued = 0, copied = 0;
    hipError_t e = hipSuccess;
    for (;;) {
        while (issued < copied + kSlots && !w.end()) {
            Ring::Slot& sl = r.slot[issued % kSlots];
            if ((e = r.dma_done(sl)) != hipSuccess) break;
            w.next(sl.p);
            sl.p.lin = r.pin + (issued % kSlots) * kChunk;
            sl.p.out = true;
            r.wait(sl.begin, sl.end);
            e = hipMemcpyAsync(sl.p.lin, (const uint8_t*)sl.p.c.dev + sl.p.off, sl.p.len, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) break;
            ++issued;
            // the last chunk is waited for by the stream itself, without an
            // event, after which the caller's next wait for it would cost 30 us
            if (w.end()) break;
            if ((e = hipEventRecord(sl.ev, s)) != hipSuccess) break;
            sl.dma = true;
        }
        if (e != hipSuccess || copied == issued) break;
        Ring::Slot& sl = r.slot[copied % kSlots];
        if ((e = sl.dma ? r.dma_done(sl) : hipStreamSynchronize(s)) != hipSuccess) break;
        sl.begin = r.next;
        pool->push(r, sl.p, alone);
        sl.end = r.next;
        ++copied;
    }
    for (const Ring::Slot& sl : r.slot) r.wait(sl.begin, sl.end);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e;
}

hipError_t Copier::to_device(hipStream_t s, const HostCopy* c, int n, Until until) {
    const bool wait_plain = until != Until::kQueued;   // the runtime may still read the host memory
    if (!pageable(c, n)) return plain(s, c, n, hipMemcpyHostToDevice, wait_plain);
    const size_t bytes = total(c, n);
    if (bytes >= kAloneUp && bytes < (n == 1 ? kPinnedOne : kPinned) && contiguous(c, n))
        return plain(s, c, n, hipMemcpyHostToDevice, wait_plain);
    CopyPool* const pool = this->pool();
    const Lent lent(pool, s);
    if (!lent.r) return plain_up(s, c, n, wait_plain);
    Ring& r = *lent.r;
    if (bytes < kAloneUp) return small(r, s, c, n, false);
    const bool alone = !pool->start_threads(bytes);
    Walk w{c, n};
    uint64_t pushed = 0, sent = 0;
    hipError_t e = hipSuccess;
    while (e == hipSuccess) {
        while (pushed < sent + kSlots && !w.end()) {
            Ring::Slot& sl = r.slot[pushed % kSlots];
            if ((e = r.dma_done(sl)) != hipSuccess) break;
            w.next(sl.p);
            sl.p.lin = r.pin + (pushed % kSlots) * kChunk;
            sl.p.out = false;
            sl.begin = r.next;
            pool->push(r, sl.p, alone);
            sl.end = r.next;
            ++pushed;
        }
        if (e != hipSuccess || sent == pushed) break;
        Ring::Slot& sl = r.slot[sent % kSlots];
        r.wait(sl.begin, sl.end);
        e = hipMemcpyAsync((uint8_t*)sl.p.c.dev + sl.p.off, sl.p.lin, sl.p.len, hipMemcpyHostToDevice, s);
        ++sent;
        // where the transfer ends with a wait for the stream, without an event
        // for the chunks that no other follows in their slots (see to_host)
        if (until == Until::kDone && w.end()) continue;
        if (e == hipSuccess) e = hipEventRecord(sl.ev, s);
        if (e == hipSuccess) sl.dma = true;
    }
    for (const Ring::Slot& sl : r.slot) r.wait(sl.begin, sl.end);   // no thread reads the caller's memory any more
    if (e == hipSuccess && until != Until::kDone) return e;
    const hipError_t d = hipStreamSynchronize(s);
    for (Ring::Slot& sl : r.slot) sl.dma = false;
    return e == hipSuccess ? d : e;
}

void Copier::copy(void* dst, const void* src, size_t bytes) {
    CopyPool* const pool = bytes < kAloneUp ? nullptr : this->pool();
    const Lent lent(pool, nullptr);
    if (!lent.r || !pool->start_threads(bytes)) {
        memcpy(dst, src, bytes);
        return;
    }
    Ring& r = *lent.r;
    const uint64_t begin = r.next;
    pool->push(r, Span{flat_copy(dst, nullptr, bytes), 0, bytes, (uint8_t*)const_cast<void*>(src), true}, false);
    r.wait(begin, r.next);
}

}  // namespace pmp
