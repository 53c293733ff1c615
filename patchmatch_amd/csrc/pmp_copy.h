// pmp_copy.h -- copies between the callers' pageable host memory and the GPU.
//
// A pageable copy is the runtime's own staging on one thread: that thread's
// memory copy, and the page faults of a buffer that nobody has touched yet,
// set its rate, not the link (51.6 MB of maps into fresh arrays: 3.8 ms,
// 14 GB/s).  Here a transfer goes through a ring of pinned chunks: the DMA
// engine works on some while several threads copy others from or to the
// caller's memory.
//
// Memory that the runtime knows (pinned, device, managed) goes straight.
//
// A Copier belongs to one context; its threads start with the first large
// transfer and end with it.  One transfer runs at a time (transfers from
// several threads take turns).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace pmp {

// rows of `row` bytes, `pitch` bytes apart in host memory and contiguous on
// the device
struct HostCopy {
    void* host;
    void* dev;
    size_t row, rows, pitch;
};

inline HostCopy flat_copy(const void* host, const void* dev, size_t bytes) {
    return HostCopy{const_cast<void*>(host), const_cast<void*>(dev), bytes, 1, bytes};
}

// What an upload has done when it returns.
enum class Until {
    kDone,     // it is complete
    kRead,     // the host memory has been read
    kQueued,   // it is queued: the caller waits for the stream before it returns (an upload that failed is not)
};

class Copier {
public:
    ~Copier();
    // Device to host after the work queued on s; complete on return.  fresh:
    // to memory that has hardly been touched since it was allocated.
    hipError_t to_host(hipStream_t s, const HostCopy* c, int n, bool fresh = false);
    // Host to device in stream order.
    hipError_t to_device(hipStream_t s, const HostCopy* c, int n, Until until = Until::kDone);
    // Host to host.
    void copy(void* dst, const void* src, size_t bytes);

private:
    // A chunk is one DMA, with 14 us of fixed costs: 48 MiB in chunks of 1 MiB
    // ran at 31 GB/s, of 2 at 40, of 4 at 46.  Its pieces are what a thread
    // copies at a time.  More than two chunks in flight gained nothing, and
    // their pinned pages cost 0.35 ms per MiB when first touched.
    static constexpr size_t kChunk = size_t(4) << 20, kPiece = size_t(256) << 10;
    static constexpr int kSlots = 2;
    static constexpr int kTasks = 256;       // a power of two above kSlots * kChunk / kPiece
    static constexpr int kThreads = 8;
    // Transfers below these are copied by the caller alone, in one chunk: waking
    // the threads costs more (normals of 328x182, 716 KB down: 66 us alone, 52
    // with them; a 614 KB image up: 75 and 76).
    static constexpr size_t kAloneDown = size_t(512) << 10, kAloneUp = size_t(768) << 10;
    // Uploads of contiguous rows from kAloneUp to this are the runtime's own: it pins the pages and
    // copies from them (five 640x320 maps to the cleaner and back: 222 us, with
    // the threads 292; of 800x400: 363 and 353; of 1363x677: 863 and 638).
    static constexpr size_t kPinned = size_t(6) << 20;
    // So are downloads to fresh memory below this: pinning takes the page
    // faults at once, which the threads would fight over (the pruner's points
    // and map: of 320x160 views 189 us, with the threads 225; of 640x320 366
    // and 375; of 1098x494 885 and 785).
    static constexpr size_t kFresh = size_t(12) << 20;
    struct Span {               // bytes [off, off + len) of c, contiguous at lin
        HostCopy c;
        size_t off, len;
        uint8_t* lin;
        bool out;               // from lin to c.host
    };
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
    struct Walk;                         // the chunks of a list of copies
    hipError_t small(hipStream_t s, const HostCopy* c, int n, bool out);
    bool start_ring();
    bool start_threads();
    static void run(const Span& p);
    bool run_one();
    void worker();
    void push(const Span& p, bool alone);
    void wait(uint64_t begin, uint64_t end);
    hipError_t dma_done(Slot& s);

    std::mutex mu_;                      // a transfer
    bool ring_tried_ = false, ring_ok_ = false, threads_tried_ = false;
    uint8_t* pin_ = nullptr;
    Slot slot_[kSlots];
    Task task_[kTasks];
    uint64_t next_ = 0;                  // the next piece's ticket; its task is ticket % kTasks
    std::atomic<uint64_t> pushed_{0}, taken_{0};
    std::atomic<int> asleep_{0};
    std::mutex sleep_mu_;
    std::condition_variable cv_;
    bool stop_ = false;
    std::vector<std::thread> threads_;
};

}  // namespace pmp
