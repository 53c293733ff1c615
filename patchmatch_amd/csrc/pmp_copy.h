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
// Rings and threads are the process's (CopyPool): a ring's pinned pages cost
// 0.38 ms per MiB when first touched, which every context's first transfers
// would pay again (the cleaner's first call on five 1920x960 maps with two
// other contexts open: 3.2 ms with a ring to each context, 1.8 with these,
// 2.5 by the runtime's copies).  A transfer borrows a ring; the pool ends with
// the last context that has used it.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <memory>
#include <mutex>

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

class CopyPool;

// A context's copies, from any threads; on the calling thread's current device.
class Copier {
public:
    // Device to host after the work queued on s; complete on return.  fresh:
    // to memory that has hardly been touched since it was allocated.
    hipError_t to_host(hipStream_t s, const HostCopy* c, int n, bool fresh = false);
    // Host to device in stream order.
    hipError_t to_device(hipStream_t s, const HostCopy* c, int n, Until until = Until::kDone);
    // Host to host.
    void copy(void* dst, const void* src, size_t bytes);

private:
    CopyPool* pool();
    std::mutex mu_;
    std::shared_ptr<CopyPool> pool_;
};

}  // namespace pmp
