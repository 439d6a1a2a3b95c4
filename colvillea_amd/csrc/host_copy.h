/* host_copy.h -- copies between device memory and a caller's pageable
 * buffers through pinned staging, by several threads for large ones. */
#ifndef CLPT_HOST_COPY_H
#define CLPT_HOST_COPY_H

#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

namespace clpt
{
/* The runtime's own copy to pageable memory moves 1 MB at a time through one
 * thread.  Here a copy is queued on the stream in parts of 2 MiB into two
 * pinned slots, and kThreads threads copy the parts out (or in) as they
 * arrive; a slot is queued again as soon as it is empty.  Copies below kMin,
 * copies to and from memory that is not pageable, and all copies where no
 * pinned memory can be had or another device is current, go the runtime's way.
 *
 * One HostCopier serves one context (it is not thread-safe).  Its staging and
 * threads are made at the first copy that needs them and kept for the
 * context's life; the host's first touch of new pinned memory costs 100 us
 * and more per MiB with all threads, so there is little of it.  A film of
 * 1920x1080 (31.6 MiB) read back, first and later times in a context: 1.9 and
 * 1.9 ms through the runtime, 3.1 and 1.08 with 32 slots of 1 MiB each queued
 * once, 1.0 and 0.85 with these two; two slots of 1 MiB 1.07 later, of 4 MiB
 * or four of 2 MiB no faster and up to 1 ms longer the first time.  Below
 * kMin nothing is gained (0.3 MiB takes 39 us, staged 45); behind a render
 * 1.2 MiB staged is 13 us sooner than the runtime's, which starts when the
 * render has ended.  But up to 16 KiB the runtime has a slower way to
 * pageable memory: such readbacks go through a slot of that size from a
 * context's third on (one alone would not repay it), 18 instead of 26 us. */
class HostCopier
{
public:
    explicit HostCopier(int device) : device_(device) {}
    ~HostCopier();
    HostCopier(const HostCopier&) = delete;
    HostCopier& operator=(const HostCopier&) = delete;

    /* Queues the copy behind the stream's work and waits for it. */
    hipError_t to_host(hipStream_t s, void* dst, const void* dev, size_t bytes);
    /* Copies src into staging and queues the transfer; src may be reused on
     * return, the stream's later work sees the data. */
    hipError_t from_host(hipStream_t s, void* dev, const void* src, size_t bytes);

private:
    static constexpr size_t   kTiny    = 16u << 10;
    static constexpr size_t   kMin     = 1u << 20;
    static constexpr size_t   kPart    = 2u << 20; /* one transfer, one slot */
    static constexpr size_t   kSlots   = 2;
    static constexpr size_t   kPiece   = 128u << 10; /* what a thread copies at a time */
    static constexpr size_t   kPer     = kPart / kPiece;
    static constexpr unsigned kThreads = 8; /* the caller's among them */

    /* staging and events for a copy; false: there are none to be had */
    bool reserve(size_t bytes);
    void touch();
    /* the slot of tiny readbacks, once there have been several */
    bool tiny();
    void wait_upload(size_t k);
    /* job(k) for k = 0..n-1 on the threads from begin() on; the caller's takes
     * those below `end` that are left in help() and all in finish(), which
     * returns when all are done */
    void begin(size_t n, const std::function<void(size_t)>& job);
    void help(size_t end);
    void finish();
    void work();

    int                      device_; /* the streams' */
    char*                    stage_ = nullptr;
    void*                    tiny_  = nullptr;
    unsigned                 ntiny_ = 0;
    size_t                   room_ = 0, slots_ = 0;
    bool                     touched_ = true;
    bool                     refused_ = false; /* pinned memory or an event could not be had */
    hipEvent_t               ev_[kSlots] = {}; /* the last transfer of each slot */
    bool                     up_pending_[kSlots] = {}; /* it was an upload and may not be done */
    std::atomic<size_t>      left_[kSlots] = {}; /* pieces of the slot's part still to be copied */
    std::vector<std::thread> threads_;
    std::mutex               mu_;
    std::condition_variable  wake_, idle_;
    const std::function<void(size_t)>* job_ = nullptr;
    std::atomic<size_t>      next_{0};
    size_t                   njobs_ = 0;
    uint64_t                 round_ = 0;
    unsigned                 busy_  = 0;
    bool                     stop_  = false;
};
} // namespace clpt

#endif
