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
/* The runtime's own copy to pageable memory goes through its staging 1 MB at
 * a time, 20 us of transfer and then 70 us in one thread that copies the
 * piece and faults its pages in: 2.9 ms for a 1080p RGBA32F film.  Here the
 * pieces of a copy are queued on the stream together, into pinned slots, and
 * kThreads threads copy them out as they arrive.  One HostCopier serves one
 * context (it is not thread-safe); it holds at most kStage bytes of pinned
 * memory and its threads, both made at the first copy that needs them and
 * kept for the context's life.  Copies to and
 * from memory that is not pageable, and all copies where no pinned memory can
 * be had, go the runtime's way. */
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
    static constexpr size_t   kPiece   = 1u << 20;
    static constexpr size_t   kSlots   = 32;
    static constexpr size_t   kStage   = kPiece * kSlots;
    static constexpr unsigned kThreads = 8; /* the caller's among them */

    /* staging, events and threads for a copy; false: there are none to be had */
    bool reserve(size_t bytes);
    void wait_upload();
    /* job(k) for k = 0..n-1 on the threads; returns when all are done */
    void run(size_t n, const std::function<void(size_t)>& job);
    void work();

    int                      device_;
    char*                    stage_ = nullptr;
    size_t                   cap_   = 0;
    bool                     refused_ = false; /* pinned memory or an event could not be had */
    hipEvent_t               ev_[kSlots] = {};
    hipEvent_t               up_ = nullptr; /* the last from_host transfer */
    bool                     up_pending_ = false;
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
