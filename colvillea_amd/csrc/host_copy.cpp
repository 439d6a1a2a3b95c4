/* host_copy.cpp -- see host_copy.h. */
#include "host_copy.h"

#include <algorithm>
#include <cstring>

namespace clpt
{
HostCopier::~HostCopier()
{
    {
        std::lock_guard<std::mutex> l(mu_);
        stop_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : threads_)
        t.join();
    for (size_t k = 0; k < kSlots; ++k)
    {
        wait_upload(k);
        if (ev_[k])
            (void)hipEventDestroy(ev_[k]);
    }
    if (stage_)
        (void)hipHostFree(stage_);
    if (tiny_)
        (void)hipHostFree(tiny_);
}

/* Whether p is ordinary memory, which the runtime would copy through staging
 * of its own; pinned and managed memory it reads and writes directly. */
static bool pageable(const void* p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess)
    {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeUnregistered;
}

/* An upload may still be reading slot k. */
void HostCopier::wait_upload(size_t k)
{
    if (up_pending_[k])
        (void)hipEventSynchronize(ev_[k]);
    up_pending_[k] = false;
}

bool HostCopier::reserve(size_t bytes)
{
    /* events are the current device's, and the stream takes its own's only */
    int device = -1;
    if (refused_ || hipGetDevice(&device) != hipSuccess || device != device_)
        return false;
    for (size_t k = 0; k < kSlots; ++k)
        wait_upload(k);
    /* as much of the first slot as is needed, or whole slots */
    const size_t need = bytes <= kPart ? 1u : std::min(kSlots, (bytes + kPart - 1) / kPart);
    const size_t room = bytes <= kPart ? (bytes + kPiece - 1) / kPiece * kPiece : need * kPart;
    hipError_t   e    = hipSuccess;
    if (room > room_)
    {
        if (stage_)
            (void)hipHostFree(stage_);
        stage_  = nullptr;
        room_   = 0;
        slots_  = 0;
        void* p = nullptr;
        e       = hipHostMalloc(&p, room, hipHostMallocDefault);
        if (e == hipSuccess)
        {
            stage_   = static_cast<char*>(p);
            room_    = room;
            slots_   = need;
            touched_ = false;
        }
    }
    for (size_t k = 0; k < need && e == hipSuccess; ++k)
        if (!ev_[k])
            e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
    if (e != hipSuccess)
    {
        (void)hipGetLastError(); /* not for the next launch to report */
        if (stage_)
            (void)hipHostFree(stage_);
        stage_   = nullptr;
        room_    = 0;
        slots_   = 0;
        refused_ = true;
        return false;
    }
    return true;
}

/* New staging's pages are mapped as the host first touches them, 100 us and
 * more per MiB: before a readback waits, while the stream's work goes on. */
void HostCopier::touch()
{
    if (touched_)
        return;
    touched_ = true;
    const std::function<void(size_t)> job = [&](size_t i) {
        for (size_t at = 0; at < kPiece; at += 4096)
            *static_cast<volatile char*>(stage_ + i * kPiece + at) = 0;
    };
    begin(room_ / kPiece, job);
    finish();
}

void HostCopier::work()
{
    uint64_t seen = 0;
    for (;;)
    {
        const std::function<void(size_t)>* job = nullptr;
        size_t                             n   = 0;
        {
            std::unique_lock<std::mutex> l(mu_);
            wake_.wait(l, [&] { return stop_ || (job_ && round_ != seen); });
            if (stop_)
                return;
            seen = round_;
            job  = job_;
            n    = njobs_;
            ++busy_;
        }
        for (size_t k = next_++; k < n; k = next_++)
            (*job)(k);
        {
            std::lock_guard<std::mutex> l(mu_);
            --busy_;
        }
        idle_.notify_one();
    }
}

void HostCopier::begin(size_t n, const std::function<void(size_t)>& job)
{
    /* a thread per MiB at most: starting one costs 10 to 15 us */
    const size_t want = std::min<size_t>(kThreads, n * kPiece >> 20);
    try
    {
        while (threads_.size() + 1 < want)
            threads_.emplace_back([this] { work(); });
    }
    catch (...)
    {
        /* as many as could be started; the caller's thread does the rest */
    }
    {
        std::lock_guard<std::mutex> l(mu_);
        job_   = &job;
        njobs_ = n;
        next_  = 0;
        ++round_;
    }
    wake_.notify_all();
}

void HostCopier::help(size_t end)
{
    for (size_t k = next_; k < end; k = next_)
        if (next_.compare_exchange_weak(k, k + 1))
            (*job_)(k);
}

void HostCopier::finish()
{
    help(njobs_);
    /* no thread takes the job up any more, and those that did are done */
    std::unique_lock<std::mutex> l(mu_);
    job_ = nullptr;
    idle_.wait(l, [&] { return busy_ == 0; });
}

bool HostCopier::tiny()
{
    if (!tiny_ && !refused_ && ++ntiny_ > 2u)
    {
        void* p = nullptr;
        if (hipHostMalloc(&p, kTiny, hipHostMallocDefault) == hipSuccess)
            tiny_ = p;
        else
        {
            (void)hipGetLastError();
            refused_ = true;
        }
    }
    return tiny_ != nullptr;
}

hipError_t HostCopier::to_host(hipStream_t s, void* dst, const void* dev, size_t bytes)
{
    if (!bytes)
        return hipStreamSynchronize(s);
    hipError_t e = hipSuccess;
    if (bytes <= kTiny && tiny())
    {
        e = hipMemcpyAsync(tiny_, dev, bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess)
            e = hipStreamSynchronize(s);
        if (e == hipSuccess)
            std::memcpy(dst, tiny_, bytes);
        return e;
    }
    if (bytes < kMin || !pageable(dst) || !reserve(bytes))
    {
        e = hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    touch();
    char*        out    = static_cast<char*>(dst);
    const char*  in     = static_cast<const char*>(dev);
    const size_t parts  = (bytes + kPart - 1) / kPart, pieces = (bytes + kPiece - 1) / kPiece;
    const auto   end_of = [&](size_t p) { return std::min(pieces, (p + 1) * kPer); };
    const auto   queue  = [&](size_t p) {
        const size_t k = p % slots_;
        left_[k]       = end_of(p) - p * kPer;
        const hipError_t q =
            hipMemcpyAsync(stage_ + k * kPart, in + p * kPart, std::min(kPart, bytes - p * kPart), hipMemcpyDeviceToHost, s);
        return q == hipSuccess ? hipEventRecord(ev_[k], s) : q;
    };
    std::atomic<size_t> arrived{0}; /* parts */
    std::atomic<bool>   failed{false};
    const std::function<void(size_t)> job = [&](size_t i) {
        const size_t p = i / kPer;
        while (arrived.load(std::memory_order_acquire) <= p)
            std::this_thread::yield();
        if (!failed)
            std::memcpy(out + i * kPiece, stage_ + p % slots_ * kPart + i % kPer * kPiece, std::min(kPiece, bytes - i * kPiece));
        left_[p % slots_].fetch_sub(1, std::memory_order_release);
    };
    for (size_t p = 0; p < std::min(slots_, parts) && e == hipSuccess; ++p)
        e = queue(p);
    /* The copies lie behind all of the stream's work, a whole render perhaps:
     * the caller's thread waits for that alone, and the others wake to
     * transfers in progress. */
    if (e == hipSuccess)
        e = hipEventSynchronize(ev_[0]);
    if (e == hipSuccess)
    {
        begin(pieces, job);
        for (size_t p = 0; p < parts; ++p)
        {
            if (p && e == hipSuccess)
                e = hipEventSynchronize(ev_[p % slots_]);
            if (e != hipSuccess)
                failed = true;
            arrived.store(p + 1, std::memory_order_release);
            help(end_of(p));
            if (p + slots_ < parts)
            {
                while (left_[p % slots_].load(std::memory_order_acquire))
                    std::this_thread::yield();
                if (e == hipSuccess)
                    e = queue(p + slots_);
                else
                    left_[p % slots_] = end_of(p + slots_) - (p + slots_) * kPer;
            }
        }
        finish();
    }
    if (e != hipSuccess)
        (void)hipStreamSynchronize(s); /* parts still queued write the staging */
    return e;
}

hipError_t HostCopier::from_host(hipStream_t s, void* dev, const void* src, size_t bytes)
{
    if (!bytes)
        return hipSuccess;
    hipError_t e = hipSuccess;
    if (bytes < kMin || !pageable(src) || !reserve(bytes))
    {
        e = hipMemcpyAsync(dev, src, bytes, hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e; /* src may be reused */
    }
    touched_ = true; /* the copy into it does */
    const char*  in     = static_cast<const char*>(src);
    char*        out    = static_cast<char*>(dev);
    const size_t parts  = (bytes + kPart - 1) / kPart, pieces = (bytes + kPiece - 1) / kPiece;
    const auto   end_of = [&](size_t p) { return std::min(pieces, (p + 1) * kPer); };
    std::atomic<size_t> open{std::min(slots_, parts)}; /* parts whose slot may be written */
    const std::function<void(size_t)> job = [&](size_t i) {
        const size_t p = i / kPer;
        while (open.load(std::memory_order_acquire) <= p)
            std::this_thread::yield();
        std::memcpy(stage_ + p % slots_ * kPart + i % kPer * kPiece, in + i * kPiece, std::min(kPiece, bytes - i * kPiece));
        left_[p % slots_].fetch_sub(1, std::memory_order_release);
    };
    for (size_t p = 0; p < open; ++p)
        left_[p] = end_of(p) - p * kPer;
    begin(pieces, job);
    for (size_t p = 0; p < parts; ++p)
    {
        const size_t k = p % slots_;
        help(end_of(p));
        while (left_[k].load(std::memory_order_acquire))
            std::this_thread::yield();
        if (e == hipSuccess)
            e = hipMemcpyAsync(out + p * kPart, stage_ + k * kPart, std::min(kPart, bytes - p * kPart), hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipEventRecord(ev_[k], s);
        up_pending_[k] = e == hipSuccess;
        if (p + slots_ < parts)
        {
            wait_upload(k);
            left_[k] = end_of(p + slots_) - (p + slots_) * kPer;
            open.store(p + slots_ + 1, std::memory_order_release);
        }
    }
    finish();
    if (e != hipSuccess)
        (void)hipStreamSynchronize(s);
    return e;
}
} // namespace clpt
