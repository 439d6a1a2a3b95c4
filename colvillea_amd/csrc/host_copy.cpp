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
    wait_upload();
    for (hipEvent_t e : ev_)
        if (e)
            (void)hipEventDestroy(e);
    if (up_)
        (void)hipEventDestroy(up_);
    if (stage_)
        (void)hipHostFree(stage_);
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

/* An upload may still be reading the staging. */
void HostCopier::wait_upload()
{
    if (up_pending_)
        (void)hipEventSynchronize(up_);
    up_pending_ = false;
}

bool HostCopier::reserve(size_t bytes)
{
    if (refused_)
        return false;
    wait_upload();
    const size_t need = std::min(kStage, std::max<size_t>((bytes + kPiece - 1) / kPiece * kPiece, kPiece));
    hipError_t   e    = hipSuccess;
    if (need > cap_)
    {
        if (stage_)
            (void)hipHostFree(stage_);
        stage_  = nullptr;
        cap_    = 0;
        void* p = nullptr;
        e       = hipHostMalloc(&p, need, hipHostMallocDefault);
        if (e == hipSuccess)
        {
            stage_ = static_cast<char*>(p);
            cap_   = need;
        }
    }
    for (size_t k = 0; k < need / kPiece && e == hipSuccess; ++k)
        if (!ev_[k])
            e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
    if (e == hipSuccess && !up_)
        e = hipEventCreateWithFlags(&up_, hipEventDisableTiming);
    if (e != hipSuccess)
    {
        (void)hipGetLastError(); /* not for the next launch to report */
        if (stage_)
            (void)hipHostFree(stage_);
        stage_   = nullptr;
        cap_     = 0;
        refused_ = true;
        return false;
    }
    /* a thread per piece at most: starting one costs 10 to 15 us, which a
     * context that only makes small copies would pay for nothing */
    const size_t want = need <= 2 * kPiece ? 0u : std::min<size_t>(kThreads, need / kPiece) - 1u;
    try
    {
        while (threads_.size() < want)
            threads_.emplace_back([this] { work(); });
    }
    catch (...)
    {
        /* as many as could be started; the caller's thread does the rest */
    }
    return true;
}

void HostCopier::work()
{
    (void)hipSetDevice(device_);
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

void HostCopier::run(size_t n, const std::function<void(size_t)>& job)
{
    if (n < 3 || threads_.empty())
    {
        for (size_t k = 0; k < n; ++k)
            job(k);
        return;
    }
    {
        std::lock_guard<std::mutex> l(mu_);
        job_   = &job;
        njobs_ = n;
        next_  = 0;
        ++round_;
    }
    wake_.notify_all();
    for (size_t k = next_++; k < n; k = next_++)
        job(k);
    /* no thread takes the job up any more, and those that did are done */
    std::unique_lock<std::mutex> l(mu_);
    job_ = nullptr;
    idle_.wait(l, [&] { return busy_ == 0; });
}

hipError_t HostCopier::to_host(hipStream_t s, void* dst, const void* dev, size_t bytes)
{
    if (!bytes)
        return hipStreamSynchronize(s);
    hipError_t e;
    if (!pageable(dst) || !reserve(bytes))
    {
        e = hipMemcpyAsync(dst, dev, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    char*       out = static_cast<char*>(dst);
    const char* in  = static_cast<const char*>(dev);
    for (size_t at = 0; at < bytes; at += cap_)
    {
        const size_t part = std::min(cap_, bytes - at), n = (part + kPiece - 1) / kPiece;
        for (size_t k = 0; k < n; ++k)
        {
            const size_t len = std::min(kPiece, part - k * kPiece);
            e = hipMemcpyAsync(stage_ + k * kPiece, in + at + k * kPiece, len, hipMemcpyDeviceToHost, s);
            if (e == hipSuccess)
                e = hipEventRecord(ev_[k], s);
            if (e != hipSuccess)
            {
                (void)hipStreamSynchronize(s); /* the pieces queued so far */
                return e;
            }
        }
        /* the copies lie behind all of the stream's work, a whole render
         * perhaps: the caller's thread waits for that alone, and the others
         * wake to transfers in progress (an event wait polls) */
        e = hipEventSynchronize(ev_[0]);
        if (e != hipSuccess)
            return e;
        std::atomic<int> bad{(int)hipSuccess};
        run(n, [&](size_t k) {
            const hipError_t w = hipEventSynchronize(ev_[k]);
            if (w != hipSuccess)
                bad = (int)w;
            else
                std::memcpy(out + at + k * kPiece, stage_ + k * kPiece, std::min(kPiece, part - k * kPiece));
        });
        if (bad != (int)hipSuccess)
            return (hipError_t)bad.load();
    }
    return hipSuccess;
}

hipError_t HostCopier::from_host(hipStream_t s, void* dev, const void* src, size_t bytes)
{
    if (!bytes)
        return hipSuccess;
    hipError_t e;
    if (!pageable(src) || !reserve(bytes))
    {
        e = hipMemcpyAsync(dev, src, bytes, hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e; /* src may be reused */
    }
    const char* in  = static_cast<const char*>(src);
    char*       out = static_cast<char*>(dev);
    for (size_t at = 0; at < bytes; at += cap_)
    {
        wait_upload();
        const size_t part = std::min(cap_, bytes - at);
        run((part + kPiece - 1) / kPiece, [&](size_t k) {
            std::memcpy(stage_ + k * kPiece, in + at + k * kPiece, std::min(kPiece, part - k * kPiece));
        });
        e = hipMemcpyAsync(out + at, stage_, part, hipMemcpyHostToDevice, s);
        if (e == hipSuccess)
            e = hipEventRecord(up_, s);
        if (e != hipSuccess)
        {
            (void)hipStreamSynchronize(s);
            return e;
        }
        up_pending_ = true;
    }
    return hipSuccess;
}
} // namespace clpt
