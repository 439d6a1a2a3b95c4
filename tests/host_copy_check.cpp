/* Host check of the staged copies (colvillea_amd/csrc/host_copy.cpp) against
 * a stand-in for the HIP calls they make: one stream whose operations a
 * thread of its own carries out in order, behind a gate that stands for a
 * render still running.  `host_copy_check CASE` prints "ok" or what failed. */
#include "../colvillea_amd/csrc/host_copy.h"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>

namespace
{
std::mutex                        mu;
std::condition_variable           cv;
std::deque<std::function<void()>> ops;
uint64_t                          queued = 0, done = 0;
bool                              gate = true, quit = false, refuse_pinned = false;
std::map<char*, size_t>           pinned;
size_t                            pinned_total = 0, pinned_calls = 0;
size_t                            staged_copies = 0, direct_copies = 0;
int                               waiting = 0; /* threads inside hipEventSynchronize */
hipError_t                        last = hipSuccess;
int                               current_device = 0; /* the stream's is 0 */

bool in_pinned(const void* p)
{
    const char* c = static_cast<const char*>(p);
    for (const auto& r : pinned)
        if (c >= r.first && c < r.first + r.second)
            return true;
    return false;
}

void device()
{
    std::unique_lock<std::mutex> l(mu);
    for (;;)
    {
        cv.wait(l, [] { return quit || (gate && !ops.empty()); });
        if (quit)
            return;
        const auto op = ops.front();
        ops.pop_front();
        l.unlock();
        op();
        l.lock();
        ++done;
        cv.notify_all();
    }
}

uint64_t enqueue(std::function<void()> f)
{
    std::lock_guard<std::mutex> l(mu);
    ops.push_back(std::move(f));
    cv.notify_all();
    return ++queued;
}

void wait_for(uint64_t at)
{
    std::unique_lock<std::mutex> l(mu);
    cv.wait(l, [&] { return done >= at; });
}

void set_gate(bool open)
{
    std::lock_guard<std::mutex> l(mu);
    gate = open;
    cv.notify_all();
}

int failures = 0;
void expect(bool good, const char* what, size_t a, size_t b)
{
    if (!good && failures++ < 10)
        std::printf("%s: %zu %zu\n", what, a, b);
}
} // namespace

struct ihipEvent_t
{
    std::atomic<uint64_t> at{0};
    int                   device = current_device;
};

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> l(mu);
    if (refuse_pinned)
        return last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    pinned[static_cast<char*>(*p)] = n;
    pinned_total += n;
    ++pinned_calls;
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    std::lock_guard<std::mutex> l(mu);
    pinned_total -= pinned[static_cast<char*>(p)];
    pinned.erase(static_cast<char*>(p));
    std::free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    std::lock_guard<std::mutex> l(mu);
    std::memset(a, 0, sizeof(*a));
    a->type = in_pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t)
{
    const void* host = kind == hipMemcpyDeviceToHost ? d : s;
    bool        page;
    {
        std::lock_guard<std::mutex> l(mu);
        page = !in_pinned(host);
        ++(page ? direct_copies : staged_copies);
    }
    const uint64_t at = enqueue([=] { std::memcpy(d, s, n); });
    if (page)
        wait_for(at); /* as the runtime does with pageable memory */
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = new ihipEvent_t;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    if (e->device != 0)
        return last = hipErrorInvalidHandle; /* not the stream's device */
    e->at = enqueue([] {});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    {
        std::lock_guard<std::mutex> l(mu);
        ++waiting;
    }
    wait_for(e->at);
    std::lock_guard<std::mutex> l(mu);
    --waiting;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    uint64_t at;
    {
        std::lock_guard<std::mutex> l(mu);
        at = queued;
    }
    wait_for(at);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d)
{
    *d = current_device;
    return hipSuccess;
}
hipError_t hipGetLastError(void)
{
    std::lock_guard<std::mutex> l(mu);
    const hipError_t e = last;
    last               = hipSuccess;
    return e;
}
}

using clpt::HostCopier;
static constexpr size_t MiB = 1u << 20;

static std::vector<char> bytes_of(size_t n, uint32_t seed)
{
    std::vector<char> v(n);
    v.reserve(n + 1); /* not null for no bytes */
    uint32_t          x = seed * 2654435761u + 1u;
    for (size_t i = 0; i < n; ++i)
    {
        x    = x * 1664525u + 1013904223u;
        v[i] = (char)(x >> 24);
    }
    return v;
}

/* n bytes down and up again; the caller's memory is as the copy left it */
static void both_ways(HostCopier& c, size_t n, uint32_t seed)
{
    const std::vector<char> src = bytes_of(n, seed);
    std::vector<char>       out(n + 1, 'x'), dev(n + 1, 'y');
    expect(c.to_host(nullptr, out.data(), src.data(), n) == hipSuccess, "to_host fails", n, 0);
    expect(std::memcmp(out.data(), src.data(), n) == 0 && out[n] == 'x', "to_host differs", n, 0);
    expect(c.from_host(nullptr, dev.data(), src.data(), n) == hipSuccess, "from_host fails", n, 0);
    (void)hipStreamSynchronize(nullptr);
    expect(std::memcmp(dev.data(), src.data(), n) == 0 && dev[n] == 'y', "from_host differs", n, 0);
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    std::thread       dev(device);
    {
        HostCopier c(0);
        if (what == "sizes")
        {
            /* around pieces, the sizes from which several threads copy, the
             * whole staging and several times it, up and down in turn */
            for (size_t n : {(size_t)0, (size_t)1, MiB - 1, MiB, MiB + 1, 5 * MiB / 4, 2 * MiB - 1, 2 * MiB, 2 * MiB + 1, 5 * MiB / 2, 3 * MiB + 7, 4 * MiB,
                             4 * MiB + 1, 8 * MiB - 1, 8 * MiB, 8 * MiB + 1, 17 * MiB / 2, 12 * MiB, 12 * MiB + 5, 16 * MiB,
                             32 * MiB + 3, 70 * MiB + 1, 5 * MiB, (size_t)100, (size_t)16383, (size_t)16384, (size_t)16385, (size_t)3})
                both_ways(c, n, (uint32_t)n + 1u);
        }
        else if (what == "no_pinned")
        {
            /* no pinned memory: the copies go the runtime's way, and leave no
             * error for the next launch to report */
            refuse_pinned = true;
            for (size_t n : {(size_t)100, 3 * MiB, 40 * MiB + 1, (size_t)7, (size_t)8, (size_t)9})
                both_ways(c, n, 3u);
            expect(hipGetLastError() == hipSuccess, "error left", 0, 0);
            expect(staged_copies == 0, "staged copies", staged_copies, 0);
            refuse_pinned = false;
        }
        else if (what == "pinned")
        {
            /* the caller's own pinned memory is written and read directly */
            const size_t n = 5 * MiB + 3;
            void*        own = nullptr;
            (void)hipHostMalloc(&own, n, 0);
            const std::vector<char> src = bytes_of(n, 9u);
            std::vector<char>       up(n);
            expect(c.to_host(nullptr, own, src.data(), n) == hipSuccess, "to_host fails", n, 0);
            expect(std::memcmp(own, src.data(), n) == 0, "to_host differs", n, 0);
            expect(c.from_host(nullptr, up.data(), own, n) == hipSuccess, "from_host fails", n, 0);
            std::memset(own, 0, n); /* src may be reused on return */
            (void)hipStreamSynchronize(nullptr);
            expect(std::memcmp(up.data(), src.data(), n) == 0, "from_host differs", n, 0);
            expect(staged_copies == 2 && direct_copies == 0, "copies", staged_copies, direct_copies);
            expect(pinned_calls == 1, "pinned allocations", pinned_calls, 1);
            (void)hipHostFree(own);
        }
        else if (what == "wait")
        {
            /* a readback behind a render in progress: one thread waits */
            set_gate(false);
            const size_t            n = 24 * MiB + 5;
            const std::vector<char> src = bytes_of(n, 5u);
            std::vector<char>       out(n);
            std::thread             caller([&] {
                expect(c.to_host(nullptr, out.data(), src.data(), n) == hipSuccess, "to_host fails", n, 0);
            });
            int most = 0;
            for (int k = 0; k < 100; ++k)
            {
                std::this_thread::sleep_for(std::chrono::milliseconds(2));
                std::lock_guard<std::mutex> l(mu);
                most = std::max(most, waiting);
            }
            expect(most == 1, "threads waiting for the render", (size_t)most, 1);
            set_gate(true);
            caller.join();
            expect(out == src, "to_host differs", n, 0);
        }
        else if (what == "setup")
        {
            /* small copies make no staging; no copy makes more than 4 MiB */
            for (size_t n : {(size_t)1, MiB / 2, MiB - 1})
                both_ways(c, n, 4u);
            expect(pinned_calls == 0, "pinned allocations of small copies", pinned_calls, 0);
            for (uint32_t k = 0; k < 5u; ++k)
            {
                both_ways(c, 16384u, k);
                both_ways(c, 1u + 100u * k, k);
            }
            expect(pinned_calls == 1 && pinned_total == 16384u, "pinned memory of tiny copies", pinned_calls, pinned_total);
            both_ways(c, 16385u, 4u);
            expect(pinned_calls == 1, "pinned allocations of small copies", pinned_calls, 1);
            both_ways(c, MiB + 1, 4u);
            expect(pinned_total < 2 * MiB, "staging of 1 MiB", pinned_total, 2 * MiB);
            both_ways(c, 70 * MiB + 1, 4u);
            expect(pinned_total <= 4 * MiB + 16384u, "staging", pinned_total, 4 * MiB);
        }
        else if (what == "device")
        {
            /* another device is current at the first large copy */
            current_device = 1;
            both_ways(c, 5 * MiB + 3, 6u);
            expect(staged_copies == 0, "staged copies", staged_copies, 0);
            current_device = 0;
            both_ways(c, 5 * MiB + 3, 7u);
            expect(staged_copies > 0, "staged copies", staged_copies, 1);
            expect(hipGetLastError() == hipSuccess, "error left", 0, 0);
        }
        else
            expect(false, "unknown case", 0, 0);
    }
    {
        std::lock_guard<std::mutex> l(mu);
        quit = true;
        cv.notify_all();
    }
    dev.join();
    expect(pinned_total == 0, "pinned memory left", pinned_total, 0);
    if (!failures)
        std::printf("ok\n");
    return failures != 0;
}
