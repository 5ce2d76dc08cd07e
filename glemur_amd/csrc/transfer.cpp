// Copies between a caller's pageable arrays and device memory, staged
// through pinned slots that several threads fill or empty while the copy
// engine moves the others.
//
// Bound by the link (57 GB/s in one large copy, about 10 us between copies).
// A plain hipMemcpy of pageable memory stages through one thread, at 25 GB/s
// up and 10 GB/s down, where fresh pages are faulted in meanwhile; one core
// copies 24 GB/s.  Measured, plain -> staged: 158 MB up 6.4 -> 3.9 ms, down
// into fresh memory 16 -> 4.0 ms; 1.2 GB up 44 -> 27 ms, down 119 -> 27 ms.
// Eight slots of 4 MB: slots of 2 MB reach 38 GB/s instead of 43, twelve
// slots or eight threads no more.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace gm {
namespace {

constexpr int kSlots = 8, kThreads = 6;
constexpr size_t kSlotBytes = 4 << 20, kMinChunk = 256 << 10;
// Below these the threads cost more than they save (plain -> staged): up
// 9 MB 0.28 -> 0.44 ms, 21 MB 0.65 -> 0.72 ms, 158 MB 6.4 -> 3.9 ms; down
// 9 MB 0.97 -> 0.70 ms, 21 MB 2.3 -> 0.85 ms.  Beside a program whose own
// threads spin (a torch program's after each host operation) a short copy
// waits for its threads to be scheduled: 11 MB down 0.7 ms plain, 2.5 ms
// staged, hence no less than 16 MB.
constexpr size_t kMinUp = 32 << 20, kMinDown = 16 << 20;

struct Staging {
    std::mutex m;             // held by the copy that uses the slots
    int users = 0;
    char *buf = nullptr;
    int device = -1;
    hipEvent_t ev[kSlots] = {};

    // Events are recorded on streams of their own device only: a caller whose
    // current device is another one than the stream's goes the plain way
    bool ready(hipStream_t s)
    {
        int d = 0;
        hipDevice_t sd = 0;
        if (hipGetDevice(&d) != hipSuccess || hipStreamGetDevice(s, &sd) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        if (sd != d) return false;
        if (!buf && hipHostMalloc((void **)&buf, kSlots * kSlotBytes, hipHostMallocPortable) != hipSuccess) {
            (void)hipGetLastError();
            buf = nullptr;
            return false;
        }
        if (d != device) {
            drop_events();
            for (auto &e : ev)
                if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    e = nullptr;
                    drop_events();
                    return false;
                }
            device = d;
        }
        return true;
    }
    void drop_events()
    {
        for (auto &e : ev) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        device = -1;
    }
};
Staging &staging()
{
    static Staging *s = new Staging;   // outlives static destructors
    return *s;
}

// Only pageable memory is staged: pinned memory copies faster as it is, and
// memory that is not the host's must not be touched from here
bool pageable(const void *p)
{
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return at.type == hipMemoryTypeUnregistered;
}

inline void relax(int &spins)
{
    if (++spins < 200) __builtin_ia32_pause();
    else std::this_thread::yield();
}

// The chunks of one copy.  Threads claim them in turn; chunk i may be worked
// on once avail > i, and done[i] says that it was.
struct Chunks {
    size_t bytes, chunk;
    long n;
    std::atomic<long> next{0}, avail{0};
    std::atomic<bool> stop{false};
    std::unique_ptr<std::atomic<bool>[]> done;
    char *slots, *host;
    bool up;
    std::vector<std::thread> threads;

    Chunks(char *slots_, char *host_, size_t bytes_, bool up_) : bytes(bytes_), slots(slots_), host(host_), up(up_)
    {
        chunk = std::min(kSlotBytes, std::max(kMinChunk, (bytes / kSlots + 4095) / 4096 * 4096));
        n = (long)((bytes + chunk - 1) / chunk);
        done.reset(new std::atomic<bool>[n]);
        for (long i = 0; i < n; ++i) done[i] = false;
        const long want = std::min<long>({kThreads, n, std::max(1, (int)std::thread::hardware_concurrency() - 1)});
        try {
            threads.reserve(want);
            for (long t = 0; t < want; ++t) threads.emplace_back([this] { work(); });
        } catch (...) {   // the threads there are do (the calling one, if none)
        }
    }
    ~Chunks()
    {
        stop = true;
        for (auto &t : threads) t.join();
    }
    size_t size(long i) const { return std::min(chunk, bytes - (size_t)i * chunk); }
    char *slot(long i) const { return slots + (i % kSlots) * kSlotBytes; }
    void move(long i)
    {
        char *h = host + (size_t)i * chunk;
        if (up) memcpy(slot(i), h, size(i));
        else memcpy(h, slot(i), size(i));
        done[i].store(true, std::memory_order_release);
    }
    void work()
    {
        for (;;) {
            const long i = next.fetch_add(1);
            if (i >= n) return;
            for (int spins = 0; avail.load(std::memory_order_acquire) <= i; relax(spins))
                if (stop) return;
            move(i);
        }
    }
    void wait(long i)
    {
        if (threads.empty()) {
            if (!done[i]) move(i);
            return;
        }
        for (int spins = 0; !done[i].load(std::memory_order_acquire);) relax(spins);
    }
};

hipError_t up(hipStream_t s, char *dst, Chunks &c, hipEvent_t *ev)
{
    hipError_t e = hipSuccess;
    c.avail = kSlots;
    for (long i = 0; i < c.n && e == hipSuccess; ++i) {
        c.wait(i);
        e = hipMemcpyAsync(dst + (size_t)i * c.chunk, c.slot(i), c.size(i), hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipEventRecord(ev[i % kSlots], s);
        const long f = i - kSlots / 2;   // half of the slots in flight, half being filled
        if (e == hipSuccess && f >= 0) {
            e = hipEventSynchronize(ev[f % kSlots]);
            c.avail.store(f + 1 + kSlots, std::memory_order_release);
        }
    }
    const hipError_t w = hipStreamSynchronize(s);   // the slots are free again
    return e == hipSuccess ? w : e;
}

hipError_t down(hipStream_t s, const char *src, Chunks &c, hipEvent_t *ev)
{
    hipError_t e = hipSuccess;
    long issued = 0;
    for (long i = 0; i < c.n && e == hipSuccess; ++i) {
        while (e == hipSuccess && issued < c.n && issued < i + kSlots) {
            if (issued >= kSlots) {
                if (issued > i && !c.done[issued - kSlots].load(std::memory_order_acquire)) break;
                c.wait(issued - kSlots);
            }
            e = hipMemcpyAsync(c.slot(issued), src + (size_t)issued * c.chunk, c.size(issued), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(ev[issued % kSlots], s);
            ++issued;
        }
        if (e == hipSuccess) e = hipEventSynchronize(ev[i % kSlots]);
        if (e != hipSuccess) break;
        c.avail.store(i + 1, std::memory_order_release);
        if (c.threads.empty()) c.move(i);
    }
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(s);
        return e;
    }
    for (long i = std::max(0L, c.n - kSlots); i < c.n; ++i) c.wait(i);
    return hipSuccess;
}

}  // namespace

void staging_retain()
{
    Staging &g = staging();
    std::lock_guard<std::mutex> l(g.m);
    ++g.users;
}

void staging_release()
{
    Staging &g = staging();
    std::lock_guard<std::mutex> l(g.m);
    if (--g.users > 0) return;
    if (g.buf) (void)hipHostFree(g.buf);
    g.buf = nullptr;
    g.drop_events();
}

// A copy that finds the slots taken by another thread's goes the plain way.
hipError_t copy_to_device(hipStream_t s, void *dst, const void *src, size_t bytes)
{
    if (bytes >= kMinUp && pageable(src)) {
        Staging &g = staging();
        std::unique_lock<std::mutex> l(g.m, std::try_to_lock);
        if (l.owns_lock() && g.ready(s)) {
            try {
                Chunks c(g.buf, (char *)src, bytes, true);
                return up(s, (char *)dst, c, g.ev);
            } catch (...) {   // no memory for the bookkeeping
            }
        }
    }
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
}

hipError_t copy_to_host(hipStream_t s, void *dst, const void *src, size_t bytes)
{
    if (bytes >= kMinDown && pageable(dst)) {
        Staging &g = staging();
        std::unique_lock<std::mutex> l(g.m, std::try_to_lock);
        if (l.owns_lock() && g.ready(s)) {
            try {
                Chunks c(g.buf, (char *)dst, bytes, false);
                return down(s, (const char *)src, c, g.ev);
            } catch (...) {
            }
        }
    }
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace gm
