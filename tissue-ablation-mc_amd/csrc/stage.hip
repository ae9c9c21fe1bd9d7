// stage.hip -- large fields to pageable host memory through a pinned ring.
//
// A copy to pageable memory runs at 10 GB/s: the runtime stages it in small
// pieces on one thread, which also takes the page faults of a new array (12
// GB/s by itself).  Here chunks go to a ring of pinned slots at the link's rate
// (56 GB/s) while a few threads move them on, converting on the way where the
// device keeps a narrower type.  To a new array, before and after:
// 64 MB 6.1 ms, 1.8; 134 MB 12.8, 3.5 (2.5 at the link's rate); 4 MB 0.7, 0.35.
// Fields that are too small for it are copied plainly (stage_route).
//
// Rings outlive a context: pinning 16 MiB takes 0.7 ms.  Idle rings are kept
// for any context (at most kIdleRings of them) and freed with the last context.
// A ring belongs to one download at a time, whatever the thread or stream.
#include "tam_internal.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include <sys/mman.h>

namespace {

constexpr int kSlots = 8;
constexpr size_t kSlotBytes = (size_t)2 << 20;         // also a huge page of the destination
constexpr int kIdleRings = 2;
// A thread per 2 MiB of the result: two for 4 MiB (0.24 ms, 0.44 on one and
// 0.28 on four), eight for 64 MiB and more (1.3 ms, 5.4 on one, 1.4 on four).
constexpr int kThreads = 8;

struct Ring {
    int dev = -1;
    char* pin = nullptr;
    hipEvent_t ev[kSlots] = {};
};

struct Pool {
    std::mutex mu;
    Ring* idle[kIdleRings] = {};
    long users = 0;
};
Pool& pool()
{
    static Pool* p = new Pool;                          // never destroyed: contexts may close at exit
    return *p;
}

// The calling thread in another capture mode for a scope: what HIP refuses while
// a stream is being captured goes by the mode of the thread that asks.
struct CaptureMode {
    hipStreamCaptureMode old;
    bool swapped;
    explicit CaptureMode(hipStreamCaptureMode mode)
        : old(mode), swapped(hipThreadExchangeStreamCaptureMode(&old) == hipSuccess)
    {
    }
    ~CaptureMode()
    {
        if (swapped) (void)hipThreadExchangeStreamCaptureMode(&old);
    }
    CaptureMode(const CaptureMode&) = delete;
};

void ring_free(Ring* r)
{
    if (!r) return;
    for (hipEvent_t e : r->ev)
        if (e) (void)hipEventDestroy(e);
    if (r->pin) (void)hipHostFree(r->pin);
    delete r;
}

// dev is the current device.  nullptr: none idle and none to be made, or no
// memory; the caller copies plainly.
Ring* ring_take(int dev, bool make)
{
    {
        std::lock_guard<std::mutex> l(pool().mu);
        for (Ring*& q : pool().idle)
            if (q && q->dev == dev) {
                Ring* r = q;
                q = nullptr;
                return r;
            }
    }
    Ring* r = make ? new (std::nothrow) Ring : nullptr;
    if (!r) return nullptr;
    r->dev = dev;
    hipError_t e;
    {
        // an allocation must not break a capture that another thread has under way
        const CaptureMode relaxed(hipStreamCaptureModeRelaxed);
        e = hipHostMalloc((void**)&r->pin, kSlots * kSlotBytes, hipHostMallocDefault);
        for (hipEvent_t& ev : r->ev)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        ring_free(r);
        return nullptr;
    }
    return r;
}

void ring_give(Ring* r)
{
    {
        std::lock_guard<std::mutex> l(pool().mu);
        if (pool().users > 0)
            for (Ring*& q : pool().idle)
                if (!q) {
                    q = r;
                    return;
                }
    }
    ring_free(r);
}

struct Job {
    Ring* ring;
    hipStream_t stream;
    const char* src;
    double* out;
    StageKind kind;
    double offset;
    long n, first, chunk, chunks;                      // elements; the first chunk ends at a huge page of `out`
    std::atomic<long> next{0};
    std::atomic<long> issued[kSlots];                  // the chunk last sent to a slot
    std::atomic<int> err{(int)hipSuccess};
};

size_t stage_size(StageKind k) { return k == STAGE_F64 ? 8 : k == STAGE_F32 ? 4 : 1; }

void span(const Job& j, long k, long& lo, long& hi)
{
    lo = k == 0 ? 0 : j.first + (k - 1) * j.chunk;
    hi = std::min(j.n, j.first + k * j.chunk);
}

void issue(Job& j, long k)
{
    long lo, hi;
    span(j, k, lo, hi);
    const int slot = (int)(k % kSlots);
    const size_t es = stage_size(j.kind);
    hipError_t e = hipMemcpyAsync(j.ring->pin + slot * kSlotBytes, j.src + lo * es, (size_t)(hi - lo) * es,
                                  hipMemcpyDeviceToHost, j.stream);
    if (e == hipSuccess) e = hipEventRecord(j.ring->ev[slot], j.stream);
    if (e != hipSuccess) j.err = (int)e;
    j.issued[slot].store(k, std::memory_order_release);
}

// Pages of a new array are made before the chunk arrives: one call instead of a
// fault per page.  A kernel that does not know the request leaves them to the
// copy.
void populate(char* lo, char* hi)
{
    constexpr uintptr_t kPage = 4096;
    constexpr int kPopulateWrite = 23;                  // MADV_POPULATE_WRITE, Linux 5.14
    const uintptr_t a = ((uintptr_t)lo + kPage - 1) & ~(kPage - 1), b = (uintptr_t)hi & ~(kPage - 1);
    if (b > a) (void)madvise((void*)a, b - a, kPopulateWrite);
}

// One of the job's threads: takes the next chunk, moves it on, sends the
// chunk that follows it in the slot.
void work(Job& j)
{
    for (long k = j.next++; k < j.chunks; k = j.next++) {
        const int slot = (int)(k % kSlots);
        long lo, hi;
        span(j, k, lo, hi);
        double* o = j.out + lo;
        populate((char*)o, (char*)(j.out + hi));
        // sent by the thread that moved chunk k - kSlots, which ends or sets err
        while (j.issued[slot].load(std::memory_order_acquire) != k) {
            if (j.err != (int)hipSuccess) return;
            std::this_thread::yield();
        }
        const hipError_t e = hipEventSynchronize(j.ring->ev[slot]);
        if (e != hipSuccess) j.err = (int)e;
        if (j.err != (int)hipSuccess) return;
        const char* in = j.ring->pin + slot * kSlotBytes;
        if (j.kind == STAGE_F64) std::memcpy(o, in, (size_t)(hi - lo) * 8);
        else if (j.kind == STAGE_F32)
            for (long i = 0; i < hi - lo; ++i) o[i] = j.offset + (double)((const float*)in)[i];
        else
            for (long i = 0; i < hi - lo; ++i) o[i] = ((const uint8_t*)in)[i];
        if (k + kSlots < j.chunks) issue(j, k + kSlots);
    }
}

}  // namespace

void stage_user(int delta)
{
    Ring* drop[kIdleRings] = {};
    {
        std::lock_guard<std::mutex> l(pool().mu);
        pool().users += delta;
        if (pool().users <= 0) std::swap_ranges(pool().idle, pool().idle + kIdleRings, drop);
    }
    for (Ring* r : drop) ring_free(r);
}

// A field by the size of its result, in us plain and through a ring (FP64; FP32 or
// bytes): 4 KiB 24, 14; 22-24, 14, so small ones take a ring that is idle, and
// make none.  32 KiB 12, 20; 256 KiB 22, 30-40; 22, 28; 500 KiB 32, 40-48; 31, 35-44;
// 1.4 MiB 87, 93-103; 70, 72.  2 MiB 122, 116; 130, 78, and all larger ones.
// (A plain copy of less than 16 KiB costs more than one of 32, and so does a
// narrower field's below 160 KiB of result: 24^3 41 us, 23.)
StageRoute stage_route(StageKind kind, long n)
{
    const size_t bytes = sizeof(double) * (size_t)n;
    if (bytes >= kSlotBytes) return STAGE_RING;
    return bytes < (size_t)(kind == STAGE_F64 ? 16 : 160) << 10 ? STAGE_IDLE : STAGE_PLAIN;
}

extern "C" int tam_internal_stage_route(int kind, int64_t n) { return (int)stage_route((StageKind)kind, (long)n); }

hipError_t stage_download(int dev, hipStream_t s, const void* src, StageKind kind, long n, double offset, double* out)
{
    if (n <= 0) return hipSuccess;
    const StageRoute route = stage_route(kind, n);
    Ring* r = route == STAGE_PLAIN ? nullptr : ring_take(dev, route == STAGE_RING);
    if (!r) return hipErrorOutOfMemory;
    Job j;
    j.ring = r;
    j.stream = s;
    j.src = (const char*)src;
    j.out = out;
    j.kind = kind;
    j.offset = offset;
    j.n = n;
    j.chunk = (long)(kSlotBytes / sizeof(double));
    j.first = std::min<long>(n, (long)((kSlotBytes - (uintptr_t)out % kSlotBytes) / sizeof(double)));
    if (j.first < 1) j.first = std::min<long>(n, j.chunk);
    j.chunks = 1 + (n - j.first + j.chunk - 1) / j.chunk;
    for (auto& q : j.issued) q = -1;
    for (long k = 0; k < std::min<long>(j.chunks, kSlots); ++k) issue(j, k);
    // the threads wait as the caller may: in its capture mode, not a new thread's
    const hipStreamCaptureMode mode = CaptureMode(hipStreamCaptureModeRelaxed).old;
    const long want = std::min<long>({(long)kThreads, j.chunks, (long)(n * sizeof(double) / kSlotBytes)});
    std::thread extra[kThreads];
    int started = 0;
    try {
        for (; started + 1 < want; ++started)
            extra[started] = std::thread([&j, dev, mode] {
                const CaptureMode own(mode);
                const hipError_t e = hipSetDevice(dev);
                if (e != hipSuccess) j.err = (int)e;
                work(j);
            });
    } catch (...) {                                     // no more threads: those there do the work
    }
    work(j);
    for (int t = 0; t < started; ++t) extra[t].join();
    // before the slots go to another download no copy to them may be on its way,
    // also where the caller's wait is refused (its capture mode) or a thread gave up
    const hipError_t done = hipStreamSynchronize(s);
    hipError_t settled = done;
    if (settled != hipSuccess) {
        const CaptureMode relaxed(hipStreamCaptureModeRelaxed);
        settled = hipStreamSynchronize(s);
    }
    const hipError_t e = (hipError_t)j.err.load();
    if (settled == hipSuccess) ring_give(r);            // else lost with its device
    return e != hipSuccess ? e : done;
}
