// Large device-to-host copies: chunks into a ring of pinned buffers, copied on to the caller's memory by a
// few threads while the next chunks arrive. A copy straight into pageable memory moves 10 GB/s on an
// MI355X host (the runtime pins the pages as it goes), the link 57; one thread's copy into fresh memory is no
// faster than that (page faults), four together reach 50. Into fresh memory, straight and so: 9 MB 0.52 and
// 0.35 ms, 19 MB 1.08 and 0.54, 151 MB 14.2 and 3.6, 1.2 GB 113 and 26; eight or twelve threads are no faster, chunks of
// 1 MB 5.0 ms at 151 MB.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <utility>

#include "ctx.hpp"

namespace cfdx {
namespace {

constexpr size_t CHUNK = (size_t)4 << 20, SLOTS = 8;
constexpr size_t STAGED_FROM = 2 * CHUNK;   // smaller copies go straight
constexpr unsigned THREADS = 4;
constexpr size_t KEPT = 2;                  // rings of a device kept for its next copy (32 MB of pinned memory each)

struct Ring {
    char *mem = nullptr;
    hipEvent_t ev[SLOTS] = {};
    int device = 0;
    Ring *next = nullptr;   // in the list of those not in use

    ~Ring()
    {
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex rings_mutex;
Ring *rings = nullptr;   // not in use, at most KEPT of each device

// the next ring of the device among those not in use, from *at on
Ring **ring_of(int device, Ring **at)
{
    while (*at && (*at)->device != device) at = &(*at)->next;
    return at;
}

Ring *ring_take(int device)
{
    {
        std::lock_guard<std::mutex> lock(rings_mutex);
        Ring **at = ring_of(device, &rings);
        if (Ring *r = *at) {
            *at = r->next;
            return r;
        }
    }
    Ring *r = new (std::nothrow) Ring;
    if (!r) return nullptr;
    r->device = device;
    hipError_t e = hipHostMalloc((void **)&r->mem, CHUNK * SLOTS, hipHostMallocDefault);
    for (auto &v : r->ev)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    if (e == hipSuccess) return r;
    (void)hipGetLastError();
    delete r;
    return nullptr;
}

void ring_give(Ring *r)
{
    {
        std::lock_guard<std::mutex> lock(rings_mutex);
        size_t kept = 0;
        for (Ring **at = ring_of(r->device, &rings); *at; at = ring_of(r->device, &(*at)->next)) ++kept;
        if (kept < KEPT) {
            r->next = std::exchange(rings, r);
            return;
        }
    }
    delete r;
}

unsigned copy_threads()
{
    cpu_set_t set;
    const int n = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
    return std::min(THREADS, (unsigned)std::max(n, 1));
}

// Whether the runtime knows the memory (pinned, managed or device memory): a copy into it needs no staging (151 MB
// into pinned memory 2.78 ms, 57 GB/s; staged 3.55).
bool known_memory(const void *p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return false;
}

// One copy. The calling thread puts chunks on the stream as slots come free and watches them arrive (one
// thread asks the runtime; eight waiting on events took 100 us a chunk); the workers take arrived chunks in
// order and copy them out. All of them spin with yields: the copy alone is over in milliseconds.
struct Copy {
    Ring &ring;
    char *dst;
    size_t bytes, chunks;
    std::atomic<size_t> arrived{0}, next{0};
    std::atomic<bool> failed{false};
    std::atomic<size_t> out[SLOTS] = {};   // per slot: chunks copied out of it

    Copy(Ring &r, void *d, size_t n) : ring(r), dst((char *)d), bytes(n), chunks((n + CHUNK - 1) / CHUNK) {}

    void work()
    {
        for (;;) {
            const size_t c = next.fetch_add(1);
            if (c >= chunks) return;
            while (arrived.load(std::memory_order_acquire) <= c) {
                if (failed.load()) return;
                std::this_thread::yield();
            }
            const size_t off = c * CHUNK;
            std::memcpy(dst + off, ring.mem + (c % SLOTS) * CHUNK, std::min(CHUNK, bytes - off));
            out[c % SLOTS].store(c / SLOTS + 1, std::memory_order_release);
        }
    }

    hipError_t run(const char *src, hipStream_t st)
    {
        size_t issued = 0, here = 0;
        hipError_t e = hipSuccess;
        while (here < chunks && e == hipSuccess) {
            if (issued < chunks && out[issued % SLOTS].load(std::memory_order_acquire) == issued / SLOTS) {
                const size_t off = issued * CHUNK;
                e = hipMemcpyAsync(ring.mem + (issued % SLOTS) * CHUNK, src + off, std::min(CHUNK, bytes - off),
                                   hipMemcpyDeviceToHost, st);
                if (e == hipSuccess) e = hipEventRecord(ring.ev[issued % SLOTS], st);
                if (e == hipSuccess) ++issued;
            }
            if (e == hipSuccess && here < issued) {
                const hipError_t q = hipEventQuery(ring.ev[here % SLOTS]);
                if (q == hipSuccess) arrived.store(++here, std::memory_order_release);
                else if (q != hipErrorNotReady) e = q;
            }
            if (here < issued && issued == chunks) std::this_thread::yield();
        }
        if (e != hipSuccess) failed.store(true);
        return e;
    }
};

}  // namespace

void staging_trim(int device)
{
    Ring *gone = nullptr;
    {
        std::lock_guard<std::mutex> lock(rings_mutex);
        for (Ring **at = ring_of(device, &rings); *at; at = ring_of(device, at)) {
            Ring *r = *at;
            *at = r->next;
            r->next = std::exchange(gone, r);
        }
    }
    while (gone) delete std::exchange(gone, gone->next);
}

int copy_to_host(cfdx_ctx *ctx, void *dst, const void *src, size_t bytes, const char *what)
{
    const unsigned nt = bytes >= STAGED_FROM && !known_memory(dst) ? copy_threads() : 0;
    Ring *ring = nt > 1 ? ring_take(ctx->device) : nullptr;
    if (!ring) {   // small, into pinned memory, one CPU, or no pinned memory left for a ring: straight
        CFDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream), what);
        CFDX_HIP(hipStreamSynchronize(ctx->stream), what);
        return CFDX_OK;
    }
    // the work queued so far may take long: it is waited for asleep, before the threads start to spin
    const hipError_t ready = hipStreamSynchronize(ctx->stream);
    if (ready != hipSuccess) {
        ring_give(ring);
        return hip_fail(ready, what);
    }
    Copy c(*ring, dst, bytes);
    std::thread threads[THREADS];
    unsigned started = 0;
    try {
        for (; started < nt; ++started) threads[started] = std::thread([&c] { c.work(); });
    } catch (const std::exception &) {
        // fewer threads than asked for: those that started do the work
    }
    if (!started) {
        ring_give(ring);
        CFDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream), what);
        CFDX_HIP(hipStreamSynchronize(ctx->stream), what);
        return CFDX_OK;
    }
    const hipError_t e = c.run((const char *)src, ctx->stream);
    for (unsigned q = 0; q < started; ++q) threads[q].join();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(ctx->stream);   // no copy into the ring is left when it is given back
        ring_give(ring);
        return hip_fail(e, what);
    }
    ring_give(ring);
    return CFDX_OK;
}

}  // namespace cfdx
