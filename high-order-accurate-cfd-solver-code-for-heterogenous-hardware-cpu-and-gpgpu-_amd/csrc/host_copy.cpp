// Large device-to-host copies: chunks into a ring of pinned buffers, copied on to the caller's memory by a
// few threads while the next chunks arrive. A copy straight into pageable memory moves 10 GB/s on an
// MI355X host (the runtime pins the pages as it goes; 4 GB/s into fresh 4 kB pages), the link 57;
// one thread's copy into fresh memory is no faster than that (5-12 GB/s, page faults), eight reach 50.
// 151 MB into fresh memory: 15.2 ms straight, 3.7 ms so.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "ctx.hpp"

namespace cfdx {
namespace {

constexpr size_t CHUNK = (size_t)4 << 20, SLOTS = 8;
constexpr size_t STAGED_FROM = 2 * CHUNK;   // smaller copies go straight
constexpr unsigned THREADS = 8;
constexpr size_t KEPT = 2;                  // rings kept for the next copy (32 MB of pinned memory each)

struct Ring {
    char *mem = nullptr;
    hipEvent_t ev[SLOTS] = {};
    int device = 0;

    ~Ring()
    {
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        if (mem) (void)hipHostFree(mem);
    }
};

std::mutex rings_mutex;
std::vector<Ring *> rings;   // not in use

Ring *ring_take(int device)
{
    {
        std::lock_guard<std::mutex> lock(rings_mutex);
        for (size_t q = 0; q < rings.size(); ++q)
            if (rings[q]->device == device) {
                Ring *r = rings[q];
                rings.erase(rings.begin() + (long)q);
                return r;
            }
    }
    Ring *r = new Ring;
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
        if (rings.size() < KEPT) {
            rings.push_back(r);
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

// One copy: `issued` chunks are on the stream, workers take them in order and mark them `done`.
struct Copy {
    Ring &ring;
    char *dst;
    size_t bytes, chunks;
    std::mutex m;
    std::condition_variable cv;
    size_t issued = 0, next = 0, done = 0;   // done: chunks copied out
    std::vector<char> out;                   // per chunk: copied out
    hipError_t err = hipSuccess;

    Copy(Ring &r, void *d, size_t n) : ring(r), dst((char *)d), bytes(n), chunks((n + CHUNK - 1) / CHUNK), out(chunks, 0) {}

    void work()
    {
        (void)hipSetDevice(ring.device);
        for (;;) {
            size_t c;
            {
                std::unique_lock<std::mutex> lock(m);
                cv.wait(lock, [&] { return err != hipSuccess || next >= chunks || next < issued; });
                if (err != hipSuccess || next >= chunks) return;
                c = next++;
            }
            const hipError_t e = hipEventSynchronize(ring.ev[c % SLOTS]);
            const size_t off = c * CHUNK;
            if (e == hipSuccess) std::memcpy(dst + off, ring.mem + (c % SLOTS) * CHUNK, std::min(CHUNK, bytes - off));
            std::lock_guard<std::mutex> lock(m);
            if (e != hipSuccess) err = e;
            out[c] = 1;
            ++done;
            cv.notify_all();
        }
    }

    // puts every chunk on the stream, each once its slot is free
    void issue(const char *src, hipStream_t st)
    {
        for (size_t c = 0; c < chunks; ++c) {
            {
                std::unique_lock<std::mutex> lock(m);
                cv.wait(lock, [&] { return err != hipSuccess || c < SLOTS || out[c - SLOTS]; });
                if (err != hipSuccess) return;
            }
            const size_t off = c * CHUNK;
            hipError_t e = hipMemcpyAsync(ring.mem + (c % SLOTS) * CHUNK, src + off, std::min(CHUNK, bytes - off),
                                          hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ring.ev[c % SLOTS], st);
            std::lock_guard<std::mutex> lock(m);
            if (e != hipSuccess) err = e;
            else issued = c + 1;
            cv.notify_all();
            if (e != hipSuccess) return;
        }
    }
};

}  // namespace

void staging_trim()
{
    std::vector<Ring *> gone;
    {
        std::lock_guard<std::mutex> lock(rings_mutex);
        gone.swap(rings);
    }
    for (Ring *r : gone) delete r;
}

int copy_to_host(cfdx_ctx *ctx, void *dst, const void *src, size_t bytes, const char *what)
{
    const unsigned nt = bytes >= STAGED_FROM ? copy_threads() : 0;
    Ring *ring = nt > 1 ? ring_take(ctx->device) : nullptr;
    if (!ring) {   // small, one CPU, or no pinned memory: straight
        CFDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream), what);
        CFDX_HIP(hipStreamSynchronize(ctx->stream), what);
        return CFDX_OK;
    }
    Copy c(*ring, dst, bytes);
    std::vector<std::thread> threads;
    try {
        threads.reserve(nt);
        for (unsigned q = 0; q < nt; ++q) threads.emplace_back([&c] { c.work(); });
    } catch (const std::exception &) {
        // fewer threads than asked for: those that started do the work
    }
    if (threads.empty()) {
        ring_give(ring);
        CFDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream), what);
        CFDX_HIP(hipStreamSynchronize(ctx->stream), what);
        return CFDX_OK;
    }
    c.issue((const char *)src, ctx->stream);
    for (auto &t : threads) t.join();
    if (c.err != hipSuccess) {
        (void)hipStreamSynchronize(ctx->stream);   // no copy into the ring is left when it is given back
        ring_give(ring);
        return hip_fail(c.err, what);
    }
    ring_give(ring);
    return CFDX_OK;
}

}  // namespace cfdx
