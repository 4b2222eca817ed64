/* The library's host sources (csrc/ctx.cpp, host_copy.cpp, common.cpp) on a HIP runtime of plain host memory that keeps
 * the books: what is allocated on which device, and the last error, which like the real one's stays until it is read.
 * No GPU, and no HIP library is linked. One check a run, named by the argument; "ok" if it holds. */
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "ctx.hpp"

namespace {
constexpr int DEVICES = 4;
std::mutex mu;
std::map<void *, size_t> device_mem, host_mem;
size_t device_free = (size_t)1 << 30;
size_t host_allocs = 0;                     // hipHostMalloc calls so far
size_t looks = 0;                           // hipMemGetInfo calls so far
bool taken = false;                         // another process takes what is freed: the free figure stays
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;

hipError_t done(hipError_t e)
{
    if (e != hipSuccess && e != hipErrorNotReady) last = e;
    return e;
}

#define CHECK(cond, ...)                        \
    do {                                        \
        if (!(cond)) {                          \
            std::printf("failed: " __VA_ARGS__); \
            std::printf(" (%s)\n", #cond);      \
            std::exit(1);                       \
        }                                       \
    } while (0)
}  // namespace

extern "C" {
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error"; }
hipError_t hipGetDeviceCount(int *n) { *n = DEVICES; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return done(d >= 0 && d < DEVICES ? hipSuccess : hipErrorInvalidDevice); }
hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lock(mu);
    if (n > device_free) return done(hipErrorOutOfMemory);
    *p = std::malloc(16);
    device_mem[*p] = n;
    device_free -= n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lock(mu);
    const auto it = device_mem.find(p);
    if (it == device_mem.end()) return done(hipErrorInvalidValue);
    device_free += it->second;
    device_mem.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    static size_t shown = 0;
    if (!taken) shown = device_free;
    *f = shown;
    ++looks;
    *t = (size_t)1 << 30;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> lock(mu);
    *p = std::malloc(n);
    host_mem[*p] = n;
    ++host_allocs;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::lock_guard<std::mutex> lock(mu);
    host_mem.erase(p);
    std::free(p);
    return hipSuccess;
}
// like the real one's older form: memory it does not know is an error
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    std::lock_guard<std::mutex> lock(mu);
    for (const auto &m : host_mem)
        if ((const char *)p >= (const char *)m.first && (const char *)p < (const char *)m.first + m.second) {
            a->type = hipMemoryTypeHost;
            return hipSuccess;
        }
    return done(hipErrorInvalidValue);
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free((void *)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void *)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
}

namespace {
cfdx_ctx *context(int device)
{
    cfdx_ctx *c = nullptr;
    CHECK(cfdx_ctx_create(device, nullptr, &c) == CFDX_OK, "context on device %d", device);
    return c;
}

// An allocation that does not fit is answered with a null pointer and leaves no error behind: the next launch check
// of the thread, on work that did fit, passes.
void pool()
{
    cfdx_ctx *c = context(0);
    size_t got = 0;
    CHECK(!cfdx::pool_take(0, (size_t)2 << 30, &got), "more than the device has");
    void *p = cfdx::pool_take(0, (size_t)256 << 20, &got);
    CHECK(p && got == (size_t)256 << 20, "what the device has");
    CHECK(cfdx::check_launch("the next launch") == CFDX_OK, "%s", cfdx_last_error());
    cfdx::pool_give(0, p, got);
    void *d = nullptr;
    CHECK(cfdx_device_alloc(c, (size_t)2 << 30, &d) == CFDX_E_NOMEM, "device_alloc past the memory");
    CHECK(cfdx::check_launch("the next launch") == CFDX_OK, "%s", cfdx_last_error());
    CHECK(cfdx_ctx_destroy(c) == CFDX_OK, "destroy");
}

// A trim whose memory is taken by others at once does not wait for the free figure to rise.
void trim()
{
    cfdx_ctx *c = context(0);
    size_t got = 0, f = 0, t = 0;
    void *p = cfdx::pool_take(0, (size_t)200 << 20, &got);
    cfdx::pool_give(0, p, got);
    (void)hipMemGetInfo(&f, &t);
    taken = true;
    const size_t before = looks;
    CHECK(cfdx_pool_trim(c) == CFDX_OK && cfdx::pool_cached(0) == 0, "trim");
    CHECK(looks - before <= 32, "%zu looks at the free figure, half a millisecond apart", looks - before);
    CHECK(cfdx_ctx_destroy(c) == CFDX_OK, "destroy");
}

// The bytes of a device-to-host copy.
void copy(cfdx_ctx *c, char *dst, const std::vector<char> &src)
{
    std::memset(dst, 0, src.size());
    CHECK(cfdx_copy_to_host(c, dst, src.data(), src.size()) == CFDX_OK, "copy: %s", cfdx_last_error());
    CHECK(std::memcmp(dst, src.data(), src.size()) == 0, "the bytes of a copy");
}

std::vector<char> bytes(size_t n)
{
    std::vector<char> b(n);
    for (size_t q = 0; q < n; ++q) b[q] = (char)(q * 31 + (q >> 12));
    return b;
}

// Large copies into pageable memory go through a pinned ring; into memory that is pinned already, also from the middle
// of it on, they go straight. Neither leaves an error behind.
void pinned()
{
    cfdx_ctx *c = context(0);
    const std::vector<char> src = bytes((size_t)20 << 20);
    void *p = nullptr;
    (void)hipHostMalloc(&p, src.size() + 4096, 0);
    const size_t own = host_allocs;
    copy(c, (char *)p, src);
    copy(c, (char *)p + 4096, src);
    CHECK(host_allocs == own, "a ring was made for a copy into pinned memory");
    std::vector<char> plain(src.size());
    copy(c, plain.data(), src);
    CHECK(host_allocs == own + 1, "%zu rings for a copy into pageable memory", host_allocs - own);
    CHECK(cfdx::check_launch("the next launch") == CFDX_OK, "%s", cfdx_last_error());
    (void)hipHostFree(p);
    CHECK(cfdx_ctx_destroy(c) == CFDX_OK, "destroy");
}

// Every device of a process keeps its rings: copies that go round the devices make one each, once. A trim gives those
// of its device back and no others.
void rings()
{
    cfdx_ctx *c[DEVICES];
    for (int d = 0; d < DEVICES; ++d) c[d] = context(d);
    const std::vector<char> src = bytes((size_t)9 << 20);
    std::vector<char> dst(src.size());
    for (int round = 0; round < 3; ++round)
        for (cfdx_ctx *x : c) copy(x, dst.data(), src);
    CHECK(host_allocs == DEVICES, "%zu rings for %d devices", host_allocs, DEVICES);
    CHECK(cfdx_pool_trim(c[1]) == CFDX_OK, "trim");
    CHECK(host_mem.size() == DEVICES - 1, "%zu rings after a trim of one device", host_mem.size());
    for (cfdx_ctx *x : c) copy(x, dst.data(), src);
    CHECK(host_allocs == DEVICES + 1, "%zu rings made", host_allocs);
    for (cfdx_ctx *x : c) CHECK(cfdx_pool_trim(x) == CFDX_OK, "trim");
    CHECK(host_mem.empty(), "%zu rings after every trim", host_mem.size());
    // at most two of a device are kept, however many copies ran at once
    std::vector<std::thread> t;
    for (int q = 0; q < 6; ++q)
        t.emplace_back([&src] {
            cfdx_ctx *x = context(2);
            std::vector<char> own(src.size());
            for (int k = 0; k < 4; ++k) copy(x, own.data(), src);
            CHECK(cfdx_ctx_destroy(x) == CFDX_OK, "destroy");
        });
    for (auto &x : t) x.join();
    CHECK(host_mem.size() <= 2, "%zu rings kept", host_mem.size());
    for (cfdx_ctx *x : c) CHECK(cfdx_ctx_destroy(x) == CFDX_OK, "destroy");
}
}  // namespace

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "pool")) pool();
    else if (!std::strcmp(what, "trim")) trim();
    else if (!std::strcmp(what, "pinned")) pinned();
    else if (!std::strcmp(what, "rings")) rings();
    else CHECK(false, "no check named '%s'", what);
    std::puts("ok");
}
