/*
 * cf_copy.hip -- device-to-host copies of whole fields into pageable memory.
 *
 * What bounds such a copy is the host: the pages of a fresh destination are
 * faulted in and zeroed by the one thread that stores to them, and the stream's
 * own copy of pageable memory waits for every chunk (101 MB into fresh memory
 * 9.5 to 24.5 ms, with the state of the host's memory; into memory in use 5.9;
 * the bus needs 1.8).  Here several threads each keep two chunks of a pinned
 * ring in flight and copy them out: 3.5 to 5.8 ms with 8 threads (where those
 * took 5.8: 6.7 with 6, 8.3 with 4, 11.9 with 2).  The caller's next passes
 * over the field take as long as after a plain copy (first read 3.7 and 3.6 ms,
 * write 2.6 and 2.6).
 *
 * The threads take fresh pages from the free lists of their own CPUs.  Where a
 * page has no memory behind it yet -- in a virtual machine, one that was never
 * used or that was free long enough to be reported to the host -- its first
 * touch costs a fault on the host, and a thread of its own meets more of those
 * than the caller, which gets back what it has just freed.  So a process that
 * begins to download by threads can pay for some copies (101 MB, each freed
 * before the next: 4, 22, ten of 15, then 3.3 ms each; plain copies beside them
 * 9.5 throughout), and other memory that it takes then as well: 18 batched
 * runs, whose fields are 2 to 17 MB, took 115 ms in place of 137 with threads
 * from 1 MB on, but a server's pass after them 302 in place of 267 (in other
 * runs 101 to 117, and no difference after).  Hence from 32 MB on, where a
 * field is not one of many.
 */
#include "chanflow.h"
#include "cf_internal_host.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#define CP_CHUNK ((size_t) 1 << 20)
#define CP_THREADS 8
#define CP_MIN ((size_t) 32 << 20)            /* below: a plain copy */
#define CP_IDLE 2                             /* rings kept for the next copies */

namespace {

/* pinned chunks and their events, two a thread */
struct Ring {
    int device = -1;
    char *buf = nullptr;
    hipEvent_t ev[2 * CP_THREADS] = {};
};

std::mutex g_lock;
Ring *g_idle[CP_IDLE] = {};
int g_users = 0;                              /* live runs; with the last one the idle rings go */

void ring_free(Ring *g)
{
    if (!g) return;
    for (hipEvent_t e : g->ev) if (e) (void) hipEventDestroy(e);
    if (g->buf) (void) hipHostFree(g->buf);
    delete g;
}

/* a ring of this device (the current one), or null */
Ring *ring_take(int device)
{
    {
        std::lock_guard<std::mutex> hold(g_lock);
        for (Ring *&g : g_idle)
            if (g && g->device == device) {
                Ring *t = g;
                g = nullptr;
                return t;
            }
    }
    Ring *g = new (std::nothrow) Ring();
    if (!g) return nullptr;
    g->device = device;
    bool ok = hipHostMalloc((void **) &g->buf, 2 * CP_THREADS * CP_CHUNK, hipHostMallocDefault) == hipSuccess;
    if (!ok) g->buf = nullptr;
    for (hipEvent_t &e : g->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) return g;
    (void) hipGetLastError();
    ring_free(g);
    return nullptr;
}

void ring_give(Ring *g)
{
    {
        std::lock_guard<std::mutex> hold(g_lock);
        if (g_users > 0) {
            for (Ring *&i : g_idle)
                if (!i) { i = g; return; }
            /* two rings of one device do not keep another's from staying */
            static_assert(CP_IDLE == 2, "compares the two kept rings");
            if (g_idle[0]->device == g_idle[1]->device && g->device != g_idle[0]->device) std::swap(g, g_idle[1]);
        }
    }
    ring_free(g);
}

} // namespace

extern "C" int cf_copy_users(int add)
{
    Ring *drop[CP_IDLE] = {};
    int users;
    {
        std::lock_guard<std::mutex> hold(g_lock);
        users = g_users += add;
        if (users == 0) std::swap(drop, g_idle);
    }
    for (Ring *g : drop) ring_free(g);
    return users;
}

extern "C" cf_status cf_copy_to_host(void *host, const void *dev, size_t bytes, int device, void *stream)
{
    const hipStream_t s = (hipStream_t) stream;
    Ring *g = nullptr;
    if (bytes >= CP_MIN) {
        /* a destination that the runtime knows (pinned, device) is copied to
         * directly */
        hipPointerAttribute_t at;
        const hipError_t e = hipPointerGetAttributes(&at, host);
        if (e != hipSuccess) (void) hipGetLastError();
        if (e != hipSuccess || at.type == hipMemoryTypeUnregistered) g = ring_take(device);
    }
    if (!g) {
        hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) return CF_OK;
        cf_set_error("copy to the host: %s", hipGetErrorString(e));
        return CF_ERR_DEVICE;
    }
    /* what the stream still has to do is waited for once, not by every thread */
    hipError_t first = hipStreamSynchronize(s);
    const size_t n = (bytes + CP_CHUNK - 1) / CP_CHUNK;
    std::atomic<size_t> next{ 0 };
    std::atomic<int> err{ (int) first };
    auto work = [&](int w) {
        char *slot[2] = { g->buf + 2 * w * CP_CHUNK, g->buf + (2 * w + 1) * CP_CHUNK };
        auto len = [&](size_t c) { return std::min(CP_CHUNK, bytes - c * CP_CHUNK); };
        auto issue = [&](size_t c, int q) {
            hipError_t e = hipMemcpyAsync(slot[q], (const char *) dev + c * CP_CHUNK, len(c), hipMemcpyDeviceToHost, s);
            if (e == hipSuccess) e = hipEventRecord(g->ev[2 * w + q], s);
            if (e != hipSuccess) err = (int) e;
        };
        if (w > 0) (void) hipSetDevice(device);
        size_t c = next++;
        if (c < n && !err) issue(c, 0);
        for (int q = 0; c < n && !err; q ^= 1) {
            const size_t c1 = next++;
            if (c1 < n) issue(c1, q ^ 1);
            const hipError_t e = hipEventSynchronize(g->ev[2 * w + q]);
            if (e != hipSuccess) { err = (int) e; break; }
            memcpy((char *) host + c * CP_CHUNK, slot[q], len(c));
            c = c1;
        }
    };
    /* a thread that does not start leaves its chunks to the others */
    std::thread th[CP_THREADS];
    for (int w = 1; w < CP_THREADS; w++) {
        try { th[w] = std::thread(work, w); } catch (...) { break; }
    }
    work(0);
    for (std::thread &t : th) if (t.joinable()) t.join();
    if (err) {
        /* copies of other threads may still be on their way into the ring */
        (void) hipStreamSynchronize(s);
        ring_free(g);
        cf_set_error("copy to the host: %s", hipGetErrorString((hipError_t) err.load()));
        return CF_ERR_DEVICE;
    }
    ring_give(g);
    return CF_OK;
}
