/*
 * pic_readback.hip -- results from the GPU into the caller's ordinary host
 * memory (fields, cell counts, particles, per-cell diagnostics).
 *
 * A copy into pageable memory runs through the runtime's own staging buffer
 * with one host thread, and a result array that was just allocated takes a
 * page fault per page on the way: 3 to 10 GB/s, where the link carries 54.
 * Here the copies land in a ring of pinned chunks and a few threads move the
 * chunks on (converting where the device holds floats or fixed point, so
 * those cross the link at their own width).  Each thread faults in the pages
 * of its chunk first, while the chunk is on its way and the kernels before it
 * run.  Six fields into fresh arrays: 22.6 to 6.5 ms at 256x128x128 cells FP32,
 * 3.2-7.0 to 2.8 at 256x64x64 FP64; twelve per-cell moments (201 MB) at
 * 256x64x64, kernels included, 24 to 11 ms.  6 threads with 1 MB chunks, and
 * 12, were within the noise of 8 with 2 MB; half a megabyte 15% slower.
 *
 * Memory the runtime knows (pinned by the caller, or a device's) is copied to
 * directly.
 */
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "pic_ctx.h"

namespace picx {

namespace {

constexpr size_t CHUNK = 2 << 20;   /* source bytes: one huge page of doubles */
constexpr int RING = 8;
constexpr int WORKERS = 8;

inline void relax() { __builtin_ia32_pause(); }

void move_chunk(char *dst, const char *src, long first, long n, ReadAs as) {
    switch (as) {
    case ReadAs::f64: std::memcpy(dst + first * 8, src, n * 8); break;
    case ReadAs::i32: std::memcpy(dst + first * 4, src, n * 4); break;
    case ReadAs::f32_to_f64: {
        double *d = (double *)dst + first;
        const float *s = (const float *)src;
        for (long k = 0; k < n; k++) d[k] = (double)s[k];
        break;
    }
    case ReadAs::fixed_to_f64: {
        double *d = (double *)dst + first;
        const long long *s = (const long long *)src;
        for (long k = 0; k < n; k++) d[k] = (double)s[k] * PIC_J_INV;
        break;
    }
    }
}

/* memory the runtime can copy to at once */
bool known_to_runtime(const void *p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type != hipMemoryTypeUnregistered;
}

}  // namespace

namespace {

/* The ring a call works with: the spare one, or a new one where another
 * thread's call has it.  One at most is kept between calls, while any context
 * lives (making one takes 1.5 ms: a program that opens a context per run would
 * pay that each time). */
struct Ring {
    char *buf = nullptr;
    int chunks = 0, dev = 0;
    hipEvent_t ev[RING] = {};
};
std::mutex ring_lock;
Ring *ring_spare = nullptr;
long contexts = 0;

void free_ring(Ring *r) {
    if (!r) return;
    if (r->buf) (void)hipHostFree(r->buf);
    for (hipEvent_t e : r->ev)
        if (e) (void)hipEventDestroy(e);
    delete r;
}

/* a ring on device dev of one chunk (want 1) or RING of them */
hipError_t take_ring(int dev, long want, Ring *&out) {
    Ring *r;
    {
        std::lock_guard<std::mutex> hold(ring_lock);
        r = ring_spare;
        ring_spare = nullptr;
    }
    if (r && r->dev == dev && (want == 1 || r->chunks == RING)) {
        out = r;
        return hipSuccess;
    }
    free_ring(r);
    r = new (std::nothrow) Ring;
    if (!r) return hipErrorOutOfMemory;
    r->dev = dev;
    r->chunks = want == 1 ? 1 : RING;
    hipError_t e = hipHostMalloc((void **)&r->buf, r->chunks * CHUNK);
    for (int k = 0; k < r->chunks && e == hipSuccess; k++)
        e = hipEventCreateWithFlags(&r->ev[k], hipEventDisableTiming);
    if (e != hipSuccess) {
        free_ring(r);
        return e;
    }
    out = r;
    return hipSuccess;
}

void give_ring(Ring *r) {
    {
        std::lock_guard<std::mutex> hold(ring_lock);
        if (!ring_spare && contexts > 0) {
            ring_spare = r;
            return;
        }
    }
    free_ring(r);
}

/* the context's device for the time of a call, which may come from a thread
 * whose current device is another: events and pinned memory belong to the
 * device current when they are made */
struct OnDevice {
    int before = -1;
    hipError_t enter(int dev) {
        const hipError_t e = hipGetDevice(&before);
        return e == hipSuccess ? hipSetDevice(dev) : e;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
};

struct Lease {
    Ring *ring = nullptr;
    ~Lease() {
        if (ring) give_ring(ring);
    }
};

}  // namespace

void readback_attach() {
    std::lock_guard<std::mutex> hold(ring_lock);
    contexts++;
}

void readback_detach() {
    Ring *r = nullptr;
    {
        std::lock_guard<std::mutex> hold(ring_lock);
        if (--contexts > 0) return;
        r = ring_spare;
        ring_spare = nullptr;
    }
    free_ring(r);
}

int readback(pic_ctx *c, void *dst_, const void *src_, long n, ReadAs as) {
    if (n <= 0) return PIC_SUCCESS;
    OnDevice here;
    HIPCHK(here.enter(c->dev));
    char *const dst = (char *)dst_;
    const char *const src = (const char *)src_;
    const size_t width = as == ReadAs::f32_to_f64 || as == ReadAs::i32 ? 4 : 8;
    const size_t bytes = n * width;
    const long nch = (long)((bytes + CHUNK - 1) / CHUNK), per = (long)(CHUNK / width);
    const bool as_is = as == ReadAs::f64 || as == ReadAs::i32;
    /* a small array as it is: the runtime's copy, 14 us where the ring takes 20 */
    if (as_is && (nch == 1 || known_to_runtime(dst))) {
        HIPCHK(hipStreamSynchronize(c->stream));
        HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
        return PIC_SUCCESS;
    }
    Lease lease;
    HIPCHK(take_ring(c->dev, nch, lease.ring));
    Ring *const r = lease.ring;
    if (nch == 1) {
        HIPCHK(hipMemcpyAsync(r->buf, src, bytes, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        move_chunk(dst, r->buf, 0, n, as);
        return PIC_SUCCESS;
    }
    const int S = r->chunks;
    auto chunk = [&](long i) { return r->buf + (i % S) * CHUNK; };
    auto size = [&](long i) { return std::min(bytes - i * CHUNK, CHUNK); };
    auto move = [&](long i) {
        move_chunk(dst, chunk(i), i * per, (long)(size(i) / width), as);
    };
    /* the pages of a chunk's destination, faulted in while the chunk is on its
     * way (and the kernels before it run), by a write that changes nothing (0
     * for 0; the instruction takes the page for writing either way): a copy
     * that fails leaves the array as it was */
    const size_t out_width = as == ReadAs::i32 ? 4 : 8;
    auto touch = [&](long i) {
        char *const p = dst + i * per * out_width;
        const size_t len = size(i) / width * out_width;
        auto take = [](char *at) {
            char was = 0;
            __atomic_compare_exchange_n(at, &was, (char)0, false, __ATOMIC_RELAXED,
                                        __ATOMIC_RELAXED);
        };
        for (size_t k = 0; k < len; k += 4096) take(p + k);
        take(p + len - 1);
    };
    auto issue = [&](long i) -> hipError_t {
        hipError_t e = hipMemcpyAsync(chunk(i), src + i * CHUNK, size(i), hipMemcpyDeviceToHost,
                                      c->stream);
        return e == hipSuccess ? hipEventRecord(r->ev[i % S], c->stream) : e;
    };
    std::atomic<long> next{0}, ready{0}, moved[RING];
    for (auto &m : moved) m.store(0, std::memory_order_relaxed);
    std::atomic<bool> stop{false};
    /* a worker whose chunk is not there within a millisecond or so (a long
     * kernel runs before it) sleeps until the next one arrives */
    constexpr int SPINS = 1 << 15;
    std::mutex arrival;
    std::condition_variable arrives;
    auto publish = [&](auto change) {
        {
            std::lock_guard<std::mutex> hold(arrival);
            change();
        }
        arrives.notify_all();
    };
    auto work = [&]() {
        for (;;) {
            const long i = next.fetch_add(1, std::memory_order_relaxed);
            if (i >= nch) return;
            touch(i);
            auto there = [&] { return ready.load(std::memory_order_acquire) > i || stop.load(); };
            for (int spins = 0; spins < SPINS && !there(); spins++) relax();
            if (!there()) {
                std::unique_lock<std::mutex> hold(arrival);
                arrives.wait(hold, there);
            }
            if (ready.load(std::memory_order_acquire) <= i) return;   /* stopped */
            move(i);
            moved[i % S].store(i + 1, std::memory_order_release);
        }
    };
    /* one thread a chunk at most; where none can be had the caller moves them */
    std::thread pool[WORKERS];
    int nw = 0;
    try {
        while (nw < WORKERS && nw < nch) {
            pool[nw] = std::thread(work);
            nw++;
        }
    } catch (...) {
    }
    hipError_t e = hipSuccess;
    long issued = 0, arrived = 0, freed = 0;
    while (arrived < nch && e == hipSuccess) {
        while (freed < arrived && moved[freed % S].load(std::memory_order_acquire) == freed + 1)
            freed++;
        if (issued < nch && issued < freed + S) {
            e = issue(issued);
            if (e == hipSuccess) issued++;
        } else if (arrived < issued) {
            e = hipEventSynchronize(r->ev[arrived % S]);
            if (e != hipSuccess) break;
            if (nw == 0) {
                move(arrived);
                moved[arrived % S].store(arrived + 1, std::memory_order_relaxed);
            }
            publish([&] { ready.store(++arrived, std::memory_order_release); });
        } else {
            relax();
        }
    }
    if (e != hipSuccess) publish([&] { stop.store(true); });
    for (int k = 0; k < nw; k++) pool[k].join();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);
        return record_hip(e, "readback");
    }
    return PIC_SUCCESS;
}

}  // namespace picx
