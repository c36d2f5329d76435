// Device-to-host copies of a download into the caller's pageable memory.
//
// A copy straight into pageable memory makes the runtime stage or pin the
// caller's pages itself, on one thread, and first touches of new pages are
// taken there too: 0.31 ms for 0.7 MB, 5.0 ms for 48 MB, 11.5 ms for 112 MB
// into new arrays, against 0.02, 0.9 and 2.1 ms for the transfer alone.  Here
// the device block is copied in chunks to pinned memory and on from there by
// the host while the next chunks arrive: 0.05, 1.4 and 3.3 ms.  What is left
// above the transfer is the host's page faults.
#include <hip/hip_runtime.h>

#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <utility>

#include "lus_device.hpp"
#include "lus_internal.hpp"

namespace lus {

// Chunks of 2 MB over four threads from 8 MB on: 48 MB take 1.4 ms with them,
// 3.6 ms on one thread; 1 MB chunks 1.9 ms, 8 MB chunks 1.7 ms, eight threads
// 1.45 ms.  Below, starting threads costs what they save (3 MB: 0.15 ms with
// one or four), and 1 MB chunks overlap better.  A download holds at most
// 16 MB of pinned memory for it.
constexpr size_t kPullSplit = (size_t)8 << 20;
constexpr size_t kPullChunk = (size_t)2 << 20;
constexpr size_t kPullSmallChunk = (size_t)1 << 20;
constexpr int kPullThreads = 4;

// a context's events
struct HostPull {
    hipEvent_t ev[2 * kPullThreads] = {};
    int nev = 0;
};

void pull_free(HostPull* hp) {
    if (!hp) return;
    for (int k = 0; k < hp->nev; ++k) (void)hipEventDestroy(hp->ev[k]);
    delete hp;
}

namespace {

// The pinned memory belongs to a download only while it runs: the contexts
// take it from these blocks in turn (allocating 16 MB takes 0.3 ms, smaller
// ones 0.02 to 0.07).  Reserving it with each scene instead made scenes longer
// to prepare (1M 3.4 -> 3.9 ms, 512 particles 0.24 -> 0.27), for a program that
// downloads nothing too; a new scene's first download takes 2.7 ms at 1M and
// 0.03 at 512 so, 3.1 and 0.04 then.  At most kPinIdle blocks are kept, and none
// once the last context is gone.
struct PinBlock {
    char* p = nullptr;
    size_t cap = 0;
};
constexpr int kPinIdle = 4;
struct PinPool {
    std::mutex m;
    PinBlock idle[kPinIdle];
    int contexts = 0;
};
// (never destroyed: at exit the runtime may be gone before it)
PinPool& pin_pool() {
    static PinPool* pool = new PinPool;
    return *pool;
}

// the smallest idle block of at least `bytes`, or a new one (p null: none to be had)
PinBlock pin_take(size_t bytes) {
    PinPool& pool = pin_pool();
    PinBlock got;
    {
        std::lock_guard<std::mutex> lock(pool.m);
        PinBlock* best = nullptr;
        for (PinBlock& b : pool.idle)
            if (b.p && b.cap >= bytes && (!best || b.cap < best->cap)) best = &b;
        if (best) std::swap(got, *best);
    }
    if (got.p) return got;
    if (hipHostMalloc((void**)&got.p, bytes, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        got.p = nullptr;
        return got;
    }
    got.cap = bytes;
    return got;
}

// back to the idle ones; with all places taken the smallest is freed
void pin_give(PinBlock b) {
    PinPool& pool = pin_pool();
    {
        std::lock_guard<std::mutex> lock(pool.m);
        for (PinBlock& q : pool.idle)
            if (q.cap < b.cap) std::swap(q, b);
    }
    if (b.p) (void)hipHostFree(b.p);
}

}  // namespace

void pull_open() {
    PinPool& pool = pin_pool();
    std::lock_guard<std::mutex> lock(pool.m);
    ++pool.contexts;
}

void pull_close() {
    PinPool& pool = pin_pool();
    PinBlock gone[kPinIdle];
    {
        std::lock_guard<std::mutex> lock(pool.m);
        if (--pool.contexts > 0) return;
        for (int k = 0; k < kPinIdle; ++k) std::swap(gone[k], pool.idle[k]);
    }
    for (const PinBlock& b : gone)
        if (b.p) (void)hipHostFree(b.p);
}

namespace {

hipError_t pull_events(HostPull* hp, int threads) {
    for (; hp->nev < 2 * threads; ++hp->nev) {
        const hipError_t e = hipEventCreateWithFlags(&hp->ev[hp->nev], hipEventDisableTiming);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

struct Pull {
    int device;
    hipStream_t s;
    const HostPull* hp;
    char* pin;
    const char* dev;
    const HostPiece* pc;
    int np, threads, chunks, n_iota;
    size_t total, chunk;
    int* iota;

    size_t first(int i) const { return chunk * (size_t)i; }
    size_t length(int i) const { return first(i) + chunk <= total ? chunk : total - first(i); }
    // slot u of thread w
    char* slot(int w, int u) const { return pin + chunk * (size_t)(2 * w + u); }

    hipError_t issue(int w, int u, int i) const {
        const hipError_t e = hipMemcpyAsync(slot(w, u), dev + first(i), length(i), hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipEventRecord(hp->ev[2 * w + u], s);
    }
    // bytes [a, a + len) of the block from q to where they belong
    void put(const char* q, size_t a, size_t len) const {
        size_t at = 0;
        for (int k = 0; k < np && at < a + len; at += pc[k].bytes, ++k) {
            const size_t b = a > at ? a : at;
            const size_t e = a + len < at + pc[k].bytes ? a + len : at + pc[k].bytes;
            if (b >= e) continue;
            memcpy(static_cast<char*>(pc[k].dst) + (b - at), q + (b - a), e - b);
            if (pc[k].also) memcpy(static_cast<char*>(pc[k].also) + (b - at), q + (b - a), e - b);
        }
    }
    // thread w's chunks: w, w + threads, ..., two in flight
    hipError_t run(int w) const {
        hipError_t e = hipSetDevice(device);
        for (int u = 0; u < 2 && e == hipSuccess; ++u)
            if (w + u * threads < chunks) e = issue(w, u, w + u * threads);
        const size_t lo = (size_t)n_iota * w / threads, hi = (size_t)n_iota * (w + 1) / threads;
        for (size_t r = lo; r < hi; ++r) iota[r] = (int)r;
        int u = 0;
        for (int i = w; i < chunks && e == hipSuccess; i += threads, u ^= 1) {
            e = hipEventSynchronize(hp->ev[2 * w + u]);
            if (e != hipSuccess) break;
            put(slot(w, u), first(i), length(i));
            if (i + 2 * threads < chunks) e = issue(w, u, i + 2 * threads);
        }
        return e;
    }
};

// memory that the runtime knows (pinned by the caller): copied to directly
bool known_memory(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

// threads, chunk and pinned bytes for a block of `total` bytes (and `more`
// written by the host alone)
static size_t pull_plan(size_t total, size_t more, int* threads, size_t* chunk) {
    *threads = total + more >= kPullSplit ? kPullThreads : 1;
    *chunk = *threads > 1 ? kPullChunk : kPullSmallChunk;
    // one chunk (a small download) needs no more than its own size
    if (*threads == 1 && total <= *chunk) return (total + 4095) & ~(size_t)4095;
    return (size_t)2 * *threads * *chunk;
}

hipError_t pull_to_host(LusGpu* c, const void* dev, const HostPiece* pc, int np, int* iota, int n_iota) {
    hipStream_t s = ctx_stream(c);
    HostPull*& hp = ctx_pull(c);
    Pull p{};
    p.device = ctx_device(c);
    p.s = s;
    p.dev = static_cast<const char*>(dev);
    p.pc = pc;
    p.np = np;
    p.iota = iota;
    p.n_iota = n_iota;
    bool direct = false;
    for (int k = 0; k < np; ++k) {
        p.total += pc[k].bytes;
        direct = direct || known_memory(pc[k].dst) || (pc[k].also && known_memory(pc[k].also));
    }
    const size_t need = pull_plan(p.total, sizeof(int) * (size_t)n_iota, &p.threads, &p.chunk);
    p.chunks = (int)((p.total + p.chunk - 1) / p.chunk);
    PinBlock pin;
    if (!direct && need > 0) {
        if (!hp) hp = new (std::nothrow) HostPull;
        if (!hp || pull_events(hp, p.threads) != hipSuccess) {
            (void)hipGetLastError();
            direct = true;
        } else {
            pin = pin_take(need);
            direct = !pin.p;
        }
    }
    if (direct) {
        size_t at = 0;
        for (int k = 0; k < np; at += pc[k].bytes, ++k) {
            if (pc[k].bytes == 0) continue;
            for (void* d : {pc[k].dst, pc[k].also}) {
                if (!d) continue;
                const hipError_t e = hipMemcpyAsync(d, p.dev + at, pc[k].bytes, hipMemcpyDeviceToHost, s);
                if (e != hipSuccess) return e;
            }
        }
        for (int r = 0; r < n_iota; ++r) iota[r] = r;
        return hipStreamSynchronize(s);
    }
    p.hp = hp;
    p.pin = pin.p;
    hipError_t err[kPullThreads] = {};
    std::thread th[kPullThreads];
    int started = 1;
    try {
        for (; started < p.threads; ++started)
            th[started] = std::thread([&p, &err, started] { err[started] = p.run(started); });
    } catch (const std::exception&) {  // no thread: its chunks are taken here
    }
    err[0] = p.run(0);
    for (int w = started; w < p.threads; ++w) err[w] = p.run(w);
    for (int w = 1; w < started; ++w) th[w].join();
    hipError_t bad = hipSuccess;
    for (hipError_t e : err)
        if (e != hipSuccess) bad = e;
    if (bad != hipSuccess) (void)hipStreamSynchronize(s);  // no copy into the slots is left in flight
    pin_give(pin);
    return bad;
}

}  // namespace lus
