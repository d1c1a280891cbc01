// hostcopy.hip — copies between the device and a caller's ordinary (pageable) host memory.
//
// hipMemcpyAsync moves such memory at 29 GB/s in and, with one thread taking the page faults of a
// fresh destination, 10 GB/s out; the link does 57.  Here a large copy is cut into chunks that
// several threads stage through page-locked slots of their own, on two streams: the host copies and
// page faults run side by side and overlap the transfers, and so do the transfers' starts and ends.
// A copy is paid for by the whole program: the threads also leave lines of its arrays in their own caches,
// and writing such an array anew, or an array in the pages that it gave back, then takes longer.  So in
// (fill_slot) the program's lines are prefetched past all but the first cache, and the sizes it starts at are
// set by the copy and the next pass over the array together.  Measured, hipMemcpyAsync -> this, us (4 threads, 2 MB
// slots, 32 MB of last-level cache; 6 and 8 threads were no faster, 1 MB slots or one stream 15-25 % slower):
//   in, and the next array's writing before it (fresh pages):
//     16 MB 586 + 270 -> 429 + 262, 24 MB 894 + 537 -> 580 + 424, 33 MB 1204 + 1126 -> 763 + 1042, 66 MB 2358 + 4569 -> 1572 + 4775
//     (without the prefetch 434 + 286, 593 + 475, 754 + 1107, 1541 + 5468)
//   out, and reading the result (fresh destination):
//     2 MB 135 + 62 -> 155 + 55, 4 MB 252 + 134 -> 230 + 98, 8 MB 527 + 276 -> 357 + 265, 33 MB 2484 + 1112 -> 1305 + 1104
// Out, it starts at 4 MB (allocating and freeing the result counted, 4.9 MB 612 -> 508 us in mapped memory, 451 -> 355
// in the heap; one state of a program's heap was seen where it lost, 737 -> 893, and 9.8 MB neither lost nor
// gained).  In, at 24 MB: a program that makes its 16 MB array out of others (a shifted 256^3
// volume) writes it in 1.80 ms instead of 1.46, for 0.04 gained in the copy, while frames of 33 and 66 MB from the
// device lose nothing (prepared in 17.9 ms, denoised in 5.85 ms without staging in, 4.58 with; 18.7 and 4.53 without
// the prefetch).
//
// The threads are started by the first copy that is large enough, sleep between copies, and end with
// vt_copy_release().  One copy runs at a time (the callers hold the runtime lock; the engine has its
// own as well).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "vt_internal.h"

namespace {

constexpr uint32_t kCopyThreads = 4;               // with the caller's
constexpr size_t kMaxChunk = (size_t)2 << 20;      // a slot
constexpr size_t kMinChunk = (size_t)512 << 10;
constexpr size_t kMinIn = (size_t)24 << 20, kMinOut = (size_t)4 << 20;   // below: hipMemcpyAsync
constexpr uint32_t kLanes = 2;                     // streams a copy is spread over

struct Slots {          // one thread's: two, so that a host copy overlaps a transfer
    char* mem[2] = {};
    hipEvent_t ev[2] = {};
    bool pending[2] = {};   // a transfer out of the slot may still run (ev); kept from copy to copy
    // The slot may be written.
    bool free_slot(uint32_t k) {
        const bool ok = !pending[k] || hipEventSynchronize(ev[k]) == hipSuccess;
        pending[k] = false;
        return ok;
    }
};

struct Job {
    char* host = nullptr;
    char* dev = nullptr;
    size_t bytes = 0, chunk = 0, chunks = 0;
    bool in = false;    // host -> device
    hipStream_t s[kLanes] = {};
    std::atomic<size_t> next{0};
    std::atomic<bool> failed{false};
};

struct Engine {
    int device = 0;
    Slots slots[kCopyThreads];
    std::vector<std::thread> threads;
    std::mutex m;
    std::condition_variable go, done;
    uint64_t epoch = 0;         // copies started
    uint32_t busy = 0;          // threads still at the current one
    bool stop = false;
    hipStream_t lane = nullptr;            // default priority
    hipEvent_t fork = nullptr, join = nullptr;
    Job job;
};

std::mutex g_copy_lock;
Engine* g_engine = nullptr;     // never destroyed at exit: its threads may be asleep in it

// Into a slot, which the device reads next: stores past the caches, which the slots would push the program's own
// data out of, and loads that leave its lines in none but the first (see above).
void fill_slot(char* dst, const char* src, size_t n) {
    typedef long long v2 __attribute__((vector_size(16)));
    constexpr size_t kAhead = 1024;
    size_t i = 0;
    for (; i + 64 <= n; i += 64) {
        if (i + kAhead < n) __builtin_prefetch(src + i + kAhead, 0, 0);   // (non-temporal)
        v2 v[4];
        std::memcpy(v, src + i, 64);
        for (int k = 0; k < 4; ++k) __builtin_nontemporal_store(v[k], reinterpret_cast<v2*>(dst + i) + k);
    }
    std::memcpy(dst + i, src + i, n - i);
    std::atomic_thread_fence(std::memory_order_seq_cst);   // before the copy is queued
}

// This thread's share of the copy: chunks off the common counter, staged through its slots.
void work(Job& j, Slots& sl, uint32_t id) {
    const hipStream_t s = j.s[id % kLanes];
    auto piece = [&](size_t c, size_t* off) {
        *off = c * j.chunk;
        return std::min(j.chunk, j.bytes - *off);
    };
    if (j.in) {
        for (uint32_t k = 0;; k ^= 1u) {
            const size_t c = j.next.fetch_add(1);
            if (c >= j.chunks || j.failed) return;
            size_t off;
            const size_t n = piece(c, &off);
            if (!sl.free_slot(k)) j.failed = true;
            fill_slot(sl.mem[k], j.host + off, n);
            if (hipMemcpyAsync(j.dev + off, sl.mem[k], n, hipMemcpyHostToDevice, s) != hipSuccess ||
                hipEventRecord(sl.ev[k], s) != hipSuccess)
                j.failed = true;
            else
                sl.pending[k] = true;
        }
    }
    // out: the next chunk's transfer is queued before the current one is waited for
    bool used[2] = {false, false};
    size_t held[2] = {0, 0};
    auto start = [&](uint32_t k) {
        used[k] = false;
        const size_t c = j.next.fetch_add(1);
        if (c >= j.chunks || j.failed) return;
        size_t off;
        const size_t n = piece(c, &off);
        if (!sl.free_slot(k) || hipMemcpyAsync(sl.mem[k], j.dev + off, n, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipEventRecord(sl.ev[k], s) != hipSuccess) {
            j.failed = true;
            return;
        }
        used[k] = true;
        held[k] = c;
    };
    start(0);
    for (uint32_t k = 0; used[k]; k ^= 1u) {
        start(k ^ 1u);
        if (hipEventSynchronize(sl.ev[k]) != hipSuccess) {
            j.failed = true;
        } else {
            size_t off;
            const size_t n = piece(held[k], &off);
            std::memcpy(j.host + off, sl.mem[k], n);
        }
        used[k] = false;
    }
}

void thread_main(Engine* e, uint32_t id) {
    hipSetDevice(e->device);
    uint64_t seen = 0;
    std::unique_lock<std::mutex> lk(e->m);
    for (;;) {
        e->go.wait(lk, [&] { return e->stop || e->epoch != seen; });
        if (e->stop) return;
        seen = e->epoch;
        lk.unlock();
        work(e->job, e->slots[id], id);
        lk.lock();
        if (--e->busy == 0) e->done.notify_one();
    }
}

void destroy(Engine* e) {
    {
        std::lock_guard<std::mutex> lk(e->m);
        e->stop = true;
    }
    e->go.notify_all();
    for (auto& t : e->threads) t.join();
    for (auto& s : e->slots)
        for (int k = 0; k < 2; ++k) {
            if (s.ev[k]) hipEventDestroy(s.ev[k]);
            hipHostFree(s.mem[k]);
        }
    if (e->fork) hipEventDestroy(e->fork);
    if (e->join) hipEventDestroy(e->join);
    if (e->lane) hipStreamDestroy(e->lane);
    delete e;
}

// The engine, made on first use; null where threads or page-locked memory are not to be had.
Engine* engine() {
    if (g_engine) return g_engine;
    Engine* e = new (std::nothrow) Engine;
    if (!e) return nullptr;
    e->device = vt_rt_device();
    bool ok = hipStreamCreateWithFlags(&e->lane, hipStreamNonBlocking) == hipSuccess &&
              hipEventCreateWithFlags(&e->fork, hipEventDisableTiming) == hipSuccess &&
              hipEventCreateWithFlags(&e->join, hipEventDisableTiming) == hipSuccess;
    for (auto& s : e->slots)
        for (int k = 0; k < 2 && ok; ++k)
            ok = hipHostMalloc(reinterpret_cast<void**>(&s.mem[k]), kMaxChunk, hipHostMallocDefault) == hipSuccess &&
                 hipEventCreateWithFlags(&s.ev[k], hipEventDisableTiming) == hipSuccess;
    if (ok) try {
        e->threads.reserve(kCopyThreads);
        for (uint32_t t = 1; t < kCopyThreads; ++t) e->threads.emplace_back(thread_main, e, t);
    } catch (...) {
        ok = false;
    }
    if (!ok) {
        (void)hipGetLastError();
        destroy(e);
        return nullptr;
    }
    return g_engine = e;
}

// Staged copy; false if it has to be done otherwise.
bool staged(void* host, void* dev, size_t bytes, bool in, hipStream_t s, hipError_t* rc) {
    if (bytes < (in ? kMinIn : kMinOut) || !vt_copy_pageable(host, bytes)) return false;
    std::lock_guard<std::mutex> own(g_copy_lock);
    Engine* e = engine();
    if (!e) return false;
    Job& j = e->job;
    j.host = static_cast<char*>(host);
    j.dev = static_cast<char*>(dev);
    j.bytes = bytes;
    // two chunks and more per thread, so that their ends meet
    j.chunk = std::min(kMaxChunk, std::max(kMinChunk, (bytes / (2 * kCopyThreads) + 4095) & ~(size_t)4095));
    j.chunks = (bytes + j.chunk - 1) / j.chunk;
    j.in = in;
    j.s[0] = s;
    j.s[1] = e->lane;
    j.next = 0;
    j.failed = false;
    if (hipEventRecord(e->fork, s) != hipSuccess || hipStreamWaitEvent(e->lane, e->fork, 0) != hipSuccess) return false;
    {
        std::lock_guard<std::mutex> lk(e->m);
        ++e->epoch;
        e->busy = (uint32_t)e->threads.size();
    }
    e->go.notify_all();
    work(j, e->slots[0], 0);
    {
        std::unique_lock<std::mutex> lk(e->m);
        e->done.wait(lk, [&] { return e->busy == 0; });
    }
    if (hipEventRecord(e->join, e->lane) != hipSuccess || hipStreamWaitEvent(s, e->join, 0) != hipSuccess) j.failed = true;
    *rc = j.failed ? hipErrorUnknown : hipSuccess;
    return true;
}

}  // namespace

// Ordinary host memory at both ends of the range: neither page-locked nor known to the device.
bool vt_copy_pageable(const void* p, size_t bytes) {
    for (const char* q : {static_cast<const char*>(p), static_cast<const char*>(p) + bytes - 1}) {
        hipPointerAttribute_t at;
        if (hipPointerGetAttributes(&at, q) != hipSuccess) (void)hipGetLastError();
        else if (at.type != hipMemoryTypeUnregistered) return false;
    }
    return true;
}

// Host to device in the order of stream s; pageable source memory may be reused on return, page-locked
// memory when the stream has passed the copy (as hipMemcpyAsync).
hipError_t vt_copy_in(void* dev, const void* host, size_t bytes, hipStream_t s) {
    hipError_t rc;
    if (staged(const_cast<void*>(host), dev, bytes, true, s, &rc)) return rc;
    return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
}

// Device to host in the order of stream s; the caller synchronises the stream before it uses the result.
hipError_t vt_copy_out(void* host, const void* dev, size_t bytes, hipStream_t s) {
    hipError_t rc;
    if (staged(host, const_cast<void*>(dev), bytes, false, s, &rc)) return rc;
    return hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
}

// Ends the threads and frees the slots (cleanup()).
void vt_copy_release() {
    std::lock_guard<std::mutex> own(g_copy_lock);
    if (g_engine) destroy(g_engine);
    g_engine = nullptr;
}
