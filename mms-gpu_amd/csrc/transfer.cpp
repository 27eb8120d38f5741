// transfer.cpp -- copies between the caller's (pageable) arrays and the device
// through a ring of pinned chunks.
//
// hipMemcpy on pageable memory moved 14 GB/s into fresh arrays and 17 GB/s into
// touched ones (48 MB: 4.7 and 2.8 ms; the first touch of the pages is part of
// it), pinned memory 57 GB/s.  Here the DMA of one chunk runs while the CPU
// copies another, over all arrays of a call back to back, and large copies use a
// few threads, since one thread touches fresh pages at 33 GB/s.  Of 48 MB
// fresh (the state of a 1024 x 1024 x 4 film) 4.7 -> 1.6 ms to the host, 1.7 ->
// 1.2 to the device.  Smaller uploads and memory that the runtime knows are left
// to the runtime.  The rings belong
// to a pool: a call takes one, so calls of several threads do not meet, at
// most kKeep are kept, and they are freed with the last context.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

#include "mms_internal.hpp"

namespace mms {
namespace {

constexpr int kSlots = 4;
constexpr size_t kChunk = 4u << 20;   // largest chunk, and a slot's size
// Below these sizes the runtime's own pageable copy is as good or better.  To
// the host: 1.5 MB 121 us against 115, 4 MB 291 against 241.  To the device it
// moves 32 GB/s by itself, a single thread's chunks 30 (set_m of 2 MB 85 us
// against 108, 4 MB 141 / 170, 8 MB 256 / 270), and only several threads are
// faster: 16 MB 474 / 465 (new arrays 625 / 569), 24 MB 681 / 625, 48 MB 1662 / 1155.
constexpr size_t kRuntimeDown = 3u << 19, kRuntimeUp = 16u << 20;
constexpr size_t kAlone = 12u << 20;   // copies of this size and more use kThreads threads
constexpr int kThreads = 4;           // divides kSlots
constexpr size_t kKeep = 4;

struct Ring {
    char *pin = nullptr;
    int device = -1;                // events belong to a device
    hipEvent_t ev[kSlots] = {};
    bool used[kSlots] = {};         // ev recorded: wait before the slot is used again
};

std::mutex g_mu;
std::vector<Ring *> g_rings;  // free rings
long g_users = 0;

void ring_free(Ring *r) {
    for (hipEvent_t e : r->ev)
        if (e) (void)hipEventDestroy(e);
    if (r->pin) (void)hipHostFree(r->pin);
    delete r;
}

Ring *ring_take(int device) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        for (size_t i = 0; i < g_rings.size(); i++)
            if (g_rings[i]->device == device) {
                Ring *r = g_rings[i];
                g_rings.erase(g_rings.begin() + i);
                return r;
            }
    }
    Ring *r = new Ring();
    r->device = device;
    bool ok = hipHostMalloc(reinterpret_cast<void **>(&r->pin), kSlots * kChunk, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t &e : r->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        ring_free(r);
        return nullptr;
    }
    return r;
}

void ring_give(Ring *r) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        if (g_users > 0 && g_rings.size() < kKeep) {
            g_rings.push_back(r);
            return;
        }
    }
    for (int i = 0; i < kSlots; i++)
        if (r->used[i]) (void)hipEventSynchronize(r->ev[i]);
    ring_free(r);
}

struct Piece { char *host; char *dev; size_t bytes; };

// every chunk c with c mod nt == w; chunk c uses slot c mod kSlots
bool run_pieces(Ring *r, const std::vector<Piece> &pieces, bool to_device, int w, int nt, hipStream_t s) {
    const int n = (int)pieces.size(), ahead = kSlots / nt;
    auto slot_free = [&](int c) {
        const int k = c % kSlots;
        if (!r->used[k]) return true;
        r->used[k] = false;
        return hipEventSynchronize(r->ev[k]) == hipSuccess;
    };
    auto mark = [&](int c) {
        r->used[c % kSlots] = true;
        return hipEventRecord(r->ev[c % kSlots], s) == hipSuccess;
    };
    auto pin = [&](int c) { return r->pin + (size_t)(c % kSlots) * kChunk; };
    if (to_device) {
        for (int c = w; c < n; c += nt) {
            const Piece &p = pieces[c];
            if (!slot_free(c)) return false;
            memcpy(pin(c), p.host, p.bytes);
            if (hipMemcpyAsync(p.dev, pin(c), p.bytes, hipMemcpyHostToDevice, s) != hipSuccess || !mark(c)) return false;
        }
        return true;
    }
    auto start = [&](int c) {
        return slot_free(c) &&
               hipMemcpyAsync(pin(c), pieces[c].dev, pieces[c].bytes, hipMemcpyDeviceToHost, s) == hipSuccess && mark(c);
    };
    int next = w;
    for (int k = 0; k < ahead && next < n; k++, next += nt)
        if (!start(next)) return false;
    for (int c = w; c < n; c += nt) {
        if (!slot_free(c)) return false;  // waits for the chunk's copy
        memcpy(pieces[c].host, pin(c), pieces[c].bytes);
        if (next < n) {
            if (!start(next)) return false;
            next += nt;
        }
    }
    return true;
}

// the runtime's own copy
int copy_runtime(const Xfer &x, bool to_device, hipStream_t s) {
    MMS_HIP(hipMemcpyAsync(to_device ? x.dev : x.host, to_device ? x.host : x.dev, x.bytes,
                           to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s));
    return 0;
}

// Memory the runtime knows (pinned, managed or a device's) is copied by DMA
// without a chunk in between, and may not be the CPU's to read.
bool pageable(const void *p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();
    return true;
}

// the arrays of `mask` through a ring; -1: no pinned memory to be had
int run_ring(const Xfer *x, int count, unsigned mask, size_t total, bool to_device, hipStream_t s) {
    // events and threads on the stream's device, whatever the caller's is
    int caller = 0;
    hipDevice_t device = 0;
    MMS_HIP(hipGetDevice(&caller));
    MMS_HIP(hipStreamGetDevice(s, &device));
    if (caller != device) MMS_HIP(hipSetDevice(device));
    Ring *r = ring_take(device);
    if (caller != device) MMS_HIP(hipSetDevice(caller));
    if (!r) {
        (void)hipGetLastError();
        return -1;
    }
    const int nt = total >= kAlone ? kThreads : 1;
    // A chunk costs about 14 us of DMA start and event on top of its bytes at
    // 53 GB/s, and the last one's CPU copy is not overlapped: both together are
    // least at a chunk of sqrt(14 us x 50 GB/s x total), in steps of 64 KB
    // (2.3 MB in two pieces, 17 MB in five).
    size_t chunk = (size_t)sqrt(7e5 * (double)total);
    chunk = std::min(kChunk, (chunk + 65535) & ~(size_t)65535);
    std::vector<Piece> pieces;
    for (int i = 0; i < count; i++)
        for (size_t o = 0; (mask >> i & 1) && o < x[i].bytes; o += chunk)
            pieces.push_back({static_cast<char *>(x[i].host) + o, static_cast<char *>(x[i].dev) + o,
                              std::min(chunk, x[i].bytes - o)});
    std::atomic<bool> ok(true);
    std::vector<std::thread> th;
    int started = 1;  // this thread takes chunks 0 mod nt
    for (; started < nt; started++) {
        const int w = started;
        try {
            th.emplace_back([&, w] {
                if (hipSetDevice(device) != hipSuccess || !run_pieces(r, pieces, to_device, w, nt, s)) ok = false;
            });
        } catch (...) {
            break;  // no thread to be had: this one does the rest
        }
    }
    if (!run_pieces(r, pieces, to_device, 0, nt, s)) ok = false;
    for (int w = started; w < nt; w++)
        if (!run_pieces(r, pieces, to_device, w, nt, s)) ok = false;
    for (std::thread &t : th) t.join();
    ring_give(r);
    MMS_CHECK(ok.load(), to_device ? "copy to the device failed" : "copy to the host failed");
    return 0;
}

// a call has at most 32 arrays (rk4_step: six)
int run(const Xfer *x, int count, bool to_device, hipStream_t s) {
    const size_t line = to_device ? kRuntimeUp : kRuntimeDown;
    size_t total = 0;
    for (int i = 0; i < count; i++)
        if (x[i].host) total += x[i].bytes;
    if (!total) return 0;
    unsigned ring = 0;  // arrays that take the chunks
    if (total >= line) {
        total = 0;
        for (int i = 0; i < count; i++)
            if (x[i].host && pageable(x[i].host)) {
                ring |= 1u << i;
                total += x[i].bytes;
            }
        if (total < line) ring = 0;
    }
    bool direct = false;
    auto runtime = [&](unsigned mask) {
        for (int i = 0; i < count; i++)
            if (x[i].host && (mask >> i & 1)) {
                direct = true;
                if (copy_runtime(x[i], to_device, s)) return 1;
            }
        return 0;
    };
    if (runtime(~ring)) return 1;
    if (ring) {
        const int st = run_ring(x, count, ring, total, to_device, s);
        if (st > 0 || (st < 0 && runtime(ring))) return 1;
    }
    // (the chunks have been waited for one by one; a wait for the stream after them takes 50 us)
    if (direct && !to_device) MMS_HIP(hipStreamSynchronize(s));
    return 0;
}

}  // namespace

int HostBuffer::alloc(size_t bytes) {
    void *m = nullptr;
    pinned = hipHostMalloc(&m, bytes, hipHostMallocDefault) == hipSuccess;
    if (!pinned) {
        (void)hipGetLastError();
        m = malloc(bytes);
    }
    p = static_cast<char *>(m);
    MMS_CHECK(p, "no host memory for the time loop");
    return 0;
}

void HostBuffer::release() {
    if (pinned) (void)hipHostFree(p);
    else free(p);
    p = nullptr;
    pinned = false;
}

int copy_to_device(const Xfer *x, int count, hipStream_t s) { return run(x, count, true, s); }
int copy_to_host(const Xfer *x, int count, hipStream_t s) { return run(x, count, false, s); }

void transfer_user(int delta) {
    std::vector<Ring *> gone;
    {
        std::lock_guard<std::mutex> lk(g_mu);
        g_users += delta;
        if (g_users == 0) gone.swap(g_rings);
    }
    for (Ring *r : gone) {
        for (int i = 0; i < kSlots; i++)
            if (r->used[i]) (void)hipEventSynchronize(r->ev[i]);
        ring_free(r);
    }
}

}  // namespace mms
