/*
 * st_copy.h - large copies between pageable host memory and the device.
 *
 * A copy call on pageable memory goes through a page-locked buffer of the
 * runtime with one thread moving the bytes: 52 MB of mesh geometry took 3.8
 * ms (14 GB/s on a link of 57), 15 MB of fresh pages for hit records 1.1 ms,
 * most of it page faults. Here the bytes go through a ring of page-locked
 * slots with several threads at its host side: 1.2 and 0.5 ms. Smaller copies
 * keep the call, which then costs less than the threads.
 */
#ifndef ST_COPY_H
#define ST_COPY_H

#include <hip/hip_runtime.h>

#include <string.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <new>
#include <thread>
#include <vector>

#define COPY_SLOTS 8u
#define COPY_SLOT_BYTES (2u << 20)
/* Bytes from which the ring is used. A depth frame into pageable memory, ring
   and call: 2 MiB 216 and 178 us, 3 MiB 269 and 257, 4 MiB 314 and 328, 8 MiB
   460 and 605. Uploads by themselves gain from some 20 MB on (creating a scene
   with a device-built mesh: 11.9 MB 1010 and 922 us, 15.9 MB 1155 and 1070,
   31.8 MB 2075 and 2300, 49.6 MB 2765 and 3515), but the launches after large
   calls pay for them, it seems where the caller's memory, pinned for the call,
   is freed: the first burst of 48 requests at a new server with four scenes of
   22 MB took 13.2 ms (15.1 in one of 8 processes) with their uploads through
   the ring, and 16.5 in 5 of 8 with calls. */
#define COPY_MIN_BYTES (4u << 20)
#define COPY_THREADS 8u

/* A launch context's ring: 16 MiB of page-locked memory and an event per
   slot, taken with the first large copy. */
struct CopyRing {
    char *base;
    hipEvent_t ev[COPY_SLOTS];
};

static inline void copy_ring_release(CopyRing *r) {
    if (r->base) (void)hipHostFree(r->base);
    for (uint32_t i = 0; i < COPY_SLOTS; i++)
        if (r->ev[i]) (void)hipEventDestroy(r->ev[i]);
    *r = CopyRing();
}
static inline bool copy_ring_ready(CopyRing *r) {
    if (r->base) return true;
    bool ok = hipHostMalloc((void **)&r->base, (size_t)COPY_SLOTS * COPY_SLOT_BYTES, hipHostMallocDefault) == hipSuccess;
    for (uint32_t i = 0; i < COPY_SLOTS && ok; i++)
        ok = hipEventCreateWithFlags(&r->ev[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        copy_ring_release(r);
        (void)hipGetLastError();
    }
    return ok;
}

struct CopySpan {
    char *dev, *host;
    size_t bytes;
    uint32_t limit;   /* an upload of indices: each 32-bit word has to be below it (0: not indices) */
    bool direct;      /* set by copy_spans: not pageable memory */
};

static inline bool words_below(const char *p, size_t bytes, uint32_t limit) {
    const uint32_t *w = (const uint32_t *)p;
    uint32_t over = 0;
    for (size_t i = 0; i < bytes / 4; i++) over |= (uint32_t)(w[i] >= limit);
    return !over;
}

/* Whether the runtime knows the memory (page-locked by whomever, or the
   device's): a plain copy call then runs at the link's rate, with no bytes
   for threads to move. */
static inline bool copy_known(const char *p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

/* Copy the spans between host memory and the device on `stream`, after the
   work queued there; complete when the call returns. Plain copy calls for
   memory that is not pageable, where the whole is small or the ring or its
   threads cannot be had, and where the spans have to be copied one after
   another (in_order: they overlap).
   *in_range (uploads) tells whether all indices are below their limits: the
   threads look while they have the bytes at hand (24 MB of indices by
   themselves, on one thread: 2 ms). */
static inline hipError_t copy_spans(hipStream_t stream, CopyRing *ring, CopySpan *spans, size_t nspans,
                                       bool download, bool in_order, bool *in_range = nullptr) {
    size_t total = 0;
    for (size_t k = 0; k < nspans; k++) total += spans[k].bytes;
    std::atomic<uint32_t> over(0);
    hipError_t e = hipSuccess;
    auto copy_calls = [&](bool direct) {
        for (size_t k = 0; k < nspans && e == hipSuccess; k++) {
            const CopySpan &s = spans[k];
            if (!s.bytes || s.direct != direct) continue;
            if (in_range && s.limit && !words_below(s.host, s.bytes, s.limit)) *in_range = false;
            e = download ? hipMemcpyAsync(s.host, s.dev, s.bytes, hipMemcpyDeviceToHost, stream)
                         : hipMemcpyAsync(s.dev, s.host, s.bytes, hipMemcpyHostToDevice, stream);
        }
    };
    auto plain = [&]() {
        copy_calls(false);
        const hipError_t w = hipStreamSynchronize(stream);
        return e != hipSuccess ? e : w;
    };
    if (in_range) *in_range = true;
    for (size_t k = 0; k < nspans; k++) spans[k].direct = false;
    if (in_order || total < COPY_MIN_BYTES) return plain();
    for (size_t k = 0; k < nspans; k++) {
        CopySpan &s = spans[k];
        s.direct = s.bytes && !s.limit && copy_known(s.host) && copy_known(s.host + s.bytes - 1);
        if (s.direct) total -= s.bytes;
    }
    copy_calls(true);
    if (e != hipSuccess || total < COPY_MIN_BYTES || !copy_ring_ready(ring)) return plain();
    /* Slot by slot, as many spans as fit: 60 images of 120 KB 1555 us (1610
       with plain calls, 2030 with a slot and an event for each). */
    struct Piece {
        char *dev, *host;
        uint32_t at, bytes, limit;   /* at: in the slot */
    };
    std::vector<Piece> piece;
    std::vector<uint32_t> first;     /* chunk i: pieces first[i] to first[i + 1] */
    /* A chunk's state: `open` says that its slot may be moved by a thread (the
       download into it is done, or the upload before it has left it), `moved`
       that a thread has done so. Threads take chunks in order. */
    std::vector<std::atomic<uint32_t>> open, moved;
    std::vector<std::thread> team;
    try {
        uint32_t used = COPY_SLOT_BYTES;
        for (size_t k = 0; k < nspans; k++)
            for (size_t done = 0; done < spans[k].bytes && !spans[k].direct;) {
                if (used >= COPY_SLOT_BYTES) {
                    first.push_back((uint32_t)piece.size());
                    used = 0;
                }
                const uint32_t n = (uint32_t)std::min(spans[k].bytes - done, (size_t)(COPY_SLOT_BYTES - used));
                piece.push_back({spans[k].dev + done, spans[k].host + done, used, n, spans[k].limit});
                used = (used + n + 255u) & ~255u;
                done += n;
            }
        first.push_back((uint32_t)piece.size());
        std::vector<std::atomic<uint32_t>>(first.size()).swap(open);
        std::vector<std::atomic<uint32_t>>(first.size()).swap(moved);
        team.reserve(COPY_THREADS);
    } catch (const std::bad_alloc &) {
        return plain();
    }
    const uint32_t chunks = (uint32_t)first.size() - 1u;
    for (uint32_t i = 0; i < chunks; i++) open[i] = moved[i] = 0;
    std::atomic<uint32_t> next(0), stop(0);
    auto work = [&]() {
        for (;;) {
            const uint32_t i = next.fetch_add(1);
            if (i >= chunks) return;
            while (!open[i].load(std::memory_order_acquire)) {
                if (stop.load()) return;
                std::this_thread::yield();
            }
            char *slot = ring->base + (size_t)(i % COPY_SLOTS) * COPY_SLOT_BYTES;
            for (uint32_t k = first[i]; k < first[i + 1]; k++) {
                const Piece &p = piece[k];
                if (download) memcpy(p.host, slot + p.at, p.bytes);
                else memcpy(slot + p.at, p.host, p.bytes);
                if (p.limit && !words_below(p.host, p.bytes, p.limit)) over = 1;
            }
            moved[i].store(1, std::memory_order_release);
        }
    };
    auto start_team = [&]() {
        try {
            for (uint32_t t = 0; t < COPY_THREADS && t < chunks; t++) team.emplace_back(work);
        } catch (const std::exception &) {   /* no thread or no memory for one: those that run do it */
        }
        return !team.empty();
    };
    auto wait_moved = [&](uint32_t i) {
        while (!moved[i].load(std::memory_order_acquire)) std::this_thread::yield();
    };
    auto queue = [&](uint32_t i) {
        char *slot = ring->base + (size_t)(i % COPY_SLOTS) * COPY_SLOT_BYTES;
        hipError_t q = hipSuccess;
        for (uint32_t k = first[i]; k < first[i + 1] && q == hipSuccess; k++) {
            const Piece &p = piece[k];
            q = download ? hipMemcpyAsync(slot + p.at, p.dev, p.bytes, hipMemcpyDeviceToHost, stream)
                         : hipMemcpyAsync(p.dev, slot + p.at, p.bytes, hipMemcpyHostToDevice, stream);
        }
        return q != hipSuccess ? q : hipEventRecord(ring->ev[i % COPY_SLOTS], stream);
    };
    if (download) {
        for (uint32_t i = 0; i < chunks && i < COPY_SLOTS && e == hipSuccess; i++) e = queue(i);
        /* the threads start when there is something to move: the stream may
           have a whole render ahead of the copies */
        if (e == hipSuccess) e = hipEventSynchronize(ring->ev[0]);
        if (e == hipSuccess && !start_team()) return plain();
        for (uint32_t i = 0; i < chunks && e == hipSuccess; i++) {
            e = hipEventSynchronize(ring->ev[i % COPY_SLOTS]);
            if (e != hipSuccess) break;
            open[i].store(1, std::memory_order_release);
            /* the slot before this one goes round again once it is empty */
            if (i >= 1 && i - 1 + COPY_SLOTS < chunks) {
                wait_moved(i - 1);
                e = queue(i - 1 + COPY_SLOTS);
            }
        }
        for (uint32_t i = 0; i < chunks && e == hipSuccess; i++) wait_moved(i);
    } else {
        if (!start_team()) return plain();
        for (uint32_t i = 0; i < chunks && i < COPY_SLOTS; i++) open[i].store(1, std::memory_order_release);
        for (uint32_t i = 0; i < chunks && e == hipSuccess; i++) {
            wait_moved(i);
            e = queue(i);
            /* the slot that has to be free next */
            if (e == hipSuccess && i + 1 >= COPY_SLOTS / 2 && i + 1 + COPY_SLOTS / 2 < chunks) {
                const uint32_t old = i + 1 - COPY_SLOTS / 2;
                e = hipEventSynchronize(ring->ev[old % COPY_SLOTS]);
                if (e == hipSuccess) open[old + COPY_SLOTS].store(1, std::memory_order_release);
            }
        }
    }
    /* the ring is free again when the call returns, also with an error */
    if (!download || e != hipSuccess) {
        const hipError_t w = hipStreamSynchronize(stream);
        if (e == hipSuccess) e = w;
    }
    stop = 1;
    for (std::thread &t : team) t.join();
    if (in_range && over) *in_range = false;
    return e;
}

#endif
