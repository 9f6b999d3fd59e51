// oe_copy.hip -- large device arrays to ordinary (pageable) host memory.
//
// The runtime copies to pageable memory through its own staging, one thread
// moving a piece after its transfer has ended: 10.5 GB/s into fresh pages, 18
// into touched ones, where the link carries 56.  A run's fields are 100 MB to
// gigabytes, read into fresh arrays, so reading them back cost a quarter of a
// 500-step run at 256^3.  Here the transfers run back to back into a ring of
// pinned pieces while a few host threads empty it into the destination (and
// take its page faults): 38 GB/s at 422 MB, 27 at 25 MB (MI355X host,
// fresh pages; 1 MB pieces 30, 3 instead of 8 pieces 28, 6 threads instead of 4
// no more).  A destination the runtime knows takes the transfers itself: pinned
// memory at 56 GB/s (192 MB; 39 through the ring), managed or device memory.
// The ring and the threads live for the call only, so nothing is shared
// between calls, threads or streams.

#include "oe_internal.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <memory>
#include <thread>

namespace oe {
namespace {

// Below: the runtime's copy.  Ring and threads cost about 0.2 ms (7.5 MB of
// gradients a training step, into warm pages, 0.43 ms either way).
constexpr size_t STAGE_MIN = 12u << 20;
constexpr int STAGE_SLOTS = 8, STAGE_THREADS = 4;

struct Piece {
    char* dst;
    const char* src;
    size_t n;
};

struct Ring {
    char* pinned = nullptr;
    hipEvent_t ev[STAGE_SLOTS] = {};
    std::vector<std::thread> threads;
    std::atomic<bool> stop{false};
    hipStream_t busy = nullptr;  // transfers into the ring may be under way on this stream
    bool make(size_t piece) {
        hipError_t err = hipHostMalloc((void**)&pinned, piece * STAGE_SLOTS, hipHostMallocDefault);
        if (err != hipSuccess) pinned = nullptr;
        for (int k = 0; k < STAGE_SLOTS && err == hipSuccess; ++k)
            if ((err = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming)) != hipSuccess) ev[k] = nullptr;
        if (err != hipSuccess) (void)hipGetLastError();
        return err == hipSuccess;
    }
    ~Ring() {
        stop.store(true);
        for (auto& t : threads) t.join();
        if (busy) (void)hipStreamSynchronize(busy);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (pinned) (void)hipHostFree(pinned);
    }
};

// *began stays false where there is no ring (nothing was copied).
hipError_t staged(const std::vector<Piece>& pieces, size_t piece, hipStream_t s, bool* began) {
    const size_t n = pieces.size();
    enum { EMPTY, FULL, DONE };
    std::unique_ptr<std::atomic<int>[]> state(new std::atomic<int>[n]);
    for (size_t q = 0; q < n; ++q) state[q].store(EMPTY);
    std::atomic<size_t> next{0};
    Ring r;
    if (!r.make(piece)) return hipErrorOutOfMemory;
    hipError_t err = hipSuccess;
    auto empty = [&] {
        for (;;) {
            const size_t c = next.fetch_add(1);
            if (c >= n) return;
            while (state[c].load(std::memory_order_acquire) != FULL) {
                if (r.stop.load()) return;
                std::this_thread::yield();
            }
            std::memcpy(pieces[c].dst, r.pinned + (c % STAGE_SLOTS) * piece, pieces[c].n);
            state[c].store(DONE, std::memory_order_release);
        }
    };
    r.threads.reserve(STAGE_THREADS);
    for (int t = 0; t < STAGE_THREADS; ++t) r.threads.emplace_back(empty);
    r.busy = s;
    *began = true;
    size_t full = 0;  // pieces whose transfer has been seen to end
    auto poll = [&](size_t issued) -> hipError_t {
        while (full < issued) {
            const hipError_t q = hipEventQuery(r.ev[full % STAGE_SLOTS]);
            if (q == hipErrorNotReady) return hipSuccess;
            if (q != hipSuccess) return q;
            state[full++].store(FULL, std::memory_order_release);
        }
        return hipSuccess;
    };
    for (size_t c = 0; c < n; ++c) {
        while (c >= STAGE_SLOTS && state[c - STAGE_SLOTS].load(std::memory_order_acquire) != DONE) {
            if ((err = poll(c)) != hipSuccess) return err;
            std::this_thread::yield();
        }
        const int k = (int)(c % STAGE_SLOTS);
        if ((err = hipMemcpyAsync(r.pinned + k * piece, pieces[c].src, pieces[c].n, hipMemcpyDeviceToHost, s)) != hipSuccess ||
            (err = hipEventRecord(r.ev[k], s)) != hipSuccess || (err = poll(c + 1)) != hipSuccess)
            return err;
    }
    while (full < n) {
        if ((err = hipEventSynchronize(r.ev[full % STAGE_SLOTS])) != hipSuccess) return err;
        state[full++].store(FULL, std::memory_order_release);
    }
    r.busy = nullptr;
    for (auto& t : r.threads) t.join();
    r.threads.clear();
    return hipSuccess;
}

// Whether p is memory that the runtime does not know: ordinary host memory.
bool pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t copy_to_host(const HostCopy* c, int n, hipStream_t s) {
    size_t total = 0;
    bool page = true;
    for (int q = 0; q < n; ++q) total += c[q].bytes;
    for (int q = 0; q < n && page && total >= STAGE_MIN; ++q) page = pageable(c[q].dst);
    if (page && total >= STAGE_MIN) {
        bool began = false;  // without memory, events or threads for the ring: the runtime's copy below
        try {
            const size_t piece = 2u << 20;
            std::vector<Piece> pieces;
            for (int q = 0; q < n; ++q)
                for (size_t o = 0; o < c[q].bytes; o += piece)
                    pieces.push_back({static_cast<char*>(c[q].dst) + o, static_cast<const char*>(c[q].src) + o,
                                      std::min(piece, c[q].bytes - o)});
            const hipError_t err = staged(pieces, piece, s, &began);
            if (began) return err;
        } catch (const std::exception&) {
        }
    }
    for (int q = 0; q < n; ++q) {
        const hipError_t err = hipMemcpyAsync(c[q].dst, c[q].src, c[q].bytes, hipMemcpyDeviceToHost, s);
        if (err != hipSuccess) return err;
    }
    return hipStreamSynchronize(s);
}

}  // namespace oe
