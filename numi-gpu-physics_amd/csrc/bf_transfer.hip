// Copies between the caller's (pageable) arrays and the device.
//
// A pageable copy moves one staging block at a time through one host thread,
// which also takes the page faults of a fresh destination: 10.7 GB/s into
// fresh memory (18 GB/s into touched memory), while the link does four times
// that; a small one costs 60 - 130 us of runtime bookkeeping.  Here the data
// passes through pinned slots.  A large copy is cut into blocks shared by a
// few threads, each owning a slot and alternating between the DMA of a block
// and its memory copy, so that the link and several cores work at the same
// time: 50 MB into fresh memory 4.8 -> 1.5 ms, 403 MB 39.6 -> 9.4 ms
// (43 GB/s; blocks of 4 MB, 8 threads; 2 MB reach 40 GB/s, 1 MB 31).  One
// thread per 4 MB: up to that one thread is as fast as several (0.25 ms), and
// the copies go through one slot with one wait (density and velocity of 24^3
// cells: 128 -> 41 us); 14 MB take 0.53 ms with three threads, 0.81 with one.
// The slots belong to the context, are made by its first copy (0.05 ms each)
// and given back with it.  Where pinned memory or threads are not to be had,
// fewer workers (down to the plain copy) do the same work.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "bf_launch.h"

namespace bf {

constexpr size_t BLOCK = size_t(4) << 20;       // bytes of a slot; work that pays for a thread

void HostPipe::release() {
    for (int i = 0; i < SLOTS; ++i) {
        if (slot[i]) (void)hipHostFree(slot[i]);
        if (done[i]) (void)hipEventDestroy(done[i]);
        slot[i] = nullptr;
        done[i] = nullptr;
    }
    slots = 0;
}

// Makes slots up to `want`, once each; returns how many there are.
static int ensure_slots(HostPipe& p, int want) {
    while (p.slots < want && !p.exhausted) {
        const int i = p.slots;
        if (hipHostMalloc(&p.slot[i], BLOCK, hipHostMallocDefault) != hipSuccess) p.slot[i] = nullptr;
        if (p.slot[i] && hipEventCreateWithFlags(&p.done[i], hipEventDisableTiming) != hipSuccess) p.done[i] = nullptr;
        if (!p.slot[i] || !p.done[i]) {
            (void)hipGetLastError();
            p.exhausted = true;
            break;
        }
        p.slots = i + 1;
    }
    return p.slots;
}

// Block `i` of the copies.
struct Piece {
    char* host;
    char* dev;
    size_t bytes;
};
static bool piece_of(const HostCopy* copies, int n, size_t i, Piece& out) {
    for (int k = 0; k < n; ++k) {
        const size_t blocks = (copies[k].bytes + BLOCK - 1) / BLOCK;
        if (i < blocks) {
            const size_t at = i * BLOCK;
            out = {(char*)copies[k].host + at, (char*)copies[k].dev + at, std::min(BLOCK, copies[k].bytes - at)};
            return true;
        }
        i -= blocks;
    }
    return false;
}

// Runs worker(t) for t < n on up to n threads, the caller's among them; the
// workers take blocks from a shared counter until none is left, so a thread
// that could not be started only leaves more for the others.
template <typename F>
static void run_workers(int n, F&& worker) {
    std::thread threads[HostPipe::SLOTS];
    int started = 0;
    for (int t = 1; t < n; ++t) {
        try {
            threads[t] = std::thread(worker, t);
            started = t;
        } catch (const std::exception&) {     // no thread, or no memory for one
            break;
        }
    }
    worker(0);
    for (int t = 1; t <= started; ++t) threads[t].join();
}

static hipError_t transfer(HostPipe& p, int device, const HostCopy* copies, int n, bool to_host, hipStream_t s) {
    size_t bytes = 0;
    for (int k = 0; k < n; ++k) bytes += copies[k].bytes;
    const int want = (int)std::min<size_t>(HostPipe::SLOTS, std::max<size_t>(1, bytes / BLOCK));
    const int have = std::min(want, ensure_slots(p, want));
    if (have == 0) {
        hipError_t e = hipSuccess;
        for (int k = 0; k < n && e == hipSuccess; ++k)
            e = hipMemcpyAsync(to_host ? copies[k].host : copies[k].dev, to_host ? copies[k].dev : copies[k].host,
                               copies[k].bytes, to_host ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    if (have == 1 && bytes <= BLOCK) {
        // everything in one slot: the copies queue up and one wait serves them
        hipError_t e = hipSuccess;
        char* at = (char*)p.slot[0];
        for (int k = 0; k < n && e == hipSuccess; at += copies[k].bytes, ++k) {
            if (!to_host) std::memcpy(at, copies[k].host, copies[k].bytes);
            e = to_host ? hipMemcpyAsync(at, copies[k].dev, copies[k].bytes, hipMemcpyDeviceToHost, s)
                        : hipMemcpyAsync(copies[k].dev, at, copies[k].bytes, hipMemcpyHostToDevice, s);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        at = (char*)p.slot[0];
        for (int k = 0; k < n && e == hipSuccess && to_host; at += copies[k].bytes, ++k)
            std::memcpy(copies[k].host, at, copies[k].bytes);
        return e;
    }
    std::atomic<size_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    run_workers(have, [&](int t) {
        hipError_t e = hipSetDevice(device);
        Piece b;
        while (e == hipSuccess && piece_of(copies, n, next.fetch_add(1), b)) {
            if (!to_host) std::memcpy(p.slot[t], b.host, b.bytes);
            e = to_host ? hipMemcpyAsync(p.slot[t], b.dev, b.bytes, hipMemcpyDeviceToHost, s)
                        : hipMemcpyAsync(b.dev, p.slot[t], b.bytes, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(p.done[t], s);
            if (e == hipSuccess) e = hipEventSynchronize(p.done[t]);   // data here, or the slot free again
            if (e == hipSuccess && to_host) std::memcpy(b.host, p.slot[t], b.bytes);
        }
        if (e != hipSuccess) error.store((int)e);
    });
    return (hipError_t)error.load();
}

hipError_t copy_to_host(HostPipe& p, int device, const HostCopy* copies, int n, hipStream_t s) {
    return transfer(p, device, copies, n, true, s);
}
hipError_t copy_to_host(HostPipe& p, int device, void* host, const void* dev, size_t bytes, hipStream_t s) {
    const HostCopy c{host, const_cast<void*>(dev), bytes};
    return transfer(p, device, &c, 1, true, s);
}
hipError_t copy_to_device(HostPipe& p, int device, void* dev, const void* host, size_t bytes, hipStream_t s) {
    const HostCopy c{const_cast<void*>(host), dev, bytes};
    return transfer(p, device, &c, 1, false, s);
}

}  // namespace bf
