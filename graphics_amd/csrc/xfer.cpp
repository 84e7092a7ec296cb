// The pinned staging ring of xfer.h.
#include "xfer.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace sphgpu {

hipError_t HostRing::reserve(size_t bytes) {
    const size_t want = std::min((bytes + 0xFFFF) & ~size_t(0xFFFF), kSlots * kChunk);
    if (want <= cap) return hipSuccess;
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    cap = 0;
    void* p = nullptr;
    if (hipError_t e = hipHostMalloc(&p, want); e != hipSuccess) return e;
    mem = static_cast<char*>(p);
    cap = want;
    for (hipEvent_t& e : done)
        if (!e)
            if (hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming); r != hipSuccess) return r;
    return hipSuccess;
}

void HostRing::release() {
    if (mem) (void)hipHostFree(mem);
    for (hipEvent_t& e : done) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    mem = nullptr;
    cap = 0;
}

hipError_t HostRing::to_host(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes == 0) return hipStreamSynchronize(st);
    if (hipError_t e = reserve(bytes); e != hipSuccess) return e;
    if (bytes <= kChunk) {
        hipError_t e = hipMemcpyAsync(mem, src, bytes, hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e == hipSuccess) std::memcpy(dst, mem, bytes);
        return e;
    }
    const int n = int((bytes + kChunk - 1) / kChunk), slots = std::min<int>(int(cap / kChunk), n);
    // slots >= 1: more than one chunk is asked for, so at least one is pinned
    std::atomic<int> next{0}, err{int(hipSuccess)};
    std::atomic<int> queued[kSlots];   // the chunk last queued into each slot
    for (auto& q : queued) q.store(-1);
    auto note = [&](hipError_t e) {
        if (e != hipSuccess) err.store(int(e));
        return e == hipSuccess;
    };
    auto queue = [&](int c) {
        const size_t b = size_t(c) * kChunk;
        const int s = c % slots;
        if (note(hipMemcpyAsync(mem + size_t(s) * kChunk, static_cast<const char*>(src) + b,
                                std::min(kChunk, bytes - b), hipMemcpyDeviceToHost, st)))
            note(hipEventRecord(done[s], st));
        queued[s].store(c);            // also after an error: the chunk's taker must not wait for ever
    };
    for (int c = 0; c < slots; ++c) queue(c);
    // chunks are taken in order; chunk c is queued by whoever finished chunk
    // c - slots, which was taken before it, so every wait ends
    auto work = [&] {
        for (int c; (c = next.fetch_add(1)) < n;) {
            const int s = c % slots;
            while (queued[s].load() != c) std::this_thread::yield();
            if (err.load() == int(hipSuccess) && note(hipEventSynchronize(done[s]))) {
                const size_t b = size_t(c) * kChunk;
                std::memcpy(static_cast<char*>(dst) + b, mem + size_t(s) * kChunk, std::min(kChunk, bytes - b));
            }
            if (c + slots < n) queue(c + slots);
        }
    };
    const int cpus = std::max(1, int(std::thread::hardware_concurrency()));
    const int extra = bytes < kThreadedBytes ? 0 : std::min({kMaxThreads, cpus, n}) - 1;
    std::thread helper[kMaxThreads - 1];
    for (int t = 0; t < extra; ++t) {
        try {
            helper[t] = std::thread(work);
        } catch (const std::system_error&) {
            break;                     // no thread to be had: the others do the work
        }
    }
    work();
    for (std::thread& t : helper)
        if (t.joinable()) t.join();
    const hipError_t e = hipStreamSynchronize(st);   // (after an error: no DMA may still write the ring)
    return err.load() != int(hipSuccess) ? hipError_t(err.load()) : e;
}

}  // namespace sphgpu
