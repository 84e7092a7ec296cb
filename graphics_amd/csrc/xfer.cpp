// The pinned staging ring of xfer.h.
#include "xfer.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace sphgpu {

hipError_t HostRing::drain(hipStream_t st) {
    if (!used) return hipSuccess;
    used = 0;
    return hipStreamSynchronize(st);
}

hipError_t HostRing::reserve(size_t bytes, hipStream_t st) {
    const size_t want = std::min((bytes + 0xFFFF) & ~size_t(0xFFFF), kSlots * kChunk);
    if (want <= cap) return hipSuccess;
    if (hipError_t e = drain(st); e != hipSuccess) return e;
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
    cap = used = 0;
}

namespace {
// runs `work` on this thread and up to `extra` more, to the end of all
template <class F>
void share(int extra, F&& work) {
    std::thread helper[HostRing::kMaxThreads - 1];
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
}
int helpers(size_t bytes, size_t from, int most, int chunks) {
    const int cpus = std::max(1, int(std::thread::hardware_concurrency()));
    return bytes < from ? 0 : std::min({most, cpus, chunks}) - 1;
}
}  // namespace

hipError_t HostRing::to_device(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes == 0) return hipSuccess;
    if (bytes <= kChunk) {
        // small ones one after another into the ring, until it is full
        if (hipError_t e = reserve(std::max(used + bytes, size_t(1) << 20), st); e != hipSuccess) return e;
        if (used + bytes > cap)
            if (hipError_t e = drain(st); e != hipSuccess) return e;
        char* at = mem + used;
        std::memcpy(at, src, bytes);
        used += (bytes + 255) & ~size_t(255);
        return hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, st);
    }
    if (hipError_t e = reserve(bytes, st); e != hipSuccess) return e;
    if (hipError_t e = drain(st); e != hipSuccess) return e;
    const int n = int((bytes + kChunk - 1) / kChunk), slots = std::min<int>(int(cap / kChunk), n);
    std::atomic<int> next{0}, err{int(hipSuccess)};
    std::atomic<int> queued[kSlots];   // the chunk last queued from each slot
    for (auto& q : queued) q.store(-1);
    auto note = [&](hipError_t e) {
        if (e != hipSuccess) err.store(int(e));
        return e == hipSuccess;
    };
    // chunks are taken in order; a slot's earlier chunk was taken before and is
    // marked by its taker whatever happens, so every wait ends
    auto work = [&] {
        for (int c; (c = next.fetch_add(1)) < n;) {
            const int s = c % slots;
            if (c >= slots) {
                while (queued[s].load() != c - slots) std::this_thread::yield();
                if (err.load() == int(hipSuccess)) note(hipEventSynchronize(done[s]));
            }
            if (err.load() == int(hipSuccess)) {
                const size_t b = size_t(c) * kChunk, k = std::min(kChunk, bytes - b);
                char* at = mem + size_t(s) * kChunk;
                std::memcpy(at, static_cast<const char*>(src) + b, k);
                if (note(hipMemcpyAsync(static_cast<char*>(dst) + b, at, k, hipMemcpyHostToDevice, st)))
                    note(hipEventRecord(done[s], st));
            }
            queued[s].store(c);
        }
    };
    used = cap;
    share(helpers(bytes, kUpThreadedBytes, kUpThreads, n), work);
    return hipError_t(err.load());
}

hipError_t HostRing::to_host(void* dst, const void* src, size_t bytes, hipStream_t st) {
    if (bytes == 0) return hipStreamSynchronize(st);
    if (hipError_t e = reserve(bytes, st); e != hipSuccess) return e;
    used = 0;   // (this transfer follows the queued ones on st, and ends with a wait)
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
    share(helpers(bytes, kThreadedBytes, kMaxThreads, n), work);
    const hipError_t e = hipStreamSynchronize(st);   // (after an error: no DMA may still write the ring)
    return err.load() != int(hipSuccess) ? hipError_t(err.load()) : e;
}

}  // namespace sphgpu
