// The pinned staging ring of xfer.h.
#include "xfer.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace sphgpu {

namespace {
struct Stage {
    int device = 0;
    char* mem = nullptr;
    size_t cap = 0;
    hipEvent_t done[HostRing::kSlots] = {};
};
struct Stages {
    std::mutex lock;
    std::vector<Stage*> idle;
    int users = 0;
    double rent = 0.0;   // us that plain copies since the last new stage took longer than through one
};
// (never destroyed: an object of static duration may release its ring late)
Stages& stages() {
    alignas(Stages) static char place[sizeof(Stages)];
    static Stages* s = new (place) Stages;
    return *s;
}
constexpr size_t kMaxIdle = 2;

void destroy(Stage* s) {
    if (s->mem) (void)hipHostFree(s->mem);
    for (hipEvent_t e : s->done)
        if (e) (void)hipEventDestroy(e);
    delete s;
}

// us that a stage of `bytes` costs when it is new (its allocation and the host's first
// touch: 0.38 a KB, or next to nothing where the process gets memory that it had
// before; half of it), and that a transfer through one takes
double price(size_t bytes) { return 25.0 + 0.19 / 1024.0 * double(bytes); }
double staged(size_t bytes, bool up) {
    return 10.0 + (up ? 0.027 : bytes <= HostRing::kChunk ? 0.05 : 0.033) / 1024.0 * double(bytes);
}

// a plain copy of a transfer that a stage would take: what it takes longer counts
// towards a stage
template <class F>
hipError_t rented(size_t bytes, bool up, hipStream_t st, F&& copy) {
    if (const hipError_t e = hipStreamSynchronize(st); e != hipSuccess) return e;   // (not the wait for other work)
    const auto from = std::chrono::steady_clock::now();
    const hipError_t e = copy();
    const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - from).count();
    Stages& all = stages();
    std::lock_guard<std::mutex> l(all.lock);
    all.rent += std::max(0.0, us - staged(bytes, up));
    return e;
}

// a stage for a transfer of `bytes` on st; nullptr where none is idle and the plain
// copies so far, with what this one would (`saves`), have not cost what a new one
// does, or there is none to be had
Stage* borrow(size_t bytes, double saves, hipStream_t st, bool& counted) {
    hipDevice_t device = 0;
    if (hipStreamGetDevice(st, &device) != hipSuccess) return nullptr;
    // up to a chunk the next power of two: a process that reads 100 KB does not
    // touch 2 MB for it, and one that reads more each time touches twice that at most
    size_t want = std::min((bytes + HostRing::kChunk - 1) / HostRing::kChunk, size_t(HostRing::kSlots)) * HostRing::kChunk;
    if (bytes <= HostRing::kChunk)
        for (want = 2 * HostRing::kDownOwnBytes; want < bytes;) want *= 2;
    Stage* s = nullptr;
    Stages& all = stages();
    {
        std::lock_guard<std::mutex> l(all.lock);
        if (!counted) ++all.users;
        counted = true;
        for (Stage* o : all.idle)
            if (o->device == device && (!s || o->cap > s->cap)) s = o;
        if (!s || s->cap < want) {
            if (all.rent + saves >= price(want)) {
                all.rent = 0.0;
            } else if (s && s->cap >= 2 * HostRing::kChunk) {
                want = s->cap;         // (two chunks in turn will do)
            } else {
                return nullptr;
            }
        }
        if (s) all.idle.erase(std::find(all.idle.begin(), all.idle.end(), s));
    }
    hipError_t err = hipSuccess;
    if (!s) {
        s = new (std::nothrow) Stage;
        if (!s) return nullptr;
        s->device = device;
        int current = 0;
        err = hipGetDevice(&current);
        if (err == hipSuccess && current != device) err = hipSetDevice(device);   // (an event is its device's)
        for (hipEvent_t& e : s->done)
            if (err == hipSuccess) err = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        if (current != device) (void)hipSetDevice(current);
    }
    if (err == hipSuccess && s->cap < want) {
        if (s->mem) (void)hipHostFree(s->mem);
        s->mem = nullptr;
        s->cap = 0;
        void* p = nullptr;
        if ((err = hipHostMalloc(&p, want)) == hipSuccess) {
            s->mem = static_cast<char*>(p);
            s->cap = want;
        }
    }
    if (err == hipSuccess) return s;
    (void)hipGetLastError();           // (the transfer goes without)
    destroy(s);
    return nullptr;
}

void give_back(Stage* s) {
    Stages& all = stages();
    {
        std::lock_guard<std::mutex> l(all.lock);
        const size_t same = std::count_if(all.idle.begin(), all.idle.end(), [s](Stage* o) { return o->device == s->device; });
        if (all.users > 0 && same < kMaxIdle) {
            try {
                all.idle.push_back(s);
                return;
            } catch (const std::bad_alloc&) {
            }
        }
    }
    destroy(s);
}
}  // namespace

hipError_t HostRing::drain(hipStream_t st) {
    if (!used) return hipSuccess;
    used = 0;
    return hipStreamSynchronize(st);
}

bool HostRing::reserve(size_t bytes, hipStream_t st) {
    const size_t want = std::min((bytes + 0xFFFF) & ~size_t(0xFFFF), kOwn);
    if (want <= cap) return true;
    if (drain(st) != hipSuccess) return false;
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    cap = 0;
    void* p = nullptr;
    if (hipHostMalloc(&p, want) != hipSuccess) {
        (void)hipGetLastError();       // (the transfer goes without)
        return false;
    }
    mem = static_cast<char*>(p);
    cap = want;
    return true;
}

void HostRing::release() {
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    cap = used = 0;
    if (!borrowed) return;
    borrowed = false;
    std::vector<Stage*> last;
    Stages& all = stages();
    {
        std::lock_guard<std::mutex> l(all.lock);
        if (--all.users == 0) {
            last.swap(all.idle);
            all.rent = 0.0;
        }
    }
    for (Stage* s : last) destroy(s);
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
    auto plain = [&] {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    };
    if (bytes <= kUpOwnBytes) {
        // small ones one after another into the ring, until it is full
        if (used + bytes > cap) {
            if (hipError_t e = drain(st); e != hipSuccess) return e;
            if (bytes > cap && bytes > kUpAtOnceBytes && !upBefore) {
                upBefore = true;
                return plain();
            }
            if (!reserve(2 * bytes, st)) return plain();
        }
        char* at = mem + used;
        std::memcpy(at, src, bytes);
        used += (bytes + 255) & ~size_t(255);
        return hipMemcpyAsync(dst, at, bytes, hipMemcpyHostToDevice, st);
    }
    if (bytes < kUpSlotsBytes) return plain();
    Stage* const stage = borrow(bytes, 0.0, st, borrowed);
    if (!stage) return rented(bytes, true, st, plain);
    char* const mem = stage->mem;
    hipEvent_t* const done = stage->done;
    const int n = int((bytes + kChunk - 1) / kChunk), slots = std::min<int>(int(stage->cap / kChunk), n);
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
    share(helpers(bytes, 0, kUpThreads, n), work);
    const hipError_t e = hipStreamSynchronize(st);   // (the stage is another transfer's next)
    give_back(stage);
    return err.load() != int(hipSuccess) ? hipError_t(err.load()) : e;
}

hipError_t HostRing::to_host(void* dst, const void* src, size_t bytes, hipStream_t st, const int* veto) {
    if (bytes == 0) return hipStreamSynchronize(st);
    // (asked for after the first bytes have arrived: the word was set before them)
    auto wanted = [veto] { return !veto || __atomic_load_n(veto, __ATOMIC_ACQUIRE) == 0; };
    auto plain = [&] {
        hipError_t e = veto ? hipStreamSynchronize(st) : hipSuccess;
        if (e != hipSuccess || !wanted()) return e;
        e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    };
    auto through = [&](char* at) {
        hipError_t e = launch_copy_out(at, src, bytes, st);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            e = hipMemcpyAsync(at, src, bytes, hipMemcpyDeviceToHost, st);
        }
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e == hipSuccess && wanted()) std::memcpy(dst, at, bytes);
        return e;
    };
    if (bytes <= kDownOwnBytes) {
        if (bytes > cap && !downBefore) {
            downBefore = true;
            return plain();
        }
        if (!reserve(bytes, st)) return plain();
        used = 0;   // (this transfer follows the queued ones on st, and ends with a wait)
        return through(mem);
    }
    // (a plain copy of 32 MB or more is bound by the destination's page faults on one
    // thread: a stage pays at the first)
    Stage* const stage = borrow(bytes, bytes < kUpSlotsBytes ? 0.0 : 0.07 / 1024.0 * double(bytes), st, borrowed);
    if (!stage) return rented(bytes, false, st, plain);
    if (bytes <= kChunk) {
        const hipError_t e = through(stage->mem);
        give_back(stage);
        return e;
    }
    char* const mem = stage->mem;
    hipEvent_t* const done = stage->done;
    const int n = int((bytes + kChunk - 1) / kChunk), slots = std::min<int>(int(stage->cap / kChunk), n);
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
            if (err.load() == int(hipSuccess) && note(hipEventSynchronize(done[s])) && wanted()) {
                const size_t b = size_t(c) * kChunk;
                std::memcpy(static_cast<char*>(dst) + b, mem + size_t(s) * kChunk, std::min(kChunk, bytes - b));
            }
            if (c + slots < n) queue(c + slots);
        }
    };
    share(helpers(bytes, kThreadedBytes, kMaxThreads, n), work);
    const hipError_t e = hipStreamSynchronize(st);   // (after an error: no DMA may still write the stage)
    give_back(stage);
    return err.load() != int(hipSuccess) ? hipError_t(err.load()) : e;
}

}  // namespace sphgpu
