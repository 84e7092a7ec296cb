// Transfers between device memory and a caller's ordinary (pageable) host
// buffer through a bounded pinned staging ring that the owning object keeps.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>

namespace sphgpu {

// A copy engine writes pinned memory at 56 GB/s, while hipMemcpy to a
// pageable buffer reaches 18 GB/s at 12 MB and 10 GB/s at 48 MB (fresh
// destination pages), and takes 85 us for 188 KB.  The ring splits a transfer
// into chunks: the DMA of the next chunks runs while the host copies the
// finished ones out.  The host copy of a large transfer is bound by the
// destination's page faults on one thread (3.4 of 3.7 ms at 48 MB), so above
// kThreadedBytes the chunks are shared by up to four threads that end before
// the call returns.  Measured (MI355X, fresh destination, engine alone): 20 KB 16 -> 9 us,
// 188 KB 85 -> 16 us, 1.4 MB 139 -> 78 us, 12 MB 777 -> 411 us, 48 MB 4.85 ->
// 1.44 ms; chunks of 1 and 4 MB were 25 and 4 % slower at 48 MB, eight
// threads no faster than four.
// To the device the runtime's own copy from a pageable buffer is as fast
// between 0.5 MB (31 us against 38) and 13 MB (383 / 406); below it costs a
// call that waits (64 KB 33 -> 10 us), and 38 MB took 1.24 ms against 1.05
// through the slots (two threads).
//
// The host's first touch of new pinned memory costs 0.4 ms a MB, several times
// the transfer.  So each object owns 1 MB at most, for small transfers, from its
// second one on (the first upload of up to 64 KB), and larger ones borrow a stage
// (the next power of two up to 2 MB, then whole chunks up to 16 MB) that the
// process's objects share: one transfer at a time has it, idle ones are kept (two at
// most, per device) while an object that has asked for one lives.  A stage is made,
// or grows, once the plain copies made instead have cost what it does: they take 32
// or 134 us for 256 KB, 75 or 420 for 1 MB, as the runtime's engine for the stream
// goes (through a stage 20 and 60), 470 for 8 MB (270), 4.9 ms for 48 MB (1.4).  (The
// first mesh of a new surfacer, MI355X, pinned at once / plain: 40^3 nodes 137 / 101
// us, 200 x 150 x 160 2.6 / 1.25 ms, 241 x 173 x 229 5.3 / 2.3 ms.)  Where no pinned
// memory is to be had, the copy is a plain one.
//
// To the host, transfers of up to a chunk are a kernel's stores to the pinned
// bytes: 15 us for 20 KB, 33 for 1 MB and 52 for 2 MB with a kernel before and the wait, where the
// runtime's copy takes 20, 39 and 57, and 60 to 130 for 20 KB in some handles' streams.
// (readback.hip; where the launch is refused, as on a stream of another device than
// the caller's or for odd addresses, the runtime's copy does it)
hipError_t launch_copy_out(void* pinned, const void* src, size_t bytes, hipStream_t st);

struct HostRing {
    static constexpr int kSlots = 8;
    static constexpr size_t kOwn = size_t(1) << 20;
    static constexpr size_t kDownOwnBytes = size_t(64) << 10;   // to the host: up to this through the own bytes
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr size_t kThreadedBytes = 2 * kChunk;
    static constexpr int kMaxThreads = 4;
    static constexpr size_t kUpOwnBytes = size_t(512) << 10;    // to the device: up to this through the own bytes,
    static constexpr size_t kUpAtOnceBytes = size_t(64) << 10;  // the first one past this without own bytes is a plain copy
    static constexpr size_t kUpSlotsBytes = size_t(32) << 20;   // from this on through the slots
    static constexpr int kUpThreads = 2;

    // device -> host; waits for everything queued on st before it, and
    // returns with `dst` complete.  veto: a pinned word that work queued before
    // the call sets; `dst` is left as it was where it is not zero
    hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t st, const int* veto = nullptr);
    // host -> device, queued on st (one past kUpOwnBytes has arrived on return); `src`
    // may be changed once it returns.  Every transfer of a ring goes through
    // one stream.
    hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t st);
    void release();

private:
    char* mem = nullptr;               // the object's own pinned bytes
    size_t cap = 0;                    // at most kOwn
    size_t used = 0;                   // bytes from `mem` on that queued transfers to the device may still read
    bool borrowed = false;             // counted among the users of the shared stages
    bool upBefore = false, downBefore = false;   // a small transfer was made without own bytes
    bool reserve(size_t bytes, hipStream_t st);
    hipError_t drain(hipStream_t st);  // waits for them
};

}  // namespace sphgpu
