// Fluid fields in ascending original id, put in order on the device.
#include "sph_common.h"
#include "xfer.h"

#include <algorithm>

namespace sphgpu {

namespace {

__device__ __forceinline__ int live_id(const Dev& D, int i) {
    const int tile = i / TILE;
    return (i - tile * TILE) < D.tileValid[tile] ? D.id[i] : -1;
}

__global__ __launch_bounds__(256) void k_live_flags(Dev D, uint32_t* __restrict__ flags) {
    const int id = live_id(D, blockIdx.x * 256 + threadIdx.x);
    if (id >= 0) flags[id] = 1u;
}

// One thread per slot writes its particle's values to the particle's place:
// its id while no particle was ever removed (rank null), else its rank among
// the live ids.  Bound by memory: 16 + 4 B read and 12 B written per particle
// for a vector field, the writes 12 B runs that neighbouring slots (which lie
// close in id too) fill into whole lines in the L2.  It replaces a host sort
// of (id, slot) pairs per call; with the transfer through the pinned ring a
// vector field of 4,000,752 particles takes 1.4 ms instead of 158 ms, of
// 117,364 particles 0.10 instead of 3.85 ms.
template <int COMP, class T>
__global__ __launch_bounds__(256) void k_field_by_id(Dev D, const T* __restrict__ src,
                                                     const uint32_t* __restrict__ rank, float* __restrict__ out,
                                                     int* __restrict__ removed) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) *removed = D.counters[C_REMOVED];
    const int id = live_id(D, i);
    if (id < 0) return;
    const size_t k = rank ? rank[id] : (uint32_t)id;
    if constexpr (COMP == 1 && sizeof(T) == 4) {
        out[k] = src[i];
    } else {
        const float4 q = src[i];
        if constexpr (COMP == 1) {
            out[k] = q.w;              // the phase, carried with the position
        } else {
            out[3 * k] = q.x;
            out[3 * k + 1] = q.y;
            out[3 * k + 2] = q.z;
        }
    }
}

// the ids themselves (64-bit); without a rank only the removal count is read
__global__ __launch_bounds__(256) void k_ids_by_rank(Dev D, const uint32_t* __restrict__ rank,
                                                     long long* __restrict__ out, int* __restrict__ removed) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i == 0) *removed = D.counters[C_REMOVED];
    const int id = rank ? live_id(D, i) : -1;
    if (id >= 0) out[rank[id]] = id;
}

// src to pinned host memory: n words, and the bytes past them.  Bound by the link:
// 20 KB takes 15 us with the wait and 2 MB 52 (40 GB/s), the runtime's copy 20 and 57,
// and 60 to 130 for 20 KB in some handles' streams
template <class T>
__global__ __launch_bounds__(256) void k_copy_out(const T* __restrict__ src, T* __restrict__ out, size_t n,
                                                  const char* __restrict__ tail, char* __restrict__ outTail, int rest) {
    for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += gridDim.x * 256ull) out[i] = src[i];
    if (blockIdx.x == 0 && (int)threadIdx.x < rest) outTail[threadIdx.x] = tail[threadIdx.x];
}

}  // namespace

hipError_t launch_copy_out(void* pinned, const void* src, size_t bytes, hipStream_t st) {
    const auto copy = [&](auto word) {
        using T = decltype(word);
        size_t n = bytes / sizeof(T), done = n * sizeof(T);
        const T* from = static_cast<const T*>(src);
        T* out = static_cast<T*>(pinned);
        const char* tail = static_cast<const char*>(src) + done;
        char* outTail = static_cast<char*>(pinned) + done;
        int rest = int(bytes - done);
        void* args[] = {&from, &out, &n, &tail, &outTail, &rest};
        const unsigned blocks = unsigned(std::clamp<size_t>((n + 255) / 256, 1, 256));
        return hipLaunchKernel(reinterpret_cast<const void*>(&k_copy_out<T>), dim3(blocks), dim3(256), args, 0, st);
    };
    const uintptr_t at = reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(pinned);
    if (at % 16 == 0) return copy(make_uint4(0, 0, 0, 0));
    return at % 4 == 0 ? copy(0u) : hipErrorInvalidValue;
}

void launch_live_ranks(const Dev& D, uint32_t* rank, int ids, uint32_t* tmp, hipStream_t st) {
    launch_fill_i32(reinterpret_cast<int*>(rank), 0, ids + 1, st);
    if (D.npad > 0) hipLaunchKernelGGL(k_live_flags, dim3(D.npad / TILE), dim3(256), 0, st, D, rank);
    exclusive_scan_u32(rank, ids + 1, tmp, st);
}

void launch_field_by_id(const Dev& D, const float4* src, int comp, const uint32_t* rank, float* out, int* removed,
                        hipStream_t st) {
    const dim3 g(D.npad / TILE), b(256);
    if (comp == 3) hipLaunchKernelGGL((k_field_by_id<3, float4>), g, b, 0, st, D, src, rank, out, removed);
    else hipLaunchKernelGGL((k_field_by_id<1, float4>), g, b, 0, st, D, src, rank, out, removed);
}

void launch_field_by_id(const Dev& D, const float* src, const uint32_t* rank, float* out, int* removed,
                        hipStream_t st) {
    hipLaunchKernelGGL((k_field_by_id<1, float>), dim3(D.npad / TILE), dim3(256), 0, st, D, src, rank, out, removed);
}

void launch_ids_by_rank(const Dev& D, const uint32_t* rank, long long* out, int* removed, hipStream_t st) {
    hipLaunchKernelGGL(k_ids_by_rank, dim3(rank ? D.npad / TILE : 1), dim3(256), 0, st, D, rank, out, removed);
}

}  // namespace sphgpu
