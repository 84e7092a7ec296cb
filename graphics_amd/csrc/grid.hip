// Uniform-grid neighbour search on the GPU (the reference's SphBase::gridSetup
// + neighbourSearch, SphBase.cpp:849-1089, re-designed): cell keys -> radix
// sort -> scene layout padded to whole tiles -> SoA reorder -> per-cell
// [start,end) tables -> ELL neighbour lists built from 9 contiguous x-runs of
// three cells each.  The pair test keeps the reference's FP32 rounding so
// that the neighbour sets are bit-identical.
#include "sph_common.h"

#include <type_traits>

namespace sphgpu {

namespace {

__device__ __forceinline__ bool slot_valid(const Dev& D, int i, int* scene) {
    int tile = i / TILE;
    *scene = D.tileScene[tile];
    return (i - tile * TILE) < D.tileValid[tile];
}


__global__ __launch_bounds__(256) void k_fluid_keys(Dev D, uint32_t* keys, uint32_t* vals) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= D.npad) return;
    uint32_t k = KEY_INVALID;
    if (D.id[i] >= 0) {
        float4 p = D.x[i];
        int s = D.tileScene[i / TILE];
        const SceneGrid G = D.grids[s];
        int cx, cy, cz;
        cell_of(G, p, cx, cy, cz);
        k = key_of(G, D.rowRank, cx, cy, cz);
    }
    keys[i] = k;
    vals[i] = (uint32_t)i;
}

__global__ __launch_bounds__(256) void k_scene_bounds(Dev D, const uint32_t* __restrict__ sk, int n) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t k = sk[i];
    if (k == KEY_INVALID) return;
    int s = scene_of_key(k, D.sceneKeyBase, D.nscenes);
    bool first = (i == 0) || sk[i - 1] == KEY_INVALID ||
                 scene_of_key(sk[i - 1], D.sceneKeyBase, D.nscenes) != s;
    bool last = (i == n - 1) || sk[i + 1] == KEY_INVALID ||
                scene_of_key(sk[i + 1], D.sceneKeyBase, D.nscenes) != s;
    if (first) D.sceneStart[s] = i;
    if (last) D.sceneCount[s] = i + 1;   // end for now; the layout kernel turns it into a count
}

// single thread: counts, padded starts, tile tables.  hostOut (mapped to the
// host by the caller via a device buffer) receives [npad_new, n_live].
__global__ void k_scene_layout(Dev D, int* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int pad = 0, live = 0;
    for (int s = 0; s < D.nscenes; ++s) {
        int st = D.sceneStart[s], en = D.sceneCount[s];
        int c = (en > st) ? en - st : 0;
        if (st < 0) c = 0;
        D.sceneCount[s] = c;
        D.scenePadStart[s] = pad;
        pad += (c + TILE - 1) / TILE * TILE;
        live += c;
    }
    D.scenePadStart[D.nscenes] = pad;
    out[0] = pad;
    out[1] = live;
}

__global__ __launch_bounds__(256) void k_tiles(Dev D, int numTiles) {
    int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= numTiles) return;
    int slot = t * TILE;
    int s = 0;
    // largest s with padStart[s] <= slot
    int lo = 0, hi = D.nscenes - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (D.scenePadStart[mid] <= slot) lo = mid; else hi = mid - 1;
    }
    s = lo;
    int valid = 0;
    if (slot < D.scenePadStart[D.nscenes]) {
        int local = slot - D.scenePadStart[s];
        valid = min(max(D.sceneCount[s] - local, 0), TILE);
    }
    D.tileScene[t] = s;
    D.tileValid[t] = valid;
}

// scatter sorted rank r to its padded slot; also marks padding slots
__global__ __launch_bounds__(256) void k_reorder(Dev D, const uint32_t* __restrict__ sk,
                                               const uint32_t* __restrict__ sv, int n) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    uint32_t k = sk[r];
    if (k == KEY_INVALID) return;
    int s = scene_of_key(k, D.sceneKeyBase, D.nscenes);
    int p = r - D.sceneStart[s] + D.scenePadStart[s];
    int src = (int)sv[r];
    D.x2[p] = D.x[src];
    D.v2[p] = D.v[src];
    D.id2[p] = D.id[src];
    D.ksum2[p] = D.ksum[src];
    D.kvsum2[p] = D.kvsum[src];
    D.key2[p] = k;
}

__global__ __launch_bounds__(256) void k_mark_padding(Dev D, int limit) {
    int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= limit) return;
    int tile = t / TILE;
    if ((t - tile * TILE) >= D.tileValid[tile]) {
        D.id2[t] = -1;
        D.key2[t] = KEY_INVALID;
    }
}

__global__ __launch_bounds__(256) void k_cell_reset(const uint32_t* __restrict__ keys, int n,
                                                  int2* __restrict__ table) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t k = keys[i];
    if (k == KEY_INVALID) return;
    if (i == 0 || keys[i - 1] != k) table[k] = make_int2(0, 0);
}

__global__ __launch_bounds__(256) void k_cell_build(const uint32_t* __restrict__ keys, int n,
                                                  int2* __restrict__ table) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    uint32_t k = keys[i];
    if (k == KEY_INVALID) return;
    if (i == 0 || keys[i - 1] != k) table[k].x = i;
    if (i == n - 1 || keys[i + 1] != k) table[k].y = i + 1;
}


// ---- counting search --------------------------------------------------------
// The order of the radix search (by cell key, stable in the old slot order)
// without its three digit passes: particles are counted per cell, the counts
// scanned into the cell table, each particle dropped into its cell's segment
// in arrival order, and its place in the segment found by counting the
// segment's smaller slot indices (a cell holds about eight particles; the
// list builder reads the particles of 27 cells per particle, so however many
// a cell holds, this is the smaller part).  Atomics only decide the arrival
// order, which the last step sorts out, so the result is the same every run.
// Four launches on a small grid, six on others, for about twenty.  Bound by
// launches and latency on a small scene, by the 104 B a particle of the reorder
// on a large one.  Kernels of one search without the list builder, MI355X: 23
// us for 15,625 particles (75 us by radix sort), 85 us for 1,000,000 (160),
// 190 us for 4,000,752 (330).
constexpr int SCAN1_THREADS = 1024;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(v, off, 64);
        if (lane >= off) v += y;
    }
    return v;
}

// exclusive prefix of v over a block of W waves; *total = the block's sum
template <int W>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* lds, uint32_t* total) {
    const int w = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(v);
    if ((threadIdx.x & 63) == 63) lds[w] = x;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const uint32_t s = lds[k];
        if (k < w) pre += s;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

// arrival rank of each lane's particle in its cell.  Neighbouring slots mostly
// share a cell, so one lane adds for each run of equal keys in the wave (every
// lane of the wave calls it; key KEY_INVALID: none).
__device__ __forceinline__ uint32_t cell_arrival(uint32_t key, uint32_t* __restrict__ cnt) {
    const int lane = lane_id();
    const uint32_t prev = __shfl_up(key, 1, 64);
    const bool head = lane == 0 || prev != key;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = heads & ((2ull << lane) - 1ull), after = heads & ~((2ull << lane) - 1ull);
    const int first = 63 - __clzll((long long)upto);
    uint32_t base = 0;
    if (head && key != KEY_INVALID) {
        const int next = after ? __ffsll((long long)after) - 1 : 64;
        base = atomicAdd(&cnt[key], (uint32_t)(next - lane));
    }
    return __shfl(base, first, 64) + (uint32_t)(lane - first);
}

__global__ __launch_bounds__(256) void k_count_fluid(Dev D, uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ arrival) {
    const int tile = blockIdx.x, i = tile * TILE + threadIdx.x;   // npad is a multiple of TILE
    uint32_t k = KEY_INVALID;
    if (D.id[i] >= 0) {
        const float4 p = D.x[i];
        const SceneGrid G = D.grids[D.tileScene[tile]];
        int cx, cy, cz;
        cell_of(G, p, cx, cy, cz);
        k = key_of(G, D.rowRank, cx, cy, cz);
    }
    keys[i] = k;
    arrival[i] = cell_arrival(k, D.cellCnt);
    const int live = __syncthreads_count(k != KEY_INVALID);
    if (threadIdx.x == 0) D.tileLive[tile] = live;
}

__global__ __launch_bounds__(256) void k_count_boundary(Dev D, const float4* __restrict__ xs,
                                                        const int* __restrict__ scene, uint32_t* __restrict__ keys,
                                                        uint32_t* __restrict__ arrival) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    uint32_t k = KEY_INVALID;
    if (i < D.nb) {
        const SceneGrid G = D.grids[scene[i]];
        int cx, cy, cz;
        cell_of(G, xs[i], cx, cy, cz);
        k = key_of(G, D.rowRank, cx, cy, cz);
    }
    const uint32_t a = cell_arrival(k, D.cellCnt);
    if (i < D.nb) {
        keys[i] = k;
        arrival[i] = a;
    }
}

__global__ __launch_bounds__(256) void k_cell_sums(Dev D) {
    __shared__ uint32_t lds[4];
    const uint32_t k0 = blockIdx.x * (uint32_t)SEARCH_KEYS + threadIdx.x;
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < SEARCH_KEYS / 256; ++q)
        if (k0 + q * 256 < D.totalKeys) s += D.cellCnt[k0 + q * 256];
    uint32_t tot;
    block_scan<4>(s, lds, &tot);
    if (threadIdx.x == 0) D.cellSums[blockIdx.x] = tot;
}

// scene counts, padded starts and tile tables, by one block; `total` = live particles
__device__ __forceinline__ void layout_block(const Dev& D, uint32_t total, int* __restrict__ out, uint32_t* lds) {
    const int tid = threadIdx.x, ns = D.nscenes, tiles = D.npad / TILE, all = D.ncap / TILE;
    __shared__ int sceneLive[MAX_SCENES];
    if (ns == 1) {
        // (no value read back from memory)
        const int pad = ((int)total + TILE - 1) / TILE * TILE;
        if (tid == 0) {
            D.sceneCount[0] = (int)total;
            D.sceneStart[0] = 0;
            D.sceneShift[0] = 0;
            D.scenePadStart[0] = 0;
            D.scenePadStart[1] = pad;
            out[0] = pad;
            out[1] = (int)total;
        }
        for (int t = tid; t < all; t += SCAN1_THREADS) {
            D.tileScene[t] = 0;
            D.tileValid[t] = min(max((int)total - t * TILE, 0), TILE);
        }
    } else {
        for (int s = tid; s < ns; s += SCAN1_THREADS) sceneLive[s] = 0;
        __syncthreads();
        // tiles of one scene lie together: one atomic per wave where they do
        for (int t0 = 0; t0 < tiles; t0 += SCAN1_THREADS) {
            const int t = t0 + tid;
            const int s = t < tiles ? D.tileScene[t] : -1;
            int c = t < tiles ? D.tileLive[t] : 0;
            const int s0 = __builtin_amdgcn_readfirstlane(s);
            if (__ballot(s != s0) == 0) {
                if (s0 < 0) continue;          // past the last tile (uniform in the wave)
                for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
                if ((tid & 63) == 0) atomicAdd(&sceneLive[s0], c);
            } else if (s >= 0) {
                atomicAdd(&sceneLive[s], c);
            }
        }
        __syncthreads();
        uint32_t start = 0, pad = 0;
        for (int s0 = 0; s0 < ns; s0 += SCAN1_THREADS) {
            const int s = s0 + tid;
            const uint32_t c = s < ns ? (uint32_t)sceneLive[s] : 0u;
            const uint32_t p = (c + TILE - 1) / TILE * TILE;
            uint32_t ct, pt;
            const uint32_t c0 = block_scan<SCAN1_THREADS / 64>(c, lds, &ct);
            const uint32_t p0 = block_scan<SCAN1_THREADS / 64>(p, lds, &pt);
            if (s < ns) {
                D.sceneCount[s] = (int)c;
                D.sceneStart[s] = (int)(start + c0);
                D.scenePadStart[s] = (int)(pad + p0);
                D.sceneShift[s] = (int)(pad + p0) - (int)(start + c0);
            }
            start += ct;
            pad += pt;
        }
        if (tid == 0) {
            D.scenePadStart[ns] = (int)pad;
            out[0] = (int)pad;
            out[1] = (int)total;
        }
        __syncthreads();
        for (int t = tid; t < all; t += SCAN1_THREADS) {
            const int slot = t * TILE;
            int lo = 0, hi = ns - 1;
            while (lo < hi) {                  // largest s with padStart[s] <= slot
                const int mid = (lo + hi + 1) >> 1;
                if (D.scenePadStart[mid] <= slot) lo = mid; else hi = mid - 1;
            }
            D.tileScene[t] = lo;
            D.tileValid[t] = slot < (int)pad ? min(max(sceneLive[lo] - (slot - D.scenePadStart[lo]), 0), TILE) : 0;
        }
    }
}

// Cell table entries of the n keys from k0 on, whose counts are in LDS, by a
// block of W waves; `first` = rank of the first key's first particle.  Each
// thread scans `per` consecutive counts in LDS (per odd: no bank conflicts);
// the table is written, and the counts cleared for the next search, key by
// lane, so both stores are whole lines (eight keys a thread straight from
// registers took 70 us for 5.3 million keys, this way 18).
template <int W>
__device__ __forceinline__ uint32_t scan_counts(uint32_t* __restrict__ c, int n, int per, uint32_t first,
                                                uint32_t* lds) {
    const int t0 = (int)threadIdx.x * per, t1 = min(t0 + per, n);
    uint32_t s = 0, tot;
    for (int k = t0; k < t1; ++k) s += c[k];
    uint32_t pre = first + block_scan<W>(s, lds, &tot);
    for (int k = t0; k < t1; ++k) {
        const uint32_t v = c[k];
        c[k] = pre;
        pre += v;
    }
    if (threadIdx.x == 0) c[n] = first + tot;
    __syncthreads();
    return tot;
}
template <bool FLUID, int W, bool CLEAR = true>
__device__ __forceinline__ void write_runs(const Dev& D, uint32_t k0, const uint32_t* __restrict__ c, int n,
                                           int2* __restrict__ table) {
    int s = -1, shift = 0;
    const bool scenes = FLUID && D.nscenes > 1;
    for (int q = threadIdx.x; q < n; q += 64 * W) {
        const uint32_t k = k0 + q;
        if (scenes) {
            if (s < 0) s = scene_of_key(k, D.sceneKeyBase, D.nscenes);
            while (k >= D.sceneKeyBase[s + 1]) ++s;
            shift = D.sceneShift[s];
        }
        table[k] = make_int2((int)c[q] + shift, (int)c[q + 1] + shift);
        if (CLEAR) D.cellCnt[k] = 0;
    }
}

// several scenes on at most SEARCH_KEYS_ONE keys: scan, layout and cell table in one block
__global__ __launch_bounds__(SCAN1_THREADS) void k_search_one(Dev D, int2* __restrict__ table, int* __restrict__ out) {
    constexpr int W = SCAN1_THREADS / 64;
    __shared__ uint32_t lds[W];
    __shared__ uint32_t c[SEARCH_KEYS_ONE + 1];
    const int n = (int)D.totalKeys, per = ((n + SCAN1_THREADS - 1) / SCAN1_THREADS) | 1;
    for (int k = threadIdx.x; k < n; k += SCAN1_THREADS) c[k] = D.cellCnt[k];
    __syncthreads();
    const uint32_t total = scan_counts<W>(c, n, per, 0, lds);
    layout_block(D, total, out, lds);
    __syncthreads();
    write_runs<true, W>(D, 0, c, n, table);
}

// The same for one scene, and for the boundary, by several blocks: each adds up the counts before its
// part for itself (the counts are in the cache, and a block that waited for the
// others' sums would take another launch); k_place clears the counts.  For
// 28,000 keys one block takes 11 us, mostly to write the table; parts of 2,048
// take 5.1.
constexpr int SEARCH_PART = 2048;
template <bool FLUID>
__global__ __launch_bounds__(SCAN1_THREADS) void k_search_part(Dev D, int2* __restrict__ table, int* __restrict__ out) {
    constexpr int W = SCAN1_THREADS / 64;
    __shared__ uint32_t lds[W];
    __shared__ uint32_t c[SEARCH_PART + 1];
    const int k0 = (int)blockIdx.x * SEARCH_PART, n = min(SEARCH_PART, (int)D.totalKeys - k0);
    for (int k = threadIdx.x; k < n; k += SCAN1_THREADS) c[k] = D.cellCnt[k0 + k];
    uint32_t s = 0, before;
    for (int k = threadIdx.x; k < k0; k += 8 * SCAN1_THREADS) {
        uint32_t v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = k + q * SCAN1_THREADS < k0 ? D.cellCnt[k + q * SCAN1_THREADS] : 0u;
#pragma unroll
        for (int q = 0; q < 8; ++q) s += v[q];
    }
    block_scan<W>(s, lds, &before);   // (its barriers also complete the staging of c)
    const uint32_t own = scan_counts<W>(c, n, (SEARCH_PART / SCAN1_THREADS) | 1, before, lds);
    write_runs<FLUID, W, false>(D, (uint32_t)k0, c, n, table);
    if (FLUID && blockIdx.x == gridDim.x - 1) layout_block(D, before + own, out, lds);
}

// larger grids: the block sums scanned (in place) by one block, which also lays out the scenes
template <bool FLUID>
__global__ __launch_bounds__(SCAN1_THREADS) void k_search_mid(Dev D, int blocks, int* __restrict__ out) {
    __shared__ uint32_t lds[SCAN1_THREADS / 64];
    uint32_t run = 0;
    for (int b0 = 0; b0 < blocks; b0 += SCAN1_THREADS) {
        const int b = b0 + (int)threadIdx.x;
        const uint32_t v = b < blocks ? D.cellSums[b] : 0u;
        uint32_t tot;
        const uint32_t pre = block_scan<SCAN1_THREADS / 64>(v, lds, &tot);
        if (b < blocks) D.cellSums[b] = run + pre;
        run += tot;
    }
    if (FLUID) layout_block(D, run, out, lds);
}

template <bool FLUID>
__global__ __launch_bounds__(256) void k_cell_runs(Dev D, int2* __restrict__ table) {
    __shared__ uint32_t lds[4];
    __shared__ uint32_t c[SEARCH_KEYS + 1];
    const uint32_t k0 = blockIdx.x * (uint32_t)SEARCH_KEYS;
    const int n = (int)min((uint32_t)SEARCH_KEYS, D.totalKeys - k0);
#pragma unroll
    for (int q = 0; q < SEARCH_KEYS / 256; ++q) {
        const int k = q * 256 + (int)threadIdx.x;
        if (k < n) c[k] = D.cellCnt[k0 + k];
    }
    __syncthreads();
    scan_counts<4>(c, n, SEARCH_KEYS / 256, D.cellSums[blockIdx.x], lds);
    write_runs<FLUID, 4>(D, k0, c, n, table);
}

__global__ __launch_bounds__(256) void k_place(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ arrival,
                                               const int2* __restrict__ table, int n, uint32_t* __restrict__ order,
                                               uint32_t* __restrict__ clear) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = keys[i];
    if (k == KEY_INVALID) return;
    order[(uint32_t)table[k].x + arrival[i]] = (uint32_t)i;
    if (clear) clear[k] = 0;
}

// place of the particle order[t] in its cell's segment: the segment's smaller indices
__device__ __forceinline__ int slot_in_cell(const uint32_t* __restrict__ order, uint32_t i, int2 seg) {
    int p = seg.x;
    for (int u = seg.x; u < seg.y; ++u) p += order[u] < i;
    return p;
}

__global__ __launch_bounds__(256) void k_reorder_cells(Dev D, const uint32_t* __restrict__ keys,
                                                       const uint32_t* __restrict__ order) {
    const int tile = blockIdx.x, t = tile * TILE + threadIdx.x;
    if ((int)threadIdx.x >= D.tileValid[tile]) {
        D.id2[t] = -1;                         // padding
        return;
    }
    const uint32_t i = order[t];
    const int p = slot_in_cell(order, i, D.cellF[keys[i]]);
    D.x2[p] = D.x[i];
    D.v2[p] = D.v[i];
    D.id2[p] = D.id[i];
    D.ksum2[p] = D.ksum[i];
    D.kvsum2[p] = D.kvsum[i];
}

__global__ __launch_bounds__(256) void k_order_boundary(Dev D, const uint32_t* __restrict__ keys,
                                                        const uint32_t* __restrict__ order, uint32_t* __restrict__ sk,
                                                        uint32_t* __restrict__ sv) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= D.nb) return;
    const uint32_t i = order[t], k = keys[i];
    const int p = slot_in_cell(order, i, D.cellB[k]);
    sk[p] = k;
    sv[p] = i;
}

// Lists are built in LDS, one column per thread, and written out group by
// group (16 bytes per particle), so each store instruction of a wave writes
// whole cache lines.  A tile whose particles span at most NB16_ROWS own rows,
// and whose row runs each fit NB16_OFF_BITS of offset, gets packed 16-bit
// lists (8 entries per group); any other tile gets 32-bit lists (4 per
// group).  NB_STAGE_GROUPS groups are staged in LDS and the rest written to
// global memory directly (6 or 8 groups: LDS per block against blocks per
// CU, chosen by the autotuner).  Both forms hold the same entries in the
// same order.
// Bound by the candidate loop (about 216 candidates a particle, 16 B of L1
// return and fifteen VALU operations each); small scenes have a builder of
// their own (k_neighbours_quarter).  The loop's short form, the slot
// bounds from the rows' end lanes only and flushing without barriers took it
// from 887 to 740 us at 4,000,752 particles, 234 to 176 us at 1,000,000 and
// 100 to 77 us at 328,233 (six groups).  Not kept: the next group's loads
// issued before this group's tests (4 % slower at 4M), the nine rows in one
// rolled loop (25 % slower).
template <int NB_STAGE_GROUPS>
__global__ __launch_bounds__(256) void k_neighbours(Dev D) {
    __shared__ int4 stage[NB_STAGE_GROUPS][256];
    __shared__ int sBase[2 * 32], sEnd[2 * 32];
    __shared__ int sRow[256];
    __shared__ int sWave[4];
    __shared__ int sOverflow;
    __shared__ int sWin[33];   // window offset of each fluid slot - (slot << NB16_OFF_BITS); [32] = size
    const int tid = threadIdx.x;
    const int tile = tile_of_block(D.tileMap);
    const int i = tile * 256 + tid;
    int scene = 0;
    const bool act = i < D.npad && slot_valid(D, i, &scene);
    int* st = reinterpret_cast<int*>(&stage[0][0]);
    uint16_t* st16 = reinterpret_cast<uint16_t*>(&stage[0][0]);
    const int stride = D.ncap;
    int cx = 0, cy = 0, cz = 0;
    float4 pa = make_float4(0.f, 0.f, 0.f, 0.f);
    SceneGrid G{};
    if (act) {
        G = D.grids[scene];
        pa = D.x[i];
        cell_of(G, pa, cx, cy, cz);
    }
    // ordinal of the particle's own row among the tile's rows: the valid
    // slots are a prefix of the tile in key order, so one row's particles
    // are contiguous
    const int row = act ? cz * G.ny + cy : -1;
    sRow[tid] = row;
    if (tid < 64) {
        sBase[tid] = INT_MAX;
        sEnd[tid] = 0;
    }
    if (tid == 0) sOverflow = 0;
    __syncthreads();
    const bool first = act && (tid == 0 || sRow[tid - 1] != row);
    const unsigned long long bal = __ballot(first);
    const int lane = tid & 63, wave = tid >> 6;
    if (lane == 0) sWave[wave] = __popcll(bal);
    __syncthreads();
    int ord = __popcll(bal & ((2ull << lane) - 1ull)) - 1;
    for (int w = 0; w < wave; ++w) ord += sWave[w];
    bool packed = sWave[0] + sWave[1] + sWave[2] + sWave[3] <= NB16_ROWS;
    // the nine fluid and boundary row runs (rows y+dy, z+dz, r = 3 (dz+1) +
    // (dy+1)), looked up once and kept in registers; empty: (0, 0)
    int2 runF[9], runB[9];
    if (D.cellRuns) {
        // without branches, so that the loads of all nine rows are in flight
        // together (three round trips instead of one after another per row)
        int rk[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int z = min(max(cz + r / 3 - 1, 0), max(G.nz - 1, 0)), y = min(max(cy + r % 3 - 1, 0), max(G.ny - 1, 0));
            rk[r] = act ? D.rowRank[G.rowBase + z * G.ny + y] : 0;
        }
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int z = cz + r / 3 - 1, y = cy + r % 3 - 1;
            const bool in = act && z >= 0 && z < G.nz && y >= 0 && y < G.ny;
            const uint32_t k0 = act ? G.keyBase + (uint32_t)rk[r] * (uint32_t)G.nx + (uint32_t)cx : 0u;
            const int2 rf = run3(D.cellF, k0, act ? cx : 0, G.nx, 1);
            const int2 rb = run3(D.cellB, k0, act ? cx : 0, G.nx, 1);
            runF[r] = in && rf.y > rf.x ? rf : make_int2(0, 0);
            runB[r] = in && rb.y > rb.x ? rb : make_int2(0, 0);
        }
    } else {
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            runF[r] = make_int2(0, 0);
            runB[r] = make_int2(0, 0);
            const int z = cz + r / 3 - 1, y = cy + r % 3 - 1;
            if (act && z >= 0 && z < G.nz && y >= 0 && y < G.ny) {
                const uint32_t k0 = key_of(G, D.rowRank, cx, y, z);
                const int2 rf = run3(D.cellF, k0, cx, G.nx, 0);
                const int2 rb = run3(D.cellB, k0, cx, G.nx, 0);
                if (rf.y > rf.x) runF[r] = rf;
                if (rb.y > rb.x) runB[r] = rb;
            }
        }
    }
    // per slot: the smallest run start and the largest run end of the tile.
    // Along the particles of one own row the runs move up, so of each wave
    // only the row's first and last particle with a run can hold them: two
    // LDS atomics of at most NB16_ROWS lanes a run (from every lane they
    // serialise on one address, 8 of the builder's 40 us on a small scene).
    if (packed && act) {
        // lanes of this wave in the particle's own row
        unsigned long long mine = 0;
#pragma unroll
        for (int o = 0; o < NB16_ROWS; ++o) {
            const unsigned long long b = __ballot(ord == o);
            if (ord == o) mine = b;
        }
        auto bounds = [&](const int2* runs, int slot0) {
#pragma unroll
            for (int r = 0; r < 9; ++r) {
                const bool has = runs[r].y > runs[r].x;
                const unsigned long long b = __ballot(has) & mine;
                if (!has) continue;
                if (__ffsll((long long)b) - 1 == lane) atomicMin(&sBase[slot0 + ord * 9 + r], runs[r].x);
                if (63 - __clzll((long long)b) == lane) atomicMax(&sEnd[slot0 + ord * 9 + r], runs[r].y);
            }
        };
        bounds(runF, 0);
        bounds(runB, 32);
    }
    __syncthreads();
    if (tid < 64 && sBase[tid] != INT_MAX && sEnd[tid] - sBase[tid] > (1 << NB16_OFF_BITS)) sOverflow = 1;
    __syncthreads();
    packed = packed && sOverflow == 0;
    // the tile's window: its fluid slot runs concatenated in slot order (the
    // order in which the solver passes stage it); entry e of slot s is
    // record e + sWin[s] of it
    if (tid < 64) {
        const int len = (packed && tid < 32 && tid != NB16_FLAG && sBase[tid] != INT_MAX) ? sEnd[tid] - sBase[tid] : 0;
        int incl = len;
        for (int off = 1; off < 32; off <<= 1) {
            const int t = __shfl_up(incl, off, 64);
            if (tid >= off) incl += t;
        }
        if (tid < 32) sWin[tid] = (incl - len) - (tid << NB16_OFF_BITS);
        if (tid == 31) sWin[32] = incl;
    }
    __syncthreads();
    const bool win = packed && sWin[32] <= WIN_MAX;
    auto to_win = [&](unsigned e) { return (e + (unsigned)sWin[e >> NB16_OFF_BITS]) & 0xffffu; };

    // staged entry k of this thread: element k * 256 + tid of the stage
    // (entries of one thread 256 elements apart, so one store instruction of
    // a wave writes consecutive elements and its address is one operation)
    auto put = [&](int* list, int k, int j) {
        if (k < NB_STAGE_GROUPS * 4) st[(k << 8) + tid] = j;
        else list[nb_slot(k, i, stride)] = j;
    };
    // bias(slot) = (slot << NB16_OFF_BITS) - base[slot]: an entry is j + bias
    auto bias16 = [&](int slot) { return packed ? (slot << NB16_OFF_BITS) - sBase[slot] : 0; };
    auto put16 = [&](int4* list, int k, int bias, int j) {
        const uint16_t e = uint16_t(j + bias);
        if (k < NB_STAGE_GROUPS * 8) {
            st16[(k << 8) + tid] = e;
        } else {
            reinterpret_cast<uint16_t*>(list)[nb16_slot(k, i, stride)] = e;
            if (win && list == D.nbF16) reinterpret_cast<uint16_t*>(D.nbW16)[nb16_slot(k, i, stride)] = uint16_t(to_win(e));
        }
    };
    // (a thread stages and flushes its own column: no barrier around either)
    auto flush = [&](int* list, int count) {
        const int ng = min((count + 3) >> 2, NB_STAGE_GROUPS);
        int4* out = reinterpret_cast<int4*>(list);
        for (int g = 0; g < ng; ++g) {
            const int b = (4 * g) << 8;
            out[(size_t)g * stride + i] = make_int4(st[b + tid], st[b + 256 + tid], st[b + 512 + tid], st[b + 768 + tid]);
        }
    };
    auto flush16 = [&](int4* out, int count) {
        const int ng = min((count + 7) >> 3, NB_STAGE_GROUPS);
        const bool towin = win && out == D.nbF16;
        for (int g = 0; g < ng; ++g) {
            unsigned w[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int b = (8 * g + 2 * q) << 8;
                w[q] = (unsigned)st16[b + tid] | (unsigned)st16[b + 256 + tid] << 16;
            }
            out[(size_t)g * stride + i] = make_int4((int)w[0], (int)w[1], (int)w[2], (int)w[3]);
            if (towin) {
                // the same group as window indices (entries past the padded
                // count are converted too, and never read)
                int r[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) r[q] = (int)(to_win(w[q] & 0xffffu) | to_win(w[q] >> 16) << 16);
                D.nbW16[(size_t)g * stride + i] = make_int4(r[0], r[1], r[2], r[3]);
            }
        }
    };
    int nbn = 0, zero = 0;
    // Candidate loop of one kind (fluid or boundary), candidates four at a
    // time (four loads in flight, tested in order).  A candidate's entry is
    // stored in LDS at the next free entry before the test decides (a miss
    // is overwritten by the next hit, or lies past the padded count that
    // the passes read).  While every lane of the wave has four staged entries
    // free, a group takes the short form: no test against the stage or the
    // list width, the self index compared in the particle's own row only
    // (the one row run that holds it), and coincident pairs counted only when
    // the smallest of the four squared distances is zero.  Otherwise entries
    // past the LDS stage go to global memory, those past the list width
    // nowhere.  n: entries found.
    auto candidates = [&](auto packed_c, auto fluid_c, const int2* runs, const float4* __restrict__ xs, int cap,
                          int slot0, int4* list16, int* list32, int& n) {
        constexpr bool PK = decltype(packed_c)::value, FLUID = decltype(fluid_c)::value;
        constexpr int STAGE = PK ? NB_STAGE_GROUPS * 8 : NB_STAGE_GROUPS * 4;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int2 rr = runs[r];
            const int bias = PK && rr.y > rr.x ? bias16(slot0 + ord * 9 + r) : 0;
            const bool own = FLUID && r == 4;   // the row run that holds the particle itself
            for (int j0 = rr.x; j0 < rr.y; j0 += 4) {
                // (up to X_TAIL records past the run are read, and not used:
                // the position arrays are that much longer)
                const float4* __restrict__ xg = xs + j0;
                float4 q[4];
                float l2[4];
                bool hit[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = xg[k];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    l2[k] = dis_square_exact(pa, q[k]);
                    hit[k] = j0 + k < rr.y && l2[k] < D.h2;
                    if (own) hit[k] = hit[k] && j0 + k != i;
                }
                if (__ballot(n > STAGE - 4) == 0) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        if (PK) st16[(n << 8) + tid] = uint16_t(j0 + k + bias);
                        else st[(n << 8) + tid] = j0 + k;
                        n += hit[k];
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int j = j0 + k;
                        if (n < STAGE) {
                            if (PK) st16[(n << 8) + tid] = uint16_t(j + bias);
                            else st[(n << 8) + tid] = j;
                        }
                        if (hit[k] && n >= STAGE && n < cap) {
                            if (PK) put16(list16, n, bias, j);
                            else put(list32, n, j);
                        }
                        n += hit[k];
                    }
                }
                if (own || fminf(fminf(l2[0], l2[1]), fminf(l2[2], l2[3])) == 0.0f) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) zero += (hit[k] && l2[k] == 0.0f);
                }
            }
        }
    };
    using PackedT = std::integral_constant<bool, true>;
    using PlainT = std::integral_constant<bool, false>;
    using FluidT = PackedT;
    using WallT = PlainT;
    // fluid neighbours (SphBase.cpp:867-905); the particle itself is skipped
    int nf = 0;
    if (packed) candidates(PackedT{}, FluidT{}, runF, D.x, NBF_CAP, 0, D.nbF16, nullptr, nf);
    else candidates(PlainT{}, FluidT{}, runF, D.x, NBF_CAP, 0, nullptr, D.nbF, nf);
    const int stored = min(nf, NBF_CAP);
    const int cf = act ? stored : 0;
    // pad: the particle itself
    for (int k = cf; k < ((cf + 3) & ~3); ++k) {
        if (packed) put16(D.nbF16, k, bias16(ord * 9 + 4), i);
        else put(D.nbF, k, i);
    }
    if (packed) flush16(D.nbF16, cf);
    else flush(D.nbF, cf);
    // boundary neighbours (SphBase.cpp:908-930); no index is skipped
    if (act) {
        if (packed) candidates(PackedT{}, WallT{}, runB, D.xb, NBB_CAP, 32, D.nbB16, nullptr, nbn);
        else candidates(PlainT{}, WallT{}, runB, D.xb, NBB_CAP, 32, nullptr, D.nbB, nbn);
    }
    const int cb = act ? min(nbn, NBB_CAP) : 0;
    // pad: the far dummy particle
    for (int k = cb; k < ((cb + 3) & ~3); ++k) {
        if (packed) {
            const uint16_t e = uint16_t(NB16_DUMMY << NB16_OFF_BITS);
            if (k < NB_STAGE_GROUPS * 8) st16[(k << 8) + tid] = e;
            else reinterpret_cast<uint16_t*>(D.nbB16)[nb16_slot(k, i, stride)] = e;
        }
        else put(D.nbB, k, D.nb);
    }
    if (packed) flush16(D.nbB16, cb);
    else flush(D.nbB, cb);
    if (tid < NB16_TAB) {
        const int slot = tid & 31;
        int v;
        if (tid == NB16_FLAG) v = packed ? 1 : 0;
        else if (tid == 32 + NB16_DUMMY) v = D.nb - (NB16_DUMMY << NB16_OFF_BITS);
        else v = sBase[tid] != INT_MAX ? sBase[tid] - (slot << NB16_OFF_BITS) : 0;
        D.nbTab[(size_t)tile * NB16_TAB + tid] = v;
        if (tid < 32) D.nbWin[(size_t)tile * 32 + tid] = packed ? sWin[tid] + (tid << NB16_OFF_BITS) : 0;
    }
    // stored fluid entries | fluid neighbours found << 8 | boundary << 16 | phase << 24
    if (i < D.npad) D.cnt[i] = cf | (act ? min(nf, 255) : 0) << 8 | (cb << 16) | ((act ? int(pa.w) : 0) << 24);
    if (!act) return;
    const int tm = nf + nbn - REF_NEIGHBOUR_CAP, over = max(nf - NBF_CAP, 0) + max(nbn - NBB_CAP, 0);
    if (tm > 0) atomicAdd(&D.counters[C_TOO_MANY], tm);
    if (over > 0) atomicAdd(&D.counters[C_LIST_OVF], over);
    if (zero > 0) atomicAdd(&D.counters[C_ZERO_DIS], zero);
}

// The list builder of scenes that leave the chip's CUs idle (launch_neighbours):
// a block takes a quarter of a tile, 64 particles, and a wave one of their nine
// row runs.  A tile's candidates (55,000 pairs) otherwise all pass through one
// CU, whose arithmetic they keep busy for 20,000 cycles; a quarter's take a
// fourth, and the chain of each thread is one row's.  Hits are bits of a mask,
// so the rows' counts are known before anything is stored, and the entries go
// to their places of the list in LDS, whose groups the waves then write out.
// Rows in one loop and both kinds of neighbour in one copy of the code: on a
// small scene a kernel's instructions are read from memory once a launch (the
// 53 KB of k_neighbours<6> cost more than its loads).
// The slot bounds come from the table's entries at the ends of the tile's rows,
// so the table has to be filled (Dev::cellRuns).  Between two particles of a row
// that are far apart they may take in a gap that k_neighbours leaves out; the
// lists hold the same neighbours in the same order.
// Bound by the pairs' arithmetic on the CUs that have a block, and under
// 10,000 particles by the chain of its phases: 1,728 particles 34 -> 10.8 us,
// 15,625 35 -> 11.8.
constexpr int NBQ_ROWS = 9, NBQ_BATCH = 8;
__global__ __launch_bounds__(64 * NBQ_ROWS) void k_neighbours_quarter(Dev D) {
    __shared__ int sRow[256], sCx[256], sOrd[256];
    __shared__ int sWave[4], sFirst[NB16_ROWS], sLast[NB16_ROWS];
    __shared__ int sBase[2 * 32], sKey[32], sOverflow;
    __shared__ int sWin[33];                  // as in k_neighbours
    __shared__ int sCount[2][NBQ_ROWS][64];
    __shared__ int sList[NBF_CAP + NBB_CAP][64];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = blockIdx.x >> 2, p = (int)(blockIdx.x & 3) * 64 + lane, i = tile * 256 + p;
    const float4 pa = D.x[i];
    const int valid = D.tileValid[tile];
    const bool act = p < valid;
    if (valid <= p - lane && p != lane) {     // uniform: none of the quarter (the first has the tile's table)
        if (w == 0) D.cnt[i] = 0;
        return;
    }
    const SceneGrid G = D.grids[D.tileScene[tile]];
    // the tile's rows
    if (tid < 256) {
        int cx = 0, cy = 0, cz = 0;
        if (tid < valid) cell_of(G, D.x[tile * 256 + tid], cx, cy, cz);
        sRow[tid] = tid < valid ? cz * G.ny + cy : -1;
        sCx[tid] = cx;
    }
    if (tid < NB16_ROWS) sFirst[tid] = sLast[tid] = -1;
    if (tid == 0) sOverflow = 0;
    __syncthreads();
    const int row = tid < 256 ? sRow[tid] : -1;
    const bool first = row >= 0 && (tid == 0 || sRow[tid - 1] != row);
    const unsigned long long bal = __ballot(first);
    if (w < 4 && lane == 0) sWave[w] = __popcll(bal);
    __syncthreads();
    const int rows = sWave[0] + sWave[1] + sWave[2] + sWave[3];
    if (tid < 256) {
        int ord = __popcll(bal & ((2ull << lane) - 1ull)) - 1;
        for (int k = 0; k < w; ++k) ord += sWave[k];
        sOrd[tid] = ord;
        if (row >= 0 && ord < NB16_ROWS) {
            if (first) sFirst[ord] = tid;
            if (tid == 255 || sRow[tid + 1] != row) sLast[ord] = tid;
        }
    }
    __syncthreads();
    // row run r of the particles of a row: the key of its first cell, or -1
    auto row_key = [&](int row, int r) {
        const int z = row / G.ny + r / 3 - 1, y = row % G.ny + r % 3 - 1;
        return z >= 0 && z < G.nz && y >= 0 && y < G.ny
                   ? int(G.keyBase + (uint32_t)D.rowRank[G.rowBase + z * G.ny + y] * (uint32_t)G.nx)
                   : -1;
    };
    // per slot: the tile's run, [start of the first particle's, end of the last's)
    if (tid < 64) {
        const int slot = lane & 31, o = slot / 9;
        int base = INT_MAX, len = 0;
        if (rows <= NB16_ROWS && o < rows) {
            const int k = row_key(sRow[sFirst[o]], slot % 9);
            if (lane < 32) sKey[slot] = k;
            if (k >= 0) {
                const int2* __restrict__ table = lane < 32 ? D.cellF : D.cellB;
                const int s = table[k + max(sCx[sFirst[o]] - 1, 0)].x, e = table[k + min(sCx[sLast[o]] + 1, G.nx - 1)].y;
                if (e > s) {
                    base = s;
                    len = e - s;
                }
            }
        }
        sBase[lane] = base;
        if (len > (1 << NB16_OFF_BITS)) sOverflow = 1;
        if (lane >= 32) len = 0;
        int incl = len;
        for (int off = 1; off < 32; off <<= 1) {
            const int t = __shfl_up(incl, off, 64);
            if (lane >= off) incl += t;
        }
        if (lane < 32) sWin[lane] = (incl - len) - (lane << NB16_OFF_BITS);
        if (lane == 31) sWin[32] = incl;
    }
    __syncthreads();
    const bool packed = rows <= NB16_ROWS && sOverflow == 0;
    const bool win = packed && sWin[32] <= WIN_MAX;
    const int ord = sOrd[p], cx = sCx[p];
    auto bias16 = [&](int slot) { return packed ? (slot << NB16_OFF_BITS) - sBase[slot] : 0; };
    // the wave's run of each kind, and the hits of its first 64 candidates
    const int key = act ? (rows <= NB16_ROWS ? sKey[ord * 9 + w] : row_key(sRow[p], w)) : -1;
    int2 runs[2];
#pragma unroll
    for (int kind = 0; kind < 2; ++kind) {
        const int2* __restrict__ table = kind ? D.cellB : D.cellF;
        const int k = key >= 0 ? key + cx : 0;
        runs[kind].x = table[key >= 0 && cx > 0 ? k - 1 : k].x;
        runs[kind].y = table[key >= 0 && cx + 1 < G.nx ? k + 1 : k].y;
        if (key < 0 || runs[kind].y < runs[kind].x) runs[kind].y = runs[kind].x;
    }
    unsigned long long mask[2];
    int zero = 0;
    const int self = w == 4 ? i : -1;         // the row run that holds the particle itself
    // a longer run, candidate by candidate
    auto walk = [&](int kind, int2 rr, auto&& each) {
        const float4* __restrict__ xs = kind ? D.xb : D.x;
#pragma unroll 1
        for (int j = rr.x; j < rr.y; ++j) {
            const float l2 = dis_square_exact(pa, xs[j]);
            if (l2 < D.h2 && (kind || j != self)) each(j, l2);
        }
    };
#pragma unroll 1
    for (int kind = 0; kind < 2; ++kind) {
        const int2 rr = kind ? runs[1] : runs[0];
        const float4* __restrict__ xs = kind ? D.xb : D.x;
        const int len = rr.y - rr.x;
        unsigned long long m = 0, z = 0;
        int n = 0;
        if (len <= 64) {
#pragma unroll 1
            for (int k0 = 0; k0 < len; k0 += NBQ_BATCH) {
                // (up to X_TAIL records past the run are read, and not used)
                const float4* __restrict__ xg = xs + rr.x + k0;
                float4 q[NBQ_BATCH];
                unsigned mk = 0, zk = 0;
#pragma unroll
                for (int k = 0; k < NBQ_BATCH; ++k) q[k] = xg[k];
#pragma unroll
                for (int k = 0; k < NBQ_BATCH; ++k) {
                    const float l2 = dis_square_exact(pa, q[k]);
                    mk |= l2 < D.h2 ? 1u << k : 0u;
                    zk |= l2 == 0.0f ? 1u << k : 0u;
                }
                m |= (unsigned long long)mk << k0;
                z |= (unsigned long long)zk << k0;
            }
            unsigned long long in = len == 64 ? ~0ull : (1ull << len) - 1ull;
            if (kind == 0 && self >= rr.x && self < rr.y) in &= ~(1ull << (self - rr.x));
            m &= in;
            n = __popcll(m);
            zero += __popcll(z & m);
        } else {
            walk(kind, rr, [&](int, float l2) {
                ++n;
                zero += l2 == 0.0f;
            });
        }
        if (kind) mask[1] = m;
        else mask[0] = m;
        sCount[kind][w][lane] = n;
    }
    __syncthreads();
    // the rows in order: each wave's entries to their places
    int found[2];
#pragma unroll
    for (int kind = 0; kind < 2; ++kind) {
        int k = 0, total = 0;
#pragma unroll
        for (int r = 0; r < NBQ_ROWS; ++r) {
            if (r == w) k = total;
            total += sCount[kind][r][lane];
        }
        found[kind] = total;
        const int cap = kind ? NBB_CAP : NBF_CAP, row0 = kind ? NBF_CAP : 0;
        const int2 rr = runs[kind];
        const int bias = rr.y > rr.x ? bias16(32 * kind + ord * 9 + w) : 0;
        if (rr.y - rr.x <= 64) {
#pragma unroll 1
            for (unsigned long long m = mask[kind]; m; m &= m - 1) {
                if (k < cap) sList[row0 + k][lane] = rr.x + __ffsll((long long)m) - 1 + bias;
                ++k;
            }
        } else {
            walk(kind, rr, [&](int j, float) {
                if (k < cap) sList[row0 + k][lane] = j + bias;
                ++k;
            });
        }
    }
    const int nf = found[0], nbn = found[1];
    const int cf = act ? min(nf, NBF_CAP) : 0, cb = act ? min(nbn, NBB_CAP) : 0;
    __syncthreads();
    // groups of eight entries, padded to four: one packed group, or two of four
#pragma unroll 1
    for (int t = w; t < (NBF_CAP + NBB_CAP) / 8; t += NBQ_ROWS) {
        const bool fluid = t < NBF_CAP / 8;
        const int g = fluid ? t : t - NBF_CAP / 8, n = fluid ? cf : cb, padded = (n + 3) & ~3;
        if (8 * g >= padded) continue;
        // pads: the particle itself, or the far dummy particle
        const int pad = fluid ? (packed ? bias16(ord * 9 + 4) : 0) + i : packed ? NB16_DUMMY << NB16_OFF_BITS : D.nb;
        int e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) e[q] = 8 * g + q < n ? sList[8 * t + q][lane] : pad;
        if (packed) {
            int v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = (e[2 * q] & 0xffff) | e[2 * q + 1] << 16;
            (fluid ? D.nbF16 : D.nbB16)[(size_t)g * D.ncap + i] = make_int4(v[0], v[1], v[2], v[3]);
            if (fluid && win) {
                auto to_win = [&](unsigned x) { return (x + (unsigned)sWin[x >> NB16_OFF_BITS]) & 0xffffu; };
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    v[q] = int(to_win((unsigned)e[2 * q] & 0xffffu) | to_win((unsigned)e[2 * q + 1] & 0xffffu) << 16);
                D.nbW16[(size_t)g * D.ncap + i] = make_int4(v[0], v[1], v[2], v[3]);
            }
        } else {
            int4* const out = reinterpret_cast<int4*>(fluid ? D.nbF : D.nbB) + (size_t)(2 * g) * D.ncap + i;
            out[0] = make_int4(e[0], e[1], e[2], e[3]);
            if (8 * g + 4 < padded) out[D.ncap] = make_int4(e[4], e[5], e[6], e[7]);
        }
    }
    if (p == lane && tid < NB16_TAB) {        // the first quarter: the tile's tables
        const int slot = tid & 31;
        int v;
        if (tid == NB16_FLAG) v = packed ? 1 : 0;
        else if (tid == 32 + NB16_DUMMY) v = D.nb - (NB16_DUMMY << NB16_OFF_BITS);
        else v = sBase[tid] != INT_MAX ? sBase[tid] - (slot << NB16_OFF_BITS) : 0;
        D.nbTab[(size_t)tile * NB16_TAB + tid] = v;
        if (tid < 32) D.nbWin[(size_t)tile * 32 + tid] = packed ? sWin[tid] + (tid << NB16_OFF_BITS) : 0;
    }
    if (zero > 0) atomicAdd(&D.counters[C_ZERO_DIS], zero);
    if (w != 0) return;
    D.cnt[i] = act ? cf | min(nf, 255) << 8 | cb << 16 | int(pa.w) << 24 : 0;
    if (!act) return;
    const int tm = nf + nbn - REF_NEIGHBOUR_CAP, over = max(nf - NBF_CAP, 0) + max(nbn - NBB_CAP, 0);
    if (tm > 0) atomicAdd(&D.counters[C_TOO_MANY], tm);
    if (over > 0) atomicAdd(&D.counters[C_LIST_OVF], over);
}

// ---- boundary --------------------------------------------------------------

__global__ __launch_bounds__(256) void k_boundary_keys(Dev D, const float4* __restrict__ xs,
                                                     const int* __restrict__ scene, uint32_t* keys,
                                                     uint32_t* vals) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= D.nb) return;
    const SceneGrid G = D.grids[scene[i]];
    int cx, cy, cz;
    cell_of(G, xs[i], cx, cy, cz);
    keys[i] = key_of(G, D.rowRank, cx, cy, cz);
    vals[i] = (uint32_t)i;
}

__global__ __launch_bounds__(256) void k_boundary_reorder(Dev D, const float4* __restrict__ xs,
                                                        const int* __restrict__ solid,
                                                        const int* __restrict__ scene,
                                                        const uint32_t* __restrict__ sk,
                                                        const uint32_t* __restrict__ sv) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= D.nb) return;
    int src = (int)sv[r];
    D.xb[r] = xs[src];
    D.vb[r] = make_float4(0.f, 0.f, 0.f, 0.f);
    D.bid[r] = src;
    D.bsolid[r] = solid[src];
    D.bscene[r] = scene[src];
    D.bkey[r] = sk[r];
}

// SphBase::prepareSolidPartWeight (SphBase.cpp:766-813): V_b = 1/(W(0) + sum over
// boundary neighbours W(r)); kerSumFromSelf = W(0) + same-solid part.
__global__ __launch_bounds__(256) void k_boundary_volume(Dev D) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= D.nb) return;
    const SceneGrid G = D.grids[D.bscene[i]];
    float4 pa = D.xb[i];
    int sa = D.bsolid[i];
    int cx, cy, cz;
    cell_of(G, pa, cx, cy, cz);
    float sumAll = D.W0, sumSelf = D.W0;
    for (int dz = -1; dz <= 1; ++dz) {
        int z = cz + dz;
        if (z < 0 || z >= G.nz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int y = cy + dy;
            if (y < 0 || y >= G.ny) continue;
            uint32_t k0 = key_of(G, D.rowRank, cx, y, z);
            int2 rb = run3(D.cellB, k0, cx, G.nx, D.cellRuns);
            for (int j = rb.x; j < rb.y; ++j) {
                if (j == i) continue;
                float4 pb = D.xb[j];
                float l2 = dis_square_exact(pa, pb);
                if (l2 < D.h2) {
                    float w = kernel_W(sqrtf(l2), D);
                    sumAll += w;
                    if (D.bsolid[j] == sa) sumSelf += w;
                }
            }
        }
    }
    pa.w = 1.0f / sumAll;
    D.xb[i] = pa;
    D.bkself[i] = sumSelf;
}

// ---- dynamic solids -----------------------------------------------------------
// SphSolid::updatePaticles (SphBase.cpp:95-128): x = T p0 (projective divide),
// v = v_lin + w x (x - com), for the particles of dynamic solids
__global__ __launch_bounds__(256) void k_rigid_pose(Dev D) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= D.nb) return;
    const SolidPose& S = D.solids[D.bsolid[i]];
    if (!S.dynamic) return;
    const float4 p = D.bloc[i];
    const float* T = S.T;
    float x = T[0] * p.x + T[4] * p.y + T[8] * p.z + T[12];
    float y = T[1] * p.x + T[5] * p.y + T[9] * p.z + T[13];
    float z = T[2] * p.x + T[6] * p.y + T[10] * p.z + T[14];
    const float a = T[3] * p.x + T[7] * p.y + T[11] * p.z + T[15];
    x /= a; y /= a; z /= a;
    const float rx = x - S.com[0], ry = y - S.com[1], rz = z - S.com[2];
    D.xb[i] = make_float4(x, y, z, D.xb[i].w);
    D.vb[i] = make_float4(S.v[0] + (S.w[1] * rz - S.w[2] * ry), S.v[1] + (S.w[2] * rx - S.w[0] * rz),
                          S.v[2] + (S.w[0] * ry - S.w[1] * rx), 0.0f);
}

// body-frame samples (original order) into sorted order; slot of each original index
__global__ __launch_bounds__(256) void k_boundary_init_local(Dev D, const float4* __restrict__ local) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= D.nb) return;
    const int k = D.bid[r];
    D.bloc[r] = local[k];
    D.brank[k] = r;
}

// boundary arrays gathered into cell-key order after the solids moved
__global__ __launch_bounds__(256) void k_boundary_regather(Dev D, const uint32_t* __restrict__ sk,
                                                         const uint32_t* __restrict__ sv) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= D.nb) return;
    const int src = (int)sv[r];
    D.xb2[r] = D.xb[src];
    D.vb2[r] = D.vb[src];
    D.bloc2[r] = D.bloc[src];
    D.bid2[r] = D.bid[src];
    D.bsolid2[r] = D.bsolid[src];
    D.bscene2[r] = D.bscene[src];
    D.bkself2[r] = D.bkself[src];
    D.bkey2[r] = sk[r];
    D.brank[D.bid[src]] = r;
}

// SphBase::updateSolidPartWeight (SphBase.cpp:817-841): V_b = 1 /
// (kerSumFromSelf + sum of W over boundary neighbours of other solids; a
// rigid body's own particles keep the part fixed at the start, kerSumFromSelf)
__global__ __launch_bounds__(256) void k_boundary_volume_update(Dev D) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= D.nb) return;
    const SceneGrid G = D.grids[D.bscene[i]];
    float4 pa = D.xb[i];
    const int sa = D.bsolid[i];
    int cx, cy, cz;
    cell_of(G, pa, cx, cy, cz);
    float vol = D.bkself[i];
    for (int dz = -1; dz <= 1; ++dz) {
        int z = cz + dz;
        if (z < 0 || z >= G.nz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int y = cy + dy;
            if (y < 0 || y >= G.ny) continue;
            int2 rb = run3(D.cellB, key_of(G, D.rowRank, cx, y, z), cx, G.nx, D.cellRuns);
            for (int j = rb.x; j < rb.y; ++j) {
                if (j == i || D.bsolid[j] == sa) continue;
                float l2 = dis_square_exact(pa, D.xb[j]);
                if (l2 < D.h2) vol += kernel_W(sqrtf(l2), D);
            }
        }
    }
    pa.w = 1.0f / vol;
    D.xb[i] = pa;
}

// Reaction force on the particles of dynamic solids from their fluid
// neighbours, summed from the boundary particle's side (a fixed order).
// mode 0 WCSPH, WcSph::wc_boundPartForce_f (WcSph.cpp:314-362): pressure x2
// (its fluid-side boundary force, WcSph.cpp:285) and artificial viscosity;
// fluid pressure f1, density v.w.
// mode 1 IISPH, IISph_M::ii_boundPartForcePressure_f (IISph_M.cpp:586-607):
// pressure x1 (the fluid-side boundary force of this implementation) and
// viscosity; pressure kr, density rho.
// mode 2 DFSPH, the constant-density solve's boundary term accumulated over
// its iterations (DFSPH.cpp:674-690, scaled by the fluid mass at 723-737):
// F_b = sum_j m_j rho0_j V_b (sum_it kappa_j / rho_j) grad_j W_jb, with
// sum_it kappa_j dt^2 = ksum_j; no viscosity.
__global__ __launch_bounds__(256) void k_rigid_reaction(Dev D, int mode) {
    int a = blockIdx.x * 256 + threadIdx.x;
    if (a >= D.nb) return;
    const SolidPose& S = D.solids[D.bsolid[a]];
    if (!S.dynamic) return;
    const SceneGrid G = D.grids[D.bscene[a]];
    const float4 pa = D.xb[a], va = D.vb[a];
    const bool iisph = mode == 1, dfsph = mode == 2;
    const float pf = iisph ? 1.0f : 2.0f;
    const float nuc = 2.0f * S.visc * D.Hs * D.cs;
    const float dt = D.dt[D.bscene[a]];
    const float rdt2 = 1.0f / (dt * dt);
    int cx, cy, cz;
    cell_of(G, pa, cx, cy, cz);
    float fx = 0.f, fy = 0.f, fz = 0.f;
    for (int dz = -1; dz <= 1; ++dz) {
        int z = cz + dz;
        if (z < 0 || z >= G.nz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int y = cy + dy;
            if (y < 0 || y >= G.ny) continue;
            int2 rf = run3(D.cellF, key_of(G, D.rowRank, cx, y, z), cx, G.nx, D.cellRuns);
            for (int j = rf.x; j < rf.y; ++j) {
                const float4 pb = D.x[j];
                const float l2 = dis_square_exact(pa, pb);
                if (!(l2 < D.h2) || l2 == 0.0f) continue;
                const int ph = (int)pb.w;
                const float frho0 = D.rho0[ph], fm0 = D.mass[ph];
                const float dx = pa.x - pb.x, dy2 = pa.y - pb.y, dz2 = pa.z - pb.z;
                const float g = kernel_gradfac(sqrtf(l2), D);
                if (dfsph) {
                    const float k = D.ksum[j] * rdt2 / D.rho[j];
                    const float force = -g * (fm0 * frho0 * pa.w * k);
                    fx += dx * force; fy += dy2 * force; fz += dz2 * force;
                    continue;
                }
                const float4 vb = D.v[j];
                const float rhob = iisph ? D.rho[j] : vb.w;
                const float pb_p = iisph ? D.kr[j] : D.f1[j];
                const float cvol = -fm0 * frho0 * pa.w;
                float force = pb_p > 0.0f ? g * (cvol * (pb_p / (rhob * rhob) * pf)) : 0.0f;
                const float pro = (va.x - vb.x) * dx + (va.y - vb.y) * dy2 + (va.z - vb.z) * dz2;
                if (pro < 0.0f) {
                    const float nu = nuc / (rhob * 2.0f);
                    const float pi = -nu * pro / (l2 + D.visc_eps);
                    force += g * (cvol * pi);
                }
                fx += dx * force; fy += dy2 * force; fz += dz2 * force;
            }
        }
    }
    D.bforce[a] = make_float4(fx, fy, fz, 0.0f);
}

// SphSolid::rigidForceJoin (SphBase.cpp:131-143) per dynamic solid: one block
// per solid over its particles in original order, in double, fixed tree
__global__ __launch_bounds__(256) void k_solid_reduce(Dev D, double* __restrict__ out) {
    __shared__ double lds[6][4];
    const int s = blockIdx.x;
    const SolidPose& S = D.solids[s];
    double acc[6] = {0, 0, 0, 0, 0, 0};
    if (S.dynamic) {
        for (int k = S.firstId + (int)threadIdx.x; k < S.endId; k += 256) {
            const int r = D.brank[k];
            const float4 f = D.bforce[r], x = D.xb[r];
            const double rx = (double)x.x - S.com[0], ry = (double)x.y - S.com[1], rz = (double)x.z - S.com[2];
            acc[0] += f.x; acc[1] += f.y; acc[2] += f.z;
            acc[3] += ry * f.z - rz * f.y;
            acc[4] += rz * f.x - rx * f.z;
            acc[5] += rx * f.y - ry * f.x;
        }
    }
    for (int q = 0; q < 6; ++q) {
        double v = acc[q];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if ((threadIdx.x & 63) == 0) lds[q][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        const int q = threadIdx.x;
        out[6 * s + q] = ((lds[q][0] + lds[q][1]) + lds[q][2]) + lds[q][3];
    }
}

// test dump: the stored neighbour lists (the ones every pass iterates), with
// original ids and correctly rounded distances
__global__ __launch_bounds__(256) void k_neighbour_dump(Dev D, int cap, int* counts, int* kinds,
                                                      long long* ids, float* dis, const int* rankOf) {
    int i = blockIdx.x * 256 + threadIdx.x;
    int scene;
    if (i >= D.npad || !slot_valid(D, i, &scene)) return;
    int o = rankOf[i];
    if (o < 0) return;
    const float4 pa = D.x[i];
    const int cnt = D.cnt[i], nf = cnt & 0xFF, nbn = (cnt >> 16) & 0xFF;
    const int* tab = D.nbTab + (size_t)(i / TILE) * NB16_TAB;
    const bool packed = tab[NB16_FLAG] != 0;
    const uint16_t* f16 = reinterpret_cast<const uint16_t*>(D.nbF16);
    const uint16_t* b16 = reinterpret_cast<const uint16_t*>(D.nbB16);
    int c = 0;
    for (int k = 0; k < nf; ++k) {
        int j;
        if (packed) {
            const int e = f16[nb16_slot(k, i, D.ncap)];
            j = tab[e >> NB16_OFF_BITS] + e;
        } else {
            j = D.nbF[nb_slot(k, i, D.ncap)];
        }
        if (c < cap) {
            size_t q = (size_t)o * cap + c;
            kinds[q] = 0; ids[q] = D.id[j]; dis[q] = sqrtf(dis_square_exact(pa, D.x[j]));
        }
        ++c;
    }
    for (int k = 0; k < nbn; ++k) {
        int j;
        if (packed) {
            const int e = b16[nb16_slot(k, i, D.ncap)];
            j = tab[32 + (e >> NB16_OFF_BITS)] + e;
        } else {
            j = D.nbB[nb_slot(k, i, D.ncap)];
        }
        if (c < cap) {
            size_t q = (size_t)o * cap + c;
            kinds[q] = 1; ids[q] = D.bid[j]; dis[q] = sqrtf(dis_square_exact(pa, D.xb[j]));
        }
        ++c;
    }
    counts[o] = c;
}

inline int blocks_for(int n) { return (n + 255) / 256; }

// counts -> cell table (and, for the fluid, the scene layout)
template <bool FLUID>
bool search_in_parts(const Dev& D) {
    return D.totalKeys <= (uint32_t)SEARCH_KEYS_ONE && (!FLUID || D.nscenes == 1);
}
template <bool FLUID>
void scan_cells(const Dev& D, int2* table, int* layoutOut, hipStream_t st) {
    if (search_in_parts<FLUID>(D)) {
        const int parts = ((int)D.totalKeys + SEARCH_PART - 1) / SEARCH_PART;
        hipLaunchKernelGGL(k_search_part<FLUID>, dim3(parts), dim3(SCAN1_THREADS), 0, st, D, table, layoutOut);
        return;
    }
    if constexpr (FLUID) {
        if (D.totalKeys <= (uint32_t)SEARCH_KEYS_ONE) {
            hipLaunchKernelGGL(k_search_one, dim3(1), dim3(SCAN1_THREADS), 0, st, D, table, layoutOut);
            return;
        }
    }
    const int blocks = int((D.totalKeys + SEARCH_KEYS - 1) / SEARCH_KEYS);
    hipLaunchKernelGGL(k_cell_sums, dim3(blocks), dim3(256), 0, st, D);
    hipLaunchKernelGGL(k_search_mid<FLUID>, dim3(1), dim3(SCAN1_THREADS), 0, st, D, blocks, layoutOut);
    hipLaunchKernelGGL(k_cell_runs<FLUID>, dim3(blocks), dim3(256), 0, st, D, table);
}

}  // namespace

void launch_search_fluid(const Dev& D, uint32_t* keys, uint32_t* arrival, uint32_t* order, int* layoutOut,
                         hipStream_t st) {
    const int tiles = D.npad / TILE;
    if (tiles > 0) hipLaunchKernelGGL(k_count_fluid, dim3(tiles), dim3(256), 0, st, D, keys, arrival);
    scan_cells<true>(D, D.cellF, layoutOut, st);
    if (tiles == 0) return;
    hipLaunchKernelGGL(k_place, dim3(tiles), dim3(256), 0, st, (const uint32_t*)keys, (const uint32_t*)arrival,
                       (const int2*)D.cellF, D.npad, order, search_in_parts<true>(D) ? D.cellCnt : nullptr);
    hipLaunchKernelGGL(k_reorder_cells, dim3(tiles), dim3(256), 0, st, D, (const uint32_t*)keys,
                       (const uint32_t*)order);
}

void launch_search_boundary(const Dev& D, const float4* xs, const int* scene, uint32_t* keys, uint32_t* arrival,
                            uint32_t* order, uint32_t* sk, uint32_t* sv, hipStream_t st) {
    const dim3 g(blocks_for(D.nb)), b(256);
    if (D.nb > 0) hipLaunchKernelGGL(k_count_boundary, g, b, 0, st, D, xs, scene, keys, arrival);
    scan_cells<false>(D, D.cellB, nullptr, st);
    if (D.nb <= 0) return;
    hipLaunchKernelGGL(k_place, g, b, 0, st, (const uint32_t*)keys, (const uint32_t*)arrival, (const int2*)D.cellB,
                       D.nb, order, search_in_parts<false>(D) ? D.cellCnt : nullptr);
    hipLaunchKernelGGL(k_order_boundary, g, b, 0, st, D, (const uint32_t*)keys, (const uint32_t*)order, sk, sv);
}

void launch_fluid_keys_into(const Dev& D, uint32_t* keys, uint32_t* vals, hipStream_t st) {
    hipLaunchKernelGGL(k_fluid_keys, dim3(blocks_for(D.npad)), dim3(256), 0, st, D, keys, vals);
}

void launch_scene_bounds(const Dev& D, const uint32_t* sk, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_scene_bounds, dim3(blocks_for(n)), dim3(256), 0, st, D, sk, n);
}

void launch_scene_layout(const Dev& D, int* out, hipStream_t st) {
    hipLaunchKernelGGL(k_scene_layout, dim3(1), dim3(64), 0, st, D, out);
    int numTiles = D.ncap / TILE;
    hipLaunchKernelGGL(k_tiles, dim3(blocks_for(numTiles)), dim3(256), 0, st, D, numTiles);
}

void launch_reorder(const Dev& D, const uint32_t* sk, const uint32_t* sv, int n, int oldPad,
                    hipStream_t st) {
    int limit = oldPad > 0 ? oldPad : n;
    hipLaunchKernelGGL(k_mark_padding, dim3(blocks_for(limit)), dim3(256), 0, st, D, limit);
    hipLaunchKernelGGL(k_reorder, dim3(blocks_for(n)), dim3(256), 0, st, D, sk, sv, n);
}

void launch_cell_reset(const Dev& D, const uint32_t* keys, int n, int2* table, hipStream_t st) {
    (void)D;
    if (n > 0) hipLaunchKernelGGL(k_cell_reset, dim3(blocks_for(n)), dim3(256), 0, st, keys, n, table);
}

void launch_cell_build(const Dev& D, const uint32_t* keys, int n, int2* table, hipStream_t st) {
    (void)D;
    if (n > 0) hipLaunchKernelGGL(k_cell_build, dim3(blocks_for(n)), dim3(256), 0, st, keys, n, table);
}

void launch_neighbours_variant(const Dev& D, int groups, hipStream_t st) {
    const dim3 g(blocks_for(D.npad)), b(256);
    if (D.cellRuns && D.npad / TILE <= QUARTER_TILES) {
        if (D.npad > 0) hipLaunchKernelGGL(k_neighbours_quarter, dim3(4 * (D.npad / TILE)), dim3(64 * NBQ_ROWS), 0, st, D);
        return;
    }
    if (groups >= 8) hipLaunchKernelGGL(k_neighbours<8>, g, b, 0, st, D);
    else hipLaunchKernelGGL(k_neighbours<6>, g, b, 0, st, D);
}

void launch_neighbours(const Dev& D, hipStream_t st) { launch_neighbours_variant(D, D.nbStage, st); }

void launch_boundary_keys_from(const Dev& D, const float4* xs, const int* scene, uint32_t* keys,
                               uint32_t* vals, hipStream_t st) {
    hipLaunchKernelGGL(k_boundary_keys, dim3(blocks_for(D.nb)), dim3(256), 0, st, D, xs, scene, keys, vals);
}

void launch_boundary_reorder(const Dev& D, const float4* srcX, const int* srcSolid, const int* srcScene,
                             const uint32_t* sk, const uint32_t* sv, hipStream_t st) {
    hipLaunchKernelGGL(k_boundary_reorder, dim3(blocks_for(D.nb)), dim3(256), 0, st, D, srcX, srcSolid,
                       srcScene, sk, sv);
}

void launch_boundary_volume(const Dev& D, hipStream_t st) {
    hipLaunchKernelGGL(k_boundary_volume, dim3(blocks_for(D.nb)), dim3(256), 0, st, D);
}

void launch_rigid_reaction(const Dev& D, int mode, hipStream_t st) {
    if (D.nb > 0) hipLaunchKernelGGL(k_rigid_reaction, dim3(blocks_for(D.nb)), dim3(256), 0, st, D, mode);
}

void launch_solid_reduce(const Dev& D, double* out, hipStream_t st) {
    if (D.nsolids > 0) hipLaunchKernelGGL(k_solid_reduce, dim3(D.nsolids), dim3(256), 0, st, D, out);
}

void launch_boundary_init_local(const Dev& D, const float4* local, hipStream_t st) {
    if (D.nb > 0) hipLaunchKernelGGL(k_boundary_init_local, dim3(blocks_for(D.nb)), dim3(256), 0, st, D, local);
}

void launch_rigid_pose(const Dev& D, hipStream_t st) {
    if (D.nb > 0) hipLaunchKernelGGL(k_rigid_pose, dim3(blocks_for(D.nb)), dim3(256), 0, st, D);
}

void launch_boundary_regather(const Dev& D, const uint32_t* sk, const uint32_t* sv, hipStream_t st) {
    if (D.nb > 0) hipLaunchKernelGGL(k_boundary_regather, dim3(blocks_for(D.nb)), dim3(256), 0, st, D, sk, sv);
}

void launch_boundary_volume_update(const Dev& D, hipStream_t st) {
    if (D.nb > 0) hipLaunchKernelGGL(k_boundary_volume_update, dim3(blocks_for(D.nb)), dim3(256), 0, st, D);
}

void launch_neighbour_dump_ranked(const Dev& D, int cap, int* counts, int* kinds, long long* ids,
                                  float* dis, const int* rankOf, hipStream_t st) {
    hipLaunchKernelGGL(k_neighbour_dump, dim3(blocks_for(D.npad)), dim3(256), 0, st, D, cap, counts,
                       kinds, ids, dis, rankOf);
}

}  // namespace sphgpu
