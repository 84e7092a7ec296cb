// Device code shared by the particle passes (solvers.hip, iisph_df.hip): the
// slot of a thread, the neighbour-list loops and the loops' convergence test.
#pragma once

#include "sph_common.h"

namespace sphgpu {

namespace {

struct Slot {
    int i, tile, scene;
    bool live;
    bool packed;   // the tile's neighbour lists are in the packed 16-bit form
    int c;         // the particle's count word (slot_nb; 0: not live)
};

// blocks: the workgroups that take tiles (0: the whole grid); K: lanes a particle
template <int K = 1>
__device__ __forceinline__ Slot slot_of(const Dev& D, bool gated, int blocks = 0) {
    Slot s;
    s.tile = tile_of_block(D.tileMap, blocks ? blocks : (int)gridDim.x);
    s.i = s.tile * TILE + (int)threadIdx.x / K;
    s.scene = D.tileScene[s.tile];
    s.live = (int)threadIdx.x / K < D.tileValid[s.tile];
    if (gated) s.live = s.live && D.active[s.scene] != 0;
    s.packed = false;
    s.c = 0;
    return s;
}

// The tile's list table (fluid slots 0..31, boundary 32..63) and the window
// offset of each fluid slot ([31]: the window size), staged in LDS by the
// kernels that read neighbour lists.
__shared__ int g_nbtab[NB16_TAB];
__shared__ int g_winoff[32];

// slot_of for kernels that read neighbour lists: every thread of the block
// calls it before any returns (it stages the tile's tables in LDS).  What
// depends on the tile or the slot alone (the tables, the count word and what
// `own`(i) loads) is requested before the scene's state is known, so that a
// pass starts with two dependent round trips to memory instead of five.  A
// gated block whose scene has converged has no live particles and returns at
// once: solver iterations launched past convergence cost little.
// QUARTER: a block takes a quarter of a tile (quarter_blocks).
template <int K = 1, bool QUARTER = false, class OWN>
__device__ __forceinline__ Slot slot_nb(const Dev& D, bool gated, OWN&& own, int blocks = 0) {
    static_assert(!QUARTER || 64 * K >= NB16_TAB + 32, "a thread for each word of the tables");
    Slot s;
    const int t = threadIdx.x;
    int at = t / K;   // the particle in the tile
    if constexpr (QUARTER) {
        s.tile = blockIdx.x >> 2;
        at += (blockIdx.x & 3) * 64;
    } else {
        s.tile = tile_of_block(D.tileMap, blocks ? blocks : (int)gridDim.x);
    }
    s.i = s.tile * TILE + at;
    int tab = D.nbTab[(size_t)s.tile * NB16_TAB + (t & (NB16_TAB - 1))];
    int win = D.nbWin[(size_t)s.tile * 32 + (t & 31)];
    const int c = D.cnt[s.i];
    own(s.i);
    s.scene = D.tileScene[s.tile];
    const int valid = D.tileValid[s.tile];
    const bool on = !gated || D.active[s.scene] != 0;
    s.live = on && at < valid;
    s.packed = false;
    s.c = s.live ? c : 0;
    asm volatile("" : "+v"(tab), "+v"(win));   // (else the loads are moved behind the branch)
    if (!on) return s;   // uniform per block
    if (t < NB16_TAB) g_nbtab[t] = tab;
    else if (t < NB16_TAB + 32) g_winoff[t - NB16_TAB] = win;
    __syncthreads();
    s.packed = __builtin_amdgcn_readfirstlane(g_nbtab[NB16_FLAG]) != 0;
    return s;
}
__device__ __forceinline__ Slot slot_nb(const Dev& D, bool gated, int blocks = 0) {
    return slot_nb<1>(D, gated, [](int) {}, blocks);
}

// mass, rest density and viscosity of a phase; one phase: no load that waits for it
__device__ __forceinline__ float mass_of(const Dev& D, int ph) { return D.nphases > 1 ? D.mass[ph] : D.mass[0]; }
__device__ __forceinline__ float visc_of(const Dev& D, int ph) { return D.nphases > 1 ? D.visc[ph] : D.visc[0]; }
__device__ __forceinline__ float rho0_of(const Dev& D, int ph) { return D.nphases > 1 ? D.rho0[ph] : D.rho0[0]; }

// A list group is read once per pass.  Where the lists and records together
// fit the last-level cache the plain load lets the next pass find the list
// there; on larger scenes a streaming load keeps the list from pushing the
// gathered records out (Dev::listNT, chosen by the autotuner).
typedef int v4i_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4 ld_group(const int4* p, bool nt) {
    if (nt) {
        const v4i_t v = __builtin_nontemporal_load(reinterpret_cast<const v4i_t*>(p));
        return make_int4(v.x, v.y, v.z, v.w);
    }
    return *p;
}

// Neighbour loops in split form: load(j) issues the gather(s) of neighbour j
// and returns the record(s), use(j, r) consumes them.  A batch of neighbours is gathered first, then the next list group is
// requested, then the batch is used: a wave waits for its memory returns in
// issue order, so a list load issued ahead of the gathers would hold up every
// batch.  W = 8: one batch of eight per packed group (single-record passes);
// W = 4: two batches of four (two-record passes: eight gathers in flight
// either way).  Entries past the padded count still gather (from the padding
// index) but are not used, so every pass sums exactly the listed entries.
template <int W, int TOFF, class LD, class US>
__device__ __forceinline__ void each_in_list16_lu(const int4* __restrict__ list, int ncap, int i, int n, int padj,
                                                  bool nt, LD&& load, US&& use) {
    static_assert(W == 4 || W == 8, "batch of four or eight");
    const int4* __restrict__ col = list + i;
    const int ng = (n + 7) >> 3;
    if (ng <= 0) return;
    const int n4 = (n + 3) & ~3;
    int4 cur = ld_group(&col[0], nt);
    for (int g = 0; g < ng; ++g) {
        const unsigned w[4] = {(unsigned)cur.x, (unsigned)cur.y, (unsigned)cur.z, (unsigned)cur.w};
        const bool second = 8 * g + 4 < n4;   // entries 8g+4..8g+7 are listed
        int j[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const unsigned e = (w[k >> 1] >> (16 * (k & 1))) & 0xffffu;
            const int jj = g_nbtab[TOFF + (e >> NB16_OFF_BITS)] + (int)e;
            j[k] = (k < 4 || second) ? jj : padj;
        }
        int4 nxt = cur;
        if (W == 8) {
            decltype(load(0)) r[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) r[k] = load(j[k]);
            __builtin_amdgcn_sched_barrier(0);
            if (g + 1 < ng) nxt = ld_group(&col[(size_t)(g + 1) * ncap], nt);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; ++k) use(j[k], r[k]);
            if (second) {
#pragma unroll
                for (int k = 4; k < 8; ++k) use(j[k], r[k]);
            }
        } else {
            decltype(load(0)) r[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] = load(j[k]);
#pragma unroll
            for (int k = 0; k < 4; ++k) use(j[k], r[k]);
#pragma unroll
            for (int k = 0; k < 4; ++k) r[k] = load(j[4 + k]);
            __builtin_amdgcn_sched_barrier(0);
            if (g + 1 < ng) nxt = ld_group(&col[(size_t)(g + 1) * ncap], nt);
            __builtin_amdgcn_sched_barrier(0);
            if (second) {
#pragma unroll
                for (int k = 0; k < 4; ++k) use(j[4 + k], r[k]);
            }
        }
        cur = nxt;
    }
}

// the same for 32-bit lists (groups of four, all listed or padding)
template <class LD, class US>
__device__ __forceinline__ void each_in_list_lu(const int* __restrict__ list, int ncap, int i, int n, bool nt,
                                                LD&& load, US&& use) {
    const int4* __restrict__ col = reinterpret_cast<const int4*>(list) + i;
    const int ng = (n + 3) >> 2;
    if (ng <= 0) return;
    int4 cur = ld_group(&col[0], nt);
    for (int g = 0; g < ng; ++g) {
        const int j[4] = {cur.x, cur.y, cur.z, cur.w};
        decltype(load(0)) r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = load(j[k]);
        int4 nxt = cur;
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 < ng) nxt = ld_group(&col[(size_t)(g + 1) * ncap], nt);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; ++k) use(j[k], r[k]);
        cur = nxt;
    }
}

template <int W, class LD, class US>
__device__ __forceinline__ void each_fluid_lu(const Dev& D, const Slot& s, int nf, LD&& load, US&& use) {
    const bool nt = __builtin_amdgcn_readfirstlane(D.listNT) != 0;
    if (s.packed) each_in_list16_lu<W, 0>(D.nbF16, D.ncap, s.i, nf, s.i, nt, load, use);
    else each_in_list_lu(D.nbF, D.ncap, s.i, nf, nt, load, use);
}

template <int W, class LD, class US>
__device__ __forceinline__ void each_boundary_lu(const Dev& D, const Slot& s, int nb, LD&& load, US&& use) {
    const bool nt = __builtin_amdgcn_readfirstlane(D.listNT) != 0;
    if (s.packed) each_in_list16_lu<W, 32>(D.nbB16, D.ncap, s.i, nb, D.nb, nt, load, use);
    else each_in_list_lu(D.nbB, D.ncap, s.i, nb, nt, load, use);
}

// ---- two lanes a particle ---------------------------------------------------
// K = 2 neighbouring lanes of a wave share a particle: of every eight list
// entries lane h gathers and evaluates entries 4 h .. 4 h + 3 (term), then lane 0
// adds the terms of the eight in list order (add), taking the other's with a DPP
// quad permute, so its sums, the particle's, have the same bits as those of one
// lane a particle (the other lane's sums are not used), as long as a term is
// rounded before it is added: a product that one lane fuses into its sum differs in
// the last place, so such a term is a pair of factors that `add` multiplies.  (Four
// lanes were slower everywhere but on the smallest scenes.)
template <int K>
struct Lanes {
    static_assert(K == 2, "two lanes a particle");
    static constexpr int E = 8 / K;   // entries of a group a lane owns
};
// v of lane O of the particle's
template <int K, int O, class T>
__device__ __forceinline__ T lane_term(const T& v) {
    if constexpr (O == 0) {
        return v;   // (lane 0's sum is the particle's)
    } else {
        constexpr int N = sizeof(T) / 4;
        int w[N];
        __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
        for (int k = 0; k < N; ++k) w[k] = __builtin_amdgcn_mov_dpp(w[k], 0xF5, 0xf, 0xf, true);
        T r;
        __builtin_memcpy(&r, w, sizeof(T));
        return r;
    }
}
// adds a group's terms in order: entries 0..3, and 4..7 where they are listed
template <int K, class T, class AD>
__device__ __forceinline__ void add_group(const T (&t)[Lanes<K>::E], bool second, AD&& add) {
    constexpr int E = Lanes<K>::E;
    add(lane_term<K, 0 / E>(t[0 % E]));
    add(lane_term<K, 1 / E>(t[1 % E]));
    add(lane_term<K, 2 / E>(t[2 % E]));
    add(lane_term<K, 3 / E>(t[3 % E]));
    if (second) {
        add(lane_term<K, 4 / E>(t[4 % E]));
        add(lane_term<K, 5 / E>(t[5 % E]));
        add(lane_term<K, 6 / E>(t[6 % E]));
        add(lane_term<K, 7 / E>(t[7 % E]));
    }
}

// a lane's four packed entries of a group: two words
template <int K>
struct Words {
    unsigned w[4 / K];
};
template <int K>
__device__ __forceinline__ Words<K> ld_words(const int4* group, int h, bool nt) {
    static_assert(K == 2, "two lanes a particle");
    typedef unsigned v2u_t __attribute__((ext_vector_type(2)));
    const v2u_t* q = reinterpret_cast<const v2u_t*>(group) + h;
    const v2u_t v = nt ? __builtin_nontemporal_load(q) : *q;
    return Words<K>{{v.x, v.y}};
}
// entry e of the words
template <int K>
__device__ __forceinline__ unsigned word_entry(const Words<K>& w, int e) {
    return (w.w[e >> 1] >> (16 * (e & 1))) & 0xffffu;
}

// each_in_list16_lu with K lanes a particle
template <int K, int TOFF, class LD, class TM, class AD>
__device__ __forceinline__ void each_in_list16_lanes(const int4* __restrict__ list, int ncap, int i, int h, int n,
                                                     int padj, bool nt, LD&& load, TM&& term, AD&& add) {
    constexpr int E = Lanes<K>::E;
    const int4* __restrict__ col = list + i;
    const int ng = (n + 7) >> 3;
    if (ng <= 0) return;
    const int n4 = (n + 3) & ~3;
    Words<K> cur = ld_words<K>(&col[0], h, nt);
    for (int g = 0; g < ng; ++g) {
        const bool second = 8 * g + 4 < n4;
        int j[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const unsigned e = word_entry<K>(cur, k);
            const int jj = g_nbtab[TOFF + (e >> NB16_OFF_BITS)] + (int)e;
            j[k] = (second || h * E + k < 4) ? jj : padj;
        }
        decltype(load(0)) r[E];
#pragma unroll
        for (int k = 0; k < E; ++k) r[k] = load(j[k]);
        __builtin_amdgcn_sched_barrier(0);
        if (g + 1 < ng) cur = ld_words<K>(&col[(size_t)(g + 1) * ncap], h, nt);
        __builtin_amdgcn_sched_barrier(0);
        decltype(term(0, r[0])) t[E];
#pragma unroll
        for (int k = 0; k < E; ++k) t[k] = term(j[k], r[k]);
        add_group<K>(t, second, add);
    }
}

// the same for 32-bit lists (groups of four, all listed or padding): lane h owns
// every second group
template <int K, class LD, class TM, class AD>
__device__ __forceinline__ void each_in_list_lanes(const int* __restrict__ list, int ncap, int i, int h, int n,
                                                   bool nt, LD&& load, TM&& term, AD&& add) {
    constexpr int E = Lanes<K>::E;
    const int4* __restrict__ col = reinterpret_cast<const int4*>(list) + i;
    const int ng = (n + 3) >> 2;
    // eight entries a turn: two groups, the lane's entries all in one of them
    for (int g = 0; g < ng; g += 2) {
        const bool second = g + 1 < ng;
        const bool mine = second || h * E < 4;
        const int4 v = ld_group(&col[(size_t)(mine ? g + (h * E) / 4 : g) * ncap], nt);
        const int w[4] = {v.x, v.y, v.z, v.w};
        decltype(load(0)) r[E];
        int j[E];
#pragma unroll
        for (int k = 0; k < E; ++k) {
            j[k] = w[k];
            r[k] = load(j[k]);
        }
        decltype(term(0, r[0])) t[E];
#pragma unroll
        for (int k = 0; k < E; ++k) t[k] = term(j[k], r[k]);
        add_group<K>(t, second, add);
    }
}

// The neighbour loops of a particle: load(j) gathers the record of neighbour
// j, term(j, r) is the pair's term, add(t) adds it.  K = 1: one lane a
// particle, W records a batch.
template <int K, int W, class LD, class TM, class AD>
__device__ __forceinline__ void each_fluid(const Dev& D, const Slot& s, int h, int nf, LD&& load, TM&& term, AD&& add) {
    if constexpr (K == 1) {
        each_fluid_lu<W>(D, s, nf, load, [&](int j, const decltype(load(0))& r) { add(term(j, r)); });
    } else {
        const bool nt = __builtin_amdgcn_readfirstlane(D.listNT) != 0;
        if (s.packed) each_in_list16_lanes<K, 0>(D.nbF16, D.ncap, s.i, h, nf, s.i, nt, load, term, add);
        else each_in_list_lanes<K>(D.nbF, D.ncap, s.i, h, nf, nt, load, term, add);
    }
}
template <int K, int W, class LD, class TM, class AD>
__device__ __forceinline__ void each_boundary(const Dev& D, const Slot& s, int h, int nb, LD&& load, TM&& term,
                                              AD&& add) {
    if constexpr (K == 1) {
        each_boundary_lu<W>(D, s, nb, load, [&](int j, const decltype(load(0))& r) { add(term(j, r)); });
    } else {
        const bool nt = __builtin_amdgcn_readfirstlane(D.listNT) != 0;
        if (s.packed) each_in_list16_lanes<K, 32>(D.nbB16, D.ncap, s.i, h, nb, D.nb, nt, load, term, add);
        else each_in_list_lanes<K>(D.nbB, D.ncap, s.i, h, nb, nt, load, term, add);
    }
}

// two gather records of one neighbour
struct Rec2 {
    float4 a, b;
};

__device__ __forceinline__ int phase_of(float4 x) { return (int)x.w; }

// the tile's sum of v, each of its particles' K lanes holding the particle's
// own: in the order of one lane a particle
template <int K>
__device__ __forceinline__ double tile_sum(double v, double* part, double* lds) {
    const int t = threadIdx.x;
    if constexpr (K > 1) {
        if (t % K == 0) part[t / K] = v;
        __syncthreads();
        v = t < TILE ? part[t] : 0.0;
    }
    return block_sum_256(v, lds);
}

__device__ __forceinline__ void write_partial(const Dev& D, int tile, int q, double v, double* lds) {
    double t = block_sum_256(v, lds);
    if (threadIdx.x == 0) D.partial[2 * tile + q] = t;
}

// packed counts: stored fluid entries | fluid neighbours found (the stored
// ones plus any beyond the list capacity, up to 255) << 8 | boundary << 16 |
// the particle's phase << 24
__device__ __forceinline__ int nf_of(int c) { return c & 0xff; }
__device__ __forceinline__ int nf_real(int c) { return (c >> 8) & 0xff; }
__device__ __forceinline__ int nb_of(int c) { return (c >> 16) & 0xff; }
__device__ __forceinline__ int phase_of_cnt(int c) { return c >> 24; }

// ------------------------------------------------------- scene reduce ----
// the copy in pinned host memory of a word of the loop-state block
template <class T>
__device__ __forceinline__ T* on_host(const Dev& D, const T* p) {
    return reinterpret_cast<T*>(D.loopHost + (reinterpret_cast<const char*>(p) - D.loopDev));
}

// mode 0: DFSPH density  err = sum(rho*/rho0)/n - 1          (DFSPH.cpp:696)
// mode 1: DFSPH divergence / IISPH error   err = sum/n      (DFSPH.cpp:896, IISph_M.cpp:353)
// mode 2: PCISPH  err = max error/rho0 (second partial)     (PciSph.cpp:344-350)
// Loop continuation (while err > tol || it < minIt; PCISPH err >= tol,
// PciSph.cpp:116), stopping at `cap`.
// Writes the scene's continuation flag to out (the active array itself, or
// the next iteration's buffer of the DFSPH loops; a scene already done stays
// done).  Every thread of the block calls it.
__device__ __forceinline__ void scene_reduce_block(const Dev& D, int sc, int mode, float tol, int minIt, int cap,
                                                   int* out) {
    __shared__ double lds[16];
    if (!D.active[sc]) {   // uniform per block
        if (threadIdx.x == 0 && out != D.active) {
            out[sc] = 0;
            *on_host(D, out + sc) = 0;
        }
        return;
    }
    int t0 = D.scenePadStart[sc] / TILE, t1 = D.scenePadStart[sc + 1] / TILE;
    __shared__ float ldsf[16];
    double s = 0.0;
    float mx = 0.0f;
    // each thread sums tiles t0 + tid, + 256, + 512, ... in that order; the
    // loads of eight of them are issued together (a larger block's further
    // threads have no part)
    for (int t = threadIdx.x < 256 ? t0 + (int)threadIdx.x : t1; t < t1; t += 256 * 8) {
        double v[8];
        float w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int tt = t + 256 * k;
            v[k] = tt < t1 ? D.partial[2 * tt] : 0.0;
            w[k] = (mode == 2 && tt < t1) ? (float)D.partial[2 * tt + 1] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (t + 256 * k < t1) s += v[k];
            mx = fmaxf(mx, w[k]);
        }
    }
    s = block_sum_256(s, lds);
    mx = block_max_256(mx, ldsf);
    if (threadIdx.x == 0) {
        int n = D.sceneCount[sc];
        double err = n > 0 ? s / n : 0.0;
        if (mode == 0) err = n > 0 ? err - 1.0 : 0.0;
        if (mode == 2) err = (double)mx;
        int it = D.iters[sc] + 1;
        D.iters[sc] = it;
        D.sceneErr[sc] = err;
        bool cont = (mode == 2 ? err >= (double)tol : err > (double)tol) || (it < minIt);
        if (cont && it >= cap) {
            cont = false;
            D.counters[C_COUNT - 1] = 1;  // max-iteration flag
        }
        out[sc] = cont ? 1 : 0;
        *on_host(D, out + sc) = cont ? 1 : 0;
        *on_host(D, D.iters + sc) = it;
        *on_host(D, D.sceneErr + sc) = err;
    }
}

// the loop's convergence test in front of a pass, scene b on block b: a pass that
// holds it has a block for every scene
__device__ __forceinline__ void loop_test(const Dev& D) {
    if (D.redMode >= 0 && (int)blockIdx.x < D.nscenes)
        scene_reduce_block(D, blockIdx.x, D.redMode, D.redTol, D.redMinIt, D.redCap, D.activeNext);
}

}  // namespace

}  // namespace sphgpu
