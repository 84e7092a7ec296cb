// The IISph class's header-consistent DFSPH (IISph.cpp:100-288
// DF_prepareAttribute, 816-1037 DF_constantDensitySolver, 1039-1217
// DF_divergenceFreeSolver), one thread per particle.
//
// Against the DFSPH class (solvers.hip) it differs in:
//   - a per-particle mass m = rho0 beta d^3 and rest density rho0 beta
//     (IISph.cpp:110-115); beta rides in the ksum array (reordered with the
//     particles, unused by this solver otherwise), the mass of each slot is
//     recomputed every step into pm;
//   - m_TH.adjustDensity (Dev::adjustDensity): the fluid-fluid density and
//     predicted-density terms use the particle's own mass (a number density);
//   - boundary terms use m_TH.boundaryDensity (Dev::boundaryDensity), which is
//     also every boundary particle's rest density, and boundary particles
//     carry their own density, alpha and kappa (bk = kappa/rho per boundary
//     particle), which the fluid's velocity pass reads;
//   - the divergence-free solve runs first, at the same positions, then the
//     constant-density solve, then updateFluids (the order of the commented
//     calls at IISph.cpp:59-60).
// Boundary particles find their neighbours once a step by scanning the 27
// cells around them (fluid through cellF, boundary through cellB, the
// reference's predicate, no pair with a particle of the same solid: every
// solid is rigid) and keep them in lists of their own; fluid particles use
// their neighbour lists.
//
// Bound: the latency of the neighbours' loads.  The lists are read in batches
// of gathers (each_fluid_lu, each_boundary_lu), one launch takes the fluid
// tiles and the boundary particles of a stiffness pass, and the convergence
// test runs in the velocity pass.  An iteration on 87,075 fluid and 33,312
// wall particles takes 33 us (114 us with one load at a time and every wall
// particle scanning its cells in every iteration).
#include "passes.h"

namespace sphgpu {

namespace {

__device__ __forceinline__ float rest_of(const Dev& D, int i, int ph) { return D.rho0[ph] * D.ksum[i]; }

// pair vector and the kernel gradient factor -|dW/dr|/r
struct Pair {
    float dx, dy, dz, r, g;
};
__device__ __forceinline__ Pair pair_of(const Dev& D, float4 a, float4 b) {
    Pair p;
    p.dx = a.x - b.x;
    p.dy = a.y - b.y;
    p.dz = a.z - b.z;
    p.r = fast_sqrt(dot3f(p.dx, p.dy, p.dz, p.dx, p.dy, p.dz));
    p.g = kernel_gradfac(p.r, D);
    return p;
}

// a gather record and one scalar of the same neighbour (mass, stiffness)
struct RecM {
    float4 x;
    float m;
};

// ---------------------------------------------------------------- masses ----
// m = rho0 beta v0 of every live slot (IISph.cpp:110-115)
__global__ __launch_bounds__(256) void k_idf_mass(Dev D) {
    const int tile = blockIdx.x, i = tile * TILE + threadIdx.x;
    if ((int)threadIdx.x >= D.tileValid[tile]) return;
    const int ph = (int)D.x[i].w;
    D.pm[i] = D.rho0[ph] * D.ksum[i] * D.v0;
}

// ------------------------------------------------------ DF_prepareAttribute --
// fluid density and alpha (IISph.cpp:143-200); publishes rho in v.w for the
// non-pressure acceleration pass
__global__ __launch_bounds__(256) void k_idf_prepare_fluid(Dev D) {
    float4 pa;
    const Slot s = slot_nb<1>(D, false, [&](int i) { pa = D.x[i]; });
    if (!s.live) return;
    const int i = s.i;
    const int ph = phase_of(pa);
    const float ma = D.pm[i], resta = rest_of(D, i, ph);
    const int c = s.c;
    Kahan rho;
    rho.init(ma * D.W0);
    float a1x = 0.f, a1y = 0.f, a1z = 0.f, a2 = 0.f;
    // (padding entries, the particle itself and the far dummy, are skipped:
    // adding a zero would change a compensated sum)
    each_fluid_lu<4>(D, s, nf_of(c), [&](int j) { return RecM{D.x[j], D.pm[j]}; }, [&](int j, RecM rec) {
        if (j == i) return;
        const Pair p = pair_of(D, pa, rec.x);
        const float mb = rec.m;
        rho.add((D.adjustDensity ? ma : mb) * kernel_W(p.r, D));     // IISph.cpp:163-164
        const float gm = p.g * mb;
        a1x += p.dx * gm; a1y += p.dy * gm; a1z += p.dz * gm;
        const float gs = gm * p.r;                                   // |dW/dr| m_b
        a2 += gs * gs;
    });
    each_boundary_lu<8>(D, s, nb_of(c), [&](int j) { return D.xb[j]; }, [&](int j, float4 pb) {
        if (j == D.nb) return;
        const Pair p = pair_of(D, pa, pb);
        rho.add(resta * pb.w * kernel_W(p.r, D));                     // IISph.cpp:187
        const float gm = p.g * D.boundaryDensity * pb.w;             // IISph.cpp:192
        a1x += p.dx * gm; a1y += p.dy * gm; a1z += p.dz * gm;
        if (D.anyDynamic && D.solids[D.bsolid[j]].dynamic) {          // IISph.cpp:193-195
            const float gs = gm * p.r;
            a2 += gs * gs;
        }
    });
    const float density = rho.s;
    float den = dot3f(a1x, a1y, a1z, a1x, a1y, a1z) + a2;
    if (den < 1.0e-6f) den = 1.0e-6f;
    D.rho[i] = density;
    D.alpha[i] = density / den;
    D.v[i].w = density;
}

// every fluid and boundary neighbour of boundary particle b, from the 27
// cells around it: fluid(j, pair), boundary(j, pair, V_j).  Candidates come
// four at a time (up to X_TAIL records past a run are read, and not used).
template <class FF, class FB>
__device__ __forceinline__ void boundary_stencil(const Dev& D, int b, float4 pa, FF&& fluid, FB&& bound) {
    const SceneGrid G = D.grids[D.bscene[b]];
    const int sa = D.bsolid[b];
    int cx, cy, cz;
    cell_of(G, pa, cx, cy, cz);
    for (int dz = -1; dz <= 1; ++dz) {
        const int z = cz + dz;
        if (z < 0 || z >= G.nz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            const int y = cy + dy;
            if (y < 0 || y >= G.ny) continue;
            const uint32_t k0 = key_of(G, D.rowRank, cx, y, z);
            const int2 rf = run3(D.cellF, k0, cx, G.nx, D.cellRuns);
            for (int j0 = rf.x; j0 < rf.y; j0 += 4) {
                float4 q[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = D.x[j0 + k];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (j0 + k < rf.y && dis_square_exact(pa, q[k]) < D.h2) fluid(j0 + k, pair_of(D, pa, q[k]));
            }
            if (D.nsolids < 2) continue;          // its own solid's particles only
            const int2 rb = run3(D.cellB, k0, cx, G.nx, D.cellRuns);
            for (int j = rb.x; j < rb.y; ++j) {
                if (j == b || D.bsolid[j] == sa) continue;
                const float4 pb = D.xb[j];
                if (dis_square_exact(pa, pb) < D.h2) bound(j, pair_of(D, pa, pb), pb.w);
            }
        }
    }
}

// the same neighbours in the same order from the lists k_idf_prepare_boundary
// keeps: fluid(j, pair, v*_j), boundary(j, pair, V_j, v_j)
template <class FF, class FB>
__device__ __forceinline__ void boundary_neighbours(const Dev& D, int b, float4 pa, FF&& fluid, FB&& bound) {
    const int c = D.bnCnt[b];
    if (c < 0) {
        boundary_stencil(D, b, pa, [&](int j, const Pair& p) { fluid(j, p, D.vs[j]); },
                         [&](int j, const Pair& p, float vol) { bound(j, p, vol, D.vb[j]); });
        return;
    }
    const int nf = c & 0xff, nb = c >> 8;
    const int4* lf = reinterpret_cast<const int4*>(D.bnF) + b;
    for (int g = 0; 4 * g < nf; ++g) {
        const int4 e = lf[(size_t)g * D.nb];
        // entries past the count are left from earlier steps: the first stands in
        const int j[4] = {e.x, 4 * g + 1 < nf ? e.y : e.x, 4 * g + 2 < nf ? e.z : e.x, 4 * g + 3 < nf ? e.w : e.x};
        Rec2 r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = Rec2{D.x[j[k]], D.vs[j[k]]};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (4 * g + k < nf) fluid(j[k], pair_of(D, pa, r[k].a), r[k].b);
    }
    for (int k = 0; k < nb; ++k) {
        const int j = D.bnB[nb_slot(k, b, D.nb)];
        const float4 pb = D.xb[j];
        bound(j, pair_of(D, pa, pb), pb.w, D.vb[j]);
    }
}

// boundary density and alpha (IISph.cpp:234-287); the mass of a boundary
// particle is boundaryDensity V_b (IISph.cpp:130).  Also keeps its neighbours
// in lists for the passes of the step's loops.
__global__ __launch_bounds__(256) void k_idf_prepare_boundary(Dev D) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= D.nb) return;
    const float4 pa = D.xb[b];
    const float ma = D.boundaryDensity * pa.w;
    Kahan rho;
    rho.init(ma * D.W0);
    float a2 = 0.0f;
    int nf = 0, nb = 0;
    boundary_stencil(D, b, pa,
        [&](int j, const Pair& p) {
            if (nf < BNF_CAP) D.bnF[nb_slot(nf, b, D.nb)] = j;
            ++nf;
            const float mf = D.pm[j];
            rho.add((D.adjustDensity ? ma : mf) * kernel_W(p.r, D));
            const float gs = p.g * p.r * mf;
            a2 += gs * gs;
        },
        [&](int j, const Pair& p, float vol) {
            if (nb < BNB_CAP) D.bnB[nb_slot(nb, b, D.nb)] = j;
            ++nb;
            rho.add(D.boundaryDensity * vol * kernel_W(p.r, D));
        });
    D.bnCnt[b] = nf <= BNF_CAP && nb <= BNB_CAP ? nf | nb << 8 : -1;
    const float density = rho.s;
    D.brho[b] = density;
    D.balpha[b] = density / (a2 < 1.0e-6f ? 1.0e-6f : a2);
}

// -------------------------------------------------------- solver passes ----
// mode 0: v_adv = v (the divergence solve starts from v, IISph.cpp:1056);
// mode 1: v = the divergence-free v_adv, v_adv = v + dt a_adv
// (IISph.cpp:833-836).  v_adv.w carries the particle's mass for the
// neighbours' gathers.
__global__ __launch_bounds__(256) void k_idf_vadv(Dev D, int mode) {
    const int tile = blockIdx.x, i = tile * TILE + threadIdx.x;
    if ((int)threadIdx.x >= D.tileValid[tile]) return;
    const float dt = D.dt[D.tileScene[tile]];
    if (mode == 0) {
        const float4 v = D.v[i];
        D.vs[i] = make_float4(v.x, v.y, v.z, D.pm[i]);
    } else {
        const float4 u = D.vs[i], a = D.f4a[i];
        D.v[i] = make_float4(u.x, u.y, u.z, D.rho[i]);
        D.vs[i] = make_float4(u.x + a.x * dt, u.y + a.y * dt, u.z + a.z * dt, u.w);
    }
}

// boundary particles' own stiffness, kappa/rho into bk:
// mode 0 density (IISph.cpp:849-904), mode 1 divergence (1069-1115)
__device__ __forceinline__ void kappa_boundary(const Dev& D, int b, int mode) {
    if (b >= D.nb) return;
    const int sc = D.bscene[b];
    if (!D.active[sc]) return;
    const float4 pa = D.xb[b], va = D.vb[b];
    const float ma = D.boundaryDensity * pa.w, rest = D.boundaryDensity;
    const bool adjust = mode == 0 && D.adjustDensity;
    float sf = 0.0f, sb = 0.0f;
    boundary_neighbours(D, b, pa,
        [&](int j, const Pair& p, float4 u) {
            sf += (adjust ? ma : u.w) * p.g * dot3f(va.x - u.x, va.y - u.y, va.z - u.z, p.dx, p.dy, p.dz);
        },
        [&](int j, const Pair& p, float vol, float4 u) {
            sb += vol * p.g * dot3f(va.x - u.x, va.y - u.y, va.z - u.z, p.dx, p.dy, p.dz);
        });
    const float dt = D.dt[sc], rho = D.brho[b];
    const float d = sf + D.boundaryDensity * sb;
    float kr;
    if (mode == 0) {
        float radv = rho + d * dt;
        if (radv < rest) radv = rest;
        kr = (radv - rest) / (dt * dt) * D.balpha[b] / rho;
    } else {
        const float dd = (d < 0.0f || (rho + d * dt) < rest) ? 0.0f : d;
        kr = dd * D.balpha[b] / dt / rho;
    }
    D.bk[b] = kr;
}

// Lanes a particle of the iterations' passes (each_fluid): with one, a wave
// waits for one batch of records after another.  A step of four iterations
// each, one lane / two: 8,000 particles 307 / 288 us, 88,704 448 / 418, 378,000
// 765 / 719, 864,000 1483 / 1374; the same bits.
constexpr int K = 2;

// fluid stiffness (mode 0 density, IISph.cpp:910-965; mode 1 divergence,
// 1120-1165) -> xk = (x, kappa/rho); partial sums of the loop's error:
// (rho_adv - rest)/rest (IISph.cpp:956-957), or Drho/Dt dt (1204-1207).
// Blocks past the tiles take the boundary particles (neither reads what the
// other writes).
__global__ __launch_bounds__(256 * K) void k_idf_kappa(Dev D, int mode, int tiles) {
    if ((int)blockIdx.x >= tiles) {
        kappa_boundary(D, ((int)blockIdx.x - tiles) * 256 * K + threadIdx.x, mode);
        return;
    }
    __shared__ double lds[4 * K], part[TILE];
    const int h = threadIdx.x % K;
    float4 pa, va;
    const Slot s = slot_nb<K>(D, true, [&](int i) { pa = D.x[i], va = D.vs[i]; }, tiles);
    if (!D.active[s.scene]) {   // uniform: a converged scene's tiles contribute nothing
        if (threadIdx.x == 0) D.partial[2 * s.tile] = 0.0;
        return;
    }
    double contrib = 0.0;
    if (s.live) {
        const int i = s.i;
        const int ph = phase_of(pa);
        const float ma = va.w, rest = rest_of(D, i, ph);
        const int c = s.c;
        const bool adjust = mode == 0 && D.adjustDensity;
        float sf = 0.0f, sb = 0.0f;
        // (weight g, v_ab.x_ab): the pair's term is their product
        each_fluid<K, 4>(D, s, h, nf_of(c), [&](int j) { return Rec2{D.x[j], D.vs[j]}; }, [&](int, const Rec2& rec) {
            const float4 u = rec.b;
            const Pair p = pair_of(D, pa, rec.a);
            return make_float2((adjust ? ma : u.w) * p.g,
                               dot3f(va.x - u.x, va.y - u.y, va.z - u.z, p.dx, p.dy, p.dz));
        }, [&](float2 t) { sf += t.x * t.y; });
        each_boundary<K, 4>(D, s, h, nb_of(c), [&](int j) { return Rec2{D.xb[j], D.vb[j]}; }, [&](int, const Rec2& rec) {
            const float4 pb = rec.a, u = rec.b;
            const Pair p = pair_of(D, pa, pb);
            return make_float2(pb.w * p.g, dot3f(va.x - u.x, va.y - u.y, va.z - u.z, p.dx, p.dy, p.dz));
        }, [&](float2 t) { sb += t.x * t.y; });
        const float dt = D.dt[s.scene], rho = D.rho[i];
        float kr;
        if (mode == 0) {
            float radv = rho + dt * (sf + D.boundaryDensity * sb);      // IISph.cpp:948
            if (radv < rest) radv = rest;
            kr = (radv - rest) / (dt * dt) * D.alpha[i] / rho;
            contrib = ((double)radv - (double)rest) / (double)rest;
        } else {
            float dd = sf + rest * sb;                                  // IISph.cpp:1156
            if (dd < 0.0f || (rho + dd * dt) < rest) dd = 0.0f;
            kr = dd * D.alpha[i] / dt / rho;
            contrib = (double)dd * (double)dt;
        }
        if (h == 0) D.xk[i] = make_float4(pa.x, pa.y, pa.z, kr);
    }
    const double sum = tile_sum<K>(contrib, part, lds);
    if (threadIdx.x == 0) D.partial[2 * s.tile] = sum;
}

// velocity pass of both loops (IISph.cpp:966-1001, 1166-1206):
// v_adv -= dt (sum_f m_b (k_a/rho_a + k_b/rho_b) gradW
//              + sum_b boundaryDensity V_b (k_a/rho_a + k_b/rho_b) gradW)
__global__ __launch_bounds__(256 * K) void k_idf_velocity(Dev D) {
    loop_test(D);   // on the stiffness pass's partial sums
    float4 pa;
    const Slot s = slot_nb<K>(D, true, [&](int i) { pa = D.xk[i]; });
    if (!s.live) return;
    const int i = s.i, h = threadIdx.x % K;
    const float ka = pa.w;
    const int c = s.c;
    float fx = 0.f, fy = 0.f, fz = 0.f, bx = 0.f, by = 0.f, bz = 0.f;
    // (x_ab, factor): the pair's term is their product
    each_fluid<K, 4>(D, s, h, nf_of(c), [&](int j) { return RecM{D.xk[j], D.pm[j]}; }, [&](int, const RecM& rec) {
        const Pair p = pair_of(D, pa, rec.x);
        return make_float4(p.dx, p.dy, p.dz, p.g * rec.m * (ka + rec.x.w));
    }, [&](float4 t) { fx += t.x * t.w; fy += t.y * t.w; fz += t.z * t.w; });
    each_boundary<K, 4>(D, s, h, nb_of(c), [&](int j) { return RecM{D.xb[j], D.bk[j]}; }, [&](int, const RecM& rec) {
        const Pair p = pair_of(D, pa, rec.x);
        return make_float4(p.dx, p.dy, p.dz, p.g * rec.x.w * (ka + rec.m));
    }, [&](float4 t) { bx += t.x * t.w; by += t.y * t.w; bz += t.z * t.w; });
    if (h != 0) return;
    const float dt = D.dt[s.scene], cb = dt * D.boundaryDensity;
    float4 v = D.vs[i];
    v.x -= dt * fx + cb * bx;
    v.y -= dt * fy + cb * by;
    v.z -= dt * fz + cb * bz;
    D.vs[i] = v;
}

inline int tiles_of(const Dev& D) { return D.npad / TILE; }
inline int bblocks(const Dev& D) { return (D.nb + 255) / 256; }

}  // namespace

void launch_idf_prepare(const Dev& D, hipStream_t st) {
    const int t = tiles_of(D);
    if (t > 0) {
        hipLaunchKernelGGL(k_idf_mass, dim3(t), dim3(256), 0, st, D);
        hipLaunchKernelGGL(k_idf_prepare_fluid, dim3(t), dim3(256), 0, st, D);
    }
    if (D.nb > 0) hipLaunchKernelGGL(k_idf_prepare_boundary, dim3(bblocks(D)), dim3(256), 0, st, D);
}

void launch_idf_vadv(const Dev& D, int mode, hipStream_t st) {
    if (tiles_of(D) > 0) hipLaunchKernelGGL(k_idf_vadv, dim3(tiles_of(D)), dim3(256), 0, st, D, mode);
}

void launch_idf_kappa(const Dev& D, int mode, hipStream_t st) {
    const int t = tiles_of(D), g = t + (D.nb + 256 * K - 1) / (256 * K);
    if (g > 0) hipLaunchKernelGGL(k_idf_kappa, dim3(g), dim3(256 * K), 0, st, D, mode, t);
}

void launch_idf_velocity(const Dev& D, hipStream_t st) {
    if (tiles_of(D) > 0) hipLaunchKernelGGL(k_idf_velocity, dim3(tiles_of(D)), dim3(256 * K), 0, st, D);
}

}  // namespace sphgpu
