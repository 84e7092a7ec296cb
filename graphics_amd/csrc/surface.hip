// Surface reconstruction on the device: the reference's offline surfacer
// (Source/re.c: surface_field::surface_setup / surface_aniso /
// surface_isotro, surface_field.cpp:8-226; marchingCubes,
// marching_cubes.cpp:45-120) as HIP kernels:
//
//   1. particles binned by a radix sort into cells of h_field = 2 r_h;
//   2. k_sf_aniso, four lanes per particle: Yu & Turk's weighted mean x_bar
//      (eq. 10, lambda = 1) and covariance (eq. 9) over the neighbours within
//      h_field (weights 1 - (r/h_field)^3, eq. 11), symmetric eigen
//      decomposition (cyclic Jacobi; equal to the SVD of the symmetric
//      positive covariance), singular values clamped to sigma0 / k_r and
//      scaled by k_s (eq. 15), G = U diag(1/sigma) U^T; fewer than N_e = 25
//      neighbours: G = k_n (3 - 2 n / N_e) I at the particle;
//   3. k_sf_field, one wave per block of 8 x 4 x 4 field nodes: det(G)
//      W(|G (p - x_bar)|) of every particle whose ellipsoid reaches the block,
//      summed in registers in particle order (float, as the reference's
//      RE_TYPE); the few particles whose box reaches further than one cell
//      from them, and all of them where the particles touch few nodes, are
//      added by k_sf_splat (one block per particle, FP32 atomics);
//   4. marching cubes: a count pass over units of nodes, an exclusive scan, a
//      pass writing triangles in cube order (x fastest, then y, then z).
#include "mc_table.h"
#include "sph_common.h"
#include "sphgpu.h"
#include "xfer.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

using namespace sphgpu;

namespace {

struct SurfParams {
    float fmin[3];        // field grid origin
    int fnum[3];          // field grid nodes per axis
    float cell;           // field grid spacing
    float gmin[3];        // particle grid origin
    int gnum[3];          // particle grid cells per axis
    float ginv;           // 1 / h_field
    float hfield, hfield2, hf3inv;
    float rh, rh2;        // kernel radius of the field (radius_h)
    int hcells;           // int(radius_h / cell)
    float ks, kr, kn, lambda;
    int Ne;
    float k1, k2, k3, k4; // spline constants times the particle volume
};

struct SurfRec {          // per particle: ellipsoid centre, symmetric G, det(G), box half-width
    float x, y, z, det;
    float g00, g01, g02, g11;
    float g12, g22;
    int ext, pad;
};

struct SurfBox {          // per particle: field nodes searched (lo..hi per axis)
    int lo[3], hi[3];
    short empty, far;     // no node of the grid; reaches further than one cell (k_sf_splat)
    int cut;              // the box may leave out nodes within the support
};

__device__ __forceinline__ int cell_axis(float v, float mn, float inv, int n) {
    int c = int((v - mn) * inv);
    return min(max(c, 0), n - 1);
}

// x: the caller's positions, three floats a particle
__global__ __launch_bounds__(256) void k_sf_keys(SurfParams S, const float* __restrict__ x, int n,
                                                 uint32_t* keys, uint32_t* vals) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const size_t q = 3 * (size_t)i;
    int cx = cell_axis(x[q], S.gmin[0], S.ginv, S.gnum[0]);
    int cy = cell_axis(x[q + 1], S.gmin[1], S.ginv, S.gnum[1]);
    int cz = cell_axis(x[q + 2], S.gmin[2], S.ginv, S.gnum[2]);
    keys[i] = (uint32_t)((cz * S.gnum[1] + cy) * S.gnum[0] + cx);
    vals[i] = (uint32_t)i;
}

__global__ __launch_bounds__(256) void k_sf_gather(const float* __restrict__ x, const uint32_t* __restrict__ vals,
                                                   int n, float4* xs) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    const size_t q = 3 * (size_t)vals[r];
    xs[r] = make_float4(x[q], x[q + 1], x[q + 2], 0.0f);
}

__global__ __launch_bounds__(256) void k_sf_fill_i2(int2* p, int n) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = make_int2(0, 0);
}

__global__ __launch_bounds__(256) void k_sf_ranges(const uint32_t* __restrict__ keys, int n, int2* ranges) {
    int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    uint32_t k = keys[r];
    if (r == 0 || keys[r - 1] != k) ranges[k].x = r;
    if (r == n - 1 || keys[r + 1] != k) ranges[k].y = r + 1;
}

// symmetric 3x3 eigen decomposition by cyclic Jacobi rotations (a fixed
// number of sweeps: deterministic); eigenvectors in the columns of V
__device__ void jacobi3(float a[3][3], float V[3][3], float ev[3]) {
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j) V[i][j] = i == j ? 1.0f : 0.0f;
    for (int sweep = 0; sweep < 8; ++sweep) {
        for (int p = 0; p < 2; ++p)
            for (int q = p + 1; q < 3; ++q) {
                const float apq = a[p][q];
                if (fabsf(apq) < 1e-30f) continue;
                const float theta = (a[q][q] - a[p][p]) / (2.0f * apq);
                const float t = (theta >= 0.0f ? 1.0f : -1.0f) / (fabsf(theta) + sqrtf(theta * theta + 1.0f));
                const float c = 1.0f / sqrtf(t * t + 1.0f), s = t * c;
                for (int k = 0; k < 3; ++k) {   // A <- A J (columns p, q)
                    const float akp = a[k][p], akq = a[k][q];
                    a[k][p] = c * akp - s * akq;
                    a[k][q] = s * akp + c * akq;
                }
                for (int k = 0; k < 3; ++k) {   // A <- J^T A (rows p, q)
                    const float apk = a[p][k], aqk = a[q][k];
                    a[p][k] = c * apk - s * aqk;
                    a[q][k] = s * apk + c * aqk;
                }
                for (int k = 0; k < 3; ++k) {
                    const float vkp = V[k][p], vkq = V[k][q];
                    V[k][p] = c * vkp - s * vkq;
                    V[k][q] = s * vkp + c * vkq;
                }
            }
    }
    for (int i = 0; i < 3; ++i) ev[i] = a[i][i];
}

// sum over the four lanes of a particle
__device__ __forceinline__ float quad_sum(float v) {
    v += __shfl_xor(v, 1, 64);
    return v + __shfl_xor(v, 2, 64);
}

// f(j, d, |d|^2) of the particles j != r of the 27 cells, every fourth one from
// `lane` on: the three cells of a row lie together (their keys are
// consecutive)
template <class F>
__device__ __forceinline__ void each_near(const SurfParams& S, const float4* __restrict__ xs,
                                          const int2* __restrict__ ranges, float4 pi, int r, int lane, F&& f) {
    const int cx = cell_axis(pi.x, S.gmin[0], S.ginv, S.gnum[0]);
    const int cy = cell_axis(pi.y, S.gmin[1], S.ginv, S.gnum[1]);
    const int cz = cell_axis(pi.z, S.gmin[2], S.ginv, S.gnum[2]);
    for (int z = max(cz - 1, 0); z <= min(cz + 1, S.gnum[2] - 1); ++z)
        for (int y = max(cy - 1, 0); y <= min(cy + 1, S.gnum[1] - 1); ++y) {
            int s = INT_MAX, e = 0;
            for (int x = max(cx - 1, 0); x <= min(cx + 1, S.gnum[0] - 1); ++x) {
                const int2 rg = ranges[(z * S.gnum[1] + y) * S.gnum[0] + x];
                if (rg.y > rg.x) {
                    s = min(s, rg.x);
                    e = max(e, rg.y);
                }
            }
            if (e <= s) continue;      // no particle in the row (s + lane would overflow)
            for (int j = s + lane; j < e; j += 4) {
                if (j == r) continue;
                const float4 pj = xs[j];
                const float dx = pj.x - pi.x, dy = pj.y - pi.y, dz = pj.z - pi.z;
                const float d2 = dx * dx + dy * dy + dz * dz;
                if (d2 > S.hfield2) continue;
                f(dx, dy, dz, d2);
            }
        }
}

// Whether the nodes p - e .. p + e + 1 hold all within w nodes of a point whose
// coordinate in nodes, cut towards zero, is p.  Above zero the next nodes outside are
// at least e + 1 away (at w itself the kernel is zero), below one less.
__device__ __forceinline__ bool holds(int e, float w, bool above) {
    return float(e) >= w + 1.0f || (above && float(e + 1) >= w * 0.99999f);
}

// The nodes with |G d| <= rh lie in the ellipsoid's bounding box, whose
// half-width along axis a is rh sqrt(sum_b (G^-1)_ab^2) (G symmetric); it is
// searched instead of the cube of half-width ext (the largest stretch along
// every axis), one node of margin added for rounding.
// A box is marked far where it reaches further than one particle cell from
// the particle itself, empty where it misses the grid.
__device__ __forceinline__ SurfBox box_of(const SurfParams& S, const SurfRec& o, float4 pi) {
    const float c00 = o.g11 * o.g22 - o.g12 * o.g12, c01 = o.g02 * o.g12 - o.g01 * o.g22;
    const float c02 = o.g01 * o.g12 - o.g02 * o.g11, c11 = o.g00 * o.g22 - o.g02 * o.g02;
    const float c12 = o.g01 * o.g02 - o.g00 * o.g12, c22 = o.g00 * o.g11 - o.g01 * o.g01;
    const float dg = o.g00 * c00 + o.g01 * c01 + o.g02 * c02;   // det G
    const float half[3] = {sqrtf(c00 * c00 + c01 * c01 + c02 * c02), sqrtf(c01 * c01 + c11 * c11 + c12 * c12),
                           sqrtf(c02 * c02 + c12 * c12 + c22 * c22)};
    const float xb[3] = {o.x, o.y, o.z}, x[3] = {pi.x, pi.y, pi.z};
    SurfBox b{};
    for (int a = 0; a < 3; ++a) {
        const long long p = int((xb[a] - S.fmin[a]) / S.cell);   // (an int even far outside the grid)
        int e = o.ext;
        bool whole = false;
        if (dg > 0.0f) {
            const float w = S.rh * half[a] / dg / S.cell;    // half-width in nodes
            if (w < float(o.ext)) e = min(o.ext, int(w) + 2);
            whole = holds(e, w, xb[a] >= S.fmin[a]);
        }
        if (!whole) b.cut = 1;
        b.lo[a] = int(max(p - e, 0LL));
        b.hi[a] = int(min(p + e + 1, (long long)S.fnum[a] - 1));
        if (b.hi[a] < b.lo[a]) b.empty = 1;
        const float l = S.fmin[a] + float(b.lo[a]) * S.cell, h = S.fmin[a] + float(b.hi[a]) * S.cell;
        if (!(l >= x[a] - S.hfield && h <= x[a] + S.hfield)) b.far = 1;
    }
    return b;
}

// Four lanes a particle, each every fourth candidate: with one lane 120,000
// particles are two waves a SIMD, which wait for one load after another (774
// us; 334 with four).
__global__ __launch_bounds__(256) void k_sf_aniso(SurfParams S, const float4* __restrict__ xs,
                                                  const int2* __restrict__ ranges, int first, int n, SurfRec* rec,
                                                  SurfBox* box, int* far, int* nfar) {
    const int r0 = first + int((blockIdx.x * 256 + threadIdx.x) >> 2), lane = threadIdx.x & 3;
    const int r = min(r0, n - 1);   // (every lane takes part in the sums)
    const float4 pi = xs[r];
    // pass 1: weighted mean (relative to the particle), neighbour count
    float sw = 0.0f, sx = 0.0f, sy = 0.0f, sz = 0.0f;
    int cnt = 0;
    each_near(S, xs, ranges, pi, r, lane, [&](float dx, float dy, float dz, float d2) {
        const float d = sqrtf(d2);
        const float w = 1.0f - d * d * d * S.hf3inv;
        sw += w; sx += w * dx; sy += w * dy; sz += w * dz;
        ++cnt;
    });
    sw = quad_sum(sw); sx = quad_sum(sx); sy = quad_sum(sy); sz = quad_sum(sz);
    cnt += __shfl_xor(cnt, 1, 64);
    cnt += __shfl_xor(cnt, 2, 64);
    SurfRec o;
    float sig0;
    if (cnt >= S.Ne) {
        const float mx = S.lambda * sx / sw, my = S.lambda * sy / sw, mz = S.lambda * sz / sw;
        // pass 2: covariance about x_bar (eq. 9 with x_bar of eq. 6)
        float c00 = 0.f, c01 = 0.f, c02 = 0.f, c11 = 0.f, c12 = 0.f, c22 = 0.f;
        each_near(S, xs, ranges, pi, r, lane, [&](float dx, float dy, float dz, float d2) {
            const float d = sqrtf(d2);
            const float w = 1.0f - d * d * d * S.hf3inv;
            const float ex = dx - mx, ey = dy - my, ez = dz - mz;
            c00 += w * ex * ex; c01 += w * ex * ey; c02 += w * ex * ez;
            c11 += w * ey * ey; c12 += w * ey * ez; c22 += w * ez * ez;
        });
        // (the four lanes of a particle have the same count: all are here)
        c00 = quad_sum(c00); c01 = quad_sum(c01); c02 = quad_sum(c02);
        c11 = quad_sum(c11); c12 = quad_sum(c12); c22 = quad_sum(c22);
        const float iw = 1.0f / sw;
        float A[3][3] = {{c00 * iw, c01 * iw, c02 * iw}, {c01 * iw, c11 * iw, c12 * iw}, {c02 * iw, c12 * iw, c22 * iw}};
        float V[3][3], ev[3];
        jacobi3(A, V, ev);
        // singular values in descending order (JAMA's SVD order)
        int o0 = 0, o1 = 1, o2 = 2;
        if (ev[o0] < ev[o1]) { int t = o0; o0 = o1; o1 = t; }
        if (ev[o1] < ev[o2]) { int t = o1; o1 = o2; o2 = t; }
        if (ev[o0] < ev[o1]) { int t = o0; o0 = o1; o1 = t; }
        float s0 = fmaxf(ev[o0], 0.0f), s1 = fmaxf(ev[o1], 0.0f), s2 = fmaxf(ev[o2], 0.0f);
        s1 = fmaxf(s1, s0 / S.kr);
        s2 = fmaxf(s2, s0 / S.kr);
        s0 *= S.ks; s1 *= S.ks; s2 *= S.ks;
        const float i0 = 1.0f / s0, i1 = 1.0f / s1, i2 = 1.0f / s2;
        const int oo[3] = {o0, o1, o2};
        const float is[3] = {i0, i1, i2};
        float G[3][3];
        for (int a = 0; a < 3; ++a)
            for (int b = 0; b < 3; ++b) {
                float g = 0.0f;
                for (int k = 0; k < 3; ++k) g += V[a][oo[k]] * is[k] * V[b][oo[k]];
                G[a][b] = g;
            }
        o.x = pi.x + mx; o.y = pi.y + my; o.z = pi.z + mz;
        o.det = i0 * i1 * i2;
        o.g00 = G[0][0]; o.g01 = 0.5f * (G[0][1] + G[1][0]); o.g02 = 0.5f * (G[0][2] + G[2][0]);
        o.g11 = G[1][1]; o.g12 = 0.5f * (G[1][2] + G[2][1]); o.g22 = G[2][2];
        sig0 = s0;
    } else {
        const float g = S.kn * (3.0f - 2.0f * float(cnt) / float(S.Ne));
        o.x = pi.x; o.y = pi.y; o.z = pi.z;
        o.det = g * g * g;
        o.g00 = g; o.g01 = 0.0f; o.g02 = 0.0f; o.g11 = g; o.g12 = 0.0f; o.g22 = g;
        sig0 = 1.0f / S.kn;
    }
    o.ext = int(float(S.hcells) * sig0);
    o.pad = cnt;
    if (lane != 0 || r0 >= n) return;
    const SurfBox bx = box_of(S, o, pi);
    rec[r] = o;
    box[r] = bx;
    if (bx.far && !bx.empty) far[atomicAdd(nfar, 1)] = r;
}

// the isotropic field's record: G = I at the particle, whole box
// (surface_field.cpp:45-75: half-width int(r_h / cell), W(|p - x|))
__device__ __forceinline__ void sphere_of(const SurfParams& S, float4 p, SurfRec& o, SurfBox& b) {
    const float xb[3] = {p.x, p.y, p.z};
    o = SurfRec{};
    o.x = p.x; o.y = p.y; o.z = p.z;
    o.det = o.g00 = o.g11 = o.g22 = 1.0f;
    o.ext = S.hcells;
    b = SurfBox{};
    for (int a = 0; a < 3; ++a) {
        const long long c = int((xb[a] - S.fmin[a]) / S.cell);
        if (!holds(S.hcells, S.rh / S.cell, xb[a] >= S.fmin[a])) b.cut = 1;
        b.lo[a] = int(max(c - S.hcells, 0LL));
        b.hi[a] = int(min(c + S.hcells + 1, (long long)S.fnum[a] - 1));
        if (b.hi[a] < b.lo[a]) b.empty = 1;
        const float l = S.fmin[a] + float(b.lo[a]) * S.cell, h = S.fmin[a] + float(b.hi[a]) * S.cell;
        if (!(l >= xb[a] - S.hfield && h <= xb[a] + S.hfield)) b.far = 1;
    }
}

__global__ __launch_bounds__(256) void k_sf_sphere(SurfParams S, const float4* __restrict__ xs, int n, SurfRec* rec,
                                                   SurfBox* box, int* far, int* nfar) {
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    SurfRec o;
    SurfBox b;
    sphere_of(S, xs[r], o, b);
    rec[r] = o;
    box[r] = b;
    if (b.far && !b.empty) far[atomicAdd(nfar, 1)] = r;
}

// cubic spline of the field (surface_field.cpp:233-250), times the particle volume
__device__ __forceinline__ float ker_field(const SurfParams& S, float r) {
    return r < 0.5f * S.rh ? S.k1 + S.k2 * r * r + S.k3 * r * r * r
                           : S.k4 * (S.rh - r) * (S.rh - r) * (S.rh - r);
}

// contribution of a particle to node (ix, iy, iz), 0 outside its support
__device__ __forceinline__ float node_value(const SurfParams& S, const SurfRec& o, int ix, int iy, int iz) {
    const float dx = S.fmin[0] + ix * S.cell - o.x;
    const float dy = S.fmin[1] + iy * S.cell - o.y;
    const float dz = S.fmin[2] + iz * S.cell - o.z;
    const float ux = o.g00 * dx + o.g01 * dy + o.g02 * dz;
    const float uy = o.g01 * dx + o.g11 * dy + o.g12 * dz;
    const float uz = o.g02 * dx + o.g12 * dy + o.g22 * dz;
    const float q2 = ux * ux + uy * uy + uz * uz;
    return q2 <= S.rh2 ? o.det * ker_field(S, sqrtf(q2)) : 0.0f;
}

// LDS accesses of the wave's lanes before it are done before those after it
// (a wave's LDS operations execute in order: this binds the compiler)
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// sqrtf of a squared distance, correctly rounded: one Newton step on the hardware's
// reciprocal root, its residual exact.  Compared on the card with sqrtf over every
// mantissa of even and odd binades: the same for every float from 2^-102 up.  Below
// 2^-100 the root of 2^-100: for the radii that come here (field_blocks) the spline
// is its value at 0 to the last place at both.  The hardware's own root is one
// place off in 15 cases of 100.  120,000 particles and 22 million nodes: the kernel
// with the hardware's root 1.72 ms, with this 1.83; the whole call 4.97 and 5.0, with
// sqrtf 5.30.
__device__ __forceinline__ float root(float x) {
    x = fmaxf(x, 0x1p-100f);
    const float y = __builtin_amdgcn_rsqf(x), g = x * y;
    return __builtin_fmaf(__builtin_fmaf(-g, g, x), 0.5f * y, g);
}

// Field nodes of one block of 8 x 4 x 4 a wave (two nodes a lane), four blocks
// along x a workgroup.  The wave looks through the particles of the cells that
// can reach its nodes, 64 at a time: each lane takes one, sets up u = G (p -
// x_bar), which is linear in the three node offsets, at the block's first node,
// and drops it where its box misses the block or |u| at the block's centre
// exceeds the support by more than |G| times the block's half diagonal.  The
// particles left are taken one after another, their u, G and det read from
// their lane into scalars, and added to the nodes in registers.  One wave alone
// sums a node, in particle order, so there are no atomics and the sums are the
// same every run.
// Bound by the arithmetic: 1.04 G wave instructions, nine tenths of the time,
// for 120,000 particles and 22 million nodes (1.83 ms).  Boxes of the particles
// over tiles of nodes in LDS took 2.5 ms (index arithmetic for each node, and
// a tile's edge cuts the boxes into parts that fill few lanes); one block per
// particle with FP32 atomics to memory 5.6 ms, at the rate of the atomics (46
// G/s).
constexpr int FB_X = 8, FB_Y = 4, FB_Z = 4, FB_WAVES = 4;
__global__ __launch_bounds__(64 * FB_WAVES) void k_sf_field(SurfParams S, const SurfRec* __restrict__ rec,
                                                          const SurfBox* __restrict__ box,
                                                          const int2* __restrict__ ranges, int tx, int ty,
                                                          float* __restrict__ field) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int bx = blockIdx.x % tx, by = (blockIdx.x / tx) % ty, bz = blockIdx.x / (tx * ty);
    // the wave's nodes [n0, n1]
    const int n0[3] = {(bx * FB_WAVES + wave) * FB_X, by * FB_Y, bz * FB_Z};
    const int n1[3] = {min(n0[0] + FB_X, S.fnum[0]) - 1, min(n0[1] + FB_Y, S.fnum[1]) - 1,
                       min(n0[2] + FB_Z, S.fnum[2]) - 1};
    if (n1[0] < n0[0]) return;      // past the grid (no barrier follows)
    const int ix = lane & 3, iy = (lane >> 2) & 3, iz = lane >> 4;
    const float kx = float(ix), ky = float(iy), kz = float(iz);
    float sum0 = 0.0f, sum1 = 0.0f;   // nodes ix and ix + 4
    // cells of the particles within one cell of the nodes along every axis
    // (a little more, for rounding); positions outside the cell grid are in
    // its border cells on both sides of the comparison
    int c0[3], c1[3];
    for (int a = 0; a < 3; ++a) {
        const float reach = S.hfield * 1.001f + S.cell;
        c0[a] = cell_axis(S.fmin[a] + float(n0[a]) * S.cell - reach, S.gmin[a], S.ginv, S.gnum[a]);
        c1[a] = cell_axis(S.fmin[a] + float(n1[a]) * S.cell + reach, S.gmin[a], S.ginv, S.gnum[a]);
    }
    const float first[3] = {S.fmin[0] + n0[0] * S.cell, S.fmin[1] + n0[1] * S.cell, S.fmin[2] + n0[2] * S.cell};
    const int ny = c1[1] - c0[1] + 1, rows = ny * (c1[2] - c0[2] + 1);
    for (int r0 = 0; r0 < rows; r0 += 64) {
        // a row of cells a lane: its particles lie together
        int s = INT_MAX, e = 0;
        if (r0 + lane < rows) {
            const int z = c0[2] + (r0 + lane) / ny, y = c0[1] + (r0 + lane) % ny;
            const int2* __restrict__ cells = ranges + (z * S.gnum[1] + y) * S.gnum[0];
            for (int x = c0[0]; x <= c1[0]; ++x) {
                const int2 rg = cells[x];
                if (rg.y > rg.x) {
                    s = min(s, rg.x);
                    e = max(e, rg.y);
                }
            }
        }
        for (unsigned long long in = __ballot(e > s); in; in &= in - 1) {
            const int row = __ffsll((long long)in) - 1;
            const int js = __builtin_amdgcn_readlane(s, row), je = __builtin_amdgcn_readlane(e, row);
            for (int j0 = js; j0 < je; j0 += 64) {
                const int j = j0 + lane;
                bool meets = false;
                SurfBox b{};
                if (j < je) {
                    b = box[j];
                    meets = !b.far && !b.empty;
                    for (int a = 0; a < 3; ++a) meets = meets && b.lo[a] <= n1[a] && b.hi[a] >= n0[a];
                }
                if (!__ballot(meets)) continue;
                const SurfRec o = rec[meets ? j : js];
                const float dx = first[0] - o.x, dy = first[1] - o.y, dz = first[2] - o.z;
                const float l_ux = o.g00 * dx + o.g01 * dy + o.g02 * dz, l_uy = o.g01 * dx + o.g11 * dy + o.g12 * dz,
                            l_uz = o.g02 * dx + o.g12 * dy + o.g22 * dz;
                const float l00 = o.g00 * S.cell, l01 = o.g01 * S.cell, l02 = o.g02 * S.cell, l11 = o.g11 * S.cell,
                            l12 = o.g12 * S.cell, l22 = o.g22 * S.cell;
                // |G v| <= (largest absolute row sum) |v|; half diagonal
                // sqrt(3.5^2 + 1.5^2 + 1.5^2) < 4.1 nodes
                const float vx = l_ux + 3.5f * l00 + 1.5f * l01 + 1.5f * l02,
                            vy = l_uy + 3.5f * l01 + 1.5f * l11 + 1.5f * l12,
                            vz = l_uz + 3.5f * l02 + 1.5f * l12 + 1.5f * l22;
                const float norm = fmaxf(fmaxf(fabsf(l00) + fabsf(l01) + fabsf(l02), fabsf(l01) + fabsf(l11) + fabsf(l12)),
                                         fabsf(l02) + fabsf(l12) + fabsf(l22));
                const float far = S.rh + 4.11f * norm;
                meets = meets && vx * vx + vy * vy + vz * vz <= 1.001f * far * far;
                const unsigned long long cut = __ballot(b.cut != 0);
                for (unsigned long long m = __ballot(meets); m; m &= m - 1) {
                    const int p = __ffsll((long long)m) - 1;
                    const float a00 = lane_value(l00, p), a01 = lane_value(l01, p), a02 = lane_value(l02, p),
                                a11 = lane_value(l11, p), a12 = lane_value(l12, p), a22 = lane_value(l22, p),
                                det = lane_value(o.det, p);
                    float ux = kx * a00 + lane_value(l_ux, p), uy = kx * a01 + lane_value(l_uy, p),
                          uz = kx * a02 + lane_value(l_uz, p);
                    ux += ky * a01 + kz * a02;
                    uy += ky * a11 + kz * a12;
                    uz += ky * a12 + kz * a22;
                    const float wx = ux + 4.0f * a00, wy = uy + 4.0f * a01, wz = uz + 4.0f * a02;
                    const float q0 = ux * ux + uy * uy + uz * uz, q1 = wx * wx + wy * wy + wz * wz;
                    bool in0 = q0 <= S.rh2, in1 = q1 <= S.rh2;
                    if (cut >> p & 1) {   // uniform: only the nodes of the box
                        bool yz = true;
                        for (int a = 1; a < 3; ++a) {
                            const int at = n0[a] + (a == 1 ? iy : iz);
                            yz = yz && at >= __builtin_amdgcn_readlane(b.lo[a], p) && at <= __builtin_amdgcn_readlane(b.hi[a], p);
                        }
                        const int lo = __builtin_amdgcn_readlane(b.lo[0], p), hi = __builtin_amdgcn_readlane(b.hi[0], p);
                        in0 = in0 && yz && n0[0] + ix >= lo && n0[0] + ix <= hi;
                        in1 = in1 && yz && n0[0] + ix + 4 >= lo && n0[0] + ix + 4 <= hi;
                    }
                    if (in0) sum0 += det * ker_field(S, root(q0));
                    if (in1) sum1 += det * ker_field(S, root(q1));
                }
            }
        }
    }
    if (n0[1] + iy > n1[1] || n0[2] + iz > n1[2]) return;
    float* const out = field + ((size_t)(n0[2] + iz) * S.fnum[1] + n0[1] + iy) * S.fnum[0] + n0[0];
    if (n0[0] + ix <= n1[0]) out[ix] = sum0;
    if (n0[0] + ix + 4 <= n1[0]) out[ix + 4] = sum1;
}

// a block's particle over the nodes of its box, added to the field with atomics
__device__ __forceinline__ void splat(const SurfParams& S, const SurfRec& o, const SurfBox& b,
                                      float* __restrict__ field) {
    const int nx = b.hi[0] - b.lo[0] + 1, ny = b.hi[1] - b.lo[1] + 1, nz = b.hi[2] - b.lo[2] + 1;
    const int total = b.empty ? 0 : nx * ny * nz;
    for (int t = threadIdx.x; t < total; t += 256) {
        const int ix = b.lo[0] + t % nx, iy = b.lo[1] + (t / nx) % ny, iz = b.lo[2] + t / (nx * ny);
        const float v = node_value(S, o, ix, iy, iz);
        if (v != 0.0f) atomicAdd(&field[((size_t)iz * S.fnum[1] + iy) * S.fnum[0] + ix], v);
    }
}

// One block per particle: every particle (list null, after the field was cleared),
// or the listed far ones, whose box reaches past the cells a block of nodes looks
// through, after the blocks are written.
__global__ __launch_bounds__(256) void k_sf_splat(SurfParams S, const SurfRec* __restrict__ rec,
                                                  const SurfBox* __restrict__ box, const int* __restrict__ list,
                                                  const int* __restrict__ count, int n, float* __restrict__ field) {
    const int m = list ? *count : n;
    for (int q = blockIdx.x; q < m; q += gridDim.x) {
        const int p = list ? list[q] : q;
        splat(S, rec[p], box[p], field);
    }
}

// The same for spheres, straight from the caller's positions: binning them costs
// more than the splat of few nodes.  Isotropic calls with their field read, MI355X:
// 4,000 particles at 4 nodes a radius 136 -> 81 us, 15,000 290 -> 229.
__global__ __launch_bounds__(256) void k_sf_splat_spheres(SurfParams S, const float* __restrict__ x, int n,
                                                          float* __restrict__ field) {
    for (int p = blockIdx.x; p < n; p += gridDim.x) {
        const size_t q = 3 * (size_t)p;
        SurfRec o;
        SurfBox b;
        sphere_of(S, make_float4(x[q], x[q + 1], x[q + 2], 0.0f), o, b);
        splat(S, o, b, field);
    }
}

struct McTable {
    unsigned short edges[256];
    signed char tris[256][16];
    unsigned char ntris[256];
};
__constant__ McTable c_mc;

// Marching cubes.  Cubes are numbered by their lowest node, n = ix + nx (iy +
// ny iz) (the nodes of the upper faces have none), triangles lie in that
// order.  A wave takes MC_UNIT nodes in chunks of 64: it loads the four node
// rows of its cubes and ballots "below iso", so a cube's case is eight bits of
// four masks and a chunk the surface does not cross is skipped after four
// loads and compares.  One pass counts the triangles of each unit, the units
// are scanned, and the second pass writes those of the units that have any, a
// lane a vertex, so that the stores are contiguous.
// Bound by the field's transfer to the device; of the kernels by reading the
// field.  9.5 million nodes, 0.2 million triangles (MI355X): a case and a
// count for each cube, a scan over all cubes and a thread a cube took 34 + 73
// + 59 us.
constexpr int MC_CHUNKS = 8;
constexpr int MC_UNIT = 64 * MC_CHUNKS;

struct McGrid {
    int nx, ny, nz;
    size_t nodes;
    float iso, mn[3], cell;
};

struct McMasks {          // "below iso" of the nodes n.. of a chunk and of those one further
    uint64_t lo[4], hi[4];   // rows (0, 0), (+y), (+z), (+y +z)
};

__device__ __forceinline__ size_t mc_row(const McGrid& G, int r) {
    return (r & 1 ? (size_t)G.nx : 0) + (r & 2 ? (size_t)G.nx * G.ny : 0);
}
// node n + the offset of row r; beyond the grid, where no cube is, its last node
__device__ __forceinline__ float mc_load(const McGrid& G, const float* __restrict__ f, size_t n, int r) {
    const size_t k = n + mc_row(G, r);
    return f[k < G.nodes ? k : G.nodes - 1];
}

// the masks of chunk k from all of a unit's loads
__device__ __forceinline__ void mc_unit(const McGrid& G, const float* __restrict__ f, size_t base, int lane,
                                        uint64_t (&m)[MC_CHUNKS][4], uint32_t& last) {
    float v[MC_CHUNKS][4];
#pragma unroll
    for (int k = 0; k < MC_CHUNKS; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[k][r] = mc_load(G, f, base + 64 * k + lane, r);
    // the node after the unit in each row: lanes 0..3
    const float e = mc_load(G, f, base + MC_UNIT, lane & 3);
#pragma unroll
    for (int k = 0; k < MC_CHUNKS; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) m[k][r] = __ballot(v[k][r] < G.iso);
    last = (uint32_t)__ballot(e < G.iso) & 15u;
}
__device__ __forceinline__ bool mc_masks(const uint64_t (&m)[MC_CHUNKS][4], uint32_t last, int k, McMasks& M) {
    uint64_t any = 0, all = ~0ull;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint64_t next = k + 1 < MC_CHUNKS ? m[k + 1 < MC_CHUNKS ? k + 1 : k][r] & 1ull : (last >> r) & 1u;
        M.lo[r] = m[k][r];
        M.hi[r] = (m[k][r] >> 1) | (next << 63);
        any |= M.lo[r] | M.hi[r];
        all &= M.lo[r] & M.hi[r];
    }
    return any != 0 && all != ~0ull;
}
// The cube's case: bit k for corner k; the corners' (x, y, z) offsets in order
// are (0,0,0) (0,0,1) (0,1,1) (0,1,0) (1,0,0) (1,0,1) (1,1,1) (1,1,0)
__device__ __forceinline__ int mc_case(const McMasks& M, int lane) {
    const int row[4] = {0, 2, 3, 1};
    int ci = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) ci |= (int((M.lo[row[k]] >> lane) & 1) << k) | (int((M.hi[row[k]] >> lane) & 1) << (4 + k));
    return ci;
}
struct McNode {
    int ix, iy, iz;
};
// position of node base + d (d < 2 MC_UNIT); base's own is wave-uniform
__device__ __forceinline__ McNode mc_node(const McGrid& G, size_t base, uint32_t d) {
    const uint64_t row = base / (uint32_t)G.nx;
    const uint32_t x = uint32_t(base - row * (uint32_t)G.nx) + d, up = x / (uint32_t)G.nx;
    const uint32_t y = uint32_t(row % (uint32_t)G.ny) + up, uz = y / (uint32_t)G.ny;
    return McNode{int(x - up * (uint32_t)G.nx), int(y - uz * (uint32_t)G.ny), int(uint32_t(row / (uint32_t)G.ny) + uz)};
}
__device__ __forceinline__ bool mc_cube(const McGrid& G, const McNode& p) {
    return p.ix < G.nx - 1 && p.iy < G.ny - 1 && p.iz < G.nz - 1;
}

__global__ __launch_bounds__(256) void k_mc_count(McGrid G, const float* __restrict__ f, int units,
                                                  uint32_t* __restrict__ count) {
    const int u = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (u >= units) return;
    const size_t base = (size_t)u * MC_UNIT;
    uint64_t m[MC_CHUNKS][4];
    uint32_t last, nt = 0;
    mc_unit(G, f, base, lane, m, last);
#pragma unroll
    for (int k = 0; k < MC_CHUNKS; ++k) {
        McMasks M;
        if (!mc_masks(m, last, k, M)) continue;
        const int ci = mc_case(M, lane);
        if (ci != 0 && ci != 255 && mc_cube(G, mc_node(G, base, 64 * k + lane))) nt += c_mc.ntris[ci];
    }
    for (int o = 32; o > 0; o >>= 1) nt += __shfl_xor(nt, o, 64);
    if (lane == 0) {
        count[u] = nt;
        if (u == units - 1) count[units] = 0;   // the total after the scan
    }
}

__global__ __launch_bounds__(256) void k_mc_emit(McGrid G, const float* __restrict__ f, int units,
                                                 const uint32_t* __restrict__ offset, float* __restrict__ out,
                                                 long long cap) {
    __shared__ uint16_t sTri[4][64 * 5];   // a chunk's triangles: lane * 8 + number in the cube
    __shared__ uint8_t sCase[4][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int u = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + w);
    if (u >= units) return;
    long long first = offset[u];
    if (offset[u + 1] == (uint32_t)first) return;
    const size_t base = (size_t)u * MC_UNIT;
    uint64_t m[MC_CHUNKS][4];
    uint32_t last;
    mc_unit(G, f, base, lane, m, last);
    const int off[8][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 1}, {0, 1, 0}, {1, 0, 0}, {1, 0, 1}, {1, 1, 1}, {1, 1, 0}};
    // an edge's corners, the one with the lower node first
    const int E[12][2] = {{0, 1}, {1, 2}, {3, 2}, {0, 3}, {4, 5}, {5, 6}, {7, 6}, {4, 7}, {0, 4}, {1, 5}, {2, 6}, {3, 7}};
#pragma unroll
    for (int k = 0; k < MC_CHUNKS; ++k) {
        McMasks M;
        if (!mc_masks(m, last, k, M)) continue;
        const int ci = mc_case(M, lane);
        int nt = 0;
        if (ci != 0 && ci != 255 && mc_cube(G, mc_node(G, base, 64 * k + lane))) nt = c_mc.ntris[ci];
        int incl = nt;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        const int total = __shfl(incl, 63, 64);
        sCase[w][lane] = (uint8_t)ci;
        for (int t = 0; t < nt; ++t) sTri[w][incl - nt + t] = uint16_t(lane * 8 + t);
        wave_order();
        for (int q = lane; q < 3 * total; q += 64) {
            const int tri = q / 3, at = q - 3 * tri;
            if (first + tri >= cap) break;
            const int code = sTri[w][tri], owner = code >> 3;
            const int e = c_mc.tris[sCase[w][owner]][3 * (code & 7) + at];
            const McNode p = mc_node(G, base, 64 * k + owner);
            // The edge's vertex by linear interpolation from its lower node,
            // with node positions from integer indices: the cubes around an
            // edge compute the same vertex (marching_cubes.cpp:40-41)
            const int a = E[e][0], b = E[e][1];
            const size_t n = base + 64 * k + owner, sy = G.nx, sz = (size_t)G.nx * G.ny;
            const float va = f[n + off[a][0] + off[a][1] * sy + off[a][2] * sz];
            const float vb = f[n + off[b][0] + off[b][1] * sy + off[b][2] * sz];
            const float mu = (G.iso - va) / (vb - va);
            const float ax = G.mn[0] + float(p.ix + off[a][0]) * G.cell, ay = G.mn[1] + float(p.iy + off[a][1]) * G.cell,
                        az = G.mn[2] + float(p.iz + off[a][2]) * G.cell;
            const float bx = G.mn[0] + float(p.ix + off[b][0]) * G.cell, by = G.mn[1] + float(p.iy + off[b][1]) * G.cell,
                        bz = G.mn[2] + float(p.iz + off[b][2]) * G.cell;
            float* o = out + 9 * (first + tri) + 3 * at;
            o[0] = ax + mu * (bx - ax);
            o[1] = ay + mu * (by - ay);
            o[2] = az + mu * (bz - az);
        }
        wave_order();
        first += total;
    }
}

}  // namespace

struct SurfRecs {          // records in cell order and the particle of each
    SurfRec* rec = nullptr;
    uint32_t* vals = nullptr;
    int cap = 0;
};

struct sphgpu_surfacer {
    SurfParams S{};
    double fmin[3], cell;
    int fnum[3];
    size_t nfield = 0, ncells = 0;
    hipStream_t st = nullptr;
    float* field = nullptr;
    int cap = 0;
    float* x = nullptr;            // positions as given
    float4* xs = nullptr;          // by cell
    uint32_t* keys = nullptr;
    int2* ranges = nullptr;
    SurfRecs spheres, ellipsoids;  // (apart: the last aniso call's stay for surfacer_particles)
    SurfBox* box = nullptr;
    int* far = nullptr;            // far particles' indices, then their number at [cap]
    HostRing ring;                 // staging of transfers
    void* sortMem = nullptr;
    SortScratch sort{};
    int keyBits = 1;
    uint32_t* mcCount = nullptr;
    uint32_t* mcTmp = nullptr;
    float* mcOut = nullptr;        // triangles
    long long mcOutCap = 0;
    int nrec = 0;                  // particles of the ellipsoids
    std::string err;
};

namespace {

int sfail(sphgpu_surfacer* s, int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    if (s) s->err = buf;
    return code;
}

#define SCHECK(s, expr)                                                                    \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess) return sfail(s, SPHGPU_E_DEVICE, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)

int ensure_particles(sphgpu_surfacer* s, int n) {
    if (s->cap > 0 && n <= s->cap) return 0;
    (void)hipFree(s->x); (void)hipFree(s->xs); (void)hipFree(s->keys);
    (void)hipFree(s->box); (void)hipFree(s->far); (void)hipFree(s->sortMem);
    s->cap = 0;
    s->box = nullptr; s->far = nullptr;
    s->x = nullptr; s->xs = nullptr; s->keys = nullptr; s->sortMem = nullptr;
    const int cap = std::max(n, 1024);
    SCHECK(s, hipMalloc(&s->x, 3 * sizeof(float) * cap));
    SCHECK(s, hipMalloc(&s->xs, sizeof(float4) * cap));
    SCHECK(s, hipMalloc(&s->keys, sizeof(uint32_t) * cap));
    SCHECK(s, hipMalloc(&s->box, sizeof(SurfBox) * cap));
    SCHECK(s, hipMalloc(&s->far, sizeof(int) * (size_t(cap) + 1)));
    SCHECK(s, hipMalloc(&s->sortMem, sort_scratch_bytes(cap)));
    sort_scratch_bind(s->sort, s->sortMem, cap);
    s->cap = cap;
    return 0;
}

void free_records(SurfRecs& r) {
    (void)hipFree(r.rec); (void)hipFree(r.vals);
    r = SurfRecs{};
}

int ensure_records(sphgpu_surfacer* s, SurfRecs& r, int n) {
    if (r.cap > 0 && n <= r.cap) return 0;
    free_records(r);
    const int cap = std::max(n, 1024);
    SCHECK(s, hipMalloc(&r.rec, sizeof(SurfRec) * cap));
    SCHECK(s, hipMalloc(&r.vals, sizeof(uint32_t) * cap));
    r.cap = cap;
    return 0;
}

// Blocks of nodes where the particles touch many nodes; where they touch few,
// the search through the particles takes longer than the atomics, and for spheres
// the binning too, which they need for it alone.  Field calls (MI355X, us: one
// block per particle / blocks of nodes), n particles, r_h = c nodes: anisotropic
// 60,000, c 8: 3201 / 1698; 60,000, c 4: 896 / 772; 15,000, c 6: 570 / 576; 30,000, c 4:
// 668 / 539; 4,000, c 8: 446 / 411; 8,000, c 6: 465 / 444; 15,000, c 4: 419 / 443; 4,000,
// c 6: 335 / 403; isotropic 15,000, c 8: 380 / 236; 30,000, c 6: 337 / 257; 8,000, c 8:
// 210 / 187; 60,000, c 4: 530 / 601; 15,000, c 6: 177 / 200; 4,000, c 8: 115 / 145.  (A
// radius under 2^-30: see root.  A thin grid of nearly 2^31 nodes can have more
// blocks than a launch holds.)
constexpr long long MAX_THREADS = 1LL << 31;   // of a launch (one of 2^32 is cut to its low 32 bits)
struct FieldGrid {
    long long x, y, z;
    long long blocks() const { return x * y * z; }
};
FieldGrid field_grid(const sphgpu_surfacer* s) {
    return {(s->fnum[0] + FB_X * FB_WAVES - 1) / (FB_X * FB_WAVES), (s->fnum[1] + FB_Y - 1) / FB_Y,
            (s->fnum[2] + FB_Z - 1) / FB_Z};
}
bool field_blocks(const sphgpu_surfacer* s, long long n, bool aniso) {
    const double c = s->S.hcells;
    return c >= 4.0 && double(n) * c * c * c >= (aniso ? 2.0e6 : 4.0e6) && s->S.rh >= 0x1p-30f &&
           field_grid(s).blocks() <= MAX_THREADS / (64 * FB_WAVES);
}

void launch_field(sphgpu_surfacer* s, const SurfRecs& r) {
    const FieldGrid g = field_grid(s);
    hipLaunchKernelGGL(k_sf_field, dim3(unsigned(g.blocks())), dim3(64 * FB_WAVES), 0, s->st, s->S,
                       (const SurfRec*)r.rec, (const SurfBox*)s->box, (const int2*)s->ranges, int(g.x), int(g.y),
                       s->field);
}

// the field of n particles: binned, ellipsoids (aniso) or spheres, tiles
int field_of(sphgpu_surfacer* s, long long n, const float* xyz, bool aniso) {
    if (n < 0 || (n > 0 && !xyz)) return sfail(s, SPHGPU_E_ARG, "bad particle array");
    if (n > (1 << 30)) return sfail(s, SPHGPU_E_CAPACITY, "too many particles");
    if (int rc = ensure_particles(s, int(n))) return rc;
    for (long long i = 0; i < n;) {   // blocks of particles, without a branch for each
        const long long end = std::min(n, i + 1024);
        bool ok = true;
        for (long long k = 3 * i; k < 3 * end; ++k) ok &= std::isfinite(xyz[k]);
        for (; !ok && i < end; ++i)
            if (!std::isfinite(xyz[3 * i]) || !std::isfinite(xyz[3 * i + 1]) || !std::isfinite(xyz[3 * i + 2]))
                return sfail(s, SPHGPU_E_ARG, "non-finite position %lld", i);
        i = end;
    }
    SCHECK(s, s->ring.to_device(s->x, xyz, 3 * sizeof(float) * size_t(n), s->st));
    // (an isotropic call of as many particles leaves the last aniso call's records)
    if (aniso || n != s->nrec) s->nrec = 0;
    const int blocks = int((n + 255) / 256);
    const bool inBlocks = field_blocks(s, n, aniso);
    // (a launch of 2^32 threads or more is cut: blocks take several particles from there)
    const dim3 splatGrid(unsigned(std::min<long long>(n, MAX_THREADS / 256)));
    if (!inBlocks) SCHECK(s, hipMemsetAsync(s->field, 0, sizeof(float) * s->nfield, s->st));
    if (!inBlocks && !aniso) {
        if (n > 0)
            hipLaunchKernelGGL(k_sf_splat_spheres, splatGrid, dim3(256), 0, s->st, s->S, (const float*)s->x, int(n),
                               s->field);
        SCHECK(s, hipGetLastError());
        SCHECK(s, hipStreamSynchronize(s->st));
        return 0;
    }
    SurfRecs& recs = aniso ? s->ellipsoids : s->spheres;
    if (int rc = ensure_records(s, recs, int(n))) return rc;
    int* const nfar = s->far + s->cap;
    SCHECK(s, hipMemsetAsync(nfar, 0, sizeof(int), s->st));
    if (n > 0) {
        hipLaunchKernelGGL(k_sf_keys, dim3(blocks), dim3(256), 0, s->st, s->S, (const float*)s->x, int(n), s->keys,
                           recs.vals);
        radix_sort_pairs(s->keys, recs.vals, int(n), s->keyBits, s->sort, s->st);
        hipLaunchKernelGGL(k_sf_gather, dim3(blocks), dim3(256), 0, s->st, (const float*)s->x,
                           (const uint32_t*)recs.vals, int(n), s->xs);
    }
    hipLaunchKernelGGL(k_sf_fill_i2, dim3(int((s->ncells + 255) / 256)), dim3(256), 0, s->st, s->ranges, int(s->ncells));
    if (n > 0) {
        hipLaunchKernelGGL(k_sf_ranges, dim3(blocks), dim3(256), 0, s->st, (const uint32_t*)s->keys, int(n), s->ranges);
        if (aniso)
            for (long long i = 0; i < n; i += MAX_THREADS / 4)
                hipLaunchKernelGGL(k_sf_aniso, dim3(unsigned((4 * std::min(n - i, MAX_THREADS / 4) + 255) / 256)),
                                   dim3(256), 0, s->st, s->S, (const float4*)s->xs, (const int2*)s->ranges, int(i),
                                   int(n), recs.rec, s->box, s->far, nfar);
        else
            hipLaunchKernelGGL(k_sf_sphere, dim3(blocks), dim3(256), 0, s->st, s->S, (const float4*)s->xs, int(n),
                               recs.rec, s->box, s->far, nfar);
    }
    if (!inBlocks) {
        if (n > 0)
            hipLaunchKernelGGL(k_sf_splat, splatGrid, dim3(256), 0, s->st, s->S, (const SurfRec*)recs.rec,
                               (const SurfBox*)s->box, (const int*)nullptr, (const int*)nullptr, int(n), s->field);
    } else {
        launch_field(s, recs);
        if (n > 0)
            hipLaunchKernelGGL(k_sf_splat, dim3(unsigned(std::min<long long>(n, 1024))), dim3(256), 0, s->st, s->S,
                               (const SurfRec*)recs.rec, (const SurfBox*)s->box, (const int*)s->far, (const int*)nfar, 0,
                               s->field);
    }
    SCHECK(s, hipGetLastError());
    SCHECK(s, hipStreamSynchronize(s->st));
    if (aniso) s->nrec = int(n);
    return 0;
}

int upload_table(sphgpu_surfacer* s) {
    const mctable::Table& t = mctable::table();
    McTable m{};
    std::memcpy(m.edges, t.edges, sizeof(m.edges));
    for (int c = 0; c < 256; ++c) {
        m.ntris[c] = t.ntris[c];
        for (int k = 0; k < 16; ++k) m.tris[c][k] = t.tris[c][k];
    }
    SCHECK(s, hipMemcpyToSymbolAsync(HIP_SYMBOL(c_mc), &m, sizeof(m), 0, hipMemcpyHostToDevice, s->st));
    SCHECK(s, hipStreamSynchronize(s->st));
    return 0;
}

}  // namespace

extern "C" {

int sphgpu_marching_cubes_table(unsigned short* edges, unsigned char* ntris, signed char* tris) {
    const mctable::Table& t = mctable::table();
    if (edges) std::memcpy(edges, t.edges, sizeof(t.edges));
    if (ntris) std::memcpy(ntris, t.ntris, sizeof(t.ntris));
    if (tris)
        for (int c = 0; c < 256; ++c) std::memcpy(tris + 16 * c, t.tris[c], 16);
    return SPHGPU_OK;
}

int sphgpu_surfacer_create(const float mn[3], const float mx[3], float radius_p, float radius_h, float cell_size,
                           sphgpu_surfacer** out) {
    if (!mn || !mx || !out) return SPHGPU_E_ARG;
    *out = nullptr;
    if (!(radius_p > 0) || !(radius_h > 0) || !(cell_size > 0)) return SPHGPU_E_ARG;
    for (int a = 0; a < 3; ++a)
        if (!(mx[a] > mn[a])) return SPHGPU_E_ARG;
    auto* s = new sphgpu_surfacer();
    SurfParams& S = s->S;
    // surface_setup (surface_field.cpp:8-43), in double on the host
    const double rp = radius_p, rh = radius_h, cell = cell_size, vol = rp * rp * rp, hf = 2.0 * rh;
    size_t nf = 1, nc = 1;
    for (int a = 0; a < 3; ++a) {
        s->fmin[a] = double(mn[a]) - rh * 0.75;
        s->fnum[a] = int((double(mx[a]) - double(mn[a]) + rh * 1.5) / cell) + 1;
        S.fmin[a] = float(s->fmin[a]);
        S.fnum[a] = s->fnum[a];
        nf *= size_t(s->fnum[a]);
        S.gmin[a] = float(double(mn[a]) - hf * 1.25);
        S.gnum[a] = int((double(mx[a]) - double(mn[a]) + hf * 2.5) / hf) + 1;
        nc *= size_t(S.gnum[a]);
    }
    if (nf > (size_t(1) << 31) || nc > (size_t(1) << 30)) {
        delete s;
        return SPHGPU_E_CAPACITY;
    }
    s->cell = cell;
    s->nfield = nf;
    s->ncells = nc;
    S.cell = float(cell);
    S.ginv = float(1.0 / hf);
    S.hfield = float(hf);
    S.hfield2 = float(hf * hf);
    S.hf3inv = float(1.0 / (hf * hf * hf));
    S.rh = float(rh);
    S.rh2 = float(rh * rh);
    S.hcells = int(rh / cell);
    S.kr = 4.0f;                                   // eq. (15), surface_field.cpp:33-37
    S.ks = float(1.0 / (0.16 * hf * hf) * 1.6);
    S.kn = 0.95f;
    S.Ne = 25;
    S.lambda = 1.0f;                               // eq. (6), surface_field.cpp:39
    S.k1 = float(8.0 / (M_PI * std::pow(rh, 3.0)) * vol);
    S.k2 = float(-48.0 / (M_PI * std::pow(rh, 5.0)) * vol);
    S.k3 = float(48.0 / (M_PI * std::pow(rh, 6.0)) * vol);
    S.k4 = float(16.0 / (M_PI * std::pow(rh, 6.0)) * vol);
    while ((1ull << s->keyBits) <= nc) ++s->keyBits;
    if (!sphgpu_device_available()) {
        *out = s;   // parameters are queryable; compute calls report E_DEVICE
        s->st = nullptr;
        return SPHGPU_OK;
    }
    if (hipStreamCreateWithFlags(&s->st, hipStreamNonBlocking) != hipSuccess ||
        hipMalloc(&s->field, sizeof(float) * nf) != hipSuccess ||
        hipMalloc(&s->ranges, sizeof(int2) * nc) != hipSuccess || upload_table(s) != 0) {
        sphgpu_surfacer_destroy(s);
        return SPHGPU_E_DEVICE;
    }
    *out = s;
    return SPHGPU_OK;
}

void sphgpu_surfacer_destroy(sphgpu_surfacer* s) {
    if (!s) return;
    if (s->st) (void)hipStreamSynchronize(s->st);
    (void)hipFree(s->field); (void)hipFree(s->ranges); (void)hipFree(s->x); (void)hipFree(s->xs);
    (void)hipFree(s->keys); (void)hipFree(s->box); (void)hipFree(s->far); (void)hipFree(s->sortMem);
    free_records(s->spheres);
    free_records(s->ellipsoids);
    s->ring.release();
    (void)hipFree(s->mcCount); (void)hipFree(s->mcTmp); (void)hipFree(s->mcOut);
    if (s->st) (void)hipStreamDestroy(s->st);
    delete s;
}

const char* sphgpu_surfacer_last_error(const sphgpu_surfacer* s) { return s ? s->err.c_str() : "null surfacer"; }

int sphgpu_surfacer_grid(const sphgpu_surfacer* s, double grid_min[3], int grid_num[3], double* cell_size) {
    if (!s) return SPHGPU_E_ARG;
    for (int a = 0; a < 3; ++a) {
        if (grid_min) grid_min[a] = s->fmin[a];
        if (grid_num) grid_num[a] = s->fnum[a];
    }
    if (cell_size) *cell_size = s->cell;
    return SPHGPU_OK;
}

int sphgpu_surfacer_aniso(sphgpu_surfacer* s, long long n, const float* xyz) {
    if (!s) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    return field_of(s, n, xyz, true);
}

int sphgpu_surfacer_isotro(sphgpu_surfacer* s, long long n, const float* xyz) {
    if (!s) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    return field_of(s, n, xyz, false);
}

int sphgpu_surfacer_particles(sphgpu_surfacer* s, float* xbar, float* G, float* det, int* neighbours) {
    if (!s) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    const int n = s->nrec;
    std::vector<SurfRec> r(size_t(std::max(n, 0)));
    std::vector<uint32_t> order(size_t(std::max(n, 0)));
    if (n > 0) {
        SCHECK(s, hipMemcpyAsync(r.data(), s->ellipsoids.rec, sizeof(SurfRec) * n, hipMemcpyDeviceToHost, s->st));
        SCHECK(s, hipMemcpyAsync(order.data(), s->ellipsoids.vals, sizeof(uint32_t) * n, hipMemcpyDeviceToHost, s->st));
    }
    SCHECK(s, hipStreamSynchronize(s->st));
    for (int k = 0; k < n; ++k) {
        const int i = int(order[k]);
        const SurfRec& o = r[k];
        if (xbar) { xbar[3 * i] = o.x; xbar[3 * i + 1] = o.y; xbar[3 * i + 2] = o.z; }
        if (G) {
            const float g[9] = {o.g00, o.g01, o.g02, o.g01, o.g11, o.g12, o.g02, o.g12, o.g22};
            std::memcpy(G + 9 * (size_t)i, g, sizeof(g));
        }
        if (det) det[i] = o.det;
        if (neighbours) neighbours[i] = o.pad;
    }
    return SPHGPU_OK;
}

int sphgpu_surfacer_get_field(sphgpu_surfacer* s, float* out) {
    if (!s || !out) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    SCHECK(s, s->ring.to_host(out, s->field, sizeof(float) * s->nfield, s->st));
    return SPHGPU_OK;
}

int sphgpu_surfacer_set_field(sphgpu_surfacer* s, const float* in) {
    if (!s || !in) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    SCHECK(s, s->ring.to_device(s->field, in, sizeof(float) * s->nfield, s->st));
    SCHECK(s, hipStreamSynchronize(s->st));
    return SPHGPU_OK;
}

int sphgpu_surfacer_marching_cubes(sphgpu_surfacer* s, float iso, float* tris, long long cap, long long* ntris) {
    if (!s || !ntris) return SPHGPU_E_ARG;
    if (!s->st) return sfail(s, SPHGPU_E_DEVICE, "no gfx9 HIP device available");
    if (!std::isfinite(iso)) return sfail(s, SPHGPU_E_ARG, "non-finite iso level");
    const int nx = s->fnum[0], ny = s->fnum[1], nz = s->fnum[2];
    *ntris = 0;
    if (nx < 2 || ny < 2 || nz < 2) return SPHGPU_OK;
    const size_t cubes = size_t(nx - 1) * (ny - 1) * (nz - 1);
    if (cubes >= (size_t(1) << 31)) return sfail(s, SPHGPU_E_CAPACITY, "too many cubes");
    const size_t nodes = size_t(nx) * ny * nz;
    // (units: fewer than 2^31, there being at most 8 nodes to a cube)
    const int units = int((nodes + MC_UNIT - 1) / MC_UNIT);
    if (!s->mcTmp) {   // the grid is the object's: its size does not change
        if (!s->mcCount) SCHECK(s, hipMalloc(&s->mcCount, sizeof(uint32_t) * (size_t(units) + 1)));
        SCHECK(s, hipMalloc(&s->mcTmp, sizeof(uint32_t) * (size_t)scan_tmp_words(units + 1)));
    }
    McGrid G{nx, ny, nz, nodes, iso, {float(s->fmin[0]), float(s->fmin[1]), float(s->fmin[2])}, float(s->cell)};
    const unsigned blocks = unsigned((units + 3) / 4);
    hipLaunchKernelGGL(k_mc_count, dim3(blocks), dim3(256), 0, s->st, G, (const float*)s->field, units, s->mcCount);
    exclusive_scan_u32(s->mcCount, units + 1, s->mcTmp, s->st);
    uint32_t total = 0;
    SCHECK(s, s->ring.to_host(&total, s->mcCount + units, sizeof(uint32_t), s->st));
    *ntris = total;
    if (!tris || total == 0) return SPHGPU_OK;
    const long long keep = std::min<long long>(cap, total);
    if (keep > 0) {
        if (s->mcOutCap < keep) {
            (void)hipFree(s->mcOut);
            s->mcOut = nullptr;
            s->mcOutCap = 0;
            long long room = keep + keep / 4;   // for a surface that grows from call to call
            if (hipMalloc(&s->mcOut, sizeof(float) * 9 * room) != hipSuccess) {
                (void)hipGetLastError();
                s->mcOut = nullptr;
                room = keep;
                SCHECK(s, hipMalloc(&s->mcOut, sizeof(float) * 9 * room));
            }
            s->mcOutCap = room;
        }
        hipLaunchKernelGGL(k_mc_emit, dim3(blocks), dim3(256), 0, s->st, G, (const float*)s->field, units,
                           (const uint32_t*)s->mcCount, s->mcOut, keep);
        if (s->ring.to_host(tris, s->mcOut, sizeof(float) * 9 * keep, s->st) != hipSuccess ||
            hipGetLastError() != hipSuccess)
            return sfail(s, SPHGPU_E_DEVICE, "marching cubes readback failed");
    }
    if (keep < (long long)total) return sfail(s, SPHGPU_E_CAPACITY, "%u triangles, room for %lld", total, cap);
    return SPHGPU_OK;
}

}  // extern "C"
