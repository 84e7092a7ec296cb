// Per-particle MLP 8 -> 64 -> 64 -> 64 -> 1 (tanh-form GELU) on the gfx950
// matrix cores: BF16 operands, FP32 accumulation (v_mfma_f32_16x16x32_bf16).
//
// Formulation: activations are kept "transposed", units x particles.  A layer
// z = W h + b is the MFMA D = A*B with A = W (out x in, from weight fragments)
// and B = h (in x 16 particles).  The D layout of a 16x16 tile is
//   lane l = 16*g + c holds D[4g + j][c], j = 0..3,
// so two consecutive 16-row tiles of one layer's output, rounded to BF16, are
// exactly the B operand of the next layer when K slot (g, j) of the 32-deep
// product carries logical index kmap(g, j) = j < 4 ? 4g + j : 16 + 4g + j - 4.
// A and B place the same logical index in the same slot, so the product does
// not depend on the hardware's own K order.
//
// Kernels: fragment packing (FP32 master weights -> BF16 A fragments),
// inference, the gradient of a slice of samples (forward, loss, backward
// through the activations, weight and bias gradients with K = samples), the
// sum of the slices, and Adam.
#include "sph_common.h"
#include "mlp.h"
#include "sphgpu.h"
#include "xfer.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

namespace sphgpu {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int kmap(int g, int j) { return j < 4 ? 4 * g + j : 16 + 4 * g + (j - 4); }

__device__ __forceinline__ __bf16 to_bf16(float x) { return (__bf16)x; }   // round to nearest even

// GELU, tanh form: 0.5 x (1 + tanh(u)), u = c (x + 0.044715 x^3),
// c = sqrt(2/pi), evaluated as x sigma(2u) = x / (1 + exp(-2u)) (the same
// function: one exponential and one hardware reciprocal per activation)
__device__ __forceinline__ float gelu_sigma(float x) {
    // exp(-2u) = exp2(t), t = x (k1 + k2 x^2), k1 = -2 c log2(e), k2 = 0.044715 k1
    const float k1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
    const float k2 = 0.044715f * k1;
    const float t = x * (k1 + k2 * (x * x));
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}
__device__ __forceinline__ float gelu(float x) { return x * gelu_sigma(x); }
// d/dx x sigma(2u) = sigma + 2 x sigma (1 - sigma) c (1 + 3 * 0.044715 x^2), sg = sigma(2u)
__device__ __forceinline__ float gelu_grad(float x, float sg) {
    const float c = 0.7978845608028654f;
    return sg + 2.0f * x * sg * (1.0f - sg) * c * (1.0f + 3.0f * 0.044715f * x * x);
}

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// --------------------------------------------------------------- layout ----
// parameter block (FP32 master): W1[64][8] b1[64] W2[64][64] b2[64] W3[64][64] b3[64] W4[1][64] b4[1]
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + 64 * 8;
constexpr int OFF_W2 = OFF_B1 + 64, OFF_B2 = OFF_W2 + 64 * 64;
constexpr int OFF_W3 = OFF_B2 + 64, OFF_B3 = OFF_W3 + 64 * 64;
constexpr int OFF_W4 = OFF_B3 + 64, OFF_B4 = OFF_W4 + 64;
static_assert(OFF_B4 + 1 == MLP_PARAMS, "parameter count");

struct LayerDim { int off_w, in, out; };
__constant__ LayerDim kLayers[4] = {{OFF_W1, 8, 64}, {OFF_W2, 64, 64}, {OFF_W3, 64, 64}, {OFF_W4, 64, 1}};

// fragment counts: forward A = W (out x in): [ceil(out/16) M tiles] x [ceil(in/32) K steps]
//   L1 4x1 (ids 0-3), L2 4x2 (4-11), L3 4x2 (12-19), L4 1x2 (20-21);
// backward A = W^T (in x out): W4^T 4x1 (0-3), W3^T 4x2 (4-11), W2^T 4x2 (12-19)
// (the first layer needs no input gradient).

// one thread per (fragment, lane): 64 lanes x 8 BF16 values
__global__ void k_mlp_pack(const float* __restrict__ P, bf16x8* __restrict__ fwd, bf16x8* __restrict__ bwd) {
    int fid = blockIdx.x, lane = threadIdx.x;
    int g = lane >> 4, c = lane & 15;
    bf16x8 v;
    if (fid < MLP_FWD_FRAGS) {
        int layer = fid < 4 ? 0 : fid < 12 ? 1 : fid < 20 ? 2 : 3;
        const int base[4] = {0, 4, 12, 20};
        const int ks[4] = {1, 2, 2, 2};
        int rel = fid - base[layer], t = rel / ks[layer], s = rel % ks[layer];
        LayerDim L = kLayers[layer];
        int out = 16 * t + c;
        for (int j = 0; j < 8; ++j) {
            int in = 32 * s + kmap(g, j);
            float w = (out < L.out && in < L.in) ? P[L.off_w + out * L.in + in] : 0.0f;
            v[j] = to_bf16(w);
        }
        fwd[fid * 64 + lane] = v;
    } else {
        int b = fid - MLP_FWD_FRAGS;
        // backward fragments: layer 3 (W4^T: 64 x 1, 4 tiles x 1 kstep) -> 0..3,
        // layer 2 (W3^T: 4 x 2) -> 4..11, layer 1 (W2^T: 4 x 2) -> 12..19
        int layer = b < 4 ? 3 : b < 12 ? 2 : 1;
        int base = b < 4 ? 0 : b < 12 ? 4 : 12;
        int ks = b < 4 ? 1 : 2;
        int rel = b - base, t = rel / ks, s = rel % ks;
        LayerDim L = kLayers[layer];   // W is out x in; A = W^T is in x out
        int in = 16 * t + c;
        for (int j = 0; j < 8; ++j) {
            int out = 32 * s + kmap(g, j);
            float w = (out < L.out && in < L.in) ? P[L.off_w + out * L.in + in] : 0.0f;
            v[j] = to_bf16(w);
        }
        bwd[b * 64 + lane] = v;
    }
}

// B operand for K step s from two D tiles (t = 2s, 2s+1) of activations
__device__ __forceinline__ bf16x8 chain(const float (&h)[4][4], int s) {
    bf16x8 b;
    for (int j = 0; j < 4; ++j) {
        b[j] = to_bf16(h[2 * s][j]);
        b[j + 4] = to_bf16(h[2 * s + 1][j]);
    }
    return b;
}

// Inference only: the 22 weight fragments stay in registers and the biases
// in LDS for all the tiles of 16 particles a wave processes (the training
// pass re-reads them per tile).  gate1: a tile whose 16 particles
// all have feature 1 below zero is skipped and its outputs are not written
// (the DFSPH warm start reads the output only where Drho/Dt > 0, and feature
// 1 is asinh of a positive multiple of Drho/Dt, negative only where it is).
__global__ __launch_bounds__(256, 3) void k_mlp_infer(const bf16x8* __restrict__ F, const float* __restrict__ P,
                                                 const float* __restrict__ feat, float* __restrict__ y, int n,
                                                 int gate1) {
    __shared__ float sb[3 * 64];
    for (int k = threadIdx.x; k < 3 * 64; k += 256) {
        const int off[3] = {OFF_B1, OFF_B2, OFF_B3};
        sb[k] = P[off[k >> 6] + (k & 63)];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    bf16x8 w[MLP_FWD_FRAGS];
#pragma unroll
    for (int f = 0; f < MLP_FWD_FRAGS; ++f) w[f] = F[f * 64 + lane];
    const float b4 = P[OFF_B4];
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int nw = (gridDim.x * blockDim.x) >> 6;
    const int ntile = (n + 15) / 16;
    for (int tile = wave; tile < ntile; tile += nw) {
        const int p = tile * 16 + c;
        bf16x8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = to_bf16(0.0f);
        bool need = false;
        if (g < 2 && p < n) {
            const float4 f = reinterpret_cast<const float4*>(feat)[p * 2 + g];
            x[0] = to_bf16(f.x); x[1] = to_bf16(f.y); x[2] = to_bf16(f.z); x[3] = to_bf16(f.w);
            need = g == 0 && !(f.y < 0.0f);
        }
        if (gate1 && __ballot(need) == 0) continue;   // uniform per wave
        float h[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = mfma(w[t], x, acc);
#pragma unroll
            for (int j = 0; j < 4; ++j) h[t][j] = gelu(acc[j] + sb[16 * t + 4 * g + j]);
        }
#pragma unroll
        for (int L = 0; L < 2; ++L) {
            const bf16x8 b0 = chain(h, 0), b1 = chain(h, 1);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                acc = mfma(w[4 + 8 * L + 2 * t], b0, acc);
                acc = mfma(w[4 + 8 * L + 2 * t + 1], b1, acc);
#pragma unroll
                for (int j = 0; j < 4; ++j) h[t][j] = gelu(acc[j] + sb[64 * (L + 1) + 16 * t + 4 * g + j]);
            }
        }
        const bf16x8 b0 = chain(h, 0), b1 = chain(h, 1);
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mfma(w[20], b0, acc);
        acc = mfma(w[21], b1, acc);
        if (g == 0 && p < n) y[p] = acc[0] + b4;
    }
}

// Tile t of the weight/bias gradient: 16x16 blocks of dW (out x in) per
// layer, then bias blocks.  L1 4x1, L2 4x4, L3 4x4, L4 1x4 (W), then bias
// tiles 4+4+4+1.
struct GradTile { int L, to, ti, bias; };
__device__ __forceinline__ GradTile grad_tile(int t) {
    GradTile r{0, 0, 0, 0};
    int k = t;
    const int wt[4] = {4, 16, 16, 4};
    while (r.L < 4 && k >= wt[r.L]) { k -= wt[r.L]; ++r.L; }
    if (r.L < 4) {
        int nin = (r.L == 0) ? 1 : 4;
        r.to = k / nin;
        r.ti = k % nin;
    } else {
        r.bias = 1;
        const int bt[4] = {4, 4, 4, 1};
        r.L = 0;
        while (r.L < 3 && k >= bt[r.L]) { k -= bt[r.L]; ++r.L; }
        r.to = k;
    }
    return r;
}

// Gradient of one slice of samples (mlp_slice_samples) a block, in chunks of
// 64: each wave takes 16 samples forward and backward, dh = W^T dz chained on
// the matrix cores like the forward pass, with loss = w e^2, e = y - target,
// w = over where e > 0 else 1 (dL/dy = 2 w e / n).  What the weight gradients
// contract over the samples, the layer inputs (features, GELU(z1..3)) and the
// output gradients (dz1..3, dL/dy), goes to LDS as BF16, unit-major, so that a
// fragment's eight samples are two 8-byte reads; after the chunk's four waves
// are done each of them accumulates every fourth of the 53 tiles
// (k_mlp_wgrad_reduce sums the slices in a fixed order: deterministic).  One
// FP64 loss partial a block.  sigma is evaluated once for GELU and its
// derivative, which stays in registers until the way back.
// Bound by the wave's chain of layers and the weights' loads at one block a CU.
// Measured (MI355X, one training iteration): 4,096 samples 18.2 us, 16,384
// 24.9 (this kernel 15.6), 60,000 35.8, 262,144 81; as separate passes that
// kept z and dz in memory 43.8, 54.5 (48.8), 98.6 and 501.  The weights staged in
// LDS (one block a CU): 20.9, 27.7, 47.6, 115; held in registers over the
// chunks: 19.6, 26.0, 46.2, 114.
constexpr int TR_CHUNK = 64;
constexpr int TR_ROW = TR_CHUNK + 4;     // LDS row pitch in BF16 (8-byte aligned, staggered banks)
constexpr int TR_DZ = 193;               // rows of output gradients: dz1 dz2 dz3 (192) and dL/dy
constexpr int TR_H = 200;                // rows of inputs: features (8), h1, h2, h3
constexpr int TR_TILES_PER_WAVE = (MLP_WGRAD_TILES + 3) / 4;

__device__ __forceinline__ bf16x8 lds_frag(const __bf16* row, int g) {
    // samples kmap(g, 0..3) = 4g..4g+3 and kmap(g, 4..7) = 16+4g..16+4g+3
    const uint2 lo = *reinterpret_cast<const uint2*>(row + 4 * g);
    const uint2 hi = *reinterpret_cast<const uint2*>(row + 16 + 4 * g);
    bf16x8 v;
    __builtin_memcpy(&v, &lo, 8);
    __builtin_memcpy(reinterpret_cast<char*>(&v) + 8, &hi, 8);
    return v;
}

__global__ __launch_bounds__(256, 2) void k_mlp_train(const bf16x8* __restrict__ F, const bf16x8* __restrict__ B,
                                                    const float* __restrict__ P, const float* __restrict__ feat,
                                                    const float* __restrict__ target, float* __restrict__ part,
                                                    double* __restrict__ lossPart, int n, int per, float over) {
    __shared__ __attribute__((aligned(16))) __bf16 sA[TR_DZ * TR_ROW];
    __shared__ __attribute__((aligned(16))) __bf16 sB[(TR_H + 1) * TR_ROW];   // last row: bias input 1 / 0
    __shared__ double sLoss[4];
    const int slice = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const int col = 16 * wave + c;           // the sample's column
    f32x4 acc[TR_TILES_PER_WAVE];
#pragma unroll
    for (int k = 0; k < TR_TILES_PER_WAVE; ++k) acc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    double loss = 0.0;
    const long long p1 = min((long long)n, (long long)(slice + 1) * per);
    for (long long q = (long long)slice * per; q < p1; q += TR_CHUNK) {
        const long long p = q + col;
        const bool ok = p < p1;
        // keeps the weights' loads in the loop: the compiler would hold the 42
        // fragments in registers over all chunks and spill for it
        int again = 0;
        asm volatile("" : "+s"(again));
        const bf16x8 *const Fc = F + again, *const Bc = B + again;
        const float* const Pc = P + again;
        float h[4][4], gp[3][4][4];
        {
            bf16x8 x = bf16x8{};
            if (g < 2) {
                if (ok) {
                    const float4 f = reinterpret_cast<const float4*>(feat)[p * 2 + g];
                    x[0] = to_bf16(f.x); x[1] = to_bf16(f.y); x[2] = to_bf16(f.z); x[3] = to_bf16(f.w);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) sB[(4 * g + j) * TR_ROW + col] = x[j];
            }
            if (g == 2) sB[TR_H * TR_ROW + col] = to_bf16(ok ? 1.0f : 0.0f);
#pragma unroll
            for (int L = 0; L < 3; ++L) {
                const bf16x8 b0 = L ? chain(h, 0) : x, b1 = L ? chain(h, 1) : x;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    if (L == 0) {
                        z = mfma(Fc[t * 64 + lane], b0, z);
                    } else {
                        z = mfma(Fc[(8 * L - 4 + 2 * t) * 64 + lane], b0, z);
                        z = mfma(Fc[(8 * L - 4 + 2 * t + 1) * 64 + lane], b1, z);
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int u = 16 * t + 4 * g + j;
                        const float v = z[j] + Pc[(L == 0 ? OFF_B1 : L == 1 ? OFF_B2 : OFF_B3) + u];
                        const float sg = gelu_sigma(v);
                        h[t][j] = v * sg;
                        gp[L][t][j] = gelu_grad(v, sg);
                        sB[(8 + 64 * L + u) * TR_ROW + col] = to_bf16(ok ? h[t][j] : 0.0f);
                    }
                }
            }
        }
        // B operand of the way back: dz4 (1 x P) in K slot (0, 0); y is row 0 of
        // the last layer's product: lanes g == 0, j == 0
        bf16x8 b = bf16x8{};
        {
            f32x4 y = {0.f, 0.f, 0.f, 0.f};
            y = mfma(Fc[20 * 64 + lane], chain(h, 0), y);
            y = mfma(Fc[21 * 64 + lane], chain(h, 1), y);
            if (g == 0) {
                if (ok) {
                    const float e = y[0] + Pc[OFF_B4] - target[p];
                    const float w = e > 0.0f ? over : 1.0f;
                    loss += (double)w * (double)e * (double)e;
                    b[0] = to_bf16(2.0f * w * e / (float)n);
                }
                sA[192 * TR_ROW + col] = b[0];
            }
        }
        // dh3 = W4^T dz4, dh2 = W3^T dz3, dh1 = W2^T dz2; dz = dh * gelu'(z)
        float d[4][4];
#pragma unroll
        for (int L = 2; L >= 0; --L) {
            const bf16x8 b0 = L == 2 ? b : chain(d, 0), b1 = L == 2 ? b : chain(d, 1);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f32x4 dh = {0.f, 0.f, 0.f, 0.f};
                if (L == 2) {
                    dh = mfma(Bc[t * 64 + lane], b0, dh);
                } else {
                    dh = mfma(Bc[(12 - 8 * L + 2 * t) * 64 + lane], b0, dh);
                    dh = mfma(Bc[(12 - 8 * L + 2 * t + 1) * 64 + lane], b1, dh);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    d[t][j] = dh[j] * gp[L][t][j];
                    sA[(64 * L + 16 * t + 4 * g + j) * TR_ROW + col] = to_bf16(ok ? d[t][j] : 0.0f);
                }
            }
        }
        __syncthreads();   // the chunk's columns are written
#pragma unroll
        for (int k = 0; k < TR_TILES_PER_WAVE; ++k) {
            const int t = wave + 4 * k;
            if (t >= MLP_WGRAD_TILES) break;
            const GradTile T = grad_tile(t);
            const int nin = (T.L == 0) ? 8 : 64, nout = (T.L == 3) ? 1 : 64;
            const int zoff = (T.L < 3) ? T.L * 64 : 192;            // rows of layer L's output gradient
            const int hoff = (T.L == 0) ? 0 : 8 + (T.L - 1) * 64;   // rows of layer L's input
            const int orow = 16 * T.to + c, icol = 16 * T.ti + c;
#pragma unroll
            for (int s = 0; s < TR_CHUNK; s += 32) {
                const bf16x8 zero = bf16x8{};
                const bf16x8 a = orow < nout ? lds_frag(sA + (zoff + orow) * TR_ROW + s, g) : zero;
                const bf16x8 v = T.bias ? lds_frag(sB + TR_H * TR_ROW + s, g)
                                        : (icol < nin ? lds_frag(sB + (hoff + icol) * TR_ROW + s, g) : zero);
                acc[k] = mfma(a, v, acc[k]);
            }
        }
        __syncthreads();   // the fragments are read: the next chunk may overwrite them
    }
    // D[4g+j][c] of each tile
#pragma unroll
    for (int k = 0; k < TR_TILES_PER_WAVE; ++k) {
        const int t = wave + 4 * k;
        if (t >= MLP_WGRAD_TILES) break;
        float* out = part + ((size_t)slice * MLP_WGRAD_TILES + t) * 256;
        for (int j = 0; j < 4; ++j) out[(4 * g + j) * 16 + c] = acc[k][j];
    }
    const double s = block_sum_256(loss, sLoss);
    if (threadIdx.x == 0) lossPart[slice] = s;
}

// Sum of the slices' partial tiles: eight threads per gradient element,
// thread group r summing slices r, r + 8, r + 16, ... in order, then the
// eight sums added in group order (a fixed order: deterministic).  Block b
// covers 32 elements of tile b / 8.
__global__ __launch_bounds__(256) void k_mlp_wgrad_reduce(const float* __restrict__ part, float* __restrict__ grad,
                                                        int slices, float scale) {
    __shared__ float red[8][32];
    const int tile = blockIdx.x >> 3, r = threadIdx.x >> 5, lane = threadIdx.x & 31;
    const int e = ((blockIdx.x & 7) << 5) | lane;
    float s = 0.0f;
#pragma unroll 4
    for (int k = r; k < slices; k += 8) s += part[((size_t)k * MLP_WGRAD_TILES + tile) * 256 + e];
    red[r][lane] = s;
    __syncthreads();
    if (r != 0) return;
#pragma unroll
    for (int k = 1; k < 8; ++k) s += red[k][lane];
    const GradTile T = grad_tile(tile);
    const int nin = (T.L == 0) ? 8 : 64, nout = (T.L == 3) ? 1 : 64;
    const int row = e >> 4, col = e & 15;
    const int out = 16 * T.to + row, in = 16 * T.ti + col;
    if (out >= nout) return;
    if (T.bias ? col != 0 : in >= nin) return;
    const int woff[4] = {OFF_W1, OFF_W2, OFF_W3, OFF_W4}, boff[4] = {OFF_B1, OFF_B2, OFF_B3, OFF_B4};
    if (T.bias) grad[boff[T.L] + out] = s * scale;
    else grad[woff[T.L] + out * nin + in] = s * scale;
}

__global__ void k_mlp_adam(float* __restrict__ P, float* __restrict__ M, float* __restrict__ V,
                           const float* __restrict__ grad, float lr, float b1, float b2, float eps, float c1,
                           float c2) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= MLP_PARAMS) return;
    float gr = grad[i];
    float m = b1 * M[i] + (1.0f - b1) * gr;
    float v = b2 * V[i] + (1.0f - b2) * gr * gr;
    M[i] = m;
    V[i] = v;
    P[i] -= lr * (m / c1) / (sqrtf(v / c2) + eps);
}

}  // namespace

// ------------------------------------------------------------------ host ----
void mlp_pack(MlpDev& m, hipStream_t st) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(MLP_FWD_FRAGS + MLP_BWD_FRAGS), dim3(64), 0, st, (const float*)m.params,
                       (bf16x8*)m.fwd, (bf16x8*)m.bwd);
}

void mlp_forward(const MlpDev& m, const float* feat, float* y, int n, hipStream_t st, bool gate1) {
    if (n <= 0) return;
    const int waves = (n + 15) / 16;
    // about three waves per SIMD, each looping over tiles
    const int blocks = std::min((waves + 3) / 4, 768);
    hipLaunchKernelGGL(k_mlp_infer, dim3(blocks), dim3(256), 0, st, (const bf16x8*)m.fwd, (const float*)m.params,
                       feat, y, n, gate1 ? 1 : 0);
}

void mlp_grad(MlpDev& m, const float* feat, const float* target, int n, hipStream_t st) {
    const int slices = mlp_slices(n);
    hipLaunchKernelGGL(k_mlp_train, dim3(slices), dim3(256), 0, st, (const bf16x8*)m.fwd, (const bf16x8*)m.bwd,
                       (const float*)m.params, feat, target, m.gradPart, m.lossPart, n, mlp_slice_samples(n),
                       m.overWeight);
    hipLaunchKernelGGL(k_mlp_wgrad_reduce, dim3(8 * MLP_WGRAD_TILES), dim3(256), 0, st, (const float*)m.gradPart,
                       m.grad, slices, 1.0f);
}

void mlp_adam(MlpDev& m, float lr, hipStream_t st) {
    m.adamStep += 1;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    float c1 = 1.0f - std::pow(b1, (float)m.adamStep), c2 = 1.0f - std::pow(b2, (float)m.adamStep);
    hipLaunchKernelGGL(k_mlp_adam, dim3((MLP_PARAMS + 255) / 256), dim3(256), 0, st, m.params, m.adamM, m.adamV,
                       (const float*)m.grad, lr, b1, b2, eps, c1, c2);
    mlp_pack(m, st);
}

// Glorot-uniform weights, zero biases, from a 64-bit LCG stream
void mlp_init_params(std::vector<float>& p, unsigned long long seed) {
    p.assign(MLP_PARAMS, 0.0f);
    unsigned long long s = seed * 6364136223846793005ULL + 1442695040888963407ULL;
    auto uni = [&]() {
        s = s * 6364136223846793005ULL + 1442695040888963407ULL;
        return double(s >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0;
    };
    const int off[4] = {OFF_W1, OFF_W2, OFF_W3, OFF_W4}, in[4] = {8, 64, 64, 64}, out[4] = {64, 64, 64, 1};
    for (int L = 0; L < 4; ++L) {
        double a = std::sqrt(6.0 / double(in[L] + out[L]));
        for (int k = 0; k < in[L] * out[L]; ++k) p[off[L] + k] = float(a * uni());
    }
}

int mlp_alloc(MlpDev& m, int cap) {
    m.cap = std::max(cap, 16);
    auto al = [](void** p, size_t b) { return hipMalloc(p, std::max<size_t>(b, 256)) == hipSuccess; };
    bool ok = al((void**)&m.params, sizeof(float) * MLP_PARAMS) && al((void**)&m.adamM, sizeof(float) * MLP_PARAMS) &&
              al((void**)&m.adamV, sizeof(float) * MLP_PARAMS) && al((void**)&m.grad, mlp_result_bytes(m.cap)) &&
              al(&m.fwd, 16 * 64 * MLP_FWD_FRAGS) && al(&m.bwd, 16 * 64 * MLP_BWD_FRAGS) &&
              al((void**)&m.gradPart, sizeof(float) * 256 * MLP_WGRAD_TILES * (size_t)mlp_max_slices(m.cap));
    m.lossPart = reinterpret_cast<double*>(reinterpret_cast<char*>(m.grad) + MLP_LOSS_OFFSET);
    if (!ok) return -1;
    hipMemset(m.adamM, 0, sizeof(float) * MLP_PARAMS);
    hipMemset(m.adamV, 0, sizeof(float) * MLP_PARAMS);
    m.adamStep = 0;
    return 0;
}

void mlp_free(MlpDev& m) {
    void* ps[] = {m.params, m.adamM, m.adamV, m.grad, m.fwd, m.bwd, m.gradPart};
    for (void* p : ps)
        if (p) hipFree(p);
    m = MlpDev{};
}

double mlp_loss_sum(const double* part, int n) {
    double s = 0.0;
    for (int k = 0; k < mlp_slices(n); ++k) s += part[k];
    return n > 0 ? s / n : 0.0;
}

// ---- gradient on caller-provided device buffers, scratch in a static array
// Every buffer mlp_grad needs beyond its inputs and outputs (weight
// fragments, loss and gradient partials) lives
// in one file-scope device array, so the entry point allocates nothing.
// Each GPU holds its own copy until the process ends; host code reaches it
// only through the address hipGetSymbolAddress returns on that device.
constexpr int MLP_DEV_MAX = SPHGPU_MLP_DEVICE_MAX;
constexpr size_t al256(size_t b) { return (b + 255) & ~size_t(255); }
constexpr size_t SCR_FWD = 0;
constexpr size_t SCR_BWD = SCR_FWD + al256(16 * 64 * MLP_FWD_FRAGS);
constexpr size_t SCR_LOSS = SCR_BWD + al256(16 * 64 * MLP_BWD_FRAGS);
constexpr size_t SCR_GPART = SCR_LOSS + al256(sizeof(double) * mlp_max_slices(MLP_DEV_MAX));
constexpr size_t SCR_BYTES = SCR_GPART + al256(sizeof(float) * 256 * MLP_WGRAD_TILES * (size_t)mlp_max_slices(MLP_DEV_MAX));

static __device__ __align__(256) unsigned char scratch[SCR_BYTES];

namespace {
// mean loss: the block partials summed in order by one thread (the order
// mlp_loss_sum sums them in), divided by n
__global__ void k_mlp_loss_final(const double* __restrict__ part, int parts, int n, double* __restrict__ out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double s = 0.0;
    for (int k = 0; k < parts; ++k) s += part[k];
    *out = s / n;
}
}  // namespace

// device address of `scratch` on the current device, looked up once per device
static int scratch_on_device(unsigned char** out) {
    static std::mutex mu;
    static unsigned char* ptr[64] = {};
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return SPHGPU_E_DEVICE;
    std::lock_guard<std::mutex> lock(mu);
    if (!ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return SPHGPU_E_DEVICE;
        ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = ptr[dev];
    return SPHGPU_OK;
}

}  // namespace sphgpu

// ------------------------------------------------------------- C-ABI ----
struct sphgpu_mlp {
    sphgpu::MlpDev m;
    hipStream_t st = nullptr;
    float* feat = nullptr;
    float* target = nullptr;
    float* y = nullptr;
    sphgpu::HostRing ring;
    std::vector<unsigned char> result;   // gradient and loss partial sums as read back
};

extern "C" int sphgpu_mlp_create(int capacity, unsigned long long seed, sphgpu_mlp** out) {
    if (!out || capacity <= 0) return SPHGPU_E_ARG;
    *out = nullptr;
    if (!sphgpu_device_available()) return SPHGPU_E_DEVICE;
    sphgpu_mlp* h = new sphgpu_mlp();
    if (hipStreamCreateWithFlags(&h->st, hipStreamNonBlocking) != hipSuccess || sphgpu::mlp_alloc(h->m, capacity) ||
        hipMalloc((void**)&h->feat, sizeof(float) * 8 * (size_t)h->m.cap) != hipSuccess ||
        hipMalloc((void**)&h->target, sizeof(float) * (size_t)h->m.cap) != hipSuccess ||
        hipMalloc((void**)&h->y, sizeof(float) * (size_t)h->m.cap) != hipSuccess) {
        sphgpu_mlp_destroy(h);
        return SPHGPU_E_DEVICE;
    }
    std::vector<float> p;
    sphgpu::mlp_init_params(p, seed);
    return sphgpu_mlp_set_params(h, p.data()) == 0 ? (*out = h, SPHGPU_OK) : (sphgpu_mlp_destroy(h), SPHGPU_E_DEVICE);
}

extern "C" void sphgpu_mlp_destroy(sphgpu_mlp* h) {
    if (!h) return;
    if (h->st) hipStreamSynchronize(h->st);
    sphgpu::mlp_free(h->m);
    if (h->feat) hipFree(h->feat);
    if (h->target) hipFree(h->target);
    if (h->y) hipFree(h->y);
    h->ring.release();
    if (h->st) hipStreamDestroy(h->st);
    delete h;
}

extern "C" int sphgpu_mlp_set_params(sphgpu_mlp* h, const float* params) {
    if (!h || !params) return SPHGPU_E_ARG;
    if (hipMemcpyAsync(h->m.params, params, sizeof(float) * sphgpu::MLP_PARAMS, hipMemcpyHostToDevice, h->st) != hipSuccess)
        return SPHGPU_E_DEVICE;
    sphgpu::mlp_pack(h->m, h->st);
    return hipStreamSynchronize(h->st) == hipSuccess ? SPHGPU_OK : SPHGPU_E_DEVICE;
}

extern "C" int sphgpu_mlp_get_params(sphgpu_mlp* h, float* params) {
    if (!h || !params) return SPHGPU_E_ARG;
    hipMemcpyAsync(params, h->m.params, sizeof(float) * sphgpu::MLP_PARAMS, hipMemcpyDeviceToHost, h->st);
    return hipStreamSynchronize(h->st) == hipSuccess ? SPHGPU_OK : SPHGPU_E_DEVICE;
}

extern "C" int sphgpu_mlp_set_loss(sphgpu_mlp* h, float over_weight) {
    if (!h || !(over_weight > 0.0f) || !std::isfinite(over_weight)) return SPHGPU_E_ARG;
    h->m.overWeight = over_weight;
    return SPHGPU_OK;
}

extern "C" int sphgpu_mlp_forward(sphgpu_mlp* h, long long n, const float* feat, float* out) {
    if (!h || n < 0 || (n > 0 && (!feat || !out))) return SPHGPU_E_ARG;
    for (long long o = 0; o < n; o += h->m.cap) {
        int k = int(std::min<long long>(h->m.cap, n - o));
        if (h->ring.to_device(h->feat, feat + 8 * o, sizeof(float) * 8 * k, h->st) != hipSuccess) return SPHGPU_E_DEVICE;
        sphgpu::mlp_forward(h->m, h->feat, h->y, k, h->st);
        if (h->ring.to_host(out + o, h->y, sizeof(float) * k, h->st) != hipSuccess) return SPHGPU_E_DEVICE;
    }
    return hipStreamSynchronize(h->st) == hipSuccess && hipGetLastError() == hipSuccess ? SPHGPU_OK : SPHGPU_E_DEVICE;
}

// uploads a batch
static int batch_to_device(sphgpu_mlp* h, int k, const float* feat, const float* target) {
    return h->ring.to_device(h->feat, feat, sizeof(float) * 8 * k, h->st) == hipSuccess &&
                   h->ring.to_device(h->target, target, sizeof(float) * k, h->st) == hipSuccess
               ? SPHGPU_OK
               : SPHGPU_E_DEVICE;
}

// gradient (where wanted) and loss of the last mlp_grad of k samples, with one transfer
static int results_to_host(sphgpu_mlp* h, int k, float* grad, double* loss) {
    const size_t bytes = sphgpu::mlp_result_bytes(k);
    h->result.resize(bytes);
    if (h->ring.to_host(h->result.data(), h->m.grad, bytes, h->st) != hipSuccess) return SPHGPU_E_DEVICE;
    if (grad) std::memcpy(grad, h->result.data(), sizeof(float) * sphgpu::MLP_PARAMS);
    if (loss)
        *loss = sphgpu::mlp_loss_sum(reinterpret_cast<const double*>(h->result.data() + sphgpu::MLP_LOSS_OFFSET), k);
    return hipGetLastError() == hipSuccess ? SPHGPU_OK : SPHGPU_E_DEVICE;
}

extern "C" int sphgpu_mlp_gradient(sphgpu_mlp* h, long long n, const float* feat, const float* target, float* grad,
                                   double* loss) {
    if (!h || n <= 0 || n > h->m.cap || !feat || !target || !grad) return SPHGPU_E_ARG;
    const int k = int(n);
    if (int rc = batch_to_device(h, k, feat, target)) return rc;
    sphgpu::mlp_grad(h->m, h->feat, h->target, k, h->st);
    return results_to_host(h, k, grad, loss);
}

extern "C" int sphgpu_mlp_train(sphgpu_mlp* h, long long n, const float* feat, const float* target, int iters, float lr,
                                double* loss) {
    if (!h || n <= 0 || n > h->m.cap || !feat || !target || iters < 0) return SPHGPU_E_ARG;
    const int k = int(n);
    if (int rc = batch_to_device(h, k, feat, target)) return rc;
    for (int it = 0; it < iters; ++it) {
        sphgpu::mlp_grad(h->m, h->feat, h->target, k, h->st);
        sphgpu::mlp_adam(h->m, lr, h->st);
    }
    sphgpu::mlp_grad(h->m, h->feat, h->target, k, h->st);
    return results_to_host(h, k, nullptr, loss);
}

extern "C" int sphgpu_mlp_gradient_device(const float* params, long long n, const float* feat, const float* target,
                                          float over_weight, float* grad, double* loss, void* stream) {
    using namespace sphgpu;
    if (!params || !feat || !target || !grad || !loss || n <= 0 || !(over_weight > 0.0f) ||
        !std::isfinite(over_weight))
        return SPHGPU_E_ARG;
    if (n > MLP_DEV_MAX) return SPHGPU_E_CAPACITY;
    unsigned char* base = nullptr;
    if (int rc = scratch_on_device(&base)) return rc;
    hipStream_t st = static_cast<hipStream_t>(stream);
    MlpDev m;
    m.params = const_cast<float*>(params);   // read only: no Adam step here
    m.grad = grad;
    m.fwd = base + SCR_FWD;
    m.bwd = base + SCR_BWD;
    m.lossPart = reinterpret_cast<double*>(base + SCR_LOSS);
    m.gradPart = reinterpret_cast<float*>(base + SCR_GPART);
    m.overWeight = over_weight;
    m.cap = MLP_DEV_MAX;
    const int k = int(n);
    // every scratch word the kernels read is written earlier in this call:
    // fragments by the pack, loss and gradient partials per slice
    mlp_pack(m, st);
    mlp_grad(m, feat, target, k, st);
    hipLaunchKernelGGL(k_mlp_loss_final, dim3(1), dim3(64), 0, st, (const double*)m.lossPart, mlp_slices(k), k,
                       loss);
    return hipGetLastError() == hipSuccess ? SPHGPU_OK : SPHGPU_E_DEVICE;
}
