// Device state of the per-particle MLP 8 -> 64 -> 64 -> 64 -> 1 (mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace sphgpu {

constexpr int MLP_IN = 8;
constexpr int MLP_PARAMS = 64 * 8 + 64 + 64 * 64 + 64 + 64 * 64 + 64 + 64 + 1;   // 8961
constexpr int MLP_FWD_FRAGS = 22;    // BF16 A fragments of the forward pass
constexpr int MLP_BWD_FRAGS = 20;    // BF16 A fragments of the backward pass
constexpr int MLP_WGRAD_TILES = 53;  // 40 weight tiles + 13 bias tiles
constexpr int MLP_SLICES = 512;      // blocks of a gradient at most: two on each CU
// Samples of a gradient block for n samples: 64, the least a block's four
// waves take, until that gives MLP_SLICES blocks; from there on a block takes
// several of its chunks and the partial gradients (54 KB a block) stay as many.
constexpr int mlp_slice_samples(long long n) { return int(64 * ((n + 64LL * MLP_SLICES - 1) / (64LL * MLP_SLICES))); }
constexpr int mlp_slices(long long n) { return int((n + mlp_slice_samples(n) - 1) / mlp_slice_samples(n)); }
// the most slices of any 1 <= n <= cap
constexpr int mlp_max_slices(long long cap) { return int((cap + 63) / 64 < MLP_SLICES ? (cap + 63) / 64 : MLP_SLICES); }

constexpr size_t MLP_LOSS_OFFSET = (sizeof(float) * MLP_PARAMS + 255) / 256 * 256;   // of lossPart behind grad

struct MlpDev {
    float* params = nullptr;    // FP32 master parameters (W1 b1 W2 b2 W3 b3 W4 b4)
    float* adamM = nullptr;
    float* adamV = nullptr;
    float* grad = nullptr;
    void* fwd = nullptr;        // MLP_FWD_FRAGS x 64 lanes x 8 BF16
    void* bwd = nullptr;        // MLP_BWD_FRAGS x 64 lanes x 8 BF16
    double* lossPart = nullptr; // mlp_max_slices(cap), behind grad in one block
    float* gradPart = nullptr;  // slices x MLP_WGRAD_TILES x 256 partial gradient tiles
    float overWeight = 1.0f;    // loss weight where the prediction exceeds the target
    int cap = 0;                // samples per gradient evaluation
    int adamStep = 0;
};

void mlp_pack(MlpDev& m, hipStream_t st);
// y[i] = MLP(feat[8 i .. 8 i + 7]); gate1: tiles of 16 particles whose feature
// 1 is negative for all 16 are skipped, their outputs left as they were
void mlp_forward(const MlpDev& m, const float* feat, float* y, int n, hipStream_t st, bool gate1 = false);
// gradient of mean((MLP(feat) - target)^2) into m.grad (n <= m.cap); loss parts in m.lossPart
void mlp_grad(MlpDev& m, const float* feat, const float* target, int n, hipStream_t st);
void mlp_adam(MlpDev& m, float lr, hipStream_t st);

}  // namespace sphgpu

#include <vector>
namespace sphgpu {
void mlp_init_params(std::vector<float>& p, unsigned long long seed);
int mlp_alloc(MlpDev& m, int cap);
void mlp_free(MlpDev& m);
// bytes from MlpDev::grad on: the gradient, then room for the loss partial sums of up to n samples
inline size_t mlp_result_bytes(long long n) { return MLP_LOSS_OFFSET + sizeof(double) * (size_t)mlp_max_slices(n); }
// mean loss of n samples from the partial sums, in order
double mlp_loss_sum(const double* part, int n);
}  // namespace sphgpu
