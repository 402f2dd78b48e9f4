// mlp_launch.hpp -- launchers of the surrogate-network kernels (mlp_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace gdtk {

hipError_t launch_mfma_probe(const float* A, const float* B, float* D, hipStream_t s);
hipError_t launch_mlp_pack(const float* W, int n_out, int n_in, int chain, unsigned short* frag, hipStream_t s);
hipError_t launch_mlp_infer(int H, int NH, const float* x, int n_in, int n, const unsigned short* frag,
                            const float* bias, int n_out, float* y, hipStream_t s, const unsigned* count = nullptr);

// One batch of training: parameters, inputs and targets, and the buffers between the kernels.
constexpr int MLP_MAX_LAYERS = 4;
struct MlpPass {
    int B, n_in, n_out;
    int bf16;  // inputs and hidden activations rounded to BF16 (the weights are by the caller)
    const float* W[MLP_MAX_LAYERS];  // [out][in]
    // inner layers' weights in operand order, of the forward and of the backward product
    const float *Wf[MLP_MAX_LAYERS], *Wb[MLP_MAX_LAYERS];
    const float* b[MLP_MAX_LAYERS];
    // Input k of batch row b at x[k xk + row xc], row = idx[b] or b; targets likewise.
    const float *x, *y;
    size_t xk, xc, yk, yc;
    const int* idx;
    float* y_out;  // forward only: [B][n_out]
    // [cell block][row, padded to 16][16 cells]: layer l's inputs and its dZ
    float* act[MLP_MAX_LAYERS];
    float* dz[MLP_MAX_LAYERS];
    float* loss;  // sum of squared errors per cell block
    int in_w[MLP_MAX_LAYERS], out_w[MLP_MAX_LAYERS];
    size_t woff[MLP_MAX_LAYERS], boff[MLP_MAX_LAYERS];
};

int mlp_blocks(int B);  // cell blocks of a batch
hipError_t launch_mlp_pass(int H, int NH, const MlpPass& net, int grad, hipStream_t s);
int mlp_grad_splits(const MlpPass& net, int nlayer, int B);
// parts: [nsplit][nparam]
hipError_t launch_mlp_weight_grad(const MlpPass& net, int nlayer, int nsplit, size_t nparam, float* parts,
                                  hipStream_t s);
hipError_t launch_mlp_sum_grads(size_t n, int nsplit, const float* parts, float* grads, hipStream_t s);
// wq (may be null): the updated parameters rounded to BF16
// packed: operands [layer][forward, backward][H H] of the sqn inner H x H layers, whose parameters
// start at sq0
hipError_t launch_mlp_operands(size_t n, const float* w, float* packed, int H, size_t sq0, size_t sqn, hipStream_t s);
hipError_t launch_mlp_adam(size_t n, int nsplit, const float* parts, float* p, float* m, float* v, float* wq,
                           float* packed, int H, size_t sq0, size_t sqn, float lr, float b1, float b2, float eps, int t,
                           hipStream_t s);
hipError_t launch_round_bf16(size_t n, const float* in, float* out, hipStream_t s);

}  // namespace gdtk
