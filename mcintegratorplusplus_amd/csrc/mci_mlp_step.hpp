// mci_mlp_step.hpp — one training iteration of the learned proposal's network in three kernels
// (mci_mlp_step.hip): forward, likelihood head and backward of a tile of samples on chip; the weight
// gradients as products over all samples; their sum with Adam.
#pragma once

#include "mci_mlp.hpp"

namespace mcim
{
constexpr int STEP_NS = 16; // samples of a workgroup's tile

// the network as the kernels read it.  dp, Hp: d and H rounded up to 32 (zero-padded copies);
// parameters in one array of npad floats: W1 [d][H], b1, W2 [H][H], b2, W3 [H][Op], b3
struct StepNet
{
    int d, H, K, Op, dp, Hp;
    int64_t oW1, ob1, oW2, ob2, oW3, ob3, npad;
    const float *p;
    // BF16 copies in the matrix instruction's operand order (step_operand): forward reads the transposes
    // W1t [Hp][dp], W2t [Hp][Hp], W3t [Op][Hp], backward the matrices W2 [Hp][Hp], W3 [Hp][Op]; one
    // array of `lines` 128-byte lines from W1t on
    bf16_t *W1t, *W2t, *W3t, *W2, *W3;
    int lines;
};

// where element (row, k) of a matrix with kp columns lies in operand order: blocks of 16 rows x 32 terms,
// in a block the eight terms that lane row % 16 + 16 (k % 32 / 8) supplies -- a wave's load is one
// contiguous KB
__host__ __device__ inline int64_t step_operand(int row, int k, int kp)
{
    return ((int64_t)(row / 16 * (kp / 32) + k / 32) * 64 + row % 16 + 16 * (k % 32 / 8)) * 8 + k % 8;
}

// a minibatch: either X, Y [d][n] given, or (snap not null) pairs drawn from the snapshots
// [nsnap][d][W]: context from one, target from another one (the context's walker with probability
// same_frac); fixed_ctx: that input for every sample
struct StepBatch
{
    int64_t n;
    const float *X, *Y;
    const float *snap, *fixed_ctx;
    int nsnap;
    int64_t W;
    uint64_t iter;
    uint32_t k0, k1;
    float same_frac;
};

// what the sample tiles leave for the weight gradients: [tile][feature][STEP_NS] in BF16, and a tile's
// sums of the three layers' output gradients [tile][Op + 2 Hp] in FP32
struct StepWork
{
    bf16_t *X, *H1, *H2, *dO, *dZ2, *dZ1;
    float *bias, *loss;
    float *ws; // [step_splits][npad]
};

// LDS of the tile kernel; the path serves every network whose tile fits a compute unit, since it is the
// faster one up to that edge: an iteration, tiles against separate products (us), d 8 H 16 K 2 1024
// samples 20 / 105, d 32 H 128 K 8 1024 samples 32 / 198, 65536 samples 464 / 2363, and at the edge
// d 32 H 512 K 8 4096 samples 84 / 520, d 8 H 640 K 8 80 / 502
size_t step_lds(int d, int H, int Op);
constexpr size_t STEP_LDS_MAX = 160 * 1024;
// splits of the sample range in the weight gradients' products
int step_splits(const StepNet &N, int64_t n);

// parameters -> the padded BF16 copies (the padding is the caller's to clear once)
hipError_t launch_step_copies(const StepNet &N, hipStream_t s);
// loss per sample and, in work.ws, the split sums of the mean loss's gradient
hipError_t launch_step_grad(const StepNet &N, const StepBatch &B, const StepWork &w, hipStream_t s);
// the gradient g[npad] from the splits
hipError_t launch_step_sum(const StepNet &N, int64_t n, const StepWork &w, float *g, hipStream_t s);
// the same with Adam: p, m, v, their BF16 copies pb[npad] and those of N
hipError_t launch_step_adam(const StepNet &N, int64_t n, const StepWork &w, float *g, float *p, float *m, float *v, bf16_t *pb, float lr,
                            float b1, float b2, float eps, float bc1, float bc2, hipStream_t s);
} // namespace mcim
