// gs_surrogate_kernels.h - launchers of the surrogate's gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

// GEMM epilogues
enum {
    EPI_STORE = 0,   // Cf = acc
    EPI_HIDDEN = 1,  // Zf = acc + bias, Cb = bf16(silu(Zf))
    EPI_OUT = 2,     // Cf = acc + bias
    EPI_DSILU = 3    // Cf = acc * silu'(Zf), Cb = bf16(Cf)
};

struct GemmArgs {
    const __bf16 *A;
    const __bf16 *B;
    int M, N, K;
    int lda, ldb, ldc;
    size_t strideA, strideB, strideC;   // per ensemble member (elements)
    const float *bias;
    size_t strideBias;
    float *Zf;                          // EPI_HIDDEN: written; EPI_DSILU: read
    float *Cf;
    __bf16 *Cb;
};

// Fused inference (all layers of a member per row tile, activations in LDS):
// hidden width 256, input and output padded to 32, 2..kMlpMaxLayers weight layers.
constexpr int kMlpMaxLayers = 8;
struct MlpArgs {
    const float *x;                     // [rows][ni] raw inputs, standardised as (x - mu) / sd
    int ni;
    float mu[32], sd[32];
    int rows, L;                        // L weight layers
    const __bf16 *Pb;                   // bf16 weights in fragment order, member stride Pm
    const float *P;                     // fp32 parameters (biases)
    size_t Pm;
    size_t woff[kMlpMaxLayers], boff[kMlpMaxLayers];
    float *Out;                         // [members][rows][32]
};

// Fused training step of the same network shape: one launch for the forward
// pass, the loss and the data gradients of every row tile, one for the weight
// and bias gradients and Adam.  rows: a multiple of 64.
struct TrainArgs {
    const __bf16 *X;                    // standardised inputs [n][32]
    const float *Y, *W;                 // targets and loss weights [n][32]
    const uint32_t *idx;                // [members][rows] rows of the minibatch; nullptr: rows 0 .. rows-1
    int rows, L;
    float *P, *Mo, *Ve, *G;             // parameters, Adam moments, gradients (member stride Pm)
    __bf16 *Pb, *PbT;                   // bf16 weights in fragment order, and with every weight transposed ([in][out])
    size_t Pm;
    size_t woff[kMlpMaxLayers], boff[kMlpMaxLayers];
    const float *wsum;                  // [members] sums of the loss weights
    // Written by the first launch for the second: bf16 operands of the products
    // over the rows in fragment order ([columns][rows]), row-major fp32 for the
    // bias sums.
    __bf16 *XT;                         // [member][32][rows] inputs
    __bf16 *ActT, *dZT;                 // [L-1][member][256][rows] activations, pre-activation gradients
    float *dZf;                         // [L-1][member][rows][256]
    __bf16 *dYT;                        // [member][32][rows] output gradients
    float *dYf;                         // [member][rows][32]
    float *loss_part;                   // [members][rows / 16]
};
struct AdamArgs {
    float lr, b1, b2, eps, wd, c1, c2;
};
// Sums of the loss weights of `steps` consecutive minibatches: wsum[step][member].
hipError_t sg_launch_wsum(const float *W, const uint32_t *idx, int rows, int steps, int members, float *wsum,
                          hipStream_t s);
hipError_t sg_launch_train_tile(const TrainArgs &g, int members, hipStream_t s);
// adam == nullptr: gradients into G; otherwise the parameters are updated.
hipError_t sg_launch_train_weights(const TrainArgs &g, const AdamArgs *adam, int members, hipStream_t s);
// Pb and PbT from P.
hipError_t sg_launch_pack(const TrainArgs &g, int members, hipStream_t s);

hipError_t sg_launch_gemm(bool a_col, bool b_col, int epi, const GemmArgs &g, int members, hipStream_t s);
hipError_t sg_launch_mlp_forward(const MlpArgs &g, int members, hipStream_t s);
hipError_t sg_launch_colsum(const float *X, int rows, int cols, size_t strideX, float *out, size_t strideOut,
                            int members, hipStream_t s);
hipError_t sg_launch_loss(const float *Y, const float *T, const float *W, int n, size_t strideY, size_t strideT,
                          float *wsum, float *dYf, __bf16 *dYb, float *loss_part, int parts, int members,
                          hipStream_t s);
hipError_t sg_launch_gather(const __bf16 *X, const float *Y, const float *W, const uint32_t *idx, int rows, int in_w,
                            int out_w, __bf16 *bx, float *by, float *bw, int members, hipStream_t s);
hipError_t sg_launch_adam(float *P, const float *G, float *Mo, float *Ve, __bf16 *Pb, size_t n, float lr, float b1,
                          float b2, float eps, float wd, float c1, float c2, hipStream_t s);
hipError_t sg_launch_to_bf16(const float *x, __bf16 *y, size_t n, hipStream_t s);
// Standardised, zero-padded bf16 rows [n][ldo] from fp32 rows [n][ni]:
// y = bf16((x - mu) / sd), with ni <= 32.
hipError_t sg_launch_standardise(const float *x, int n, int ni, int ldo, const float *mu, const float *sd, __bf16 *y,
                                 hipStream_t s);
// Ensemble mean and spread of the outputs Y [E][n][32], first no columns, and
// the fallback flags of the raw inputs x [n][ni]: 0x1 spread above limit on an
// output of mask, 0x2 input outside [lo, hi]; no, ni <= 32.  mean, sd and flags
// may be null.
hipError_t sg_launch_query_stats(const float *Y, int E, int n, int no, const float *x, int ni, uint32_t mask, float limit,
                                 const float *lo, const float *hi, float *mean, float *sd, uint8_t *flags,
                                 hipStream_t s);
