// gs_surrogate.hip - MLP-ensemble surrogate kernels for gfx950 (BF16 MFMA,
// FP32 accumulate): forward, backward, loss, Adam, ensemble statistics.
//
// One GEMM kernel serves every product of training and inference:
//   C[m][n] = sum_k A(m,k) B(n,k)
// with A(m,k) stored row-major (A[m*lda + k]) or column-major (A[k*lda + m])
// and likewise B(n,k), so that
//   forward        Z = X W^T        A = X (row),  B = W (row)
//   data gradient  dX = dZ W        A = dZ (row), B(n=i,k=o) = W[o][i] (col)
//   weight grad    dW = dZ^T X      A(m=o,k=b) = dZ[b][o] (col), B(n=i,k=b) = X[b][i] (col)
// Tiles: a 256-thread workgroup owns a 64x64 block of C; each wave a 32x32
// quarter as 2x2 v_mfma_f32_16x16x32_bf16 tiles.  K advances 32 at a time
// through LDS (rows padded to 40 bf16 so the 16-byte fragment reads of a
// wave spread over the banks).  Fragment layout of the 16x16x32 MFMA
// (checked on the device): lane l holds A[l%16][8(l/16)..8(l/16)+7],
// B[8(l/16)..+7][l%16], and result D[4(l/16)+v][l%16], v = 0..3.
// The ensemble index is blockIdx.z; every operand has a per-member stride.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gs_surrogate_kernels.h"

namespace gs {
namespace sg {

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TM = 64, TN = 64, TK = 32, LDS_ROW = TK + 8;

// Fragment order of a matrix M[n][k], k a multiple of 32: blocks of 16 n x 32 k
// as the 64 lanes of an MFMA hold them, lane l the 8 values M[16 nt + l % 16][32
// ks + 8 (l / 16) ..], so that a wave's operand load is 1 KB of consecutive
// bytes.  Read row by row (16 pieces of 64 bytes per load) the same operands
// came at 8 to 16 bytes per cycle and CU.
__host__ __device__ inline size_t frag_at(int n, int k, int K) {
    return (((size_t)(n >> 4) * (size_t)(K >> 5) + (size_t)(k >> 5)) * 64 + (size_t)((k >> 3) & 3) * 16 + (size_t)(n & 15)) * 8 +
           (size_t)(k & 7);
}
// Lane `lane`'s fragment of block (nt, ks).
__device__ __forceinline__ bf16x8 frag(const __bf16 *M, int K, int nt, int ks, int lane) {
    return *(const bf16x8 *)(M + (((size_t)nt * (size_t)(K >> 5) + (size_t)ks) * 64 + (size_t)lane) * 8);
}

// bf16(silu(z)) = bf16(z / (1 + e^-z)) from ez = e^-z and z / 4, with one Newton step in
// place of the IEEE division (div_fixup keeps its zeros, infinities and NaN): (z / 4) /
// (1/4 + e^-z / 4), so that the reciprocal stays a normal number up to the largest
// finite e^-z.  Over all 2^32 floats z the bf16 value of the division but for 512 with
// |z| < 5e-38, whose subnormal results differ in the last bit.  The division was half of
// the activation's instructions.
__device__ __forceinline__ __bf16 silu_of(float ez, float z4) {
    const float d = fmaf(ez, 0.25f, 0.25f), y = __builtin_amdgcn_rcpf(d), q = z4 * y;
    return (__bf16)__builtin_amdgcn_div_fixupf(fmaf(fmaf(-d, q, z4), y, q), d, z4);
}
// (training: dsilu takes the same e^-z)
__device__ __forceinline__ __bf16 silu_act(float z) { return silu_of(__expf(-z), 0.25f * z); }
__device__ __forceinline__ __bf16 silu_of_quarter(float z4) {
    constexpr float kM4Log2E = -4.0f * 1.44269504088896340736f;
    return silu_of(__builtin_amdgcn_exp2f(z4 * kM4Log2E), z4);
}
__device__ __forceinline__ float dsilu(float z) {
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

template <bool A_COL, bool B_COL, int EPI>
__global__ void __launch_bounds__(256) gemm_kernel(GemmArgs g) {
    __shared__ __bf16 sA[TM * LDS_ROW];
    __shared__ __bf16 sB[TN * LDS_ROW];
    const int e = blockIdx.z;
    const __bf16 *A = g.A + (size_t)e * g.strideA;
    const __bf16 *B = g.B + (size_t)e * g.strideB;
    const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4 acc[2][2];
    for (int i = 0; i < 2; ++i)
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int k0 = 0; k0 < g.K; k0 += TK) {
        // ---- global -> LDS, 8 bf16 per thread per operand, zero outside M/N
        if (!A_COL) {
            const int r = t >> 2, c = (t & 3) * 8, m = m0 + r;
            bf16x8 v = {};
            if (m < g.M) v = *(const bf16x8 *)(A + (size_t)m * g.lda + k0 + c);
            *(bf16x8 *)(sA + r * LDS_ROW + c) = v;
        } else {
            const int kk = t >> 3, c = (t & 7) * 8;
            const __bf16 *src = A + (size_t)(k0 + kk) * g.lda + m0 + c;
#pragma unroll
            for (int i = 0; i < 8; ++i) sA[(c + i) * LDS_ROW + kk] = (m0 + c + i < g.M) ? src[i] : (__bf16)0.0f;
        }
        if (!B_COL) {
            const int r = t >> 2, c = (t & 3) * 8, n = n0 + r;
            bf16x8 v = {};
            if (n < g.N) v = *(const bf16x8 *)(B + (size_t)n * g.ldb + k0 + c);
            *(bf16x8 *)(sB + r * LDS_ROW + c) = v;
        } else {
            const int kk = t >> 3, c = (t & 7) * 8;
            const __bf16 *src = B + (size_t)(k0 + kk) * g.ldb + n0 + c;
#pragma unroll
            for (int i = 0; i < 8; ++i) sB[(c + i) * LDS_ROW + kk] = (n0 + c + i < g.N) ? src[i] : (__bf16)0.0f;
        }
        __syncthreads();
        const int fr = lane & 15, fk = (lane >> 4) * 8;
        bf16x8 a[2], b[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) a[i] = *(const bf16x8 *)(sA + (wm + 16 * i + fr) * LDS_ROW + fk);
#pragma unroll
        for (int j = 0; j < 2; ++j) b[j] = *(const bf16x8 *)(sB + (wn + 16 * j + fr) * LDS_ROW + fk);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        __syncthreads();
    }
    // ---- epilogue
    const size_t eo = (size_t)e * g.strideC;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + v;
                const int n = n0 + wn + 16 * j + (lane & 15);
                if (m >= g.M || n >= g.N) continue;
                const size_t o = eo + (size_t)m * g.ldc + n;
                const float x = acc[i][j][v];
                if (EPI == EPI_HIDDEN) {
                    const float z = x + g.bias[(size_t)e * g.strideBias + n];
                    if (g.Zf) g.Zf[o] = z;   // kept for the backward pass only
                    g.Cb[o] = silu_act(z);
                } else if (EPI == EPI_OUT) {
                    g.Cf[o] = x + g.bias[(size_t)e * g.strideBias + n];
                } else if (EPI == EPI_DSILU) {
                    const float d = x * dsilu(g.Zf[o]);
                    g.Cf[o] = d;
                    g.Cb[o] = (__bf16)d;
                } else {   // EPI_STORE
                    g.Cf[o] = x;
                }
            }
}

// Fused inference of one member over a tile of rows: standardisation of the
// raw inputs, every layer in one workgroup with the bf16 activations in LDS,
// no activation in memory.  Hidden width 256, padded input and output widths 32.
// Each output element sees the MFMA sequence of gemm_kernel (16x16x32 steps, k
// ascending) and the same epilogue, so the outputs equal the layer-by-layer
// forward pass bit for bit.
//  - The weights are the MFMA's first operand: a lane's four results are then
//    neighbouring outputs of one row, which go to LDS as 8 bytes and to memory
//    as 16.
//  - Weight fragments stream from L2 (fragment order) kAheadK k steps ahead of
//    their use, across layers, so that the epilogue of a layer hides the first
//    loads of the next.
//  - The SiLU is most of the vector work (two transcendentals and seven other
//    operations per element): see silu_of_quarter.
// RT row tiles of 16 by NW waves, chosen by sg_launch_mlp_forward.  Four waves per SIMD: two
// (four waves of 64 columns each) gave 195 us instead of 160 for 65,536 rows of
// four members.  There the products alone take 114 us (947 TFLOP/s; a large matrix
// product reaches 1,297 on this card) and the activations 48 us; before, with IEEE
// divisions, 2-byte LDS writes and two k steps of loads, 190 us.  Ping-pong tiles
// with the activations of one row tile scheduled into the products of the next
// (twice the LDS, half the rows) gave 174 us, wave priorities nothing.
template <int RT, int NW>
struct MlpShape {
    static constexpr int kRows = 16 * RT, kCols = 256 / NW, kColTiles = kCols / 16;
    static constexpr int kAheadK = RT >= 4 ? 2 : RT == 2 ? 4 : 8;   // registers allow no more
};
constexpr int FH = 256, FLD = FH + 8;

template <int RT, int NW>
__global__ void __launch_bounds__(NW * 64, 4) mlp_forward_kernel(MlpArgs g) {
    using S = MlpShape<RT, NW>;
    constexpr int CJ = S::kColTiles, AK = S::kAheadK;
    __shared__ __bf16 act[S::kRows * FLD];
    const int e = blockIdx.y, row0 = blockIdx.x * S::kRows;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int fr = lane & 15, quad = lane >> 4, ct0 = wave * CJ;   // first column tile
    const __bf16 *Pb = g.Pb + (size_t)e * g.Pm;
    const float *P = g.P + (size_t)e * g.Pm;
    bf16x8 w[AK][CJ];
    f32x4 acc[RT][CJ];
    // the first layer's weights and the second's first steps
    bf16x8 w0[CJ];
#pragma unroll
    for (int j = 0; j < CJ; ++j) w0[j] = frag(Pb + g.woff[0], 32, ct0 + j, 0, lane);
    if (g.L > 2) {
#pragma unroll
        for (int k = 0; k < AK; ++k)
#pragma unroll
            for (int j = 0; j < CJ; ++j) w[k][j] = frag(Pb + g.woff[1], FH, ct0 + j, k, lane);
    }
    // standardised inputs, zero beyond the last row and column
    const int sh = g.ni <= 8 ? 3 : g.ni <= 16 ? 4 : 5;
    for (int q = t; q < S::kRows << sh; q += NW * 64) {
        const int r = q >> sh, c = q & ((1 << sh) - 1);
        float v = 0.0f;
        if (c < g.ni && row0 + r < g.rows) v = (g.x[(size_t)(row0 + r) * g.ni + c] - g.mu[c]) / g.sd[c];
        act[r * FLD + c] = (__bf16)v;
    }
    if (sh < 5)
        for (int q = t; q < S::kRows * 3; q += NW * 64) {
            const int r = q / 3, c = 8 * (q % 3 + 1);
            if (c >= 1 << sh) *(bf16x8 *)(act + r * FLD + c) = bf16x8{};
        }
    __syncthreads();
    auto epilogue = [&](const float *bias) {   // all waves have read the tile
#pragma unroll
        for (int j = 0; j < CJ; ++j) {
            const int n = 16 * (ct0 + j) + 4 * quad;
            const f32x4 b = *(const f32x4 *)(bias + n);
            float b4[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) b4[v] = 0.25f * b[v];
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                bf16x4 a;
#pragma unroll
                for (int v = 0; v < 4; ++v) a[v] = silu_of_quarter(fmaf(acc[i][j][v], 0.25f, b4[v]));   // (acc + b) / 4
                *(bf16x4 *)(act + (16 * i + fr) * FLD + n) = a;
            }
        }
    };
    auto row_frag = [&](int i, int k) { return *(const bf16x8 *)(act + (16 * i + fr) * FLD + 32 * k + 8 * quad); };
    // ---- first layer, K = 32
#pragma unroll
    for (int i = 0; i < RT; ++i) {
        const bf16x8 a = row_frag(i, 0);
#pragma unroll
        for (int j = 0; j < CJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0[j], a, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
    __syncthreads();
    epilogue(P + g.boff[0]);
    __syncthreads();
    // ---- hidden layers, K = 256
#pragma unroll 1
    for (int l = 1; l < g.L - 1; ++l) {
        const __bf16 *W = Pb + g.woff[l], *Wn = Pb + g.woff[l + 1 < g.L - 1 ? l + 1 : l];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const bf16x8 a = row_frag(i, k);
#pragma unroll
                for (int j = 0; j < CJ; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k % AK][j], a, k ? acc[i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < CJ; ++j)   // (after the last layer: its own first steps again, unused)
                w[k % AK][j] = k + AK < 8 ? frag(W, FH, ct0 + j, k + AK, lane) : frag(Wn, FH, ct0 + j, k + AK - 8, lane);
        }
        __syncthreads();
        epilogue(P + g.boff[l]);
        __syncthreads();
    }
    // ---- output layer, 32 padded columns: 2 RT tiles over the waves
    const __bf16 *W = Pb + g.woff[g.L - 1];
    const float *bias = P + g.boff[g.L - 1];
#pragma unroll
    for (int task = 0; task < 2 * RT; task += NW) {
        const int q = task + wave, i = q >> 1, j = q & 1;
        if (q >= 2 * RT) break;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 8; ++k) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(W, FH, j, k, lane), row_frag(i, k), o, 0, 0, 0);
        const int n = 16 * j + 4 * quad, row = row0 + 16 * i + fr;
        const f32x4 b = *(const f32x4 *)(bias + n);
        if (row < g.rows) *(f32x4 *)(g.Out + ((size_t)e * g.rows + row) * 32 + n) = f32x4{o[0] + b[0], o[1] + b[1], o[2] + b[2], o[3] + b[3]};
    }
}

// Column sums of a [rows x cols] fp32 matrix per member (bias gradients).
// One thread per column, rows added in order: deterministic.  Networks without
// the fused training kernels only; 16 rows are loaded ahead of their sums.
__global__ void colsum_kernel(const float *X, int rows, int cols, size_t strideX, float *out, size_t strideOut) {
    const int e = blockIdx.y;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cols) return;
    const float *x = X + (size_t)e * strideX;
    float s = 0.f;
    int r = 0;
    for (; r + 16 <= rows; r += 16) {
        float v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = x[(size_t)(r + i) * cols + c];
#pragma unroll
        for (int i = 0; i < 16; ++i) s += v[i];
    }
    for (; r < rows; ++r) s += x[(size_t)r * cols + c];
    out[(size_t)e * strideOut + c] = s;
}

// Weighted squared error: L = sum w (y - t)^2 / sum w per member.
// dY = 2 w (y - t) / sum w, in fp32 and bf16.  wsum[e] holds sum w.
__global__ void loss_grad_kernel(const float *Y, const float *T, const float *W, int n, size_t strideY,
                                 size_t strideT, const float *wsum, float *dYf, __bf16 *dYb, float *loss_part) {
    const int e = blockIdx.y;
    __shared__ float red[256];
    float l = 0.f;
    const float inv = 1.0f / fmaxf(wsum[e], 1e-30f);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float y = Y[(size_t)e * strideY + i], t = T[(size_t)e * strideT + i], w = W[(size_t)e * strideT + i];
        const float d = y - t;
        l += w * d * d * inv;
        const float gr = 2.0f * w * d * inv;
        dYf[(size_t)e * strideY + i] = gr;
        dYb[(size_t)e * strideY + i] = (__bf16)gr;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[(size_t)e * gridDim.x + blockIdx.x] = red[0];
}

// Sum of the loss weights of each member's batch.
__global__ void wsum_kernel(const float *W, int n, size_t strideT, float *wsum) {
    const int e = blockIdx.x;
    __shared__ float red[256];
    float s = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += W[(size_t)e * strideT + i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) wsum[e] = red[0];
}

// Gather a member's minibatch: rows idx[e][r] of the resident data set.
__global__ void gather_kernel(const __bf16 *X, const float *Y, const float *W, const uint32_t *idx, int rows,
                              int in_w, int out_w, __bf16 *bx, float *by, float *bw) {
    const int e = blockIdx.y;
    const int r = blockIdx.x;
    if (r >= rows) return;
    const uint32_t s = idx[(size_t)e * rows + r];
    for (int c = threadIdx.x; c < in_w; c += blockDim.x)
        bx[((size_t)e * rows + r) * in_w + c] = X[(size_t)s * in_w + c];
    for (int c = threadIdx.x; c < out_w; c += blockDim.x) {
        by[((size_t)e * rows + r) * out_w + c] = Y[(size_t)s * out_w + c];
        bw[((size_t)e * rows + r) * out_w + c] = W[(size_t)s * out_w + c];
    }
}

// Adam (decoupled weight decay) of one parameter, the fused multiply-adds
// written out so that every kernel rounds alike.
__device__ __forceinline__ float adam_update(float p, float g, float &mo, float &ve, float lr, float b1, float b2,
                                             float eps, float wd, float c1, float c2) {
    const float m = fmaf(1.0f - b1, g, b1 * mo);
    const float v = fmaf(g, (1.0f - b2) * g, b2 * ve);
    mo = m;
    ve = v;
    return fmaf(-lr, fmaf(wd, p, (m / c1) / (sqrtf(v / c2) + eps)), p);
}

// Adam over the flat parameter vector of every member; refreshes the bf16
// copy the GEMMs read.
__global__ void adam_kernel(float *P, const float *G, float *Mo, float *Ve, __bf16 *Pb, size_t n, float lr,
                            float b1, float b2, float eps, float wd, float c1, float c2) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        float m = Mo[i], v = Ve[i];
        const float p = adam_update(P[i], G[i], m, v, lr, b1, b2, eps, wd, c1, c2);
        Mo[i] = m;
        Ve[i] = v;
        P[i] = p;
        Pb[i] = (__bf16)p;
    }
}

// ---------------------------------------------------------------- fused training step
// Layer by layer a training step was 29 launches, of which the column sums
// (one thread per column, one row after another) took 590 of 870 us at
// minibatches of 512 rows and 4 members.  Here a step is two launches:
//  - train_tile_kernel takes a tile of 16 rows of one member through the
//    forward pass, the loss and the data gradients.  A row's gradient chain
//    touches no other row, so activations pass from layer to layer in LDS and
//    pre-activations stay in the registers of the lanes that formed them
//    (forward and backward give a lane the same elements).  What the weight
//    gradients need goes out in their fragment order (frag_at, along the rows).
//  - train_weights_kernel forms every layer's weight gradient (a wave takes
//    32 x 16 elements over the whole minibatch, operands straight from L2)
//    and bias gradient, and applies Adam to them where they are: the gradient
//    never goes to memory.
// 16 rows: at 512 rows x 4 members 128 workgroups.  16 waves (20.9 us at 8, 38 at
// 4): a lone wave issues every 5 to 6 cycles and the SiLU of 16 elements each
// was as long as a layer's product; a layer's 128 KB of weights are loaded into
// registers while the layer before finishes.  Every sum is taken in the
// layer-by-layer order (k ascending by 32 in the MFMAs, rows ascending in the
// bias sums), so results are the same bits.
// Measured per step, 512 rows x 4 members: 870 us of kernels before; 19 + 15 us.
constexpr int BR = 16, BLD = 256 + 8;
// Work item of workgroup b of n: items in order go to one die (workgroup b runs
// on die b mod 8) in runs, so that a die reads the parameters of one member or
// two instead of all.
__device__ __forceinline__ int item_of(int b, int n) {
    const int q = n / 8, r = n % 8, x = b % 8;
    return x * q + (x < r ? x : r) + b / 8;
}
constexpr int TW = 16, TC = 256 / TW, TJ = TC / 16;   // waves per tile, columns and column tiles per wave

struct WFrag {
    bf16x8 f[8][TJ];   // [k step][column tile]
};
// The fragments of this wave's columns of a weight matrix with rows of K.
template <int K>
__device__ __forceinline__ void load_weights(WFrag &w, const __bf16 *W, int n0, int lane) {
#pragma unroll
    for (int k = 0; k < K / 32; ++k)
#pragma unroll
        for (int j = 0; j < TJ; ++j) w.f[k][j] = frag(W, K, n0 / 16 + j, k, lane);
}
template <int K>
__device__ __forceinline__ void tile_product(f32x4 (&acc)[TJ], const __bf16 *buf, const WFrag &w, int fr, int fk) {
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < K / 32; ++k) {
        const bf16x8 a = *(const bf16x8 *)(buf + fr * BLD + 32 * k + fk);
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w.f[k][j], acc[j], 0, 0, 0);
    }
}


// NH hidden layers of 256.
template <int NH>
__global__ void __launch_bounds__(TW * 64) train_tile_kernel(TrainArgs g) {
    __shared__ __bf16 tile[2][BR * BLD];
    __shared__ float red[2];
    const int tiles = g.rows / BR, item = item_of((int)blockIdx.x, (int)gridDim.x);
    const int e = item / tiles, tile_no = item % tiles, row0 = tile_no * BR;
    const size_t E = gridDim.x / tiles;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int fr = lane & 15, quad = lane >> 4, fk = quad * 8, n0 = wave * TC;
    const __bf16 *Pb = g.Pb + (size_t)e * g.Pm, *PbT = g.PbT + (size_t)e * g.Pm;
    const float *P = g.P + (size_t)e * g.Pm;
    const uint32_t *idx = g.idx ? g.idx + (size_t)e * g.rows : nullptr;
    const size_t B = (size_t)g.rows;
    // this lane's place in a column tile of the second launch's operands
    // (fragments along the rows): 4 rows from row0 + 4 quad
    const int b0 = row0 + 4 * quad;
    auto operand = [&](__bf16 *M, size_t columns_before, int n) {
        return (bf16x4 *)(M + columns_before * B + frag_at(n, b0, g.rows));
    };
    WFrag w;
    load_weights<32>(w, Pb + g.woff[0], n0, lane);
    if (t < BR * 4) {   // input tile
        const int r = t >> 2, c = (t & 3) * 8;
        const size_t row = idx ? (size_t)idx[row0 + r] : (size_t)(row0 + r);
        const bf16x8 v = *(const bf16x8 *)(g.X + row * 32 + c);
        *(bf16x8 *)(tile[0] + r * BLD + c) = v;
#pragma unroll
        for (int i = 0; i < 8; ++i) g.XT[(size_t)e * 32 * B + frag_at(c + i, row0 + r, g.rows)] = v[i];
    }
    __syncthreads();
    // ---- forward: layer l reads tile[l % 2] and writes the other
    f32x4 z[NH][TJ];
#pragma unroll
    for (int l = 0; l < NH; ++l) {
        f32x4 acc[TJ];
        if (l == 0) tile_product<32>(acc, tile[0], w, fr, fk);
        else tile_product<256>(acc, tile[l & 1], w, fr, fk);
        if (l + 1 < NH) load_weights<256>(w, Pb + g.woff[l + 1], n0, lane);
        __bf16 *out = tile[(l + 1) & 1];
        const float *bias = P + g.boff[l];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int n = n0 + 16 * j + fr;
            const float bn = bias[n];
            bf16x4 a;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                z[l][j][v] = acc[j][v] + bn;
                a[v] = silu_act(z[l][j][v]);
                out[(4 * quad + v) * BLD + n] = a[v];
            }
            *operand(g.ActT, ((size_t)l * E + e) * 256, n) = a;
        }
        __syncthreads();
    }
    // ---- output layer, loss and its gradient: waves 0 and 1, 16 columns each
    const __bf16 *act = tile[NH & 1];
    __bf16 *dout = tile[(NH + 1) & 1];
    load_weights<32>(w, PbT + g.woff[NH], n0, lane);   // the first data gradient's
    if (wave < 2) {
        const int n = 16 * wave + fr;
        const __bf16 *W = Pb + g.woff[NH];
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k0 = 0; k0 < 256; k0 += 32) {
            const bf16x8 a = *(const bf16x8 *)(act + fr * BLD + k0 + fk);
            const bf16x8 b = frag(W, 256, wave, k0 / 32, lane);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
        const float bn = P[g.boff[NH] + n];
        const float inv = 1.0f / fmaxf(g.wsum[e], 1e-30f);
        float loss = 0.f;
        bf16x4 gb;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = row0 + 4 * quad + v;
            const size_t row = idx ? (size_t)idx[r] : (size_t)r;
            const float y = acc[v] + bn, tt = g.Y[row * 32 + n], ww = g.W[row * 32 + n];
            const float d = y - tt;
            loss += ww * d * d * inv;
            const float gr = 2.0f * ww * d * inv;
            g.dYf[((size_t)e * B + r) * 32 + n] = gr;
            gb[v] = (__bf16)gr;
            dout[(4 * quad + v) * BLD + n] = gb[v];
        }
        *operand(g.dYT, (size_t)e * 32, n) = gb;
#pragma unroll
        for (int s = 32; s > 0; s >>= 1) loss += __shfl_xor(loss, s);
        if (lane == 0) red[wave] = loss;
    }
    __syncthreads();
    if (t == 0) g.loss_part[(size_t)e * tiles + tile_no] = red[0] + red[1];
    // ---- data gradients: layer l's dZ from layer l + 1's
#pragma unroll
    for (int l = NH - 1; l >= 0; --l) {
        const __bf16 *in = tile[(NH + 1 + NH - 1 - l) & 1];
        __bf16 *out = tile[(NH + NH - 1 - l) & 1];
        f32x4 acc[TJ];
        if (l == NH - 1) tile_product<32>(acc, in, w, fr, fk);
        else tile_product<256>(acc, in, w, fr, fk);
        if (l > 0) load_weights<256>(w, PbT + g.woff[l], n0, lane);
        const size_t at = ((size_t)l * E + e) * 256;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int n = n0 + 16 * j + fr;
            bf16x4 db;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float d = acc[j][v] * dsilu(z[l][j][v]);
                g.dZf[at * B + (size_t)(row0 + 4 * quad + v) * 256 + n] = d;
                db[v] = (__bf16)d;
                if (l > 0) out[(4 * quad + v) * BLD + n] = db[v];
            }
            *operand(g.dZT, at, n) = db;
        }
        if (l > 0) __syncthreads();
    }
}

// Workgroup x of a member: 64 x 64 elements of one layer's weight gradient
// (a wave 32 x 16), or, beyond those, 64 columns of a layer's bias gradient (one
// wave: 512 dependent additions set its time, so the columns are spread).  The
// output layer has 32 rows, the first layer 32 columns: the waves beyond have
// nothing to do.
constexpr int kBiasBlocks = 4;   // per layer; the output layer uses one
template <bool kAdam>
__global__ void __launch_bounds__(512) train_weights_kernel(TrainArgs g, AdamArgs a) {
    const int L = g.L, blocks = 8 + 16 * (L - 2) + kBiasBlocks * (L - 1) + 1;   // of a member
    const int item = item_of((int)blockIdx.x, (int)gridDim.x), e = item / blocks, bx = item % blocks;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const size_t B = (size_t)g.rows, E = gridDim.x / blocks;
    const int n_tiles = 4 + 16 * (L - 2) + 4;
    float *P = g.P + (size_t)e * g.Pm, *G = g.G + (size_t)e * g.Pm;
    float *Mo = g.Mo + (size_t)e * g.Pm, *Ve = g.Ve + (size_t)e * g.Pm;
    __bf16 *Pb = g.Pb + (size_t)e * g.Pm, *PbT = g.PbT + (size_t)e * g.Pm;
    if (bx >= n_tiles) {   // bias of layer l: rows added in order
        const int q = bx - n_tiles, l = q / kBiasBlocks, c = q % kBiasBlocks * 64 + t;
        const int cols = l == L - 1 ? 32 : 256;
        if (t >= 64 || c >= cols) return;
        const float *x = l == L - 1 ? g.dYf + (size_t)e * B * 32 + c : g.dZf + ((size_t)l * E + e) * 256 * B + c;
        const size_t o = g.boff[l] + c;
        float m = 0.f, v = 0.f, p = 0.f;
        if (kAdam) {
            m = Mo[o];
            v = Ve[o];
            p = P[o];
        }
        float s = 0.f;
        auto add_rows = [&](size_t r, auto rows) {
            constexpr int R = decltype(rows)::value;
            float d[R];
#pragma unroll
            for (int i = 0; i < R; ++i) d[i] = x[(r + i) * cols];
#pragma unroll
            for (int i = 0; i < R; ++i) s += d[i];
        };
        size_t r = 0;
        for (; r + 128 <= B; r += 128) add_rows(r, std::integral_constant<int, 128>());
        for (; r < B; r += 64) add_rows(r, std::integral_constant<int, 64>());
        if (kAdam) {
            p = adam_update(p, s, m, v, a.lr, a.b1, a.b2, a.eps, a.wd, a.c1, a.c2);
            Mo[o] = m;
            Ve[o] = v;
            P[o] = p;
        } else {
            G[o] = s;
        }
        return;
    }
    int l, tm, tn;   // layer, tile row (outputs), tile column (inputs)
    if (bx < 4) {
        l = 0; tm = bx; tn = 0;
    } else if (bx < n_tiles - 4) {
        const int q = bx - 4;
        l = 1 + q / 16; tm = (q % 16) / 4; tn = q % 4;
    } else {
        l = L - 1; tm = 0; tn = bx - (n_tiles - 4);
    }
    const int out_w = l == L - 1 ? 32 : 256, in_w = l == 0 ? 32 : 256;
    const int m0 = tm * 64 + (wave >> 2) * 32, c0 = tn * 64 + (wave & 3) * 16;
    if (m0 >= out_w || c0 >= in_w) return;
    const __bf16 *A = l == L - 1 ? g.dYT + (size_t)e * 32 * B : g.dZT + ((size_t)l * E + e) * 256 * B;
    const __bf16 *Bm = l == 0 ? g.XT + (size_t)e * 32 * B : g.ActT + ((size_t)(l - 1) * E + e) * 256 * B;
    const int fr = lane & 15, quad = lane >> 4;
    // Adam's operands, loaded before the product needs its own
    const size_t o = g.woff[l] + (size_t)(m0 + 4 * quad) * in_w + c0 + fr;
    float p[2][4], mo[2][4], ve[2][4];
    if (kAdam) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const size_t ov = o + (size_t)(16 * i + v) * in_w;
                p[i][v] = P[ov];
                mo[i][v] = Mo[ov];
                ve[i][v] = Ve[ov];
            }
    }
    f32x4 acc[2];
    acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // 256 rows of loads in flight at once
    auto rows_from = [&](int k0, auto steps) {
        constexpr int S = decltype(steps)::value;
        bf16x8 fa[S][2], fb[S];
#pragma unroll
        for (int k = 0; k < S; ++k) {
            fb[k] = frag(Bm, g.rows, c0 / 16, k0 / 32 + k, lane);
#pragma unroll
            for (int i = 0; i < 2; ++i) fa[k][i] = frag(A, g.rows, m0 / 16 + i, k0 / 32 + k, lane);
        }
#pragma unroll
        for (int k = 0; k < S; ++k)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[k][i], fb[k], acc[i], 0, 0, 0);
    };
    int k0 = 0;
    for (; k0 + 256 <= g.rows; k0 += 256) rows_from(k0, std::integral_constant<int, 8>());
    for (; k0 < g.rows; k0 += 64) rows_from(k0, std::integral_constant<int, 2>());
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (kAdam) {
            bf16x4 pt;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const size_t ov = o + (size_t)(16 * i + v) * in_w;
                const float pn = adam_update(p[i][v], acc[i][v], mo[i][v], ve[i][v], a.lr, a.b1, a.b2, a.eps, a.wd, a.c1, a.c2);
                Mo[ov] = mo[i][v];
                Ve[ov] = ve[i][v];
                P[ov] = pn;
                pt[v] = (__bf16)pn;
                Pb[g.woff[l] + frag_at(m0 + 16 * i + 4 * quad + v, c0 + fr, in_w)] = pt[v];
            }
            *(bf16x4 *)(PbT + g.woff[l] + frag_at(c0 + fr, m0 + 16 * i + 4 * quad, out_w)) = pt;
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) G[o + (size_t)(16 * i + v) * in_w] = acc[i][v];
        }
    }
}

// wsum[step][e] in the order of wsum_kernel over the gathered minibatch.
__global__ void __launch_bounds__(256) wsum_steps_kernel(const float *W, const uint32_t *idx, int rows, float *wsum) {
    __shared__ float red[256];
    const uint32_t *ix = idx ? idx + (size_t)blockIdx.x * rows : nullptr;
    const int c = threadIdx.x & 31;
    float s = 0.f;
    for (int r = threadIdx.x >> 5; r < rows; r += 64) {   // rows: a multiple of 64
        float w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = W[(ix ? (size_t)ix[r + 8 * i] : (size_t)(r + 8 * i)) * 32 + c];
#pragma unroll
        for (int i = 0; i < 8; ++i) s += w[i];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) wsum[blockIdx.x] = red[0];
}

// The weights of every layer in bf16 and fragment order: W [out][in] into Pb,
// its transpose into PbT (when parameters are set; afterwards
// train_weights_kernel keeps both).
__global__ void __launch_bounds__(256) pack_kernel(TrainArgs g) {
    const int e = blockIdx.y, l = blockIdx.z;
    const int out_w = l == g.L - 1 ? 32 : 256, in_w = l == 0 ? 32 : 256;
    const size_t at = (size_t)e * g.Pm + g.woff[l];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < out_w * in_w; i += gridDim.x * 256) {
        const int o = i / in_w, c = i % in_w;
        const __bf16 v = (__bf16)g.P[at + i];
        g.Pb[at + frag_at(o, c, in_w)] = v;
        g.PbT[at + frag_at(c, o, out_w)] = v;
    }
}

__global__ void to_bf16_kernel(const float *x, __bf16 *y, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        y[i] = (__bf16)x[i];
}

struct StdArgs {
    float mu[32], sd[32];
};

// One thread per padded element.  The subtraction and the IEEE-rounded
// division are those the host would do, so the rows equal a host
// standardisation followed by the bf16 conversion.
__global__ void standardise_kernel(const float *x, int n, int ni, int ldo, StdArgs a, __bf16 *y) {
    const size_t total = (size_t)n * ldo;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / ldo;
        const int c = (int)(i - r * ldo);
        float v = 0.0f;
        if (c < ni) v = (x[r * ni + c] - a.mu[c]) / a.sd[c];
        y[i] = (__bf16)v;
    }
}

struct FlagArgs {
    float lo[32], hi[32];
};

// Per query, half a wave: mean and (population) standard deviation over the
// members of the outputs [E][n][32], first `no` columns, and the fallback flags:
// bit 0x1 when an output selected by `mask` has a spread that is not <= `limit`
// (NaN included), bit 0x2 when one of its ni inputs lies outside [lo, hi] (NaN
// included).  mean, sd and flags may be null.  Reads 128 bytes per query and
// member and is bound by that: as three launches (statistics, flags from the
// spread in memory) it took 17 us for 65,536 queries.
__global__ void __launch_bounds__(256) query_stats_kernel(const float *Y, int E, int n, int no, const float *x, int ni,
                                                         uint32_t mask, float limit, FlagArgs b, float *mean, float *sd,
                                                         uint8_t *flags) {
    const int c = threadIdx.x & 31, lane = threadIdx.x & 63;
    for (size_t r = (size_t)blockIdx.x * 8 + (threadIdx.x >> 5); r < (size_t)n; r += (size_t)gridDim.x * 8) {
        float s = 0.f, s2 = 0.f;
        for (int e = 0; e < E; ++e) {
            const float y = Y[((size_t)e * n + r) * 32 + c];
            s += y;
            s2 = fmaf(y, y, s2);
        }
        const float mu = s / E;
        const float sp = sqrtf(fmaxf(fmaf(-mu, mu, s2 / E), 0.f));
        if (c < no) {
            if (mean) mean[r * no + c] = mu;
            if (sd) sd[r * no + c] = sp;
        }
        if (flags) {
            bool out = false;
            if (c < ni) {
                const float v = x[r * ni + c];
                out = !(v >= b.lo[c] && v <= b.hi[c]);
            }
            const uint64_t wide = __ballot(c < no && ((mask >> c) & 1u) && !(sp <= limit)), outside = __ballot(out);
            const int half = lane & 32;
            if (c == 0) flags[r] = (uint8_t)(((uint32_t)(wide >> half) ? 0x1u : 0u) | ((uint32_t)(outside >> half) ? 0x2u : 0u));
        }
    }
}

}  // namespace sg
}  // namespace gs

using namespace gs::sg;

template <bool AC, bool BC, int EPI>
static hipError_t launch_gemm_t(const GemmArgs &g, int members, hipStream_t s) {
    const dim3 grid((g.N + TN - 1) / TN, (g.M + TM - 1) / TM, members);
    hipLaunchKernelGGL((gemm_kernel<AC, BC, EPI>), grid, dim3(256), 0, s, g);
    return hipGetLastError();
}

hipError_t sg_launch_gemm(bool a_col, bool b_col, int epi, const GemmArgs &g, int members, hipStream_t s) {
    if (g.K % TK != 0 || g.M <= 0 || g.N <= 0 || members <= 0) return hipErrorInvalidValue;
    // the column-major loaders read 8 consecutive m (n) values per thread
    if ((a_col && (g.lda % 8)) || (b_col && (g.ldb % 8)) || (!a_col && (g.lda % 8)) || (!b_col && (g.ldb % 8)))
        return hipErrorInvalidValue;
    if (!a_col && !b_col) {
        if (epi == EPI_HIDDEN) return launch_gemm_t<false, false, EPI_HIDDEN>(g, members, s);
        if (epi == EPI_OUT) return launch_gemm_t<false, false, EPI_OUT>(g, members, s);
        return launch_gemm_t<false, false, EPI_STORE>(g, members, s);
    }
    if (!a_col && b_col) {
        if (epi == EPI_DSILU) return launch_gemm_t<false, true, EPI_DSILU>(g, members, s);
        return launch_gemm_t<false, true, EPI_STORE>(g, members, s);
    }
    if (a_col && b_col) return launch_gemm_t<true, true, EPI_STORE>(g, members, s);
    return hipErrorInvalidValue;
}

template <int RT, int NW>
static hipError_t launch_mlp(const MlpArgs &g, int members, hipStream_t s) {
    const int tile = MlpShape<RT, NW>::kRows;
    hipLaunchKernelGGL((mlp_forward_kernel<RT, NW>), dim3((unsigned)((g.rows + tile - 1) / tile), (unsigned)members),
                       dim3(NW * 64), 0, s, g);
    return hipGetLastError();
}

hipError_t sg_launch_mlp_forward(const MlpArgs &g, int members, hipStream_t s) {
    if (g.rows <= 0 || members <= 0 || g.L < 2 || g.L > kMlpMaxLayers || g.ni < 1 || g.ni > 32) return hipErrorInvalidValue;
    // The smallest tiles that fill the CUs: latency, and no long last wave of
    // workgroups.  One call, four members, in us (tiles of 16 / 32 / 64 / 128 rows):
    // 1 row 23 / 25 / 28 / 38; 2,048 rows 34 / 28 / 30 / 41; 8,192 rows 77 / 48 / 42 / 45;
    // 20,011 rows 159 / 93 / 73 / 80; 40,000 rows 297 / 165 / 126 / 123; 65,536 rows
    // 471 / 258 / 198 / 183.  256 CUs, two workgroups of 64 or 128 rows each.
    const size_t rows = (size_t)g.rows * (size_t)members;
    if (rows <= 16 * 256) return launch_mlp<1, 16>(g, members, s);
    if (rows <= 32 * 256) return launch_mlp<2, 8>(g, members, s);
    if (rows <= 64 * 2048) return launch_mlp<4, 8>(g, members, s);
    return launch_mlp<8, 8>(g, members, s);
}

hipError_t sg_launch_wsum(const float *W, const uint32_t *idx, int rows, int steps, int members, float *wsum,
                          hipStream_t s) {
    if (rows <= 0 || rows % 64 || steps <= 0 || members <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(wsum_steps_kernel, dim3((unsigned)steps * (unsigned)members), dim3(256), 0, s, W, idx, rows, wsum);
    return hipGetLastError();
}

hipError_t sg_launch_train_tile(const TrainArgs &g, int members, hipStream_t s) {
    if (g.rows <= 0 || g.rows % 64 || members <= 0 || g.L < 2 || g.L > kMlpMaxLayers) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(g.rows / BR) * (unsigned)members), block(TW * 64);
    switch (g.L - 1) {
    case 1: hipLaunchKernelGGL(train_tile_kernel<1>, grid, block, 0, s, g); break;
    case 2: hipLaunchKernelGGL(train_tile_kernel<2>, grid, block, 0, s, g); break;
    case 3: hipLaunchKernelGGL(train_tile_kernel<3>, grid, block, 0, s, g); break;
    case 4: hipLaunchKernelGGL(train_tile_kernel<4>, grid, block, 0, s, g); break;
    case 5: hipLaunchKernelGGL(train_tile_kernel<5>, grid, block, 0, s, g); break;
    case 6: hipLaunchKernelGGL(train_tile_kernel<6>, grid, block, 0, s, g); break;
    default: hipLaunchKernelGGL(train_tile_kernel<7>, grid, block, 0, s, g); break;
    }
    return hipGetLastError();
}

hipError_t sg_launch_train_weights(const TrainArgs &g, const AdamArgs *adam, int members, hipStream_t s) {
    if (g.rows <= 0 || g.rows % 64 || members <= 0 || g.L < 2 || g.L > kMlpMaxLayers) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(8 + 16 * (g.L - 2) + kBiasBlocks * (g.L - 1) + 1) * (unsigned)members), block(512);
    if (adam) hipLaunchKernelGGL(train_weights_kernel<true>, grid, block, 0, s, g, *adam);
    else hipLaunchKernelGGL(train_weights_kernel<false>, grid, block, 0, s, g, AdamArgs{});
    return hipGetLastError();
}

hipError_t sg_launch_pack(const TrainArgs &g, int members, hipStream_t s) {
    if (members <= 0 || g.L < 2 || g.L > kMlpMaxLayers) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pack_kernel, dim3(32, (unsigned)members, (unsigned)g.L), dim3(256), 0, s, g);
    return hipGetLastError();
}

hipError_t sg_launch_colsum(const float *X, int rows, int cols, size_t strideX, float *out, size_t strideOut,
                            int members, hipStream_t s) {
    hipLaunchKernelGGL(colsum_kernel, dim3((cols + 255) / 256, members), dim3(256), 0, s, X, rows, cols, strideX,
                       out, strideOut);
    return hipGetLastError();
}

hipError_t sg_launch_loss(const float *Y, const float *T, const float *W, int n, size_t strideY, size_t strideT,
                          float *wsum, float *dYf, __bf16 *dYb, float *loss_part, int parts, int members,
                          hipStream_t s) {
    hipLaunchKernelGGL(wsum_kernel, dim3(members), dim3(256), 0, s, W, n, strideT, wsum);
    hipLaunchKernelGGL(loss_grad_kernel, dim3(parts, members), dim3(256), 0, s, Y, T, W, n, strideY, strideT, wsum,
                       dYf, dYb, loss_part);
    return hipGetLastError();
}

hipError_t sg_launch_gather(const __bf16 *X, const float *Y, const float *W, const uint32_t *idx, int rows, int in_w,
                            int out_w, __bf16 *bx, float *by, float *bw, int members, hipStream_t s) {
    hipLaunchKernelGGL(gather_kernel, dim3(rows, members), dim3(64), 0, s, X, Y, W, idx, rows, in_w, out_w, bx, by,
                       bw);
    return hipGetLastError();
}

hipError_t sg_launch_adam(float *P, const float *G, float *Mo, float *Ve, __bf16 *Pb, size_t n, float lr, float b1,
                          float b2, float eps, float wd, float c1, float c2, hipStream_t s) {
    hipLaunchKernelGGL(adam_kernel, dim3(1024), dim3(256), 0, s, P, G, Mo, Ve, Pb, n, lr, b1, b2, eps, wd, c1, c2);
    return hipGetLastError();
}

hipError_t sg_launch_to_bf16(const float *x, __bf16 *y, size_t n, hipStream_t s) {
    hipLaunchKernelGGL(to_bf16_kernel, dim3(1024), dim3(256), 0, s, x, y, n);
    return hipGetLastError();
}

hipError_t sg_launch_standardise(const float *x, int n, int ni, int ldo, const float *mu, const float *sd, __bf16 *y,
                                 hipStream_t s) {
    if (ni < 1 || ni > 32 || ni > ldo) return hipErrorInvalidValue;
    StdArgs a{};
    for (int c = 0; c < ni; ++c) {
        a.mu[c] = mu[c];
        a.sd[c] = sd[c];
    }
    hipLaunchKernelGGL(standardise_kernel, dim3(1024), dim3(256), 0, s, x, n, ni, ldo, a, y);
    return hipGetLastError();
}

hipError_t sg_launch_query_stats(const float *Y, int E, int n, int no, const float *x, int ni, uint32_t mask, float limit,
                                 const float *lo, const float *hi, float *mean, float *sd, uint8_t *flags,
                                 hipStream_t s) {
    if (E <= 0 || n <= 0 || no < 0 || no > 32 || ni < 1 || ni > 32) return hipErrorInvalidValue;
    FlagArgs b{};
    for (int c = 0; c < ni; ++c) {
        b.lo[c] = lo[c];
        b.hi[c] = hi[c];
    }
    hipLaunchKernelGGL(query_stats_kernel, dim3((unsigned)((n + 7) / 8)), dim3(256), 0, s, Y, E, n, no, x, ni, mask, limit, b,
                       mean, sd, flags);
    return hipGetLastError();
}
