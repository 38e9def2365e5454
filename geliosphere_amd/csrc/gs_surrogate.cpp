// gs_surrogate.cpp - host side of the MLP-ensemble surrogate (C ABI in
// include/gs_surrogate.h).  All tensors live on the device; the host only
// draws initial weights and minibatch orders and launches kernels.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/gs_surrogate.h"
#include "gs_surrogate_kernels.h"

namespace {

constexpr int kPad = 32;   // padded width of the input and output layers

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
};

}  // namespace

struct gs_surrogate {
    int device = 0;
    hipStream_t stream = nullptr;
    gs_surrogate_config cfg{};
    int E = 0, L = 0;                  // members, weight layers (hidden layers + 1)
    std::vector<int> dims;             // dims[0] = kPad, hidden..., dims[L] = kPad
    std::vector<size_t> woff, boff;    // per-member offsets (floats)
    size_t Pm = 0;                     // floats per member
    float *P = nullptr, *G = nullptr, *Mo = nullptr, *Ve = nullptr;
    __bf16 *Pb = nullptr;              // row-major; fragment order for the fused kernels' shapes
    __bf16 *PbT = nullptr;             // those shapes: every weight transposed, fragment order
    uint64_t step = 0;
    bool normalized = false;
    float mu[GS_SG_MAX_INPUTS], sd[GS_SG_MAX_INPUTS], lo[GS_SG_MAX_INPUTS], hi[GS_SG_MAX_INPUTS];
    // work buffers, grown on demand
    std::vector<DevBuf> bufs;
    // host predictions: two halves of pinned memory and their events (pin_half)
    char *pin = nullptr;
    size_t pin_half = 0;
    hipEvent_t pin_done[2] = {nullptr, nullptr};
    std::string err;
};

namespace {

gs_status fail(gs_surrogate *s, gs_status st, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (s) s->err = buf;
    return st;
}

#define SG_TRY(s, call)                                                                       \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return fail((s), e_ == hipErrorOutOfMemory ? GS_ERR_OUT_OF_MEMORY : GS_ERR_HIP,   \
                        "%s failed: %s", #call, hipGetErrorString(e_));                       \
    } while (0)

// Named work buffers (index into s->bufs).
enum Buf {
    B_X = 0,      // data set inputs, bf16 [n][kPad]
    B_XF,         // staging fp32 [n][n_inputs]
    B_Y,          // data set targets fp32 [n][kPad]
    B_W,          // data set weights fp32 [n][kPad]
    B_IDX,        // minibatch rows uint32 [E][B]
    B_BX, B_BY, B_BW,     // minibatch per member
    B_Z,          // pre-activations fp32 [L-1][E][B][H]
    B_ACT,        // activations bf16 [L-1][E][B][H]
    B_OUT,        // outputs fp32 [E][B][kPad]
    B_DYF, B_DYB, // output gradient
    B_DZF0, B_DZB0, B_DZF1, B_DZB1,   // hidden gradients, ping-pong
    B_WSUM, B_LOSS,
    B_MEAN, B_SD,
    B_FLAGS,      // predict: fallback flags uint8 [n]
    B_DZF, B_DZT, // fused training: hidden gradients [L-1][E][H][B], fp32 and bf16
    B_COUNT_
};

template <class T>
gs_status need(gs_surrogate *s, int which, size_t count, T **out) {
    DevBuf &b = s->bufs[which];
    const size_t bytes = std::max<size_t>(count * sizeof(T), 256);
    if (b.bytes < bytes) {
        if (b.p) (void)hipFree(b.p);
        b.p = nullptr;
        b.bytes = 0;
        SG_TRY(s, hipMalloc(&b.p, bytes));
        b.bytes = bytes;
    }
    *out = (T *)b.p;
    return GS_OK;
}

#define SG_NEED(s, which, count, ptr)                       \
    do {                                                    \
        gs_status st_ = need((s), (which), (count), &(ptr)); \
        if (st_ != GS_OK) return st_;                       \
    } while (0)

// Forward pass for `rows` rows per member.  X: bf16 [rows][kPad] with
// member stride xstride (0: all members read the same rows).  Zbuf null
// skips the pre-activations (inference).
gs_status forward(gs_surrogate *s, const __bf16 *X, size_t xstride, int rows, float *Zbuf, __bf16 *Act,
                  float *Out) {
    const int H = (int)s->cfg.hidden;
    const size_t layer_stride = (size_t)s->E * rows * H;
    for (int l = 0; l < s->L; ++l) {
        GemmArgs g{};
        const bool last = l == s->L - 1;
        g.A = l == 0 ? X : Act + (size_t)(l - 1) * layer_stride;
        g.strideA = l == 0 ? xstride : (size_t)rows * H;
        g.lda = s->dims[l];
        g.B = s->Pb + s->woff[l];
        g.strideB = s->Pm;
        g.ldb = s->dims[l];
        g.M = rows;
        g.N = s->dims[l + 1];
        g.K = s->dims[l];
        g.ldc = s->dims[l + 1];
        g.strideC = (size_t)rows * s->dims[l + 1];
        g.bias = s->P + s->boff[l];
        g.strideBias = s->Pm;
        if (last) {
            g.Cf = Out;
            SG_TRY(s, sg_launch_gemm(false, false, EPI_OUT, g, s->E, s->stream));
        } else {
            g.Zf = Zbuf ? Zbuf + (size_t)l * layer_stride : nullptr;
            g.Cb = Act + (size_t)l * layer_stride;
            SG_TRY(s, sg_launch_gemm(false, false, EPI_HIDDEN, g, s->E, s->stream));
        }
    }
    return GS_OK;
}

// Inference forward pass into Out [E][rows][kPad]: the fused kernel when the
// network has its shape (hidden 256, at most kMlpMaxLayers weight layers),
// otherwise the layer-by-layer GEMMs through the activation buffer.
bool fused_shape(const gs_surrogate *s) {
    return s->cfg.hidden == 256 && s->L >= 2 && s->L <= kMlpMaxLayers && s->dims[0] == 32 && s->dims[s->L] == 32;
}

// The parameters as the fused kernels take them.
TrainArgs param_args(const gs_surrogate *s) {
    TrainArgs g{};
    g.L = s->L;
    g.P = s->P; g.Mo = s->Mo; g.Ve = s->Ve; g.G = s->G;
    g.Pb = s->Pb; g.PbT = s->PbT;
    g.Pm = s->Pm;
    for (int l = 0; l < s->L; ++l) {
        g.woff[l] = s->woff[l];
        g.boff[l] = s->boff[l];
    }
    return g;
}

// The buffers and parameters of the fused training step for `rows` rows.
gs_status train_args(gs_surrogate *s, int rows, TrainArgs &g) {
    const size_t E = (size_t)s->E, B = (size_t)rows, hidden = (size_t)(s->L - 1) * E * 256;
    g = param_args(s);
    g.rows = rows;
    SG_NEED(s, B_BX, E * kPad * B, g.XT);
    SG_NEED(s, B_ACT, hidden * B, g.ActT);
    SG_NEED(s, B_DZT, hidden * B, g.dZT);
    SG_NEED(s, B_DZF, hidden * B, g.dZf);
    SG_NEED(s, B_DYB, E * kPad * B, g.dYT);
    SG_NEED(s, B_DYF, E * kPad * B, g.dYf);
    return GS_OK;
}

// The members' outputs [E][rows][kPad] of raw inputs x [rows][n_inputs] in
// device memory, or for fused shapes pinned host memory.
gs_status forward_infer(gs_surrogate *s, const float *x, int rows, float *Out) {
    const uint32_t ni = s->cfg.n_inputs;
    if (fused_shape(s)) {
        MlpArgs g{};
        g.x = x;
        g.ni = (int)ni;
        std::copy(s->mu, s->mu + ni, g.mu);
        std::copy(s->sd, s->sd + ni, g.sd);
        g.rows = rows;
        g.L = s->L;
        g.Pb = s->Pb;
        g.P = s->P;
        g.Pm = s->Pm;
        for (int l = 0; l < s->L; ++l) {
            g.woff[l] = s->woff[l];
            g.boff[l] = s->boff[l];
        }
        g.Out = Out;
        SG_TRY(s, sg_launch_mlp_forward(g, s->E, s->stream));
        return GS_OK;
    }
    __bf16 *act, *X;
    SG_NEED(s, B_ACT, (size_t)(s->L - 1) * s->E * rows * s->cfg.hidden, act);
    SG_NEED(s, B_X, (size_t)rows * kPad, X);
    SG_TRY(s, sg_launch_standardise(x, rows, (int)ni, kPad, s->mu, s->sd, X, s->stream));
    return forward(s, X, 0, rows, nullptr, act, Out);
}

// Backward pass from dY (fp32 and bf16 [E][rows][kPad]) into s->G.
gs_status backward(gs_surrogate *s, const __bf16 *X, size_t xstride, int rows, const float *Zbuf,
                   const __bf16 *Act, const float *dYf, const __bf16 *dYb) {
    const int H = (int)s->cfg.hidden;
    const size_t layer_stride = (size_t)s->E * rows * H;
    float *dzf[2];
    __bf16 *dzb[2];
    SG_NEED(s, B_DZF0, layer_stride, dzf[0]);
    SG_NEED(s, B_DZB0, layer_stride, dzb[0]);
    SG_NEED(s, B_DZF1, layer_stride, dzf[1]);
    SG_NEED(s, B_DZB1, layer_stride, dzb[1]);
    const float *cur_f = dYf;
    const __bf16 *cur_b = dYb;
    for (int l = s->L - 1; l >= 0; --l) {
        const int out_w = s->dims[l + 1], in_w = s->dims[l];
        const __bf16 *in_act = l == 0 ? X : Act + (size_t)(l - 1) * layer_stride;
        const size_t in_stride = l == 0 ? xstride : (size_t)rows * H;
        // dW[o][i] = sum_b dZ[b][o] in[b][i]
        GemmArgs gw{};
        gw.A = cur_b;
        gw.strideA = (size_t)rows * out_w;
        gw.lda = out_w;
        gw.B = in_act;
        gw.strideB = in_stride;
        gw.ldb = in_w;
        gw.M = out_w;
        gw.N = in_w;
        gw.K = rows;
        gw.ldc = in_w;
        gw.strideC = s->Pm;
        gw.Cf = s->G + s->woff[l];
        SG_TRY(s, sg_launch_gemm(true, true, EPI_STORE, gw, s->E, s->stream));
        SG_TRY(s, sg_launch_colsum(cur_f, rows, out_w, (size_t)rows * out_w, s->G + s->boff[l], s->Pm, s->E,
                                   s->stream));
        if (l == 0) break;
        // dZ_prev[b][i] = (sum_o dZ[b][o] W[o][i]) silu'(Z_prev[b][i])
        const int nxt = (l & 1);
        GemmArgs gd{};
        gd.A = cur_b;
        gd.strideA = (size_t)rows * out_w;
        gd.lda = out_w;
        gd.B = s->Pb + s->woff[l];
        gd.strideB = s->Pm;
        gd.ldb = in_w;
        gd.M = rows;
        gd.N = in_w;
        gd.K = out_w;
        gd.ldc = in_w;
        gd.strideC = (size_t)rows * in_w;
        gd.Zf = const_cast<float *>(Zbuf) + (size_t)(l - 1) * layer_stride;
        gd.Cf = dzf[nxt];
        gd.Cb = dzb[nxt];
        SG_TRY(s, sg_launch_gemm(false, true, EPI_DSILU, gd, s->E, s->stream));
        cur_f = dzf[nxt];
        cur_b = dzb[nxt];
    }
    return GS_OK;
}

// fp32 rows [n][n_inputs] in host memory -> standardised, padded bf16 rows
// [n][kPad] on the device.
gs_status upload_inputs(gs_surrogate *s, const float *x, uint32_t n, __bf16 **out) {
    const uint32_t ni = s->cfg.n_inputs;
    float *xf;
    __bf16 *xb;
    SG_NEED(s, B_XF, (size_t)n * ni, xf);
    SG_NEED(s, B_X, (size_t)n * kPad, xb);
    SG_TRY(s, hipMemcpyAsync(xf, x, (size_t)n * ni * sizeof(float), hipMemcpyHostToDevice, s->stream));
    SG_TRY(s, sg_launch_standardise(xf, (int)n, (int)ni, kPad, s->mu, s->sd, xb, s->stream));
    SG_TRY(s, hipStreamSynchronize(s->stream));
    *out = xb;
    return GS_OK;
}

std::vector<float> pad_rows(const float *v, uint32_t n, uint32_t width) {
    std::vector<float> h((size_t)n * kPad, 0.0f);
    for (uint32_t r = 0; r < n; ++r)
        for (uint32_t c = 0; c < width; ++c) h[(size_t)r * kPad + c] = v[(size_t)r * width + c];
    return h;
}

bool check_cfg(const gs_surrogate_config *c, std::string &msg) {
    if (c->n_members < 1 || c->n_members > 64) { msg = "n_members must be 1..64"; return false; }
    if (c->n_inputs < 1 || c->n_inputs > GS_SG_MAX_INPUTS) { msg = "n_inputs must be 1..32"; return false; }
    if (c->n_outputs < 1 || c->n_outputs > GS_SG_MAX_OUTPUTS) { msg = "n_outputs must be 1..32"; return false; }
    if (c->hidden < 64 || c->hidden % 64 || c->hidden > 4096) { msg = "hidden must be a multiple of 64 up to 4096"; return false; }
    if (c->n_hidden_layers < 1 || c->n_hidden_layers > 16) { msg = "n_hidden_layers must be 1..16"; return false; }
    if (c->batch < 64 || c->batch % 64 || c->batch > 65536) { msg = "batch must be a multiple of 64 up to 65536"; return false; }
    if (!(c->lr > 0) || !(c->beta1 >= 0 && c->beta1 < 1) || !(c->beta2 >= 0 && c->beta2 < 1) || !(c->eps > 0)) {
        msg = "bad Adam hyper-parameters";
        return false;
    }
    return true;
}

}  // namespace

extern "C" {

gs_status gs_surrogate_default_config(gs_surrogate_config *c) {
    if (!c) return GS_ERR_INVALID_ARG;
    std::memset(c, 0, sizeof *c);
    c->n_members = 4;
    c->n_inputs = 8;
    c->n_outputs = 30;
    c->hidden = 256;
    c->n_hidden_layers = 4;
    c->batch = 1024;
    c->seed = 1;
    c->lr = 1e-3f;
    c->beta1 = 0.9f;
    c->beta2 = 0.999f;
    c->eps = 1e-8f;
    c->weight_decay = 0.0f;
    c->std_limit = 0.01f;
    c->std_outputs = 0xffffffffu;
    return GS_OK;
}

const char *gs_surrogate_last_error(const gs_surrogate *s) { return s ? s->err.c_str() : "no surrogate"; }

gs_status gs_surrogate_create(int device, const gs_surrogate_config *cfg, gs_surrogate **out) {
    if (!out || !cfg) return GS_ERR_INVALID_ARG;
    *out = nullptr;
    std::string msg;
    if (!check_cfg(cfg, msg)) return GS_ERR_INVALID_ARG;
    int nd = 0;
    if (hipGetDeviceCount(&nd) != hipSuccess || nd <= 0) return GS_ERR_NO_DEVICE;
    if (device < 0 || device >= nd) return GS_ERR_INVALID_ARG;
    gs_surrogate *s = new gs_surrogate();
    s->device = device;
    s->cfg = *cfg;
    s->E = (int)cfg->n_members;
    s->L = (int)cfg->n_hidden_layers + 1;
    s->bufs.resize(B_COUNT_);
    s->dims.push_back(kPad);
    for (uint32_t i = 0; i < cfg->n_hidden_layers; ++i) s->dims.push_back((int)cfg->hidden);
    s->dims.push_back(kPad);
    size_t off = 0;
    for (int l = 0; l < s->L; ++l) {
        s->woff.push_back(off);
        off += (size_t)s->dims[l + 1] * s->dims[l];
        s->boff.push_back(off);
        off += (size_t)s->dims[l + 1];
    }
    s->Pm = (off + 7) / 8 * 8;   // keeps every member's block 16-byte aligned in bf16
    for (int i = 0; i < GS_SG_MAX_INPUTS; ++i) { s->mu[i] = 0.f; s->sd[i] = 1.f; s->lo[i] = -INFINITY; s->hi[i] = INFINITY; }
    hipError_t e = hipSetDevice(device);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking);
    const size_t np = (size_t)s->E * s->Pm;
    if (e == hipSuccess) e = hipMalloc((void **)&s->P, np * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&s->G, np * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&s->Mo, np * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&s->Ve, np * sizeof(float));
    if (e == hipSuccess) e = hipMalloc((void **)&s->Pb, np * sizeof(__bf16));
    if (e == hipSuccess && fused_shape(s)) e = hipMalloc((void **)&s->PbT, np * sizeof(__bf16));
    if (e != hipSuccess) {
        gs_surrogate_destroy(s);
        return e == hipErrorOutOfMemory ? GS_ERR_OUT_OF_MEMORY : GS_ERR_HIP;
    }
    // He-uniform weights over the real fan-in, zero biases and padding;
    // the output layer starts ten times smaller.
    std::vector<float> h(np, 0.0f);
    for (int m = 0; m < s->E; ++m) {
        std::mt19937_64 rng(cfg->seed * 0x9E3779B97F4A7C15ull + (uint64_t)m * 1000003ull + 17);
        for (int l = 0; l < s->L; ++l) {
            const int out_real = l == s->L - 1 ? (int)cfg->n_outputs : s->dims[l + 1];
            const int in_real = l == 0 ? (int)cfg->n_inputs : s->dims[l];
            const float a = std::sqrt(6.0f / in_real) * (l == s->L - 1 ? 0.1f : 1.0f);
            std::uniform_real_distribution<float> U(-a, a);
            for (int o = 0; o < out_real; ++o)
                for (int i = 0; i < in_real; ++i)
                    h[(size_t)m * s->Pm + s->woff[l] + (size_t)o * s->dims[l] + i] = U(rng);
        }
    }
    gs_status st = gs_surrogate_set_params(s, h.data(), h.size());
    if (st != GS_OK) {
        gs_surrogate_destroy(s);
        return st;
    }
    *out = s;
    return GS_OK;
}

void gs_surrogate_destroy(gs_surrogate *s) {
    if (!s) return;
    (void)hipSetDevice(s->device);
    if (s->stream) (void)hipStreamSynchronize(s->stream);
    for (DevBuf &b : s->bufs)
        if (b.p) (void)hipFree(b.p);
    for (hipEvent_t e : s->pin_done)
        if (e) (void)hipEventDestroy(e);
    if (s->pin) (void)hipHostFree(s->pin);
    for (void *p : {(void *)s->P, (void *)s->G, (void *)s->Mo, (void *)s->Ve, (void *)s->Pb, (void *)s->PbT})
        if (p) (void)hipFree(p);
    if (s->stream) (void)hipStreamDestroy(s->stream);
    delete s;
}

gs_status gs_surrogate_layout(const gs_surrogate *s, uint64_t *per_member, uint64_t *layout, uint32_t cap) {
    if (!s) return GS_ERR_INVALID_ARG;
    if (per_member) *per_member = s->Pm;
    if (layout) {
        if (cap < 4u * (uint32_t)s->L) return GS_ERR_INVALID_ARG;
        for (int l = 0; l < s->L; ++l) {
            layout[4 * l + 0] = s->woff[l];
            layout[4 * l + 1] = s->boff[l];
            layout[4 * l + 2] = (uint64_t)s->dims[l + 1];
            layout[4 * l + 3] = (uint64_t)s->dims[l];
        }
    }
    return GS_OK;
}

gs_status gs_surrogate_get_params(gs_surrogate *s, float *p, uint64_t count) {
    if (!s || !p) return GS_ERR_INVALID_ARG;
    if (count != (uint64_t)s->E * s->Pm) return fail(s, GS_ERR_INVALID_ARG, "count must be %zu", (size_t)s->E * s->Pm);
    SG_TRY(s, hipSetDevice(s->device));
    SG_TRY(s, hipMemcpyAsync(p, s->P, count * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    SG_TRY(s, hipStreamSynchronize(s->stream));
    return GS_OK;
}

gs_status gs_surrogate_set_params(gs_surrogate *s, const float *p, uint64_t count) {
    if (!s || !p) return GS_ERR_INVALID_ARG;
    if (count != (uint64_t)s->E * s->Pm) return fail(s, GS_ERR_INVALID_ARG, "count must be %zu", (size_t)s->E * s->Pm);
    SG_TRY(s, hipSetDevice(s->device));
    SG_TRY(s, hipMemcpyAsync(s->P, p, count * sizeof(float), hipMemcpyHostToDevice, s->stream));
    SG_TRY(s, hipMemsetAsync(s->Mo, 0, count * sizeof(float), s->stream));
    SG_TRY(s, hipMemsetAsync(s->Ve, 0, count * sizeof(float), s->stream));
    if (fused_shape(s)) SG_TRY(s, sg_launch_pack(param_args(s), s->E, s->stream));
    else SG_TRY(s, sg_launch_to_bf16(s->P, s->Pb, count, s->stream));
    SG_TRY(s, hipStreamSynchronize(s->stream));
    s->step = 0;
    return GS_OK;
}

gs_status gs_surrogate_get_normalization(const gs_surrogate *s, float *mean, float *sd, float *lo, float *hi) {
    if (!s) return GS_ERR_INVALID_ARG;
    for (uint32_t i = 0; i < s->cfg.n_inputs; ++i) {
        if (mean) mean[i] = s->mu[i];
        if (sd) sd[i] = s->sd[i];
        if (lo) lo[i] = s->lo[i];
        if (hi) hi[i] = s->hi[i];
    }
    return GS_OK;
}

gs_status gs_surrogate_set_normalization(gs_surrogate *s, const float *mean, const float *sd, const float *lo,
                                         const float *hi) {
    if (!s || !mean || !sd || !lo || !hi) return GS_ERR_INVALID_ARG;
    for (uint32_t i = 0; i < s->cfg.n_inputs; ++i) {
        if (!(sd[i] > 0) || !std::isfinite(mean[i])) return fail(s, GS_ERR_INVALID_ARG, "bad normalization");
        s->mu[i] = mean[i];
        s->sd[i] = sd[i];
        s->lo[i] = lo[i];
        s->hi[i] = hi[i];
    }
    s->normalized = true;
    return GS_OK;
}

gs_status gs_surrogate_train(gs_surrogate *s, const float *x, const float *y, const float *w, uint32_t n,
                             uint32_t epochs, float *last_loss) {
    if (!s) return GS_ERR_INVALID_ARG;
    if (!x || !y || !w) return fail(s, GS_ERR_INVALID_ARG, "NULL data");
    const int B = (int)s->cfg.batch;
    if (n < (uint32_t)B) return fail(s, GS_ERR_INVALID_ARG, "need at least one minibatch (%d rows)", B);
    SG_TRY(s, hipSetDevice(s->device));
    const uint32_t ni = s->cfg.n_inputs, no = s->cfg.n_outputs;
    for (size_t i = 0; i < (size_t)n * no; ++i)
        if (!std::isfinite(y[i]) && w[i] != 0.0f) return fail(s, GS_ERR_INVALID_ARG, "non-finite target with weight");
    if (!s->normalized) {
        for (uint32_t c = 0; c < ni; ++c) {
            double m = 0, m2 = 0;
            float lo = INFINITY, hi = -INFINITY;
            for (uint32_t r = 0; r < n; ++r) {
                const double v = x[(size_t)r * ni + c];
                m += v;
                m2 += v * v;
                lo = std::min(lo, (float)v);
                hi = std::max(hi, (float)v);
            }
            m /= n;
            const double var = std::max(0.0, m2 / n - m * m);
            s->mu[c] = (float)m;
            s->sd[c] = var > 1e-12 ? (float)std::sqrt(var) : 1.0f;
            s->lo[c] = lo;
            s->hi[c] = hi;
        }
        s->normalized = true;
    }
    __bf16 *X;
    gs_status st = upload_inputs(s, x, n, &X);
    if (st != GS_OK) return st;
    std::vector<float> yh = pad_rows(y, n, no), wh = pad_rows(w, n, no);
    for (size_t i = 0; i < yh.size(); ++i)
        if (wh[i] == 0.0f) yh[i] = 0.0f;   // unweighted targets may be NaN (empty bins)
    float *Y, *W;
    SG_NEED(s, B_Y, yh.size(), Y);
    SG_NEED(s, B_W, wh.size(), W);
    SG_TRY(s, hipMemcpyAsync(Y, yh.data(), yh.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
    SG_TRY(s, hipMemcpyAsync(W, wh.data(), wh.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
    const int E = s->E, H = (int)s->cfg.hidden;
    const bool fused = fused_shape(s);
    uint32_t *idx;
    __bf16 *bx = nullptr, *act = nullptr, *dyb = nullptr;
    float *by = nullptr, *bw = nullptr, *Z = nullptr, *out = nullptr, *dyf = nullptr, *wsum, *loss;
    const int steps = (int)(n / (uint32_t)B);
    const int parts = fused ? B / 16 : 8;
    TrainArgs ta;
    SG_NEED(s, B_IDX, (size_t)E * B * steps, idx);
    if (fused) {
        st = train_args(s, B, ta);
        if (st != GS_OK) return st;
        ta.X = X;
        ta.Y = Y;
        ta.W = W;
    } else {
        SG_NEED(s, B_BX, (size_t)E * B * kPad, bx);
        SG_NEED(s, B_BY, (size_t)E * B * kPad, by);
        SG_NEED(s, B_BW, (size_t)E * B * kPad, bw);
        SG_NEED(s, B_Z, (size_t)(s->L - 1) * E * B * H, Z);
        SG_NEED(s, B_ACT, (size_t)(s->L - 1) * E * B * H, act);
        SG_NEED(s, B_OUT, (size_t)E * B * kPad, out);
        SG_NEED(s, B_DYF, (size_t)E * B * kPad, dyf);
        SG_NEED(s, B_DYB, (size_t)E * B * kPad, dyb);
    }
    SG_NEED(s, B_WSUM, fused ? (size_t)E * steps : (size_t)E, wsum);
    SG_NEED(s, B_LOSS, (size_t)E * parts * steps, loss);
    std::vector<uint32_t> order(n), hidx((size_t)E * B * steps);
    std::vector<float> hl((size_t)E * parts * steps);
    const gs_surrogate_config &c = s->cfg;
    double last = 0.0;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        for (int m = 0; m < E; ++m) {
            std::mt19937_64 rng(c.seed ^ (0xD1B54A32D192ED03ull * (s->step + 1)) ^ ((uint64_t)m << 48));
            for (uint32_t i = 0; i < n; ++i) order[i] = i;
            std::shuffle(order.begin(), order.end(), rng);
            for (int k = 0; k < steps; ++k)
                std::copy(order.begin() + (size_t)k * B, order.begin() + (size_t)(k + 1) * B,
                          hidx.begin() + ((size_t)k * E + m) * B);
        }
        SG_TRY(s, hipMemcpyAsync(idx, hidx.data(), hidx.size() * sizeof(uint32_t), hipMemcpyHostToDevice, s->stream));
        if (fused) SG_TRY(s, sg_launch_wsum(W, idx, B, steps, E, wsum, s->stream));
        for (int k = 0; k < steps; ++k) {
            if (fused) {
                ta.idx = idx + (size_t)k * E * B;
                ta.wsum = wsum + (size_t)k * E;
                ta.loss_part = loss + (size_t)k * E * parts;
                SG_TRY(s, sg_launch_train_tile(ta, E, s->stream));
                ++s->step;
                const AdamArgs aa{c.lr, c.beta1, c.beta2, c.eps, c.weight_decay, 1.0f - std::pow(c.beta1, (float)s->step),
                                  1.0f - std::pow(c.beta2, (float)s->step)};
                SG_TRY(s, sg_launch_train_weights(ta, &aa, E, s->stream));
                continue;
            }
            SG_TRY(s, sg_launch_gather(X, Y, W, idx + (size_t)k * E * B, B, kPad, kPad, bx, by, bw, E, s->stream));
            st = forward(s, bx, (size_t)B * kPad, B, Z, act, out);
            if (st != GS_OK) return st;
            SG_TRY(s, sg_launch_loss(out, by, bw, B * kPad, (size_t)B * kPad, (size_t)B * kPad, wsum, dyf, dyb,
                                     loss + (size_t)k * E * parts, parts, E, s->stream));
            st = backward(s, bx, (size_t)B * kPad, B, Z, act, dyf, dyb);
            if (st != GS_OK) return st;
            ++s->step;
            const float c1 = 1.0f - std::pow(c.beta1, (float)s->step), c2 = 1.0f - std::pow(c.beta2, (float)s->step);
            SG_TRY(s, sg_launch_adam(s->P, s->G, s->Mo, s->Ve, s->Pb, (size_t)E * s->Pm, c.lr, c.beta1, c.beta2,
                                     c.eps, c.weight_decay, c1, c2, s->stream));
        }
        if (ep + 1 == epochs) {
            SG_TRY(s, hipMemcpyAsync(hl.data(), loss, hl.size() * sizeof(float), hipMemcpyDeviceToHost, s->stream));
            SG_TRY(s, hipStreamSynchronize(s->stream));
            double tot = 0;
            for (float v : hl) tot += v;
            last = tot / ((double)steps * E);
        }
    }
    SG_TRY(s, hipStreamSynchronize(s->stream));
    if (last_loss) *last_loss = (float)last;
    return GS_OK;
}

gs_status gs_surrogate_gradients(gs_surrogate *s, const float *x, const float *y, const float *w, uint32_t n,
                                 float *grads, float *loss_out) {
    if (!s) return GS_ERR_INVALID_ARG;
    if (!x || !y || !w || !grads || n == 0 || n > 65536) return fail(s, GS_ERR_INVALID_ARG, "bad arguments");
    SG_TRY(s, hipSetDevice(s->device));
    const uint32_t rows = (n + 63) / 64 * 64;   // padded rows carry zero weight
    std::vector<float> xp((size_t)rows * s->cfg.n_inputs, 0.0f), yp((size_t)rows * s->cfg.n_outputs, 0.0f),
        wp((size_t)rows * s->cfg.n_outputs, 0.0f);
    std::copy(x, x + (size_t)n * s->cfg.n_inputs, xp.begin());
    std::copy(y, y + (size_t)n * s->cfg.n_outputs, yp.begin());
    std::copy(w, w + (size_t)n * s->cfg.n_outputs, wp.begin());
    __bf16 *X;
    gs_status st = upload_inputs(s, xp.data(), rows, &X);
    if (st != GS_OK) return st;
    const int E = s->E, H = (int)s->cfg.hidden;
    std::vector<float> yh = pad_rows(yp.data(), rows, s->cfg.n_outputs), wh = pad_rows(wp.data(), rows, s->cfg.n_outputs);
    const bool fused = fused_shape(s);
    const int parts = fused ? (int)rows / 16 : 8;
    float *by, *bw, *wsum, *loss;
    SG_NEED(s, B_WSUM, (size_t)E, wsum);
    SG_NEED(s, B_LOSS, (size_t)E * parts, loss);
    std::vector<float> ye, we;   // must outlive the copies
    if (fused) {   // every member reads the same rows
        SG_NEED(s, B_BY, yh.size(), by);
        SG_NEED(s, B_BW, wh.size(), bw);
        SG_TRY(s, hipMemcpyAsync(by, yh.data(), yh.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
        SG_TRY(s, hipMemcpyAsync(bw, wh.data(), wh.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
        TrainArgs ta;
        st = train_args(s, (int)rows, ta);
        if (st != GS_OK) return st;
        ta.X = X;
        ta.Y = by;
        ta.W = bw;
        ta.wsum = wsum;
        ta.loss_part = loss;
        for (int m = 0; m < E; ++m) SG_TRY(s, sg_launch_wsum(bw, nullptr, (int)rows, 1, 1, wsum + m, s->stream));
        SG_TRY(s, sg_launch_train_tile(ta, E, s->stream));
        SG_TRY(s, sg_launch_train_weights(ta, nullptr, E, s->stream));
    } else {
        float *Z, *out, *dyf;
        __bf16 *act, *dyb;
        // the same rows for every member
        for (int m = 0; m < E; ++m) {
            ye.insert(ye.end(), yh.begin(), yh.end());
            we.insert(we.end(), wh.begin(), wh.end());
        }
        SG_NEED(s, B_BY, ye.size(), by);
        SG_NEED(s, B_BW, we.size(), bw);
        SG_NEED(s, B_Z, (size_t)(s->L - 1) * E * rows * H, Z);
        SG_NEED(s, B_ACT, (size_t)(s->L - 1) * E * rows * H, act);
        SG_NEED(s, B_OUT, (size_t)E * rows * kPad, out);
        SG_NEED(s, B_DYF, (size_t)E * rows * kPad, dyf);
        SG_NEED(s, B_DYB, (size_t)E * rows * kPad, dyb);
        SG_TRY(s, hipMemcpyAsync(by, ye.data(), ye.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
        SG_TRY(s, hipMemcpyAsync(bw, we.data(), we.size() * sizeof(float), hipMemcpyHostToDevice, s->stream));
        st = forward(s, X, 0, (int)rows, Z, act, out);
        if (st != GS_OK) return st;
        SG_TRY(s, sg_launch_loss(out, by, bw, (int)rows * kPad, (size_t)rows * kPad, (size_t)rows * kPad, wsum, dyf, dyb,
                                 loss, parts, E, s->stream));
        // The first layer reads the shared inputs (member stride 0).
        st = backward(s, X, 0, (int)rows, Z, act, dyf, dyb);
        if (st != GS_OK) return st;
    }
    SG_TRY(s, hipMemcpyAsync(grads, s->G, (size_t)E * s->Pm * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    std::vector<float> hl((size_t)E * parts);
    SG_TRY(s, hipMemcpyAsync(hl.data(), loss, hl.size() * sizeof(float), hipMemcpyDeviceToHost, s->stream));
    SG_TRY(s, hipStreamSynchronize(s->stream));
    if (loss_out)
        for (int m = 0; m < E; ++m) {
            double t = 0;
            for (int p = 0; p < parts; ++p) t += hl[(size_t)m * parts + p];
            loss_out[m] = (float)t;
        }
    return GS_OK;
}

// Whether the inputs share no memory with the outputs.
static bool apart(const gs_surrogate *s, const float *x, size_t n, const float *mean, const float *sd,
                  const uint8_t *fallback) {
    const uintptr_t b = (uintptr_t)x, e = b + n * s->cfg.n_inputs * sizeof(float);
    auto from_x = [&](const void *p, size_t bytes) { return !p || (uintptr_t)p >= e || (uintptr_t)p + bytes <= b; };
    const size_t out = n * s->cfg.n_outputs * sizeof(float);
    return from_x(mean, out) && from_x(sd, out) && from_x(fallback, n);
}

// Whether kernels of this surrogate may read x in place: memory of its device,
// apart from the outputs (the statistics read the inputs again after other
// queries' results are written).
static bool reads_in_place(const gs_surrogate *s, const float *x, size_t n, const float *mean, const float *sd,
                           const uint8_t *fallback) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, x) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeDevice && a.device == s->device && apart(s, x, n, mean, sd, fallback);
}

// Pinned memory for host predictions of `bytes` per half, at most kHostChunk rows
// each; false where there is none.
static bool pin_halves(gs_surrogate *s, size_t bytes) {
    for (hipEvent_t &e : s->pin_done)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            e = nullptr;
            return false;
        }
    if (s->pin_half >= bytes) return true;
    if (s->pin) (void)hipHostFree(s->pin);
    s->pin = nullptr;
    s->pin_half = 0;
    if (hipHostMalloc((void **)&s->pin, 2 * bytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        s->pin = nullptr;
        return false;
    }
    s->pin_half = bytes;
    return true;
}

// The statistics of one block of rows whose inputs x and outputs the kernels can
// reach.
static gs_status infer_rows(gs_surrogate *s, const float *x, uint32_t rows, float *mean, float *sd, uint8_t *fallback) {
    const int E = s->E, no = (int)s->cfg.n_outputs, ni = (int)s->cfg.n_inputs;
    float *out;
    SG_NEED(s, B_OUT, (size_t)E * rows * kPad, out);
    gs_status st = forward_infer(s, x, (int)rows, out);
    if (st != GS_OK) return st;
    SG_TRY(s, sg_launch_query_stats(out, E, (int)rows, no, x, ni, s->cfg.std_outputs, s->cfg.std_limit, s->lo, s->hi,
                                    mean, sd, fallback, s->stream));
    return GS_OK;
}

// Host buffers through pinned memory that the kernels write themselves, in
// blocks of kHostChunk rows: while the device works on one block the host copies
// the results of the one before.  Pageable copies, four to a call with one in and
// three out, were two thirds of a small call and took turns with the kernels in a
// large one.  In us, before / now: 1 row 52 / 29, 512 82 / 33, 4,096 87 / 63, 20,011
// 281 / 193 (four members, means and flags).
// The inputs of up to kDirectRows rows are read from pinned memory too (each by
// every member); of more, copied first (4,096 rows: 63 read, 70 copied; 20,011: 281, 251).
constexpr uint32_t kHostChunk = 8192, kDirectRows = 4096;
static gs_status predict_pinned(gs_surrogate *s, const float *x, uint32_t n, float *mean, float *sd, uint8_t *fallback) {
    const size_t no = s->cfg.n_outputs, ni = s->cfg.n_inputs;
    const size_t most = std::min(n, kHostChunk);
    // a half: inputs, means, spreads, flags
    auto half = [&](uint32_t c) { return s->pin + (c & 1) * s->pin_half; };
    auto take = [&](uint32_t c) -> gs_status {   // results of block c, when they are there
        const size_t r0 = (size_t)c * kHostChunk, rows = std::min<size_t>(n - r0, kHostChunk);
        SG_TRY(s, hipEventSynchronize(s->pin_done[c & 1]));
        const float *m = (const float *)half(c) + most * ni, *d = m + most * no;
        const uint8_t *f = (const uint8_t *)(d + most * no);
        if (mean) std::memcpy(mean + r0 * no, m, rows * no * sizeof(float));
        if (sd) std::memcpy(sd + r0 * no, d, rows * no * sizeof(float));
        if (fallback) std::memcpy(fallback + r0, f, rows);
        return GS_OK;
    };
    const uint32_t blocks = (n - 1) / kHostChunk + 1;   // n > 0
    gs_status st = GS_OK;
    for (uint32_t c = 0; c < blocks && st == GS_OK; ++c) {
        if (c >= 2 && (st = take(c - 2)) != GS_OK) break;
        const size_t r0 = (size_t)c * kHostChunk;
        const uint32_t rows = (uint32_t)std::min<size_t>(n - r0, kHostChunk);
        float *px = (float *)half(c), *m = px + most * ni, *d = m + most * no;
        std::memcpy(px, x + r0 * ni, rows * ni * sizeof(float));
        const float *in = px;
        if (rows > kDirectRows) {
            float *xf;
            SG_NEED(s, B_XF, (size_t)rows * ni, xf);
            SG_TRY(s, hipMemcpyAsync(xf, px, rows * ni * sizeof(float), hipMemcpyHostToDevice, s->stream));
            in = xf;
        }
        st = infer_rows(s, in, rows, mean ? m : nullptr, sd ? d : nullptr, fallback ? (uint8_t *)(d + most * no) : nullptr);
        if (st == GS_OK) SG_TRY(s, hipEventRecord(s->pin_done[c & 1], s->stream));
    }
    if (st == GS_OK && blocks > 1) st = take(blocks - 2);
    if (st == GS_OK) st = take(blocks - 1);
    return st;
}

// Both predict entry points: host buffers (through pinned memory, or where
// there is none, or the inputs share memory with the outputs, copied through the
// surrogate's stream) or device buffers (read and written in place).
static gs_status predict_rows(gs_surrogate *s, const float *x, uint32_t n, float *mean, float *sd,
                              uint8_t *fallback, bool on_device) {
    if (!s) return GS_ERR_INVALID_ARG;
    if (!x && n) return fail(s, GS_ERR_INVALID_ARG, "NULL inputs");
    if (n == 0) return GS_OK;
    SG_TRY(s, hipSetDevice(s->device));
    const uint32_t no = s->cfg.n_outputs, ni = s->cfg.n_inputs;
    // (results go out block by block before later inputs are read)
    if (!on_device && apart(s, x, n, mean, sd, fallback) &&
        pin_halves(s, (size_t)std::min(n, kHostChunk) * ((ni + 2 * no) * sizeof(float) + 1) + 64))
        return predict_pinned(s, x, n, mean, sd, fallback);
    const uint32_t chunk = 65536;
    const bool in_place = on_device && reads_in_place(s, x, n, mean, sd, fallback);
    for (uint32_t r0 = 0; r0 < n; r0 += chunk) {
        const uint32_t rows = std::min(chunk, n - r0);
        const float *xr = x + (size_t)r0 * ni;
        float *dm = mean ? mean + (size_t)r0 * no : nullptr, *ds = sd ? sd + (size_t)r0 * no : nullptr;
        uint8_t *fl = fallback ? fallback + r0 : nullptr;
        if (!in_place) {
            float *xf;
            SG_NEED(s, B_XF, (size_t)rows * ni, xf);
            SG_TRY(s, hipMemcpyAsync(xf, xr, (size_t)rows * ni * sizeof(float),
                                     on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, s->stream));
            xr = xf;
        }
        if (!on_device) {
            if (mean) SG_NEED(s, B_MEAN, (size_t)rows * no, dm);
            if (sd) SG_NEED(s, B_SD, (size_t)rows * no, ds);
            if (fallback) SG_NEED(s, B_FLAGS, (size_t)rows, fl);
        }
        const gs_status st = infer_rows(s, xr, rows, dm, ds, fl);
        if (st != GS_OK) return st;
        if (!on_device) {
            const size_t bytes = (size_t)rows * no * sizeof(float);
            if (fallback) SG_TRY(s, hipMemcpyAsync(fallback + r0, fl, rows, hipMemcpyDeviceToHost, s->stream));
            if (mean) SG_TRY(s, hipMemcpyAsync(mean + (size_t)r0 * no, dm, bytes, hipMemcpyDeviceToHost, s->stream));
            if (sd) SG_TRY(s, hipMemcpyAsync(sd + (size_t)r0 * no, ds, bytes, hipMemcpyDeviceToHost, s->stream));
        }
    }
    // the buffers are the next call's, and the outputs the caller's
    SG_TRY(s, hipStreamSynchronize(s->stream));
    return GS_OK;
}

gs_status gs_surrogate_predict(gs_surrogate *s, const float *x, uint32_t n, float *mean, float *sd,
                               uint8_t *fallback) {
    return predict_rows(s, x, n, mean, sd, fallback, false);
}

gs_status gs_surrogate_predict_device(gs_surrogate *s, const float *x, uint32_t n, float *mean, float *sd,
                                      uint8_t *fallback) {
    return predict_rows(s, x, n, mean, sd, fallback, true);
}

}  // extern "C"
