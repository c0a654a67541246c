// Learned initial guess for the Stokes solve: host side of the U-Net.
//
// The network maps two fields resampled to element centres of a uniform
// mesh -- temperature and log10 viscosity -- to three: u_x, u_z and p at the
// element centres, in units of Ra (Stokes flow is linear in the buoyancy Ra T,
// so the solution at any Ra is Ra times the solution at Ra = 1) and scaled by a
// dataset constant.  Architecture: 4 levels, two 3x3 convolutions with ReLU per
// level (32, 64, 128, 256 channels), 2x2 average pooling down, nearest 2x
// upsampling up with the encoder activation concatenated, a 1x1 head.
// Training data are snapshots of the solver's own fields captured on the
// device; training runs on the device with the kernels of mcl_unet.hip (bf16
// MFMA products, FP32 accumulation and master weights, Adam).  The guess is
// accepted only if its momentum residual is smaller than that of the current
// (previous-step) guess.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "mcl.h"
#include "mcl_net.h"

// kernels of mcl_unet.hip
struct ConvShape {
    int B, H, W;
    int Cin, Cout;
    int cs_in, ci_off;
    int cs_out, co_off;
};
struct NetLayer {
    int off, nw, nb, Cin;
    uint16_t *Wf, *Wd;
};
struct NetLayers {
    NetLayer l[15];
};
__global__ void k_conv3_fwd(ConvShape s, const uint16_t *in, const uint16_t *Wf, const float *bias, uint16_t *out,
                            int relu);
__global__ void k_conv3_dgrad(ConvShape s, const uint16_t *dout, const uint16_t *act, const uint16_t *Wd,
                              uint16_t *din);
__global__ void k_conv3_wgrad(ConvShape s, const uint16_t *dout, const uint16_t *in, float *dW, int pix_per_split);
template <int MR, int NB, int WX, int WY, bool DG>
__global__ void k_conv3_tile(ConvShape s, const uint16_t *X, const uint16_t *act, const uint16_t *Wt, const float *bias,
                             uint16_t *Y, int relu);
__global__ void k_conv3_mm(ConvShape s, int dgrad, const uint16_t *X, const uint16_t *act, const uint16_t *Wt,
                           const float *bias, uint16_t *Y, int relu);
__global__ void k_conv3_wgrad_mm(ConvShape s, const uint16_t *dout, const uint16_t *in, float *dW, float *db,
                                 int tiles_per_split);
template <int NBLK, int TH>
__global__ void k_conv3_wgrad_tile(ConvShape s, const uint16_t *dout, const uint16_t *in, float *dW, float *db,
                                   int tiles_per_split);
__global__ void k_bias_grad(int M, int Cout, int cs, int coff, const uint16_t *dout, float *db);
__global__ void k_pool_fwd(int B, int H, int W, int C, const uint16_t *in, int cs_in, int ci_off, uint16_t *out,
                           int cs_out, int co_off);
__global__ void k_pool_bwd(int B, int H, int W, int C, const uint16_t *dout, int cs_out, int co_off,
                           const uint16_t *act, uint16_t *din, int cs_in, int ci_off);
__global__ void k_up_fwd(int B, int H, int W, int C, const uint16_t *in, int cs_in, int ci_off, uint16_t *out,
                         int cs_out, int co_off);
__global__ void k_up_bwd(int B, int H, int W, int C, const uint16_t *dout, int cs_out, int co_off, uint16_t *din,
                         int cs_in, int ci_off);
__global__ void k_head_fwd(int M, const uint16_t *x, int cs, const float *Wh, const float *bh, float *y);
__global__ void k_head_bwd(int M, const uint16_t *x, int cs, const float *Wh, const float *y, const float *tgt,
                           float scale, uint16_t *dx, float *dWh, float *dbh, float *loss);
template <bool STEP>
__global__ void k_update_weights(NetLayers ls, float *w, const float *g, float *m1, float *m2, float lr, float b1,
                                 float b2, float eps, float c1, float c2);
__global__ void k_f32_to_bf16(size_t n, const float *x, uint16_t *y);
__global__ void k_bf16_to_f32(size_t n, const uint16_t *x, float *y);

namespace {

struct Act {           // one NHWC bf16 activation buffer and its gradient
    int H = 0, W = 0, C = 0;
    uint16_t *y = nullptr, *g = nullptr;
};

struct Conv {          // one 3x3 convolution layer
    int Cin = 0, Cout = 0;
    size_t nw = 0;     // Cout*9*Cin
    float *w = nullptr, *b = nullptr, *dw = nullptr, *db = nullptr;   // in mcl_net's params and grads
    uint16_t *Wf = nullptr, *Wd = nullptr;
};

}  // namespace

struct mcl_net {
    int H = 0, W = 0, B = 0;
    hipStream_t stream = nullptr;
    std::vector<void *> owned;
    std::string err;
    // activations (encoder, concat buffers, decoder)
    Act x0, e1a, cat1, p1, e2a, cat2, p2, e3a, cat3, p3, b1, b2, d3a, d3b, d2a, d2b, d1a, d1b;
    Conv enc1a, enc1b, enc2a, enc2b, enc3a, enc3b, bota, botb, dec3a, dec3b, dec2a, dec2b, dec1a, dec1b;
    // head (1x1, 32 -> 3, FP32)
    float *wh = nullptr, *bh = nullptr, *dwh = nullptr, *dbh = nullptr;
    // Parameters, gradients and Adam moments, each one buffer in the flat order
    // of mcl_net_get_params, so that clearing, reading and updating them is one
    // call for the network; the loss lies behind the gradients and is cleared
    // with them.
    size_t np = 0;
    float *params = nullptr, *grads = nullptr, *m1 = nullptr, *m2 = nullptr;
    NetLayers layers{};
    float *y = nullptr, *tgt = nullptr, *xin = nullptr, *loss = nullptr;
    long long adam_t = 0;
    float out_scale[3] = {1.0f, 1.0f, 1.0f};   // per output channel (RMS of the training targets)
    bool scaled = false;
    // dataset of snapshots on the device: inputs [N][H][W][2], targets [N][H][W][3]
    std::vector<float *> ds_x, ds_t;
};

#define NCHK(call)                                                                       \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess) {                                                          \
            n->err = std::string(#call) + ": " + hipGetErrorString(e_);                   \
            return MCL_E_DEVICE;                                                         \
        }                                                                                \
    } while (0)

template <typename T>
static int nalloc(mcl_net *n, T **p, size_t count)
{
    void *q = nullptr;
    NCHK(hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)));
    NCHK(hipMemset(q, 0, std::max<size_t>(count, 1) * sizeof(T)));
    n->owned.push_back(q);
    *p = (T *)q;
    return 0;
}

static int make_act(mcl_net *n, Act &a, int H, int W, int C)
{
    a.H = H;
    a.W = W;
    a.C = C;
    size_t cnt = (size_t)n->B * H * W * C;
    if (nalloc(n, &a.y, cnt) || nalloc(n, &a.g, cnt)) return MCL_E_DEVICE;
    return 0;
}

// Normal deviates of mean 0 (Marsaglia's polar method in float, the values of
// libstdc++'s std::normal_distribution<float>): generate_canonical computes two
// long double logarithms for every uniform, which took 76-134 ms of a
// network's creation (the same code, by its alignment); this takes 20.
struct Normal {
    float sd, saved = 0.f;
    bool have = false;
    explicit Normal(float s) : sd(s) {}
    static float unit(std::mt19937_64 &rng)
    {
        const float u = (float)rng() * 0x1p-64f;
        return u >= 1.0f ? 0x1.fffffep-1f : u;
    }
    float operator()(std::mt19937_64 &rng)
    {
        if (have) {
            have = false;
            return saved * sd + 0.f;   // + the mean: no negative zeros
        }
        float x, y, r2;
        do {
            x = (float)(2.0f * unit(rng) - 1.0);
            y = (float)(2.0f * unit(rng) - 1.0);
            r2 = x * x + y * y;
        } while (r2 > 1.0f || r2 == 0.0f);
        const float m = std::sqrt(-2 * std::log(r2) / r2);
        saved = x * m;
        have = true;
        return (y * m) * sd + 0.f;
    }
};

// Convolution i, its parameters at offset `off` of the flat order (moved past them).
static int make_conv(mcl_net *n, int i, Conv &c, int Cin, int Cout, size_t &off)
{
    c.Cin = Cin;
    c.Cout = Cout;
    c.nw = (size_t)Cout * 9 * Cin;
    if (nalloc(n, &c.Wf, c.nw) || nalloc(n, &c.Wd, c.nw)) return MCL_E_DEVICE;
    c.w = n->params + off;
    c.b = c.w + c.nw;
    c.dw = n->grads + off;
    c.db = c.dw + c.nw;
    n->layers.l[i] = {(int)off, (int)c.nw, Cout, Cin, c.Wf, c.Wd};
    off += c.nw + Cout;
    return 0;
}

static unsigned gblocks(size_t n) { return (unsigned)std::min<size_t>((n + 255) / 256, 8192); }

// MCL_CONV_DIRECT=1 keeps the unstaged kernels everywhere (for comparisons).
static bool conv_direct()
{
    const char *e = getenv("MCL_CONV_DIRECT");
    return e && atoi(e);
}

// One 3x3 product of `dg` = false: the forward pass, true: the data gradient.
// Tiles of whole 16-pixel runs (k_conv3_tile) need a width that is a multiple
// of 16 and 16-byte aligned pixels of the summed buffer; the tile is the
// largest that leaves a workgroup for each of the 256 CUs (the large ones stage
// less and read less LDS per MFMA; a layer with few pixels is bound by the
// latency of its chunks, which only more workgroups hide).  A forward pass of 15
// images of 32 x 256 takes 362 us with that line at one workgroup a CU, 371 at
// two, 384 at four; the 14 products of one 256 x 256 image take 119 us (280 us as
// 64 pixels x 64 channels a workgroup throughout).  Narrower layers whose 64
// consecutive pixels form a rectangle of one image take k_conv3_mm, the rest the
// unstaged kernels.
template <bool DG>
static void conv_product(mcl_net *n, const ConvShape &s, const uint16_t *X, const uint16_t *act, const uint16_t *Wt,
                         const float *bias, uint16_t *Y, int relu)
{
    const int Kc = DG ? s.Cout : s.Cin, N = DG ? s.Cin : s.Cout;
    const int xst = DG ? s.cs_out : s.cs_in, xof = DG ? s.co_off : s.ci_off;
    const int M = s.B * s.H * s.W;
    const bool staged = !conv_direct() && Kc % 8 == 0 && xst % 8 == 0 && xof % 8 == 0;
    if (staged && s.W % 16 == 0 && s.H % 4 == 0 && N % 32 == 0) {
        auto fits = [&](int px, int tw, int th, int nt, int least) {
            return s.W % tw == 0 && s.H % th == 0 && N % nt == 0 && (long long)(M / px) * (N / nt) >= least;
        };
#define CONV_TILE(MR, NB, WX, WY)                                                                                   \
    hipLaunchKernelGGL((k_conv3_tile<MR, NB, WX, WY, DG>), dim3((M / (16 * WX * MR * WY)) * (N / (16 * NB))),         \
                       dim3(64 * WX * WY), 0, n->stream, s, X, act, Wt, bias, Y, relu)
        if (fits(256, 32, 8, 64, 256)) CONV_TILE(4, 4, 2, 2);
        else if (fits(256, 32, 8, 32, 256)) CONV_TILE(4, 2, 2, 2);
        else if (fits(128, 32, 4, 32, 256)) CONV_TILE(2, 2, 2, 2);
        else if (fits(64, 32, 2, 32, 1)) CONV_TILE(1, 2, 2, 2);
        else CONV_TILE(1, 2, 1, 4);
#undef CONV_TILE
        return;
    }
    const int TW = s.W < 64 ? s.W : 64;
    if (staged && s.W % TW == 0 && 64 % TW == 0 && s.H % (64 / TW) == 0) {
        hipLaunchKernelGGL(k_conv3_mm, dim3(M / 64, (N + 63) / 64), dim3(256), 0, n->stream, s, DG ? 1 : 0, X, act, Wt,
                           bias, Y, relu);
        return;
    }
    if constexpr (DG)
        hipLaunchKernelGGL(k_conv3_dgrad, dim3((M + 63) / 64, (N + 63) / 64), dim3(256), 0, n->stream, s, X, act, Wt, Y);
    else
        hipLaunchKernelGGL(k_conv3_fwd, dim3((M + 63) / 64, (N + 63) / 64), dim3(256), 0, n->stream, s, X, Wt, bias, Y,
                           relu);
}

static void conv_fwd(mcl_net *n, Conv &c, const Act &in, int ci_off, Act &out, int co_off, bool relu)
{
    ConvShape s{n->B, in.H, in.W, c.Cin, c.Cout, in.C, ci_off, out.C, co_off};
    conv_product<false>(n, s, in.y, nullptr, c.Wf, c.b, out.y, relu ? 1 : 0);
}

// Backward of a ReLU convolution whose output gradient out.g is already zero
// where the ReLU was: weight and bias gradients, and the data gradient into
// in.g (skipped when din is false), zeroed where the input is not positive if
// the input is a ReLU's output (in_relu).
static void conv_bwd(mcl_net *n, Conv &c, const Act &in, int ci_off, Act &out, int co_off, bool din, bool in_relu)
{
    ConvShape s{n->B, in.H, in.W, c.Cin, c.Cout, in.C, ci_off, out.C, co_off};
    const int M = n->B * in.H * in.W;
    const uint16_t *g = out.g, *x = in.y;
    const int TW = in.W < 64 ? in.W : 64;
    const bool staged = !conv_direct() && c.Cin % 8 == 0 && in.C % 8 == 0 && ci_off % 8 == 0 && out.C % 8 == 0 &&
                        co_off % 8 == 0;
    // (32 output channels: the full-resolution layers, whose height 8 divides)
    if (staged && in.W % 32 == 0 && c.Cout % 32 == 0 && in.H % (c.Cout % 64 == 0 ? 4 : 8) == 0) {
        // tiles of 32 x 8 pixels (32 x 4 on lower images), about 512
        // workgroups, each summing at least two tiles where there are that many
        const int th = in.H % 8 == 0 ? 8 : 4, tiles = M / (32 * th), nblk = c.Cout % 64 == 0 ? 64 : 32;
        const int nbn = c.Cout / nblk, nbc = (c.Cin + 31) / 32;
        int splits = std::max(1, std::min((tiles + 1) / 2, 512 / (nbn * nbc)));
        const int tps = (tiles + splits - 1) / splits;
        splits = (tiles + tps - 1) / tps;
        const dim3 grid(nbn, nbc, splits);
#define WGRAD_TILE(NBLK, TH) \
    hipLaunchKernelGGL((k_conv3_wgrad_tile<NBLK, TH>), grid, dim3(256), 0, n->stream, s, g, x, c.dw, c.db, tps)
        if (nblk == 64 && th == 8) WGRAD_TILE(64, 8);
        else if (nblk == 64) WGRAD_TILE(64, 4);
        else WGRAD_TILE(32, 8);
#undef WGRAD_TILE
    } else if (staged && TW % 8 == 0 && in.W % TW == 0 && 64 % TW == 0 && in.H % (64 / TW) == 0) {
        // narrow and low levels: workgroups of 64 x 32 x 9 taps, about 512 in
        // all, each summing at least 8 runs of 64 pixels (a step of 128 x 128,
        // batch 32: 2.2 ms, 3.1 with the unstaged kernel on its two 16-wide layers)
        const int tiles = M / 64, nbn = (c.Cout + 63) / 64, nbc = (c.Cin + 31) / 32;
        int splits = std::max(1, std::min(tiles / 8, 512 / (nbn * nbc)));
        const int tps = (tiles + splits - 1) / splits;
        splits = (tiles + tps - 1) / tps;
        hipLaunchKernelGGL(k_conv3_wgrad_mm, dim3(nbn, nbc, splits), dim3(256), 0, n->stream, s, g, x, c.dw, c.db, tps);
    } else {
        int splits = std::max(1, std::min(256, M / 4096));
        int pps = ((M + splits - 1) / splits + 15) / 16 * 16;
        splits = (M + pps - 1) / pps;
        dim3 gw((c.Cout + 63) / 64, (9 * c.Cin + 63) / 64, splits);
        hipLaunchKernelGGL(k_conv3_wgrad, gw, dim3(256), 0, n->stream, s, g, x, c.dw, pps);
        hipLaunchKernelGGL(k_bias_grad, dim3(std::min(1024, (M + 63) / 64)), dim3(256), 0, n->stream, M, c.Cout,
                           out.C, co_off, g, c.db);
    }
    if (din) conv_product<true>(n, s, g, in_relu ? x : nullptr, c.Wd, nullptr, in.g, 0);
}

static Conv *convs(mcl_net *n, int i)
{
    Conv *all[] = {&n->enc1a, &n->enc1b, &n->enc2a, &n->enc2b, &n->enc3a, &n->enc3b, &n->bota,
                   &n->botb,  &n->dec3a, &n->dec3b, &n->dec2a, &n->dec2b, &n->dec1a, &n->dec1b};
    return i < 14 ? all[i] : nullptr;
}

// One row of workgroups for each layer: 256 of 256 threads cover the largest
// (589 824 weights and 256 biases) in ten rounds, the last for the biases.
static const dim3 update_grid(256, 15);

static void weights_bf16(mcl_net *n)
{
    hipLaunchKernelGGL(k_update_weights<false>, update_grid, dim3(256), 0, n->stream, n->layers, n->params,
                       (const float *)nullptr, (float *)nullptr, (float *)nullptr, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
}

int mcl_net_create(int H, int W, int batch, unsigned long long seed, mcl_net **out)
{
    if (!out || H % 8 || W % 8 || H < 16 || W < 16 || batch < 1) return MCL_E_ARG;
    mcl_net *n = new mcl_net();
    n->H = H;
    n->W = W;
    n->B = batch;
    if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
        delete n;
        return MCL_E_DEVICE;
    }
    std::mt19937_64 rng(seed);
    int rc = 0;
    rc |= make_act(n, n->x0, H, W, 16);
    rc |= make_act(n, n->e1a, H, W, 32);
    rc |= make_act(n, n->cat1, H, W, 96);
    rc |= make_act(n, n->p1, H / 2, W / 2, 32);
    rc |= make_act(n, n->e2a, H / 2, W / 2, 64);
    rc |= make_act(n, n->cat2, H / 2, W / 2, 192);
    rc |= make_act(n, n->p2, H / 4, W / 4, 64);
    rc |= make_act(n, n->e3a, H / 4, W / 4, 128);
    rc |= make_act(n, n->cat3, H / 4, W / 4, 384);
    rc |= make_act(n, n->p3, H / 8, W / 8, 128);
    rc |= make_act(n, n->b1, H / 8, W / 8, 256);
    rc |= make_act(n, n->b2, H / 8, W / 8, 256);
    rc |= make_act(n, n->d3a, H / 4, W / 4, 128);
    rc |= make_act(n, n->d3b, H / 4, W / 4, 128);
    rc |= make_act(n, n->d2a, H / 2, W / 2, 64);
    rc |= make_act(n, n->d2b, H / 2, W / 2, 64);
    rc |= make_act(n, n->d1a, H, W, 32);
    rc |= make_act(n, n->d1b, H, W, 32);
    static const int chan[14][2] = {{16, 32}, {32, 32}, {32, 64}, {64, 64}, {64, 128}, {128, 128}, {128, 256},
                                    {256, 256}, {384, 128}, {128, 128}, {192, 64}, {64, 64}, {96, 32}, {32, 32}};
    for (auto &c : chan) n->np += (size_t)c[1] * (9 * c[0] + 1);
    n->np += 3 * 32 + 3;
    rc |= nalloc(n, &n->params, n->np) | nalloc(n, &n->grads, n->np + 1) | nalloc(n, &n->m1, n->np) |
          nalloc(n, &n->m2, n->np);
    size_t off = 0;
    for (int i = 0; i < 14 && !rc; i++) rc |= make_conv(n, i, *convs(n, i), chan[i][0], chan[i][1], off);
    size_t M = (size_t)batch * H * W;
    rc |= nalloc(n, &n->y, 3 * M) | nalloc(n, &n->tgt, 3 * M) | nalloc(n, &n->xin, 2 * M);
    if (rc) {
        mcl_net_destroy(n);
        return MCL_E_DEVICE;
    }
    n->wh = n->params + off;
    n->bh = n->wh + 3 * 32;
    n->dwh = n->grads + off;
    n->dbh = n->dwh + 3 * 32;
    n->loss = n->grads + n->np;
    n->layers.l[14] = {(int)off, 0, 3 * 32 + 3, 0, nullptr, nullptr};
    // He initialisation for the ReLU layers, zero biases
    std::vector<float> p(n->np, 0.f);
    off = 0;
    for (int i = 0; i < 14; i++) {
        const Conv &c = *convs(n, i);
        Normal nd(std::sqrt(2.0f / (9.0f * (float)c.Cin)));
        for (size_t k = 0; k < c.nw; k++) p[off + k] = nd(rng);
        off += c.nw + c.Cout;
    }
    Normal nd(std::sqrt(1.0f / 32.0f));
    for (int k = 0; k < 96; k++) p[off + k] = nd(rng);
    if (hipMemcpy(n->params, p.data(), n->np * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
        mcl_net_destroy(n);
        return MCL_E_DEVICE;
    }
    weights_bf16(n);
    *out = n;
    return 0;
}

void mcl_net_destroy(mcl_net *n)
{
    if (!n) return;
    if (n->stream) (void)hipStreamSynchronize(n->stream);
    for (void *p : n->owned) (void)hipFree(p);
    for (float *p : n->ds_x) (void)hipFree(p);
    for (float *p : n->ds_t) (void)hipFree(p);
    if (n->stream) (void)hipStreamDestroy(n->stream);
    delete n;
}

const char *mcl_net_last_error(const mcl_net *n) { return n ? n->err.c_str() : "null network"; }

// x0 (bf16, 16 channels, 2 used) from FP32 [B][H][W][2] on the device
__global__ void k_pack_input(size_t M, const float *__restrict__ x, uint16_t *__restrict__ x0)
{
    for (size_t m = blockIdx.x * (size_t)blockDim.x + threadIdx.x; m < M; m += (size_t)gridDim.x * blockDim.x) {
        for (int c = 0; c < 16; c++) {
            float v = c < 2 ? x[m * 2 + c] : 0.f;
            unsigned u = __float_as_uint(v);
            u += 0x7fffu + ((u >> 16) & 1u);
            x0[m * 16 + c] = (uint16_t)(u >> 16);
        }
    }
}

static void forward(mcl_net *n)
{
    const int B = n->B;
    size_t M = (size_t)B * n->H * n->W;
    hipLaunchKernelGGL(k_pack_input, dim3(gblocks(M)), dim3(256), 0, n->stream, M, (const float *)n->xin, n->x0.y);
    conv_fwd(n, n->enc1a, n->x0, 0, n->e1a, 0, true);
    conv_fwd(n, n->enc1b, n->e1a, 0, n->cat1, 64, true);
    hipLaunchKernelGGL(k_pool_fwd, dim3(gblocks(M / 4 * 4)), dim3(256), 0, n->stream, B, n->H, n->W, 32,
                       (const uint16_t *)n->cat1.y, 96, 64, n->p1.y, 32, 0);
    conv_fwd(n, n->enc2a, n->p1, 0, n->e2a, 0, true);
    conv_fwd(n, n->enc2b, n->e2a, 0, n->cat2, 128, true);
    hipLaunchKernelGGL(k_pool_fwd, dim3(gblocks(M / 16 * 8)), dim3(256), 0, n->stream, B, n->H / 2, n->W / 2, 64,
                       (const uint16_t *)n->cat2.y, 192, 128, n->p2.y, 64, 0);
    conv_fwd(n, n->enc3a, n->p2, 0, n->e3a, 0, true);
    conv_fwd(n, n->enc3b, n->e3a, 0, n->cat3, 256, true);
    hipLaunchKernelGGL(k_pool_fwd, dim3(gblocks(M / 64 * 16)), dim3(256), 0, n->stream, B, n->H / 4, n->W / 4, 128,
                       (const uint16_t *)n->cat3.y, 384, 256, n->p3.y, 128, 0);
    conv_fwd(n, n->bota, n->p3, 0, n->b1, 0, true);
    conv_fwd(n, n->botb, n->b1, 0, n->b2, 0, true);
    hipLaunchKernelGGL(k_up_fwd, dim3(gblocks(M / 16 * 32)), dim3(256), 0, n->stream, B, n->H / 8, n->W / 8, 256,
                       (const uint16_t *)n->b2.y, 256, 0, n->cat3.y, 384, 0);
    conv_fwd(n, n->dec3a, n->cat3, 0, n->d3a, 0, true);
    conv_fwd(n, n->dec3b, n->d3a, 0, n->d3b, 0, true);
    hipLaunchKernelGGL(k_up_fwd, dim3(gblocks(M / 4 * 16)), dim3(256), 0, n->stream, B, n->H / 4, n->W / 4, 128,
                       (const uint16_t *)n->d3b.y, 128, 0, n->cat2.y, 192, 0);
    conv_fwd(n, n->dec2a, n->cat2, 0, n->d2a, 0, true);
    conv_fwd(n, n->dec2b, n->d2a, 0, n->d2b, 0, true);
    hipLaunchKernelGGL(k_up_fwd, dim3(gblocks(M * 8)), dim3(256), 0, n->stream, B, n->H / 2, n->W / 2, 64,
                       (const uint16_t *)n->d2b.y, 64, 0, n->cat1.y, 96, 0);
    conv_fwd(n, n->dec1a, n->cat1, 0, n->d1a, 0, true);
    conv_fwd(n, n->dec1b, n->d1a, 0, n->d1b, 0, true);
    hipLaunchKernelGGL(k_head_fwd, dim3(gblocks(M)), dim3(256), 0, n->stream, (int)M, (const uint16_t *)n->d1b.y,
                       32, (const float *)n->wh, (const float *)n->bh, n->y);
}

static void zero_grads(mcl_net *n)
{
    (void)hipMemsetAsync(n->grads, 0, (n->np + 1) * sizeof(float), n->stream);
}

static void backward(mcl_net *n)
{
    const int B = n->B;
    const int M = B * n->H * n->W;
    float scale = 2.0f / (3.0f * (float)M);
    hipLaunchKernelGGL(k_head_bwd, dim3(std::min(1024, (M + 255) / 256)), dim3(256), 0, n->stream, M,
                       (const uint16_t *)n->d1b.y, 32, (const float *)n->wh, (const float *)n->y,
                       (const float *)n->tgt, scale, n->d1b.g, n->dwh, n->dbh, n->loss);
    conv_bwd(n, n->dec1b, n->d1a, 0, n->d1b, 0, true, true);
    conv_bwd(n, n->dec1a, n->cat1, 0, n->d1a, 0, true, true);
    hipLaunchKernelGGL(k_up_bwd, dim3(gblocks((size_t)M / 4 * 8)), dim3(256), 0, n->stream, B, n->H / 2, n->W / 2, 64,
                       (const uint16_t *)n->cat1.g, 96, 0, n->d2b.g, 64, 0);
    conv_bwd(n, n->dec2b, n->d2a, 0, n->d2b, 0, true, true);
    conv_bwd(n, n->dec2a, n->cat2, 0, n->d2a, 0, true, true);
    hipLaunchKernelGGL(k_up_bwd, dim3(gblocks((size_t)M / 16 * 16)), dim3(256), 0, n->stream, B, n->H / 4, n->W / 4,
                       128, (const uint16_t *)n->cat2.g, 192, 0, n->d3b.g, 128, 0);
    conv_bwd(n, n->dec3b, n->d3a, 0, n->d3b, 0, true, true);
    conv_bwd(n, n->dec3a, n->cat3, 0, n->d3a, 0, true, true);
    hipLaunchKernelGGL(k_up_bwd, dim3(gblocks((size_t)M / 64 * 32)), dim3(256), 0, n->stream, B, n->H / 8, n->W / 8,
                       256, (const uint16_t *)n->cat3.g, 384, 0, n->b2.g, 256, 0);
    conv_bwd(n, n->botb, n->b1, 0, n->b2, 0, true, true);
    conv_bwd(n, n->bota, n->p3, 0, n->b1, 0, true, false);
    hipLaunchKernelGGL(k_pool_bwd, dim3(gblocks((size_t)M / 16 * 16)), dim3(256), 0, n->stream, B, n->H / 4, n->W / 4,
                       128, (const uint16_t *)n->p3.g, 128, 0, (const uint16_t *)n->cat3.y, n->cat3.g, 384, 256);
    conv_bwd(n, n->enc3b, n->e3a, 0, n->cat3, 256, true, true);
    conv_bwd(n, n->enc3a, n->p2, 0, n->e3a, 0, true, false);
    hipLaunchKernelGGL(k_pool_bwd, dim3(gblocks((size_t)M / 4 * 8)), dim3(256), 0, n->stream, B, n->H / 2, n->W / 2,
                       64, (const uint16_t *)n->p2.g, 64, 0, (const uint16_t *)n->cat2.y, n->cat2.g, 192, 128);
    conv_bwd(n, n->enc2b, n->e2a, 0, n->cat2, 128, true, true);
    conv_bwd(n, n->enc2a, n->p1, 0, n->e2a, 0, true, false);
    hipLaunchKernelGGL(k_pool_bwd, dim3(gblocks((size_t)M * 4)), dim3(256), 0, n->stream, B, n->H, n->W, 32,
                       (const uint16_t *)n->p1.g, 32, 0, (const uint16_t *)n->cat1.y, n->cat1.g, 96, 64);
    conv_bwd(n, n->enc1b, n->e1a, 0, n->cat1, 64, true, true);
    conv_bwd(n, n->enc1a, n->x0, 0, n->e1a, 0, false, false);
}

static void adam_step(mcl_net *n, float lr)
{
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    n->adam_t++;
    float c1 = 1.0f - std::pow(b1, (float)n->adam_t), c2 = 1.0f - std::pow(b2, (float)n->adam_t);
    hipLaunchKernelGGL(k_update_weights<true>, update_grid, dim3(256), 0, n->stream, n->layers, n->params,
                       (const float *)n->grads, n->m1, n->m2, lr, b1, b2, eps, c1, c2);
}

int mcl_net_forward(mcl_net *n, const float *x_host, float *y_host)
{
    if (!n || !x_host || !y_host) return MCL_E_ARG;
    size_t M = (size_t)n->B * n->H * n->W;
    NCHK(hipMemcpyAsync(n->xin, x_host, 2 * M * sizeof(float), hipMemcpyHostToDevice, n->stream));
    forward(n);
    NCHK(hipGetLastError());
    NCHK(hipMemcpyAsync(y_host, n->y, 3 * M * sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NCHK(hipStreamSynchronize(n->stream));
    return 0;
}

int mcl_net_train_step(mcl_net *n, const float *x_host, const float *t_host, float lr, float *loss)
{
    if (!n || !x_host || !t_host) return MCL_E_ARG;
    size_t M = (size_t)n->B * n->H * n->W;
    NCHK(hipMemcpyAsync(n->xin, x_host, 2 * M * sizeof(float), hipMemcpyHostToDevice, n->stream));
    NCHK(hipMemcpyAsync(n->tgt, t_host, 3 * M * sizeof(float), hipMemcpyHostToDevice, n->stream));
    zero_grads(n);
    forward(n);
    backward(n);
    if (lr > 0.f) adam_step(n, lr);
    NCHK(hipGetLastError());
    float l = 0.f;
    NCHK(hipMemcpyAsync(&l, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
    NCHK(hipStreamSynchronize(n->stream));
    if (loss) *loss = l / (3.0f * (float)M);
    return 0;
}

// Parameters in a flat FP32 vector: for each conv in order w[Cout][3][3][Cin]
// then b[Cout]; then the head w[3][32], b[3].
long long mcl_net_num_params(const mcl_net *n) { return (long long)n->np; }

static int copy_params(mcl_net *n, float *host, bool get, bool grads)
{
    if (get) {
        NCHK(hipMemcpy(host, grads ? n->grads : n->params, n->np * sizeof(float), hipMemcpyDeviceToHost));
        return 0;
    }
    NCHK(hipMemcpy(n->params, host, n->np * sizeof(float), hipMemcpyHostToDevice));
    weights_bf16(n);
    NCHK(hipStreamSynchronize(n->stream));
    return 0;
}

int mcl_net_get_params(mcl_net *n, float *host) { return n && host ? copy_params(n, host, true, false) : MCL_E_ARG; }
int mcl_net_set_params(mcl_net *n, const float *host)
{
    return n && host ? copy_params(n, const_cast<float *>(host), false, false) : MCL_E_ARG;
}
int mcl_net_get_grads(mcl_net *n, float *host) { return n && host ? copy_params(n, host, true, true) : MCL_E_ARG; }

// ------------------------------------------------- internal interface, data
float *mcl_net_in(mcl_net *n) { return n->xin; }
float *mcl_net_out(mcl_net *n) { return n->y; }
float *mcl_net_tgt(mcl_net *n) { return n->tgt; }
hipStream_t mcl_net_stream(mcl_net *n) { return n->stream; }
float mcl_net_out_scale(const mcl_net *n, int ch) { return (ch >= 0 && ch < 3) ? n->out_scale[ch] : 0.f; }

int mcl_net_dims(const mcl_net *n, int *H, int *W, int *B)
{
    if (!n) return MCL_E_ARG;
    *H = n->H;
    *W = n->W;
    *B = n->B;
    return 0;
}

int mcl_net_forward_device(mcl_net *n)
{
    forward(n);
    NCHK(hipGetLastError());
    return 0;
}

// sum of squares of each of the 3 channels of npix pixels [npix][3] (order of
// accumulation irrelevant: it only sets the output scales)
__global__ void k_sumsq3(size_t npix, const float *__restrict__ x, double *__restrict__ out)
{
    double s[3] = {0.0, 0.0, 0.0};
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < npix; i += (size_t)gridDim.x * blockDim.x)
        for (int c = 0; c < 3; c++) s[c] += (double)x[3 * i + c] * x[3 * i + c];
    for (int c = 0; c < 3; c++) {
        for (int o = 32; o > 0; o >>= 1) s[c] += __shfl_xor(s[c], o, 64);
        if ((threadIdx.x & 63) == 0) atomicAdd(out + c, s[c]);
    }
}

__global__ void k_scale3(size_t npix, float a0, float a1, float a2, float *__restrict__ x)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < npix; i += (size_t)gridDim.x * blockDim.x) {
        x[3 * i] *= a0;
        x[3 * i + 1] *= a1;
        x[3 * i + 2] *= a2;
    }
}

// Mirror one sample in x (column ix <-> W-1-ix) in place: inputs [H][W][2],
// targets [H][W][3] with the horizontal velocity negated (the box, its
// boundary conditions and gravity are symmetric under x -> L - x).
__global__ void k_flip_x(int H, int W, float *__restrict__ x, float *__restrict__ t)
{
    const int half = W / 2;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < H * half; q += gridDim.x * blockDim.x) {
        const int iz = q / half, ix = q - iz * half;
        const int a = iz * W + ix, b = iz * W + (W - 1 - ix);
        for (int c = 0; c < 2; c++) {
            float u = x[2 * a + c], v = x[2 * b + c];
            x[2 * a + c] = v;
            x[2 * b + c] = u;
        }
        for (int c = 0; c < 3; c++) {
            float u = t[3 * a + c], v = t[3 * b + c];
            float sg = c == 0 ? -1.f : 1.f;
            t[3 * a + c] = sg * v;
            t[3 * b + c] = sg * u;
        }
    }
}

int mcl_net_add_snapshot(mcl_net *n, const float *x_dev, const float *t_dev)
{
    size_t P = (size_t)n->H * n->W;
    float *x = nullptr, *t = nullptr;
    NCHK(hipMalloc(&x, 2 * P * sizeof(float)));
    NCHK(hipMalloc(&t, 3 * P * sizeof(float)));
    NCHK(hipMemcpyAsync(x, x_dev, 2 * P * sizeof(float), hipMemcpyDeviceToDevice, n->stream));
    NCHK(hipMemcpyAsync(t, t_dev, 3 * P * sizeof(float), hipMemcpyDeviceToDevice, n->stream));
    NCHK(hipStreamSynchronize(n->stream));
    n->ds_x.push_back(x);
    n->ds_t.push_back(t);
    return 0;
}

long long mcl_net_dataset_size(const mcl_net *n) { return n ? (long long)n->ds_x.size() : 0; }

int mcl_net_train(mcl_net *n, int epochs, float lr, unsigned long long seed, float *losses)
{
    if (!n || epochs < 0) return MCL_E_ARG;
    const size_t N = n->ds_x.size();
    if (N < (size_t)n->B) {
        n->err = "dataset smaller than one batch";
        return MCL_E_STATE;
    }
    const size_t P = (size_t)n->H * n->W;
    // output scales: RMS of each target channel over the dataset (set once)
    if (!n->scaled) {
        double *acc = nullptr;
        NCHK(hipMalloc(&acc, 3 * sizeof(double)));
        NCHK(hipMemsetAsync(acc, 0, 3 * sizeof(double), n->stream));
        for (size_t i = 0; i < N; i++)
            hipLaunchKernelGGL(k_sumsq3, dim3(gblocks(P)), dim3(256), 0, n->stream, P, (const float *)n->ds_t[i], acc);
        double sq[3] = {0.0, 0.0, 0.0};
        NCHK(hipMemcpyAsync(sq, acc, 3 * sizeof(double), hipMemcpyDeviceToHost, n->stream));
        NCHK(hipStreamSynchronize(n->stream));
        (void)hipFree(acc);
        for (int c = 0; c < 3; c++) {
            double rms = std::sqrt(sq[c] / ((double)P * N));
            n->out_scale[c] = rms > 0 ? (float)rms : 1.0f;
        }
        n->scaled = true;
    }
    std::mt19937_64 rng(seed);
    std::vector<size_t> order(N);
    for (size_t i = 0; i < N; i++) order[i] = i;
    const size_t nb = N / n->B;
    for (int ep = 0; ep < epochs; ep++) {
        std::shuffle(order.begin(), order.end(), rng);
        double sum = 0.0;
        for (size_t b = 0; b < nb; b++) {
            for (int k = 0; k < n->B; k++) {
                size_t s = order[b * n->B + k];
                NCHK(hipMemcpyAsync(n->xin + k * 2 * P, n->ds_x[s], 2 * P * sizeof(float), hipMemcpyDeviceToDevice,
                                    n->stream));
                NCHK(hipMemcpyAsync(n->tgt + k * 3 * P, n->ds_t[s], 3 * P * sizeof(float), hipMemcpyDeviceToDevice,
                                    n->stream));
                if (rng() & 1)
                    hipLaunchKernelGGL(k_flip_x, dim3(gblocks(P / 2)), dim3(256), 0, n->stream, n->H, n->W,
                                       n->xin + k * 2 * P, n->tgt + k * 3 * P);
            }
            hipLaunchKernelGGL(k_scale3, dim3(gblocks(P * n->B)), dim3(256), 0, n->stream, P * n->B,
                               1.0f / n->out_scale[0], 1.0f / n->out_scale[1], 1.0f / n->out_scale[2], n->tgt);
            zero_grads(n);
            forward(n);
            backward(n);
            adam_step(n, lr);
            NCHK(hipGetLastError());
            float l = 0.f;
            NCHK(hipMemcpyAsync(&l, n->loss, sizeof(float), hipMemcpyDeviceToHost, n->stream));
            NCHK(hipStreamSynchronize(n->stream));
            sum += l / (3.0 * P * n->B);
        }
        if (losses) losses[ep] = (float)(sum / nb);
    }
    return 0;
}

double mcl_net_get_scale(const mcl_net *n, int channel)
{
    return (n && channel >= 0 && channel < 3) ? n->out_scale[channel] : 0.0;
}

int mcl_net_set_scale(mcl_net *n, int channel, double scale)
{
    if (!n || channel < 0 || channel > 2 || !(scale > 0)) return MCL_E_ARG;
    n->out_scale[channel] = (float)scale;
    n->scaled = true;
    return 0;
}
