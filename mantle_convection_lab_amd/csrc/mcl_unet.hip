// Learned initial guess: the U-Net's forward, backward and Adam kernels (gfx950).
//
// Activations are NHWC bf16 (stored as 16-bit words), weights are FP32 master
// copies plus bf16 copies in the two layouts the products need:
//   Wf[co][tap][ci]   forward      out[m,co]  = sum_{tap,ci} in[m+off(tap),ci] Wf[co][tap][ci]
//   Wd[ci][tap][co]   data grad    din[m,ci]  = sum_{tap,co} g[m-off(tap),co] Wd[ci][tap][co]
// and the weight gradient dW[co][tap][ci] = sum_m g[m,co] in[m+off(tap),ci].
// All three are implicit GEMMs on bf16 MFMAs with FP32 accumulation.  A
// gradient buffer holds the gradient behind its layer's ReLU: whoever writes
// it zeroes it where the activation is not positive, so no reader needs the
// activation.
// The unstaged kernels (v_mfma_f32_16x16x16_bf16): a workgroup (4 waves)
// computes a 64 x 64 output tile; each wave a 32 x 32 block of four 16 x 16
// MFMA tiles.  Operand lane layout of the instruction (K = 16): A[i][k] in lane
// i + 16*(k/4), element k%4; B[k][j] in lane j + 16*(k/4), element k%4; D[i][j]
// in lane j + 16*(i/4), element i%4.
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned u4 __attribute__((ext_vector_type(4)));   // 16 bytes being staged

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((unsigned)h) << 16); }

// round to nearest even
__device__ __forceinline__ uint16_t f2bf(float f)
{
    unsigned u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

struct ConvShape {
    int B, H, W;          // batch and spatial size (same for input and output: 3x3, stride 1, pad 1)
    int Cin, Cout;        // channels of this convolution
    int cs_in, ci_off;    // channel stride / offset of the input buffer
    int cs_out, co_off;   // channel stride / offset of the output buffer
};

struct NetLayer {
    int off, nw, nb;      // first parameter in the flat order, 3x3 weights, parameters after them (biases, the head)
    int Cin;
    uint16_t *Wf, *Wd;    // bf16 weights of a 3x3 layer
};
struct NetLayers {
    NetLayer l[15];       // 14 convolutions, the head
};

// Load 4 consecutive bf16 channels (8-byte aligned) or zeros.
__device__ __forceinline__ s4 load4(const uint16_t *p, bool valid)
{
    if (!valid) return s4{0, 0, 0, 0};
    uint2 v = *(const uint2 *)p;
    s4 r;
    r[0] = (short)(v.x & 0xffff);
    r[1] = (short)(v.x >> 16);
    r[2] = (short)(v.y & 0xffff);
    r[3] = (short)(v.y >> 16);
    return r;
}

// ------------------------------------------------------------------ forward
// out[m, co] = relu?(bias[co] + sum in[m + off, ci] Wf[co][tap][ci]); requires
// Cin % 16 == 0 and Cout % 32 == 0, channel offsets/strides multiples of 4.
__global__ void __launch_bounds__(256) k_conv3_fwd(ConvShape s, const uint16_t *__restrict__ in,
                                                   const uint16_t *__restrict__ Wf, const float *__restrict__ bias,
                                                   uint16_t *__restrict__ out, int relu)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int M = s.B * s.H * s.W;
    const int m0 = blockIdx.x * 64 + (wave >> 1) * 32;
    const int n0 = blockIdx.y * 64 + (wave & 1) * 32;
    if (n0 >= s.Cout) return;  // whole wave idle (Cout = 32)
    f4 acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = f4{0, 0, 0, 0};
    // this lane's A rows (pixels) for the two 16-row tiles
    int ph[2], pw[2], pn[2];
    bool pv[2];
    for (int a = 0; a < 2; a++) {
        int m = m0 + a * 16 + (lane & 15);
        pv[a] = m < M;
        int mm = pv[a] ? m : 0;
        pn[a] = mm / (s.H * s.W);
        int r = mm - pn[a] * s.H * s.W;
        ph[a] = r / s.W;
        pw[a] = r - ph[a] * s.W;
    }
    const int kq = (lane >> 4) * 4;  // this lane's 4 k values within a 16-chunk
    for (int tap = 0; tap < 9; tap++) {
        const int dh = tap / 3 - 1, dw = tap % 3 - 1;
        const uint16_t *ap[2];
        bool av[2];
        for (int a = 0; a < 2; a++) {
            int h = ph[a] + dh, w = pw[a] + dw;
            av[a] = pv[a] && h >= 0 && h < s.H && w >= 0 && w < s.W;
            ap[a] = in + ((size_t)((pn[a] * s.H + (av[a] ? h : 0)) * s.W + (av[a] ? w : 0))) * s.cs_in + s.ci_off;
        }
        for (int c0 = 0; c0 < s.Cin; c0 += 16) {
            s4 A[2], Bv[2];
            for (int a = 0; a < 2; a++) A[a] = load4(ap[a] + c0 + kq, av[a]);
            for (int b = 0; b < 2; b++) {
                int co = n0 + b * 16 + (lane & 15);
                Bv[b] = load4(Wf + ((size_t)co * 9 + tap) * s.Cin + c0 + kq, co < s.Cout);
            }
            for (int a = 0; a < 2; a++)
                for (int b = 0; b < 2; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A[a], Bv[b], acc[a][b], 0, 0, 0);
        }
    }
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) {
            int co = n0 + b * 16 + (lane & 15);
            if (co >= s.Cout) continue;
            float bi = bias ? bias[co] : 0.f;
            for (int e = 0; e < 4; e++) {
                int m = m0 + a * 16 + (lane >> 4) * 4 + e;
                if (m >= M) continue;
                float v = acc[a][b][e] + bi;
                if (relu) v = fmaxf(v, 0.f);
                out[(size_t)m * s.cs_out + s.co_off + co] = f2bf(v);
            }
        }
}

// ------------------------------------------- LDS-staged forward / data grad
// Implicit-GEMM 3x3 convolution on v_mfma_f32_16x16x32_bf16 (gfx950) with the
// operands staged in LDS:
//   forward   Y[m, n] = relu?(bias[n] + sum_{tap,c} X[m + off(tap), c] Wt[n][tap][c])
//     with X = in, Wt = Wf, Y = out;
//   data grad Y[m, n] = sum_{tap,c} X[m - off(tap), c] Wt[n][tap][c]
//     with X = dout (already zero where the layer's ReLU was), Wt = Wd, Y =
//     din, zeroed where the input activation act is not positive (act != NULL:
//     the input is itself a ReLU's output, or a copy of one).
// A workgroup of WX x WY waves computes a rectangle of 16 WX x MR WY pixels of
// one image and 16 NB output channels, each wave 16 x MR pixels and all the
// channels.  For every 32-channel chunk of the summed channels it stages the
// rectangle with one pixel around and the chunk's weights for all nine taps;
// the next chunk's loads are in flight while the nine taps run.  Per chunk a
// wave reads its (MR + 2) x 3 shifted pixel rows once and uses them for every
// tap, so MR = 4, NB = 4 does 144 MFMAs for 54 LDS reads (the LDS pipe and the
// matrix pipe then take the same time); a 64-pixel, 64-channel workgroup of 32
// x 32 waves needs 36 reads for 36 MFMAs and stages the weights four times as
// often.  Measured at 256 x 256, batch 32, mean over the forward and data
// gradient products: 284 -> 104 us where the output has a multiple of 64
// channels (MR = 4, NB = 4), 313 -> 141 us for 32 and 96 (NB = 2), which are
// within 2x of their memory traffic.
// Every output is the same chain of MFMAs, chunk by chunk and tap by tap,
// whatever the tile, so the variants agree bit for bit.
// LDS rows are 64 bytes (32 channels of a pixel or of a weight row), the
// 16-byte unit q of row r stored at q ^ (r / 4 mod 4): 16 consecutive rows'
// equal units then lie in different banks.
// Operand layout of the instruction (K = 32): A[i][k] in lane i + 16 (k / 8),
// element k % 8; B[k][j] in lane j + 16 (k / 8), element k % 8; D[i][j] in
// lane j + 16 (i / 4), element i % 4.  A = weights (i = channel), B = pixels
// (j): a lane then holds four consecutive channels of its pixel, one 8-byte
// store.
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));

constexpr int CV_KC = 32;            // summed channels per stage

// round two floats to bf16, packed
__device__ __forceinline__ unsigned pack_bf(float a, float b) { return f2bf(a) | ((unsigned)f2bf(b) << 16); }

// a bf16 pair of g, 0 where y is not positive (a ReLU's gradient)
__device__ __forceinline__ unsigned mask_bf16x2(unsigned g, unsigned y)
{
    return (bf2f((uint16_t)(y & 0xffffu)) <= 0.f ? 0u : g & 0xffffu) |
           (bf2f((uint16_t)(y >> 16)) <= 0.f ? 0u : g & 0xffff0000u);
}

// Workgroup -> (tile, group of output channels).  Workgroups are dealt to the
// eight XCDs in turn, so the groups of one tile, which read the same pixels,
// are eight workgroups apart: they share the XCD's L2.
__device__ __forceinline__ void tile_group(int tiles, int groups, int &tile, int &group)
{
    const int id = blockIdx.x;
    if (tiles % 8 == 0) {
        group = (id >> 3) % groups;
        tile = (id / (8 * groups)) * 8 + (id & 7);
    } else {
        group = id % groups;
        tile = id / groups;
    }
}

template <int MR, int NB, int WX, int WY, bool DG>
__global__ void __launch_bounds__(64 * WX * WY)
    k_conv3_tile(ConvShape s, const uint16_t *__restrict__ X, const uint16_t *__restrict__ act,
                 const uint16_t *__restrict__ Wt, const float *__restrict__ bias, uint16_t *__restrict__ Y, int relu)
{
    constexpr int NTHR = 64 * WX * WY, TW = 16 * WX, TH = MR * WY, PW = TW + 2, NP = PW * (TH + 2), NT = 16 * NB;
    constexpr int XU = (NP * 4 + NTHR - 1) / NTHR, WU = (9 * NT * 4 + NTHR - 1) / NTHR;
    __shared__ u4 xs[NP * 4], ws[9 * NT * 4];
    const int Kc = DG ? s.Cout : s.Cin, N = DG ? s.Cin : s.Cout;
    const int xst = DG ? s.cs_out : s.cs_in, xof = DG ? s.co_off : s.ci_off;
    const int yst = DG ? s.cs_in : s.cs_out, yof = DG ? s.ci_off : s.co_off;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wx = wave % WX, wy = wave / WX;
    const int tx = s.W / TW, ty = s.H / TH;
    int tile, group;
    tile_group(s.B * tx * ty, N / NT, tile, group);
    const int img = tile / (tx * ty), tr = tile - img * tx * ty;
    const int h0 = (tr / tx) * TH, w0 = (tr % tx) * TW, n0 = group * NT;
    u4 rx[XU], rw[WU];
    auto fetch = [&](int c0) {
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int k = threadIdx.x + u * NTHR, row = k >> 2, c = c0 + 8 * (k & 3);
            const int hh = h0 - 1 + row / PW, ww = w0 - 1 + row % PW;
            rx[u] = u4{0, 0, 0, 0};
            if (k < NP * 4 && c < Kc && hh >= 0 && hh < s.H && ww >= 0 && ww < s.W)
                rx[u] = *(const u4 *)(X + ((size_t)(img * s.H + hh) * s.W + ww) * xst + xof + c);
        }
#pragma unroll
        for (int u = 0; u < WU; u++) {
            const int k = threadIdx.x + u * NTHR, row = k >> 2, c = c0 + 8 * (k & 3), tap = row / NT, n = row % NT;
            rw[u] = u4{0, 0, 0, 0};
            if (k < 9 * NT * 4 && c < Kc) rw[u] = *(const u4 *)(Wt + ((size_t)(n0 + n) * 9 + tap) * Kc + c);
        }
    };
    f4 acc[MR][NB];
#pragma unroll
    for (int m = 0; m < MR; m++)
#pragma unroll
        for (int b = 0; b < NB; b++) acc[m][b] = f4{0, 0, 0, 0};
    const int q = lane >> 4, j = lane & 15;
    const int wunit = j * 4 + (q ^ ((j >> 2) & 3));   // this lane's unit in 16 weight rows
    fetch(0);
    for (int c0 = 0; c0 < Kc; c0 += CV_KC) {
        if (c0) __syncthreads();   // the previous chunk's products are done with the LDS
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int k = threadIdx.x + u * NTHR, row = k >> 2;
            if (k < NP * 4) xs[row * 4 + ((k & 3) ^ ((row >> 2) & 3))] = rx[u];
        }
#pragma unroll
        for (int u = 0; u < WU; u++) {
            const int k = threadIdx.x + u * NTHR, row = k >> 2;
            if (k < 9 * NT * 4) ws[row * 4 + ((k & 3) ^ ((row >> 2) & 3))] = rw[u];
        }
        __syncthreads();
        if (c0 + CV_KC < Kc) fetch(c0 + CV_KC);
        bf8 P[MR + 2][3];
#pragma unroll
        for (int r = 0; r < MR + 2; r++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const int row = (wy * MR + r) * PW + wx * 16 + j + d;
                P[r][d] = *(const bf8 *)(xs + row * 4 + (q ^ ((row >> 2) & 3)));
            }
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            const int dr = DG ? 2 - tap / 3 : tap / 3, dc = DG ? 2 - tap % 3 : tap % 3;
            bf8 A[NB];
#pragma unroll
            for (int b = 0; b < NB; b++) A[b] = *(const bf8 *)(ws + (tap * NT + 16 * b) * 4 + wunit);
#pragma unroll
            for (int m = 0; m < MR; m++)
#pragma unroll
                for (int b = 0; b < NB; b++)
                    acc[m][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[b], P[m + dr][dc], acc[m][b], 0, 0, 0);
        }
    }
#pragma unroll
    for (int m = 0; m < MR; m++) {
        const size_t pix = (size_t)(img * s.H + h0 + wy * MR + m) * s.W + w0 + wx * 16 + j;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int n = n0 + 16 * b + 4 * q;
            f4 v = acc[m][b];
            uint2 o;
            if constexpr (!DG) {
                v += *(const f4 *)(bias + n);
                if (relu)
#pragma unroll
                    for (int e = 0; e < 4; e++) v[e] = fmaxf(v[e], 0.f);
            }
            o.x = pack_bf(v[0], v[1]);
            o.y = pack_bf(v[2], v[3]);
            if (DG && act) {
                const uint2 y = *(const uint2 *)(act + pix * yst + yof + n);
                o.x = mask_bf16x2(o.x, y.x);
                o.y = mask_bf16x2(o.y, y.y);
            }
            *(uint2 *)(Y + pix * yst + yof + n) = o;
        }
    }
}

// The variants: large tiles where they fill the device, small ones where a
// layer has few pixels (see conv_product in mcl_net.cpp).
#define CONV3_TILE(MR, NB, WX, WY)                                                                              \
    template __global__ void k_conv3_tile<MR, NB, WX, WY, false>(ConvShape, const uint16_t *, const uint16_t *, \
                                                                 const uint16_t *, const float *, uint16_t *, int); \
    template __global__ void k_conv3_tile<MR, NB, WX, WY, true>(ConvShape, const uint16_t *, const uint16_t *,  \
                                                                const uint16_t *, const float *, uint16_t *, int);
CONV3_TILE(4, 4, 2, 2)
CONV3_TILE(4, 2, 2, 2)
CONV3_TILE(2, 2, 2, 2)
CONV3_TILE(1, 2, 2, 2)
CONV3_TILE(1, 2, 1, 4)

// 64 pixels x 64 channels in one run of consecutive pixels (a rectangle of one
// image TW = min(W, 64) wide): the layers whose width is not a multiple of 16.
// Waves of 32 x 32, rows padded by 16 bytes.
constexpr int CV_ROW = CV_KC + 8;    // bf16 words per staged pixel or weight row

__global__ void __launch_bounds__(256) k_conv3_mm(ConvShape s, int dgrad, const uint16_t *__restrict__ X,
                                                  const uint16_t *__restrict__ act, const uint16_t *__restrict__ Wt,
                                                  const float *__restrict__ bias, uint16_t *__restrict__ Y, int relu)
{
    constexpr int MT = 64, NT = 64;
    __shared__ __attribute__((aligned(16))) uint16_t xs[3 * (MT + 2) * CV_ROW];
    __shared__ __attribute__((aligned(16))) uint16_t ws[9 * NT * CV_ROW];
    const int Kc = dgrad ? s.Cout : s.Cin, N = dgrad ? s.Cin : s.Cout;
    const int xst = dgrad ? s.cs_out : s.cs_in, xof = dgrad ? s.co_off : s.ci_off;
    const int yst = dgrad ? s.cs_in : s.cs_out, yof = dgrad ? s.ci_off : s.co_off;
    const int sg = dgrad ? -1 : 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / 2, wn = wave % 2;
    const int TW = s.W < MT ? s.W : MT, TH = MT / TW, PW = TW + 2, np = (TH + 2) * PW;
    const int m0 = blockIdx.x * MT, n0 = blockIdx.y * NT;
    const int img = m0 / (s.H * s.W), r0 = m0 - img * s.H * s.W;
    const int h0 = r0 / s.W, w0 = r0 - h0 * s.W;
    const bool active = n0 + wn * 32 < N;
    f4 acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = f4{0, 0, 0, 0};
    // this lane's pixels (patch coordinates of the tap-free position)
    int py[2], px[2];
    for (int a = 0; a < 2; a++) {
        const int ml = wm * 32 + a * 16 + (lane & 15);
        py[a] = ml / TW + 1;
        px[a] = ml - (py[a] - 1) * TW + 1;
    }
    const int kq = 8 * (lane >> 4);
    for (int c0 = 0; c0 < Kc; c0 += CV_KC) {
        __syncthreads();   // the previous chunk's products are done with the LDS
        for (int t = threadIdx.x; t < np * 4; t += 256) {
            const int p = t >> 2, q = t & 3, c = c0 + 8 * q;
            const int hh = h0 - 1 + p / PW, ww = w0 - 1 + p % PW;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (c < Kc && hh >= 0 && hh < s.H && ww >= 0 && ww < s.W)
                v = *(const uint4 *)(X + ((size_t)(img * s.H + hh) * s.W + ww) * xst + xof + c);
            *(uint4 *)(xs + p * CV_ROW + 8 * q) = v;
        }
        for (int t = threadIdx.x; t < 9 * NT * 4; t += 256) {
            const int q = t & 3, row = t >> 2, nl = row % NT, tap = row / NT, c = c0 + 8 * q;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (c < Kc && n0 + nl < N) v = *(const uint4 *)(Wt + ((size_t)(n0 + nl) * 9 + tap) * Kc + c);
            *(uint4 *)(ws + (tap * NT + nl) * CV_ROW + 8 * q) = v;
        }
        __syncthreads();
        if (active) {
            for (int tap = 0; tap < 9; tap++) {
                const int dh = sg * (tap / 3 - 1), dw = sg * (tap % 3 - 1);
                bf8 A[2], B[2];
                for (int a = 0; a < 2; a++)
                    A[a] = *(const bf8 *)(xs + ((py[a] + dh) * PW + px[a] + dw) * CV_ROW + kq);
                for (int b = 0; b < 2; b++)
                    B[b] = *(const bf8 *)(ws + (tap * NT + wn * 32 + b * 16 + (lane & 15)) * CV_ROW + kq);
                for (int a = 0; a < 2; a++)
                    for (int b = 0; b < 2; b++)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a], B[b], acc[a][b], 0, 0, 0);
            }
        }
    }
    if (!active) return;
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) {
            const int n = n0 + wn * 32 + b * 16 + (lane & 15);
            if (n >= N) continue;
            const float bi = (!dgrad && bias) ? bias[n] : 0.f;
            for (int e = 0; e < 4; e++) {
                const size_t idx = (size_t)(m0 + wm * 32 + a * 16 + (lane >> 4) * 4 + e) * yst + yof + n;
                float v = acc[a][b][e] + bi;
                if (relu) v = fmaxf(v, 0.f);
                if (act && bf2f(act[idx]) <= 0.f) v = 0.f;
                Y[idx] = f2bf(v);
            }
        }
}

// ---------------------------------------------------------------- data grad
// din[m, ci] = sum_{tap,co} dout[m - off(tap), co] Wd[ci][tap][co], 0 where act
// (the forward input) is not positive when act != NULL.  Output channels ci of
// the input buffer (stride/offset of the forward input).  Requires Cout % 16 ==
// 0, Cin % 32 == 0.
__global__ void __launch_bounds__(256) k_conv3_dgrad(ConvShape s, const uint16_t *__restrict__ dout,
                                                     const uint16_t *__restrict__ act,
                                                     const uint16_t *__restrict__ Wd, uint16_t *__restrict__ din)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int M = s.B * s.H * s.W;
    const int m0 = blockIdx.x * 64 + (wave >> 1) * 32;
    const int n0 = blockIdx.y * 64 + (wave & 1) * 32;
    if (n0 >= s.Cin) return;
    f4 acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = f4{0, 0, 0, 0};
    int ph[2], pw[2], pn[2];
    bool pv[2];
    for (int a = 0; a < 2; a++) {
        int m = m0 + a * 16 + (lane & 15);
        pv[a] = m < M;
        int mm = pv[a] ? m : 0;
        pn[a] = mm / (s.H * s.W);
        int r = mm - pn[a] * s.H * s.W;
        ph[a] = r / s.W;
        pw[a] = r - ph[a] * s.W;
    }
    const int kq = (lane >> 4) * 4;
    for (int tap = 0; tap < 9; tap++) {
        const int dh = tap / 3 - 1, dw = tap % 3 - 1;
        size_t off[2];
        bool av[2];
        for (int a = 0; a < 2; a++) {
            int h = ph[a] - dh, w = pw[a] - dw;
            av[a] = pv[a] && h >= 0 && h < s.H && w >= 0 && w < s.W;
            off[a] = ((size_t)((pn[a] * s.H + (av[a] ? h : 0)) * s.W + (av[a] ? w : 0))) * s.cs_out + s.co_off;
        }
        for (int c0 = 0; c0 < s.Cout; c0 += 16) {
            s4 A[2], Bv[2];
            for (int a = 0; a < 2; a++) A[a] = load4(dout + off[a] + c0 + kq, av[a]);
            for (int b = 0; b < 2; b++) {
                int ci = n0 + b * 16 + (lane & 15);
                Bv[b] = load4(Wd + ((size_t)ci * 9 + tap) * s.Cout + c0 + kq, ci < s.Cin);
            }
            for (int a = 0; a < 2; a++)
                for (int b = 0; b < 2; b++)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A[a], Bv[b], acc[a][b], 0, 0, 0);
        }
    }
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) {
            int ci = n0 + b * 16 + (lane & 15);
            if (ci >= s.Cin) continue;
            for (int e = 0; e < 4; e++) {
                int m = m0 + a * 16 + (lane >> 4) * 4 + e;
                if (m >= M) continue;
                size_t idx = (size_t)m * s.cs_in + s.ci_off + ci;
                float v = acc[a][b][e];
                if (act && bf2f(act[idx]) <= 0.f) v = 0.f;
                din[idx] = f2bf(v);
            }
        }
}

// -------------------------------------------------------------- weight grad
// dW[co][tap][ci] += sum over a slice of pixels of dout[m,co] in[m+off(tap),ci]
// (FP32 atomics; the pixel range is split over blockIdx.z).  GEMM rows co,
// columns (tap, ci) with ci fastest, K = pixels.
__global__ void __launch_bounds__(256) k_conv3_wgrad(ConvShape s, const uint16_t *__restrict__ dout,
                                                     const uint16_t *__restrict__ in, float *__restrict__ dW,
                                                     int pix_per_split)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int M = s.B * s.H * s.W;
    const int NC = 9 * s.Cin;
    const int r0 = blockIdx.x * 64 + (wave >> 1) * 32;   // co
    const int c0 = blockIdx.y * 64 + (wave & 1) * 32;    // (tap, ci)
    if (r0 >= s.Cout || c0 >= NC) return;
    const int mbeg = blockIdx.z * pix_per_split;
    const int mend = min(M, mbeg + pix_per_split);
    f4 acc[2][2];
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) acc[a][b] = f4{0, 0, 0, 0};
    const int kq = (lane >> 4) * 4;
    int col_tap[2], col_ci[2];
    bool col_ok[2];
    for (int b = 0; b < 2; b++) {
        int c = c0 + b * 16 + (lane & 15);
        col_ok[b] = c < NC;
        int cc = col_ok[b] ? c : 0;
        col_tap[b] = cc / s.Cin;
        col_ci[b] = cc - col_tap[b] * s.Cin;
    }
    for (int mk = mbeg; mk < mend; mk += 16) {
        s4 A[2], Bv[2];
        for (int a = 0; a < 2; a++) {
            int co = r0 + a * 16 + (lane & 15);
            for (int e = 0; e < 4; e++) {
                int m = mk + kq + e;
                short v = 0;
                if (m < mend && co < s.Cout) v = (short)dout[(size_t)m * s.cs_out + s.co_off + co];
                A[a][e] = v;
            }
        }
        for (int b = 0; b < 2; b++) {
            const int dh = col_tap[b] / 3 - 1, dw = col_tap[b] % 3 - 1;
            for (int e = 0; e < 4; e++) {
                int m = mk + kq + e;
                short v = 0;
                if (m < mend && col_ok[b]) {
                    int n = m / (s.H * s.W);
                    int r = m - n * s.H * s.W;
                    int h = r / s.W + dh, w = r % s.W + dw;
                    if (h >= 0 && h < s.H && w >= 0 && w < s.W)
                        v = (short)in[((size_t)((n * s.H + h) * s.W + w)) * s.cs_in + s.ci_off + col_ci[b]];
                }
                Bv[b][e] = v;
            }
        }
        for (int a = 0; a < 2; a++)
            for (int b = 0; b < 2; b++)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(A[a], Bv[b], acc[a][b], 0, 0, 0);
    }
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++) {
            int c = c0 + b * 16 + (lane & 15);
            if (c >= NC) continue;
            for (int e = 0; e < 4; e++) {
                int co = r0 + a * 16 + (lane >> 4) * 4 + e;
                if (co >= s.Cout) continue;
                atomicAdd(&dW[(size_t)co * NC + c], acc[a][b][e]);
            }
        }
}

// LDS-staged weight gradient on v_mfma_f32_16x16x32_bf16 (K = pixels):
// dW[n][tap][c] += sum_m G[m, n] X[m + off(tap), c], G = dout, X = in.  A
// workgroup owns NBLK output channels n, 32 input channels c and all nine taps
// and sums over tiles_per_split tiles of 32 x TH pixels of one image; the
// partial sums are added to dW with FP32 atomics, and the workgroups of the
// first channel block add the bias gradient db[n] = sum_m G[m, n].
// G and X lie in LDS as in memory (a pixel's channels together; X with one
// pixel around): the operands want eight consecutive pixels of one channel,
// which the transposing LDS read gives (ds_read_b64_tr_b16: among 16 lanes,
// lane i gets element i % 4 of the lanes 4 j + i / 4, j = 0..3), for the
// shifted taps at another pixel offset of the same copy.  A wave has 32 n x 16
// c x 9 taps (18 accumulators); it walks down the tile's rows and keeps the
// fragments of three rows, so that a row costs 10 transposing reads for 18
// MFMAs.  (Before, G was transposed and X copied three times with 2-byte LDS
// writes: 399 us a layer at 256 x 256, batch 32, now 110.)  With NBLK = 32 two of
// the waves take the lower half of the rows.  The next tile's loads are in flight
// while the products run.
typedef short bs4 __attribute__((ext_vector_type(4)));

template <int ROWB>
__device__ __forceinline__ bf8 tr_frag(const char *p)
{
    // rows (pixels) 0..3 and 4..7 of this lane's eight
    typedef __attribute__((address_space(3))) bs4 lds_s4;
    const bs4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(p));
    const bs4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(p + 4 * ROWB));
    union {
        bs4 h[2];
        bf8 v;
    } u;
    u.h[0] = lo;
    u.h[1] = hi;
    return u.v;
}

template <int NBLK, int TH>
__global__ void __launch_bounds__(256) k_conv3_wgrad_tile(ConvShape s, const uint16_t *__restrict__ dout,
                                                          const uint16_t *__restrict__ in, float *__restrict__ dW,
                                                          float *__restrict__ db, int tiles_per_split)
{
    constexpr int TW = 32, PW = TW + 2, NP = PW * (TH + 2), GP = TW * TH, GQ = NBLK / 8;
    constexpr int XROW = 64, GROW = NBLK == 64 ? 144 : 64;   // bytes a pixel (G of 64 channels padded: banks)
    constexpr int XU = (NP * 4 + 255) / 256, GU = GP * GQ / 256;
    constexpr int ROWS = NBLK == 64 ? TH : TH / 2;           // rows of a wave
    __shared__ __attribute__((aligned(16))) char xs[NP * XROW], gs[GP * GROW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wn = NBLK == 64 ? wave & 1 : 0, wc = NBLK == 64 ? wave >> 1 : wave & 1;
    const int y0 = NBLK == 64 ? 0 : (wave >> 1) * ROWS;
    const int tx = s.W / TW, ty = s.H / TH, ntiles = s.B * tx * ty;
    const int n0 = blockIdx.x * NBLK, c0 = blockIdx.y * 32;
    const int tb = blockIdx.z * tiles_per_split, te = min(ntiles, tb + tiles_per_split);
    const bool bias = blockIdx.y == 0 && wc == 0;
    u4 rx[XU], rg[GU];
    auto fetch = [&](int tile) {
        const int img = tile / (tx * ty), tr = tile - img * tx * ty;
        const int h0 = (tr / tx) * TH, w0 = (tr % tx) * TW;
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int k = threadIdx.x + u * 256, row = k >> 2, c = c0 + 8 * (k & 3);
            const int hh = h0 - 1 + row / PW, ww = w0 - 1 + row % PW;
            rx[u] = u4{0, 0, 0, 0};
            if (k < NP * 4 && c < s.Cin && hh >= 0 && hh < s.H && ww >= 0 && ww < s.W)
                rx[u] = *(const u4 *)(in + ((size_t)(img * s.H + hh) * s.W + ww) * s.cs_in + s.ci_off + c);
        }
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int k = threadIdx.x + u * 256, p = k / GQ, q = k % GQ;
            rg[u] = *(const u4 *)(dout + ((size_t)(img * s.H + h0 + p / TW) * s.W + w0 + p % TW) * s.cs_out +
                                     s.co_off + n0 + 8 * q);
        }
    };
    f4 acc[9][2];
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int a = 0; a < 2; a++) acc[t][a] = f4{0, 0, 0, 0};
    float bsum[2] = {0.f, 0.f};   // this lane's share of sum_m G[m, n], n = n0 + 32 wn + 16 a + lane % 16
    // this lane's pixel and channels in a transposing read
    const int pix = 8 * (lane >> 4) + ((lane & 15) >> 2), ch = 4 * (lane & 3);
    const char *gp = gs + pix * GROW + 2 * (32 * wn + ch), *xp = xs + pix * XROW + 2 * (16 * wc + ch);
    if (tb < te) fetch(tb);
    for (int tile = tb; tile < te; tile++) {
        __syncthreads();   // the previous tile's products are done with the LDS
#pragma unroll
        for (int u = 0; u < XU; u++) {
            const int k = threadIdx.x + u * 256;
            if (k < NP * 4) *(u4 *)(xs + (k >> 2) * XROW + 16 * (k & 3)) = rx[u];
        }
#pragma unroll
        for (int u = 0; u < GU; u++) {
            const int k = threadIdx.x + u * 256;
            *(u4 *)(gs + (k / GQ) * GROW + 16 * (k % GQ)) = rg[u];
        }
        __syncthreads();
        if (tile + 1 < te) fetch(tile + 1);
        bf8 F0[3], F1[3], F2[3];   // rows y, y + 1, y + 2 of the patch
#pragma unroll
        for (int d = 0; d < 3; d++) {
            F1[d] = tr_frag<XROW>(xp + (y0 * PW + d) * XROW);
            F2[d] = tr_frag<XROW>(xp + ((y0 + 1) * PW + d) * XROW);
        }
#pragma unroll
        for (int y = 0; y < ROWS; y++) {
#pragma unroll
            for (int d = 0; d < 3; d++) {
                F0[d] = F1[d];
                F1[d] = F2[d];
                F2[d] = tr_frag<XROW>(xp + ((y0 + y + 2) * PW + d) * XROW);
            }
            bf8 A[2];
#pragma unroll
            for (int a = 0; a < 2; a++) A[a] = tr_frag<GROW>(gp + (y0 + y) * TW * GROW + 32 * a);
            if (bias)
#pragma unroll
                for (int a = 0; a < 2; a++)
#pragma unroll
                    for (int k = 0; k < 8; k++) bsum[a] += (float)A[a][k];
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const bf8 X = t < 3 ? F0[t] : t < 6 ? F1[t - 3] : F2[t - 6];
#pragma unroll
                for (int a = 0; a < 2; a++)
                    acc[t][a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[a], X, acc[t][a], 0, 0, 0);
            }
        }
    }
    if (bias)
#pragma unroll
        for (int a = 0; a < 2; a++) {
            float v = bsum[a];
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (lane < 16) atomicAdd(&db[n0 + 32 * wn + 16 * a + lane], v);
        }
    const int c = c0 + 16 * wc + (lane & 15);
    if (c >= s.Cin) return;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                atomicAdd(&dW[((size_t)(n0 + 32 * wn + 16 * a + (lane >> 4) * 4 + e) * 9 + t) * s.Cin + c],
                          acc[t][a][e]);
}

template __global__ void k_conv3_wgrad_tile<64, 8>(ConvShape, const uint16_t *, const uint16_t *, float *, float *, int);
template __global__ void k_conv3_wgrad_tile<64, 4>(ConvShape, const uint16_t *, const uint16_t *, float *, float *, int);
template __global__ void k_conv3_wgrad_tile<32, 8>(ConvShape, const uint16_t *, const uint16_t *, float *, float *, int);

// The same for the levels that k_conv3_wgrad_tile has no tile for: 8 or 16
// pixels wide, or 32 and 64 with a height that 4 does not divide.  A workgroup
// owns 64 output channels n, 32 input channels c and all nine taps (waves: 16 n
// each, 18 tiles of 16 x 16), and sums over tiles_per_split runs of 64 pixels
// (TH x TW rectangles of one image, as k_conv3_mm).  Per run it stages G
// transposed (channel-major, 64 pixels a row) and three copies of the X patch
// shifted by -1, 0, +1 columns, channel-major, so that every operand fragment --
// 8 consecutive pixels of one channel -- is one 16-byte LDS read; what bounds it
// is that staging by 2-byte writes (39 us a launch in a 64 x 64 network, batch
// 32).  Requires TW % 8 == 0 (the host checks the shapes).  A training step with
// these levels on the unstaged kernel and on this one: 64 x 64, batch 32, 3.1 and
// 1.13 ms; 256 x 64, batch 4, 2.6 and 0.89 ms; 512 x 16, batch 8, 7.1 and 3.0 ms.
constexpr int WG_XP = 72;   // bf16 words per staged G row (64 pixels + pad)

__global__ void __launch_bounds__(256) k_conv3_wgrad_mm(ConvShape s, const uint16_t *__restrict__ dout,
                                                        const uint16_t *__restrict__ in, float *__restrict__ dW,
                                                        float *__restrict__ db, int tiles_per_split)
{
    __shared__ __attribute__((aligned(16))) uint16_t gt[64 * WG_XP];
    __shared__ __attribute__((aligned(16))) uint16_t xs[3 * 32 * 3 * 72];   // largest: TW = 64, TH + 2 = 3
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int TW = s.W < 64 ? s.W : 64, TH = 64 / TW, PR = TH + 2, XP = TW + 8;
    const int n0 = blockIdx.x * 64, c0 = blockIdx.y * 32;
    const int ntiles = s.B * s.H * s.W / 64;
    const int tb = blockIdx.z * tiles_per_split, te = min(ntiles, tb + tiles_per_split);
    const bool active = n0 + 16 * wave < s.Cout;
    const bool bias = blockIdx.y == 0;
    float bsum = 0.f;   // this lane's share of sum_m G[m, n] for n = n0 + 16 wave + lane % 16
    f4 acc[9][2];
    for (int t = 0; t < 9; t++)
        for (int b = 0; b < 2; b++) acc[t][b] = f4{0, 0, 0, 0};
    const int kq = 8 * (lane >> 4);
    for (int tile = tb; tile < te; tile++) {
        const int m0 = tile * 64;
        const int img = m0 / (s.H * s.W), r0 = m0 - img * s.H * s.W;
        const int h0 = r0 / s.W, w0 = r0 - h0 * s.W;
        __syncthreads();   // the previous tile's products are done with the LDS
        // G^T: 64 pixels x 64 channels (8 channels per 16-byte load)
        for (int t = threadIdx.x; t < 64 * 8; t += 256) {
            const int p = t >> 3, q = t & 7, n = n0 + 8 * q;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (n < s.Cout) v = *(const uint4 *)(dout + (size_t)(m0 + p) * s.cs_out + s.co_off + n);
            const uint16_t *e = (const uint16_t *)&v;
#pragma unroll
            for (int k = 0; k < 8; k++) gt[(8 * q + k) * WG_XP + p] = e[k];
        }
        // X patch (PR rows x TW + 2 columns) into the three shifted copies
        const int pw = TW + 2;
        for (int t = threadIdx.x; t < PR * pw * 4; t += 256) {
            const int pp = t >> 2, q = t & 3, c = c0 + 8 * q;
            const int prow = pp / pw, pcol = pp - prow * pw;
            const int hh = h0 - 1 + prow, ww = w0 - 1 + pcol;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (c < s.Cin && hh >= 0 && hh < s.H && ww >= 0 && ww < s.W)
                v = *(const uint4 *)(in + ((size_t)(img * s.H + hh) * s.W + ww) * s.cs_in + s.ci_off + c);
            const uint16_t *e = (const uint16_t *)&v;
            // copy sh holds X at column col + sh - 1 of the tile: col = pcol - sh
#pragma unroll
            for (int sh = 0; sh < 3; sh++) {
                const int col = pcol - sh;
                if (col < 0 || col >= TW) continue;
#pragma unroll
                for (int k = 0; k < 8; k++) xs[((sh * 32 + 8 * q + k) * PR + prow) * XP + col] = e[k];
            }
        }
        __syncthreads();
        if (!active) continue;
        for (int kk = 0; kk < 64; kk += 32) {
            const bf8 A = *(const bf8 *)(gt + (16 * wave + (lane & 15)) * WG_XP + kk + kq);
            if (bias) {
                const uint4 a4 = *(const uint4 *)(gt + (16 * wave + (lane & 15)) * WG_XP + kk + kq);
                const uint16_t *e = (const uint16_t *)&a4;
#pragma unroll
                for (int k = 0; k < 8; k++) bsum += bf2f(e[k]);
            }
            const int p = kk + kq, py = p / TW, px = p - py * TW;
            for (int tap = 0; tap < 9; tap++) {
                const int dh = tap / 3 - 1, sh = tap % 3;
                for (int b = 0; b < 2; b++) {
                    const bf8 B = *(const bf8 *)(xs + ((sh * 32 + 16 * b + (lane & 15)) * PR + py + dh + 1) * XP + px);
                    acc[tap][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, acc[tap][b], 0, 0, 0);
                }
            }
        }
    }
    if (!active) return;
    if (bias) {
        bsum += __shfl_xor(bsum, 16, 64);
        bsum += __shfl_xor(bsum, 32, 64);
        const int n = n0 + 16 * wave + lane;
        if (lane < 16 && n < s.Cout) atomicAdd(&db[n], bsum);
    }
    const int NC = 9 * s.Cin;
    for (int tap = 0; tap < 9; tap++)
        for (int b = 0; b < 2; b++) {
            const int c = c0 + 16 * b + (lane & 15);
            if (c >= s.Cin) continue;
            for (int e = 0; e < 4; e++) {
                const int n = n0 + 16 * wave + (lane >> 4) * 4 + e;
                if (n < s.Cout) atomicAdd(&dW[(size_t)n * NC + tap * s.Cin + c], acc[tap][b][e]);
            }
        }
}

// db[co] += sum_m dout[m, co]
__global__ void k_bias_grad(int M, int Cout, int cs, int coff, const uint16_t *__restrict__ dout,
                            float *__restrict__ db)
{
    int co = threadIdx.x % Cout;
    int lanes = blockDim.x / Cout;
    int sub = threadIdx.x / Cout;
    if (sub >= lanes) return;
    float s = 0.f;
    for (int m = blockIdx.x * lanes + sub; m < M; m += gridDim.x * lanes)
        s += bf2f(dout[(size_t)m * cs + coff + co]);
    atomicAdd(&db[co], s);
}

// ------------------------------------------------------- pooling / upsampling
// One thread moves eight channels of a pixel (16-byte accesses): C, the strides
// and the offsets are multiples of 8.
union Bf8 {
    uint4 q;
    uint16_t e[8];
};

// 2x2 average pooling: out (B, H/2, W/2) from in (B, H, W), C channels.
__global__ void k_pool_fwd(int B, int H, int W, int C, const uint16_t *__restrict__ in, int cs_in, int ci_off,
                           uint16_t *__restrict__ out, int cs_out, int co_off)
{
    const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
    const size_t total = (size_t)B * Ho * Wo * C8;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(t % C8) * 8;
        const size_t p = t / C8;
        const int w = p % Wo, h = (p / Wo) % Ho, n = p / ((size_t)Wo * Ho);
        Bf8 v[4], o;
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k].q = *(const uint4 *)(in + ((size_t)((n * H + 2 * h + k / 2) * W + 2 * w + k % 2)) * cs_in + ci_off + c);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 4; k++) s += bf2f(v[k].e[e]);
            o.e[e] = f2bf(0.25f * s);
        }
        *(uint4 *)(out + p * cs_out + co_off + c) = o.q;
    }
}

// din += pool^T dout, 0 where act (the pooled activation) is not positive
__global__ void k_pool_bwd(int B, int H, int W, int C, const uint16_t *__restrict__ dout, int cs_out, int co_off,
                           const uint16_t *__restrict__ act, uint16_t *__restrict__ din, int cs_in, int ci_off)
{
    const int Ho = H / 2, Wo = W / 2, C8 = C / 8;
    const size_t total = (size_t)B * H * W * C8;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(t % C8) * 8;
        const size_t p = t / C8;
        const int w = p % W, h = (p / W) % H, n = p / ((size_t)W * H);
        const size_t idx = p * cs_in + ci_off + c;
        Bf8 g, d, y, o;
        g.q = *(const uint4 *)(dout + ((size_t)((n * Ho + h / 2) * Wo + w / 2)) * cs_out + co_off + c);
        d.q = *(const uint4 *)(din + idx);
        y.q = *(const uint4 *)(act + idx);
#pragma unroll
        for (int e = 0; e < 8; e++)
            o.e[e] = bf2f(y.e[e]) <= 0.f ? (uint16_t)0 : f2bf(0.25f * bf2f(g.e[e]) + bf2f(d.e[e]));
        *(uint4 *)(din + idx) = o.q;
    }
}

// nearest 2x upsampling: out (B, 2H, 2W) from in (B, H, W)
__global__ void k_up_fwd(int B, int H, int W, int C, const uint16_t *__restrict__ in, int cs_in, int ci_off,
                         uint16_t *__restrict__ out, int cs_out, int co_off)
{
    const int Ho = 2 * H, Wo = 2 * W, C8 = C / 8;
    const size_t total = (size_t)B * Ho * Wo * C8;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(t % C8) * 8;
        const size_t p = t / C8;
        const int w = p % Wo, h = (p / Wo) % Ho, n = p / ((size_t)Wo * Ho);
        *(uint4 *)(out + p * cs_out + co_off + c) =
            *(const uint4 *)(in + ((size_t)((n * H + h / 2) * W + w / 2)) * cs_in + ci_off + c);
    }
}

// din = up^T dout: the sum of the four copies' gradients
__global__ void k_up_bwd(int B, int H, int W, int C, const uint16_t *__restrict__ dout, int cs_out, int co_off,
                         uint16_t *__restrict__ din, int cs_in, int ci_off)
{
    const int Ho = 2 * H, Wo = 2 * W, C8 = C / 8;
    const size_t total = (size_t)B * H * W * C8;
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const int c = (int)(t % C8) * 8;
        const size_t p = t / C8;
        const int w = p % W, h = (p / W) % H, n = p / ((size_t)W * H);
        Bf8 v[4], o;
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k].q = *(const uint4 *)(dout + ((size_t)((n * Ho + 2 * h + k / 2) * Wo + 2 * w + k % 2)) * cs_out +
                                      co_off + c);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < 4; k++) s += bf2f(v[k].e[e]);
            o.e[e] = f2bf(s);
        }
        *(uint4 *)(din + p * cs_in + ci_off + c) = o.q;
    }
}

// ------------------------------------------------------------- head and loss
// The 1x1 head: 32 channels -> 3 outputs (FP32).  A pixel's 32 bf16 channels
// are four 16-byte loads (channel stride a multiple of 8).
constexpr int HC = 32, HO = 3;

__device__ __forceinline__ void load32(const uint16_t *p, float (&x)[HC])
{
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint4 v = *(const uint4 *)(p + 8 * q);
        const uint16_t *e = (const uint16_t *)&v;
#pragma unroll
        for (int k = 0; k < 8; k++) x[8 * q + k] = bf2f(e[k]);
    }
}

// y[m, o] = bh[o] + sum_c Wh[o][c] x[m, c]
__global__ void __launch_bounds__(256) k_head_fwd(int M, const uint16_t *__restrict__ x, int cs,
                                                  const float *__restrict__ Wh, const float *__restrict__ bh,
                                                  float *__restrict__ y)
{
    __shared__ float w[HO * HC + HO];
    for (int t = threadIdx.x; t < HO * HC + HO; t += blockDim.x) w[t] = t < HO * HC ? Wh[t] : bh[t - HO * HC];
    __syncthreads();
    for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        float xv[HC];
        load32(x + (size_t)m * cs, xv);
#pragma unroll
        for (int o = 0; o < HO; o++) {
            float s = w[HO * HC + o];
#pragma unroll
            for (int c = 0; c < HC; c++) s += w[o * HC + c] * xv[c];
            y[(size_t)m * HO + o] = s;
        }
    }
}

// dy = 2 (y - t) / (M O), loss partials; dx[m,c] = sum_o Wh[o][c] dy, 0 where x is not positive; dWh,
// dbh and the loss summed per thread in registers, then per workgroup, then
// one atomic per value and workgroup.
__global__ void __launch_bounds__(256) k_head_bwd(int M, const uint16_t *__restrict__ x, int cs,
                                                  const float *__restrict__ Wh, const float *__restrict__ y,
                                                  const float *__restrict__ tgt, float scale,
                                                  uint16_t *__restrict__ dx, float *__restrict__ dWh,
                                                  float *__restrict__ dbh, float *__restrict__ loss)
{
    constexpr int NV = HO * HC + HO + 1;   // dWh, dbh, loss
    __shared__ float w[HO * HC];
    __shared__ float red[4][NV];
    for (int t = threadIdx.x; t < HO * HC; t += blockDim.x) w[t] = Wh[t];
    __syncthreads();
    float aw[HO * HC], ab[HO], ls = 0.f;
#pragma unroll
    for (int k = 0; k < HO * HC; k++) aw[k] = 0.f;
#pragma unroll
    for (int o = 0; o < HO; o++) ab[o] = 0.f;
    for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < M; m += gridDim.x * blockDim.x) {
        float dy[HO];
#pragma unroll
        for (int o = 0; o < HO; o++) {
            const float r = y[(size_t)m * HO + o] - tgt[(size_t)m * HO + o];
            ls += r * r;
            dy[o] = scale * r;
            ab[o] += dy[o];
        }
        float xv[HC];
        load32(x + (size_t)m * cs, xv);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            uint4 v;
            uint16_t *e = (uint16_t *)&v;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int c = 8 * q + k;
                float g = 0.f;
#pragma unroll
                for (int o = 0; o < HO; o++) {
                    g += w[o * HC + c] * dy[o];
                    aw[o * HC + c] += dy[o] * xv[c];
                }
                e[k] = xv[c] <= 0.f ? (uint16_t)0 : f2bf(g);   // x is a ReLU's output
            }
            *(uint4 *)(dx + (size_t)m * cs + 8 * q) = v;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        float v = k < HO * HC ? aw[k] : k < HO * HC + HO ? ab[k - HO * HC] : ls;
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
        if (lane == 0) red[wave][k] = v;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < NV; k += blockDim.x) {
        const float v = red[0][k] + red[1][k] + red[2][k] + red[3][k];
        if (k < HO * HC) atomicAdd(&dWh[k], v);
        else if (k < HO * HC + HO) atomicAdd(&dbh[k - HO * HC], v);
        else atomicAdd(loss, v);
    }
}

// ----------------------------------------------------------------- Adam etc.
// Adam step (STEP; Kingma & Ba 2015) on the FP32 master weights [co][tap][ci],
// and the bf16 weights of every layer from them: Wf ([co][tap][ci]) and Wd
// ([ci][tap][co]).  blockIdx.y is the layer; one launch, where one a tensor for
// each of the two took 44.  What bounds it is the rounds of the largest layer:
// 24 to 35 us with the step, 28 without.
template <bool STEP>
__global__ void __launch_bounds__(256)
k_update_weights(NetLayers ls, float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m1,
                 float *__restrict__ m2, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const NetLayer l = ls.l[blockIdx.y];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < l.nw + l.nb; i += gridDim.x * blockDim.x) {
        const int j = l.off + i;
        float wi = w[j];
        if (STEP) {
            float gi = g[j];
            float a = b1 * m1[j] + (1.f - b1) * gi;
            float b = b2 * m2[j] + (1.f - b2) * gi * gi;
            m1[j] = a;
            m2[j] = b;
            wi -= lr * (a / c1) / (sqrtf(b / c2) + eps);
            w[j] = wi;
        }
        if (i < l.nw) {
            const int ci = i % l.Cin, tap = (i / l.Cin) % 9, co = i / (9 * l.Cin);
            const uint16_t v = f2bf(wi);
            l.Wf[i] = v;
            l.Wd[((size_t)ci * 9 + tap) * l.nb + co] = v;
        }
    }
}
template __global__ void k_update_weights<true>(NetLayers, float *, const float *, float *, float *, float, float,
                                                float, float, float, float);
template __global__ void k_update_weights<false>(NetLayers, float *, const float *, float *, float *, float, float,
                                                 float, float, float, float);

__global__ void k_f32_to_bf16(size_t n, const float *__restrict__ x, uint16_t *__restrict__ y)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        y[i] = f2bf(x[i]);
}

__global__ void k_bf16_to_f32(size_t n, const uint16_t *__restrict__ x, float *__restrict__ y)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        y[i] = bf2f(x[i]);
}
