// warmstart.hip -- the warm-start network's kernels (gfx950) and its trainer.
//
// Convolutions with 32 input channels run on the matrix cores as implicit
// GEMMs with v_mfma_f32_16x16x32_bf16: M = 16 output channels, N = 16
// pixels of one image row, K = the 32 input channels of one tap, accumulated
// over the 9 taps in FP32.  The backward pass of such a layer with respect to
// its input is the same kernel with the taps flipped and the channel roles
// swapped; its weight gradient is a GEMM with K = pixels (M = input channels,
// N = output channels).  The 32 -> 1 output layer is VALU work.
//
// Operand layout of the 16x16x32 BF16 MFMA (64 lanes): lane l holds row
// l % 16 of A and column l % 16 of B, each with 8 K-values at positions
// 8*(l/16) .. 8*(l/16)+7; the result lane l holds column l % 16, rows
// 4*(l/16) .. 4*(l/16)+3.  A and B use the same K positions, so any
// permutation of K inside the hardware leaves the product unchanged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/tea_warmstart.h"
#include "ws_net.hpp"

#define EXPORT extern "C" __attribute__((visibility("default")))

namespace ws {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned int)))) unsigned int uintx4;

constexpr int BLOCK = 256;
constexpr int NPLANES = 6;   // training sample: f0, f1, f2, target, Kx, Ky

__device__ __forceinline__ floatx4 mfma(bf16x8 a, bf16x8 b, floatx4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float bf16_round(float x) { return (float)(__bf16)x; }

// Flat index of pixel (y, x) of image b in a padded image batch (y, x interior
// coordinates; -1 and H / W address the zero border).
__device__ __forceinline__ long padded(int b, int y, int x, int H, int W)
{
    return ((long)b * (H + 2) + (y + 1)) * (W + 2) + (x + 1);
}

// ---------------------------------------------------------------- parameters

__global__ void k_pack(const float *__restrict__ p, __bf16 *__restrict__ packed, float *__restrict__ w6)
{
    const int e = blockIdx.x * BLOCK + threadIdx.x;
    if (e < TAPS * CH) w6[e] = bf16_round(p[OFF_W6 + e]);
    if (e >= PK_TOTAL) return;
    float v;
    if (e >= PK_OUT) {   // layer 6: W6 in row 0 (lanes 0, 16, 32, 48), zeros elsewhere
        const int r = e - PK_OUT, t = r / FRAG, lane = (r / 8) % 64, i = r % 8;
        v = lane % 16 == 0 ? p[OFF_W6 + t * CH + (lane / 16) * 8 + i] : 0.0f;
    } else if (e < PK_HID) {
        const int nb = e / FRAG, lane = (e / 8) % 64, i = e % 8;
        const int k = (lane / 16) * 8 + i, co = nb * 16 + lane % 16;
        v = k < K1 ? p[OFF_W1 + k * CH + co] : 0.0f;
    } else {
        const int e2 = e - PK_HID;
        const int per_layer = TAPS * 2 * FRAG;
        const bool bwd = e2 >= HIDDEN * per_layer;
        const int r0 = e2 % (HIDDEN * per_layer);
        const int l = r0 / per_layer + 2, r = r0 % per_layer;
        const int t = r / (2 * FRAG), nb = (r / FRAG) % 2, lane = (r / 8) % 64, i = r % 8;
        const int k = (lane / 16) * 8 + i, n = nb * 16 + lane % 16;
        const float *w = p + off_w(l);
        // forward: K = ci, N = co; backward: K = co, N = ci, tap mirrored
        v = bwd ? w[((TAPS - 1 - t) * CH + n) * CH + k] : w[(t * CH + k) * CH + n];
    }
    packed[e] = (__bf16)v;
}

// ---------------------------------------------------------------- forward

// planes[b][f][y][x] (npl planes per image, the first three are the features)
// -> x1[b][y][x][k], k = tap*3 + f, zero for k >= 27 and outside the image.
__global__ void k_im2col(const float *__restrict__ planes, int npl, __bf16 *__restrict__ x1, int B, int H, int W)
{
    const long p = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (p >= (long)B * H * W) return;
    const int x = (int)(p % W), y = (int)((p / W) % H), b = (int)(p / ((long)W * H));
    const float *pl = planes + (long)b * npl * H * W;
    bf16x8 v[4];
#pragma unroll
    for (int k = 0; k < CH; k++) {
        float f = 0.0f;
        if (k < K1) {
            const int t = k / 3, c = k % 3;
            const int yy = y + t / 3 - 1, xx = x + t % 3 - 1;
            if (yy >= 0 && yy < H && xx >= 0 && xx < W) f = pl[(long)c * H * W + (long)yy * W + xx];
        }
        v[k / 8][k % 8] = (__bf16)f;
    }
    bf16x8 *dst = (bf16x8 *)(x1 + padded(b, y, x, H, W) * CH);
#pragma unroll
    for (int q = 0; q < 4; q++) dst[q] = v[q];
}

// Convolution kernels: a workgroup of CONV_ROWS waves computes rows
// y0 .. y0+CONV_ROWS-1, 64 pixels from x0, one row per wave (4 blocks of 16
// pixels) and all 32 output channels (2 blocks of 16).  It first stages its
// input window (rows y0-1 .. y0+CONV_ROWS, pixels x0-1 .. x0+64) in LDS with
// 16-byte loads; the taps then read the window from LDS.  The MFMA's A operand
// is the weight fragment (rows = output channels), B the activations
// (columns = pixels), so each lane's result is 4 consecutive channels of one
// pixel, stored as one 8-byte vector.  Grid (W/64, H/ROWS, B); ROWS = 8
// where H allows it (a smaller share of re-read halo rows), else 4.
constexpr int WIN_X = 64 + 2;
constexpr int LDS_PIX = CH + 8;   // bf16 per staged pixel: an 80-byte stride spreads 16-byte reads over the banks
inline int conv_rows(int H) { return H % 8 == 0 ? 8 : 4; }

// Stages rows y0-1 .. y0+ROWS of a padded NHWC32 image into win.
template <int ROWS>
__device__ __forceinline__ void stage_nhwc32(const __bf16 *__restrict__ in, __bf16 *win, int b, int y0, int x0,
                                             int H, int W)
{
    constexpr int CHUNKS = (ROWS + 2) * WIN_X * 4;   // 16-byte pieces, 4 per pixel
    for (int c = threadIdx.x; c < CHUNKS; c += ROWS * 64) {
        const int r = c / (WIN_X * 4), rem = c - r * (WIN_X * 4), px = rem >> 2, q = rem & 3;
        const bf16x8 v = *(const bf16x8 *)(in + padded(b, y0 - 1 + r, x0 - 1 + px, H, W) * CH + q * 8);
        *(bf16x8 *)(win + (r * WIN_X + px) * LDS_PIX + q * 8) = v;
    }
    __syncthreads();
}

// acc (4 pixel blocks x 2 channel blocks) -> out at row y, pixels x0..x0+63.
// Forward: bf16(relu(acc + bias)); backward (BWD): bf16(acc * (mask > 0)).
template <bool BWD>
__device__ __forceinline__ void store_nhwc32(const floatx4 (&acc)[4][2], __bf16 *__restrict__ out,
                                             const float *__restrict__ bias, const __bf16 *__restrict__ mask, int b,
                                             int y, int x0, int H, int W)
{
    const int lane = threadIdx.x & 63, m = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) {
            const int co = nb * 16 + kg * 4;
            const long idx = padded(b, y, x0 + mb * 16 + m, H, W) * CH + co;
            bf16x4 o;
            bf16x4 mk;
            if (BWD) mk = *(const bf16x4 *)(mask + idx);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = acc[mb][nb][i];
                if (BWD) v = (float)mk[i] > 0.0f ? v : 0.0f;
                else v = fmaxf(v + bias[co + i], 0.0f);
                o[i] = (__bf16)v;
            }
            *(bf16x4 *)(out + idx) = o;
        }
}

// 32 -> 32 channels, 3x3 taps.
// Forward:  out = bf16(relu(conv(in) + bias)).
// Backward (BWD): out = bf16(conv(in) * (mask > 0)), mask = the layer's forward input.
template <int ROWS, bool BWD>
__global__ __launch_bounds__(ROWS * 64) void k_conv32(const __bf16 *__restrict__ in, __bf16 *__restrict__ out,
                                                      const bf16x8 *__restrict__ frag, const float *__restrict__ bias,
                                                      const __bf16 *__restrict__ mask, int H, int W)
{
    __shared__ __attribute__((aligned(16))) __bf16 win[(ROWS + 2) * WIN_X * LDS_PIX];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int y0 = blockIdx.y * ROWS, x0 = blockIdx.x * 64, b = blockIdx.z;
    stage_nhwc32<ROWS>(in, win, b, y0, x0, H, W);
    floatx4 acc[4][2];
#pragma unroll
    for (int mb = 0; mb < 4; mb++) acc[mb][0] = acc[mb][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < TAPS; t++) {
        const int dy = t / 3 - 1, dx = t % 3 - 1;
        const bf16x8 w0 = frag[(t * 2 + 0) * 64 + lane];
        const bf16x8 w1 = frag[(t * 2 + 1) * 64 + lane];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) {
            const bf16x8 a = *(const bf16x8 *)(win + ((wave + 1 + dy) * WIN_X + 1 + mb * 16 + m + dx) * LDS_PIX + kg * 8);
            acc[mb][0] = mfma(w0, a, acc[mb][0]);
            acc[mb][1] = mfma(w1, a, acc[mb][1]);
        }
    }
    store_nhwc32<BWD>(acc, out, bias, mask, b, y0 + wave, x0, H, W);
}

// Layer 1 straight from the feature planes (planes[b][f][y][x], npl planes
// per image, features f = 0..2): the im2col value k = tap*3 + f (zero for
// k >= 27 and outside the image) of each pixel is formed from the staged
// planes, then one MFMA K-block does the whole 3x3x3 -> 32 convolution.
template <int ROWS>
__global__ __launch_bounds__(ROWS * 64) void k_conv_first(const float *__restrict__ planes, int npl,
                                                          __bf16 *__restrict__ out, const bf16x8 *__restrict__ frag,
                                                          const float *__restrict__ bias, int H, int W)
{
    constexpr int WIN_Y = ROWS + 2;
    __shared__ float feat[NFEAT][WIN_Y][WIN_X];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int y0 = blockIdx.y * ROWS, x0 = blockIdx.x * 64, b = blockIdx.z;
    const float *pl = planes + (long)b * npl * H * W;
    for (int c = threadIdx.x; c < NFEAT * WIN_Y * WIN_X; c += ROWS * 64) {
        const int f = c / (WIN_Y * WIN_X), rem = c - f * (WIN_Y * WIN_X), r = rem / WIN_X, px = rem - r * WIN_X;
        const int y = y0 - 1 + r, x = x0 - 1 + px;
        feat[f][r][px] = (y >= 0 && y < H && x >= 0 && x < W) ? pl[(long)f * H * W + (long)y * W + x] : 0.0f;
    }
    __syncthreads();
    // this lane's 8 K-values: offsets into feat relative to the pixel
    int off[8];
    bool real[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int k = kg * 8 + i, t = k / 3, f = k - 3 * t;
        real[i] = k < K1;
        off[i] = real[i] ? (f * WIN_Y + (t / 3 - 1)) * WIN_X + (t % 3 - 1) : 0;
    }
    const float *base = &feat[0][wave + 1][1];
    const bf16x8 w0 = frag[lane], w1 = frag[64 + lane];
    floatx4 acc[4][2];
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
        bf16x8 a;
#pragma unroll
        for (int i = 0; i < 8; i++) a[i] = (__bf16)(real[i] ? base[mb * 16 + m + off[i]] : 0.0f);
        const floatx4 z = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        acc[mb][0] = mfma(w0, a, z);
        acc[mb][1] = mfma(w1, a, z);
    }
    store_nhwc32<false>(acc, out, bias, (const __bf16 *)nullptr, b, y0 + wave, x0, H, W);
}

// Layer 6 (32 -> 1) on the matrix cores: the A fragment (packed at PK_OUT)
// holds W6 in its first row (output channel 0) and zeros elsewhere;
// out[b][y][x] = b6 + acc.
template <int ROWS>
__global__ __launch_bounds__(ROWS * 64) void k_conv_out(const __bf16 *__restrict__ a5, const bf16x8 *__restrict__ frag,
                                                        const float *__restrict__ b6, float *__restrict__ out, int H,
                                                        int W)
{
    __shared__ __attribute__((aligned(16))) __bf16 win[(ROWS + 2) * WIN_X * LDS_PIX];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int y0 = blockIdx.y * ROWS, x0 = blockIdx.x * 64, b = blockIdx.z;
    stage_nhwc32<ROWS>(a5, win, b, y0, x0, H, W);
    floatx4 acc[4];
#pragma unroll
    for (int mb = 0; mb < 4; mb++) acc[mb] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < TAPS; t++) {
        const int dy = t / 3 - 1, dx = t % 3 - 1;
        const bf16x8 w = frag[t * 64 + lane];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) {
            const bf16x8 a = *(const bf16x8 *)(win + ((wave + 1 + dy) * WIN_X + 1 + mb * 16 + m + dx) * LDS_PIX + kg * 8);
            acc[mb] = mfma(w, a, acc[mb]);
        }
    }
    if (kg == 0) {
        const float bv = b6[0];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) out[((long)b * H + y0 + wave) * W + x0 + mb * 16 + m] = acc[mb][0] + bv;
    }
}

// The 32-channel-input layers (k_conv32 forward, k_conv_out) as a march down a
// run of run_rows rows of one 64-pixel band (inference): the workgroup keeps
// the ROWS + 2 input rows of the current block of ROWS output rows in an LDS
// ring (row y in slot (y + 1) % (ROWS + 2)) and, while the matrix cores work
// on that block, has the next block's ROWS new rows in flight into registers;
// they replace the rows no later block needs once every wave is done.  So
// each input row is read once per run (a window per block re-reads 2 of every
// ROWS + 2), and the loads of a block overlap the products of the one before.
// The operands and their order are those of the windowed kernels, so the
// values are the same.  Grid (W/64, H/run_rows, B); run_rows a multiple of ROWS.
template <int ROWS> struct MarchRing {
    static constexpr int NR = ROWS + 2;
    static constexpr int PIECES = WIN_X * 4;                    // 16-byte pieces per staged row
    static constexpr int NEW = ROWS * PIECES;                   // pieces per block of new rows
    static constexpr int PER = (NEW + ROWS * 64 - 1) / (ROWS * 64);
    __bf16 *win;
    const __bf16 *in;
    int b, x0, H, W;
    __device__ __forceinline__ static int slot(int y) { return (y + 1) % NR; }
    __device__ __forceinline__ const bf16x8 *src(int y, int px, int q) const
    {
        return (const bf16x8 *)(in + padded(b, y, x0 - 1 + px, H, W) * CH + q * 8);
    }
    __device__ __forceinline__ bf16x8 *dst(int y, int px, int q) const
    {
        return (bf16x8 *)(win + (slot(y) * WIN_X + px) * LDS_PIX + q * 8);
    }
    // rows y_first .. y_first + n - 1 straight into the ring
    __device__ __forceinline__ void stage(int y_first, int n) const
    {
        for (int c = threadIdx.x; c < n * PIECES; c += ROWS * 64) {
            const int r = c / PIECES, rem = c - r * PIECES;
            *dst(y_first + r, rem >> 2, rem & 3) = *src(y_first + r, rem >> 2, rem & 3);
        }
    }
    __device__ __forceinline__ void prefetch(bf16x8 (&pf)[PER], int y_first) const
    {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = threadIdx.x + j * ROWS * 64;
            if (c < NEW) {
                const int r = c / PIECES, rem = c - r * PIECES;
                pf[j] = *src(y_first + r, rem >> 2, rem & 3);
            }
        }
    }
    __device__ __forceinline__ void commit(const bf16x8 (&pf)[PER], int y_first) const
    {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = threadIdx.x + j * ROWS * 64;
            if (c < NEW) {
                const int r = c / PIECES, rem = c - r * PIECES;
                *dst(y_first + r, rem >> 2, rem & 3) = pf[j];
            }
        }
    }
    // input row y, pixel x0 + px (px = -1 .. 64), this lane's 8 channels
    __device__ __forceinline__ bf16x8 at(int y, int px, int kg) const
    {
        return *(const bf16x8 *)(win + (slot(y) * WIN_X + 1 + px) * LDS_PIX + kg * 8);
    }
};

// body(ring, y0): the products and stores of the block of output rows y0 .. y0+ROWS-1
template <int ROWS, typename Body>
__device__ __forceinline__ void conv_march(const __bf16 *__restrict__ in, __bf16 *win, int H, int W, int run_rows,
                                           Body body)
{
    using Ring = MarchRing<ROWS>;
    const Ring ring{win, in, (int)blockIdx.z, (int)blockIdx.x * 64, H, W};
    const int ya = blockIdx.y * run_rows, yb = ya + run_rows < H ? ya + run_rows : H;
    ring.stage(ya - 1, ROWS + 2);
    bf16x8 pf[Ring::PER];
    for (int y0 = ya; y0 < yb; y0 += ROWS) {
        const bool more = y0 + ROWS < yb;
        if (more) ring.prefetch(pf, y0 + ROWS + 1);   // the next block's new rows
        __syncthreads();                              // rows y0-1 .. y0+ROWS in the ring
        body(ring, y0);
        __syncthreads();                              // rows y0-1 .. y0+ROWS-2 no longer read
        if (more) ring.commit(pf, y0 + ROWS + 1);
    }
}

// The weight fragments and biases are read once per workgroup, into LDS and
// registers: a global read inside the march would wait for the next block's
// rows in flight before it (the memory counter completes in order).
template <int ROWS>
__global__ __launch_bounds__(ROWS * 64) void k_conv32_march(const __bf16 *__restrict__ in, __bf16 *__restrict__ out,
                                                            const bf16x8 *__restrict__ frag,
                                                            const float *__restrict__ bias, int H, int W, int run_rows)
{
    __shared__ __attribute__((aligned(16))) __bf16 win[(ROWS + 2) * WIN_X * LDS_PIX];
    __shared__ bf16x8 wsh[TAPS * 2 * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    for (int i = threadIdx.x; i < TAPS * 2 * 64; i += ROWS * 64) wsh[i] = frag[i];
    float bv[2][4];
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int i = 0; i < 4; i++) bv[nb][i] = bias[nb * 16 + kg * 4 + i];
    conv_march<ROWS>(in, win, H, W, run_rows, [&](const MarchRing<ROWS> &ring, int y0) {
        floatx4 acc[4][2];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) acc[mb][0] = acc[mb][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < TAPS; t++) {
            const int dy = t / 3 - 1, dx = t % 3 - 1;
            const bf16x8 w0 = wsh[(t * 2 + 0) * 64 + lane];
            const bf16x8 w1 = wsh[(t * 2 + 1) * 64 + lane];
#pragma unroll
            for (int mb = 0; mb < 4; mb++) {
                const bf16x8 a = ring.at(y0 + wave + dy, mb * 16 + m + dx, kg);
                acc[mb][0] = mfma(w0, a, acc[mb][0]);
                acc[mb][1] = mfma(w1, a, acc[mb][1]);
            }
        }
        // store_nhwc32's forward expression with the biases held in registers
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int nb = 0; nb < 2; nb++) {
                const long idx = padded(ring.b, y0 + wave, ring.x0 + mb * 16 + m, H, W) * CH + nb * 16 + kg * 4;
                bf16x4 o;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = (__bf16)fmaxf(acc[mb][nb][i] + bv[nb][i], 0.0f);
                *(bf16x4 *)(out + idx) = o;
            }
    });
}

// Layers 1 and 2 in one march (inference, one image): the rows of layer 1's
// output that layer 2's window needs are formed in the LDS ring from the
// feature planes as the march reaches them (k_conv_first's operands and
// expressions, zero outside the image as its padded output holds), instead
// of being stored and read back: 12 bytes per pixel read instead of
// 12 + 64 written + 64 read.  Layer 1 covers 80 pixels (five 16-pixel
// blocks from x0 - 8) of which the ring keeps x0 - 1 .. x0 + 64.  The next
// block's feature rows are in flight into registers while layer 2 works.
// The same values as k_conv_first followed by k_conv32.
template <int ROWS> struct FirstRows {
    static constexpr int FX = 82;                       // feature columns x0 - 9 .. x0 + 72
    static constexpr int FY = ROWS + 2;                 // feature rows of ROWS layer-1 rows
    static constexpr int N = NFEAT * FY * FX;
    static constexpr int PER = (N + ROWS * 64 - 1) / (ROWS * 64);
    const float *pl;
    int H, W, x0;
    // feature f at row y, column x0 - 9 + px (zero outside the image)
    __device__ __forceinline__ float load(int c, int y_first) const
    {
        const int f = c / (FY * FX), rem = c - f * (FY * FX), r = rem / FX, px = rem - r * FX;
        const int y = y_first - 1 + r, x = x0 - 9 + px;
        return (y >= 0 && y < H && x >= 0 && x < W) ? pl[(long)f * H * W + (long)y * W + x] : 0.0f;
    }
    __device__ __forceinline__ void prefetch(float (&pf)[PER], int y_first) const
    {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = threadIdx.x + j * ROWS * 64;
            if (c < N) pf[j] = load(c, y_first);
        }
    }
    __device__ __forceinline__ void commit(float *fb, const float (&pf)[PER]) const
    {
#pragma unroll
        for (int j = 0; j < PER; j++) {
            const int c = threadIdx.x + j * ROWS * 64;
            if (c < N) fb[c] = pf[j];
        }
    }
};

template <int ROWS>
__global__ __launch_bounds__(ROWS * 64) void k_first_conv32_march(const float *__restrict__ planes, int npl,
                                                                  __bf16 *__restrict__ out,
                                                                  const bf16x8 *__restrict__ frag1,
                                                                  const float *__restrict__ bias1,
                                                                  const bf16x8 *__restrict__ frag2,
                                                                  const float *__restrict__ bias2, int H, int W,
                                                                  int run_rows)
{
    using FR = FirstRows<ROWS>;
    __shared__ __attribute__((aligned(16))) __bf16 win[(ROWS + 2) * WIN_X * LDS_PIX];
    __shared__ float fb[FR::N];
    __shared__ bf16x8 wsh1[2 * 64], wsh2[TAPS * 2 * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    const int x0 = blockIdx.x * 64, b = blockIdx.z;
    const FR fr{planes + (long)b * npl * H * W, H, W, x0};
    const MarchRing<ROWS> ring{win, nullptr, b, x0, H, W};
    for (int i = threadIdx.x; i < TAPS * 2 * 64; i += ROWS * 64) wsh2[i] = frag2[i];
    for (int i = threadIdx.x; i < 2 * 64; i += ROWS * 64) wsh1[i] = frag1[i];
    float bv1[2][4], bv2[2][4];
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            bv1[nb][i] = bias1[nb * 16 + kg * 4 + i];
            bv2[nb][i] = bias2[nb * 16 + kg * 4 + i];
        }
    // this lane's 8 im2col K-values: offsets into fb relative to the pixel (k_conv_first's)
    int off[8];
    bool real[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int k = kg * 8 + i, t = k / 3, f = k - 3 * t;
        real[i] = k < K1;
        off[i] = real[i] ? (f * FR::FY + (t / 3 - 1)) * FR::FX + (t % 3 - 1) : 0;
    }
    // layer-1 rows y_first .. y_first + n - 1 (wave w: row y_first + w) into the ring from the
    // features in fb (rows y_first - 1 .. y_first + n)
    auto form = [&](int y_first, int n) {
        if (wave >= n) return;
        const int y = y_first + wave;
        const bool row_in = y >= 0 && y < H;
        const float *base = fb + (wave + 1) * FR::FX + 9;   // pixel x0 + 0 of row y
        const bf16x8 w0 = wsh1[lane], w1 = wsh1[64 + lane];
#pragma unroll
        for (int mb = 0; mb < 5; mb++) {
            const int px = mb * 16 + m - 8;   // relative to x0
            bf16x8 a;
#pragma unroll
            for (int i = 0; i < 8; i++) a[i] = (__bf16)(real[i] ? base[px + off[i]] : 0.0f);
            const floatx4 z = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            const floatx4 acc[2] = {mfma(w0, a, z), mfma(w1, a, z)};
            if (px >= -1 && px <= 64) {
                const bool in = row_in && x0 + px >= 0 && x0 + px < W;
#pragma unroll
                for (int nb = 0; nb < 2; nb++) {
                    bf16x4 o;
#pragma unroll
                    for (int i = 0; i < 4; i++) o[i] = in ? (__bf16)fmaxf(acc[nb][i] + bv1[nb][i], 0.0f) : (__bf16)0.0f;
                    *(bf16x4 *)(win + (MarchRing<ROWS>::slot(y) * WIN_X + 1 + px) * LDS_PIX + nb * 16 + kg * 4) = o;
                }
            }
        }
    };
    const int ya = blockIdx.y * run_rows, yb = ya + run_rows < H ? ya + run_rows : H;
    float pf[FR::PER];
    // prologue: layer-1 rows ya - 1 .. ya + ROWS
    fr.prefetch(pf, ya - 1);
    fr.commit(fb, pf);
    __syncthreads();
    form(ya - 1, ROWS);
    __syncthreads();
    fr.prefetch(pf, ya - 1 + ROWS);
    fr.commit(fb, pf);
    __syncthreads();
    form(ya - 1 + ROWS, 2);
    for (int y0 = ya; y0 < yb; y0 += ROWS) {
        const bool more = y0 + ROWS < yb;
        if (more) fr.prefetch(pf, y0 + ROWS + 1);   // features of the next block's layer-1 rows
        __syncthreads();                            // layer-1 rows y0-1 .. y0+ROWS in the ring
        floatx4 acc[4][2];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) acc[mb][0] = acc[mb][1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < TAPS; t++) {
            const int dy = t / 3 - 1, dx = t % 3 - 1;
            const bf16x8 w0 = wsh2[(t * 2 + 0) * 64 + lane];
            const bf16x8 w1 = wsh2[(t * 2 + 1) * 64 + lane];
#pragma unroll
            for (int mb = 0; mb < 4; mb++) {
                const bf16x8 a = ring.at(y0 + wave + dy, mb * 16 + m + dx, kg);
                acc[mb][0] = mfma(w0, a, acc[mb][0]);
                acc[mb][1] = mfma(w1, a, acc[mb][1]);
            }
        }
#pragma unroll
        for (int mb = 0; mb < 4; mb++)
#pragma unroll
            for (int nb = 0; nb < 2; nb++) {
                const long idx = padded(b, y0 + wave, x0 + mb * 16 + m, H, W) * CH + nb * 16 + kg * 4;
                bf16x4 o;
#pragma unroll
                for (int i = 0; i < 4; i++) o[i] = (__bf16)fmaxf(acc[mb][nb][i] + bv2[nb][i], 0.0f);
                *(bf16x4 *)(out + idx) = o;
            }
        __syncthreads();   // layer-1 rows y0-1 .. y0+ROWS-2 and the features no longer read
        if (more) {
            fr.commit(fb, pf);
            __syncthreads();
            form(y0 + ROWS + 1, ROWS);
        }
    }
}

template <int ROWS>
__global__ __launch_bounds__(ROWS * 64) void k_conv_out_march(const __bf16 *__restrict__ a5,
                                                              const bf16x8 *__restrict__ frag,
                                                              const float *__restrict__ b6, float *__restrict__ out,
                                                              int H, int W, int run_rows)
{
    __shared__ __attribute__((aligned(16))) __bf16 win[(ROWS + 2) * WIN_X * LDS_PIX];
    __shared__ bf16x8 wsh[TAPS * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4;
    for (int i = threadIdx.x; i < TAPS * 64; i += ROWS * 64) wsh[i] = frag[i];
    const float bv = b6[0];
    conv_march<ROWS>(a5, win, H, W, run_rows, [&](const MarchRing<ROWS> &ring, int y0) {
        floatx4 acc[4];
#pragma unroll
        for (int mb = 0; mb < 4; mb++) acc[mb] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < TAPS; t++) {
            const int dy = t / 3 - 1, dx = t % 3 - 1;
            const bf16x8 w = wsh[t * 64 + lane];
#pragma unroll
            for (int mb = 0; mb < 4; mb++) acc[mb] = mfma(w, ring.at(y0 + wave + dy, mb * 16 + m + dx, kg), acc[mb]);
        }
        if (kg == 0) {
#pragma unroll
            for (int mb = 0; mb < 4; mb++)
                out[((long)ring.b * H + y0 + wave) * W + ring.x0 + mb * 16 + m] = acc[mb][0] + bv;
        }
    });
}

// ---------------------------------------------------------------- loss and backward

// Loss over the cells M at least `margin` from the crop edge, e = out - target:
//   MSE:    sum_M e^2 / |M|,            g6 = 2 e / |M|
//   energy: sum_M e (A_M e) / |M|,      g6 = 2 (A_M e) / |M|
// where A_M e = e + sum over the faces between two cells of M of
// k_face (e_i - e_j), k_face = Kx (left face, plane 4) or Ky (bottom face,
// plane 5): the error's squared norm in the timestep operator I - dt div K grad,
// restricted to M.  One FP64 partial sum per workgroup.
__device__ __forceinline__ float err_at(const float *out, const float *tgt, long p, long q) { return out[p] - tgt[q]; }

__global__ __launch_bounds__(BLOCK) void k_loss(const float *__restrict__ out, const float *__restrict__ samples,
                                                float *__restrict__ g6, double *__restrict__ part, int B, int H,
                                                int W, int margin, float scale, int energy)
{
    __shared__ double lds[BLOCK / 64];
    const long p = (long)blockIdx.x * BLOCK + threadIdx.x;
    double s = 0.0;
    if (p < (long)B * H * W) {
        const int x = (int)(p % W), y = (int)((p / W) % H), b = (int)(p / ((long)W * H));
        const bool in = x >= margin && x < W - margin && y >= margin && y < H - margin;
        const long hw = (long)H * W, q = (long)y * W + x;
        const float *smp = samples + (long)b * NPLANES * hw;
        const float *tgt = smp + 3 * hw;
        const float *pout = out + (long)b * hw;
        const float e = pout[q] - tgt[q];
        float ae = e;
        if (energy && in) {
            const float *kx = smp + 4 * hw, *ky = smp + 5 * hw;
            if (x - 1 >= margin) ae += kx[q] * (e - err_at(pout, tgt, q - 1, q - 1));
            if (x + 1 < W - margin) ae += kx[q + 1] * (e - err_at(pout, tgt, q + 1, q + 1));
            if (y - 1 >= margin) ae += ky[q] * (e - err_at(pout, tgt, q - W, q - W));
            if (y + 1 < H - margin) ae += ky[q + W] * (e - err_at(pout, tgt, q + W, q + W));
        }
        g6[padded(b, y, x, H, W)] = in ? scale * ae : 0.0f;
        if (in) s = (double)e * ae;
    }
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = lds[0] + lds[1] + lds[2] + lds[3];
}

// Layer 6 backward to its input: g5 = bf16(relu'(a5) * sum_tap g6[p - tap] W6[tap]).
__global__ void k_out_bwd(const float *__restrict__ g6, const float *__restrict__ w6, const __bf16 *__restrict__ a5,
                          __bf16 *__restrict__ g5, int B, int H, int W)
{
    const long p = (long)blockIdx.x * BLOCK + threadIdx.x;
    if (p >= (long)B * H * W) return;
    const int x = (int)(p % W), y = (int)((p / W) % H), b = (int)(p / ((long)W * H));
    float s[CH];
#pragma unroll
    for (int c = 0; c < CH; c++) s[c] = 0.0f;
    for (int t = 0; t < TAPS; t++) {
        const float g = g6[padded(b, y - (t / 3 - 1), x - (t % 3 - 1), H, W)];
#pragma unroll
        for (int c = 0; c < CH; c++) s[c] += g * w6[t * CH + c];
    }
    const long base = padded(b, y, x, H, W) * CH;
    const bf16x8 *am = (const bf16x8 *)(a5 + base);
    bf16x8 *dst = (bf16x8 *)(g5 + base);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const bf16x8 a = am[q];
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = (__bf16)((float)a[i] > 0.0f ? s[q * 8 + i] : 0.0f);
        dst[q] = v;
    }
}

// Workgroups of a weight-gradient reduction: each sums its share of the pixels
// in registers and writes one partial, which k_sum_parts adds in a fixed order.
// 512 (two per compute unit) keeps the partials at 19 MB per layer.
constexpr int WG_PARTS = 512;

// Layer 6 weight and bias gradients, dW6[tap][ci] = sum_p a5[p + tap][ci] g6[p]
// and db6 = sum_p g6[p].
//
// The weights are summed over the input pixels q = p + tap (a5 and g6 are zero
// on the border).  One product per 72 loaded values, so that part is bound by
// reading a5 once: a lane holds 8 channels of one pixel column (one 16-byte load
// per pixel), marches down a run of rows and keeps the 3x3 window of g6 and the
// 72 sums in registers; 4 lanes cover a pixel, a wave 16 columns.  32 x 128 x 128
// pixels: 1060 us with one thread per weight walking every pixel, 20 us here (29
// with the bias).  tasks: (image, 16 columns, run of rows).
//
// Under the energy loss g6 is made of fluxes that cancel in db6 (the sum of
// |g6| is 13 to 7000 times |db6| over 40 batches of 32 x 128 x 128), so the order
// of its FP32 sum shows in db6, and the order is fixed: BIAS_RUNS runs of
// consecutive pixels, each summed first pixel to last, then the runs' sums first
// to last (k_sum_runs).
// One wave per run, in the workgroups after the first `wparts`, beside the others'
// reads of a5: it loads 64 pixels side by side and adds them one by one out of its
// lanes.  Bound by that chain (35 us with one such load under way instead of eight).
constexpr int BIAS_RUNS = 256;

// s + v of lane 0 + v of lane 1 + ... of the first n lanes, in that order
__device__ __forceinline__ float add_in_order(float s, float v, int n)
{
    if (n == 64) {
#pragma unroll
        for (int k = 0; k < 64; k++) s += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
    } else {
        for (int k = 0; k < n; k++) s += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k));
    }
    return s;
}

__global__ __launch_bounds__(BLOCK) void k_out_wgrad(const __bf16 *__restrict__ a5, const float *__restrict__ g6,
                                                     float *__restrict__ part, float *__restrict__ runs, int B, int H,
                                                     int W, int rows, int nruns, long tasks, int wparts)
{
    constexpr int NOUT = TAPS * CH, NW = BLOCK / 64, AHEAD = 8;
    __shared__ float lds[NW][NOUT];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if ((int)blockIdx.x >= wparts) {
        const int c = ((int)blockIdx.x - wparts) * NW + wave;
        if (c >= BIAS_RUNS) return;
        // (pixels are counted in 32 bits: 2^31 of them would be 137 GB per layer)
        const long n = (long)B * H * W;
        const unsigned p1 = (unsigned)(n * (c + 1) / BIAS_RUNS);
        auto pixel = [&](unsigned p) {
            if (p >= p1) return 0.0f;
            const unsigned row = p / (unsigned)W, b = row / (unsigned)H;
            return g6[padded((int)b, (int)(row - b * H), (int)(p - row * W), H, W)];
        };
        unsigned p = (unsigned)(n * c / BIAS_RUNS);
        float s = 0.0f, next[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; u++) next[u] = pixel(p + u * 64 + lane);
        for (; p < p1; p += AHEAD * 64) {
            float v[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; u++) {
                v[u] = next[u];
                next[u] = pixel(p + (AHEAD + u) * 64 + lane);   // under way while these are added
            }
#pragma unroll
            for (int u = 0; u < AHEAD; u++) s = add_in_order(s, v[u], (int)min(64l, max(0l, (long)p1 - p - u * 64)));
        }
        if (lane == 0) runs[c] = s;
        return;
    }
    const int q = lane & 3, px = lane >> 2;
    const int cols = W / 16;
    float acc[TAPS][8];
#pragma unroll
    for (int t = 0; t < TAPS; t++)
#pragma unroll
        for (int i = 0; i < 8; i++) acc[t][i] = 0.0f;
    for (long task = (long)blockIdx.x * NW + wave; task < tasks; task += (long)wparts * NW) {
        const int run = (int)(task % nruns);
        const int xg = (int)((task / nruns) % cols), b = (int)(task / nruns / cols);
        const int x = xg * 16 + px, y0 = run * rows, y1 = min(y0 + rows, H);
        // gw[k][j] = g6 at row y - 1 + k, column x - 1 + j
        float gw[3][3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            gw[1][j] = g6[padded(b, y0 - 1, x - 1 + j, H, W)];
            gw[2][j] = g6[padded(b, y0, x - 1 + j, H, W)];
        }
        for (int y = y0; y < y1; y++) {
#pragma unroll
            for (int j = 0; j < 3; j++) {
                gw[0][j] = gw[1][j];
                gw[1][j] = gw[2][j];
                gw[2][j] = g6[padded(b, y + 1, x - 1 + j, H, W)];
            }
            const bf16x8 a = *(const bf16x8 *)(a5 + padded(b, y, x, H, W) * CH + q * 8);
#pragma unroll
            for (int t = 0; t < TAPS; t++) {
                const float g = gw[2 - t / 3][2 - t % 3];   // g6 at p = q - tap
#pragma unroll
                for (int i = 0; i < 8; i++) acc[t][i] += (float)a[i] * g;
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 4; off >>= 1) {
#pragma unroll
        for (int t = 0; t < TAPS; t++)
#pragma unroll
            for (int i = 0; i < 8; i++) acc[t][i] += __shfl_xor(acc[t][i], off, 64);
    }
    if (px == 0) {
#pragma unroll
        for (int t = 0; t < TAPS; t++)
#pragma unroll
            for (int i = 0; i < 8; i++) lds[wave][t * CH + q * 8 + i] = acc[t][i];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NOUT; e += BLOCK)
        part[(long)blockIdx.x * NOUT + e] = (lds[0][e] + lds[1][e]) + (lds[2][e] + lds[3][e]);
}

// db6 from the runs' sums, in order.
__global__ __launch_bounds__(64) void k_sum_runs(const float *__restrict__ runs, float *__restrict__ dst)
{
    float s = 0.0f, v[BIAS_RUNS / 64];
#pragma unroll
    for (int k = 0; k < BIAS_RUNS / 64; k++) v[k] = runs[k * 64 + threadIdx.x];
#pragma unroll
    for (int k = 0; k < BIAS_RUNS / 64; k++) s = add_in_order(s, v[k], 64);
    if (threadIdx.x == 0) *dst = s;
}

// Weight and bias gradients of a 32-channel layer: dW[tap][ci][co] =
// sum_q in[q][ci] g[q - tap][co] over the input pixels q (both images are zero
// on the border) and db[co] = sum_p g[p][co], as products with K = 32 pixels of
// a row on the matrix cores.  Both operands need 8 consecutive pixels of one
// channel per lane, across the images' layout, so rows are turned on their way
// into LDS ([channel][pixel], pixels in pairs: one 4-byte store per two) and
// each staged row serves all nine taps: `in` rows meet a ring of g rows, and the
// left and right taps come from the centre fragment by funnel shifts.  A
// workgroup marches down a run of rows of a 64-pixel band, two rows per step;
// wave (cb, nb) owns one 16 x 16 block of every tap, so no sums cross waves,
// and the bias is a tenth product with a row of ones.  Reading the two images
// once is the floor (13 us at 32 x 128 x 128); one workgroup per tap gathering
// 2-byte values took 82 us and the bias alone 132 us, this takes 29 us for both.
// NTAP = 1: the im2col image of layer 1 (27 of 32 rows kept, centre tap only).
constexpr int WGR_IN = 36, WGR_G = 44;   // 4-byte words per channel row: 16-byte aligned rows, spread over the banks
constexpr int WGR_G0 = 8;                // index of the band's first pixel in a g row
template <int NTAP>
__global__ __launch_bounds__(BLOCK) void k_wgrad32(const __bf16 *__restrict__ in, const __bf16 *__restrict__ g,
                                                   float *__restrict__ part, int H, int W, int rows, int nruns,
                                                   long tasks)
{
    constexpr int NIN = NTAP == 1 ? K1 : CH, NPART = NTAP * NIN * CH + CH;
    constexpr int RING = 4;   // g rows y - 1 .. y + 2 of a step
    __shared__ __attribute__((aligned(16))) unsigned int tin[2][CH * WGR_IN];
    __shared__ __attribute__((aligned(16))) unsigned int tg[RING][CH * WGR_G];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kg = lane >> 4, cb = wave >> 1, nb = wave & 1;
    const int bands = W / 64;
    // two pixels x 8 channels of a row, px and px + 1 (each inside the padded
    // row or zero), to word `word` of the 8 channel rows
    auto turn = [&](const __bf16 *img, int b, int y, int x0, int px, int lo, int hi, int q8, unsigned int *dst,
                    int stride, int word) {
        uintx4 v[2];   // channels 2j, 2j + 1 of a pixel in word j
#pragma unroll
        for (int k = 0; k < 2; k++) {
            v[k] = uintx4{0, 0, 0, 0};
            if (px + k >= lo && px + k <= hi && y <= H)
                v[k] = *(const uintx4 *)(img + padded(b, y, x0 + px + k, H, W) * CH + q8 * 8);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            dst[(q8 * 8 + 2 * j) * stride + word] = (v[0][j] & 0xffffu) | (v[1][j] << 16);
            dst[(q8 * 8 + 2 * j + 1) * stride + word] = (v[0][j] >> 16) | (v[1][j] & 0xffff0000u);
        }
    };
    auto stage_in = [&](int b, int y, int x0, unsigned int *dst, int t0) {
        for (int e = t0; e < 32 * 4; e += BLOCK / 2) turn(in, b, y, x0, (e >> 2) * 2, 0, 63, e & 3, dst, WGR_IN, e >> 2);
    };
    auto stage_g = [&](int b, int y, int x0, unsigned int *dst, int t0) {   // pixels -1 .. 64
        for (int e = t0; e < 34 * 4; e += BLOCK / 2)
            turn(g, b, y, x0, (e >> 2) * 2 - 2, -1, 64, e & 3, dst, WGR_G, WGR_G0 / 2 - 1 + (e >> 2));
    };
    floatx4 acc[NTAP], accb = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < NTAP; t++) acc[t] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = (__bf16)1.0f;
    const int half = threadIdx.x / (BLOCK / 2), t0 = threadIdx.x % (BLOCK / 2);
    for (long task = blockIdx.x; task < tasks; task += gridDim.x) {
        const int run = (int)(task % nruns);
        const int band = (int)((task / nruns) % bands), b = (int)(task / nruns / bands);
        const int x0 = band * 64, y0 = run * rows, y1 = min(y0 + rows, H);
        __syncthreads();   // the last task's reads are done
        if (NTAP > 1) stage_g(b, y0 - 1 + half, x0, tg[(y0 - 1 + half + RING) % RING], t0);
        for (int y = y0; y < y1; y += 2) {
            stage_in(b, y + half, x0, tin[half], t0);
            const int yg = NTAP > 1 ? y + 1 + half : y + half;
            stage_g(b, yg, x0, tg[yg % RING], t0);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < 2; k++) {
                if (y + k >= y1) continue;
#pragma unroll
                for (int grp = 0; grp < 2; grp++) {
                    const int px = grp * 32 + kg * 8;
                    const bf16x8 av =
                        __builtin_bit_cast(bf16x8, *(const uintx4 *)&tin[k][(cb * 16 + m) * WGR_IN + px / 2]);
#pragma unroll
                    for (int dy = NTAP > 1 ? -1 : 0; dy <= (NTAP > 1 ? 1 : 0); dy++) {
                        // tap row dy + 1 meets g row y - dy
                        const unsigned int *gr =
                            &tg[(y + k - dy + RING) % RING][(nb * 16 + m) * WGR_G + (WGR_G0 + px) / 2];
                        const uintx4 w = *(const uintx4 *)gr;
                        const bf16x8 gc = __builtin_bit_cast(bf16x8, w);
                        if (NTAP == 1) {
                            acc[0] = mfma(av, gc, acc[0]);
                        } else {
                            // dx = 1 takes g one pixel to the left, dx = -1 one to the right
                            const unsigned int wl = gr[-1], wr = gr[4];
                            uintx4 l, r;
                            l[0] = __builtin_amdgcn_alignbit(w[0], wl, 16);
                            l[1] = __builtin_amdgcn_alignbit(w[1], w[0], 16);
                            l[2] = __builtin_amdgcn_alignbit(w[2], w[1], 16);
                            l[3] = __builtin_amdgcn_alignbit(w[3], w[2], 16);
                            r[0] = l[1];
                            r[1] = l[2];
                            r[2] = l[3];
                            r[3] = __builtin_amdgcn_alignbit(wr, w[3], 16);
                            const int t = (dy + 1) * 3;
                            acc[t % NTAP] = mfma(av, __builtin_bit_cast(bf16x8, r), acc[t % NTAP]);
                            acc[(t + 1) % NTAP] = mfma(av, gc, acc[(t + 1) % NTAP]);
                            acc[(t + 2) % NTAP] = mfma(av, __builtin_bit_cast(bf16x8, l), acc[(t + 2) % NTAP]);
                        }
                        if (dy == 0 && cb == 0) accb = mfma(ones, gc, accb);
                    }
                }
            }
            __syncthreads();
        }
    }
    float *dst = part + (long)blockIdx.x * NPART;
#pragma unroll
    for (int t = 0; t < NTAP; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int ci = cb * 16 + kg * 4 + i;
            if (ci < NIN) dst[(t * NIN + ci) * CH + nb * 16 + m] = acc[t][i];
        }
    if (cb == 0 && kg == 0) dst[NTAP * NIN * CH + nb * 16 + m] = accb[0];
}

// dst[e] = sum_c part[c*n + e], e < n (fixed order): 32 consecutive e per
// workgroup, every 8th partial per thread, then the 8 sums in order.  Bound by
// reading the partials; one thread walking all of them took 58 us for 256 x
// 9216 values, this takes 5 us for 512 x 9248.
__global__ __launch_bounds__(BLOCK) void k_sum_parts(const float *__restrict__ part, int chunks, int n,
                                                     float *__restrict__ dst)
{
    __shared__ float lds[BLOCK / 32][32];
    const int k = threadIdx.x & 31, sub = threadIdx.x >> 5, e = blockIdx.x * 32 + k;
    float s = 0.0f;
    if (e < n) {
#pragma unroll 8
        for (int c = sub; c < chunks; c += BLOCK / 32) s += part[(long)c * n + e];
    }
    lds[sub][k] = s;
    __syncthreads();
    if (sub == 0 && e < n) {
        for (int j = 1; j < BLOCK / 32; j++) s += lds[j][k];
        dst[e] = s;
    }
}

// Adam (Kingma and Ba, 2015) on the FP32 master parameters.
__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int e = blockIdx.x * BLOCK + threadIdx.x;
    if (e >= n) return;
    const float ge = g[e];
    const float me = b1 * m[e] + (1.0f - b1) * ge;
    const float ve = b2 * v[e] + (1.0f - b2) * ge * ge;
    m[e] = me;
    v[e] = ve;
    p[e] -= lr * (me / c1) / (sqrtf(ve / c2) + eps);
}

// Training samples from dense FP64 interior fields (row-major ny x nx):
// sample k = crop of size `crop` at origins[2k], origins[2k+1] (x, y), planes
//   0: (log10 rho - 0.5) / 1.5
//   1: (u0 - u_prev) / s
//   2: u0 / s_u
//   3: target ((u_next - u0) - c0 (u0 - u_prev) - c1 (u_prev - u_prev2)) / s
//   4, 5: Kx (left face), Ky (bottom face) of the timestep operator
__global__ void k_make_samples(const double *__restrict__ rho, const double *__restrict__ u_prev2,
                               const double *__restrict__ u_prev, const double *__restrict__ u0,
                               const double *__restrict__ u_next, const double *__restrict__ kx,
                               const double *__restrict__ ky, int nx, int ny, double c0, double c1, double inv_s,
                               double inv_su, const int *__restrict__ origins, int n, int crop,
                               float *__restrict__ out)
{
    const long p = (long)blockIdx.x * BLOCK + threadIdx.x;
    const long per = (long)crop * crop;
    if (p >= per * n) return;
    const int k = (int)(p / per);
    const int cy = (int)((p % per) / crop), cx = (int)(p % crop);
    const int ox = origins[2 * k], oy = origins[2 * k + 1];
    const int x = ox + cx, y = oy + cy;
    float *o = out + (long)k * NPLANES * per + (long)cy * crop + cx;
    if (x < 0 || x >= nx || y < 0 || y >= ny) {
        for (int q = 0; q < NPLANES; q++) o[q * per] = 0.0f;
        return;
    }
    const long i = (long)y * nx + x;
    const double dprev = u0[i] - u_prev[i];
    o[0] = (float)((log10(rho[i]) - 0.5) / 1.5);
    o[per] = (float)(dprev * inv_s);
    o[2 * per] = (float)(u0[i] * inv_su);
    o[3 * per] = (float)(((u_next[i] - u0[i]) - c0 * dprev - c1 * (u_prev[i] - u_prev2[i])) * inv_s);
    o[4 * per] = (float)kx[i];
    o[5 * per] = (float)ky[i];
}

// sums of (u0 - u_prev)^2 and u0^2 over dense fields, one FP64 pair per workgroup
__global__ __launch_bounds__(BLOCK) void k_scales(const double *__restrict__ u_prev, const double *__restrict__ u0,
                                                  long n, double *__restrict__ part)
{
    __shared__ double lds[2][BLOCK / 64];
    double a = 0.0, c = 0.0;
    for (long i = (long)blockIdx.x * BLOCK + threadIdx.x; i < n; i += (long)gridDim.x * BLOCK) {
        const double d = u0[i] - u_prev[i];
        a += d * d;
        c += u0[i] * u0[i];
    }
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off, 64);
        c += __shfl_xor(c, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        lds[0][threadIdx.x >> 6] = a;
        lds[1][threadIdx.x >> 6] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = lds[0][0] + lds[0][1] + lds[0][2] + lds[0][3];
        part[2 * blockIdx.x + 1] = lds[1][0] + lds[1][1] + lds[1][2] + lds[1][3];
    }
}

// ---------------------------------------------------------------- host side

static unsigned nblocks(long n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }

hipError_t net_alloc(Net &net)
{
    hipError_t e;
    if ((e = hipMalloc(&net.params, NPARAM * sizeof(float))) != hipSuccess) return e;
    if ((e = hipMalloc(&net.packed, PK_TOTAL * sizeof(__bf16))) != hipSuccess) return e;
    return hipMalloc(&net.w6, TAPS * CH * sizeof(float));
}

void net_free(Net &net)
{
    if (net.params) (void)hipFree(net.params);
    if (net.packed) (void)hipFree(net.packed);
    if (net.w6) (void)hipFree(net.w6);
    net = Net();
}

void net_pack(const Net &net, hipStream_t stream)
{
    hipLaunchKernelGGL(k_pack, dim3(nblocks(PK_TOTAL)), dim3(BLOCK), 0, stream, net.params, net.packed, net.w6);
}

hipError_t net_upload(Net &net, const float *host_params, hipStream_t stream)
{
    hipError_t e = hipMemcpyAsync(net.params, host_params, NPARAM * sizeof(float), hipMemcpyHostToDevice, stream);
    if (e != hipSuccess) return e;
    net_pack(net, stream);
    return hipStreamSynchronize(stream);
}

hipError_t acts_alloc(Acts &a, int B, int H, int W, bool training)
{
    a.B = B;
    a.H = H;
    a.W = W;
    const size_t bytes = act_bytes(B, H, W);
    const int distinct = training ? 5 : 2;
    hipError_t e;
    if (training) {   // the im2col image is only needed for layer 1's weight gradient
        if ((e = hipMalloc(&a.x1, bytes)) != hipSuccess) return e;
        if ((e = hipMemset(a.x1, 0, bytes)) != hipSuccess) return e;
    }
    for (int l = 1; l <= distinct; l++) {
        if ((e = hipMalloc(&a.a[l], bytes)) != hipSuccess) return e;
        if ((e = hipMemset(a.a[l], 0, bytes)) != hipSuccess) return e;
    }
    for (int l = distinct + 1; l <= 5; l++) a.a[l] = a.a[l - 2];  // inference: ping-pong
    return hipMalloc(&a.out, (size_t)B * H * W * sizeof(float));
}

void acts_free(Acts &a)
{
    if (a.x1) (void)hipFree(a.x1);
    for (int l = 1; l <= 5; l++) {
        bool alias = false;
        for (int k = 1; k < l; k++) alias |= a.a[k] == a.a[l];
        if (a.a[l] && !alias) (void)hipFree(a.a[l]);
    }
    if (a.out) (void)hipFree(a.out);
    a = Acts();
}

void im2col(const Acts &a, const float *planes, int npl, hipStream_t stream)
{
    hipLaunchKernelGGL(k_im2col, dim3(nblocks((long)a.B * a.H * a.W)), dim3(BLOCK), 0, stream, planes, npl, a.x1,
                       a.B, a.H, a.W);
}

// Rows per run of the marching layers: about one workgroup (95 KB of LDS)
// per compute unit, a multiple of rows.
int march_run_rows(int H, int W, int B, int rows)
{
    static int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
            n = 256;
        return n;
    }();
    const long bands = (long)(W / 64) * B;
    const long runs = bands >= cus ? 1 : cus / bands;
    const long per = (H + runs - 1) / runs;
    return (int)((per + rows - 1) / rows * rows);
}

// The marching layers (k_first_conv32_march, k_conv32_march,
// k_conv_out_march) for one image where the height is a multiple of 16,
// unless TEA_WS_MARCH=0.  Not before a backward pass (layers_too): the march keeps
// layer 1's output in LDS, and the gradients of layers 1 and 2 read it from memory.
template <int ROWS>
void forward_rows(const Net &net, const Acts &a, const float *planes, int npl, hipStream_t stream, bool layers_too)
{
    const dim3 grid(a.W / 64, a.H / ROWS, a.B), block(ROWS * 64);
    const bf16x8 *pk = (const bf16x8 *)net.packed;
    const char *env = getenv("TEA_WS_MARCH");
    const bool march = ROWS == 16 && a.B == 1 && !layers_too && !(env && env[0] == '0');
    int run_rows = march_run_rows(a.H, a.W, a.B, ROWS);
    // TEA_WS_MARCH_ROWS=<rows> sets the run length (tests march several blocks on small images)
    if (const char *s = getenv("TEA_WS_MARCH_ROWS")) {
        const int v = atoi(s);
        if (v > 0) run_rows = (v + ROWS - 1) / ROWS * ROWS;
    }
    const dim3 mgrid(a.W / 64, (a.H + run_rows - 1) / run_rows, a.B);
    if (march)   // layers 1 and 2 in one march (layer 1's output stays in LDS)
        hipLaunchKernelGGL(k_first_conv32_march<ROWS>, mgrid, block, 0, stream, planes, npl, a.a[2], pk + PK_L1 / 8,
                           net.params + OFF_B1, pk + pk_fwd(2) / 8, net.params + off_b(2), a.H, a.W, run_rows);
    else
        hipLaunchKernelGGL(k_conv_first<ROWS>, grid, block, 0, stream, planes, npl, a.a[1], pk + PK_L1 / 8,
                           net.params + OFF_B1, a.H, a.W);
    for (int l = march ? 3 : 2; l <= 5; l++) {
        if (march)
            hipLaunchKernelGGL(k_conv32_march<ROWS>, mgrid, block, 0, stream, a.a[l - 1], a.a[l], pk + pk_fwd(l) / 8,
                               net.params + off_b(l), a.H, a.W, run_rows);
        else
            hipLaunchKernelGGL((k_conv32<ROWS, false>), grid, block, 0, stream, a.a[l - 1], a.a[l],
                               pk + pk_fwd(l) / 8, net.params + off_b(l), (const __bf16 *)nullptr, a.H, a.W);
    }
    if (march)
        hipLaunchKernelGGL(k_conv_out_march<ROWS>, mgrid, block, 0, stream, a.a[5], pk + PK_OUT / 8,
                           net.params + OFF_B6, a.out, a.H, a.W, run_rows);
    else
        hipLaunchKernelGGL(k_conv_out<ROWS>, grid, block, 0, stream, a.a[5], pk + PK_OUT / 8, net.params + OFF_B6,
                           a.out, a.H, a.W);
}

// Inference takes workgroups of 16 rows where the height allows it: a smaller
// share of re-read halo rows (18/16 against 10/8 per staged window).
void forward(const Net &net, const Acts &a, const float *planes, int npl, hipStream_t stream, bool layers_too)
{
    if (a.H % 16 == 0) forward_rows<16>(net, a, planes, npl, stream, layers_too);
    else if (conv_rows(a.H) == 8) forward_rows<8>(net, a, planes, npl, stream, layers_too);
    else forward_rows<4>(net, a, planes, npl, stream, layers_too);
}

}  // namespace ws

// =============================================================================
// Trainer C-ABI
// =============================================================================
namespace {

char g_ws_error[512] = "";

int ws_fail(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_ws_error, sizeof g_ws_error, fmt, ap);
    va_end(ap);
    return -1;
}

#define WS_OK(call)                                                                     \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess) return ws_fail("%s: %s", #call, hipGetErrorString(e_));  \
    } while (0)

struct Trainer {
    int B = 0, H = 0, W = 0, margin = 0, energy = 0;
    long step = 0;
    hipStream_t stream = nullptr;
    ws::Net net;
    ws::Acts acts;
    float *g6 = nullptr;            // padded FP32 gradient of the output layer
    __bf16 *g[2] = {};              // padded NHWC32 gradients (ping-pong)
    float *grad = nullptr, *m = nullptr, *v = nullptr;
    float *part = nullptr;          // weight-gradient partials
    double *loss_part = nullptr;
    int loss_blocks = 0;
};

void destroy(Trainer *t)
{
    if (!t) return;
    if (t->stream) (void)hipStreamSynchronize(t->stream);
    ws::net_free(t->net);
    ws::acts_free(t->acts);
    for (void *p : {(void *)t->g6, (void *)t->g[0], (void *)t->g[1], (void *)t->grad, (void *)t->m, (void *)t->v,
                    (void *)t->part, (void *)t->loss_part})
        if (p) (void)hipFree(p);
    if (t->stream) (void)hipStreamDestroy(t->stream);
    delete t;
}

int forward_pass(Trainer *t, const float *samples, bool layers_too)
{
    ws::im2col(t->acts, samples, ws::NPLANES, t->stream);
    ws::forward(t->net, t->acts, samples, ws::NPLANES, t->stream, layers_too);
    WS_OK(hipGetLastError());
    return 0;
}

void sum_parts(const float *part, int parts, int n, float *dst, hipStream_t s)
{
    hipLaunchKernelGGL(ws::k_sum_parts, dim3((n + 31) / 32), dim3(ws::BLOCK), 0, s, part, parts, n, dst);
}

// loss, then every gradient into t->grad (same layout as the parameters)
int backward_pass(Trainer *t, const float *samples)
{
    using namespace ws;
    const int B = t->B, H = t->H, W = t->W;
    const long npix = (long)B * H * W;
    const long inner = (long)B * (H - 2 * t->margin) * (W - 2 * t->margin);
    const float scale = 2.0f / (float)inner;
    hipStream_t s = t->stream;
    hipLaunchKernelGGL(k_loss, dim3(t->loss_blocks), dim3(BLOCK), 0, s, t->acts.out, samples, t->g6, t->loss_part,
                       B, H, W, t->margin, scale, t->energy);
    // layer 6
    {
        // about 2048 waves; a run no shorter than 8 rows (two more are read for the window)
        const long cols = (long)B * (W / 16);
        const int rows = (int)std::min<long>(H, std::max<long>(8, (cols * H + 2047) / 2048));
        const int nruns = (H + rows - 1) / rows;
        const long tasks = cols * nruns;
        const int parts = (int)std::min<long>(WG_PARTS, (tasks + 3) / 4);
        float *runs = t->part + (long)WG_PARTS * TAPS * CH;
        hipLaunchKernelGGL(k_out_wgrad, dim3(parts + BIAS_RUNS / (BLOCK / 64)), dim3(BLOCK), 0, s, t->acts.a[5],
                           t->g6, t->part, runs, B, H, W, rows, nruns, tasks, parts);
        hipLaunchKernelGGL(k_sum_runs, dim3(1), dim3(64), 0, s, runs, t->grad + OFF_B6);
        sum_parts(t->part, parts, TAPS * CH, t->grad + OFF_W6, s);
    }
    hipLaunchKernelGGL(k_out_bwd, dim3(nblocks(npix)), dim3(BLOCK), 0, s, t->g6, t->net.w6, t->acts.a[5], t->g[0],
                       B, H, W);
    // the 32-channel layers: two workgroups per compute unit, runs of an even number of rows (two per step),
    // no shorter than 8 (the run's g rows above and below are read twice)
    const long bands = (long)B * (W / 64);
    const int wrows = (int)std::min<long>(H, std::max<long>(8, (bands * H + WG_PARTS - 1) / WG_PARTS + 1) & ~1L);
    const int wruns = (H + wrows - 1) / wrows;
    const int wparts = (int)std::min<long>(WG_PARTS, bands * wruns);
    // layers 5..2: weight and bias gradients from g(l), then g(l-1)
    const int rows = conv_rows(H);
    const dim3 grid(W / 64, H / rows, B), block(rows * 64);
    const bf16x8 *pk = (const bf16x8 *)t->net.packed;
    int cur = 0;
    for (int l = 5; l >= 2; l--) {
        // weights and bias are neighbours in the parameter vector
        hipLaunchKernelGGL((k_wgrad32<TAPS>), dim3(wparts), dim3(BLOCK), 0, s, t->acts.a[l - 1], t->g[cur], t->part,
                           H, W, wrows, wruns, bands * wruns);
        sum_parts(t->part, wparts, HID_SIZE, t->grad + off_w(l), s);
        if (rows == 8)
            hipLaunchKernelGGL((k_conv32<8, true>), grid, block, 0, s, t->g[cur], t->g[1 - cur], pk + pk_bwd(l) / 8,
                               (const float *)nullptr, t->acts.a[l - 1], H, W);
        else
            hipLaunchKernelGGL((k_conv32<4, true>), grid, block, 0, s, t->g[cur], t->g[1 - cur], pk + pk_bwd(l) / 8,
                               (const float *)nullptr, t->acts.a[l - 1], H, W);
        cur = 1 - cur;
    }
    // layer 1 (im2col input, no input gradient)
    hipLaunchKernelGGL((k_wgrad32<1>), dim3(wparts), dim3(BLOCK), 0, s, t->acts.x1, t->g[cur], t->part, H, W, wrows,
                       wruns, bands * wruns);
    sum_parts(t->part, wparts, K1 * CH + CH, t->grad + OFF_W1, s);
    WS_OK(hipGetLastError());
    return 0;
}

int read_loss(Trainer *t, double *loss)
{
    if (!loss) return 0;
    std::vector<double> h(t->loss_blocks);
    WS_OK(hipMemcpyAsync(h.data(), t->loss_part, h.size() * sizeof(double), hipMemcpyDeviceToHost, t->stream));
    WS_OK(hipStreamSynchronize(t->stream));
    double s = 0.0;
    for (double x : h) s += x;
    const long inner = (long)t->B * (t->H - 2 * t->margin) * (t->W - 2 * t->margin);
    *loss = s / (double)inner;
    return 0;
}

}  // namespace

EXPORT const char *tea_ws_last_error(void) { return g_ws_error; }

EXPORT int tea_ws_param_count(void) { return ws::NPARAM; }

EXPORT void *tea_ws_trainer_create(int batch, int height, int width, int margin, int loss)
{
    if (loss != 0 && loss != 1) {
        ws_fail("tea_ws_trainer_create: loss %d is not 0 (MSE) or 1 (energy)", loss);
        return nullptr;
    }
    if (batch < 1 || !ws::shape_ok(height, width)) {
        ws_fail("tea_ws_trainer_create: need batch >= 1, height %% 4 == 0, width %% 64 == 0 (got %d, %d, %d)", batch,
                height, width);
        return nullptr;
    }
    if (margin < 0 || 2 * margin >= height || 2 * margin >= width) {
        ws_fail("tea_ws_trainer_create: margin %d leaves no pixels", margin);
        return nullptr;
    }
    Trainer *t = new Trainer();
    t->B = batch;
    t->H = height;
    t->W = width;
    t->margin = margin;
    t->energy = loss;
    const long npix = (long)batch * height * width;
    t->loss_blocks = (int)ws::nblocks(npix);
    const size_t gbytes = ws::act_bytes(batch, height, width);
    const size_t g6bytes = (size_t)batch * (height + 2) * (width + 2) * sizeof(float);
    const size_t part_floats = (size_t)ws::WG_PARTS * ws::HID_SIZE;
    bool ok = hipStreamCreateWithFlags(&t->stream, hipStreamNonBlocking) == hipSuccess &&
              ws::net_alloc(t->net) == hipSuccess && ws::acts_alloc(t->acts, batch, height, width, true) == hipSuccess &&
              hipMalloc(&t->g6, g6bytes) == hipSuccess && hipMemset(t->g6, 0, g6bytes) == hipSuccess &&
              hipMalloc(&t->g[0], gbytes) == hipSuccess && hipMemset(t->g[0], 0, gbytes) == hipSuccess &&
              hipMalloc(&t->g[1], gbytes) == hipSuccess && hipMemset(t->g[1], 0, gbytes) == hipSuccess &&
              hipMalloc(&t->grad, ws::NPARAM * sizeof(float)) == hipSuccess &&
              hipMalloc(&t->m, ws::NPARAM * sizeof(float)) == hipSuccess &&
              hipMalloc(&t->v, ws::NPARAM * sizeof(float)) == hipSuccess &&
              hipMalloc(&t->part, part_floats * sizeof(float)) == hipSuccess &&
              hipMalloc(&t->loss_part, t->loss_blocks * sizeof(double)) == hipSuccess &&
              hipDeviceSynchronize() == hipSuccess;
    if (!ok) {
        ws_fail("tea_ws_trainer_create: device allocation failed (%s)", hipGetErrorString(hipGetLastError()));
        destroy(t);
        return nullptr;
    }
    return t;
}

EXPORT void tea_ws_trainer_destroy(void *h) { destroy((Trainer *)h); }

EXPORT int tea_ws_trainer_set_params(void *h, const float *host_params)
{
    Trainer *t = (Trainer *)h;
    if (!t || !host_params) return ws_fail("tea_ws_trainer_set_params: null argument");
    WS_OK(ws::net_upload(t->net, host_params, t->stream));
    WS_OK(hipMemsetAsync(t->m, 0, ws::NPARAM * sizeof(float), t->stream));
    WS_OK(hipMemsetAsync(t->v, 0, ws::NPARAM * sizeof(float), t->stream));
    WS_OK(hipStreamSynchronize(t->stream));
    t->step = 0;
    return 0;
}

EXPORT int tea_ws_trainer_get_params(void *h, float *host_params)
{
    Trainer *t = (Trainer *)h;
    if (!t || !host_params) return ws_fail("tea_ws_trainer_get_params: null argument");
    WS_OK(hipMemcpyAsync(host_params, t->net.params, ws::NPARAM * sizeof(float), hipMemcpyDeviceToHost, t->stream));
    WS_OK(hipStreamSynchronize(t->stream));
    return 0;
}

EXPORT int tea_ws_trainer_forward(void *h, const float *samples, float *out_host)
{
    Trainer *t = (Trainer *)h;
    if (!t || !samples || !out_host) return ws_fail("tea_ws_trainer_forward: null argument");
    if (forward_pass(t, samples, false)) return -1;
    WS_OK(hipMemcpyAsync(out_host, t->acts.out, (size_t)t->B * t->H * t->W * sizeof(float), hipMemcpyDeviceToHost,
                         t->stream));
    WS_OK(hipStreamSynchronize(t->stream));
    return 0;
}

EXPORT int tea_ws_trainer_gradient(void *h, const float *samples, float *grad_host, double *loss)
{
    Trainer *t = (Trainer *)h;
    if (!t || !samples || !grad_host) return ws_fail("tea_ws_trainer_gradient: null argument");
    if (forward_pass(t, samples, true) || backward_pass(t, samples)) return -1;
    WS_OK(hipMemcpyAsync(grad_host, t->grad, ws::NPARAM * sizeof(float), hipMemcpyDeviceToHost, t->stream));
    WS_OK(hipStreamSynchronize(t->stream));
    return read_loss(t, loss);
}

EXPORT int tea_ws_trainer_step(void *h, const float *samples, float lr, double *loss)
{
    Trainer *t = (Trainer *)h;
    if (!t || !samples) return ws_fail("tea_ws_trainer_step: null argument");
    if (forward_pass(t, samples, true) || backward_pass(t, samples)) return -1;
    if (loss && read_loss(t, loss)) return -1;
    t->step++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)t->step), c2 = 1.0f - powf(b2, (float)t->step);
    hipLaunchKernelGGL(ws::k_adam, dim3(ws::nblocks(ws::NPARAM)), dim3(ws::BLOCK), 0, t->stream, t->net.params,
                       t->grad, t->m, t->v, ws::NPARAM, lr, b1, b2, 1e-8f, c1, c2);
    ws::net_pack(t->net, t->stream);
    WS_OK(hipGetLastError());
    return 0;
}

EXPORT int tea_ws_trainer_sync(void *h)
{
    Trainer *t = (Trainer *)h;
    if (!t) return ws_fail("tea_ws_trainer_sync: null argument");
    WS_OK(hipStreamSynchronize(t->stream));
    return 0;
}

EXPORT int tea_ws_make_samples(const double *rho, const double *u_prev2, const double *u_prev, const double *u0,
                               const double *u_next, const double *kx, const double *ky, int nx, int ny, double c0,
                               double c1, const int *origins, int n, int crop, float *out, double *scales)
{
    if (!rho || !u_prev2 || !u_prev || !u0 || !u_next || !kx || !ky || !origins || !out || !scales || nx < 1 ||
        ny < 1 || n < 1 || crop < 1)
        return ws_fail("tea_ws_make_samples: bad argument");
    const long cells = (long)nx * ny;
    const int blocks = 1024;
    double *part = nullptr;
    WS_OK(hipMalloc(&part, 2 * blocks * sizeof(double)));
    hipLaunchKernelGGL(ws::k_scales, dim3(blocks), dim3(ws::BLOCK), 0, nullptr, u_prev, u0, cells, part);
    std::vector<double> h(2 * blocks);
    hipError_t e = hipMemcpy(h.data(), part, h.size() * sizeof(double), hipMemcpyDeviceToHost);
    (void)hipFree(part);
    WS_OK(e);
    double a = 0.0, c = 0.0;
    for (int b = 0; b < blocks; b++) {
        a += h[2 * b];
        c += h[2 * b + 1];
    }
    scales[0] = std::sqrt(a / (double)cells);
    scales[1] = std::sqrt(c / (double)cells);
    if (!(scales[0] > 0.0) || !(scales[1] > 0.0)) return ws_fail("tea_ws_make_samples: zero field scale");
    const long total = (long)n * crop * crop;
    hipLaunchKernelGGL(ws::k_make_samples, dim3(ws::nblocks(total)), dim3(ws::BLOCK), 0, nullptr, rho, u_prev2,
                       u_prev, u0, u_next, kx, ky, nx, ny, c0, c1, 1.0 / scales[0], 1.0 / scales[1], origins, n, crop,
                       out);
    WS_OK(hipGetLastError());
    WS_OK(hipDeviceSynchronize());
    return 0;
}
