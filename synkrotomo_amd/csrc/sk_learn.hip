// sk_learn.hip -- kernels of the learned SIRT correction (no reference counterpart) and the
// GPU phantom generator used to train it.
//
// Network: y = x + conv4(relu(conv3(relu(conv2(relu(conv1(x))))))), 3x3 convolutions with
// stride 1 and zero padding 1; conv1: 1 -> 32 channels, conv2/conv3: 32 -> 32, conv4: 32 -> 1.
// Activations are BF16 in NHWC layout ([image][row][col][32]); images, biases and every
// accumulation are FP32; weights are BF16 in [Cout][ky][kx][Cin] layout.
//
//   k_conv32      32 -> 32 (the FLOP-heavy layers) as an implicit GEMM on gfx950 MFMA
//                 (v_mfma_f32_16x16x32_bf16): M = 16 output channels, N = 16 output pixels
//                 of one row, K = 32 input channels of one tap; 9 taps accumulate.  Persistent
//                 blocks compute 16x16-pixel x 32-channel tiles from an LDS-staged 18x18x32
//                 input patch (the next tile's patch loaded during the MFMAs) and the 32x9x32
//                 weights, staged once per block.  The same kernel computes the data
//                 gradient: with weights that the caller flipped and transposed, the ReLU derivative
//                 of the layer's output in the staging of its input (mask); or with the forward
//                 weights, flipped while they are staged, and the derivative of the layer below in
//                 its output (omask; four library launches less in a backward pass of the
//                 network: 285 and 259 us for one of 7 images of 86^2, where launches count).
//   k_conv_in     1 or 2 -> 32 (288 MACs per pixel and input channel) on VALU with fused bias and
//                 ReLU, in FP32 on the FP32 input (the image, or the image and the SIRT update
//                 direction interleaved); the data gradient of the last layer likewise.
//   k_conv_out_mfma  32 -> 1: per 16x16 tile, the 9 tap products of every halo pixel in one
//                 MFMA per 16 pixels, then a 9-term shifted sum per output, fused bias and
//                 residual; the data gradient of the first layer likewise.
//   k_wgrad32_mfma  weight and bias gradients of the 32 -> 32 layers on MFMA (K = pixels),
//                 tiles staged in LDS as they are and transposed by the reads; per-block partial
//                 sums (deterministic), then k_reduce_partials.
//   k_wgrad_thin  weight and bias gradients of the thin layers (1 -> 32, 32 -> 1) on VALU, the
//                 same per-block partials.
//   k_phantom     random-ellipse phantoms, evaluated in FP64 exactly as the numpy
//                 generator (synkrotomo_amd/phantom.py) does.
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "sk_common.h"

namespace sk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CT = 16;    // conv tile side (pixels)
constexpr int CP = 40;    // LDS channel stride (bf16 elements): 80 B, keeps 16 B alignment
constexpr int NCH = 32;   // hidden channels

// ---------------------------------------------------------------------- 32 -> 32, MFMA
// Persistent blocks: each stages the 32x9x32 weights in LDS once, then walks output tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...  A tile's 18x18x32 input patch is loaded into
// registers while the previous tile's MFMAs run, then stored to LDS.  The MFMA's M is the 16
// output channels of a channel block (A = weights), N the 16 pixels of a row (B = input), so
// each lane's accumulator holds 4 consecutive channels of one pixel: 8-byte stores.
constexpr int PATCH_Q = (CT + 2) * (CT + 2) * 4;      // 16-byte quads of a patch
constexpr int PATCH_PER_T = (PATCH_Q + 255) / 256;    // per thread

// MASK_OUT: y is zeroed where omask <= 0 (the gradient of the pre-activation of the layer below, so
// that none of its readers needs the mask again).
template <bool MASK_IN, bool BIAS_RELU, bool MASK_OUT = false>
__global__ __launch_bounds__(256) void k_conv32(int H, int W, long ntiles, const __bf16* __restrict__ x,
                                                const __bf16* __restrict__ mask,
                                                const __bf16* __restrict__ w,
                                                const float* __restrict__ bias,
                                                __bf16* __restrict__ y,
                                                const __bf16* __restrict__ omask = nullptr) {
  __shared__ __attribute__((aligned(16))) __bf16 sx[(CT + 2) * (CT + 2) * CP];
  __shared__ __attribute__((aligned(16))) __bf16 sw[NCH * 9 * CP];
  const int tiles_x = (W + CT - 1) / CT;
  const long tiles_img = (long)tiles_x * ((H + CT - 1) / CT);
  for (int c = threadIdx.x; c < NCH * 9 * 4; c += 256) {
    const int row = c >> 2, q = c & 3;  // row = co*9 + tap
    const bf16x8 v = *(const bf16x8*)(w + row * NCH + q * 8);
    if constexpr (MASK_OUT) {  // a data gradient: the forward weights flipped and transposed
      const int co = row / 9, tap = row - 9 * co;
      for (int i = 0; i < 8; ++i) sw[((q * 8 + i) * 9 + 8 - tap) * CP + co] = v[i];
    } else {
      *(bf16x8*)(sw + row * CP + q * 8) = v;
    }
  }
  bf16x8 pf[PATCH_PER_T];
  auto load_patch = [&](long t) {
    const long b = t / tiles_img;
    const int r = (int)(t - b * tiles_img);
    const int tx0 = (r % tiles_x) * CT, ty0 = (r / tiles_x) * CT;
    const size_t img = (size_t)b * H * W;
#pragma unroll
    for (int k = 0; k < PATCH_PER_T; ++k) {
      const int c = threadIdx.x + 256 * k;
      bf16x8 v;
      for (int i = 0; i < 8; ++i) v[i] = (__bf16)0.0f;
      const int pix = c >> 2, q = c & 3;
      const int py = pix / (CT + 2), px = pix - py * (CT + 2);
      const int gy = ty0 + py - 1, gx = tx0 + px - 1;
      if (c < PATCH_Q && gy >= 0 && gy < H && gx >= 0 && gx < W) {
        const size_t off = (img + (size_t)gy * W + gx) * NCH + q * 8;
        v = *(const bf16x8*)(x + off);
        if constexpr (MASK_IN) {
          const bf16x8 m = *(const bf16x8*)(mask + off);
          for (int i = 0; i < 8; ++i)
            if (!((float)m[i] > 0.0f)) v[i] = (__bf16)0.0f;
        }
      }
      pf[k] = v;
    }
  };
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  long t = blockIdx.x;
  if (t < ntiles) load_patch(t);
  for (; t < ntiles; t += gridDim.x) {  // uniform over the block: every thread reaches each barrier
    __syncthreads();  // the previous tile's LDS reads (and, first, the weight stores) are done
#pragma unroll
    for (int k = 0; k < PATCH_PER_T; ++k) {
      const int c = threadIdx.x + 256 * k;
      if (c < PATCH_Q) *(bf16x8*)(sx + (c >> 2) * CP + (c & 3) * 8) = pf[k];
    }
    __syncthreads();
    const long tn = t + gridDim.x;
    if (tn < ntiles) load_patch(tn);  // in flight during this tile's MFMAs
    const long b = t / tiles_img;
    const int r = (int)(t - b * tiles_img);
    const int tx0 = (r % tiles_x) * CT, ty0 = (r / tiles_x) * CT;
    const size_t img = (size_t)b * H * W;
    [[maybe_unused]] bf16x4 om[4][2];
    if constexpr (MASK_OUT) {
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const int oy = min(ty0 + wv * 4 + mb, H - 1), ox = min(tx0 + m, W - 1);  // in bounds; used where written
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          om[mb][nb] = *(const bf16x4*)(omask + (img + (size_t)oy * W + ox) * NCH + nb * 16 + 4 * kq);
      }
    }
    f32x4 acc[4][2];
    for (int a = 0; a < 4; ++a)
      for (int c = 0; c < 2; ++c) acc[a][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int tp = 0; tp < 9; ++tp) {
      const int ky = tp / 3, kx = tp - 3 * (tp / 3);
      // A: weights of output channels nb*16 + m, input channels 8kq..8kq+7 of tap tp
      const bf16x8 w0 = *(const bf16x8*)(sw + ((0 * 16 + m) * 9 + tp) * CP + 8 * kq);
      const bf16x8 w1 = *(const bf16x8*)(sw + ((1 * 16 + m) * 9 + tp) * CP + 8 * kq);
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        const int oy = wv * 4 + mb;
        // B: input channels 8kq..8kq+7 of pixel m of output row oy, shifted by the tap
        const bf16x8 a = *(const bf16x8*)(sx + ((oy + ky) * (CT + 2) + m + kx) * CP + 8 * kq);
        acc[mb][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, a, acc[mb][0], 0, 0, 0);
        acc[mb][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, a, acc[mb][1], 0, 0, 0);
      }
    }
    // C: lane holds output channels nb*16 + 4kq + i (i < 4) of pixel m of row oy.
    const int ox = tx0 + m;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int oy = ty0 + wv * 4 + mb;
      if (oy >= H || ox >= W) continue;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const int co = nb * 16 + 4 * kq;
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[mb][nb][i];
          if constexpr (BIAS_RELU) v = fmaxf(v + bias[co + i], 0.0f);
          if constexpr (MASK_OUT) v = (float)om[mb][nb][i] > 0.0f ? v : 0.0f;
          o[i] = (__bf16)v;
        }
        *(bf16x4*)(y + (img + (size_t)oy * W + ox) * NCH + co) = o;
      }
    }
  }
}

// ---------------------------------------------------------------------- CIN -> 32, VALU
// h[p][co] = relu(b[co] + sum_t sum_c w[co][t][c] x[p + off_t][c]); x: FP32 [B][H][W][CIN]
// (CIN = 1: an image; CIN = 2: the image and the SIRT update direction, interleaved), w: BF16
// [32][9][CIN].  Grid (pixel blocks of one image, images).  The weights are read as BF16 pairs
// through readfirstlane (wave-uniform values: scalar loads into SGPRs, unpacked on the scalar
// unit, operands of the FMAs): no LDS reads for them and no per-lane conversion.  Same
// operations in the same order as a plain per-pixel loop: bias, then taps 0..8 (channels in
// order within a tap).  The block's 256 x 32 BF16 outputs (16 KB, contiguous in NHWC) go out
// through LDS so that every store instruction writes 1 KB of consecutive bytes.  w2: the
// weights as 144 * CIN words.
template <int CIN>
__global__ __launch_bounds__(256) void k_conv_in(int H, int W, const float* __restrict__ x,
                                                 const uint32_t* __restrict__ w2,
                                                 const float* __restrict__ bias,
                                                 __bf16* __restrict__ h) {
  __shared__ bf16x8 st[256 * 4];
  const int r0 = blockIdx.x * 256;
  const int r = r0 + threadIdx.x;
  const bool live = r < H * W;
  const size_t img = (size_t)blockIdx.y * H * W;
  const int py = r / W, px = r - py * W;
  float v[9][CIN];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int yy = py + t / 3 - 1, xx = px + t % 3 - 1;
    const bool in = live && yy >= 0 && yy < H && xx >= 0 && xx < W;
#pragma unroll
    for (int c = 0; c < CIN; ++c) v[t][c] = in ? x[(img + (size_t)yy * W + xx) * CIN + c] : 0.0f;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int co = q * 8 + i;
      float s = bias[co];
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int c = 0; c < CIN; ++c) {
          const int k = (co * 9 + t) * CIN + c;
          const uint32_t pr = __builtin_amdgcn_readfirstlane(w2[k >> 1]);
          s = fmaf(__builtin_bit_cast(float, (k & 1) ? (pr & 0xffff0000u) : (pr << 16)), v[t][c], s);
        }
      o[i] = (__bf16)fmaxf(s, 0.0f);
    }
    st[threadIdx.x * 4 + q] = o;
  }
  __syncthreads();
  bf16x8* out = (bf16x8*)(h + (img + r0) * NCH);
  const int n = min(256, H * W - r0) * 4;  // 16-byte chunks of this block's pixels
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c < n) out[c] = st[c];
  }
}

// 32 -> 1 on MFMA: for a 16x16 output tile, the 18x18 input pixels of its halo each get
// U[q][t] = sum_ci h[q][ci] w[t][ci] for the 9 taps t in one GEMM ([pixels x 32] x [32 x 16],
// taps 9..15 zero: one v_mfma_f32_16x16x32_bf16 per 16 pixels), kept in LDS; each output
// pixel then sums its 9 shifted taps: y[p] = res[p] + (sum_t U[p + off_t][t] + bias).
// Each activation is read once per tile (the halo adds 27%).
constexpr int CO_SLOTS = 21 * 16;  // 18*18 = 324 halo pixels in groups of 16

__global__ __launch_bounds__(256) void k_conv_out_mfma(int H, int W, const __bf16* __restrict__ h,
                                                       const __bf16* __restrict__ w,
                                                       const float* __restrict__ bias,
                                                       const float* __restrict__ res,
                                                       float* __restrict__ y) {
  __shared__ float U[CO_SLOTS * 9];
  const int tiles_x = (W + CT - 1) / CT;
  const int tx0 = (blockIdx.x % tiles_x) * CT, ty0 = (blockIdx.x / tiles_x) * CT;
  const size_t img = (size_t)blockIdx.y * H * W;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  // B: w[tap m][8kq .. 8kq+7] for taps 0..8, zero columns for m >= 9
  bf16x8 wb;
  for (int i = 0; i < 8; ++i) wb[i] = (__bf16)0.0f;
  if (m < 9) wb = *(const bf16x8*)(w + m * NCH + 8 * kq);
  // wave wv takes pixel groups wv, wv + 4, ...: all of its loads are issued before the MFMAs
  constexpr int NG = CO_SLOTS / 16, GPW = (NG + 3) / 4;
  bf16x8 a[GPW];
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int slot = (wv + 4 * k) * 16 + m;  // A row m: halo pixel `slot`
    const int hy = slot / (CT + 2), hx = slot - hy * (CT + 2);
    const int gy = ty0 + hy - 1, gx = tx0 + hx - 1;
    for (int i = 0; i < 8; ++i) a[k][i] = (__bf16)0.0f;
    if (slot < (CT + 2) * (CT + 2) && gy >= 0 && gy < H && gx >= 0 && gx < W)
      a[k] = *(const bf16x8*)(h + (img + (size_t)gy * W + gx) * NCH + 8 * kq);
  }
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int g = wv + 4 * k;
    if (g >= NG) break;  // wave-uniform
    const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k], wb, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
    // C: lane holds U[pixel g*16 + 4kq + i][tap m]
    if (m < 9)
      for (int i = 0; i < 4; ++i) U[(g * 16 + 4 * kq + i) * 9 + m] = c[i];
  }
  __syncthreads();
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
  const int oy = ty0 + ty, ox = tx0 + tx;
  if (oy >= H || ox >= W) return;
  float sum = 0.0f;
#pragma unroll
  for (int t = 0; t < 9; ++t) sum += U[((ty + t / 3) * (CT + 2) + tx + t % 3) * 9 + t];
  const size_t p = img + (size_t)oy * W + ox;
  y[p] = res[p] + (sum + bias[0]);
}

// d h[q][ci] = sum_t w[t][ci] g[q - off_t]   (data gradient of the 32 -> 1 layer), zeroed where h <= 0
// with MASK_OUT.  The block's 256 x 32 BF16 outputs go out through LDS (and its mask comes in the
// same order): every store instruction writes 1 KB of consecutive bytes.
template <bool MASK_OUT>
__global__ __launch_bounds__(256) void k_conv_out_dgrad(int H, int W, long npix, const float* __restrict__ g,
                                                        const __bf16* __restrict__ w,
                                                        __bf16* __restrict__ dh,
                                                        const __bf16* __restrict__ h) {
  __shared__ float sw[9 * NCH];
  __shared__ bf16x8 st[256 * 4];
  for (int i = threadIdx.x; i < 9 * NCH; i += 256) sw[i] = (float)w[i];
  const long p0 = (long)blockIdx.x * 256;
  const int n = (int)min(256L, npix - p0) * 4;  // 16-byte chunks of this block's pixels
  [[maybe_unused]] bf16x8 mk[4];
  if constexpr (MASK_OUT) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int c = threadIdx.x + 256 * k;
      mk[k] = ((const bf16x8*)(h + p0 * NCH))[c < n ? c : 0];
    }
  }
  __syncthreads();
  const long p = p0 + threadIdx.x;
  const long b = p / ((long)H * W);
  const int r = (int)(p - b * H * W);
  const int py = r / W, px = r - py * W;
  float gv[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int yy = py - (t / 3 - 1), xx = px - (t % 3 - 1);
    gv[t] = (p < npix && yy >= 0 && yy < H && xx >= 0 && xx < W) ? g[(b * H + yy) * W + xx] : 0.0f;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int ci = q * 8 + i;
      float s = 0.0f;
#pragma unroll
      for (int t = 0; t < 9; ++t) s = fmaf(sw[t * NCH + ci], gv[t], s);
      o[i] = (__bf16)s;
    }
    st[threadIdx.x * 4 + q] = o;
  }
  __syncthreads();
  bf16x8* out = (bf16x8*)(dh + p0 * NCH);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c >= n) continue;
    bf16x8 o = st[c];
    if constexpr (MASK_OUT) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (!((float)mk[k][i] > 0.0f)) o[i] = (__bf16)0.0f;
    }
    out[c] = o;
  }
}

// dx[q][c] = sum_{t,co} w[co][t][c] g1[q - off_t][co],  g1 = dh * (h > 0) (MASK) or dh   (data gradient of
// k_conv_in; dx FP32 [B][H][W][CIN]).  As k_conv_out_mfma: per 16x16 tile and input channel c, each
// of the 18x18 halo pixels of g1 gets U[p][t] = sum_co g1[p][co] w[co][t][c] for the 9 taps in one
// MFMA per 16 pixels (products of BF16 values, exact in the FP32 accumulator's input), then each
// output sums its 9 shifted taps.  Bound by the two activation streams: 8 x 512^2, 1.21 times 134 MB
// each, 69 us = 4.7 TB/s (on VALU with one thread per pixel re-reading every neighbour's 32
// channels: 851 us); 31 us for a gradient that needs no mask.
template <int CIN, bool MASK>
__global__ __launch_bounds__(256) void k_conv_in_dgrad(int H, int W, long ntiles,
                                                       const __bf16* __restrict__ dh,
                                                       const __bf16* __restrict__ hmask,
                                                       const __bf16* __restrict__ w,
                                                       float* __restrict__ dx) {
  __shared__ float U[CO_SLOTS * 9];
  const int tiles_x = (W + CT - 1) / CT, tiles_img = tiles_x * ((H + CT - 1) / CT);
  const long block = (long)blockIdx.y * gridDim.x + blockIdx.x;
  if (block >= ntiles) return;  // uniform
  const long b = block / tiles_img;
  const int tile = (int)(block - b * tiles_img);
  const int tx0 = (tile % tiles_x) * CT, ty0 = (tile / tiles_x) * CT;
  const size_t img = (size_t)b * H * W;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  constexpr int NG = CO_SLOTS / 16, GPW = (NG + 3) / 4;
  bf16x8 a[GPW];
#pragma unroll
  for (int k = 0; k < GPW; ++k) {
    const int slot = (wv + 4 * k) * 16 + m;  // A row m: halo pixel `slot`
    const int hy = slot / (CT + 2), hx = slot - hy * (CT + 2);
    const int gy = ty0 + hy - 1, gx = tx0 + hx - 1;
    for (int i = 0; i < 8; ++i) a[k][i] = (__bf16)0.0f;
    if (slot < (CT + 2) * (CT + 2) && gy >= 0 && gy < H && gx >= 0 && gx < W) {
      const size_t off = (img + (size_t)gy * W + gx) * NCH + 8 * kq;
      const bf16x8 g = *(const bf16x8*)(dh + off);
      if constexpr (MASK) {
        const bf16x8 mk = *(const bf16x8*)(hmask + off);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if ((float)mk[i] > 0.0f) a[k][i] = g[i];
      } else {
        a[k] = g;
      }
    }
  }
  const int ty = threadIdx.x >> 4, tx = threadIdx.x & 15;
  const int oy = ty0 + ty, ox = tx0 + tx;
#pragma unroll
  for (int c = 0; c < CIN; ++c) {
    if (c > 0) __syncthreads();  // the previous channel's sums have been read
    // B: w[co 8kq .. 8kq+7][tap m][c] for taps 0..8, zero columns for m >= 9
    bf16x8 wb;
#pragma unroll
    for (int i = 0; i < 8; ++i) wb[i] = m < 9 ? w[((8 * kq + i) * 9 + m) * CIN + c] : (__bf16)0.0f;
#pragma unroll
    for (int k = 0; k < GPW; ++k) {
      const int g = wv + 4 * k;
      if (g >= NG) break;  // wave-uniform
      const f32x4 u = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k], wb, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
      if (m < 9)
        for (int i = 0; i < 4; ++i) U[(g * 16 + 4 * kq + i) * 9 + m] = u[i];
    }
    __syncthreads();
    if (oy < H && ox < W) {
      // tap t of output (ty, tx) comes from halo pixel (ty + 1 - (t/3 - 1), tx + 1 - (t%3 - 1))
      float sum = 0.0f;
#pragma unroll
      for (int t = 0; t < 9; ++t) sum += U[((ty + 2 - t / 3) * (CT + 2) + tx + 2 - t % 3) * 9 + t];
      dx[(img + (size_t)oy * W + ox) * CIN + c] = sum;
    }
  }
}

// ---------------------------------------------------------------------- weight gradients
// dW[co][t][ci] = sum_p G[p][co] X[p + off_t][ci],  db[co] = sum_p G[p][co], over every pixel p.
//
// Thin layers: 32 BF16 channels V (NHWC, zeroed where M <= 0 when M is given) against CI FP32
// channels F ([B][H][W][CI]): K[ch][t][c] = sum_p V[p][ch] F[p + off_t][c] on VALU, FP32 FMAs of the
// unrounded FP32 values.  V = the gradient and F = the input for conv1 (TAIL false: out = K, then
// db[ch] = sum V).  For conv4 (TAIL true) V = its input and F = the gradient: sum_p g[p] V[p +
// off_t] = sum_q V[q] g[q - off_t], i.e. tap 8 - t of K, out [t][ch], then db = sum of F (as two
// floats, high and low part).
// A wave walks 16x4 pixels of a 16x16 tile at a time: lane l holds channels 2(l%16) and +1 of row
// l/16, so a pixel's V is one coalesced dword per lane and its 9 F values are read from LDS rows
// into registers once per tile row; sums stay in registers over all of the block's tiles.
// 8 x 512^2 (134 MB of V): 41 us for either without M, 109 us with it; one weight per thread over
// LDS tiles: 195 and 236 us.
template <int CI, bool TAIL>
__global__ __launch_bounds__(256) void k_wgrad_thin(int H, int W, int B, const __bf16* __restrict__ V,
                                                    const __bf16* __restrict__ M, const float* __restrict__ F,
                                                    float* __restrict__ partials) {
  constexpr int NW = NCH * 9 * CI, NOUT = NW + (TAIL ? 2 : NCH);
  constexpr int FS = CT + 4;  // LDS row of F (floats): 18 columns, 16-byte multiple
  __shared__ __attribute__((aligned(16))) float sf[CI][CT + 2][FS];
  __shared__ float red[NOUT];
  [[maybe_unused]] __shared__ double red_f[4];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int cp = lane & 15, sub = lane >> 4;
  float acc[CI][2][9], accb[2] = {0.0f, 0.0f};
  // TAIL: a sum of one sign-changing value per pixel, the one output without BF16 factors: it can
  // cancel to any size, so it stays in FP64 up to the output (a block's partial is two floats)
  double sum_f = 0.0;
#pragma unroll
  for (int c = 0; c < CI; ++c)
#pragma unroll
    for (int t = 0; t < 9; ++t) acc[c][0][t] = acc[c][1][t] = 0.0f;
  const int tiles_x = (W + CT - 1) / CT, tiles_y = (H + CT - 1) / CT;
  const long ntiles = (long)tiles_x * tiles_y * B;
  for (long tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {  // uniform over the block
    const long b = tile / ((long)tiles_x * tiles_y);
    const int tr = (int)(tile - b * tiles_x * tiles_y);
    const int ty0 = (tr / tiles_x) * CT, tx0 = (tr % tiles_x) * CT;
    const size_t img = (size_t)b * H * W;
    // this lane's row of V: 16 pixels, two channels each
    const int gy = ty0 + 4 * wv + sub;
    uint32_t v[CT];
#pragma unroll
    for (int x = 0; x < CT; ++x) {
      v[x] = 0u;
      if (gy < H && tx0 + x < W) {
        const size_t off = ((img + (size_t)gy * W + tx0 + x) * NCH >> 1) + cp;
        v[x] = ((const uint32_t*)V)[off];
        if (M) {
          const uint32_t mk = ((const uint32_t*)M)[off];
          // BF16 > 0 of each half (NaN is not): the sign and magnitude as FP32
          if (!(__builtin_bit_cast(float, mk << 16) > 0.0f)) v[x] &= 0xffff0000u;
          if (!(__builtin_bit_cast(float, mk & 0xffff0000u) > 0.0f)) v[x] &= 0x0000ffffu;
        }
      }
    }
    __syncthreads();  // the previous tile's F has been read
    for (int e = threadIdx.x; e < (CT + 2) * (CT + 2) * CI; e += 256) {
      const int pix = e / CI, c = e - pix * CI;
      const int py = pix / (CT + 2), px = pix - py * (CT + 2);
      const int fy = ty0 + py - 1, fx = tx0 + px - 1;
      sf[c][py][px] = (fy >= 0 && fy < H && fx >= 0 && fx < W) ? F[(img + (size_t)fy * W + fx) * CI + c] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CI; ++c) {
      float f[3][CT + 2];
#pragma unroll
      for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int x = 0; x < CT + 2; ++x) f[r][x] = sf[c][4 * wv + sub + r][x];
#pragma unroll
      for (int x = 0; x < CT; ++x) {
        const float v0 = __builtin_bit_cast(float, v[x] << 16), v1 = __builtin_bit_cast(float, v[x] & 0xffff0000u);
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          acc[c][0][t] = fmaf(v0, f[t / 3][x + t % 3], acc[c][0][t]);
          acc[c][1][t] = fmaf(v1, f[t / 3][x + t % 3], acc[c][1][t]);
        }
        if (!TAIL && c == 0) {
          accb[0] += v0;
          accb[1] += v1;
        }
      }
      if constexpr (TAIL) {  // the row's own 16 pixels of F
#pragma unroll
        for (int x = 0; x < CT; ++x) sum_f += (gy < H && tx0 + x < W) ? (double)f[1][x + 1] : 0.0;
      }
    }
  }
  if constexpr (TAIL) {
    sum_f += __shfl_xor(sum_f, 16);
    sum_f += __shfl_xor(sum_f, 32);
    if (lane == 0) red_f[wv] = sum_f;
  }
  // the wave's four rows ((0 + 1) + (2 + 3)), then the waves in order
  auto rows = [](float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (!TAIL) accb[k] = rows(accb[k]);
#pragma unroll
    for (int c = 0; c < CI; ++c)
#pragma unroll
      for (int t = 0; t < 9; ++t) acc[c][k][t] = rows(acc[c][k][t]);
  }
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wv != w || sub != 0) continue;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int ch = 2 * cp + k;
#pragma unroll
      for (int c = 0; c < CI; ++c)
#pragma unroll
        for (int t = 0; t < 9; ++t) {
          const int o = TAIL ? (8 - t) * NCH + ch : (ch * 9 + t) * CI + c;
          red[o] = (w ? red[o] : 0.0f) + acc[c][k][t];
        }
      if constexpr (!TAIL) red[NW + ch] = (w ? red[NW + ch] : 0.0f) + accb[k];
    }
  }
  if constexpr (TAIL) {
    if (threadIdx.x == 0) {
      const double f = (red_f[0] + red_f[1]) + (red_f[2] + red_f[3]);
      red[NW] = (float)f;
      red[NW + 1] = (float)(f - (double)red[NW]);
    }
  }
  __syncthreads();
  for (int o = threadIdx.x; o < NOUT; o += 256) partials[(size_t)blockIdx.x * NOUT + o] = red[o];
}

// 32 -> 32 weight and bias gradients on MFMA: for each tap t, dW[co][t][ci] is a GEMM with M = 16
// output channels, N = 16 input channels and K = pixels (v_mfma_f32_16x16x32_bf16, K = 32 pixels
// per step); db[co] is the same GEMM against a column of ones.  The MFMA takes 8 consecutive K
// values (pixels) per lane, the activations hold a pixel's channels side by side: the tiles go to
// LDS as they are (16-byte stores) and ds_read_b64_tr_b16 transposes on the way out -- a group of 16
// lanes reads 4 pixels x 16 channels and each lane gets one channel's 4 pixels -- so a tap's shift
// is only another first pixel.  A pixel's 64 bytes are two halves of 16 channels, swapped where
// bit 1 of the pixel's index is set: any 4 consecutive pixels then cover all 32 banks once.
// Wave w of 8 takes channel block (cb, nb) = (w/2 % 2, w % 2) and K steps 4(w/4) .. +3 of every tile
// of its block (two pixel rows per step: lane group kq holds row 2s + kq/2, columns 8(kq%2) .. +7).
// The next tile is loaded into registers during this one's MFMAs.  At the end the two waves of a
// channel block are added and the block writes one partial (deterministic).
// 8 x 512^2: 82 us for the two streams' 268 MB, 102 us with M (16-bit transposing stores of three
// shifted copies: 280 us).
constexpr int WG_NOUT = NCH * 9 * NCH + NCH;
constexpr int WG_T = 512;                                       // threads
constexpr int WG_GQ = CT * CT * 4 / WG_T;                       // 16-byte quads per thread: gradient
constexpr int WG_XQ = ((CT + 2) * (CT + 2) * 4 + WG_T - 1) / WG_T;  // and input halo

typedef __attribute__((address_space(3))) __bf16 lds_bf16;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// LDS element of channel 8q of pixel pix.
__device__ __forceinline__ int wg_at(int pix, int q) { return pix * NCH + (((q >> 1) ^ (pix >> 1 & 1)) << 4) + ((q & 1) << 3); }

// 8 pixels from pix of channel block blk (16 channels), one channel per lane m of the 16-lane group.
__device__ __forceinline__ bf16x8 wg_read(const __bf16* s, int pix, int blk, int m) {
  const int p0 = pix + (m >> 2), p1 = p0 + 4;
  const int c = (m & 3) << 2;
  union { s16x4 h[2]; bf16x8 v; } u;
  u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(s + p0 * NCH + ((blk ^ (p0 >> 1 & 1)) << 4) + c));
  u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(s + p1 * NCH + ((blk ^ (p1 >> 1 & 1)) << 4) + c));
  return u.v;
}

__global__ __launch_bounds__(WG_T, 4) void k_wgrad32_mfma(int H, int W, int B, const __bf16* __restrict__ G,
                                                          const __bf16* __restrict__ M,
                                                          const __bf16* __restrict__ X,
                                                          float* __restrict__ partials) {
  constexpr int GE = CT * CT * NCH, XE = (CT + 2) * (CT + 2) * NCH;
  __shared__ __attribute__((aligned(16))) __bf16 sg[GE + XE];
  __bf16* sx = sg + GE;
  static_assert(sizeof(__bf16) * (GE + XE) >= sizeof(float) * WG_NOUT, "reduction buffer");
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int m = lane & 15, kq = lane >> 4;
  const int cb = wv >> 1 & 1, nb = wv & 1, half = wv >> 2;
  f32x4 acc[9], accb = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.0f;
  const int tiles_x = (W + CT - 1) / CT, tiles_y = (H + CT - 1) / CT;
  const long ntiles = (long)tiles_x * tiles_y * B;
  bf16x8 pg[WG_GQ], px[WG_XQ];
  auto load = [&](long tile) {
    const long b = tile / ((long)tiles_x * tiles_y);
    const int tr = (int)(tile - b * tiles_x * tiles_y);
    const int ty0 = (tr / tiles_x) * CT, tx0 = (tr % tiles_x) * CT;
    const size_t img = (size_t)b * H * W;
#pragma unroll
    for (int k = 0; k < WG_GQ; ++k) {
      const int c = threadIdx.x + WG_T * k, pix = c >> 2, q = c & 3;
      const int gy = ty0 + (pix >> 4), gx = tx0 + (pix & 15);
      bf16x8 v;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (__bf16)0.0f;
      if (gy < H && gx < W) {
        const size_t off = (img + (size_t)gy * W + gx) * NCH + 8 * q;
        v = *(const bf16x8*)(G + off);
        if (M) {
          const bf16x8 mk = *(const bf16x8*)(M + off);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (!((float)mk[i] > 0.0f)) v[i] = (__bf16)0.0f;
        }
      }
      pg[k] = v;
    }
#pragma unroll
    for (int k = 0; k < WG_XQ; ++k) {
      const int c = threadIdx.x + WG_T * k, pix = c >> 2, q = c & 3;
      const int hy = pix / (CT + 2), hx = pix - hy * (CT + 2);
      const int gy = ty0 + hy - 1, gx = tx0 + hx - 1;
      bf16x8 v;
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = (__bf16)0.0f;
      if (pix < (CT + 2) * (CT + 2) && gy >= 0 && gy < H && gx >= 0 && gx < W)
        v = *(const bf16x8*)(X + (img + (size_t)gy * W + gx) * NCH + 8 * q);
      px[k] = v;
    }
  };
  long tile = blockIdx.x;
  if (tile < ntiles) load(tile);
  for (; tile < ntiles; tile += gridDim.x) {  // uniform over the block
    __syncthreads();                          // the previous tile's LDS reads are done
#pragma unroll
    for (int k = 0; k < WG_GQ; ++k) {
      const int c = threadIdx.x + WG_T * k;
      *(bf16x8*)(sg + wg_at(c >> 2, c & 3)) = pg[k];
    }
#pragma unroll
    for (int k = 0; k < WG_XQ; ++k) {
      const int c = threadIdx.x + WG_T * k;
      if ((c >> 2) < (CT + 2) * (CT + 2)) *(bf16x8*)(sx + wg_at(c >> 2, c & 3)) = px[k];
    }
    __syncthreads();
    if (tile + gridDim.x < ntiles) load(tile + gridDim.x);  // in flight during the MFMAs
#pragma unroll
    for (int ss = 0; ss < 4; ++ss) {
      const int py = 2 * (4 * half + ss) + (kq >> 1), px0 = (kq & 1) * 8;
      // A: gradient of output channels cb*16 + m at the 8 pixels (py, px0 .. px0 + 7)
      const bf16x8 a = wg_read(sg, py * CT + px0, cb, m);
      if (nb == 0) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, accb, 0, 0, 0);  // wave-uniform
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        // B: input channel nb*16 + m at the same pixels shifted by the tap
        const bf16x8 bv = wg_read(sx, (py + t / 3) * (CT + 2) + px0 + t % 3, nb, m);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv, acc[t], 0, 0, 0);
      }
    }
  }
  // C: lane (m, kq) holds rows 4kq + i (output channels cb*16 + 4kq + i) of column m (input
  // channel nb*16 + m).  The waves of K steps 4..7 go through LDS to those of 0..3.
  float* red = (float*)sg;
  float* out = partials + (size_t)blockIdx.x * WG_NOUT;
  __syncthreads();
#pragma unroll
  for (int ph = 0; ph < 2; ++ph) {
    if (half == 1 - ph) {
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int o = ((cb * 16 + 4 * kq + i) * 9 + t) * NCH + nb * 16 + m;
          if (ph == 0)
            red[o] = acc[t][i];
          else
            out[o] = acc[t][i] + red[o];
        }
      if (nb == 0 && m == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int o = NCH * 9 * NCH + cb * 16 + 4 * kq + i;
          if (ph == 0)
            red[o] = accb[i];
          else
            out[o] = accb[i] + red[o];
        }
    }
    if (ph == 0) __syncthreads();
  }
}

// out[o] = sum over blocks b of partials[b][o], rows of `row` floats (nout, or nout + 1 with the last
// output's low parts behind it), in a fixed order (deterministic): a workgroup of 1024
// threads takes OUTS consecutive outputs (coalesced rows of the partials); strand s of 1024/OUTS
// sums the blocks b = s, s + strands, ..., eight loads in flight, then the strands' sums are added
// in order.  OUTS = 64 for the 9248 outputs of the 32 -> 32 layers, 16 for the few hundred of the
// thin ones (512 blocks x 9248 outputs: 5.0 us; before, with 64 outputs and four strands a workgroup,
// 42 us on average over a training step's calls).
template <int OUTS>
__global__ __launch_bounds__(1024) void k_reduce_partials(const float* __restrict__ partials, int nblocks,
                                                          int nout, int row, float* __restrict__ out) {
  constexpr int STR = 1024 / OUTS;
  __shared__ double sh[STR][OUTS];
  const int c = threadIdx.x % OUTS, r = threadIdx.x / OUTS;
  const int o = blockIdx.x * OUTS + c;
  double s = 0.0;  // FP64: the sums of a bias gradient cancel, and the adds hide behind the loads
  auto column = [&](int col) {
    int b = r;
    for (; b + 7 * STR < nblocks; b += 8 * STR) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = partials[(size_t)(b + k * STR) * row + col];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += (double)v[k];
    }
    for (; b < nblocks; b += STR) s += (double)partials[(size_t)b * row + col];
  };
  if (o < nout) {
    column(o);
    if (o == nout - 1 && row > nout) column(nout);
  }
  sh[r][c] = s;
  __syncthreads();
  if (r == 0 && o < nout) {
    double t = sh[0][c];
    for (int k = 1; k < STR; ++k) t += sh[k][c];
    out[o] = (float)t;
  }
}

// ---------------------------------------------------------------------- phantoms
// params[b][e] = (cx, cy, a, b, cos t, sin t, value); pixel centres at (2j+1)/N - 1.
__global__ __launch_bounds__(256) void k_phantom(int N, int E, long npix, const double* __restrict__ params,
                                                 float* __restrict__ out) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  if (p >= npix) return;
  const long b = p / ((long)N * N);
  const int r = (int)(p - b * N * N);
  const int i = r / N, j = r - i * N;
  const double x = (2.0 * j + 1.0) / N - 1.0, y = (2.0 * i + 1.0) / N - 1.0;
  double acc = 0.0;
  const double* P = params + b * E * 7;
  for (int e = 0; e < E; ++e) {
    const double* q = P + e * 7;
    const double dx = x - q[0], dy = y - q[1];
    const double u = (dx * q[4] + dy * q[5]) / q[2];
    const double w = (-dx * q[5] + dy * q[4]) / q[3];
    acc += (u * u + w * w <= 1.0) ? q[6] : 0.0;
  }
  acc = acc < 0.0 ? 0.0 : (acc > 1.0 ? 1.0 : acc);
  out[p] = (float)acc;
}

}  // namespace sk

using namespace sk;

static int check_ctx(sk_ctx* ctx) {
  if (!ctx) return SK_EINVAL;
  SK_HIP(&ctx->c, hipSetDevice(ctx->c.device));
  return SK_OK;
}

extern "C" {

static int conv32_go(sk_ctx* ctx, int B, int H, int W, const void* x, const void* mask, const void* w,
                     const float* bias, void* y, const void* omask, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (B < 1 || B > 65535 || H < 1 || W < 1 || !x || !w || !y)
    return fail(&ctx->c, SK_EINVAL, "conv32: bad arguments");
  const bool relu = bias != nullptr;
  const long ntiles = (long)((W + CT - 1) / CT) * ((H + CT - 1) / CT) * B;
  // persistent grid: the resident blocks of the chip (queried once per process and device)
  static int per_cu[64] = {0}, cus[64] = {0};
  const int dev = ctx->c.device < 64 ? ctx->c.device : 63;
  if (!per_cu[dev]) {
    SK_HIP(&ctx->c, hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, ctx->c.device));
    SK_HIP(&ctx->c, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu[dev], k_conv32<true, true>, 256, 0));
    per_cu[dev] = std::max(1, per_cu[dev]);
  }
  const long resident = (long)cus[dev] * per_cu[dev];
  dim3 grid((unsigned)std::min(ntiles, resident));
  hipStream_t s = (hipStream_t)stream;
  const __bf16 *X = (const __bf16*)x, *Mk = (const __bf16*)mask, *Wt = (const __bf16*)w, *Om = (const __bf16*)omask;
  __bf16* Y = (__bf16*)y;
  if (omask)
    hipLaunchKernelGGL((k_conv32<false, false, true>), grid, dim3(256), 0, s, H, W, ntiles, X, Mk, Wt, bias, Y, Om);
  else if (mask && relu)
    hipLaunchKernelGGL((k_conv32<true, true>), grid, dim3(256), 0, s, H, W, ntiles, X, Mk, Wt, bias, Y, Om);
  else if (mask)
    hipLaunchKernelGGL((k_conv32<true, false>), grid, dim3(256), 0, s, H, W, ntiles, X, Mk, Wt, bias, Y, Om);
  else if (relu)
    hipLaunchKernelGGL((k_conv32<false, true>), grid, dim3(256), 0, s, H, W, ntiles, X, Mk, Wt, bias, Y, Om);
  else
    hipLaunchKernelGGL((k_conv32<false, false>), grid, dim3(256), 0, s, H, W, ntiles, X, Mk, Wt, bias, Y, Om);
  return launched(&ctx->c, "conv32 kernel");
}

int sk_conv32(sk_ctx* ctx, int B, int H, int W, const void* x, const void* mask, const void* w,
              const float* bias, void* y, void* stream) {
  return conv32_go(ctx, B, H, W, x, mask, w, bias, y, nullptr, stream);
}

int sk_conv32_dgrad_relu(sk_ctx* ctx, int B, int H, int W, const void* g, const void* w, const void* h, void* dh,
                         void* stream) {
  if (ctx && !h) return fail(&ctx->c, SK_EINVAL, "conv32_dgrad_relu: bad arguments");
  return conv32_go(ctx, B, H, W, g, nullptr, w, nullptr, dh, h, stream);
}

static int conv_in_go(sk_ctx* ctx, int cin, int B, int H, int W, const float* x, const void* w, const float* bias,
                      void* h, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (B < 1 || H < 1 || W < 1 || !x || !w || !bias || !h) return fail(&ctx->c, SK_EINVAL, "conv_in: bad arguments");
  if (B > 65535 || (long)H * W >= (1L << 31)) return fail(&ctx->c, SK_EINVAL, "conv_in: batch or image too large");
  if ((uintptr_t)w % 4) return fail(&ctx->c, SK_EINVAL, "conv_in: weights must be 4-byte aligned");
  const dim3 grid((unsigned)((H * W + 255) / 256), B);
  if (cin == 1)
    hipLaunchKernelGGL(k_conv_in<1>, grid, dim3(256), 0, (hipStream_t)stream, H, W, x, (const uint32_t*)w, bias,
                       (__bf16*)h);
  else
    hipLaunchKernelGGL(k_conv_in<2>, grid, dim3(256), 0, (hipStream_t)stream, H, W, x, (const uint32_t*)w, bias,
                       (__bf16*)h);
  return launched(&ctx->c, "conv_in kernel");
}

int sk_conv_in(sk_ctx* ctx, int B, int H, int W, const float* x, const void* w, const float* bias,
               void* h, void* stream) {
  return conv_in_go(ctx, 1, B, H, W, x, w, bias, h, stream);
}

int sk_conv_in2(sk_ctx* ctx, int B, int H, int W, const float* x2, const void* w, const float* bias,
                void* h, void* stream) {
  return conv_in_go(ctx, 2, B, H, W, x2, w, bias, h, stream);
}

int sk_conv_out(sk_ctx* ctx, int B, int H, int W, const void* h, const void* w, const float* bias,
                const float* res, float* y, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (B < 1 || H < 1 || W < 1 || !h || !w || !bias || !res || !y)
    return fail(&ctx->c, SK_EINVAL, "conv_out: bad arguments");
  if (B > 65535) return fail(&ctx->c, SK_EINVAL, "conv_out: batch must be <= 65535");
  dim3 grid(((W + CT - 1) / CT) * ((H + CT - 1) / CT), B);
  hipLaunchKernelGGL(k_conv_out_mfma, grid, dim3(256), 0, (hipStream_t)stream, H, W, (const __bf16*)h,
                     (const __bf16*)w, bias, res, y);
  return launched(&ctx->c, "conv_out kernel");
}

static int conv_out_dgrad_go(sk_ctx* ctx, int B, int H, int W, const float* g, const void* w, const void* h,
                             void* dh, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (B < 1 || H < 1 || W < 1 || !g || !w || !dh) return fail(&ctx->c, SK_EINVAL, "conv_out_dgrad: bad arguments");
  const long npix = (long)B * H * W;
  const dim3 grid((unsigned)((npix + 255) / 256));
  if (h)
    hipLaunchKernelGGL(k_conv_out_dgrad<true>, grid, dim3(256), 0, (hipStream_t)stream, H, W, npix, g,
                       (const __bf16*)w, (__bf16*)dh, (const __bf16*)h);
  else
    hipLaunchKernelGGL(k_conv_out_dgrad<false>, grid, dim3(256), 0, (hipStream_t)stream, H, W, npix, g,
                       (const __bf16*)w, (__bf16*)dh, (const __bf16*)nullptr);
  return launched(&ctx->c, "conv_out_dgrad kernel");
}

int sk_conv_out_dgrad(sk_ctx* ctx, int B, int H, int W, const float* g, const void* w, void* dh,
                      void* stream) {
  return conv_out_dgrad_go(ctx, B, H, W, g, w, nullptr, dh, stream);
}

int sk_conv_out_dgrad_relu(sk_ctx* ctx, int B, int H, int W, const float* g, const void* w, const void* h, void* dh,
                           void* stream) {
  if (ctx && !h) return fail(&ctx->c, SK_EINVAL, "conv_out_dgrad_relu: bad arguments");
  return conv_out_dgrad_go(ctx, B, H, W, g, w, h, dh, stream);
}

}  // extern "C"

template <bool MASK>
static int conv_in_dgrad_go(sk_ctx* ctx, int cin, int B, int H, int W, const void* dh, const void* hmask,
                            const void* w, float* dx, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (cin < 1 || cin > 2 || B < 1 || H < 1 || W < 1 || !dh || (MASK && !hmask) || !w || !dx)
    return fail(&ctx->c, SK_EINVAL, "conv_in_dgrad: bad arguments");
  const long ntiles = (long)((W + CT - 1) / CT) * ((H + CT - 1) / CT) * B;
  const long across = std::min(ntiles, 1L << 22);  // a dimension of a launch holds fewer than 2^32 threads
  const dim3 grid((unsigned)across, (unsigned)((ntiles + across - 1) / across));
  if (cin == 1)
    hipLaunchKernelGGL((k_conv_in_dgrad<1, MASK>), grid, dim3(256), 0, (hipStream_t)stream, H, W, ntiles,
                       (const __bf16*)dh, (const __bf16*)hmask, (const __bf16*)w, dx);
  else
    hipLaunchKernelGGL((k_conv_in_dgrad<2, MASK>), grid, dim3(256), 0, (hipStream_t)stream, H, W, ntiles,
                       (const __bf16*)dh, (const __bf16*)hmask, (const __bf16*)w, dx);
  return launched(&ctx->c, "conv_in_dgrad kernel");
}

extern "C" {

int sk_conv_in_dgrad(sk_ctx* ctx, int B, int H, int W, const void* dh, const void* hmask,
                     const void* w, float* dx, void* stream) {
  return conv_in_dgrad_go<true>(ctx, 1, B, H, W, dh, hmask, w, dx, stream);
}

int sk_conv_in2_dgrad(sk_ctx* ctx, int B, int H, int W, const void* dh, const void* hmask,
                      const void* w, float* dx2, void* stream) {
  return conv_in_dgrad_go<true>(ctx, 2, B, H, W, dh, hmask, w, dx2, stream);
}

int sk_conv_in_dgrad_relu(sk_ctx* ctx, int cin, int B, int H, int W, const void* g, const void* w, float* dx,
                          void* stream) {
  return conv_in_dgrad_go<false>(ctx, cin, B, H, W, g, nullptr, w, dx, stream);
}

// kind 0: conv1 (G = 32-ch gradient masked by h1, X = fp32 image) -> dW [32][9], db [32]
// kind 1: conv2/3 (G masked, X = 32-ch activation)                  -> dW [32][9][32], db [32]
// kind 2: conv4 (G = fp32 image gradient, X = 32-ch activation)     -> dW [9][32], db [1]
// kind 3: conv1 with two input channels (G masked, X = fp32 [B][H][W][2]) -> dW [32][9][2], db [32]
// out: CO*9*CI weight gradients followed by CO bias gradients (fp32).
int sk_conv_wgrad(sk_ctx* ctx, int kind, int B, int H, int W, const void* g, const void* mask,
                  const void* x, float* out, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  Ctx* c = &ctx->c;
  if (B < 1 || H < 1 || W < 1 || !g || !x || !out || kind < 0 || kind > 3)
    return fail(c, SK_EINVAL, "conv_wgrad: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  const long ntiles = (long)((W + CT - 1) / CT) * ((H + CT - 1) / CT) * B;
  // one resident set of blocks, each with one partial (queried once per device)
  static int cus[64] = {0};
  const int dev = c->device < 64 ? c->device : 63;
  if (!cus[dev])
    SK_HIP(c, hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, c->device));
  const long cap = kind == 1 ? 2L * cus[dev] : 4L * cus[dev];
  const int nblocks = (int)std::min<long>(ntiles, cap);
  const int nout = kind == 0 ? NCH * 9 + NCH
                             : (kind == 1 ? NCH * 9 * NCH + NCH : (kind == 2 ? 9 * NCH + 1 : NCH * 9 * 2 + NCH));
  const int row = nout + (kind == 2 ? 1 : 0);  // floats of a block's partial
  void* ws = nullptr;
  rc = scratch(c, sizeof(float) * (size_t)nblocks * row, s, &ws);
  if (rc) return rc;
  float* part = (float*)ws;
  const __bf16* Mk = (const __bf16*)mask;
  if (kind == 0)
    hipLaunchKernelGGL((k_wgrad_thin<1, false>), dim3(nblocks), dim3(256), 0, s, H, W, B, (const __bf16*)g, Mk,
                       (const float*)x, part);
  else if (kind == 1)
    hipLaunchKernelGGL(k_wgrad32_mfma, dim3(nblocks), dim3(WG_T), 0, s, H, W, B, (const __bf16*)g, Mk,
                       (const __bf16*)x, part);
  else if (kind == 2)
    hipLaunchKernelGGL((k_wgrad_thin<1, true>), dim3(nblocks), dim3(256), 0, s, H, W, B, (const __bf16*)x,
                       (const __bf16*)nullptr, (const float*)g, part);
  else
    hipLaunchKernelGGL((k_wgrad_thin<2, false>), dim3(nblocks), dim3(256), 0, s, H, W, B, (const __bf16*)g, Mk,
                       (const float*)x, part);
  rc = launched(c, "wgrad kernel");
  if (rc) return rc;
  if (nout > 1024)
    hipLaunchKernelGGL(k_reduce_partials<64>, dim3((nout + 63) / 64), dim3(1024), 0, s, part, nblocks, nout, row,
                       out);
  else
    hipLaunchKernelGGL(k_reduce_partials<16>, dim3((nout + 15) / 16), dim3(1024), 0, s, part, nblocks, nout, row,
                       out);
  return launched(c, "partials reduction kernel");
}

int sk_phantoms(sk_ctx* ctx, int B, int N, int E, const double* d_params, float* d_out, void* stream) {
  int rc = check_ctx(ctx);
  if (rc) return rc;
  if (B < 1 || N < 1 || E < 0 || !d_params || !d_out) return fail(&ctx->c, SK_EINVAL, "phantoms: bad arguments");
  const long npix = (long)B * N * N;
  hipLaunchKernelGGL(k_phantom, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0, (hipStream_t)stream, N, E,
                     npix, d_params, d_out);
  return launched(&ctx->c, "phantom kernel");
}

}  // extern "C"
