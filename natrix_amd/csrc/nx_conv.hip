// 3x3 convolution staged in LDS (gfx950): the training path's forward and input
// gradient, wherever no split of K and no tiled weights are asked for and the
// image is more than a few pixels (conv3x3_lds has the line).
// Layouts and arithmetic as in nx_unet.hip: NHWC bfloat16 activations, KRSC
// bfloat16 weights, and for every output the chain of v_mfma_f32_32x32x16_bf16
// over the K steps in order (16 channels of one tap, taps outermost), so the
// results are bitwise those of k_conv3x3.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/natrix.h"
#include "nx_common.h"
#include "nx_conv.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// A block of 4 waves makes TH rows x 16 columns of pixels (TH = 16 / WN) by
// 32 NT WN output channels; a wave makes 64 pixels x 32 NT channels, 2 NT
// MFMAs per K step from 2 + NT fragments.  The pixels' surround is staged in
// LDS once for all taps, [pixel][channel] with 16 bytes between pixels (an odd
// multiple of 16 bytes, so that 8 lanes' 16-byte reads fall on different
// banks), zero beyond the image; the weights go through LDS in chunks of CH K
// steps, which are contiguous in the KRSC rows, double buffered, one barrier a
// chunk.  The outputs leave through LDS in 16-byte stores.
// WN = 2 halves the staged pixels where the channels are many; the whole
// depth has to fit, since the taps are the outer loop of the sum.
// Bound: LDS reads, 4 KiB per wave and K step against 128 MFMA cycles; two
// blocks per CU overlap one's staging with the other's products.  32 x 64 x 64
// pixels, 64 -> 64 channels: 24 us (400 TFLOP/s), where loading each fragment
// from the caches, once per tap, took 51; 192 -> 64 on the same pixels, one
// block per CU: 118 us.
template <int CPS, int NT, int WN, int CH>
struct ConvShape {
  static constexpr int TH = 16 / WN, XW = 18, XP = (TH + 2) * XW;
  static constexpr int XS = CPS * 16 + 8;  // halfwords from pixel to pixel
  static constexpr int BS = CH * 16 + 8;   // halfwords from output channel to output channel
  static constexpr int CO = 32 * NT * WN;
  static constexpr int OS = 32 * NT + 8;   // halfwords from pixel to pixel of a wave's output
  static constexpr int LDS_IN = XP * XS + 2 * CO * BS, LDS_OUT = 4 * 64 * OS;
  static constexpr int BYTES = 2 * (LDS_IN > LDS_OUT ? LDS_IN : LDS_OUT);
  static_assert(9 * CPS % CH == 0, "whole chunks");
  static_assert(BYTES <= 160 * 1024, "LDS of a compute unit");
};

template <int CPS, int NT, int WN, int CH>
__global__ void __launch_bounds__(256, 2)
    k_conv3x3_lds(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                  const float* __restrict__ bias, uint16_t* __restrict__ y, int H, int W,
                  int Cout, int relu, int tiles_x, int tiles_img) {
  using S = ConvShape<CPS, NT, WN, CH>;
  constexpr int Cin = CPS * 16, K = 9 * Cin;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  uint16_t* lx = lds;
  uint16_t* lw = lds + S::XP * S::XS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wp = wave / WN, wn = wave % WN;
  const int r = lane & 31, kb = lane >> 5;
  const int img = blockIdx.x / tiles_img, rem = blockIdx.x - img * tiles_img;
  const int y0 = rem / tiles_x * S::TH, x0 = rem % tiles_x * 16;
  const int co0 = blockIdx.y * S::CO;
  const long long pix0 = (long long)img * H * W;

  // weights: 16-byte chunks, CH * 2 per output channel
  constexpr int WCHUNKS = S::CO * CH * 2, WJ = (WCHUNKS + 255) / 256;
  uint4 rw[WJ];
  auto load_w = [&](int c) {
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int q = threadIdx.x + 256 * j;
      if (WCHUNKS % 256 == 0 || q < WCHUNKS)
        rw[j] = *reinterpret_cast<const uint4*>(w + (long long)(co0 + q / (CH * 2)) * K +
                                                c * CH * 16 + (q % (CH * 2)) * 8);
    }
  };
  auto store_w = [&](int buf) {
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int q = threadIdx.x + 256 * j;
      if (WCHUNKS % 256 == 0 || q < WCHUNKS)
        *reinterpret_cast<uint4*>(lw + buf * S::CO * S::BS + q / (CH * 2) * S::BS +
                                  (q % (CH * 2)) * 8) = rw[j];
    }
  };
  load_w(0);

  constexpr int XCHUNKS = S::XP * CPS * 2, BATCH = 8;
  for (int q0 = 0; q0 < XCHUNKS; q0 += 256 * BATCH) {
    uint4 v[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const int q = q0 + threadIdx.x + 256 * j, px = q / (CPS * 2);
      const int yy = y0 + px / S::XW - 1, xx = x0 + px % S::XW - 1;
      v[j] = make_uint4(0, 0, 0, 0);
      if (q < XCHUNKS && yy >= 0 && yy < H && xx >= 0 && xx < W)
        v[j] = *reinterpret_cast<const uint4*>(x + (pix0 + (long long)yy * W + xx) * Cin +
                                               (q % (CPS * 2)) * 8);
    }
#pragma unroll
    for (int j = 0; j < BATCH; ++j) {
      const int q = q0 + threadIdx.x + 256 * j;
      if (q < XCHUNKS)
        *reinterpret_cast<uint4*>(lx + q / (CPS * 2) * S::XS + (q % (CPS * 2)) * 8) = v[j];
    }
  }
  store_w(0);
  __syncthreads();

  f32x16 acc[2][NT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // fragment i: rows 4 wp + 2 i + r / 16, column r % 16
  const uint16_t* xa = lx + ((4 * wp + (r >> 4)) * S::XW + (r & 15)) * S::XS + kb * 8;
  const uint16_t* wb = lw + (32 * NT * wn + r) * S::BS + kb * 8;
  constexpr int CHUNKS = 9 * CPS / CH;
  for (int c = 0; c < CHUNKS; ++c) {
    if (c + 1 < CHUNKS) load_w(c + 1);
    const uint16_t* wc = wb + (c & 1) * S::CO * S::BS;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int ks = c * CH + j, tap = ks / CPS, s = ks - tap * CPS;
      const int off = (tap / 3 * S::XW + tap % 3) * S::XS + s * 16;
      bf16x8 a[2], b[NT];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(xa + off + 2 * i * S::XW * S::XS);
#pragma unroll
      for (int n = 0; n < NT; ++n)
        b[n] = *reinterpret_cast<const bf16x8*>(wc + 32 * n * S::BS + j * 16);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n)
          acc[i][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[n], acc[i][n], 0, 0, 0);
    }
    if (c + 1 < CHUNKS) store_w((c + 1) & 1);
    __syncthreads();
  }

  // out through LDS: [64 pixels of the wave][32 NT channels]
  uint16_t* lo = lds + wave * 64 * S::OS;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const int co = 32 * n + r;
      const float bv = bias ? bias[co0 + 32 * NT * wn + co] : 0.0f;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float v = acc[i][n][e] + bv;
        if (relu) v = fmaxf(v, 0.0f);
        lo[(32 * i + 8 * (e >> 2) + 4 * kb + (e & 3)) * S::OS + co] =
            (uint16_t)nx::f32_to_bf16(v);
      }
    }
  __syncthreads();
  constexpr int OC = 4 * NT;  // 16-byte chunks of a pixel
#pragma unroll
  for (int j = 0; j < OC; ++j) {
    const int q = lane + 64 * j, px = q / OC, ch = (q % OC) * 8;
    const int yy = y0 + 4 * wp + (px >> 4), xx = x0 + (px & 15);
    if (yy < H && xx < W)
      *reinterpret_cast<uint4*>(y + (pix0 + (long long)yy * W + xx) * Cout + co0 + 32 * NT * wn +
                                ch) = *reinterpret_cast<const uint4*>(lo + px * S::OS + ch);
  }
}

template <int CPS, int NT, int WN, int CH>
hipError_t launch(const uint16_t* x, const uint16_t* w, const float* bias, uint16_t* y, int n,
                  int h, int wd, int cout, int relu, hipStream_t s) {
  using S = ConvShape<CPS, NT, WN, CH>;
  const int tx = (wd + 15) / 16, ti = tx * ((h + S::TH - 1) / S::TH);
  if (S::BYTES > 65536) {
    const hipError_t e = hipFuncSetAttribute(
        reinterpret_cast<const void*>(&k_conv3x3_lds<CPS, NT, WN, CH>),
        hipFuncAttributeMaxDynamicSharedMemorySize, S::BYTES);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((unsigned)((long long)n * ti), cout / S::CO);
  k_conv3x3_lds<CPS, NT, WN, CH>
      <<<grid, 256, S::BYTES, s>>>(x, w, bias, y, h, wd, cout, relu, tx, ti);
  return hipGetLastError();
}

}  // namespace

namespace nx {

bool conv3x3_lds(const uint16_t* x, const uint16_t* w, const float* bias, uint16_t* y, int n,
                 int h, int wd, int cin, int cout, int relu, hipStream_t s, hipError_t* err) {
  if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) != 0) return false;
  if ((long long)n * ((h + 7) / 8) * ((wd + 15) / 16) > 0x7FFFFFFF) return false;
  // A few pixels: k_conv3x3, whose waves take 32 or 64 of them, starts on its
  // first fragments while a block here still stages the weights of 128 channels
  // or more.  us with k_conv3x3 / here, at 16, 48 and 64 pixels: 128 -> 128
  // channels 25.4 / 28.6, 30.1 / 28.9, 33.1 / 28.8; 256 -> 256 45.0 / 54.5,
  // 50.7 / 54.6, 54.6 / 54.7.  With 32 to 96 channels (64 -> 64: 13.3 / 12.3 at
  // one pixel) and with 192 and 384 (384 -> 128: 62 / 50) staging wins from one
  // pixel on.
  if ((cin == 128 || cin == 256) && (long long)n * h * wd * 3 <= cin) return false;
  const bool n2 = cout % 64 == 0, n4 = cout % 128 == 0;
#define NX_CONV(CPS, NT, WN, CH) \
  return *err = launch<CPS, NT, WN, CH>(x, w, bias, y, n, h, wd, cout, relu, s), true
  switch (cin) {
    case 32:
      if (n2) NX_CONV(2, 2, 1, 6);
      NX_CONV(2, 1, 1, 6);
    case 64:
      if (n2) NX_CONV(4, 2, 1, 6);
      NX_CONV(4, 1, 1, 6);
    case 96:
      if (n2) NX_CONV(6, 2, 1, 6);
      NX_CONV(6, 1, 1, 6);
    case 128:
      if (n4) NX_CONV(8, 2, 2, 6);
      if (n2) NX_CONV(8, 1, 2, 6);
      NX_CONV(8, 1, 1, 6);
    case 192:
      if (n4) NX_CONV(12, 2, 2, 6);
      if (n2) NX_CONV(12, 1, 2, 6);
      return false;
    case 256:
      if (n4) NX_CONV(16, 2, 2, 6);
      if (n2) NX_CONV(16, 1, 2, 6);
      return false;
    case 384:
      if (n2) NX_CONV(24, 1, 2, 4);
      return false;
    default:
      return false;
  }
#undef NX_CONV
}

}  // namespace nx
