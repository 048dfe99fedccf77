// Backward kernels of the U-Net's layers (gfx950): the 3x3 convolution's
// weight gradient, ReLU's gradient with the bias gradient, column sums and
// the head's backward.  Layouts as in nx_unet.hip: NHWC bfloat16
// activations, float32 gradients of the parameters.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/natrix.h"
#include "nx_common.h"

namespace nx {
int set_error(int code, const std::string& msg);
}

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ __forceinline__ float bf(uint16_t h) { return nx::bf16_to_f32(h); }
__device__ __forceinline__ uint16_t tobf(float f) { return (uint16_t)nx::f32_to_bf16(f); }

// ------------------------------------------------------------- sum of splits
// out[i] = sum over s of part[s n + i], in a fixed order: a block of 1024
// threads takes 1024 / G elements, its G thread groups add the splits g,
// g + G, ... and the group sums are added pairwise in LDS.  Each thread's
// loads are independent, so a sum is a few memory round trips long whatever
// the number of splits (one thread walking 1024 records of a 64-channel
// bias gradient took 122 us; this takes 5).
__global__ void __launch_bounds__(1024)
    k_sum_splits(const float* __restrict__ part, float* __restrict__ out, long long n,
                 int splits, int lg) {
  __shared__ float acc[1024];
  const int el = threadIdx.x & ((1024 >> lg) - 1), g = threadIdx.x >> (10 - lg);
  const int G = 1 << lg;
  const long long i = (long long)blockIdx.x * (1024 >> lg) + el;
  float s = 0.0f;
  if (i < n) {
    int k = g;
    for (; k + 3 * G < splits; k += 4 * G) {
      const float a = part[(long long)k * n + i], b = part[(long long)(k + G) * n + i];
      const float c = part[(long long)(k + 2 * G) * n + i];
      const float d = part[(long long)(k + 3 * G) * n + i];
      s += (a + b) + (c + d);
    }
    for (; k < splits; k += G) s += part[(long long)k * n + i];
  }
  acc[threadIdx.x] = s;
  for (int h = G >> 1; h > 0; h >>= 1) {
    __syncthreads();
    if (g < h) acc[threadIdx.x] += acc[threadIdx.x + h * (1024 >> lg)];
  }
  if (g == 0 && i < n) out[i] = acc[threadIdx.x];
}

// groups: as many as there are splits (a power of two, at most 32, so that a
// group still reads 128 consecutive bytes)
void launch_sum_splits(const float* part, float* out, long long n, int splits, hipStream_t s) {
  int lg = 0;
  while (lg < 5 && (2 << lg) <= splits) ++lg;
  const long long per = 1024 >> lg;
  k_sum_splits<<<(unsigned)((n + per - 1) / per), 1024, 0, s>>>(part, out, n, splits, lg);
}

// ---------------------------------------------------------------- row passes
// One pass over a (rows x C) matrix that leaves per-block column sums in
// part[block][C (+ 1)]; V consecutive channels per thread (8: one 16-byte
// access, for C % 8 == 0; else 1).
//   SUM_PLAIN  column sums of a
//   SUM_RELU   dz = dy where y > 0 else 0, written, and its column sums (the
//              bias gradient), in one pass: dz is read where it is made
//   SUM_HEAD   dx[p][c] = dout[p] w[c], column sums of dout[p] x[p][c] and,
//              as column C, of dout: that one in pixel order, since under a
//              mean-free loss it is a sum of opposites, all round-off, and
//              its value is the order's
// Memory bound: SUM_RELU moves 6 bytes a value; 131072 x 64 in 12 us, where a
// ReLU pass and a column-sum pass of one row per block step took 18 + 32.
enum { SUM_PLAIN = 0, SUM_RELU = 1, SUM_HEAD = 2 };

template <int MODE, int V>
__global__ void __launch_bounds__(256)
    k_rows(const uint16_t* __restrict__ a, const uint16_t* __restrict__ dy,
           uint16_t* __restrict__ dz, const float* __restrict__ w,
           const float* __restrict__ dout, float* __restrict__ part, long long rows, int C,
           long long rows_per_block) {
  extern __shared__ float acc[];  // [groups][C], groups > 1
  const int cg = C / V;           // channel groups of a row
  const int gang = cg < 256 ? cg : 256;
  const int groups = 256 / gang;  // rows a block works on at once
  const int g = threadIdx.x / gang, c0 = threadIdx.x - g * gang;
  const int width = MODE == SUM_HEAD ? C + 1 : C;
  const long long r0 = blockIdx.x * rows_per_block;
  const long long r1 = r0 + rows_per_block < rows ? r0 + rows_per_block : rows;
  if (g < groups) {
    for (int c = c0; c < cg; c += gang) {
      float s[V], wv[V];
#pragma unroll
      for (int j = 0; j < V; ++j) {
        s[j] = 0.0f;
        wv[j] = MODE == SUM_HEAD ? w[c * V + j] : 0.0f;
      }
#pragma unroll 4
      for (long long r = r0 + g; r < r1; r += groups) {
        const long long at = r * C + (long long)c * V;
        uint16_t av[V], yv[V], ov[V];
        if (V == 8) {
          *reinterpret_cast<uint4*>(av) = *reinterpret_cast<const uint4*>(a + at);
          if (MODE == SUM_RELU)
            *reinterpret_cast<uint4*>(yv) = *reinterpret_cast<const uint4*>(dy + at);
        } else {
          av[0] = a[at];
          if (MODE == SUM_RELU) yv[0] = dy[at];
        }
        const float d = MODE == SUM_HEAD ? dout[r] : 0.0f;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          if (MODE == SUM_PLAIN) s[j] += bf(av[j]);
          if (MODE == SUM_RELU) {
            ov[j] = bf(av[j]) > 0.0f ? yv[j] : (uint16_t)0;
            s[j] += bf(ov[j]);
          }
          if (MODE == SUM_HEAD) {
            ov[j] = tobf(d * wv[j]);
            s[j] += d * bf(av[j]);
          }
        }
        if (MODE != SUM_PLAIN) {
          if (V == 8)
            *reinterpret_cast<uint4*>(dz + at) = *reinterpret_cast<const uint4*>(ov);
          else
            dz[at] = ov[0];
        }
      }
      // a row as wide as the block: the thread's sum is the block's
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if (groups > 1)
          acc[g * C + c * V + j] = s[j];
        else
          part[(long long)blockIdx.x * width + c * V + j] = s[j];
      }
    }
  }
  if (groups > 1) {
    __syncthreads();
    for (int c = threadIdx.x; c < C; c += 256) {
      float s = 0.0f;
      for (int q = 0; q < groups; ++q) s += acc[q * C + c];
      part[(long long)blockIdx.x * width + c] = s;
    }
  }
  if (MODE == SUM_HEAD) {
    __shared__ float d[1024];
    float s = 0.0f;
    for (long long r = r0; r < r1; r += 1024) {
      __syncthreads();
      for (int j = threadIdx.x; j < 1024 && r + j < r1; j += 256) d[j] = dout[r + j];
      __syncthreads();
      const int m = r1 - r < 1024 ? (int)(r1 - r) : 1024;
      if (threadIdx.x == 0)
        for (int j = 0; j < m; ++j) s += d[j];
    }
    if (threadIdx.x == 0) part[(long long)blockIdx.x * width + C] = s;
  }
}

// the head's records: column c < C summed by the block's threads, column C in
// block order
__global__ void __launch_bounds__(256)
    k_head_sum(const float* __restrict__ part, float* __restrict__ out, int C, int blocks) {
  __shared__ float v[1024];
  const int c = blockIdx.x;
  for (int b = threadIdx.x; b < blocks; b += 256) v[b] = part[(long long)b * (C + 1) + c];
  __syncthreads();
  if (c == C) {
    if (threadIdx.x == 0) {
      float s = 0.0f;
      for (int b = 0; b < blocks; ++b) s += v[b];
      out[c] = s;
    }
    return;
  }
  float s = 0.0f;
  for (int b = threadIdx.x; b < blocks; b += 256) s += v[b];
  __syncthreads();
  v[threadIdx.x] = s;
  for (int h = 128; h > 0; h >>= 1) {
    __syncthreads();
    if ((int)threadIdx.x < h) v[threadIdx.x] += v[threadIdx.x + h];
  }
  if (threadIdx.x == 0) out[c] = v[0];
}

// blocks: at most 1024 (the callers' work buffers hold 1024 records), each
// with at least 64 rows, which is what its record costs to add up; the
// head's blocks hold ceil(rows / 1024) rows, which fixes its bias' sum
template <int MODE>
int launch_rows(const uint16_t* a, const uint16_t* dy, uint16_t* dz, const float* w,
                const float* dout, float* out, float* part, long long rows, int C,
                hipStream_t s) {
  if (rows < 1 || C < 1) return nx::set_error(NX_ERR_ARG, "row pass: rows and channels >= 1");
  const int width = MODE == SUM_HEAD ? C + 1 : C;
  long long blocks = MODE == SUM_HEAD ? rows : (rows + 63) / 64;
  if (blocks > 1024) blocks = 1024;
  const long long per = (rows + blocks - 1) / blocks;
  blocks = (rows + per - 1) / per;
  const bool vec = C % 8 == 0 &&
                   (((uintptr_t)a | (uintptr_t)dy | (uintptr_t)dz) & 15) == 0;
  const int cg = vec ? C / 8 : C;
  const int groups = cg < 256 ? 256 / cg : 1;
  const size_t lds = groups > 1 ? (size_t)groups * C * sizeof(float) : 0;  // at most 8 KiB
  if (vec)
    k_rows<MODE, 8><<<(unsigned)blocks, 256, lds, s>>>(a, dy, dz, w, dout, part, rows, C, per);
  else
    k_rows<MODE, 1><<<(unsigned)blocks, 256, lds, s>>>(a, dy, dz, w, dout, part, rows, C, per);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) {
    if (MODE == SUM_HEAD)
      k_head_sum<<<width, 256, 0, s>>>(part, out, C, (int)blocks);
    else
      launch_sum_splits(part, out, width, (int)blocks, s);
    e = hipGetLastError();
  }
  return e == hipSuccess ? NX_OK : nx::set_error(NX_ERR_HIP, hipGetErrorString(e));
}

// ------------------------------------------------------------ weight gradient
// dw[co][tap][ci] = sum over pixels m of dy[m][co] x[m moved by tap][ci].
// A block of 4 waves makes all nine taps of a 32 x 32 channel tile over the
// spatial tiles of its split: a tile of 8 rows x 16 columns of dy and its 10
// x 18 surround of x are staged in LDS as they lie in memory, [pixel][32
// channels], once for the nine taps, and wave w runs the K steps (16 pixels
// of a row) of rows 2 w and 2 w + 1.  MFMA wants 8 consecutive K, here
// pixels, of one channel per lane: ds_read_b64_tr_b16 transposes on the way
// out of LDS (in each group of 16 lanes, lane i addresses 4 channels of pixel
// i / 4 and receives 4 pixels of channel i), so a tap's shift is only another
// pixel address, whatever its alignment.  A pixel row of 64 bytes puts the
// four rows of two lane groups on 64 different banks.
// A column beyond the image points its lanes at zeros with no row stride
// (its dy is staged as zero, and x may hold an infinity there); rows beyond
// the image are left out.
// Bound: LDS reads and MFMA issue, about equal (28 reads, 18 MFMAs of 32
// cycles per wave and tile).  32 x 64 x 64 pixels, 64 -> 64 channels: 29 us
// (330 TFLOP/s) and 5 us for the sum of the splits, where a form that staged
// each tap of 64 x 64 channels anew, transposed by 2-byte LDS stores, took
// 182 and 122.
constexpr int WG_TH = 8, WG_TW = 16, WG_XW = WG_TW + 2, WG_XH = WG_TH + 2;
constexpr int WG_DY = WG_TH * WG_TW, WG_X = WG_XH * WG_XW;  // pixels
constexpr int WG_BUF = (WG_DY + WG_X) * 32;                 // halfwords of one stage
constexpr int WG_ZERO = 3 * 32;                             // three pixels of zeros

__global__ void __launch_bounds__(256, 2)
    k_conv3x3_wgrad(const uint16_t* __restrict__ x, const uint16_t* __restrict__ dy,
                    float* __restrict__ part, int H, int W, int Cin, int Cout, int tiles,
                    int tiles_x, int tiles_img, int per) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * WG_BUF + WG_ZERO];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ci_tiles = (Cin + 31) / 32;
  const int co0 = (blockIdx.x / ci_tiles) * 32, ci0 = (blockIdx.x % ci_tiles) * 32;
  const int t_begin = blockIdx.y * per, t_end = min(t_begin + per, tiles);
  for (int i = threadIdx.x; i < WG_ZERO; i += 256) lds[2 * WG_BUF + i] = 0;

  // staging: 16-byte chunks (8 channels of a pixel), 2 of dy and 3 of x per
  // thread; chunk j of a thread is chunk threadIdx.x + 256 j of the array
  uint4 rdy[2], rx[3];
  auto load = [&](int t) {
    const int img = t / tiles_img, rem = t - img * tiles_img;
    const int y0 = rem / tiles_x * WG_TH, x0 = rem % tiles_x * WG_TW;
    const long long pix0 = (long long)img * H * W;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c = threadIdx.x + 256 * j, px = c >> 2, ch = co0 + (c & 3) * 8;
      const int yy = y0 + (px >> 4), xx = x0 + (px & 15);
      rdy[j] = make_uint4(0, 0, 0, 0);
      if (yy < H && xx < W && ch < Cout)
        rdy[j] = *reinterpret_cast<const uint4*>(dy + (pix0 + (long long)yy * W + xx) * Cout + ch);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int c = threadIdx.x + 256 * j, px = c >> 2, ch = ci0 + (c & 3) * 8;
      const int yy = y0 + px / WG_XW - 1, xx = x0 + px % WG_XW - 1;
      rx[j] = make_uint4(0, 0, 0, 0);
      if (px < WG_X && yy >= 0 && yy < H && xx >= 0 && xx < W && ch < Cin)
        rx[j] = *reinterpret_cast<const uint4*>(x + (pix0 + (long long)yy * W + xx) * Cin + ch);
    }
  };
  auto store = [&](uint16_t* buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<uint4*>(buf + (threadIdx.x + 256 * j) * 8) = rdy[j];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int c = threadIdx.x + 256 * j;
      if (c < WG_X * 4) *reinterpret_cast<uint4*>(buf + WG_DY * 32 + c * 8) = rx[j];
    }
  };

  const int grp = lane >> 4, i = lane & 15;
  const int kpx = 8 * (grp >> 1) + (i >> 2);         // pixel of the first read; + 4: second
  const int chn = 16 * (grp & 1) + 4 * (i & 3);      // channels of the lane's address
  f32x16 acc[9];
#pragma unroll
  for (int t = 0; t < 9; ++t)
    for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;

  auto frag = [&](const uint16_t* p0, const uint16_t* p1) -> bf16x8 {
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
    typedef __attribute__((__vector_size__(8 * sizeof(short)))) short s16x8;
    const s16x8 v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
  };

  if (t_begin < t_end) {
    load(t_begin);
    store(lds);
  }
  __syncthreads();
  for (int t = t_begin; t < t_end; ++t) {
    uint16_t* buf = lds + ((t - t_begin) & 1) * WG_BUF;
    const bool more = t + 1 < t_end;
    if (more) load(t + 1);
    const int rem = t % tiles_img;
    const int y0 = rem / tiles_x * WG_TH, x0 = rem % tiles_x * WG_TW;
    // lanes of a column beyond the image: the zeros, with no row stride
    const bool in0 = x0 + kpx < W, in1 = x0 + kpx + 4 < W;
    const uint16_t* xb = buf + WG_DY * 32 + chn;
    const uint16_t* zero = lds + 2 * WG_BUF + chn;
    const uint16_t* xa0 = in0 ? xb + kpx * 32 : zero;
    const uint16_t* xa1 = in1 ? xb + (kpx + 4) * 32 : zero;
    const int rs0 = in0 ? WG_XW * 32 : 0, rs1 = in1 ? WG_XW * 32 : 0;
    const uint16_t* da = buf + kpx * 32 + chn;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int ry = 2 * wave + q;
      if (y0 + ry >= H) continue;  // wave-uniform
      const uint16_t* dr = da + ry * WG_TW * 32;
      const bf16x8 a = frag(dr, dr + 4 * 32);
#pragma unroll
      for (int ty = 0; ty < 3; ++ty)
#pragma unroll
        for (int tx = 0; tx < 3; ++tx) {
          const bf16x8 b = frag(xa0 + (ry + ty) * rs0 + tx * 32, xa1 + (ry + ty) * rs1 + tx * 32);
          acc[3 * ty + tx] =
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[3 * ty + tx], 0, 0, 0);
        }
    }
    if (more) store(lds + ((t + 1 - t_begin) & 1) * WG_BUF);
    __syncthreads();
  }

  // the four waves' sums of one tap at a time, added in wave order
  float* red = reinterpret_cast<float*>(lds);  // [4][32][32], 16 KiB
  float* base = part + (long long)blockIdx.y * Cout * 9 * Cin;
  const int r = lane & 31, kb = lane >> 5;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      red[wave * 1024 + (8 * (e >> 2) + 4 * kb + (e & 3)) * 32 + r] = acc[t][e];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int o = threadIdx.x + 256 * j, co = co0 + (o >> 5), ci = ci0 + (o & 31);
      const float v = (red[o] + red[1024 + o]) + (red[2048 + o] + red[3072 + o]);
      if (co < Cout && ci < Cin) base[((long long)co * 9 + t) * Cin + ci] = v;
    }
    __syncthreads();
  }
}
static_assert((2 * WG_BUF + WG_ZERO) * 2 >= 4 * 1024 * 4, "the final sums reuse the stages");

}  // namespace

#define NX_U(stream) ((hipStream_t)(stream))
#define NX_BWD_RET()                                                            \
  do {                                                                          \
    hipError_t e_ = hipGetLastError();                                          \
    return e_ == hipSuccess ? NX_OK                                             \
                            : nx::set_error(NX_ERR_HIP, hipGetErrorString(e_)); \
  } while (0)

extern "C" {

// dw: float32 [cout][9][cin]; work: float32, splits * cout * 9 * cin
int nx_conv3x3_wgrad(const void* x, const void* dy, float* dw, float* work, int splits,
                     int n, int h, int wd, int cin, int cout, void* stream) {
  if (!x || !dy || !dw || !work || splits < 1 || n < 1 || h < 1 || wd < 1 || cin < 8 ||
      cout < 8 || cin % 8 || cout % 8)
    return nx::set_error(NX_ERR_ARG, "conv3x3 wgrad: cin % 8 == 0 and cout % 8 == 0");
  const int tiles_x = (wd + WG_TW - 1) / WG_TW;
  const int tiles_img = tiles_x * ((h + WG_TH - 1) / WG_TH);
  const long long tiles = (long long)tiles_img * n;
  if (tiles > 0x7FFFFFFF) return nx::set_error(NX_ERR_ARG, "conv3x3 wgrad: too many pixels");
  // grid.y at most 65535; every split has at least one tile
  long long used = splits < tiles ? splits : tiles;
  if (used > 65535) used = 65535;
  const int per = (int)((tiles + used - 1) / used);
  used = (tiles + per - 1) / per;
  const hipStream_t s = NX_U(stream);
  const dim3 grid(((cout + 31) / 32) * ((cin + 31) / 32), (unsigned)used);
  float* to = used == 1 ? dw : work;
  k_conv3x3_wgrad<<<grid, 256, 0, s>>>((const uint16_t*)x, (const uint16_t*)dy, to, h, wd, cin,
                                       cout, (int)tiles, tiles_x, tiles_img, per);
  if (hipGetLastError() != hipSuccess) return nx::set_error(NX_ERR_HIP, "wgrad failed");
  if (used > 1) launch_sum_splits(work, dw, (long long)cout * 9 * cin, (int)used, s);
  NX_BWD_RET();
}

// column sums of a bf16 (rows x c) matrix into out[c] (float32);
// work: 1024 * c floats
int nx_colsum(const void* a, float* out, float* work, long long rows, int c, void* stream) {
  return launch_rows<SUM_PLAIN>((const uint16_t*)a, nullptr, nullptr, nullptr, nullptr, out,
                                work, rows, c, NX_U(stream));
}

int nx_relu_bwd_colsum(const void* y, const void* dy, void* dz, float* db, float* work,
                       long long rows, int c, void* stream) {
  if (!y || !dy || !dz || !db || !work)
    return nx::set_error(NX_ERR_ARG, "relu backward: null argument");
  return launch_rows<SUM_RELU>((const uint16_t*)y, (const uint16_t*)dy, (uint16_t*)dz, nullptr,
                               nullptr, db, work, rows, c, NX_U(stream));
}

// dw[c] (c floats) and db (1 float) into dwb[0..c]; work: 1024 * (c+1) floats
int nx_head_bwd(const void* x, const float* w, const float* dout, void* dx, float* dwb,
                float* work, long long pixels, int c, void* stream) {
  return launch_rows<SUM_HEAD>((const uint16_t*)x, nullptr, (uint16_t*)dx, w, dout, dwb, work,
                               pixels, c, NX_U(stream));
}

}  // extern "C"
