// Fused [advection ->] curl -> confinement -> [viscosity] -> divergence ->
// first sweep, one LDS-staged 64x16 tile (shared by the single-grid and batched
// kernels).
#pragma once
#include "nx_cells.h"
#include "nx_common.h"

namespace nx {
namespace fused {

constexpr int TX = 64, TY = 16;  // output tile
constexpr int HMAX = 4;

struct Tile {
  int ox, oy, W, H;
  __device__ int cx(int vx) const { return clampi(vx, 0, W - 1); }
  __device__ int cy(int vy) const { return clampi(vy, 0, H - 1); }
};

// index of grid coordinate (gx, gy) in a stage array of halo hs
__device__ __forceinline__ int sidx(const Tile& t, int hs, int gx, int gy) {
  return (gy - t.oy + hs) * (TX + 2 * hs) + (gx - t.ox + hs);
}

__device__ __forceinline__ float2 confine_cell(float2 u, float wc, float wl,
                                               float wr, float wb, float wt,
                                               float dt, float scale) {
  // shader.ApplyVorticity.comp:33-39
  float fx = 0.5f * (fabsf(wt) - fabsf(wb));
  float fy = 0.5f * (fabsf(wr) - fabsf(wl));
  const float mag = fmaxf(VORTICITY_EPSILON, fx * fx + fy * fy);
  const float inv = 1.0f / sqrtf(mag);
  fx = fx * inv;
  fy = fy * inv;
  const float s = scale * wc;
  fx = fx * s;
  fy = fy * (-s);
  return make_float2(u.x + fx * dt, u.y + fy * dt);
}

// The advection of the velocity that enters a tile (Advect::on), with the
// walls' treatment on its reads; off: the input is the advected velocity.
struct Advect {
  int on;
  float speed, diss;
  BcParams bc;
};

// Stages of one 64x16 output tile with halo HA (3, or 4 with viscosity);
// every stage walks its region as one flat index range over the block's NT
// threads, so no lane idles on the few columns past a multiple of 64.  In
// an INTERIOR tile (halo inside the grid) no coordinate clamps, and the
// stencil neighbours of a stage slot are fixed offsets in the previous
// stage's array; border tiles evaluate the clamped coordinates.
template <class S, bool VISC, bool INTERIOR, bool ADV, int NT>
__device__ __forceinline__ void fused_tile_stages(
    float2* A, float* Wc, float2* V2, const Tile& t, const typename S::s2* __restrict__ uin,
    const uint8_t* __restrict__ mask, typename S::s2* __restrict__ uout,
    typename S::s1* __restrict__ div, typename S::s1* __restrict__ p1, float dt,
    float scale, float alpha, float rbeta, const Advect& adv) {
  constexpr int hA = VISC ? 4 : 3, hW = hA - 1, hV2 = hA - 2;
  constexpr int WA = TX + 2 * hA, HA = TY + 2 * hA;
  constexpr int WW = TX + 2 * hW, HW = TY + 2 * hW;
  constexpr int WV = TX + 2 * hV2, HV = TY + 2 * hV2;
  const int tid = threadIdx.y * 64 + threadIdx.x;
  const int W = t.W;
  // the viscosity output reuses A's storage: A is last read by the
  // confinement stage, which a barrier separates from the viscosity stage
  float2* const V3 = A;

  // 1. advected velocity at clamped coordinates; advected here, the halo's
  //    cells are advected by every tile that reads them, and rounded to
  //    storage as a pass of its own would leave them
  auto slot = [&](int k, int& gx, int& gy) {
    const int j = k / WA, i = k - j * WA;
    gy = INTERIOR ? t.oy - hA + j : t.cy(t.oy - hA + j);
    gx = INTERIOR ? t.ox - hA + i : t.cx(t.ox - hA + i);
  };
  if (ADV) {
    // a thread's slots in groups of G: the group's velocities in flight
    // together, then its corners; cells and corners of the grid's outermost
    // ring, whose values the walls make, are read once more through them
    constexpr int N = (WA * HA + NT - 1) / NT, G = N < 4 ? N : 4;
    auto ring = [&](int x, int y) { return x == 0 || y == 0 || x == W - 1 || y == t.H - 1; };
#pragma unroll
    for (int g0 = 0; g0 < N; g0 += G) {
      int gx[G], gy[G];
      float2 v[G];
      uint8_t m[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        slot(min(tid + NT * (g0 + g), WA * HA - 1), gx[g], gy[g]);
        v[g] = S::ld2(uin, gy[g] * W + gx[g]);
        m[g] = mask[gy[g] * W + gx[g]];
      }
      Bilin c[G];
      float2 lt[G], rt[G], lb[G], rb[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (ring(gx[g], gy[g])) v[g] = load_bc<S>(uin, gx[g], gy[g], W, t.H, adv.bc);
        c[g] = bilinear_corners((float)gx[g] - (v[g].x * dt) * adv.speed,
                                (float)gy[g] - (v[g].y * dt) * adv.speed, W, t.H);
        lt[g] = S::ld2(uin, c[g].lt);
        rt[g] = S::ld2(uin, c[g].rt);
        lb[g] = S::ld2(uin, c[g].lb);
        rb[g] = S::ld2(uin, c[g].rb);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (c[g].bx == 0 || c[g].by == 0 || c[g].tx == W - 1 || c[g].ty == t.H - 1) {
          lt[g] = load_bc<S>(uin, c[g].bx, c[g].ty, W, t.H, adv.bc);
          rt[g] = load_bc<S>(uin, c[g].tx, c[g].ty, W, t.H, adv.bc);
          lb[g] = load_bc<S>(uin, c[g].bx, c[g].by, W, t.H, adv.bc);
          rb[g] = load_bc<S>(uin, c[g].tx, c[g].by, W, t.H, adv.bc);
        }
        const float2 q = bilinear_mix<float2>(lt[g], rt[g], lb[g], rb[g], c[g].dx, c[g].dy);
        const bool fluid = m[g] == 0;
        typename S::s2 w;
        S::st2(&w, 0, make_float2(fluid ? clampf(q.x * adv.diss, -1.0f, 1.0f) : 0.0f,
                                  fluid ? clampf(q.y * adv.diss, -1.0f, 1.0f) : 0.0f));
        if (tid + NT * (g0 + g) < WA * HA) A[tid + NT * (g0 + g)] = S::ld2(&w, 0);
      }
    }
  } else {
    for (int k = tid; k < WA * HA; k += NT) {
      int gx, gy;
      slot(k, gx, gy);
      A[k] = S::ld2(uin, gy * W + gx);
    }
  }
  __syncthreads();

  // 2. curl, shader.CalcVorticity.comp:21-26
  for (int k = tid; k < WW * HW; k += NT) {
    const int j = k / WW, i = k - j * WW;
    float2 vL, vR, vB, vT;
    if (INTERIOR) {
      const int a = (j + 1) * WA + (i + 1);
      vL = A[a - 1];
      vR = A[a + 1];
      vB = A[a - WA];
      vT = A[a + WA];
    } else {
      const int gy = t.cy(t.oy - hW + j), gx = t.cx(t.ox - hW + i);
      const int yb = t.cy(gy - 1), yt = t.cy(gy + 1);
      const int xl = t.cx(gx - 1), xr = t.cx(gx + 1);
      vL = A[sidx(t, hA, xl, gy)];
      vR = A[sidx(t, hA, xr, gy)];
      vB = A[sidx(t, hA, gx, yb)];
      vT = A[sidx(t, hA, gx, yt)];
    }
    Wc[k] = 0.5f * ((vR.y - vL.y) - (vT.x - vB.x));
  }
  __syncthreads();

  // 3. confinement, shader.ApplyVorticity.comp:26-39
  for (int k = tid; k < WV * HV; k += NT) {
    const int j = k / WV, i = k - j * WV;
    if (INTERIOR) {
      const int w = (j + 1) * WW + (i + 1);
      V2[k] = confine_cell(A[(j + 2) * WA + (i + 2)], Wc[w], Wc[w - 1], Wc[w + 1],
                           Wc[w - WW], Wc[w + WW], dt, scale);
    } else {
      const int gy = t.cy(t.oy - hV2 + j), gx = t.cx(t.ox - hV2 + i);
      const int yb = t.cy(gy - 1), yt = t.cy(gy + 1);
      const int xl = t.cx(gx - 1), xr = t.cx(gx + 1);
      V2[k] = confine_cell(A[sidx(t, hA, gx, gy)], Wc[sidx(t, hW, gx, gy)],
                           Wc[sidx(t, hW, xl, gy)], Wc[sidx(t, hW, xr, gy)],
                           Wc[sidx(t, hW, gx, yb)], Wc[sidx(t, hW, gx, yt)], dt, scale);
    }
  }
  __syncthreads();

  // 4. viscosity, shader.Viscosity.comp:25-31 (only when nu > 0)
  const float2* Vf = V2;
  int hf = hV2;
  if (VISC) {
    constexpr int W3 = TX + 2, H3 = TY + 2;
    for (int k = tid; k < W3 * H3; k += NT) {
      const int j = k / W3, i = k - j * W3;
      float2 L, R, B, T, c;
      if (INTERIOR) {
        const int v = (j + 1) * WV + (i + 1);
        L = V2[v - 1];
        R = V2[v + 1];
        B = V2[v - WV];
        T = V2[v + WV];
        c = V2[v];
      } else {
        const int gy = t.cy(t.oy - 1 + j), gx = t.cx(t.ox - 1 + i);
        const int yb = t.cy(gy - 1), yt = t.cy(gy + 1);
        const int xl = t.cx(gx - 1), xr = t.cx(gx + 1);
        L = V2[sidx(t, hV2, xl, gy)];
        R = V2[sidx(t, hV2, xr, gy)];
        B = V2[sidx(t, hV2, gx, yb)];
        T = V2[sidx(t, hV2, gx, yt)];
        c = V2[sidx(t, hV2, gx, gy)];
      }
      V3[k] = make_float2(((((L.x + R.x) + B.x) + T.x) + c.x * alpha) * rbeta,
                          ((((L.y + R.y) + B.y) + T.y) + c.y * alpha) * rbeta);
    }
    __syncthreads();
    Vf = V3;
    hf = 1;
  }

  // 5. divergence (Divergence.comp:22-40) and the first sweep from p = 0:
  //    ((((0+0)+0)+0) - b) * 0.25 = (0 - b) * 0.25 (Poisson.comp:37)
  const int Wf = TX + 2 * hf;
  for (int k = tid; k < TX * TY; k += NT) {
    const int j = k / TX, i = k - j * TX;
    const int gy = t.oy + j, gx = t.ox + i;
    if (!INTERIOR && (gy >= t.H || gx >= W)) continue;
    const int pos = gy * W + gx;
    float2 vl, vr, vb, vt, vc;
    int ml, mr, mb, mt;
    if (INTERIOR) {
      const int v = (j + hf) * Wf + (i + hf);
      vl = Vf[v - 1];
      vr = Vf[v + 1];
      vb = Vf[v - Wf];
      vt = Vf[v + Wf];
      vc = Vf[v];
      ml = pos - 1;
      mr = pos + 1;
      mb = pos - W;
      mt = pos + W;
    } else {
      const int yb = t.cy(gy - 1), yt = t.cy(gy + 1);
      const int xl = t.cx(gx - 1), xr = t.cx(gx + 1);
      vl = Vf[sidx(t, hf, xl, gy)];
      vr = Vf[sidx(t, hf, xr, gy)];
      vb = Vf[sidx(t, hf, gx, yb)];
      vt = Vf[sidx(t, hf, gx, yt)];
      vc = Vf[sidx(t, hf, gx, gy)];
      ml = gy * W + xl;
      mr = gy * W + xr;
      mb = yb * W + gx;
      mt = yt * W + gx;
    }
    const float x1 = mask[ml] ? 0.0f : vl.x;
    const float x2 = mask[mr] ? 0.0f : vr.x;
    const float y1 = mask[mb] ? 0.0f : vb.y;
    const float y2 = mask[mt] ? 0.0f : vt.y;
    const float d = 0.5f * ((x2 - x1) + (y2 - y1));
    S::st2(uout, pos, vc);
    S::st(div, pos, d);
    if (p1) S::st(p1, pos, (0.0f - d) * 0.25f);
  }
}

// One 64x16 output tile with origin (ox, oy); NT threads as (64, NT / 64).
// Velocity, divergence and p1 are stored in format S; the chain is float32.
template <class S = F32S, bool ADV = false, int NT = 256>
__device__ __forceinline__ void fused_vort_div_tile(
    int ox, int oy, const typename S::s2* __restrict__ uin,
    const uint8_t* __restrict__ mask, typename S::s2* __restrict__ uout,
    typename S::s1* __restrict__ div, typename S::s1* __restrict__ p1, int W,
    int H, float dt, float scale, int viscous, float alpha, float rbeta,
    const Advect& adv = Advect{0, 0.0f, 0.0f, BcParams{0, 0, 0.0f}}) {
  __shared__ float2 A[(TX + 2 * HMAX) * (TY + 2 * HMAX)];
  __shared__ float Wc[(TX + 2 * HMAX - 2) * (TY + 2 * HMAX - 2)];
  __shared__ float2 V2[(TX + 2 * HMAX - 4) * (TY + 2 * HMAX - 4)];
  const Tile t{ox, oy, W, H};
  const int h = viscous ? 4 : 3;
  const bool interior = ox - h >= 0 && oy - h >= 0 && ox + TX + h <= W && oy + TY + h <= H;
  if (viscous) {
    if (interior)
      fused_tile_stages<S, true, true, ADV, NT>(A, Wc, V2, t, uin, mask, uout, div, p1, dt, scale,
                                            alpha, rbeta, adv);
    else
      fused_tile_stages<S, true, false, ADV, NT>(A, Wc, V2, t, uin, mask, uout, div, p1, dt, scale,
                                             alpha, rbeta, adv);
  } else {
    if (interior)
      fused_tile_stages<S, false, true, ADV, NT>(A, Wc, V2, t, uin, mask, uout, div, p1, dt, scale,
                                             alpha, rbeta, adv);
    else
      fused_tile_stages<S, false, false, ADV, NT>(A, Wc, V2, t, uin, mask, uout, div, p1, dt, scale,
                                              alpha, rbeta, adv);
  }
}

// threads of a block of the kernels with the advection in front: with few tiles
// the block's own latency counts and 1024 threads shorten it (128^2: 18 to 13 us
// for the stages of a step, 1001 x 699, 704 tiles: 31 to 26); with many, blocks
// of 256 overlap better (2048^2: 69 us a step of three simulators in turn
// against 77)
inline int advect_threads(int W, int H) {
  return ((W + TX - 1) / TX) * ((H + TY - 1) / TY) <= 768 ? 1024 : 256;
}

}  // namespace fused
}  // namespace nx
