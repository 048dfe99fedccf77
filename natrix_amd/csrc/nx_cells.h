// Per-cell device functions shared by the single-grid and batched kernels,
// so both evaluate the reference shaders with identical code.
#pragma once
#include "nx_common.h"

namespace nx {

// S2, shader.AdvectVelocity.comp:27-49, velocity read through the wall
// treatment of S1
template <class S = F32S>
__device__ __forceinline__ float2 advect_cell(
    const typename S::s2* __restrict__ uin, const uint8_t* __restrict__ mask,
    int x, int y, int W, int H, float dt, float speed, float diss,
    const BcParams& bc) {
  if (mask[y * W + x] != 0) return make_float2(0.0f, 0.0f);
  const float2 vel = load_bc<S>(uin, x, y, W, H, bc);
  const float fx = (float)x - (vel.x * dt) * speed;
  const float fy = (float)y - (vel.y * dt) * speed;
  const Bilin c = bilinear_corners(fx, fy, W, H);
  const float2 v = bilinear_mix<float2>(
      load_bc<S>(uin, c.bx, c.ty, W, H, bc), load_bc<S>(uin, c.tx, c.ty, W, H, bc),
      load_bc<S>(uin, c.bx, c.by, W, H, bc), load_bc<S>(uin, c.tx, c.by, W, H, bc),
      c.dx, c.dy);
  return make_float2(clampf(v.x * diss, -1.0f, 1.0f),
                     clampf(v.y * diss, -1.0f, 1.0f));
}

// S9, shader.SubtractGradient.comp:24-46 (pressure always float32)
template <class S = F32S>
__device__ __forceinline__ float2 subgrad_cell(
    const typename S::s2* __restrict__ uin, const float* __restrict__ p,
    const uint8_t* __restrict__ mask, int x, int y, int W, int H) {
  const int pos = y * W + x;
  const int iL = y * W + max(x - 1, 0), iR = y * W + min(x + 1, W - 1);
  const int iB = max(y - 1, 0) * W + x, iT = min(y + 1, H - 1) * W + x;
  const float pc = p[pos];
  const float x1 = mask[iL] ? pc : p[iL];
  const float x2 = mask[iR] ? pc : p[iR];
  const float y1 = mask[iB] ? pc : p[iB];
  const float y2 = mask[iT] ? pc : p[iT];
  float2 v = S::ld2(uin, pos);
  v.x -= 0.5f * (x2 - x1);
  v.y -= 0.5f * (y2 - y1);
  return v;
}

// S11, demo/shaders/shader.AdvectParticle.comp:21-69 (dye grid P, velocity
// grid V); sx, sy: the quotients of their sides, one division for the grid
template <class S = F32S>
__device__ __forceinline__ float advect_dye_cell(
    const typename S::s1* __restrict__ qin, const typename S::s2* __restrict__ u,
    const uint8_t* __restrict__ mask, int x, int y, int Wp, int Hp, int Wv,
    int Hv, float sx, float sy, float dt, float speed, float diss) {
  const float nx = ((float)x / (float)Wp) * (float)Wv;
  const float ny = ((float)y / (float)Hp) * (float)Hv;
  // uint() truncation (n >= 0); x/Wp < 1 keeps it below Wv, the min() only
  // guards the memory access
  const int opos = min((int)ny, Hv - 1) * Wv + min((int)nx, Wv - 1);
  if (mask[opos] != 0) return 0.0f;
  const Bilin cv = bilinear_corners(nx, ny, Wv, Hv);
  const float2 vel =
      bilinear_mix<float2>(S::ld2(u, cv.lt), S::ld2(u, cv.rt), S::ld2(u, cv.lb),
                           S::ld2(u, cv.rb), cv.dx, cv.dy);
  const float vx = vel.x * sx, vy = vel.y * sy;
  const float fx = (float)x - (vx * dt) * speed;
  const float fy = (float)y - (vy * dt) * speed;
  const Bilin c = bilinear_corners(fx, fy, Wp, Hp);
  return bilinear_mix<float>(S::ld(qin, c.lt), S::ld(qin, c.rt),
                             S::ld(qin, c.lb), S::ld(qin, c.rb), c.dx, c.dy) *
         diss;
}

// e2: w = float(exp(double(-(dx*dx + dy*dy) / (r*r)))).  Below -104 the
// exponent's weight rounds to zero (exp(-104) < 2^-150), and beyond 105 r*r the
// quotient is below that whatever its rounding.  SKIP: waves with no cell within
// 10.25 radii of the splat leave out the division and the float64 exponential,
// which were the kernel's time (4096^2 bf16, 8 splats: 167 to 96 us).
template <bool SKIP>
__device__ __forceinline__ float gaussian_weight(const Splat& s, int x, int y,
                                                 int W, int H) {
  const float sx = s.px * (float)W, sy = s.py * (float)H;
  const float dx = sx - (float)x, dy = sy - (float)y;
  const float d2 = dx * dx + dy * dy, r2 = s.radius * s.radius;
  if (SKIP && d2 > 105.0f * r2) return 0.0f;
  return (float)exp((double)(-d2 / r2));
}

// Share of a W x H grid in the box of a splat's reach, 10.25 radii; a centre or
// radius that is no number counts as all of it.
inline float splat_share(const Splat& s, int W, int H) {
  const float w = (float)W, h = (float)H, x = s.px * w, y = s.py * h;
  const float reach = 10.25f * fabsf(s.radius);
  const float bw = fminf(x + reach, w) - fmaxf(x - reach, 0.0f);
  const float bh = fminf(y + reach, h) - fmaxf(y - reach, 0.0f);
  return fmaxf(bw, 0.0f) / w * (fmaxf(bh, 0.0f) / h);
}

// SKIP pays while less than this share of the (cell, splat) pairs is within reach:
// its branch makes a near pair cost 1.2 of what it costs without.  2048^2, 8
// splats, us without / with at shares of 0.04, 0.36, 0.57, 0.76 and 1: 39.8 / 21.1,
// 39.7 / 33.4, 39.9 / 38.7, 40.2 / 42.7, 40.4 / 47.8.
constexpr float SPLAT_SKIP_SHARE = 0.55f;

}  // namespace nx
