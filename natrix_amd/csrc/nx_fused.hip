// Fused middle of the fluid step:
//   curl (CalcVorticity.comp) -> confinement (ApplyVorticity.comp)
//   -> [viscosity (Viscosity.comp)] -> divergence (Divergence.comp)
//   -> first Jacobi sweep from the zero guess (ClearBuffer + Poisson.comp).
//
// One 64x16 output tile per block.  The advected velocity is read once into LDS
// with a halo of 3 (4 with viscosity) and every intermediate field lives in LDS
// on a shrinking halo, so the kernel reads velocity + mask and writes velocity,
// divergence and p1: 8+1 -> 8+4+4 bytes per cell instead of the
// 12+20+(16)+13+4+13 bytes the separate passes move.  With the advection in
// front (the merged step) the block makes the advected velocity itself, halo
// included, instead of reading what a pass of its own wrote: 25 bytes a cell
// instead of 42, for 1.5 times the gathers.  Bound by the gathers' latency, so
// that at 2048^2 the bytes saved buy little (48.0 us for 20.7 + 28.9) and the gain
// is a launch less (128^2 9 us against 12.5) and, in bf16, the conversions of the
// stored velocity (4096^2 137 us against 167).
//
// Each LDS slot holds its stage's value at the CLAMPED grid coordinate of the
// slot, and neighbours are looked up at clamp(c +- 1) as common.sh:14-17 does,
// so border tiles need no special case and every value is bitwise the one
// the separate per-stage kernels produce.
#include "nx_fused_tile.h"
#include "nx_kernels.h"

namespace nx {

namespace {

using fused::TX;
using fused::TY;

template <bool ADV, int NT>
__global__ void __launch_bounds__(NT)
    k_fused_vort_div(const float2* __restrict__ uin,
                     const uint8_t* __restrict__ mask,
                     float2* __restrict__ uout, float* __restrict__ div,
                     float* __restrict__ p1, int W, int H, float dt,
                     float scale, int viscous, float alpha, float rbeta, fused::Advect adv) {
  // 1D grid of TX x TY tiles in XCD order
  const int gx = (W + TX - 1) / TX;
  const int t = xcd_tile((int)blockIdx.x, gx * ((H + TY - 1) / TY));
  fused::fused_vort_div_tile<F32S, ADV, NT>((t % gx) * TX, (t / gx) * TY, uin, mask, uout, div,
                                            p1, W, H, dt, scale, viscous, alpha, rbeta, adv);
}

}  // namespace

hipError_t launch_fused_vort_div(const float2* uin, const uint8_t* mask,
                                 float2* uout, float* div, float* p1, int W,
                                 int H, float dt, float scale, int viscous,
                                 float alpha, float rbeta, hipStream_t s) {
  const dim3 grid(((W + TX - 1) / TX) * ((H + TY - 1) / TY), 1, 1);
  k_fused_vort_div<false, 256><<<grid, dim3(64, 4), 0, s>>>(
      uin, mask, uout, div, p1, W, H, dt, scale, viscous, alpha, rbeta, fused::Advect{});
  return hipGetLastError();
}

hipError_t launch_advect_vort_div(const float2* uin, const uint8_t* mask, float2* uout,
                                  float* div, float* p1, int W, int H, float dt, float speed,
                                  float diss, BcParams bc, float scale, int viscous, float alpha,
                                  float rbeta, hipStream_t s) {
  const dim3 grid(((W + TX - 1) / TX) * ((H + TY - 1) / TY), 1, 1);
  const fused::Advect adv{1, speed, diss, bc};
  if (fused::advect_threads(W, H) == 1024)
    k_fused_vort_div<true, 1024><<<grid, dim3(64, 16), 0, s>>>(
        uin, mask, uout, div, p1, W, H, dt, scale, viscous, alpha, rbeta, adv);
  else
    k_fused_vort_div<true, 256><<<grid, dim3(64, 4), 0, s>>>(
        uin, mask, uout, div, p1, W, H, dt, scale, viscous, alpha, rbeta, adv);
  return hipGetLastError();
}

}  // namespace nx
