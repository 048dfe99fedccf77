// Temporal-blocked Chebyshev smoothing of the fine pressure system.
//
// Chebyshev iteration for -L x = -b on the eigenvalue interval [lmin, 8] of
// -L (three-term recurrence of Saad, Iterative Methods for Sparse Linear
// Systems, 2nd ed., Algorithm 12.1), with L the 5-point operator of the
// Jacobi sweep (shader.Poisson.comp:26-37: a solid or out-of-grid neighbour
// reads the centre value):
//   setup:      r = L x - b,  d = r / theta
//   iteration:  x += d,  r += L d,  d = (rho' rho) d + (2 rho' / delta) r
//               (one fused multiply-add: fma(cd, d, cr r))
// with theta = (8 + lmin) / 2, delta = (8 - lmin) / 2, sigma = theta /
// delta, rho_0 = 1 / sigma, rho' = 1 / (2 sigma - rho) (the scalar
// recurrence runs on the host; a launch takes its passes' coefficients).
// -L is symmetric positive semi-definite with spectrum in [0, 8], so the
// error polynomial is at most 1 in magnitude on all of [0, 8] and at most
// 1 / T_n(sigma) on [lmin, 8]: n iterations damp every mode above lmin,
// which n Jacobi sweeps (factor (1 - lambda / 4)^n) leave nearly untouched
// near lmin.
//
// Only d needs neighbours, so a launch carries (x, r, d) of a register tile
// through k stencil passes (nx_cheb_tile.h).  The first launch of a run spends
// its first pass on the setup, the last one (RES) its last pass on the FP64
// residual of the result.  Every pass evaluates each cell's expressions in a
// fixed order: L v = (((u + l) + r) + d) - 4 v with u, d the cells above and
// below and l, r the lane-shifted ones, so that each shift is the DPP operand
// of an addition (no separate move); the -4 v is one fused multiply-add, which
// rounds like the subtraction because 4 v is exact; and the d update is the one
// fused multiply-add written above.  The result is bitwise independent of the
// tile shape and of k.
#include "../../include/natrix.h"
#include "nx_cheb_tile.h"
#include "nx_kernels.h"

namespace nx {

namespace {

template <int ROWS, int WAVES, int COLS, bool RES>
__global__ void __launch_bounds__(WAVES * 64)
    __attribute__((amdgpu_waves_per_eu(jt::cheb_waves_per_eu<ROWS * COLS>())))
    k_cheb_tb(jt::ChebArgs a, ChebCoef cf) {
  jt::cheb_tile<ROWS, WAVES, COLS, false, RES>(a, cf,
                                               xcd_tile<XCD_RUNS>((int)blockIdx.x, gridDim.x));
}

template <int ROWS, int WAVES, int COLS>
hipError_t launch_cheb(const jt::ChebArgs& a, const ChebCoef& cf, hipStream_t st) {
  const int grid = jt::cheb_tiles(a.W, a.H, 64 * COLS, ROWS * WAVES, a.halo);
  if (a.red)
    k_cheb_tb<ROWS, WAVES, COLS, true><<<grid, WAVES * 64, 0, st>>>(a, cf);
  else
    k_cheb_tb<ROWS, WAVES, COLS, false><<<grid, WAVES * 64, 0, st>>>(a, cf);
  return hipGetLastError();
}

}  // namespace

// Tile shapes (rows per wave, waves per block, columns per lane).
#define NX_CHEB_SHAPES(X) \
  X(2, 16, 2)             \
  X(4, 8, 2)              \
  X(4, 16, 2)             \
  X(4, 16, 1)             \
  X(8, 8, 1)              \
  X(8, 16, 1)             \
  X(8, 8, 2)

bool cheb_cfg_supported(JacobiCfg c) {
  bool shape = false;
#define NX_CHEB_CHECK(R, WV, CL) shape |= (c.rows == R && c.waves == WV && c.cols == CL);
  NX_CHEB_SHAPES(NX_CHEB_CHECK)
#undef NX_CHEB_CHECK
  return shape && c.k >= 1 && c.k <= CHEB_MAX_PASSES && 64 * c.cols - 2 * c.k >= 8 &&
         c.rows * c.waves - 2 * c.k >= 8;
}

// A residual launch's last stencil is the residual's, and its last iteration
// reads no neighbour: its cells depend on c.k - 1 stencils (one without
// iterations).
static int residual_halo(JacobiCfg c) { return c.k > 2 ? c.k - 1 : 1; }

int cheb_launch_blocks(int W, int H, JacobiCfg c) {
  return jt::cheb_tiles(W, H, 64 * c.cols, c.rows * c.waves, residual_halo(c));
}

hipError_t launch_cheb_tb(hipStream_t st, JacobiCfg c, const float* xin, const float* rin,
                          const float* din, const float* b, const uint8_t* mask, float* xout,
                          float* rout, float* dout, int W, int H, int setup, float theta,
                          const ChebCoef& cf, double* red, const float* dapp,
                          const double* line) {
  const int its = c.k - (setup ? 1 : 0) - (red ? 1 : 0);
  if (!cheb_cfg_supported(c) || its < 0) return hipErrorInvalidValue;
  const jt::ChebArgs a{xin,  rin,  din, b, mask,      nullptr, xout,
                       rout, dout, W,   H, its,       setup ? 1 : 0, red ? residual_halo(c) : c.k,
                       theta, red, dapp, line};
#define NX_CHEB_LAUNCH(R, WV, CL)                   \
  if (c.rows == R && c.waves == WV && c.cols == CL) \
    return launch_cheb<R, WV, CL>(a, cf, st);
  NX_CHEB_SHAPES(NX_CHEB_LAUNCH)
#undef NX_CHEB_LAUNCH
  return hipErrorInvalidValue;
}

ChebRecurrence::ChebRecurrence(float lambda_min) {
  theta = 0.5f * (8.0f + lambda_min);
  delta = 0.5f * (8.0f - lambda_min);
  sigma = theta / delta;
  rho = 1.0f / sigma;
}

void ChebRecurrence::next(int first, int passes, ChebCoef& cf) {
  for (int i = first; i < passes; ++i) {
    const float rho1 = 1.0f / (2.0f * sigma - rho);
    cf.cd[i] = rho1 * rho;
    cf.cr[i] = 2.0f * rho1 / delta;
    rho = rho1;
  }
}

}  // namespace nx
