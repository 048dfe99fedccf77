// Temporal-blocked Chebyshev tile of the fine (solid cells) and the coarse
// (face weights) pressure systems; the iteration is stated in nx_cheb.hip.
//
// A launch carries (x, r, d) of a register tile through its stencil passes as
// the Jacobi tile carries p: lane l of wave w owns COLS columns and ROWS rows,
// horizontal neighbours come by DPP lane shifts, the rows next to a wave's strip
// through a double-buffered LDS exchange, and tiles lie inside the grid
// (axis_tiles): a side loses one cell per pass only where it has a neighbour.
//
// What bounds it: a launch reads and writes up to 29 bytes a cell, once for all
// its passes; the passes are VALU work, 8 instructions a cell, of which the
// overlapping halos are the larger part when many passes run on a small tile,
// and each pass waits once for the exchange (0.3 us).  Tiles inside the grid,
// masks taken as words and only by the waves next to solids, and no spills (x, r,
// d of up to 16 cells a lane; d is the only array with neighbours, and larger
// strips are walked up and down in turn, so that a new row takes the registers
// of the old one before it) took a learned step's 20 passes at 2048^2 from 107
// to 82 us (8 x 8 x 1, 10 a launch; 87 at 8 x 8 x 2, 104 at 4 x 16 x 2 and at
// 8 x 16 x 1), 74 passes at 1000 x 700 from 124 (10 a launch) to 84 (15), and
// 4096^2 (18 iterations) from 464 us (4 x 8 x 2, 8 a launch) to 255 (8 x 8 x 2,
// 10).  20 or 24 cells a lane spill (18 iterations at 2048^2: 95 to 109 us).
#pragma once
#include "nx_jacobi_tile.h"
#include "nx_kernels.h"

namespace nx {
namespace jt {

// Waves per SIMD asked of the compiler (amdgpu_waves_per_eu) for CELLS cells a lane
template <int CELLS>
constexpr int cheb_waves_per_eu() { return CELLS <= 4 ? 8 : CELLS <= 8 ? 5 : 4; }

struct ChebArgs {
  const float *x, *r, *d, *b;  // r: b at the first launch; d unread there
  const uint8_t* mask;         // fine system: solid cells
  const float* faces;          // coarse system: east, then south weights
  float *xout, *rout, *dout;   // rout null: only x is written
  int W, H;
  int its, first;  // iterations; whether r and d are set up from x and b
  int halo;        // stencils the written cells depend on
  float theta;
  double* red;          // RES: 5 sums a tile
  const float* dapp;    // first launch: x += line[0] dapp on fluid cells
  const double* line;
};

// tiles of a launch with `halo` stencils
inline int cheb_tiles(int W, int H, int EX, int EY, int halo) {
  return axis_tiles(W, EX, halo) * axis_tiles(H, EY, halo);
}

// FACES: a neighbour across a face of weight w enters the sum as the centre c
// when w = 0 (as a solid neighbour does), as itself when w = 1, and as
// fma(w, v - c, c) between, so that the sum minus 4 c is the sum of w (v - c).
// RES: after the iterations the exact FP64 residual r = b - L x on the tile's
// own fluid cells, as red[5 tile + {sum r, sum r^2, sum b, sum b^2, cells}].
template <int ROWS, int WAVES, int COLS, bool FACES, bool RES>
__device__ __forceinline__ void cheb_tile(const ChebArgs& a, const ChebCoef& cf, int tile) {
  constexpr int EX = 64 * COLS, EY = ROWS * WAVES;
  const int W = a.W, H = a.H;
  const int lane = threadIdx.x & 63;
  // wave-uniform: a scalar register, so branches on it are scalar branches
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nx = axis_tiles(W, EX, a.halo), ny = axis_tiles(H, EY, a.halo);
  const int bx = tile % nx, by = tile / nx;
  const AxisTile ax = axis_tile(bx, nx, W, EX, a.halo), ay = axis_tile(by, ny, H, EY, a.halo);
  const int tcol0 = COLS * lane;
  const int gx0 = ax.o + tcol0, gy0 = ay.o + wave * ROWS;
  const bool idle = gy0 >= H;  // beyond a grid smaller than the tile: barriers only
  const bool inside = W >= EX && H >= EY;
  const int right = W - 1 - gx0;  // the lane's column of the grid's last cell
  const int last = H - 1 - gy0;   // the strip's row of the grid's last row

  // cells of the lane's columns in row y (clamped to the grid; the cells
  // beyond it hold its edge, which no cell of the grid reads)
  auto load_row = [&](const float* __restrict__ p, int y, float(&v)[COLS]) {
    const long long row = (long long)min(max(y, 0), H - 1) * W;
    if (inside) {
      load_cols<F32S, COLS>(p + row + ax.o, tcol0, v);
    } else {
#pragma unroll
      for (int c = 0; c < COLS; ++c) v[c] = p[row + min(gx0 + c, W - 1)];
    }
  };
  auto mask_row = [&](int y) -> uint32_t {  // a bit per solid column
    const uint8_t* row = a.mask + (long long)min(max(y, 0), H - 1) * W;
    uint32_t m = 0;
#pragma unroll
    for (int c = 0; c < COLS; ++c) m |= (row[min(gx0 + c, W - 1)] ? 1u : 0u) << c;
    return m;
  };

  // every load is issued before the first use
  float x[ROWS][COLS], r[ROWS][COLS], d[ROWS][COLS];
  const float* rsrc = a.first ? a.b : a.r;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    load_row(a.x, gy0 + i, x[i]);
    load_row(rsrc, gy0 + i, r[i]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!a.first) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      load_row(a.d, gy0 + i, d[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < ROWS; ++i)
#pragma unroll
      for (int c = 0; c < COLS; ++c) d[i][c] = 0.0f;
  }

  // solid cells, a bit per cell of the strip and of the rows next to it, and a
  // bit per row for the cells left (0..15) and right (16..31) of the lane's
  // columns; cells beyond the grid count as solid
  static_assert((ROWS + 2) * COLS <= 32 && ROWS <= 16, "flags of a strip in a word");
  uint32_t sol = 0, side = 0;
  bool special = false;
  if (!FACES) {
    if (inside) {
      using M = typename Pack<uint8_t, COLS>::type;
      M m[ROWS + 2];
#pragma unroll
      for (int i = 0; i < ROWS + 2; ++i)
        m[i] = *reinterpret_cast<const M*>(
            a.mask + (long long)min(max(gy0 - 1 + i, 0), H - 1) * W + ax.o + tcol0);
#pragma unroll
      for (int i = 0; i < ROWS + 2; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) sol |= (m[i][c] ? 1u : 0u) << (i * COLS + c);
    } else {
#pragma unroll
      for (int i = 0; i < ROWS + 2; ++i) sol |= mask_row(gy0 - 1 + i) << (i * COLS);
    }
    special = __any(sol != 0);
    if (special || RES) {
      constexpr uint32_t ROW = (1u << COLS) - 1;
      const uint32_t beyond = right >= COLS - 1 ? 0 : right < 0 ? ROW : (ROW << (right + 1)) & ROW;
#pragma unroll
      for (int i = 0; i < ROWS + 2; ++i) {
        const bool row_in = gy0 + i > 0 && i - 1 <= last;
        sol |= (row_in ? beyond : ROW) << (i * COLS);
      }
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int own = (int)(sol >> ((i + 1) * COLS));
        const uint32_t fl = (uint32_t)ilane_from_left((own >> (COLS - 1)) & 1);
        const uint32_t fr = (uint32_t)ilane_from_right(own & 1);
        side |= (gx0 == 0 ? 1u : fl) << i;
        side |= (right < COLS ? 1u : fr) << (16 + i);
      }
    }
  }
  // face weights: east of the strip's cells, south of them and of the row before;
  // shut at the grid's edge (stored so for the east and south ones)
  constexpr int FR = FACES ? ROWS : 1;
  bool partial = false;
  float fe[FR][COLS], fs[FR + 1][COLS], fw[FR];
  if (FACES) {
    const float* south = a.faces + (long long)W * H;
#pragma unroll
    for (int i = 0; i < FR; ++i) load_row(a.faces, gy0 + i, fe[i]);
#pragma unroll
    for (int i = 0; i <= FR; ++i) load_row(south, gy0 - 1 + i, fs[i]);
    // a weight outside [0, 1] is an open face
    auto clean = [](float& w) { w = w >= 0.0f && w < 1.0f ? w : 1.0f; };
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      clean(fs[0][c]);
#pragma unroll
      for (int i = 0; i < FR; ++i) {
        clean(fe[i][c]);
        clean(fs[i + 1][c]);
      }
    }
    bool any = false;
    auto inner = [](float w) { return w > 0.0f && w < 1.0f; };
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        // the grid's edge is the edge rule's business; cells beyond it nobody's
        any |= fe[i][c] != 1.0f && c < right && i <= last;
        any |= fs[i + 1][c] != 1.0f && c <= right && i < last;
        any |= i == 0 && gy0 > 0 && fs[0][c] != 1.0f && c <= right;
        if (c >= right) fe[i][c] = 0.0f;
        if (i >= last) fs[i + 1][c] = 0.0f;
        if (i == 0 && gy0 == 0) fs[0][c] = 0.0f;
        partial |= c <= right && i <= last &&
                   (inner(fe[i][c]) || inner(fs[i + 1][c]) || (i == 0 && inner(fs[0][c])));
      }
#pragma unroll
    for (int i = 0; i < FR; ++i) {
      // west of the lane's first column: the left lane's east face
      fw[i] = lane_from_left(fe[i][COLS - 1]);
      if (gx0 == 0) fw[i] = 0.0f;
      any |= fw[i] != 1.0f && gx0 > 0 && lane > 0 && right >= 0 && i <= last;
      partial |= inner(fw[i]) && right >= 0 && i <= last;
    }
    special = __any(any);
    partial = __any(partial);
  }

  // a pending line-search step, as the apply of the line search would have
  // stored it
  if (a.dapp) {
    const float al = (float)a.line[0];
    if (al != 0.0f) {
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        float la[COLS];
        load_row(a.dapp, gy0 + i, la);
#pragma unroll
        for (int c = 0; c < COLS; ++c)
          if (FACES || !((sol >> ((i + 1) * COLS + c)) & 1)) x[i][c] = x[i][c] + al * la[c];
      }
    }
  }

  __shared__ __attribute__((aligned(16))) float xch[2][2][WAVES][EX];
  // The rows above and below a wave's strip come from its neighbours in the
  // block; the first and the last wave read their own row back: at the grid's
  // edge that is the edge's rule, elsewhere the cells that see it are outside
  // the valid region.
  const bool top = wave == WAVES - 1 || gy0 + ROWS >= H;
  const int dn_slot = wave > 0 ? 1 : 0, dn_wave = wave > 0 ? wave - 1 : 0;
  const int up_slot = top ? 1 : 0, up_wave = top ? wave : wave + 1;
  struct alignas(sizeof(float) * COLS) Cells { float v[COLS]; };
  auto publish = [&](int buf, const float(&v)[ROWS][COLS]) {
    Cells lo, hi;
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      lo.v[c] = v[0][c];
      hi.v[c] = v[ROWS - 1][c];
    }
    *reinterpret_cast<Cells*>(&xch[buf][0][wave][tcol0]) = lo;
    *reinterpret_cast<Cells*>(&xch[buf][1][wave][tcol0]) = hi;
  };
  auto collect = [&](int buf, float(&prev)[COLS], float(&above)[COLS]) {
    __syncthreads();
    const Cells lo = *reinterpret_cast<const Cells*>(&xch[buf][dn_slot][dn_wave][tcol0]);
    const Cells hi = *reinterpret_cast<const Cells*>(&xch[buf][up_slot][up_wave][tcol0]);
#pragma unroll
    for (int c = 0; c < COLS; ++c) {
      prev[c] = lo.v[c];
      above[c] = hi.v[c];
    }
  };

  // the last iteration of a residual launch only adds d to x
  const int full = RES ? max(a.its - 1, 0) : a.its;
  // flag of cell (i, c), all ones where the centre replaces it as a neighbour
  auto flag = [&](int i, int c) -> uint32_t {
    const int bit = c < 0 ? i : c >= COLS ? 16 + i : (i + 1) * COLS + c;
    return (uint32_t)__builtin_amdgcn_sbfe((int)(c < 0 || c >= COLS ? side : sol), bit, 1);
  };
  auto insert = [](uint32_t m, float pc, float v) -> float {
    return __uint_as_float((m & __float_as_uint(pc)) | (~m & __float_as_uint(v)));
  };
  // neighbours of cell (i, c) before any edge rule
  auto around = [&](const float(&v)[ROWS][COLS], int i, int c, const float(&prev)[COLS],
                    const float(&above)[COLS], float& l, float& q, float& u, float& n) {
    l = c > 0 ? v[i][c > 0 ? c - 1 : 0] : lane_shr0(v[i][COLS - 1]);
    q = c < COLS - 1 ? v[i][c < COLS - 1 ? c + 1 : c] : lane_shl0(v[i][0]);
    u = i > 0 ? v[i > 0 ? i - 1 : 0][c] : prev[c];
    n = i < ROWS - 1 ? v[i < ROWS - 1 ? i + 1 : i][c] : above[c];
  };
  auto flagged = [&](float pc, int i, int c, float& l, float& q, float& u, float& n) {
    l = insert(flag(i, c - 1), pc, l);
    q = insert(flag(i, c + 1), pc, q);
    u = insert(flag(i - 1, c), pc, u);
    n = insert(flag(i + 1, c), pc, n);
  };
  int buf = 0;
  // Small strips keep their masks as conditions, lane masks in scalar registers:
  // one select a neighbour.  Larger ones make each mask from its bit where it is
  // used: conditions would take a wave a SIMD from 4 x 2 cells (83 vector registers
  // against 73: 2048^2, 72 iterations without solids, 386 us against 341).
  constexpr bool FEW = ROWS * COLS <= 4;
  // The passes of one wave; XE, YE the edge rules as in the Jacobi tile (XE: 0
  // away from the grid's sides, 1 the tile's first and last column, 2 any
  // column; YE: the grid's last row is inside the strip).  SP: 0 no solid cell and
  // no face but open ones in or next to the strip; 1 solid cells or shut faces,
  // every neighbour taken through its mask; 2 partial faces.
  auto run = [&](auto xec, auto yec, auto spc) {
    constexpr int XE = decltype(xec)::value, SP = decltype(spc)::value;
    constexpr bool YE = decltype(yec)::value;
    // conditions of the strip's neighbours: solid (or beyond the grid) in the
    // strip, in the rows next to it and left and right of the lane's columns; of
    // its faces: shut, and partial
    constexpr bool CONDS = SP && !FACES && FEW;
    constexpr int CR = CONDS ? ROWS + 2 : 1, MR = SP && FACES ? ROWS : 1;
    bool fl[CR][COLS], fo[CR][2], ve[MR][COLS], vs[MR + 1][COLS], vw[MR];
    bool pe[MR][COLS], ps[MR + 1][COLS], pw[MR];
    if (CONDS) {
#pragma unroll
      for (int i = 0; i < CR; ++i) {
        fo[i][0] = (side >> i) & 1;
        fo[i][1] = (side >> (16 + i)) & 1;
#pragma unroll
        for (int c = 0; c < COLS; ++c) fl[i][c] = (sol >> (i * COLS + c)) & 1;
      }
    }
    if (SP && FACES) {
      auto cut = [](float w) { return w > 0.0f && w < 1.0f; };
#pragma unroll
      for (int i = 0; i < MR; ++i) {
        vw[i] = fw[FACES ? i : 0] == 0.0f;
        pw[i] = cut(fw[FACES ? i : 0]);
      }
#pragma unroll
      for (int i = 0; i <= MR; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          vs[i][c] = fs[FACES ? i : 0][c] == 0.0f;
          ps[i][c] = cut(fs[FACES ? i : 0][c]);
          if (i < MR) {
            ve[i < MR ? i : 0][c] = fe[FACES && i < MR ? i : 0][c] == 0.0f;
            pe[i < MR ? i : 0][c] = cut(fe[FACES && i < MR ? i : 0][c]);
          }
        }
    }
    auto through = [&](bool shut, bool cut, float w, float pc, float v) -> float {
      const float o = shut ? pc : v;
      if (SP < 2) return o;
      const float t = __builtin_fmaf(w, v - pc, pc);
      return cut ? t : o;
    };
    auto neighbours = [&](const float(&v)[ROWS][COLS], int i, int c, const float(&prev)[COLS],
                          const float(&above)[COLS], float& l, float& q, float& u, float& n) {
      const float pc = v[i][c];
      around(v, i, c, prev, above, l, q, u, n);
      if (CONDS) {
        const int ci = CONDS ? i : 0, c1 = CONDS ? i + 1 : 0, c2 = CONDS ? i + 2 : 0;
        l = (c > 0 ? fl[c1][c > 0 ? c - 1 : 0] : fo[ci][0]) ? pc : l;
        q = (c < COLS - 1 ? fl[c1][c < COLS - 1 ? c + 1 : c] : fo[ci][1]) ? pc : q;
        u = fl[ci][c] ? pc : u;
        n = fl[c2][c] ? pc : n;
      } else if (SP && !FACES) {
        flagged(pc, i, c, l, q, u, n);
      } else if (SP) {
        const int fi = FACES ? i : 0;
        const int mi = SP && FACES ? i : 0;
        l = through(c > 0 ? ve[mi][c > 0 ? c - 1 : 0] : vw[mi],
                    c > 0 ? pe[mi][c > 0 ? c - 1 : 0] : pw[mi],
                    c > 0 ? fe[fi][c > 0 ? c - 1 : 0] : fw[fi], pc, l);
        q = through(ve[mi][c], pe[mi][c], fe[fi][c], pc, q);
        u = through(vs[mi][c], ps[mi][c], fs[fi][c], pc, u);
        n = through(vs[mi + 1][c], ps[mi + 1][c], fs[FACES ? i + 1 : 0][c], pc, n);
      } else {
        if (XE && c == 0) l = lane == 0 ? pc : l;
        if (XE == 2 || (XE == 1 && c == COLS - 1)) q = c == right ? pc : q;
        if (YE) n = i == last ? pc : n;
      }
    };
    // L v = (((u + l) + r) + d) - 4 v: 4 v is exact, so the fused multiply-add
    // rounds once, like the subtraction
    auto lap = [&](const float(&v)[ROWS][COLS], int i, int c, const float(&prev)[COLS],
                   const float(&above)[COLS]) -> float {
      float l, q, u, n;
      neighbours(v, i, c, prev, above, l, q, u, n);
      return __builtin_fmaf(-4.0f, v[i][c], ((u + l) + q) + n);
    };

    if (a.first) {
      float prev[COLS], above[COLS];
      publish(0, x);
      collect(0, prev, above);
      buf = 1;
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          r[i][c] = lap(x, i, c, prev, above) - r[i][c];
          d[i][c] = r[i][c] / a.theta;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    // Small strips (up to 8 cells a lane) are bound by the exchange's latency:
    // half of the inner rows run while the neighbours' rows are on their way out
    // of LDS, then the edge rows, published at once, then what is left.  Larger
    // ones are walked downwards and upwards in turn: a new row takes the registers
    // of the old one before it and two iterations bring every row back.
    constexpr bool SMALL = ROWS * COLS <= 8;
    auto iterate = [&](auto downc, int it, const float(&in)[ROWS][COLS], float(&out)[ROWS][COLS]) {
      constexpr bool DOWN = decltype(downc)::value;
      float prev[COLS], above[COLS];
      collect(buf, prev, above);
      buf ^= 1;
      if (SP && !FACES && !CONDS) asm volatile("" : "+v"(sol), "+v"(side));  // masks made where used
      const float cdd = cf.cd[a.first + it], crr = cf.cr[a.first + it];
      auto row = [&](int i) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          r[i][c] = r[i][c] + lap(in, i, c, prev, above);
          out[i][c] = __builtin_fmaf(cdd, in[i][c], crr * r[i][c]);
        }
      };
      auto add = [&](int i) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) x[i][c] = x[i][c] + in[i][c];
      };
      if (SMALL) {
        constexpr int HALF = 1 + (ROWS - 2) / 2;
#pragma unroll
        for (int i = 1; i < HALF; ++i) row(i);
        __builtin_amdgcn_sched_barrier(0);
        row(0);
        if (ROWS > 1) row(ROWS - 1);
        publish(buf, out);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = HALF; i < ROWS - 1; ++i) row(i);
#pragma unroll
        for (int i = 0; i < ROWS; ++i) add(i);
      } else {
#pragma unroll
        for (int k = 0; k < ROWS; ++k) {
          const int i = DOWN ? k : ROWS - 1 - k;
          add(i);
          row(i);
          __builtin_amdgcn_sched_barrier(0);  // keep the walk: fewer rows live
        }
        publish(buf, out);
      }
    };
    publish(buf, d);
    float e[ROWS][COLS];
    int it = 0;
    while (it + 1 < full) {
      iterate(std::true_type(), it, d, e);
      iterate(std::false_type(), it + 1, e, d);
      it += 2;
    }
    if (it < full) {
      iterate(std::true_type(), it, d, e);
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) d[i][c] = e[i][c];
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  if (idle) {
    for (int s = 0; s < a.first + full; ++s) __syncthreads();
  } else if (FACES && partial) {
    run(I0(), I0(), I2());
  } else if (special) {
    run(I0(), I0(), I1());
  } else if (W < EX || gy0 + ROWS > H) {
    run(I2(), I1(), I0());
  } else if (bx == 0 || bx == nx - 1) {
    run(I1(), I0(), I0());
  } else {
    run(I0(), I0(), I0());
  }

  double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (RES) {
    if (a.its > 0)
#pragma unroll
      for (int i = 0; i < ROWS; ++i)
#pragma unroll
        for (int c = 0; c < COLS; ++c) x[i][c] = x[i][c] + d[i][c];
    float prev[COLS], above[COLS], bb[ROWS][COLS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      load_row(a.b, gy0 + i, bb[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
    publish(buf, x);
    collect(buf, prev, above);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const bool row_in = gy0 + i >= ay.own0 && gy0 + i < ay.own1;
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        float l, q, u, n;
        around(x, i, c, prev, above, l, q, u, n);
        flagged(x[i][c], i, c, l, q, u, n);
        if (row_in && gx0 + c >= ax.own0 && gx0 + c < ax.own1 && flag(i, c) == 0) {
          const double bd = (double)bb[i][c];
          const double rr = bd - (((((double)l + (double)q) + (double)u) + (double)n) -
                                  4.0 * (double)x[i][c]);
          acc[0] += rr;
          acc[1] += rr * rr;
          acc[2] += bd;
          acc[3] += bd * bd;
          acc[4] += 1.0;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  const bool whole = gx0 >= ax.own0 && gx0 + COLS <= ax.own1;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int gy = gy0 + i;
    if (gy < ay.own0 || gy >= ay.own1) continue;
    const long long row = (long long)gy * W + ax.o;
    if (whole) {
      store_cols<F32S, COLS>(a.xout + row, tcol0, x[i]);
      if (a.rout) {
        store_cols<F32S, COLS>(a.rout + row, tcol0, r[i]);
        store_cols<F32S, COLS>(a.dout + row, tcol0, d[i]);
      }
    } else {
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        if (gx0 + c < ax.own0 || gx0 + c >= ax.own1) continue;
        (a.xout + row)[tcol0 + c] = x[i][c];
        if (a.rout) {
          (a.rout + row)[tcol0 + c] = r[i][c];
          (a.dout + row)[tcol0 + c] = d[i][c];
        }
      }
    }
  }

  if (RES) {
    __shared__ double part[WAVES][5];
#pragma unroll
    for (int j = 0; j < 5; ++j) acc[j] = wave_sum(acc[j]);
    if (lane == 0)
#pragma unroll
      for (int j = 0; j < 5; ++j) part[wave][j] = acc[j];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int j = 0; j < 5; ++j) {
        double t = 0.0;
        for (int w = 0; w < WAVES; ++w) t += part[w][j];
        a.red[5 * tile + j] = t;
      }
  }
}

}  // namespace jt
}  // namespace nx
