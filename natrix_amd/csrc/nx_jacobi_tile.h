// Temporal-blocked Jacobi tile (shared by the single-grid and batched
// kernels); see nx_jacobi.hip for the scheme.
#pragma once
#include <type_traits>

#include "nx_common.h"

namespace nx {
namespace jt {

// Waves per SIMD asked of the compiler for a tile kernel of CELLS cells
// per lane (amdgpu_waves_per_eu).  Jacobi: what the strip,
// its right-hand side and, next to solids, its masks fit in without spills in
// the sweeps; asked for one step more (8 for 16 cells, 5 for 32) the spills
// cost more than the waves give (2048^2, three simulators in turn: (12, 8, 8, 2)
// 1.51 to 1.58 us per sweep, (13, 8, 8, 2) 1.42 to 1.47).
template <int CELLS>
constexpr int jacobi_waves_per_eu() {
  return CELLS <= 8 ? 8 : CELLS <= 16 ? 6 : CELLS <= 32 ? 4 : 2;
}
__device__ __forceinline__ double wave_sum(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ float lane_from_left(float v) {
  // lane i receives lane i-1 (wave_shr:1); lane 0 keeps its own value
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x138,
                                  0xf, 0xf, false));
}

__device__ __forceinline__ float lane_from_right(float v) {
  // lane i receives lane i+1 (wave_shl:1); lane 63 keeps its own value
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), 0x130,
                                  0xf, 0xf, false));
}

__device__ __forceinline__ int ilane_from_left(int v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false);
}

__device__ __forceinline__ int ilane_from_right(int v) {
  return __builtin_amdgcn_update_dpp(v, v, 0x130, 0xf, 0xf, false);
}

// The same shifts with the edge lane reading 0 (bound_ctrl): no old value
// to keep, so the compiler folds the shift into the instruction that
// consumes it as a DPP source operand (v_add_f32_dpp), at no cost of its
// own.  For callers whose edge lanes hold cells outside the valid region.
__device__ __forceinline__ float lane_shr0(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}

__device__ __forceinline__ float lane_shl0(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));
}

// ---- tiling -----------------------------------------------------------
// Tiles of E cells along an axis of N cells for k sweeps.  Every tile lies
// inside the grid (as long as N >= E): the first starts at cell 0, the last
// ends at cell N, and where a tile meets the grid's edge the edge's own rule
// (a neighbour beyond it is the centre value) holds exactly, so there the
// valid region does not shrink with the sweeps.  Only sides inside the grid
// lose k cells: tile i starts at min(i (E - 2k), N - E) and owns cells
// [i (E - 2k) + k, (i + 1) (E - 2k) + k), the first from 0, the last to N.
// Against tiles laid with a halo of k beyond the grid's edges this loads no
// cell that does not exist and needs no out-of-grid rule in the sweeps: a
// 2048^2 grid at k = 10 on 128 x 128 tiles takes 19 x 19 tiles either way, a
// 128^2 grid one instead of four.
__host__ __device__ constexpr int axis_tiles(int N, int E, int k) {
  return N <= E ? 1 : 1 + (N - E + (E - 2 * k) - 1) / (E - 2 * k);
}

struct AxisTile {
  int o;         // first cell
  int own0, own1;  // cells the tile writes
};

__device__ __forceinline__ AxisTile axis_tile(int i, int n, int N, int E, int k) {
  const int V = E - 2 * k;
  AxisTile t;
  t.o = n == 1 ? 0 : min(i * V, N - E);
  t.own0 = i == 0 ? 0 : i * V + k;
  t.own1 = i == n - 1 ? N : (i + 1) * V + k;
  return t;
}

// COLS consecutive stored values as one access.  The address is aligned to one
// of them only (odd grid widths), which the hardware's wide accesses allow.
template <int BYTES>
struct RawBits;
template <>
struct RawBits<1> { using type = uint8_t; };
template <>
struct RawBits<2> { using type = uint16_t; };
template <>
struct RawBits<4> { using type = uint32_t; };
template <class T, int COLS>
struct Pack {
  using raw = typename RawBits<sizeof(T)>::type;
  typedef raw type __attribute__((ext_vector_type(COLS), aligned(sizeof(raw))));
};

template <class S, int COLS>
__device__ __forceinline__ void load_cols(const typename S::s1* __restrict__ p, int i,
                                          float (&out)[COLS]) {
  using P = Pack<typename S::s1, COLS>;
  const typename P::type t = *reinterpret_cast<const typename P::type*>(p + i);
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    const typename P::raw v = t[c];
    out[c] = S::ld(reinterpret_cast<const typename S::s1*>(&v), 0);
  }
}

template <class S, int COLS>
__device__ __forceinline__ void store_cols(typename S::s1* __restrict__ p, int i,
                                           const float (&in)[COLS]) {
  using P = Pack<typename S::s1, COLS>;
  typename P::type t;
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    typename P::raw v;
    S::st(reinterpret_cast<typename S::s1*>(&v), 0, in[c]);
    t[c] = v;
  }
  *reinterpret_cast<typename P::type*>(p + i) = t;
}

// The projection a tile runs on the pressure it ends with (SubtractGradient.
// comp:24-46 and the obstacle clear): velocity in place, the next step's mask.
template <class S>
struct Project {
  typename S::s2* u;
  uint8_t* mask_next;
};

// ROWS x COLS cells per lane: lane `l` of wave `w` owns tile columns
// [COLS*l, COLS*l + COLS) and tile rows [ROWS*w, ROWS*w + ROWS).
// k sweeps on tile (bx, by) of the nx x ny tiles of a W x H grid; `rid` is
// the partial-sum record this tile writes when RES.  Uses __syncthreads():
// every thread of the block must call it.
// p and b are stored in format S and held in float32 registers across the k
// sweeps; p is rounded to S once, at the store.
// RES: the last sweep also accumulates the FP64 residual of its input iterate
// over the tile's own fluid cells.
// CORR (residual correction): the first of the k passes computes the float32
// residual r = b - A p of the stored iterate instead of a sweep, the other
// k-1 passes are Jacobi sweeps of A e = r from e = 0, and the tile writes
// the float32 pressure p + e to pout32 (pout is unused).
// PROJ: the tile also projects the velocity with the pressure it ends with
// (p + e with CORR), which needs the pressure's neighbours: it owns what k + 1
// sweeps would leave valid.
template <int ROWS, int WAVES, int COLS, class S = F32S, bool CORR = false, bool RES = false,
          bool PROJ = false>
__device__ __forceinline__ void jacobi_tb_tile(
    int bx, int by, int nx, int ny, const typename S::s1* __restrict__ pin,
    const typename S::s1* __restrict__ b, const uint8_t* __restrict__ mask,
    typename S::s1* __restrict__ pout, int W, int H, int k,
    double* __restrict__ red, int rid, float* __restrict__ pout32 = nullptr,
    const Project<S>& proj = Project<S>{nullptr, nullptr}) {
  constexpr int EX = 64 * COLS, EY = ROWS * WAVES;
  const int lane = threadIdx.x & 63;
  // wave-uniform: a scalar register, so branches on it are scalar branches
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kt = PROJ ? k + 1 : k;
  const AxisTile ax = axis_tile(bx, nx, W, EX, kt), ay = axis_tile(by, ny, H, EY, kt);
  const int tcol0 = COLS * lane;
  const int gx0 = ax.o + tcol0, gy0 = ay.o + wave * ROWS;

  // a wave that lies beyond a grid smaller than the tile only keeps the
  // block's barriers
  const bool idle = gy0 >= H;

  // Rows are addressed by a scalar row pointer plus the lane's column offset.
  // All of a lane's loads are issued before the first is used; the scheduling
  // barriers keep the row pointers from piling up in scalar registers.
  float p[ROWS][COLS], bb[ROWS][COLS];
  static_assert(COLS <= 4, "a row's mask bytes in one word");
  // mask bytes of the lane's columns in row y, clamped to the grid: cells
  // beyond it read its edge, a value no cell of the grid uses
  auto mask_at = [&](int y) -> uint32_t {
    const uint8_t* row = mask + (long long)min(max(y, 0), H - 1) * W;
    uint32_t m = 0;
#pragma unroll
    for (int c = 0; c < COLS; ++c) m |= (uint32_t)row[min(gx0 + c, W - 1)] << (8 * c);
    return m;
  };
  // the masks of the strip's rows and, last, of the rows below and above it, a
  // byte a column: kept from this one read until the waves with solids have their
  // bits (a second read by those waves alone, a memory latency more per launch,
  // took 5 to 8 % of a step with obstacles: 1024^2, (10, 4, 16, 2), rectangles
  // 140.9 against 129.9 us)
  uint32_t mrow[ROWS + 2];
  if (W >= EX && H >= EY) {  // the whole tile is inside the grid
    // not aligned to more than a byte
    typedef typename RawBits<COLS>::type M __attribute__((aligned(1), may_alias));
    auto mask_in = [&](int y) -> uint32_t {
      return *reinterpret_cast<const M*>(mask + (long long)y * W + ax.o + tcol0);
    };
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const long long row = (long long)(gy0 + r) * W + ax.o;
      load_cols<S, COLS>(pin + row, tcol0, p[r]);
      load_cols<S, COLS>(b + row, tcol0, bb[r]);
      mrow[r] = mask_in(gy0 + r);
      __builtin_amdgcn_sched_barrier(0);
    }
    mrow[ROWS] = mask_in(max(gy0 - 1, 0));
    mrow[ROWS + 1] = mask_in(min(gy0 + ROWS, H - 1));
  } else {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int y = min(gy0 + r, H - 1);
#pragma unroll
      for (int c = 0; c < COLS; ++c) {
        p[r][c] = S::ld(pin + (long long)y * W, min(gx0 + c, W - 1));
        bb[r][c] = S::ld(b + (long long)y * W, min(gx0 + c, W - 1));
      }
      mrow[r] = mask_at(y);
      __builtin_amdgcn_sched_barrier(0);
    }
    mrow[ROWS] = mask_at(gy0 - 1);
    mrow[ROWS + 1] = mask_at(gy0 + ROWS);
  }
  uint32_t any = 0;
#pragma unroll
  for (int r = 0; r < ROWS + 2; ++r) any |= mrow[r];
  const bool special = __any(any != 0);
  // one bit per solid cell of the strip and of the rows next to it, made by the
  // waves that have any
  constexpr int WORDS = (ROWS * COLS + 31) / 32;
  uint32_t sol[WORDS], sol_lo = 0, sol_hi = 0;
#pragma unroll
  for (int w = 0; w < WORDS; ++w) sol[w] = 0;
  if (special) {
    auto bits = [](uint32_t m) -> uint32_t {
      uint32_t v = 0;
#pragma unroll
      for (int c = 0; c < COLS; ++c) v |= ((m >> (8 * c)) & 0xFF ? 1u : 0u) << c;
      return v;
    };
#pragma unroll
    for (int r = 0; r < ROWS; ++r) sol[r * COLS / 32] |= bits(mrow[r]) << (r * COLS % 32);
    sol_lo = bits(mrow[ROWS]);
    sol_hi = bits(mrow[ROWS + 1]);
  }
  static_assert(32 % COLS == 0, "a row's bits in one word");
  auto solid = [&](int r, int c) -> uint32_t {  // r = -1, ROWS: the rows next to the strip
    if (r < 0) return (sol_lo >> c) & 1;
    if (r >= ROWS) return (sol_hi >> c) & 1;
    return (sol[(r * COLS + c) >> 5] >> ((r * COLS + c) & 31)) & 1;
  };

  __shared__ __attribute__((aligned(16))) float xch[2][2][WAVES][EX];
  // The rows above and below a wave's strip come from its neighbours in the
  // block.  The first and the last wave read their own row back: at the
  // grid's edge that is the edge's rule, elsewhere the cells that see it are
  // outside the valid region.
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

  constexpr bool SMALL = ROWS * COLS <= 8;
  // Small strips of few rows keep their masks as conditions, one lane mask in
  // scalar registers each (20 pairs for 4 x 2 cells), which saves an extraction
  // per side and the vector registers; 8 rows' 26 pairs spill (1024^2 bf16, 100
  // iterations: (10, 4, 16, 2) with obstacles 138.6 to 135.7 us a step, (10, 8, 8,
  // 1) without any 132 to 134.5).
  constexpr bool CONDS = SMALL && ROWS <= 4;
  double sr = 0.0, srr = 0.0;
  // The passes of one wave.  XE, the x neighbours at the grid's sides: 0 none
  // (a tile away from them), 1 the tile's first and last column, 2 any column
  // (a grid narrower than the tile).  YE: the grid's last row is inside the
  // strip (a grid lower than the tile).  SP, solid cells: 0 none in or next to
  // the strip; 1 some: every neighbour is taken through the mask of its cell,
  // all ones where the centre replaces it, one bit-field insert (cells beyond
  // the grid count as solid); 2 only solid cells in and next to the strip:
  // every neighbour is the centre, nothing is read from other lanes or waves.
  // Lane 0's left and lane 63's right neighbour are outside the valid region
  // unless an edge rule says otherwise; the zero-filled lane shift folds into
  // the addition.
  auto run = [&](auto xec, auto yec, auto spc) {
    constexpr int XE = decltype(xec)::value, SP = decltype(spc)::value;
    constexpr bool YE = decltype(yec)::value;
    const int right = W - 1 - gx0;  // the lane's column of the grid's last cell
    const int last = H - 1 - gy0;   // the strip's row of the grid's last row
    // masks of the lane's cells and of the rows next to the strip; bits of the
    // cells left and right of the lane's columns, 2 per row
    constexpr int MR = SP == 1 ? ROWS + 2 : 1, OW = SP == 1 ? (2 * ROWS + 31) / 32 : 1;
    uint32_t msk[MR][COLS], outer[OW];
    bool fl[MR][COLS], fo[MR][2];
    if (SP == 1 && CONDS) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int l = ilane_from_left((int)solid(r, COLS - 1));
        const int q = ilane_from_right((int)solid(r, 0));
        fo[SP == 1 ? r : 0][0] = gx0 == 0 || l != 0;
        fo[SP == 1 ? r : 0][1] = right < COLS || q != 0;
      }
#pragma unroll
      for (int r = -1; r <= ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c)
          fl[SP == 1 ? r + 1 : 0][c] = c > right || r > last || solid(r, c) != 0;
    } else if (SP == 1) {
#pragma unroll
      for (int q = 0; q < OW; ++q) outer[q] = 0;
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t fl = (uint32_t)ilane_from_left((int)solid(r, COLS - 1));
        const uint32_t fr = (uint32_t)ilane_from_right((int)solid(r, 0));
        outer[2 * r / 32] |= (gx0 == 0 ? 1u : fl) << (2 * r % 32);
        outer[2 * r / 32] |= (right < COLS ? 1u : fr) << ((2 * r + 1) % 32);
      }
#pragma unroll
      for (int r = -1; r <= ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c)
          msk[SP == 1 ? r + 1 : 0][c] =
              c > right || r > last ? 0xFFFFFFFFu
                                    : (uint32_t)__builtin_amdgcn_sbfe((int)solid(r, c), 0, 1);
    }
    auto insert = [](uint32_t m, float pc, float x) -> float {
      return __uint_as_float((m & __float_as_uint(pc)) | (~m & __float_as_uint(x)));
    };
    auto neighbours = [&](const float(&v)[ROWS][COLS], int r, int c, const float(&prev)[COLS],
                          const float(&above)[COLS], float& x1, float& x2, float& y1, float& y2) {
      const float pc = v[r][c];
      if (SP == 2) {
        x1 = x2 = y1 = y2 = pc;
        return;
      }
      x1 = c > 0 ? v[r][c > 0 ? c - 1 : 0] : lane_shr0(v[r][COLS - 1]);
      x2 = c < COLS - 1 ? v[r][c < COLS - 1 ? c + 1 : c] : lane_shl0(v[r][0]);
      y1 = r > 0 ? v[r > 0 ? r - 1 : 0][c] : prev[c];
      y2 = r < ROWS - 1 ? v[r < ROWS - 1 ? r + 1 : r][c] : above[c];
      if (SP == 1 && CONDS) {
        const int m = SP == 1 ? r : 0;
        const int m1 = SP == 1 ? r + 1 : 0, m2 = SP == 1 ? r + 2 : 0;
        x1 = (c > 0 ? fl[m1][c > 0 ? c - 1 : 0] : fo[m][0]) ? pc : x1;
        x2 = (c < COLS - 1 ? fl[m1][c < COLS - 1 ? c + 1 : c] : fo[m][1]) ? pc : x2;
        y1 = fl[m][c] ? pc : y1;
        y2 = fl[m2][c] ? pc : y2;
      } else if (SP == 1) {
        auto side = [&](int bit) -> uint32_t {
          return (uint32_t)__builtin_amdgcn_sbfe((int)outer[SP == 1 ? (2 * r + bit) / 32 : 0],
                                                 (2 * r + bit) % 32, 1);
        };
        x1 = insert(c > 0 ? msk[SP == 1 ? r + 1 : 0][c > 0 ? c - 1 : 0] : side(0), pc, x1);
        x2 = insert(c < COLS - 1 ? msk[SP == 1 ? r + 1 : 0][c < COLS - 1 ? c + 1 : c] : side(1),
                    pc, x2);
        y1 = insert(msk[SP == 1 ? r : 0][c], pc, y1);
        y2 = insert(msk[SP == 1 ? r + 2 : 0][c], pc, y2);
      } else {
        if (XE && c == 0) x1 = lane == 0 ? pc : x1;
        if (XE == 2 || (XE == 1 && c == COLS - 1)) x2 = c == right ? pc : x2;
        if (YE) y2 = r == last ? pc : y2;
      }
    };
    // pass s reads the edge rows published in buffer s & 1 and publishes its own
    // for the next; one barrier a pass
    int s = 0;
    publish(0, p);
    if (CORR) {
      // pass 0: r = b - ((((x1 + x2) + y1) + y2) - 4 p), float32
      float prev[COLS], above[COLS];
      collect(0, prev, above);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          float x1, x2, y1, y2;
          neighbours(p, r, c, prev, above, x1, x2, y1, y2);
          bb[r][c] = bb[r][c] - ((((x1 + x2) + y1) + y2) - 4.0f * p[r][c]);
        }
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) p[r][c] = 0.0f;
      s = 1;
      publish(1, p);
    }
    // Small strips (up to 8 cells a lane), bound by the exchange's latency: half
    // of the inner rows run while the neighbours' rows are on their way out of
    // LDS, then the edge rows, which are published at once, then the other half
    // while those are on their way in.
    // Larger ones walk the strip row by row, upwards and downwards in turn: when
    // row r is done the old row before it is dead, so the new row can take its
    // registers, and two sweeps bring every row back to where it was.  A strip
    // lives in ROWS + 1 rows of registers, without copies and without a second
    // strip of neighbour sums.
    auto sweep = [&](auto upc, const float(&in)[ROWS][COLS], float(&out)[ROWS][COLS]) {
      constexpr bool UP = decltype(upc)::value;
      float prev[COLS], above[COLS];
      auto row = [&](int r) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          float x1, x2, y1, y2;
          neighbours(in, r, c, prev, above, x1, x2, y1, y2);
          out[r][c] = ((((x1 + x2) + y1) + y2) - bb[r][c]) * 0.25f;
        }
      };
      collect(s & 1, prev, above);
      ++s;
      if (SMALL) {
        constexpr int HALF = 1 + (ROWS - 2) / 2;
#pragma unroll
        for (int r = 1; r < HALF; ++r) row(r);
        __builtin_amdgcn_sched_barrier(0);
        row(0);
        if (ROWS > 1) row(ROWS - 1);
        publish(s & 1, out);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = HALF; r < ROWS - 1; ++r) row(r);
      } else {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
          row(UP ? i : ROWS - 1 - i);
          __builtin_amdgcn_sched_barrier(0);  // keep the walk: fewer rows live
        }
        publish(s & 1, out);
      }
    };
    const int plain = RES ? k - 1 : k;
    float q[ROWS][COLS];
    while (s + 1 < plain) {
      sweep(std::true_type(), p, q);
      sweep(std::false_type(), q, p);
    }
    if (s < plain) {
      sweep(std::true_type(), p, q);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) p[r][c] = q[r][c];
    }
    if (RES) {
      float prev[COLS], above[COLS], np[ROWS][COLS];
      collect(s & 1, prev, above);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          float x1, x2, y1, y2;
          neighbours(p, r, c, prev, above, x1, x2, y1, y2);
          np[r][c] = ((((x1 + x2) + y1) + y2) - bb[r][c]) * 0.25f;
          const int gx = gx0 + c, gy = gy0 + r;
          if (gx >= ax.own0 && gx < ax.own1 && gy >= ay.own0 && gy < ay.own1 &&
              solid(r, c) == 0) {
            const double rr =
                (double)bb[r][c] -
                (((((double)x1 + (double)x2) + (double)y1) + (double)y2) - 4.0 * (double)p[r][c]);
            sr += rr;
            srr += rr * rr;
          }
        }
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c) p[r][c] = np[r][c];
    }
    if (PROJ) {
      if (CORR) {
        // the pressure the projection takes is the stored iterate + e
#pragma unroll
        for (int r = 0; r < ROWS; ++r)
#pragma unroll
          for (int c = 0; c < COLS; ++c)
            p[r][c] = S::ld(pin + (long long)min(gy0 + r, H - 1) * W, min(gx0 + c, W - 1)) +
                      p[r][c];
        publish(s & 1, p);
      }
      float prev[COLS], above[COLS];
      collect(s & 1, prev, above);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const int gy = gy0 + r;
        if (gy < ay.own0 || gy >= ay.own1) continue;
        const long long row = (long long)gy * W + ax.o;
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
          float x1, x2, y1, y2;
          neighbours(p, r, c, prev, above, x1, x2, y1, y2);
          if (gx0 + c >= ax.own0 && gx0 + c < ax.own1) {
            float2 v = S::ld2(proj.u + row, tcol0 + c);
            v.x -= 0.5f * (x2 - x1);
            v.y -= 0.5f * (y2 - y1);
            S::st2(proj.u + row, tcol0 + c, v);
            (proj.mask_next + row)[tcol0 + c] = (mask + row)[tcol0 + c] & MASK_PERSIST;
          }
        }
      }
    }
  };

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  if (idle) {
    for (int s = 0; s < kt; ++s) __syncthreads();
  } else if (special) {
    bool all = sol_lo == (1u << COLS) - 1 && sol_hi == (1u << COLS) - 1;
#pragma unroll
    for (int w = 0; w < WORDS; ++w)
      all &= sol[w] == (ROWS * COLS >= 32 * (w + 1) ? 0xFFFFFFFFu
                                                    : (1u << (ROWS * COLS % 32)) - 1);
    if (__all(all) && W >= EX && gy0 + ROWS <= H)
      run(I0(), I0(), I2());
    else
      run(I0(), I0(), I1());
  } else if (W < EX || gy0 + ROWS > H) {
    run(I2(), I1(), I0());
  } else if (bx == 0 || bx == nx - 1) {
    run(I1(), I0(), I0());
  } else {
    run(I0(), I0(), I0());
  }

  const bool whole = gx0 >= ax.own0 && gx0 + COLS <= ax.own1;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int gy = gy0 + r;
    if (gy < ay.own0 || gy >= ay.own1) continue;
    const long long row = (long long)gy * W + ax.o;
    if (CORR) {
#pragma unroll
      for (int c = 0; c < COLS; ++c)
        if (gx0 + c >= ax.own0 && gx0 + c < ax.own1)
          (pout32 + row)[tcol0 + c] = PROJ ? p[r][c] : S::ld(pin + row, tcol0 + c) + p[r][c];
    } else if (whole) {
      store_cols<S, COLS>(pout + row, tcol0, p[r]);
    } else {
#pragma unroll
      for (int c = 0; c < COLS; ++c)
        if (gx0 + c >= ax.own0 && gx0 + c < ax.own1) S::st(pout + row, tcol0 + c, p[r][c]);
    }
  }

  if (RES) {
    __shared__ double part[WAVES][2];
    sr = wave_sum(sr);
    srr = wave_sum(srr);
    if (lane == 0) {
      part[wave][0] = sr;
      part[wave][1] = srr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double a = 0.0, c2 = 0.0;
      for (int w = 0; w < WAVES; ++w) {
        a += part[w][0];
        c2 += part[w][1];
      }
      red[2 * rid + 0] = a;
      red[2 * rid + 1] = c2;
    }
  }
}

}  // namespace jt
}  // namespace nx
