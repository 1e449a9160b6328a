// Several Euler steps per launch on block tiles (temporal blocking with the
// state in registers).
//
// A block of NW waves owns a tile of NW R rows and 64 columns (one per lane)
// and advances it up to K steps ("levels"). Wave w keeps u, v, w and the static
// coefficients (D and its two first differences) of its R rows in registers
// for the whole launch. Per level a wave needs u on 4 rows above and below its
// own: each wave puts its rows of u in LDS, one barrier, and reads its
// neighbours' 8 rows (two buffers, so one barrier per level); along the columns
// the neighbours come from the lanes next door (DPP).
//
// What bounds it. A dependent launch costs 2.2 us on this GPU and its loads and
// stores 1.5 to 5 us more that nothing overlaps in a grid of one round of
// tiles; K steps share both, and the stencil's static parts. A wave whose cells
// are all at rest, or all excited, evaluates only its side of the gates. A
// level is then about 61 VALU operations per cell (105 in the one-step kernel).
// Against that stand the 4 K columns on each inner side of the tile that only
// feed the stencil and 4 rows per level and side (a wave outside the rows that
// later levels reach skips the level). On a small grid a level takes 1.0 to
// 1.3 us whatever its rows: the latency of one wave's 250 operations.
// Measured figures stand at the rule that chooses the tiling (auto_variant).
//
// Arithmetic. Every cell of every level is computed by the operations of
// stream_tile in the same order (contraction off, explicit fmaf), so K levels
// equal K launches of k_stream bit for bit.
//
// Boundaries (cardiax/solve.py:225-254: edge padding, one-sided differences).
// Columns: a tile that reaches over a side holds the column beyond it, which
// takes the edge column's value at load time (clamped loads) and after every
// level; the one-sided rules are compiled in for those tiles only. Rows: a wave
// whose window reaches over an edge takes the edge's rules, at compile time
// where it holds exactly the grid's first or last rows, else by row index.
#pragma once

#include <type_traits>

#include "fk_stream.h"
#include "fk_stream_t.h"

namespace fk {

// Tiles along one axis of N cells: T cells per tile of which the outer h on an
// inner side only feed the stencil; pad cells beyond the grid at its ends.
// Outputs are disjoint: tile s writes [a, b).
struct BlockAxis {
  int n, N, T, h, pad;
};

struct BlockSpan {
  int o, a, b;  // first cell of the tile (may lie beyond the grid), outputs [a, b)
};

__host__ __device__ inline BlockAxis make_block_axis(int N, int T, int h, int pad) {
  BlockAxis x{1, N, T, h, pad};
  if (N + 2 * pad > T) {
    const int rest = N - 2 * (T - pad - h), inner = T - 2 * h;
    x.n = 2 + (rest > 0 ? (rest + inner - 1) / inner : 0);
  }
  return x;
}

__host__ __device__ inline BlockSpan block_span(const BlockAxis& x, int s) {
  const int first = x.T - x.pad - x.h, inner = x.T - 2 * x.h;
  BlockSpan p;
  p.a = s == 0 ? 0 : first + (s - 1) * inner;
  p.b = s == x.n - 1 ? x.N : first + s * inner;
  p.o = s == 0 ? -x.pad : s == x.n - 1 ? x.N + x.pad - x.T : p.a - x.h;
  return p;
}

template <int R, int NW, int K>
struct BlockCfg {
  static constexpr int rows = R, waves = NW, steps = K;
  static constexpr int T = NW * R, C = 64;            // owned rows, columns
  static constexpr int hr = 4 * (K - 1), hc = 4 * K;  // rows, columns that only feed the stencil
  static_assert(R >= 2 && T - 2 * hr >= 2 && C - 2 * hc >= 2, "tile too small for its levels");
  static __host__ __device__ BlockAxis row_axis(int H) { return make_block_axis(H, T, hr, 0); }
  static __host__ __device__ BlockAxis col_axis(int W) { return make_block_axis(W, C, hc, 1); }
  static constexpr int buf = (T + 8) * C;  // floats of one LDS buffer: tile rows -4 .. T+3
  static constexpr int lds_floats = 2 * buf;
};

// Stimulus fields of a launch: field m is active at level l when bit m of
// act[l] is set (list order, later ones override).
constexpr int kBlockMaxSteps = 4;
struct BlockStim {
  uint32_t act[kBlockMaxSteps];
  const float* f[FK_MAX_STIMULI];
};

struct BlockStimArgs {
  const BlockStim& s;
  __device__ uint32_t active(int l) const { return s.act[l]; }
  __device__ const float* field(int m) const { return s.f[m]; }
};

// 12 x first differences across columns, by the rules of d1_lanes. YG: bit 0
// the tile reaches over the left side, bit 1 over the right one; left / right:
// the lane's column is <= 0 / >= W-1 and takes the one-sided rule. (Also the
// second difference from first differences: its one-sided columns are 0 and
// W-1, and nothing reads it beyond the grid.) Every lane evaluates every shift.
template <int YG>
__device__ __forceinline__ float diff_cols(float x, bool left, bool right) {
#pragma clang fp contract(off)
  const float m1 = from_left(x), p1 = from_right(x);
  const float m2 = from_left(m1), p2 = from_right(p1);
  float g = s1_interior(m2, m1, p1, p2);
  if constexpr (YG & 1) {
    const float f = s1_forward(x, p1, p2, from_right(p2));
    g = left ? f : g;
  }
  if constexpr (YG & 2) {
    const float b = s1_backward(from_left(m2), m2, m1, x);
    g = right ? b : g;
  }
  return g;
}

// Which side of the gate u >= V_c the cells of a wave lie on.
enum GateSide { kRest, kExcited, kMixed };

// Gates and currents of reaction() by the same operations, one side only
// where the whole wave lies on it.
template <int SIDE>
__device__ __forceinline__ void reaction_side(const Coef& c, float v, float w, float u, float& dv,
                                              float& dw, float& jion) {
#pragma clang fp contract(off)
  if constexpr (SIDE == kMixed) {
    reaction_sel(c, v, w, u, dv, dw, jion);
  } else {
    float fo;
    if constexpr (SIDE == kExcited) {
      const float a = (u - c.V_c) * (1.0f - u);
      fo = fmaf(-(v * a), c.inv_td, c.inv_tr);
      dv = -v * c.inv_tvp;
      dw = -w * c.inv_twp;
    } else {
      fo = u * c.inv_t0;
      const float inv_tvm = (u >= c.V_v) ? c.inv_tv2m : c.inv_tv1m;
      dv = (1.0f - v) * inv_tvm;
      dw = (1.0f - w) * c.inv_twm;
    }
    const float s = fmaf(-(w * c.inv_tsi), half_one_plus_tanh(c, u), fo);
    jion = -s * c.inv_cm;
  }
}

// Inputs and outputs of a tile. Level l (from 1) writes to o_* + (l - 1)
// o_stride when `all` is set (a trajectory), else the last one to o_*.
struct BlockIO {
  const float *D, *v, *w, *u;
  float *o_v, *o_w, *o_u;
  size_t o_stride;
  bool all;
};

// How the window of 4 rows on each side of a wave's rows i0 .. i0+R-1 lies:
// inside the grid, over its top with i0 = 0, over its bottom with i0 + R = H,
// or any other overlap.
enum RowEdge { kInside, kTop, kBottom, kAnyEdge };

__device__ __forceinline__ int row_edge(int i0, int R, int H) {
  if (i0 >= 4 && i0 + R + 4 <= H) return kInside;
  if (i0 == 0 && R + 4 <= H) return kTop;
  if (i0 >= 4 && i0 + R == H) return kBottom;
  return kAnyEdge;
}

// The tile at (rsp, csp) over n_lev <= K levels. lds: Cfg::lds_floats floats.
// Every wave of the block calls it (a barrier between levels). HEUN: levels
// come in pairs, the two stages of a Heun step (cardiax/solve.py:73-85): an odd
// level forms x1 = x0 + dt k1 and keeps x0 and k1, the even one x0 + (k1 + k2)
// dt / 2, by the operations of stream_tile's stages; n_lev is even.
template <class Cfg, int YG, bool HEUN, class SV>
__device__ __forceinline__ void block_tile(const Coef& c, const BlockIO& io, int H, int W,
                                           const SV& sv, int n_lev, float dt, float inv_dx2,
                                           const BlockSpan& rsp, const BlockSpan& csp,
                                           float* lds) {
#pragma clang fp contract(off)  // explicit fmaf only: the rounding of stream_tile
  constexpr int R = Cfg::rows, T = Cfg::T, C = Cfg::C;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int i0 = rsp.o + wave * R;  // first row of the wave
  const int col = csp.o + lane;
  const uint32_t off = (uint32_t)(YG ? clampi(col, 0, W - 1) : col) * 4u;
  const bool left = col <= 0, right = col >= W - 1;
  auto row = [&](const float* a, int r) { return a + (size_t)clampi(r, 0, H - 1) * (size_t)W; };
  auto ldr = [&](const float* a, int r) { return ld(row(a, r), off); };
  // LDS by tile row t in [-4, T+4), this lane's column
  auto cell = [&](int buf, int t) -> float& { return lds[buf * Cfg::buf + (t + 4) * C + lane]; };
  // grid row r, clamped into the grid and what LDS holds
  auto lds_row = [&](int buf, int r) {
    return cell(buf, clampi(clampi(r, 0, H - 1) - rsp.o, -4, T + 3));
  };
  const int xe = row_edge(i0, R, H);
  const float k2 = inv_dx2 * (1.0f / 144.0f);

  float u[R], v[R], w[R], Dc[R], Dx[R], Dy[R];
  float x0[HEUN ? 3 * R : 1], k1[HEUN ? 3 * R : 1];  // v, w, u of the rows
#pragma unroll
  for (int k = 0; k < R; ++k) {
    u[k] = ldr(io.u, i0 + k);
    Dc[k] = ldr(io.D, i0 + k);
  }
  // the rows beyond the tile that its first level reads: 4 of u (buffer 0) and
  // 2 of D (buffer 1) above and below, one row per wave
  for (int h = wave; h < 12; h += Cfg::waves) {
    const int t = h < 4 ? h - 4 : h < 8 ? T + h - 4 : h < 10 ? h - 10 : T + h - 10;
    cell(h < 8 ? 0 : 1, t) = ldr(h < 8 ? io.u : io.D, rsp.o + t);
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    v[k] = ldr(io.v, i0 + k);
    w[k] = ldr(io.w, i0 + k);
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    cell(0, wave * R + k) = u[k];
    cell(1, wave * R + k) = Dc[k];
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < R; ++k) Dy[k] = diff_cols<YG>(Dc[k], left, right);
  auto slope_D = [&](auto edge) {  // 12 D_x of the wave's rows
    constexpr int XE = decltype(edge)::value;
    if constexpr (XE != kAnyEdge) {
      float dd[R + 4];  // D rows i0-2 .. i0+R+1
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        dd[k] = XE == kTop ? Dc[0] : cell(1, wave * R - 2 + k);
        dd[R + 2 + k] = XE == kBottom ? Dc[R - 1] : cell(1, wave * R + R + k);
      }
#pragma unroll
      for (int k = 0; k < R; ++k) dd[k + 2] = Dc[k];
#pragma unroll
      for (int k = 0; k < R; ++k)
        Dx[k] = XE == kTop && k == 0 ? s1_forward(dd[2], dd[3], dd[4], dd[5])
                : XE == kBottom && k == R - 1
                    ? s1_backward(dd[R - 2], dd[R - 1], dd[R], dd[R + 1])
                    : s1_interior(dd[k], dd[k + 1], dd[k + 3], dd[k + 4]);
    } else {
      float dd[R + 6];  // D rows i0-3 .. i0+R+2
#pragma unroll
      for (int k = 0; k < R + 6; ++k) dd[k] = lds_row(1, i0 - 3 + k);
#pragma unroll
      for (int k = 0; k < R; ++k) {
        float g = s1_interior(dd[k + 1], dd[k + 2], dd[k + 4], dd[k + 5]);
        if (k == 0 && i0 == 0)  // row 0 is the first row of a wave
          g = s1_forward(dd[3], dd[4], dd[5], dd[6]);
        else if (i0 + k == H - 1)
          g = s1_backward(dd[k], dd[k + 1], dd[k + 2], dd[k + 3]);
        Dx[k] = g;
      }
    }
  };
  switch (xe) {
    case kInside: slope_D(std::integral_constant<int, kInside>{}); break;
    case kTop: slope_D(std::integral_constant<int, kTop>{}); break;
    case kBottom: slope_D(std::integral_constant<int, kBottom>{}); break;
    default: slope_D(std::integral_constant<int, kAnyEdge>{}); break;
  }
  lds_barrier();  // buffer 1 may be overwritten

#pragma unroll 1
  for (int l = 1; l <= n_lev; ++l) {
    const int in = (l - 1) & 1, out = l & 1;
    // the wave's first row, opaque to the loop: row addresses derived from it
    // are recomputed per level instead of being kept in registers for all
    int ib = i0;
    asm volatile("" : "+s"(ib));
    // rows later levels still reach: 4 per level, 5 at an edge's one-sided rule
    const int reach = (rsp.o == 0 || rsp.o + T >= H ? 5 : 4) * (n_lev - l);
    const bool need = i0 < min(H, rsp.b + reach) && i0 + R > max(0, rsp.a - reach);
    if (need) {
      float del[R];  // the diffusion term
      auto diffuse = [&](int k, float uxx, float gx) {
        const float gy = diff_cols<YG>(u[k], left, right);
        const float uyy = diff_cols<YG>(gy, left, right);
        del[k] = fmaf(Dy[k], gy, fmaf(Dx[k], gx, Dc[k] * (uxx + uyy))) * k2;
      };
      auto diffusion = [&](auto edge) {
        constexpr int XE = decltype(edge)::value;
        if constexpr (XE != kAnyEdge) {
          float win[R + 8];  // u rows i-4 .. i+R+3 (i = ib)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            win[k] = XE == kTop ? u[0] : cell(in, wave * R - 4 + k);
            win[R + 4 + k] = XE == kBottom ? u[R - 1] : cell(in, wave * R + R + k);
          }
#pragma unroll
          for (int k = 0; k < R; ++k) win[k + 4] = u[k];
          float gx[R + 4];  // 12 u_x at rows i-2 .. i+R+1
#pragma unroll
          for (int k = 0; k < R + 4; ++k)
            gx[k] = XE == kTop && (k == 1 || k == 2)
                        ? s1_forward(win[k + 2], win[k + 3], win[k + 4], win[k + 5])
                    : XE == kBottom && (k == R + 1 || k == R + 2)
                        ? s1_backward(win[k - 1], win[k], win[k + 1], win[k + 2])
                        : s1_interior(win[k], win[k + 1], win[k + 3], win[k + 4]);
#pragma unroll
          for (int k = 0; k < R; ++k)
            diffuse(k,
                    XE == kTop && k == 0 ? s1_forward(gx[2], gx[3], gx[4], gx[5])
                    : XE == kBottom && k == R - 1
                        ? s1_backward(gx[R - 2], gx[R - 1], gx[R], gx[R + 1])
                        : s1_interior(gx[k], gx[k + 1], gx[k + 3], gx[k + 4]),
                    gx[k + 2]);
        } else {
          float win[R + 9];  // u rows i-5 .. i+R+3
#pragma unroll
          for (int k = 0; k < R + 9; ++k) win[k] = lds_row(in, ib - 5 + k);
          float gx[R + 5];  // 12 u_x at rows p = i-3 .. i+R+1, each by its rule
#pragma unroll
          for (int k = 0; k < R + 5; ++k) {
            const int p = ib - 3 + k;
            float g = s1_interior(win[k], win[k + 1], win[k + 3], win[k + 4]);
            if (k + 5 < R + 9 && p <= 0)  // p <= 0 lies in the window's first rows
              g = s1_forward(win[k + 2], win[k + 3], win[k + 4], win[k + 5 < R + 9 ? k + 5 : 0]);
            else if (k >= 1 && p >= H - 1)
              g = s1_backward(win[k >= 1 ? k - 1 : 0], win[k], win[k + 1], win[k + 2]);
            gx[k] = g;
          }
#pragma unroll
          for (int k = 0; k < R; ++k) {
            float uxx = s1_interior(gx[k + 1], gx[k + 2], gx[k + 4], gx[k + 5 < R + 5 ? k + 5 : R + 4]);
            if (k == 0 && ib == 0)
              uxx = s1_forward(gx[3], gx[4], gx[5], gx[6]);
            else if (ib + k == H - 1)
              uxx = s1_backward(gx[k], gx[k + 1], gx[k + 2], gx[k + 3]);
            diffuse(k, uxx, gx[k + 3]);
          }
        }
      };
      switch (xe) {
        case kInside: diffusion(std::integral_constant<int, kInside>{}); break;
        case kTop: diffusion(std::integral_constant<int, kTop>{}); break;
        case kBottom: diffusion(std::integral_constant<int, kBottom>{}); break;
        default: diffusion(std::integral_constant<int, kAnyEdge>{}); break;
      }
      uint64_t any = 0, all = ~0ull;  // cells with u >= V_c
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const uint64_t p = __builtin_amdgcn_ballot_w64(u[k] >= c.V_c);
        any |= p;
        all &= p;
      }
      const uint32_t act = sv.active(l - 1);
      auto react = [&](auto side) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
          float dv, dw, jion;
          reaction_side<decltype(side)::value>(c, v[k], w[k], u[k], dv, dw, jion);
          if (decltype(side)::value == kMixed && act) {
            float sval = 0.0f;
            for (uint32_t m = act; m; m &= m - 1) {
              const float f = ldr(sv.field(__builtin_ctz(m)), ib + k);
              sval = (f != 0.0f) ? f : sval;
            }
            jion = (sval != 0.0f) ? sval : jion;
          }
          const float du = del[k] + jion;
          if (HEUN && (l & 1) == 0) {
            const float half = dt * 0.5f;
            v[k] = fmaf(k1[3 * k] + dv, half, x0[3 * k]);
            w[k] = fmaf(k1[3 * k + 1] + dw, half, x0[3 * k + 1]);
            u[k] = fmaf(k1[3 * k + 2] + du, half, x0[3 * k + 2]);
            continue;
          }
          if constexpr (HEUN) {
            x0[3 * k] = v[k], x0[3 * k + 1] = w[k], x0[3 * k + 2] = u[k];
            k1[3 * k] = dv, k1[3 * k + 1] = dw, k1[3 * k + 2] = du;
          }
          v[k] = fmaf(dt, dv, v[k]);
          w[k] = fmaf(dt, dw, w[k]);
          u[k] = fmaf(dt, du, u[k]);
        }
      };
      if (any == 0 && !act)
        react(std::integral_constant<int, kRest>{});
      else if (all == ~0ull && !act)
        react(std::integral_constant<int, kExcited>{});
      else
        react(std::integral_constant<int, kMixed>{});
      if constexpr (YG & 1) {  // column -1 (lane 0) takes column 0's value
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int e = __builtin_amdgcn_readlane(__float_as_int(u[k]), 1);
          u[k] = lane == 0 ? __int_as_float(e) : u[k];
        }
      }
      if constexpr (YG & 2) {  // column W takes column W-1's value
        const int pw = W - csp.o;  // its lane
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int e = __builtin_amdgcn_readlane(__float_as_int(u[k]), pw - 1);
          u[k] = lane == pw ? __int_as_float(e) : u[k];
        }
      }
      if (l < n_lev)
#pragma unroll
        for (int k = 0; k < R; ++k) cell(out, wave * R + k) = u[k];
      if ((io.all || l == n_lev) && col >= csp.a && col < csp.b) {
        const size_t lo = io.all ? (size_t)(l - 1) * io.o_stride : 0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
          const int i = ib + k;
          if (i < rsp.a || i >= rsp.b) continue;
          const size_t ro = lo + (size_t)i * (size_t)W;
          st(io.o_v + ro, off, v[k]);
          st(io.o_w + ro, off, w[k]);
          st(io.o_u + ro, off, u[k]);
        }
      }
    }
    if (l < n_lev) lds_barrier();
  }
}

// The sides a column span reaches over: the YG of block_tile.
__device__ __forceinline__ int block_sides(const BlockSpan& c, int C, int W) {
  return (c.o < 0 ? 1 : 0) | (c.o + C > W ? 2 : 0);
}

// block_tile over the spans of one tile, by the sides it reaches over.
template <class Cfg, bool HEUN, class SV>
__device__ __forceinline__ void block_tile_any(const Coef& c, const BlockIO& io, int H, int W,
                                               const SV& sv, int n_lev, float dt, float inv_dx2,
                                               const BlockSpan& r, const BlockSpan& s,
                                               float* lds) {
  switch (block_sides(s, Cfg::C, W)) {
    case 0: block_tile<Cfg, 0, HEUN>(c, io, H, W, sv, n_lev, dt, inv_dx2, r, s, lds); break;
    case 1: block_tile<Cfg, 1, HEUN>(c, io, H, W, sv, n_lev, dt, inv_dx2, r, s, lds); break;
    case 2: block_tile<Cfg, 2, HEUN>(c, io, H, W, sv, n_lev, dt, inv_dx2, r, s, lds); break;
    default: block_tile<Cfg, 3, HEUN>(c, io, H, W, sv, n_lev, dt, inv_dx2, r, s, lds); break;
  }
}

// Which tile a workgroup of k_block takes. Workgroup b runs on XCD b % 8, and
// each XCD has an L2 of its own: an XCD takes a contiguous run of the tiles
// ordered by groups of 8 bands, strip by strip within a group, so the 32 to 96
// tiles it has in flight form a patch whose shared halos (2 of 3 rows and a
// third of the columns are read by a neighbour too) come from its L2. In plain
// order (bands of a strip, workgroup b tile b) every neighbour sits on another
// XCD; times per step of the 32-row 2-step tiling, plain and so: 760^2 5.2 and
// 4.2 us, 1200^2 9.4 and 7.3, 2048^2 22.4 and 15.9, 4096^2 90 and 69. Groups of
// 4 or 16 bands are within 3% of 8, of 32 up to 15% slower. A solve's launches
// go through each run forward and backward in turn (`back`): where the fields
// exceed the 256 MB cache, what a launch wrote last is still there for the next
// (4096^2 69.9 and 66.5 us per step, 5000^2 104 and 100; no change below).
constexpr int kBlockGroup = 8;

struct BlockOrder {
  int per_xcd, extra;  // the first `extra` XCDs take one tile more
  float inv_group;     // 1 / tiles of a group of bands
  int back;            // each XCD's run from its end
};

struct BlockPlace {
  int band, strip;
};

inline BlockOrder make_block_order(const BlockAxis& ra, const BlockAxis& ca, bool back) {
  const int n = ra.n * ca.n;
  return {n / kXcds, n % kXcds, 1.0f / (float)(kBlockGroup * ca.n), back ? 1 : 0};
}

__device__ __forceinline__ BlockPlace block_place(int b, const BlockOrder& o, const BlockAxis& ra,
                                                  const BlockAxis& ca) {
  const int x = b % kXcds, k = b / kXcds;
  const int last = o.per_xcd - (x < o.extra ? 0 : 1);
  const int t = x * o.per_xcd + min(x, o.extra) + (o.back ? last - k : k);
  const int per = kBlockGroup * ca.n;
  // t / per: the float quotient is within one of it (below 2^15, t below 2^24)
  int g = __builtin_amdgcn_readfirstlane((int)((float)t * o.inv_group));
  g -= g * per > t;
  g += (g + 1) * per <= t;
  const int rem = t - g * per, left = ra.n - g * kBlockGroup;
  const int strip = left >= kBlockGroup ? rem / kBlockGroup : rem / left;
  const int bands = min(left, kBlockGroup);
  return {g * kBlockGroup + rem - strip * bands, strip};
}

template <class Cfg, bool HEUN>
__global__ void __launch_bounds__(Cfg::waves * 64)
k_block(Coef c, BlockIO io, int H, int W, BlockStim st, int n_lev, float dt, float inv_dx2,
        BlockAxis ra, BlockAxis ca, BlockOrder ord) {
  __shared__ float lds[Cfg::lds_floats];
  const BlockPlace at = block_place(blockIdx.x, ord, ra, ca);
  const BlockStimArgs sv{st};
  block_tile_any<Cfg, HEUN>(c, io, H, W, sv, n_lev, dt, inv_dx2, block_span(ra, at.band),
                            block_span(ca, at.strip), lds);
}

// The tilings of Euler steps, and the choice among those offered. A launch takes
// the GPU's 256 CUs in rounds of tiles, and each tiling's time per step is close
// to a + b ceil(tiles / 256) us, measured from 64^2 to 2500^2: few steps per
// launch cost the launch (a), many cost the columns and rows that only feed the
// stencil (b). The least is taken. Of the tilings tried (1 and 2 columns per lane,
// 2 to 6 rows per wave, 4 to 16 waves, 2 to 4 steps) these four were the fastest
// somewhere. Where a step's 28 bytes per cell exceed the 256 MB cache, two steps
// per launch wait for memory (32 rows 66.5 us at 4096^2 and 100 at 5000^2, 48 rows
// and three steps 65.1 and 95.3; at 3000^2 30.8 and 34.7): a larger b there.
typedef BlockCfg<2, 16, 4> Block32x4;
typedef BlockCfg<4, 8, 2> Block32x2;
typedef BlockCfg<4, 12, 3> Block48x3;
typedef BlockCfg<4, 16, 3> Block64x3;

struct LeastRounds {
  const bool streams;
  int best = -1;
  double least = 0.0;
  explicit LeastRounds(int64_t cells) : streams(28 * cells > (256 << 20)) {}
  void offer(int id, int64_t tiles, double a, double b) {
    const double us = a + b * (double)((tiles + 255) / 256);
    if (best < 0 || us < least) best = id, least = us;
  }
  void offer(int id, Block32x4, int64_t tiles) { offer(id, tiles, 1.0, 1.05); }
  void offer(int id, Block48x3, int64_t tiles) { offer(id, tiles, 1.7, 1.25); }
  void offer(int id, Block64x3, int64_t tiles) { offer(id, tiles, 1.4, 2.05); }
  void offer(int id, Block32x2, int64_t tiles) { offer(id, tiles, 2.2, streams ? 1.15 : 1.0); }
};

template <class Cfg>
inline int64_t block_tiles(int H, int W) {
  return (int64_t)Cfg::row_axis(H).n * Cfg::col_axis(W).n;
}

}  // namespace fk
