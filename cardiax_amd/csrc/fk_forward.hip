// Forward kernels of the Fenton-Karma step and the C-ABI entry points of the
// single-simulation path (include/cardiax_amd.h).
//
// Two kernels compute the same step (cardiax/solve.py:26-70):
//   k_plain  one thread per cell, every neighbour read from global memory with
//            clamped indices (the edge padding), no LDS. The unoptimised
//            baseline and a structurally independent cross-check.
//   k_tile   64 x TH output tile per 256-thread workgroup. u (halo 4) and D
//            (halo 2) are staged in LDS once; the first derivatives u_x, u_y
//            are formed once per cell into LDS and reused by the 5-point second
//            derivative; v, w are read straight from HBM into registers. One
//            HBM pass per step: read v, w, u, D, write v, w, u.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "cardiax_amd.h"
#include "fk_block.h"
#include "fk_device.h"
#include "fk_host.h"
#include "fk_stream.h"
#include "fk_stream2.h"
#include "fk_stream_t.h"

namespace fk {

// ---------------------------------------------------------------------------
// Plain kernel
// ---------------------------------------------------------------------------
template <bool EULER>
__global__ void __launch_bounds__(256)
k_plain(Coef c, const float* __restrict__ D, const float* __restrict__ v,
        const float* __restrict__ w, const float* __restrict__ u, int H, int W, StimArgs sa,
        float dt, float inv_dx2, float* __restrict__ o_v, float* __restrict__ o_w,
        float* __restrict__ o_u) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  const int i = blockIdx.y * 4 + threadIdx.y;
  if (i >= H || j >= W) return;
  cell_general<EULER>(c, D, v, w, u, H, W, i, j, sa, dt, inv_dx2, o_v, o_w, o_u);
}

// ---------------------------------------------------------------------------
// LDS-tiled kernel
// ---------------------------------------------------------------------------
constexpr int TW = 64;  // tile width = one wavefront of columns

// Tile origin along an axis of N cells: tiles of T cells, the last one shifted
// back to end at N (overlapping its neighbour, which then writes identical
// values twice) so that every cell at index N-1 sits >= 3 rows inside its tile
// and the one-sided rules only read inside the staged halo.
__device__ __forceinline__ int tile_origin(int b, int T, int N) {
  const int o = b * T;
  return (N >= T && o > N - T) ? N - T : o;
}

template <int TH, bool EULER>
__global__ void __launch_bounds__(256)
k_tile(Coef c, const float* __restrict__ D, const float* __restrict__ v,
       const float* __restrict__ w, const float* __restrict__ u, int H, int W, StimArgs sa,
       float dt, float inv_dx2, float* __restrict__ o_v, float* __restrict__ o_w,
       float* __restrict__ o_u) {
  static_assert(TH % 4 == 0, "TH must be a multiple of 4");
  constexpr int UR = TH + 8, UC = TW + 8;  // u, halo 4
  constexpr int DR = TH + 4, DC = TW + 4;  // D, halo 2
  constexpr int NU = UR / 4, ND = DR / 4, NO = TH / 4;  // rows per wave
  __shared__ float s_u[UR][UC];
  __shared__ float s_D[DR][DC];
  __shared__ float s_gx[TH + 4][TW];  // u_x at tile rows -2 .. TH+1
  __shared__ float s_gy[TH][TW + 4];  // u_y at tile cols -2 .. TW+1

  const int lane = threadIdx.x;  // column in tile
  const int wv = threadIdx.y;    // 0..3
  const int r0 = tile_origin(blockIdx.y, TH, H);
  const int c0 = tile_origin(blockIdx.x, TW, W);

  // Issue every global load of the tile before the first LDS store so their
  // latencies overlap. Clamped indices *are* the edge padding.
  float ru[NU], ru2[NU], rD[ND], rD2[ND], rv[NO], rw[NO];
  const int cu = clampi(c0 - 4 + lane, 0, W - 1), cu2 = clampi(c0 + TW - 4 + lane, 0, W - 1);
  const int cd = clampi(c0 - 2 + lane, 0, W - 1), cd2 = clampi(c0 + TW - 2 + lane, 0, W - 1);
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    const float* row = u + (size_t)clampi(r0 - 4 + wv + 4 * k, 0, H - 1) * W;
    ru[k] = row[cu];
    ru2[k] = lane < 8 ? row[cu2] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    const float* row = D + (size_t)clampi(r0 - 2 + wv + 4 * k, 0, H - 1) * W;
    rD[k] = row[cd];
    rD2[k] = lane < 4 ? row[cd2] : 0.0f;
  }
  const int gj = c0 + lane, gjc = min(gj, W - 1);
#pragma unroll
  for (int k = 0; k < NO; ++k) {
    const size_t idx = (size_t)min(r0 + wv + 4 * k, H - 1) * W + gjc;
    rv[k] = v[idx];
    rw[k] = w[idx];
  }
#pragma unroll
  for (int k = 0; k < NU; ++k) {
    s_u[wv + 4 * k][lane] = ru[k];
    if (lane < 8) s_u[wv + 4 * k][TW + lane] = ru2[k];
  }
#pragma unroll
  for (int k = 0; k < ND; ++k) {
    s_D[wv + 4 * k][lane] = rD[k];
    if (lane < 4) s_D[wv + 4 * k][TW + lane] = rD2[k];
  }
  __syncthreads();

  // Every first/second derivative this tile needs is a central one.
  const bool interior =
      (r0 >= 3) && (r0 + TH + 3 <= H) && (c0 >= 3) && (c0 + TW + 3 <= W);

  // u_x on tile rows lr in [-2, TH+2), column `lane`; u_y on rows [0, TH),
  // tile columns lc in [-2, TW+2).
  if (interior) {
#pragma unroll
    for (int k = 0; k < (TH + 4) / 4; ++k) {
      const int r = wv + 4 * k;
      const int a = r + 2;  // s_u row of tile row lr = r - 2
      s_gx[r][lane] = d1_interior(s_u[a - 2][lane + 4], s_u[a - 1][lane + 4],
                                  s_u[a + 1][lane + 4], s_u[a + 2][lane + 4]);
    }
#pragma unroll
    for (int k = 0; k < TH / 4; ++k) {
      const int r = wv + 4 * k;
      const float* ur = s_u[r + 4];
      {
        const int b = lane + 2;  // s_u column of tile column lc = lane - 2
        s_gy[r][lane] = d1_interior(ur[b - 2], ur[b - 1], ur[b + 1], ur[b + 2]);
      }
      if (lane < 4) {
        const int b = TW + 2 + lane;
        s_gy[r][TW + lane] = d1_interior(ur[b - 2], ur[b - 1], ur[b + 1], ur[b + 2]);
      }
    }
  } else {
    for (int r = wv; r < TH + 4; r += 4) {
      const int q = r0 + r - 2;  // global row
      auto f = [&](int gr) { return s_u[gr - r0 + 4][lane + 4]; };
      s_gx[r][lane] = d1_general(f, q, H);
    }
    for (int r = wv; r < TH; r += 4) {
      const float* ur = s_u[r + 4];
      auto f = [&](int gc) { return ur[gc - c0 + 4]; };
      s_gy[r][lane] = d1_general(f, c0 + lane - 2, W);
      if (lane < 4) s_gy[r][TW + lane] = d1_general(f, c0 + TW - 2 + lane, W);
    }
  }
  __syncthreads();

#pragma unroll
  for (int k = 0; k < NO; ++k) {
    const int r = wv + 4 * k;
    const int gi = r0 + r;
    float uxx, uyy, dDx, dDy;
    if (interior) {
      uxx = d1_interior(s_gx[r][lane], s_gx[r + 1][lane], s_gx[r + 3][lane],
                        s_gx[r + 4][lane]);
      uyy = d1_interior(s_gy[r][lane], s_gy[r][lane + 1], s_gy[r][lane + 3],
                        s_gy[r][lane + 4]);
      dDx = d1_interior(s_D[r][lane + 2], s_D[r + 1][lane + 2], s_D[r + 3][lane + 2],
                        s_D[r + 4][lane + 2]);
      dDy = d1_interior(s_D[r + 2][lane], s_D[r + 2][lane + 1], s_D[r + 2][lane + 3],
                        s_D[r + 2][lane + 4]);
    } else {
      auto gx = [&](int q) { return s_gx[q - r0 + 2][lane]; };
      auto gy = [&](int q) { return s_gy[r][q - c0 + 2]; };
      auto Dx = [&](int q) { return s_D[q - r0 + 2][lane + 2]; };
      auto Dy = [&](int q) { return s_D[r + 2][q - c0 + 2]; };
      uxx = d2_from_d1(gx, gi, H);
      uyy = d2_from_d1(gy, gj, W);
      dDx = d1_general(Dx, gi, H);
      dDy = d1_general(Dy, gj, W);
    }
    if (gi >= H || gj >= W) continue;
    const float Dc = s_D[r + 2][lane + 2];
    const float del_u =
        (Dc * (uxx + uyy) + dDx * s_gx[r + 2][lane] + dDy * s_gy[r][lane + 2]) * inv_dx2;
    const size_t idx = (size_t)gi * W + gj;
    const float vc = rv[k], wc = rw[k], uc = s_u[r + 4][lane + 4];
    float dv, dw, jion;
    reaction(c, vc, wc, uc, dv, dw, jion);
    jion = stimulate_cell(sa, idx, jion);
    const float du = del_u + jion;
    if (EULER) {
      o_v[idx] = vc + dt * dv;
      o_w[idx] = wc + dt * dw;
      o_u[idx] = uc + dt * du;
    } else {
      o_v[idx] = dv;
      o_w[idx] = dw;
      o_u[idx] = du;
    }
  }
}


// ---------------------------------------------------------------------------
// Small kernels: init, gradient, stimulate
// ---------------------------------------------------------------------------
// Static diffusion coefficients of one cell, precomputed once per solve:
// (D, 12 D_x, 12 D_y) with the reference's rules (edge padding, one-sided
// differences at the two outermost padded entries), each times
// inv_dx2 / 144, so that the step's diffusion term is
// x (12^2 u_xx + 12^2 u_yy) + y (12 u_x) + z (12 u_y).
__global__ void __launch_bounds__(256)
k_stream_coef(const float* __restrict__ D, int H, int W, float k2, float4* __restrict__ cf) {
  const int j = blockIdx.x * 64 + (threadIdx.x & 63);
  const int i = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= H || j >= W) return;
  auto at = [&](int r, int q) {
    return D[(size_t)clampi(r, 0, H - 1) * W + clampi(q, 0, W - 1)];
  };
  float dx, dy;
  if (i == 0) dx = s1_forward(at(0, j), at(1, j), at(2, j), at(3, j));
  else if (i == H - 1) dx = s1_backward(at(i - 3, j), at(i - 2, j), at(i - 1, j), at(i, j));
  else dx = s1_interior(at(i - 2, j), at(i - 1, j), at(i + 1, j), at(i + 2, j));
  if (j == 0) dy = s1_forward(at(i, 0), at(i, 1), at(i, 2), at(i, 3));
  else if (j == W - 1) dy = s1_backward(at(i, j - 3), at(i, j - 2), at(i, j - 1), at(i, j));
  else dy = s1_interior(at(i, j - 2), at(i, j - 1), at(i, j + 1), at(i, j + 2));
  cf[(size_t)i * W + j] = make_float4(at(i, j) * k2, dx * k2, dy * k2, 0.0f);
}

__global__ void k_fill(float* a, size_t n, float x) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    a[i] = x;
}

// field = x on columns [0, c1) of every row, 0 elsewhere.
__global__ void k_fill_cols(float* a, int H, int W, int c1, float x) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)H * W;
       i += (size_t)gridDim.x * blockDim.x)
    a[i] = (int)(i % (size_t)W) < c1 ? x : 0.0f;
}

__global__ void k_init(float* v, float* w, float* u, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    v[i] = 1.0f;
    w[i] = 1.0f;
    u[i] = 0.0f;
  }
}

// Sets *flag when any of the n values is NaN or infinite. The flag word is
// cleared by k_clear_flag first (a kernel rather than a memset, so the pair
// can sit in a captured graph).
__global__ void k_clear_flag(unsigned* flag) {
  if (blockIdx.x == 0 && threadIdx.x == 0) flag[0] = 0u;
}

__global__ void __launch_bounds__(256)
k_nonfinite(const float* __restrict__ a, int64_t n, unsigned* flag) {
  bool bad = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * 256)
    bad |= !isfinite(a[i]);
  if (bad) atomicOr(flag, 1u);
}

// cardiax/solve.py:225-254 on an unpadded (rows, cols) array.
__global__ void k_gradient(const float* __restrict__ a, float* __restrict__ out, int rows,
                           int cols, int axis) {
  const int j = blockIdx.x * 64 + threadIdx.x;
  const int i = blockIdx.y * 4 + threadIdx.y;
  if (i >= rows || j >= cols) return;
  const int n = axis == 0 ? rows : cols;
  const int p = axis == 0 ? i : j;
  auto f = [&](int k) {
    return axis == 0 ? a[(size_t)k * cols + j] : a[(size_t)i * cols + k];
  };
  float g;
  if (p <= 1)
    g = d1_forward(f(p), f(p + 1), f(p + 2), f(p + 3));
  else if (p >= n - 2)
    g = d1_backward(f(p - 3), f(p - 2), f(p - 1), f(p));
  else
    g = d1_interior(f(p - 2), f(p - 1), f(p + 1), f(p + 2));
  out[(size_t)i * cols + j] = g;
}

__global__ void k_stimulate(const float* __restrict__ X, float* __restrict__ out, int64_t n,
                            StimArgs sa) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = stimulate_cell(sa, (size_t)i, X[i]);
}

// ---------------------------------------------------------------------------
// Host-side launch helpers
// ---------------------------------------------------------------------------
// Kernel variants of one step (the value of fk_set_forward_variant).
enum Variant : int {
  kAuto = 0,
  kPlain = 1,
  kTile16 = 2,
  kTile32 = 3,
  kStream8 = 4,
  kStream16 = 5,
  kStream32 = 6,
  kBlock32x2 = 7,   // block tiles (fk_block.h) of 32 rows, 2 steps per launch
  kBlock48x3 = 8,   // 48 rows, 3 steps
  kBlock64x3 = 9,   // 64 rows, 3 steps
  kBlock32x4 = 10,  // 32 rows, 4 steps
  kStreamC8 = 11,   // streaming bands of 8 / 16 rows with the static diffusion
  kStreamC16 = 12,  // coefficients precomputed once per solve
  kStream4 = 13,    // streaming bands of 4 rows
  kStreamC4 = 14,   // ... with precomputed coefficients
  kStream2 = 15,    // streaming bands of 2 rows
  kStreamC2 = 16,   // ... with precomputed coefficients
  kPair2 = 17,      // streaming bands of 2 / 4 rows, two adjacent columns per lane
  kPair4 = 18,      // (W odd: the one-column kernels 15 / 13)
  kStreamT8 = 19,   // two steps per launch on streaming bands of 8 / 12 / 16 / 24
  kStreamT12 = 20,  // rows (grids too small for them: 15)
  kStreamT16 = 21,
  kStreamT24 = 22,
  kNumVariants = 23
};

static bool is_pc(int v) {
  return v == kStreamC8 || v == kStreamC16 || v == kStreamC4 || v == kStreamC2;
}

// The streaming variant a precomputed-coefficient variant falls back to for
// single steps.
static int pc_base(int v) {
  return v == kStreamC8 ? kStream8 : v == kStreamC4 ? kStream4 : v == kStreamC2 ? kStream2
                                                                                 : kStream16;
}

static bool is_block(int v) { return v >= kBlock32x2 && v <= kBlock32x4; }

static int block_steps(int v) { return v == kBlock32x2 ? 2 : v == kBlock32x4 ? 4 : 3; }

// Steps of the next launch of block variant v with `left` to go, and in *v the
// variant that runs them. Where a step's fields exceed the 256 MB cache (`streams`),
// a tile of three steps takes as long for two of them as for three, so a solve of
// 3 a + 1 or 3 a + 2 steps ends in two launches or one of two steps on 32 rows
// (4096^2: two steps 140 us in place of 189, four 278 in place of 353).
static int block_launch(int* v, int64_t left, bool streams) {
  if (streams && *v == kBlock48x3 && (left == 2 || left == 4)) {
    *v = kBlock32x2;
    return 2;
  }
  return (int)std::min<int64_t>(block_steps(*v), left);
}

static bool is_two_step(int v) { return v >= kStreamT8 && v <= kStreamT24; }

// Whether the two-step variant v fits an H x W grid (else stream2 runs).
static bool two_step_fits(int v, int H, int W) {
  switch (v) {
    case kStreamT8: return stream_t_fits<8>(H, W);
    case kStreamT12: return stream_t_fits<12>(H, W);
    case kStreamT16: return stream_t_fits<16>(H, W);
    default: return stream_t_fits<24>(H, W);
  }
}

template <int R>
static void launch_stream_t(const Coef& c, const float* D, const float* v, const float* w,
                            const float* u, int H, int W, const StimArgs& s1,
                            const StimArgs& s2, float dt, float inv_dx2, float* ov, float* ow,
                            float* ou, hipStream_t s) {
  const StreamTGeom g = make_stream_t_geom<R>(H, W);
  k_stream_t<R><<<g.blocks, 256, 0, s>>>(c, D, v, w, u, H, W, s1, s2, dt, inv_dx2, ov, ow, ou,
                                         g);
}

// Two Euler steps (times t and t+1) with the two-step variant v.
static hipError_t launch_two_step(int v, const Coef& c, const float* D, const float* x0,
                                  const float* x1, const float* x2, int H, int W,
                                  const StimArgs& s1, const StimArgs& s2, float dt,
                                  float inv_dx2, float* ov, float* ow, float* ou,
                                  hipStream_t s) {
  switch (v) {
    case kStreamT8: launch_stream_t<8>(c, D, x0, x1, x2, H, W, s1, s2, dt, inv_dx2, ov, ow, ou, s); break;
    case kStreamT12: launch_stream_t<12>(c, D, x0, x1, x2, H, W, s1, s2, dt, inv_dx2, ov, ow, ou, s); break;
    case kStreamT16: launch_stream_t<16>(c, D, x0, x1, x2, H, W, s1, s2, dt, inv_dx2, ov, ow, ou, s); break;
    default: launch_stream_t<24>(c, D, x0, x1, x2, H, W, s1, s2, dt, inv_dx2, ov, ow, ou, s); break;
  }
  return hipGetLastError();
}

static std::atomic<int> g_variant{kAuto};

int current_forward_variant() { return g_variant.load(); }

// Autotuner results: grid shape -> fastest variant measured on this device
// (fk_autotune_forward). Read on every automatic launch, written by the
// tuner; guarded by a mutex.
static std::mutex g_tune_mu;
static std::map<std::pair<int, int>, int> g_tuned;

static int tuned_variant(int H, int W) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  const auto it = g_tuned.find({H, W});
  return it == g_tuned.end() ? (int)kAuto : it->second;
}

// Streaming default when no variant is set and the shape was not tuned: the
// kernel of single steps, and what auto_variant's solves replace. Up to 1.1 M
// cells, streaming bands of 2 rows: small bands give enough waves to hide
// latency, and a grid this small is limited by issue rate more than by memory.
// Above, two steps per launch (bands of 8 rows up to 2.5 M cells, of 16 above),
// which single steps run as 2-row bands. Grids too small for those run 4-row
// bands up to 8 M cells and the LDS tile above.
static int default_variant(int H, int W) {
  const size_t n = (size_t)H * W;
  if (n <= 1100 * 1024) return kStream2;
  if (n <= 2560 * 1024 && stream_t_fits<8>(H, W)) return kStreamT8;
  if (stream_t_fits<16>(H, W)) return kStreamT16;
  return n <= 8 * 1024 * 1024 ? (int)kStream4 : (int)kTile16;
}
// The variant an automatic solve of several steps runs when the shape was not
// tuned: block tiles, which equal the streaming kernels of default_variant bit
// for bit, in the tiling that LeastRounds finds. Against the best streaming
// kernel, us per step: 128^2 2.05 and 3.07 (32 rows, 4 steps), 500^2 3.0 and 3.9
// (48 rows, 3), 700 x 600 3.5 and 5.4 (64 rows, 3), 1024^2 6.1 and 7.2, 1200^2 7.2
// and 10.0, 2048^2 15.6 and 17.2 (32 rows, 2), 4096^2 65 and 78 (48 rows, 3).
static int auto_variant(int H, int W) {
  const int d = default_variant(H, W);
  if (d == kTile16) return d;  // narrow grids above 8 M cells: another rounding
  LeastRounds r((int64_t)H * W);
  r.offer(kBlock32x4, Block32x4{}, block_tiles<Block32x4>(H, W));
  r.offer(kBlock48x3, Block48x3{}, block_tiles<Block48x3>(H, W));
  r.offer(kBlock64x3, Block64x3{}, block_tiles<Block64x3>(H, W));
  r.offer(kBlock32x2, Block32x2{}, block_tiles<Block32x2>(H, W));
  return r.best;
}

// The variant whose kernel a grid takes in place of v. A launch holds fewer than
// 2^32 threads: 32 rows and 4 steps take 4 per cell (48 rows and 3 steps 0.6).
static int on_grid(int v, int H, int W) {
  if (v == kBlock32x4 && block_tiles<Block32x4>(H, W) * (Block32x4::waves * 64) > UINT32_MAX)
    return kBlock48x3;
  if (W % 2 && v == kPair2) return kStream2;
  if (W % 2 && v == kPair4) return kStream4;
  if (is_two_step(v) && !two_step_fits(v, H, W)) return kStream2;
  return v;
}

// The variant of a solve of several steps.
static int resolve_solve(int v, int H, int W) {
  if (v == kAuto) v = tuned_variant(H, W);
  return on_grid(v != kAuto ? v : auto_variant(H, W), H, W);
}

// The setting, else the tuned variant, else the streaming default.
static int resolve_for(int v, int H, int W) {
  if (v == kAuto) v = tuned_variant(H, W);
  return on_grid(v != kAuto ? v : default_variant(H, W), H, W);
}

// The one-step variant that runs a single step in place of v. Of the variants
// with several steps per launch that is the 2-row bands, the single step of an
// untuned shape too (1024^2 6.7 us a step and 9.2 with 8-row bands, 2048^2 24.0
// and 31.7).
static int step_variant(int v) {
  if (is_pc(v)) return pc_base(v);  // no coefficient precompute to amortise
  if (is_two_step(v) || is_block(v)) return kStream2;
  return v;
}

template <int R>
static void launch_stream(bool euler, const Coef& c, const float* D, const float* v,
                          const float* w, const float* u, int H, int W, const StimArgs& sa,
                          float dt, float inv_dx2, float* ov, float* ow, float* ou,
                          hipStream_t s) {
  const StreamGeom g = make_stream_geom<R>(H, W);
  const int blocks = g.blocks;
  if (euler)
    k_stream<R, true><<<blocks, 256, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                            ou, g);
  else
    k_stream<R, false><<<blocks, 256, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                             ou, g);
}

template <int R>
static void launch_stream2(bool euler, const Coef& c, const float* D, const float* v,
                           const float* w, const float* u, int H, int W, const StimArgs& sa,
                           float dt, float inv_dx2, float* ov, float* ow, float* ou,
                           hipStream_t s) {
  const StreamGeom2 g = make_stream_geom2<R>(H, W);
  if (euler)
    k_stream2<R, true><<<g.blocks, 256, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                               ou, g);
  else
    k_stream2<R, false><<<g.blocks, 256, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                                ou, g);
}

template <int R>
static void launch_stream_c(const Coef& c, const float4* cf, const float* v, const float* w,
                            const float* u, int H, int W, const StimArgs& sa, float dt,
                            float* ov, float* ow, float* ou, hipStream_t s) {
  const StreamGeom g = make_stream_geom<R>(H, W);
  k_stream_c<R><<<g.blocks, 256, 0, s>>>(c, cf, v, w, u, H, W, sa, dt, ov, ow, ou, g);
}

// Forward workspace: ping-pong state (3 fields), then, 256-byte aligned, the
// precomputed diffusion coefficients (one float4 per cell).
static size_t coef_offset(int H, int W) {
  return (3 * (size_t)H * W * sizeof(float) + 255) / 256 * 256;
}

template <int TH>
static void launch_tile(bool euler, const Coef& c, const float* D, const float* v,
                        const float* w, const float* u, int H, int W, const StimArgs& sa,
                        float dt, float inv_dx2, float* ov, float* ow, float* ou,
                        hipStream_t s) {
  const dim3 block(64, 4), grid((W + TW - 1) / TW, (H + TH - 1) / TH);
  if (euler)
    k_tile<TH, true><<<grid, block, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou);
  else
    k_tile<TH, false><<<grid, block, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                             ou);
}

static hipError_t launch_step(int variant, bool euler, const Coef& c, const float* D,
                              const float* v, const float* w, const float* u, int H, int W,
                              const StimArgs& sa, float dt, float inv_dx2, float* ov,
                              float* ow, float* ou, hipStream_t s) {
  switch (step_variant(on_grid(variant, H, W))) {
    case kPlain: {
      const dim3 block(64, 4), grid((W + 63) / 64, (H + 3) / 4);
      if (euler)
        k_plain<true><<<grid, block, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou);
      else
        k_plain<false><<<grid, block, 0, s>>>(c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow,
                                              ou);
      break;
    }
    case kTile16: launch_tile<16>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kTile32: launch_tile<32>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kStream32: launch_stream<32>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kStream16: launch_stream<16>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kStream4: launch_stream<4>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kStream2: launch_stream<2>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kPair2: launch_stream2<2>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kPair4: launch_stream2<4>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
    case kStream8:
    default: launch_stream<8>(euler, c, D, v, w, u, H, W, sa, dt, inv_dx2, ov, ow, ou, s); break;
  }
  return hipGetLastError();
}

// n_lev (at most Cfg::steps) levels on every tile. back: see BlockOrder.
template <class Cfg, bool HEUN>
static hipError_t launch_tiles(const Coef& c, const BlockIO& io, int H, int W,
                               const BlockStim& st, int n_lev, float dt, float inv_dx2, bool back,
                               hipStream_t s) {
  const BlockAxis ra = Cfg::row_axis(H), ca = Cfg::col_axis(W);
  k_block<Cfg, HEUN><<<(unsigned)(ra.n * ca.n), Cfg::waves * 64, 0, s>>>(
      c, io, H, W, st, n_lev, dt, inv_dx2, ra, ca, make_block_order(ra, ca, back));
  return hipGetLastError();
}

// n_lev steps (at most the variant's) of block variant v.
static hipError_t launch_block(int v, const Coef& c, const BlockIO& io, int H, int W,
                               const BlockStim& st, int n_lev, float dt, float inv_dx2, bool back,
                               hipStream_t s) {
  switch (v) {
    case kBlock32x2:
      return launch_tiles<Block32x2, false>(c, io, H, W, st, n_lev, dt, inv_dx2, back, s);
    case kBlock48x3:
      return launch_tiles<Block48x3, false>(c, io, H, W, st, n_lev, dt, inv_dx2, back, s);
    case kBlock64x3:
      return launch_tiles<Block64x3, false>(c, io, H, W, st, n_lev, dt, inv_dx2, back, s);
    default: return launch_tiles<Block32x4, false>(c, io, H, W, st, n_lev, dt, inv_dx2, back, s);
  }
}

// The stimuli of the n_lev steps from time t on.
static void block_stim(const StimSchedule& sched, double t, int n_lev, BlockStim& st) {
  for (int j = 0; j < kBlockMaxSteps; ++j)
    st.act[j] = j < n_lev ? sched.mask(t + (double)j) : 0u;
}

// Heun steps per launch (n <= 2) on block tiles, each two levels. The tiling is
// chosen as in auto_variant. Two launches per step of a streaming kernel, the
// slope k1 in memory between them, and this, us per step: 150 x 170 7.3 and 4.7
// (32 rows, 2 steps), 517 x 389 9.1 and 6.1 (48 rows, 2 steps), 760^2 14.1 and 9.8
// (64 rows, 1 step), 1000 x 760 18.1 and 11.6, 1200^2 30.1 and 18.9, 3000 x 2000 101
// and 57 (40 rows, 1 step).
typedef BlockCfg<2, 16, 4> Heun32x2;
typedef BlockCfg<3, 16, 4> Heun48x2;
typedef BlockCfg<4, 16, 2> Heun64x1;
typedef BlockCfg<5, 8, 2> Heun40x1;

enum HeunTiling { kHeun32x2, kHeun48x2, kHeun64x1, kHeun40x1 };

static int heun_tiling(int H, int W) {
  LeastRounds r((int64_t)H * W);
  r.offer(kHeun32x2, block_tiles<Heun32x2>(H, W), 2.0, 2.9);
  r.offer(kHeun48x2, block_tiles<Heun48x2>(H, W), 1.8, 4.2);
  r.offer(kHeun64x1, block_tiles<Heun64x1>(H, W), 2.2, 7.45);
  r.offer(kHeun40x1, block_tiles<Heun40x1>(H, W), 4.3, 3.55);
  return r.best;
}

static int heun_steps(int tiling) { return tiling == kHeun32x2 || tiling == kHeun48x2 ? 2 : 1; }

static hipError_t launch_heun(int tiling, const Coef& c, const BlockIO& io, int H, int W,
                              const BlockStim& st, int n, float dt, float inv_dx2, bool back,
                              hipStream_t s) {
  const int l = 2 * n;
  switch (tiling) {
    case kHeun32x2: return launch_tiles<Heun32x2, true>(c, io, H, W, st, l, dt, inv_dx2, back, s);
    case kHeun48x2: return launch_tiles<Heun48x2, true>(c, io, H, W, st, l, dt, inv_dx2, back, s);
    case kHeun64x1: return launch_tiles<Heun64x1, true>(c, io, H, W, st, l, dt, inv_dx2, back, s);
    default: return launch_tiles<Heun40x1, true>(c, io, H, W, st, l, dt, inv_dx2, back, s);
  }
}

// Heun steps at times t .. t_end-1 (cardiax/solve.py:103-111) from `in` to
// `out`; the workspace holds a ping-pong state.
static int32_t heun_loop(const fk_params* params, const float* D, const float* const in[3],
                         int32_t H, int32_t W, const fk_stimulus* stimuli, int32_t n_stimuli,
                         double t, int64_t steps, float dt, float dx, float* const out[3],
                         void* work, hipStream_t s) {
  const size_t n = (size_t)H * W;
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  float* wk = (float*)work;
  float* ping[3] = {wk, wk + n, wk + 2 * n};
  float* const* bufs[2] = {out, ping};
  const int tiling = heun_tiling(H, W), per = heun_steps(tiling);
  const int64_t launches = (steps + per - 1) / per;
  int dst = (launches % 2 == 1) ? 0 : 1;  // the last launch lands in `out`
  const float* src[3] = {in[0], in[1], in[2]};
  const StimSchedule sched(stimuli, n_stimuli);
  BlockStim st{};
  for (int i = 0; i < n_stimuli; ++i) st.f[i] = stimuli[i].field;
  for (int64_t k = 0; k < steps; k += per) {
    const int m = (int)std::min<int64_t>(per, steps - k);
    for (int l = 0; l < 2 * m; ++l)  // both stages of step k + j at time t + k + j
      st.act[l] = sched.mask(t + (double)(k + l / 2));
    float* const* d = bufs[dst];
    const BlockIO io{D, src[0], src[1], src[2], d[0], d[1], d[2], 0, false};
    HIP_CHECK(launch_heun(tiling, c, io, H, W, st, m, dt, inv_dx2, dst == 1, s));
    src[0] = d[0];
    src[1] = d[1];
    src[2] = d[2];
    dst ^= 1;
  }
  return FK_OK;
}

int32_t forward_loop(int variant, const fk_params* params, const float* D, const float* v_in,
                     const float* w_in, const float* u_in, int32_t H, int32_t W,
                     const fk_stimulus* stimuli, int32_t n_stimuli, double t, double t_end,
                     float dt, float dx, float* v_out, float* w_out, float* u_out, void* work,
                     size_t work_bytes, void* stream, bool state_only) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v_in, w_in, u_in, v_out, w_out, u_out}) || !check_time(t, t_end) ||
      !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  const size_t n = (size_t)H * W;
  const int64_t steps = loop_count(t, t_end);
  const size_t need = state_only ? 3 * n * sizeof(float) : fk_forward_workspace_bytes(H, W);
  if (steps >= 2 && (work == nullptr || work_bytes < need))
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu", need,
                     work_bytes);
  hipStream_t s = (hipStream_t)stream;
  if (steps == 0) {
    for (auto pr : {std::make_pair(v_in, v_out), std::make_pair(w_in, w_out),
                    std::make_pair(u_in, u_out)})
      HIP_CHECK(hipMemcpyAsync(pr.second, pr.first, n * sizeof(float),
                               hipMemcpyDeviceToDevice, s));
    return FK_OK;
  }
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  float* wk = (float*)work;
  float* bufs[2][3] = {{v_out, w_out, u_out}, {wk, wk + n, wk + 2 * n}};
  int v = steps < 2 ? resolve_for(variant, H, W) : resolve_solve(variant, H, W);
  // nothing to amortise, or no room for the coefficients
  if (is_pc(v) && (steps < 2 || state_only)) v = pc_base(v);
  float4* cf = nullptr;
  if (is_pc(v)) {
    cf = (float4*)((char*)work + coef_offset(H, W));
    const dim3 grid((W + 63) / 64, (H + 3) / 4);
    k_stream_coef<<<grid, 256, 0, s>>>(D, H, W, (float)(inv_dx2 / 144.0), cf);
    HIP_CHECK(hipGetLastError());
  }
  const int depth = is_block(v) ? block_steps(v) : is_two_step(v) ? 2 : 1;
  const int64_t launches = (steps + depth - 1) / depth;
  // Ping-pong so that the last launch lands in the output buffers.
  int dst = (launches % 2 == 1) ? 0 : 1;
  const float* src[3] = {v_in, w_in, u_in};
  StimSchedule sched(stimuli, n_stimuli);
  BlockStim st{};
  for (int i = 0; i < n_stimuli; ++i) st.f[i] = stimuli[i].field;
  for (int64_t k = 0, ns = depth; k < steps; k += ns) {
    float** d = bufs[dst];
    if (is_two_step(v)) {
      const StimArgs s1 = sched.at(t + (double)k);  // copies: at() reuses its storage
      if (steps - k >= 2) {
        const StimArgs s2 = sched.at(t + (double)(k + 1));
        HIP_CHECK(launch_two_step(v, c, D, src[0], src[1], src[2], H, W, s1, s2, dt, inv_dx2,
                                  d[0], d[1], d[2], s));
      } else {  // an odd last step
        HIP_CHECK(launch_step(kStream2, true, c, D, src[0], src[1], src[2], H, W, s1, dt,
                              inv_dx2, d[0], d[1], d[2], s));
      }
    } else if (is_block(v) && steps - k > 1) {
      int bv = v;
      ns = block_launch(&bv, steps - k, LeastRounds((int64_t)n).streams);
      block_stim(sched, t + (double)k, (int)ns, st);
      const BlockIO io{D, src[0], src[1], src[2], d[0], d[1], d[2], 0, false};
      HIP_CHECK(launch_block(bv, c, io, H, W, st, (int)ns, dt, inv_dx2, dst == 1, s));
    } else if (is_block(v)) {  // a single last step
      HIP_CHECK(launch_step(kStream2, true, c, D, src[0], src[1], src[2], H, W,
                            sched.at(t + (double)k), dt, inv_dx2, d[0], d[1], d[2], s));
    } else if (is_pc(v)) {
      const StimArgs& sa = sched.at(t + (double)k);
      if (v == kStreamC8)
        launch_stream_c<8>(c, cf, src[0], src[1], src[2], H, W, sa, dt, d[0], d[1], d[2], s);
      else if (v == kStreamC4)
        launch_stream_c<4>(c, cf, src[0], src[1], src[2], H, W, sa, dt, d[0], d[1], d[2], s);
      else if (v == kStreamC2)
        launch_stream_c<2>(c, cf, src[0], src[1], src[2], H, W, sa, dt, d[0], d[1], d[2], s);
      else
        launch_stream_c<16>(c, cf, src[0], src[1], src[2], H, W, sa, dt, d[0], d[1], d[2], s);
      HIP_CHECK(hipGetLastError());
    } else {
      const StimArgs& sa = sched.at(t + (double)k);
      HIP_CHECK(launch_step(v, true, c, D, src[0], src[1], src[2], H, W, sa, dt, inv_dx2,
                            d[0], d[1], d[2], s));
    }
    src[0] = d[0];
    src[1] = d[1];
    src[2] = d[2];
    dst ^= 1;
  }
  return FK_OK;
}

// Times every variant but the plain one over n_steps Euler steps from
// (v, w, u) at time t with the given problem (HIP events on `s`, which is
// synchronised): a warm-up of 8 steps, then the timed run, results into
// y (3 H W floats); the inputs are not modified. The three fastest are
// timed three more times, interleaved, and keep their minimum.
// times_ms[variant] receives each time (-1 for the untimed), *best the
// fastest.
static int32_t time_candidates(const fk_params* p, const float* D, const float* v,
                               const float* w, const float* u, int H, int W,
                               const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                               int32_t n_steps, float dt, float dx, float* y, void* wk,
                               size_t wb, hipStream_t s, float* times_ms, int32_t* best) {
  const size_t n = (size_t)H * W;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  int best_v = default_variant(H, W);
  float best_ms = 0.0f;
  const int cand[] = {kStream8,  kStream4,  kStream2,   kStream16,  kStream32,  kStreamC8,
                      kStreamC4, kStreamC2, kStreamC16, kPair2,     kPair4,     kTile16,
                      kTile32,   kBlock32x2, kBlock48x3, kBlock64x3, kBlock32x4, kStreamT8,
                      kStreamT12, kStreamT16, kStreamT24};
  int32_t rc = FK_OK;
  // one warm-up launch of 8 steps, then n_steps timed with events on `s`
  auto time_one = [&](int var, float* ms) {
    rc = forward_loop(var, p, D, v, w, u, H, W, stimuli, n_stimuli, t, t + 8.0, dt, dx, y,
                      y + n, y + 2 * n, wk, wb, s, false);
    if (rc == FK_OK) e = hipEventRecord(e0, s);
    if (rc == FK_OK && e == hipSuccess)
      rc = forward_loop(var, p, D, v, w, u, H, W, stimuli, n_stimuli, t, t + (double)n_steps,
                        dt, dx, y, y + n, y + 2 * n, wk, wb, s, false);
    if (rc == FK_OK && e == hipSuccess) e = hipEventRecord(e1, s);
    if (rc == FK_OK && e == hipSuccess) e = hipEventSynchronize(e1);
    *ms = 0.0f;
    if (rc == FK_OK && e == hipSuccess) e = hipEventElapsedTime(ms, e0, e1);
    return rc == FK_OK && e == hipSuccess;
  };
  float t_all[kNumVariants];
  for (int k = 0; k < kNumVariants; ++k) t_all[k] = -1.0f;
  for (int var : cand) {
    if (e != hipSuccess) break;
    float ms;
    if (!time_one(var, &ms)) break;
    t_all[var] = ms;
  }
  // The three fastest again, three interleaved rounds, the minimum of each:
  // a transient slowdown during one candidate's single run cannot decide.
  int top[3] = {-1, -1, -1};
  if (rc == FK_OK && e == hipSuccess) {
    for (int var : cand) {
      if (t_all[var] < 0.0f) continue;
      for (int k = 0; k < 3; ++k) {
        if (top[k] < 0 || t_all[var] < t_all[top[k]]) {
          for (int m = 2; m > k; --m) top[m] = top[m - 1];
          top[k] = var;
          break;
        }
      }
    }
    for (int round = 0; round < 3 && rc == FK_OK && e == hipSuccess; ++round)
      for (int k = 0; k < 3; ++k) {
        if (top[k] < 0) continue;
        float ms;
        if (!time_one(top[k], &ms)) break;
        t_all[top[k]] = std::min(t_all[top[k]], ms);
      }
    for (int k = 0; k < 3; ++k)
      if (top[k] >= 0 && (best_ms == 0.0f || t_all[top[k]] < best_ms)) {
        best_ms = t_all[top[k]];
        best_v = top[k];
      }
  }
  if (times_ms)
    for (int k = 0; k < kNumVariants; ++k) times_ms[k] = t_all[k];
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (rc != FK_OK) return rc;
  if (e != hipSuccess) return set_error(FK_ERR_HIP, "autotune failed: %s", hipGetErrorString(e));
  *best = best_v;
  return FK_OK;
}

}  // namespace fk

using namespace fk;

extern "C" {

int32_t fk_abi_version(void) { return 4; }

int32_t fk_set_forward_variant(int32_t variant) {
  ErrorScope es;
  if (variant < 0 || variant >= kNumVariants)
    return set_error(FK_ERR_ARG, "unknown forward variant %d", variant);
  return g_variant.exchange(variant);
}

int32_t fk_init(float* v, float* w, float* u, int64_t n_cells, void* stream) {
  ErrorScope es;
  if (!check_ptrs({v, w, u}) || n_cells < 0)
    return set_error(FK_ERR_ARG, "fk_init: null pointer or negative size");
  if (n_cells == 0) return FK_OK;
  const int blocks = (int)std::min<int64_t>((n_cells + 255) / 256, 4096);
  k_init<<<blocks, 256, 0, (hipStream_t)stream>>>(v, w, u, n_cells);
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

int32_t fk_check_finite(const float* const* fields, int32_t n_fields, int64_t n_cells,
                        void* work, void* stream) {
  ErrorScope es;
  if (!fields || !work || n_fields < 1 || n_cells < 0)
    return set_error(FK_ERR_ARG, "fk_check_finite: null pointer or bad count");
  for (int32_t k = 0; k < n_fields; ++k)
    if (!fields[k]) return set_error(FK_ERR_ARG, "fk_check_finite: field %d is null", k);
  hipStream_t s = (hipStream_t)stream;
  unsigned* flag = (unsigned*)work;
  k_clear_flag<<<1, 64, 0, s>>>(flag);
  const int blocks = (int)std::max<int64_t>(1, std::min<int64_t>((n_cells + 255) / 256, 2048));
  for (int32_t k = 0; k < n_fields; ++k)
    k_nonfinite<<<blocks, 256, 0, s>>>(fields[k], n_cells, flag);
  HIP_CHECK(hipGetLastError());
  unsigned host = 0;
  HIP_CHECK(hipMemcpyAsync(&host, flag, sizeof(host), hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  if (host) return set_error(FK_ERR_NONFINITE, "non-finite values (NaN or inf) in the fields");
  return FK_OK;
}

int32_t fk_step(const fk_params* params, const float* D, const float* v, const float* w,
                const float* u, int32_t H, int32_t W, const fk_stimulus* stimuli,
                int32_t n_stimuli, double t, float dx, float* dv, float* dw, float* du,
                void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v, w, u, dv, dw, du}) || !check_time(t, t) || !check_dx(dx))
    return last_code();
  StimSchedule sched(stimuli, n_stimuli);
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  HIP_CHECK(launch_step(resolve_for(g_variant.load(), H, W), false, c, D, v, w, u, H, W,
                        sched.at(t), 0.0f, inv_dx2, dv, dw, du, (hipStream_t)stream));
  return FK_OK;
}

int32_t fk_step_euler(const fk_params* params, const float* D, const float* v,
                      const float* w, const float* u, int32_t H, int32_t W,
                      const fk_stimulus* stimuli, int32_t n_stimuli, double t, float dt,
                      float dx, float* v_out, float* w_out, float* u_out, void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v, w, u, v_out, w_out, u_out}) || !check_time(t, t) ||
      !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  StimSchedule sched(stimuli, n_stimuli);
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  HIP_CHECK(launch_step(resolve_for(g_variant.load(), H, W), true, c, D, v, w, u, H, W,
                        sched.at(t), dt, inv_dx2, v_out, w_out, u_out, (hipStream_t)stream));
  return FK_OK;
}

size_t fk_forward_workspace_bytes(int32_t H, int32_t W) {
  if (H <= 0 || W <= 0) return 0;
  return coef_offset(H, W) + (size_t)H * (size_t)W * sizeof(float4);
}

int32_t fk_forward_euler(const fk_params* params, const float* D, const float* v_in,
                         const float* w_in, const float* u_in, int32_t H, int32_t W,
                         const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                         double t_end, float dt, float dx, float* v_out, float* w_out,
                         float* u_out, void* work, size_t work_bytes, void* stream) {
  return forward_loop(g_variant.load(), params, D, v_in, w_in, u_in, H, W, stimuli, n_stimuli, t,
                      t_end, dt, dx, v_out, w_out, u_out, work, work_bytes, stream, false);
}

int32_t fk_autotune_forward(int32_t H, int32_t W, int32_t n_steps, void* stream,
                            float* times_ms, int32_t* best) {
  ErrorScope es;
  if (!check_grid(H, W)) return last_code();
  if (n_steps < 1 || n_steps > 100000)
    return set_error(FK_ERR_ARG, "n_steps must be in [1, 100000], got %d", n_steps);
  hipStream_t s = (hipStream_t)stream;
  const size_t n = (size_t)H * W;
  const size_t wb = fk_forward_workspace_bytes(H, W);
  float* mem = nullptr;
  HIP_CHECK(hipMalloc((void**)&mem, 8 * n * sizeof(float) + 256 + wb));
  float *D = mem, *x = mem + n, *y = mem + 4 * n, *f = mem + 7 * n;
  float* wk = (float*)(((uintptr_t)(mem + 8 * n) + 255) / 256 * 256);
  const int blocks = (int)std::min<size_t>((n + 255) / 256, 4096);
  k_fill<<<blocks, 256, 0, s>>>(D, n, 1e-3f);
  k_init<<<blocks, 256, 0, s>>>(y, y + n, y + 2 * n, (int64_t)n);
  // PARAMSET_3 (cardiax/params.py:60-62)
  const fk_params p{3.33f, 19.6f, 1250.0f, 870.0f, 41.0f, 0.25f, 12.5f,
                    33.33f, 29.0f, 10.0f, 0.85f, 0.13f, 0.04f, 1.0f};
  // The gates compile to branches in some kernels, so a step costs more where
  // waves hold excited or mixed cells than at rest. The candidates are timed
  // from the state 200 steps after an S1 pulse over the left 40% of the
  // columns: that part excited, the rest at rest, a wavefront between them.
  // No stimulus is active while timing, as for all but a few steps of a real
  // solve. fk_autotune_forward_state times on the caller's own problem.
  k_fill_cols<<<blocks, 256, 0, s>>>(f, H, W, (W * 2) / 5, 20.0f);
  HIP_CHECK(hipGetLastError());
  int32_t rc;
  {
    const fk_stimulus s1{0.0, 2.0, 1e9, f};
    rc = forward_loop(kStream2, &p, D, y, y + n, y + 2 * n, H, W, &s1, 1, 0.0, 200.0, 0.01f,
                      0.01f, x, x + n, x + 2 * n, wk, wb, s, false);
  }
  int32_t best_v = 0;
  if (rc == FK_OK)
    rc = time_candidates(&p, D, x, x + n, x + 2 * n, H, W, nullptr, 0, 0.0, n_steps, 0.01f,
                         0.01f, y, wk, wb, s, times_ms, &best_v);
  const hipError_t ef = hipFree(mem);
  if (rc != FK_OK) return rc;
  if (ef != hipSuccess) return set_error(FK_ERR_HIP, "autotune failed: %s", hipGetErrorString(ef));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[{H, W}] = best_v;
  }
  if (best) *best = best_v;
  return FK_OK;
}

int32_t fk_autotune_forward_state(const fk_params* params, const float* D, const float* v,
                                  const float* w, const float* u, int32_t H, int32_t W,
                                  const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                                  int32_t n_steps, float dt, float dx, void* stream,
                                  float* times_ms, int32_t* best) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v, w, u}) || !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  if (n_steps < 1 || n_steps > 100000)
    return set_error(FK_ERR_ARG, "n_steps must be in [1, 100000], got %d", n_steps);
  if (!check_time(t, t + (double)n_steps)) return last_code();
  hipStream_t s = (hipStream_t)stream;
  const size_t n = (size_t)H * W;
  const size_t wb = fk_forward_workspace_bytes(H, W);
  float* mem = nullptr;
  HIP_CHECK(hipMalloc((void**)&mem, 3 * n * sizeof(float) + 256 + wb));
  float* wk = (float*)(((uintptr_t)(mem + 3 * n) + 255) / 256 * 256);
  int32_t best_v = 0;
  const int32_t rc = time_candidates(params, D, v, w, u, H, W, stimuli, n_stimuli, t, n_steps,
                                     dt, dx, mem, wk, wb, s, times_ms, &best_v);
  const hipError_t ef = hipFree(mem);
  if (rc != FK_OK) return rc;
  if (ef != hipSuccess) return set_error(FK_ERR_HIP, "autotune failed: %s", hipGetErrorString(ef));
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[{H, W}] = best_v;
  }
  if (best) *best = best_v;
  return FK_OK;
}

int32_t fk_autotune_lookup(int32_t H, int32_t W) { return tuned_variant(H, W); }

void fk_autotune_reset(void) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tuned.clear();
}

int32_t fk_forward_variant_for(int32_t H, int32_t W) {
  ErrorScope es;
  if (H < 3 || W < 3) return set_error(FK_ERR_ARG, "grid %d x %d: H, W must be >= 3", H, W);
  return resolve_for(g_variant.load(), H, W);
}

int32_t fk_solve_variant_for(int32_t H, int32_t W) {
  ErrorScope es;
  if (!check_grid(H, W)) return last_code();
  return resolve_solve(g_variant.load(), H, W);
}

int32_t fk_step_variant_for(int32_t H, int32_t W) {
  ErrorScope es;
  if (!check_grid(H, W)) return last_code();
  return step_variant(resolve_for(g_variant.load(), H, W));
}

int32_t fk_forward_trajectory(const fk_params* params, const float* D, const float* v0,
                              const float* w0, const float* u0, int32_t H, int32_t W,
                              const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                              int32_t n_steps, float dt, float dx, float* states,
                              void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v0, w0, u0}) || !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  if (n_steps < 0) return set_error(FK_ERR_ARG, "n_steps must be >= 0, got %d", n_steps);
  if (n_steps == 0) return FK_OK;
  if (states == nullptr) return set_error(FK_ERR_ARG, "null states pointer");
  if (!check_time(t, t + (double)n_steps)) return last_code();
  const size_t n = (size_t)H * W;
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  StimSchedule sched(stimuli, n_stimuli);
  const int v = resolve_solve(g_variant.load(), H, W);  // two-step variants: stream2
  const float* src[3] = {v0, w0, u0};
  BlockStim st{};
  for (int i = 0; i < n_stimuli; ++i) st.f[i] = stimuli[i].field;
  for (int32_t k = 0; k < n_steps;) {
    float* d = states + (size_t)k * 3 * n;
    if (is_block(v) && n_steps - k > 1) {  // every level of a block is a state
      const int ns = std::min(block_steps(v), n_steps - k);
      block_stim(sched, t + (double)k, ns, st);
      const BlockIO io{D, src[0], src[1], src[2], d, d + n, d + 2 * n, 3 * n, true};
      HIP_CHECK(launch_block(v, c, io, H, W, st, ns, dt, inv_dx2, false, (hipStream_t)stream));
      d += (size_t)(ns - 1) * 3 * n;
      src[0] = d;
      src[1] = d + n;
      src[2] = d + 2 * n;
      k += ns;
      continue;
    }
    HIP_CHECK(launch_step(v, true, c, D, src[0], src[1], src[2], H, W, sched.at(t + (double)k),
                          dt, inv_dx2, d, d + n, d + 2 * n, (hipStream_t)stream));
    src[0] = d;
    src[1] = d + n;
    src[2] = d + 2 * n;
    ++k;
  }
  return FK_OK;
}

int32_t fk_forward_euler_plain(const fk_params* params, const float* D, const float* v_in,
                               const float* w_in, const float* u_in, int32_t H, int32_t W,
                               const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                               double t_end, float dt, float dx, float* v_out,
                               float* w_out, float* u_out, void* work, size_t work_bytes,
                               void* stream) {
  return forward_loop(kPlain, params, D, v_in, w_in, u_in, H, W, stimuli, n_stimuli,
                      t, t_end, dt, dx, v_out, w_out, u_out, work, work_bytes, stream, false);
}

size_t fk_heun_workspace_bytes(int32_t H, int32_t W) {
  if (H <= 0 || W <= 0) return 0;
  return 6 * (size_t)H * (size_t)W * sizeof(float);
}

int32_t fk_step_heun(const fk_params* params, const float* D, const float* v, const float* w,
                     const float* u, int32_t H, int32_t W, const fk_stimulus* stimuli,
                     int32_t n_stimuli, double t, float dt, float dx, float* v_out,
                     float* w_out, float* u_out, void* work, size_t work_bytes, void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v, w, u, v_out, w_out, u_out, work}) || !check_time(t, t) ||
      !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  if (work_bytes < fk_heun_workspace_bytes(H, W))
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu",
                     fk_heun_workspace_bytes(H, W), work_bytes);
  const float* in[3] = {v, w, u};
  float* out[3] = {v_out, w_out, u_out};
  return heun_loop(params, D, in, H, W, stimuli, n_stimuli, t, 1, dt, dx, out, work,
                   (hipStream_t)stream);
}

int32_t fk_forward_heun(const fk_params* params, const float* D, const float* v_in,
                        const float* w_in, const float* u_in, int32_t H, int32_t W,
                        const fk_stimulus* stimuli, int32_t n_stimuli, double t, double t_end,
                        float dt, float dx, float* v_out, float* w_out, float* u_out,
                        void* work, size_t work_bytes, void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v_in, w_in, u_in, v_out, w_out, u_out}) || !check_time(t, t_end) ||
      !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  const int64_t steps = loop_count(t, t_end);
  hipStream_t s = (hipStream_t)stream;
  const size_t n = (size_t)H * W;
  if (steps == 0) {
    for (auto pr : {std::make_pair(v_in, v_out), std::make_pair(w_in, w_out),
                    std::make_pair(u_in, u_out)})
      HIP_CHECK(hipMemcpyAsync(pr.second, pr.first, n * sizeof(float),
                               hipMemcpyDeviceToDevice, s));
    return FK_OK;
  }
  if (work == nullptr || work_bytes < fk_heun_workspace_bytes(H, W))
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu",
                     fk_heun_workspace_bytes(H, W), work_bytes);
  const float* in[3] = {v_in, w_in, u_in};
  float* out[3] = {v_out, w_out, u_out};
  return heun_loop(params, D, in, H, W, stimuli, n_stimuli, t, steps, dt, dx, out, work, s);
}

int32_t fk_gradient(const float* a, float* out, int32_t rows, int32_t cols, int32_t axis,
                    void* stream) {
  ErrorScope es;
  if (!check_ptrs({a, out})) return FK_ERR_ARG;
  if (axis != 0 && axis != 1) return set_error(FK_ERR_ARG, "axis must be 0 or 1, got %d", axis);
  if (rows <= 0 || cols <= 0) return set_error(FK_ERR_ARG, "empty array %dx%d", rows, cols);
  const int n = axis == 0 ? rows : cols;
  if (n < 5)
    return set_error(FK_ERR_ARG, "gradient needs >= 5 entries along axis %d, got %d", axis, n);
  const dim3 block(64, 4), grid((cols + 63) / 64, (rows + 3) / 4);
  k_gradient<<<grid, block, 0, (hipStream_t)stream>>>(a, out, rows, cols, axis);
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

int32_t fk_stimulate(double t, const float* X, float* out, int64_t n_cells,
                     const fk_stimulus* stimuli, int32_t n_stimuli, void* stream) {
  ErrorScope es;
  if (n_cells < 0) return set_error(FK_ERR_ARG, "fk_stimulate: negative size");
  if (!check_ptrs({X, out}) || !check_stimuli(stimuli, n_stimuli) || !check_time(t, t))
    return last_code();
  if (n_cells == 0) return FK_OK;
  StimSchedule sched(stimuli, n_stimuli);
  const int blocks = (int)std::min<int64_t>((n_cells + 255) / 256, 4096);
  k_stimulate<<<blocks, 256, 0, (hipStream_t)stream>>>(X, out, n_cells, sched.at(t));
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

}  // extern "C"
