// Adjoint (reverse mode) of one forward-Euler step, for gradients of a loss
// with respect to the diffusivity map D and the time constants tau_d, tau_r,
// tau_si.
//
// Forward step (cardiax/solve.py:26-70): x' = x + dt f(x), f = (f_v, f_w, f_u),
//   f_u = [D (A2x u + A2y u) + (A1x D)(A1x u) + (A1y D)(A1y u)] / dx^2 + J,
// where A1 = crop(G(pad(.))) and A2 = crop(G(G(pad(.)))) are the effective
// per-axis operators of the reference's `gradient` with edge padding, and J is
// j_ion, replaced by the stimulus where one is active. Reverse step, with the
// Heaviside gates p = [u >= V_c], q = [u >= V_v] held as fixed masks and the
// stimulus selection routing no cotangent to j_ion (the semantics jax.grad
// gives greater_equal and where):
//   lam_v' = lam_v + dt (df_v/dv lam_v + dJ/dv lam_u*)
//   lam_w' = lam_w + dt (df_w/dw lam_w + dJ/dw lam_u*)
//   lam_u' = lam_u + dt (dJ/du lam_u* + [A2x^T(D lam_u) + A2y^T(D lam_u)
//                        + A1x^T(D_x lam_u) + A1y^T(D_y lam_u)] / dx^2)
//   gD    += dt [lam_u (A2x u + A2y u) + A1x^T(lam_u A1x u) + A1y^T(lam_u A1y u)] / dx^2
//   g_tau += dt sum(dJ/dtau lam_u*)            (tau_d, tau_r, tau_si)
// with lam_u* = lam_u outside active stimulus cells and 0 inside.
//
// The operators' rows away from the edges are the central stencils; those near
// an edge are tabulated per call by k_adj_tables, which composes the
// reference's gradient rules exactly (any N >= 3). One launch reverses one step
// (adj_tile).
#include <hip/hip_runtime.h>

#include "cardiax_amd.h"
#include "fk_adjoint.h"
#include "fk_device.h"
#include "fk_host.h"

namespace fk {

// Band rows of a reverse step on one grid: a small grid's step takes as long as
// its slowest wave (256^2: 7.0 us with 2 rows, 8.9 with 4, 13.9 with 8); the
// halo rows of short bands cost less (1120^2: 24.7, 23.9 and 29.8).
constexpr int kRevRows = 2;

// The table rows of both axes, one d = -5 .. 5 per thread.
__global__ void k_adj_tables(int H, int W, AdjAxisTab* tab) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  constexpr int per_axis = kAdjSlots * 12;
  if (t >= 2 * per_axis) return;
  const int axis = t / per_axis, slot = t % per_axis / 12, d = t % 12 - kA2;
  const int N = axis == 0 ? H : W;
  const int i = N <= kAdjSlots || slot < kAdjT ? slot : slot + (N - kAdjSlots);
  float a1, a2, t1, t2;  // 0 for d = 6 and for cells off a short axis
  adj_coef(i, d <= kA2 ? i + d : -1, N, a1, a2);
  adj_coef(d <= kA2 ? i - d : -1, i, N, t1, t2);
  AdjRow& r = tab[axis].r[slot];
  r.a2[d + kA2] = a2;
  r.t2[d + kA2] = t2;
  if (d >= -kA1 && d <= kA1 + 1) {
    r.a1[d + kA1] = d <= kA1 ? a1 : 0.0f;
    r.t1[d + kA1] = d <= kA1 ? t1 : 0.0f;
  }
}

// One reverse step: a wave per (strip, band of R rows), four per block.
// A die takes a run of whole bands across the strips (see k_adj_rev_row); forward
// and backward over 100 steps, strips first in plain order and so: 600^2 1.75 and
// 1.64 ms, 1000^2 3.16 and 2.86.
template <int R>
__global__ void __launch_bounds__(256)
k_adj_rev(Coef c, AdjArgs a, int H, int W, StimArgs sa, float dt, float inv_dx2, int n_strips,
          int n_tiles) {
  __shared__ AdjAxisTab tab[4][2];
  const int x = blockIdx.x % kXcds, q = gridDim.x / kXcds, r = gridDim.x % kXcds;
  const int blk = x * q + min(x, r) + blockIdx.x / kXcds;
  const int tile = __builtin_amdgcn_readfirstlane(blk * 4 + (int)(threadIdx.x >> 6));
  if (tile >= n_tiles) return;  // whole wave leaves; the kernel has no barrier
  const int band = tile / n_strips, strip = tile - band * n_strips;
  const int rs = R * band, cs = kRevOut * strip;
  const AdjStimList sv{sa};
  adj_tile_any<R>(c, a, H, W, sv, dt, inv_dx2, rs, cs,
                  (adj_edge_band(rs, R, H) ? 1 : 0) | (adj_edge_strip(cs, W) ? 2 : 0),
                  tab[threadIdx.x >> 6]);
}

// The same with a wave per row, a pair of rows per block. A die takes a run of
// whole bands across the strips, so that neighbours' windows come from its L2 and
// the edge strips spread over all dies; forward and backward over 200 steps
// (with the rows of a pair still adding their tau terms together), strips first
// in plain order and so: 256^2 1.88 and 1.76 ms, 350^2 2.33 and 2.16,
// 400^2 2.32 and 2.30 (runs along a strip: 1.82, 2.19 and 2.46).
__global__ void __launch_bounds__(128)
k_adj_rev_row(Coef c, AdjArgs a, int H, int W, StimArgs sa, float dt, float inv_dx2,
              int n_strips) {
  __shared__ AdjAxisTab tab[2][2];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int x = blockIdx.x % kXcds, q = gridDim.x / kXcds, r = gridDim.x % kXcds;
  const int t = x * q + min(x, r) + blockIdx.x / kXcds;  // a die's pairs are neighbours
  const int band = t / n_strips;
  const int rs = 2 * band + wave, cs = kRevOut * (t - band * n_strips);
  if (rs >= H) return;  // an odd last row; the kernel has no barrier
  const AdjStimList sv{sa};
  adj_tile_any<1>(c, a, H, W, sv, dt, inv_dx2, rs, cs,
                  (adj_edge_band(rs, 1, H) ? 1 : 0) | (adj_edge_strip(cs, W) ? 2 : 0),
                  tab[wave]);
}

__global__ void k_adj_zero(float* a, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    a[i] = 0.0f;
}


// Sums of the three tau accumulators (n triples of doubles): each
// block reduces a grid-stride slice into part[block][0..2] (k_adj_reduce),
// then one block adds the block sums (k_adj_reduce_final). Fixed order:
// deterministic.
__global__ void __launch_bounds__(256)
k_adj_reduce(const double* __restrict__ acc, size_t n, double* __restrict__ part) {
  __shared__ double s[3][256];
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x; b < n;
       b += (size_t)gridDim.x * blockDim.x) {
    a0 += acc[3 * b];
    a1 += acc[3 * b + 1];
    a2 += acc[3 * b + 2];
  }
  s[0][threadIdx.x] = a0;
  s[1][threadIdx.x] = a1;
  s[2][threadIdx.x] = a2;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o)
      for (int k = 0; k < 3; ++k) s[k][threadIdx.x] += s[k][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 3; ++k) part[3 * (size_t)blockIdx.x + k] = s[k][0];
}

__global__ void __launch_bounds__(256)
k_adj_reduce_final(const double* __restrict__ part, int n_part, float* g_tau) {
  __shared__ double s[3][256];
  for (int k = 0; k < 3; ++k) {
    double a = 0.0;
    for (int b = threadIdx.x; b < n_part; b += blockDim.x) a += part[3 * b + k];
    s[k][threadIdx.x] = a;
  }
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o)
      for (int k = 0; k < 3; ++k) s[k][threadIdx.x] += s[k][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    for (int k = 0; k < 3; ++k) g_tau[k] = (float)s[k][0];
}

// Reverse step: cotangents lam_in (v, w, u; inj, if not null, adds to u) ->
// lam_out.
static hipError_t launch_rev(const AdjLayout& L, char* wk, const Coef& c, const float* D,
                             const float* v, const float* w, const float* u, int H, int W,
                             const StimArgs& sa, float dt, float inv_dx2,
                             const float* const lam_in[3], const float* inj,
                             float* const lam_out[3], float* gD, hipStream_t s) {
  const AdjArgs a{v, w, u, D, lam_in[0], lam_in[1], lam_in[2], inj, lam_out[0], lam_out[1],
                  lam_out[2], gD, (double*)(wk + L.part), (const AdjAxisTab*)(wk + L.tab)};
  const int strips = adj_strips(W), bands = (H + kRevRows - 1) / kRevRows;
  const int tiles = strips * bands;
  if (tiles <= kRevRowTiles) {
    const int pairs = (H + 1) / 2;
    k_adj_rev_row<<<strips * pairs, 128, 0, s>>>(c, a, H, W, sa, dt, inv_dx2, strips);
    return hipGetLastError();
  }
  k_adj_rev<kRevRows><<<(tiles + 3) / 4, 256, 0, s>>>(c, a, H, W, sa, dt, inv_dx2, strips, tiles);
  return hipGetLastError();
}

}  // namespace fk

using namespace fk;

extern "C" {

size_t fk_adjoint_workspace_bytes(int32_t H, int32_t W) {
  if (H <= 0 || W <= 0) return 0;
  return adj_layout(H, W).total;
}

int32_t fk_adjoint_prepare(const float* D, int32_t H, int32_t W, void* work, size_t work_bytes,
                           void* stream) {
  ErrorScope es;
  if (!check_grid(H, W) || !check_ptrs({D, work})) return last_code();
  const AdjLayout L = adj_layout(H, W);
  if (work_bytes < L.total)
    return set_error(FK_ERR_ARG, "adjoint workspace too small: need %zu bytes, got %zu",
                     L.total, work_bytes);
  hipStream_t s = (hipStream_t)stream;
  char* wk = (char*)work;
  AdjAxisTab* tab = (AdjAxisTab*)(wk + L.tab);
  const int n_tab = 2 * kAdjSlots * 12;
  k_adj_tables<<<(n_tab + 255) / 256, 256, 0, s>>>(H, W, tab);
  HIP_CHECK(hipGetLastError());
  k_adj_zero<<<256, 256, 0, s>>>((float*)(wk + L.part), 6 * adj_n_groups(H, W));
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

int32_t fk_adjoint_step(const fk_params* params, const float* D, const float* v,
                        const float* w, const float* u, int32_t H, int32_t W,
                        const fk_stimulus* stimuli, int32_t n_stimuli, double t, float dt,
                        float dx, const float* lam_v, const float* lam_w, const float* lam_u,
                        float* lam_v_out, float* lam_w_out, float* lam_u_out, float* grad_D,
                        void* work, size_t work_bytes, void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, v, w, u, lam_v, lam_w, lam_u, lam_v_out, lam_w_out, lam_u_out, grad_D,
                   work}) ||
      !check_scalar("t", t) || !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  const AdjLayout L = adj_layout(H, W);
  if (work_bytes < L.total)
    return set_error(FK_ERR_ARG, "adjoint workspace too small: need %zu bytes, got %zu",
                     L.total, work_bytes);
  StimSchedule sched(stimuli, n_stimuli);
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  const float* lin[3] = {lam_v, lam_w, lam_u};
  float* lout[3] = {lam_v_out, lam_w_out, lam_u_out};
  hipStream_t s = (hipStream_t)stream;
  HIP_CHECK(launch_rev(L, (char*)work, c, D, v, w, u, H, W, sched.at(t), dt, inv_dx2, lin,
                       nullptr, lout, grad_D, s));
  return FK_OK;
}

int32_t fk_adjoint_segment(const fk_params* params, const float* D, int32_t H, int32_t W,
                           const fk_stimulus* stimuli, int32_t n_stimuli, double t,
                           int32_t n_steps, float dt, float dx, const float* states,
                           const float* const* inject, float* lam_v, float* lam_w,
                           float* lam_u, float* grad_D, void* work, size_t work_bytes,
                           void* stream) {
  ErrorScope es;
  if (!check_params(params) || !check_grid(H, W) || !check_stimuli(stimuli, n_stimuli) ||
      !check_ptrs({D, lam_v, lam_w, lam_u, grad_D, work}) || !check_scalar("t", t) ||
      !check_scalar("dt", dt) || !check_dx(dx))
    return last_code();
  if (n_steps < 0) return set_error(FK_ERR_ARG, "n_steps must be >= 0, got %d", n_steps);
  if (n_steps > 0 && states == nullptr) return set_error(FK_ERR_ARG, "null states pointer");
  if (t + (double)n_steps > 16777216.0)
    return set_error(FK_ERR_ARG, "time index must stay below 2^24");
  const AdjLayout L = adj_layout(H, W);
  if (work_bytes < L.total)
    return set_error(FK_ERR_ARG, "adjoint workspace too small: need %zu bytes, got %zu",
                     L.total, work_bytes);
  hipStream_t s = (hipStream_t)stream;
  char* wk = (char*)work;
  const size_t n = (size_t)H * W;
  float* alt = (float*)(wk + L.lam);
  float* bufs[2][3] = {{lam_v, lam_w, lam_u}, {alt, alt + n, alt + 2 * n}};
  StimSchedule sched(stimuli, n_stimuli);
  const Coef c = make_coef(*params);
  const float inv_dx2 = (float)(1.0 / ((double)dx * (double)dx));
  int cur = 0;
  for (int32_t k = n_steps - 1; k >= 0; --k) {
    const float* x = states + (size_t)k * 3 * n;
    const float* lin[3] = {bufs[cur][0], bufs[cur][1], bufs[cur][2]};
    HIP_CHECK(launch_rev(L, wk, c, D, x, x + n, x + 2 * n, H, W, sched.at(t + (double)k), dt,
                         inv_dx2, lin, inject ? inject[k] : nullptr, bufs[cur ^ 1], grad_D, s));
    cur ^= 1;
  }
  if (cur == 1)
    for (int f = 0; f < 3; ++f)
      HIP_CHECK(hipMemcpyAsync(bufs[0][f], bufs[1][f], n * sizeof(float),
                               hipMemcpyDeviceToDevice, s));
  return FK_OK;
}

int32_t fk_adjoint_tau_grads(void* work, int32_t H, int32_t W, float* g_tau, void* stream) {
  ErrorScope es;
  if (!check_grid(H, W) || !check_ptrs({work, g_tau})) return last_code();
  const AdjLayout L = adj_layout(H, W);
  const size_t n = adj_n_groups(H, W);
  const int blocks = (int)std::min<size_t>((n + 255) / 256, (size_t)kRedBlocks);
  double* part = (double*)((char*)work + L.red);
  k_adj_reduce<<<blocks, 256, 0, (hipStream_t)stream>>>(
      (const double*)((char*)work + L.part), n, part);
  k_adj_reduce_final<<<1, 256, 0, (hipStream_t)stream>>>(part, blocks, g_tau);
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

}  // extern "C"
