// Device side of the adjoint of one forward-Euler step, shared by the per-grid
// kernel (fk_adjoint.hip) and the batched rollout (fk_rollout_batch.hip): one
// code path, so both give identical bits. The mathematics is described at the
// top of fk_adjoint.hip.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "fk_stream.h"

namespace fk {

// The per-axis operators A1 = crop G pad and A2 = crop G G pad of an axis of N
// cells (G: the gradient rule of cardiax/solve.py:230-250, one-sided on the two
// outermost padded entries of each side). Away from the edges their rows are
// central stencils. The rows of the kAdjB cells nearest each edge, and the
// transposed rows of the kAdjT cells nearest it, come from a table.
constexpr int kAdjB = 8, kAdjT = 13;
constexpr int kA1 = 3, kA2 = 5;  // |column - row| <= 3 in A1, <= 5 in A2
constexpr int kAdjSlots = 2 * kAdjT;

struct AdjRow {
  float a1[8], a2[12];  // A[i][i + d], d = -3 .. 3 and -5 .. 5 (and padding)
  float t1[8], t2[12];  // A[i - d][i]
};
struct alignas(16) AdjAxisTab {
  AdjRow r[kAdjSlots];
};

// Whether cell i lies within B of an edge (of a short axis: any cell).
__host__ __device__ inline bool adj_near(int i, int N, int B) {
  return N <= 2 * B || i < B || i >= N - B;
}
// Table row of a cell within kAdjT of an edge.
__host__ __device__ inline int adj_slot(int i, int N) {
  return N <= kAdjSlots || i < kAdjT ? i : i - (N - kAdjSlots);
}

// Central rows of A1 (d = -2..2) and A2 (d = -4..4).
#define FK_A1(d) ((d) == -2 ? 1.0f / 12.0f : (d) == -1 ? -2.0f / 3.0f : (d) == 1 ? 2.0f / 3.0f : (d) == 2 ? -1.0f / 12.0f : 0.0f)
#define FK_A2(d)                                                                          \
  ((d) == 0 ? -65.0f / 72.0f                                                              \
            : ((d) == 1 || (d) == -1) ? 1.0f / 9.0f                                       \
            : ((d) == 2 || (d) == -2) ? 4.0f / 9.0f                                       \
            : ((d) == 3 || (d) == -3) ? -1.0f / 9.0f                                      \
            : ((d) == 4 || (d) == -4) ? 1.0f / 144.0f : 0.0f)

// Gradient rule as a matrix on n padded entries: the coefficient of entry q in
// row p.
__host__ __device__ inline double g_coef(int p, int q, int n) {
  const int d = q - p;
  if (p <= 1) {
    const double c[4] = {-11.0 / 6.0, 3.0, -1.5, 1.0 / 3.0};
    return (d >= 0 && d <= 3) ? c[d] : 0.0;
  }
  if (p >= n - 2) {
    const double c[4] = {-1.0 / 3.0, 1.5, -3.0, 11.0 / 6.0};
    return (d >= -3 && d <= 0) ? c[d + 3] : 0.0;
  }
  const double c[5] = {1.0 / 12.0, -2.0 / 3.0, 0.0, 2.0 / 3.0, -1.0 / 12.0};
  return (d >= -2 && d <= 2) ? c[d + 2] : 0.0;
}

// Edge padding as a matrix: padded entry q takes original cell clamp(q-1).
__host__ __device__ inline double pad_coef(int q, int i, int N) {
  int s = q - 1;
  s = s < 0 ? 0 : (s > N - 1 ? N - 1 : s);
  return s == i ? 1.0 : 0.0;
}

// A1[j][i] and A2[j][i] (0 off the axis): the rules composed exactly for the
// rows near an edge, the central stencils elsewhere.
__host__ __device__ inline void adj_coef(int j, int i, int N, float& a1, float& a2) {
  a1 = a2 = 0.0f;
  if (j < 0 || j >= N || i < 0 || i >= N) return;
  const int d = i - j;
  if (!adj_near(j, N, kAdjB)) {
    a1 = FK_A1(d);
    a2 = FK_A2(d);
    return;
  }
  const int n = N + 2, pj = j + 1;  // padded row of original j
  double s1 = 0.0, s2 = 0.0;
  for (int q = pj - 3; q <= pj + 3; ++q) {
    if (q < 0 || q >= n) continue;
    const double gq = g_coef(pj, q, n);
    if (gq == 0.0) continue;
    s1 += gq * pad_coef(q, i, N);
    double gp = 0.0;  // A2 = crop G G pad: row pj of G times column i of G pad
    for (int s = q - 3; s <= q + 3; ++s)
      if (s >= 0 && s < n) gp += g_coef(q, s, n) * pad_coef(s, i, N);
    s2 += gq * gp;
  }
  a1 = (float)s1;
  a2 = (float)s2;
}

// Sums of taps in the order of d. dL/dD adds L A2 u and A1^T (L A1 u), which
// nearly cancel, so it carries the rounding of these sums many times over: two
// differences of differences in their place take fewer operations, but moved
// dL/dD by 7e-5 over 500 steps and gained under 2 us of 29.
// sum_d A1(d) x[s d], x[0] the centre; s = -1 the transposed row.
template <int s>
__device__ __forceinline__ float a1_sum(const float* x) {
  float g = FK_A1(-2) * x[-2 * s];
  g = fmaf(FK_A1(-1), x[-s], g);
  g = fmaf(FK_A1(1), x[s], g);
  return fmaf(FK_A1(2), x[2 * s], g);
}

__device__ __forceinline__ float a2_sum(const float* x) {
  float g = FK_A2(-4) * x[-4];
#pragma unroll
  for (int d = -3; d <= 4; ++d) g = fmaf(FK_A2(d), x[d], g);
  return g;
}

// The same with a table row, each product rounded.
__device__ __forceinline__ float tab_sum(const float* t, const float* x, int n) {
#pragma clang fp contract(off)
  float g = 0.0f;
#pragma unroll
  for (int d = -n; d <= n; ++d) g = g + t[d + n] * x[d];
  return g;
}

// sum_d A2(d) y2[-d] + A1(d) y1[-d]: the transposed diffusion operators.
__device__ __forceinline__ float at_sum(const float* y2, const float* y1) {
  float g = 0.0f;
#pragma unroll
  for (int d = -4; d <= 4; ++d) {
    g = fmaf(FK_A2(d), y2[-d], g);
    if (d >= -2 && d <= 2 && d != 0) g = fmaf(FK_A1(d), y1[-d], g);
  }
  return g;
}

// A value and its neighbours up to n columns away: x[n + d] is column + d.
template <int n>
__device__ __forceinline__ void lane_window(float y, float x[2 * n + 1]) {
  x[n] = y;
#pragma unroll
  for (int d = 1; d <= n; ++d) {
    x[n + d] = from_right(x[n + d - 1]);
    x[n - d] = from_left(x[n - d + 1]);
  }
}

constexpr int kRevOut = 54;   // output columns per wave: 5 halo lanes on each side
constexpr int kRevHalo = 5;   // what an edge's rules reach (4 away from the edges)

// Tau accumulators: one triple of doubles per strip and row. At most 54 terms are
// added in float before a sum goes to its double, and the sums do not depend on
// the band height.
__host__ __device__ inline int adj_strips(int W) { return (W + kRevOut - 1) / kRevOut; }
__host__ __device__ inline size_t adj_n_groups(int H, int W) {
  return (size_t)adj_strips(W) * (size_t)H;
}

// Stimulus fields of one step as an active list (count(), on(m), field(m)).
struct AdjStimList {
  const StimArgs& sa;
  __device__ int count() const { return sa.n; }
  __device__ bool on(int) const { return true; }
  __device__ const float* field(int m) const { return sa.f[m]; }
};

// Sums over the wave of up to four values, each into its own 16 lanes, by lane
// moves (no LDS): half the operations of a tree for each value.
// x of the lanes 0-15 and 32-47 and y of the same, each with the 16 lanes above
// it: x's sums go to the lower 16, y's to the upper.
__device__ __forceinline__ float pair_sum16(float x, float y) {
  const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false,
                                                  false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// The same of the lower and the upper 32 lanes.
__device__ __forceinline__ float pair_sum32(float x, float y) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false,
                                                  false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
// Sum over each 16 lanes, in all of them.
__device__ __forceinline__ float row_sum(float x) {
  auto add = [](float a, auto ctrl) {
    const int m = __builtin_amdgcn_update_dpp(0, __float_as_int(a), decltype(ctrl)::value, 0xf,
                                              0xf, false);
    return a + __int_as_float(m);
  };
  using std::integral_constant;
  x = add(x, integral_constant<int, 0x128>{});  // row_ror:8
  x = add(x, integral_constant<int, 0x124>{});  // row_ror:4
  x = add(x, integral_constant<int, 0x122>{});  // row_ror:2
  return add(x, integral_constant<int, 0x121>{});  // row_ror:1
}

struct AdjArgs {
  const float *v, *w, *u, *D;        // the state of the step, the D-map
  const float *lv, *lw, *lu, *inj;   // cotangent of the next state; inj (may be null) adds to lu
  float *lv_o, *lw_o, *lu_o, *gD;    // cotangent of this state; dL/dD (accumulated)
  double* g_tau;                     // tau accumulators
  const AdjAxisTab* tab;             // rows, columns
};

// One reverse step of the band of R rows at rs of the strip at cs: one
// wave, lane l on column cs - 5 + l, rows walked as the forward streaming tile
// walks them: windows of u, D and the cotangent L = lu + inj in registers,
// column neighbours by DPP, no LDS. The fields that the transposed operators
// read (D L, D_x L, L u_x and the same along y) are formed from those windows,
// so a reverse step reads and writes only what it must (state 12 bytes,
// cotangent 12 in and 12 out, D 4, dL/dD 8: 48 per cell, and the windows' halo
// rows). It replaced a kernel that kept seven derived fields in memory (104
// bytes by design, 121-142 measured), two threads per cell:
// 59.1 us before, 27.3 now per step of 12 problems of 128^2 to 512^2 (1.26 M
// cells; 161 registers, three waves per SIMD); 61 us for 3.84 M cells (3.0 TB/s of
// the 48 bytes); 7.05 and, a wave per row, 5.7 to 6.0 at 256^2, where a launch and an edge
// wave's own instructions bound both.
// XG, YG: a row within 13 of an edge, a column within 13 of a side. In such a
// band each row, and in such a strip each lane, takes the table or the central
// taps by itself, so neither the band height nor the strip changes a bit.
// tab: the wave's LDS copy of the tables, filled here where they are used (read
// from memory one row after another they were most of an edge wave's time: a
// dozen dependent scalar loads, 33 us in place of 29 for the 12 problems).
// The waves of a block may run different instantiations (an edge band next to an
// inner one), so it holds no workgroup barrier.
template <int R, bool XG, bool YG, class SV>
__device__ __forceinline__ void adj_tile(const Coef& c, const AdjArgs& a, int H, int W,
                                         const SV& sv, float dt, float inv_dx2, int rs, int cs,
                                         AdjAxisTab* tab) {
#pragma clang fp contract(off)
  static_assert(R == 1 || R == 2 || R == 4, "the tau sums of a band");
  constexpr int E = XG ? kRevHalo : 4;  // window rows above and below the band
  constexpr int NW = R + 2 * E, NG = NW - 4;  // window; its first differences
  const int lane = threadIdx.x & 63;
  const int col = cs - kRevHalo + lane;
  const bool in_col = col >= 0 && col < W;
  // the lane's cell near a side, and its table row
  const bool nearB = YG && in_col && adj_near(col, W, kAdjB);
  const bool nearT = YG && in_col && adj_near(col, W, kAdjT);
  const int tslot = nearT ? adj_slot(col, W) : 0;
  const uint32_t off = (uint32_t)(YG ? clampi(col, 0, W - 1) : col) * 4u;
  auto at = [&](const float* f, int r) {
    return ld(f + (size_t)(XG ? clampi(r, 0, H - 1) : r) * (size_t)W, off);
  };

  constexpr int kTab4 = (int)(sizeof(AdjAxisTab) / sizeof(f32x4)), kTabN = (kTab4 + 63) / 64;
  f32x4 tx[XG ? kTabN : 1], ty[YG ? kTabN : 1];
#pragma unroll
  for (int k = 0; k < kTabN; ++k) {
    const uint32_t o = (uint32_t)min(64 * k + lane, kTab4 - 1);
    if constexpr (XG) tx[k] = ((const f32x4 __attribute__((address_space(1)))*)(gcbytes)a.tab)[o];
    if constexpr (YG)
      ty[k] = ((const f32x4 __attribute__((address_space(1)))*)(gcbytes)(a.tab + 1))[o];
  }
  float uu[NW], dd[NW], LL[NW];
#pragma unroll
  for (int k = 0; k < NW; ++k) uu[k] = at(a.u, rs - E + k);
#pragma unroll
  for (int k = 0; k < NW; ++k) LL[k] = at(a.lu, rs - E + k);
#pragma unroll
  for (int k = 0; k < NW; ++k) dd[k] = at(a.D, rs - E + k);
  if (a.inj) {
#pragma unroll
    for (int k = 0; k < NW; ++k) LL[k] = LL[k] + at(a.inj, rs - E + k);
  }
  // The tau sums of the band's rows: lane 16 k + f holds sum f of row k and loads
  // it here, so that it arrives with the rest (read where it is added to, it
  // ended the wave with a trip to memory).
  const int tau_row = lane >> 4, tau_f = lane & 15;
  const bool has_tau = tau_f < 3 && tau_row < (XG ? min(R, H - rs) : R);
  double __attribute__((address_space(1)))* gt =
      (double __attribute__((address_space(1)))*)a.g_tau +
      3 * ((size_t)(cs / kRevOut) * H + rs + tau_row) + tau_f;
  const double g0 = has_tau ? *gt : 0.0;
  float vv[R], ww[R], lvv[R], lww[R], gd[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    vv[k] = at(a.v, rs + k);
    ww[k] = at(a.w, rs + k);
    lvv[k] = at(a.lv, rs + k);
    lww[k] = at(a.lw, rs + k);
    gd[k] = at(a.gD, rs + k);
  }
  if constexpr (XG || YG) {
#pragma unroll
    for (int k = 0; k < kTabN; ++k) {
      const int o = min(64 * k + lane, kTab4 - 1);
      if constexpr (XG) ((f32x4*)&tab[0])[o] = tx[k];
      if constexpr (YG) ((f32x4*)&tab[1])[o] = ty[k];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // read by this wave only
    __builtin_amdgcn_wave_barrier();
  }
  if (XG || YG) {  // no cotangent beyond the grid
#pragma unroll
    for (int k = 0; k < NW; ++k) {
      const int i = rs - E + k;
      LL[k] = (!XG || (i >= 0 && i < H)) && (!YG || in_col) ? LL[k] : 0.0f;
    }
  }

  // A1 of a window at its entry m, row r; `fused`: of the D-map
  auto slope = [&](const float* x, int m, int r, bool fused) {
    if (XG && r >= 0 && r < H && adj_near(r, H, kAdjB)) {
      const float* t = tab[0].r[adj_slot(r, H)].a1;
      float g = 0.0f;
#pragma unroll
      for (int d = -kA1; d <= kA1; ++d)
        if (m + d >= 0 && m + d < NW) {  // taps beyond the window are 0
          const float y = x[m + d];
          g = fused ? fmaf(t[d + kA1], y, g) : g + t[d + kA1] * y;
        }
      return g;
    }
    return a1_sum<1>(x + m);
  };
  // Q2 = D L; u_x, P = L u_x and Q1 = D_x L
  float q2[NW], pp[NG], q1[NG];
#pragma unroll
  for (int k = 0; k < NW; ++k) q2[k] = dd[k] * LL[k];
#pragma unroll
  for (int k = 0; k < NG; ++k) {
    const int m = k + 2, r = rs - E + m;
    pp[k] = LL[m] * slope(uu, m, r, false);
    q1[k] = slope(dd, m, r, true) * LL[m];
  }

  float even[3], ts[3];  // tau terms of an even row; of the rows so far, by 16 lanes
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int i = rs + k, m = k + E, mf = m - 2;  // row, its entries in the windows
    const float uc = uu[m], L = LL[m];
    // along the rows: A2 u, s = A2^T Q2 + A1^T Q1, e = A1^T P
    float lapx, sx, ex;
    if (XG && i < H && adj_near(i, H, kAdjB))
      lapx = tab_sum(tab[0].r[adj_slot(i, H)].a2, uu + m, kA2);
    else
      lapx = a2_sum(uu + m);
    if (XG && i < H && adj_near(i, H, kAdjT)) {
      const AdjRow& t = tab[0].r[adj_slot(i, H)];
      sx = ex = 0.0f;
#pragma unroll
      for (int d = -kA2; d <= kA2; ++d) {
        if (d >= -kA1 && d <= kA1) {
          sx = fmaf(t.t1[d + kA1], q1[mf - d], sx);
          ex = fmaf(t.t1[d + kA1], pp[mf - d], ex);
        }
        sx = fmaf(t.t2[d + kA2], q2[m - d], sx);
      }
    } else {
      sx = at_sum(q2 + m, q1 + mf);
      ex = a1_sum<-1>(pp + mf);
    }
    // along the columns
    float lapy, sy, ey;
    if constexpr (!YG) {
      float x[9], z[5], y2[9], y1[5], yp[5];
      lane_window<4>(uc, x);
      lane_window<2>(dd[m], z);
      lapy = a2_sum(x + 4);
      lane_window<4>(q2[m], y2);
      lane_window<2>(a1_sum<1>(z + 2) * L, y1);
      lane_window<2>(L * a1_sum<1>(x + 4), yp);
      sy = at_sum(y2 + 4, y1 + 2);
      ey = a1_sum<-1>(yp + 2);
    } else {
      // the lane's table row, loaded anew for each row of the band: kept, it
      // would hold 40 registers (lane shifts are evaluated by the whole wave,
      // then selected)
      int slot = tslot;
      asm volatile("" : "+v"(slot));
      const AdjRow& t = tab[1].r[slot];
      float x[11], z[7], y2[11], y1[7], yp[7];
      lane_window<5>(uc, x);
      lane_window<3>(dd[m], z);
      const float lt = tab_sum(t.a2, x + 5, kA2), gt = tab_sum(t.a1, x + 5, kA1);
      float ft = 0.0f;
#pragma unroll
      for (int d = -kA1; d <= kA1; ++d) ft = fmaf(t.a1[d + kA1], z[d + 3], ft);
      const float lc = a2_sum(x + 5), gc = a1_sum<1>(x + 5), fc = a1_sum<1>(z + 3);
      lapy = nearB ? lt : lc;
      lane_window<5>(q2[m], y2);
      lane_window<3>((nearB ? ft : fc) * L, y1);
      lane_window<3>(L * (nearB ? gt : gc), yp);
      float s = 0.0f, e = 0.0f;
#pragma unroll
      for (int d = -kA2; d <= kA2; ++d) {
        if (d >= -kA1 && d <= kA1) {
          s = fmaf(t.t1[d + kA1], y1[3 - d], s);
          e = fmaf(t.t1[d + kA1], yp[3 - d], e);
        }
        s = fmaf(t.t2[d + kA2], y2[5 - d], s);
      }
      const float sc = at_sum(y2 + 5, y1 + 3), ec = a1_sum<-1>(yp + 3);
      sy = nearT ? s : sc;
      ey = nearT ? e : ec;
    }
    const float lap = lapx + lapy;
    // reaction, gates as fixed masks
    const bool q = uc >= c.V_c;
    const float inv_tvm = (uc >= c.V_v) ? c.inv_tv2m : c.inv_tv1m;
    const float dfv_dv = q ? -c.inv_tvp : -inv_tvm;
    const float dfw_dw = q ? -c.inv_twp : -c.inv_twm;
    const float S = half_one_plus_tanh(c, uc);  // (1 + tanh(k (u - V_csi))) / 2
    // dS/du = 2k S (1 - S); kk = -2 k log2(e)
    const float dS = -c.kk * 0.69314718055994531f * S * (1.0f - S);
    // j_ion = -(j_fi + j_so + j_si) / Cm
    const float a1 = (uc - c.V_c) * (1.0f - uc) * c.inv_td * c.inv_cm;
    const float djdv = q ? a1 : 0.0f;
    const float djdw = S * c.inv_tsi * c.inv_cm;
    const float a0 = q ? -vv[k] * fmaf(-2.0f, uc, 1.0f + c.V_c) * c.inv_td : c.inv_t0;
    const float djdu = -fmaf(-(ww[k] * dS), c.inv_tsi, a0) * c.inv_cm;
    // a stimulus replaces j_ion: no cotangent reaches it where one is active
    bool stim = false;
    for (int f = 0; f < sv.count(); ++f)
      if (sv.on(f)) stim = stim || at(sv.field(f), i) != 0.0f;
    const float lus = stim ? 0.0f : L;
    const bool out = lane >= kRevHalo && lane < kRevHalo + kRevOut && col < W && (!XG || i < H);
    if (out) {
      const size_t ro = (size_t)i * (size_t)W;
      st(a.lv_o + ro, off, fmaf(dt, fmaf(dfv_dv, lvv[k], djdv * lus), lvv[k]));
      st(a.lw_o + ro, off, fmaf(dt, fmaf(dfw_dw, lww[k], djdw * lus), lww[k]));
      st(a.lu_o + ro, off, fmaf(dt, fmaf(djdu, lus, (sx + sy) * inv_dx2), L));
      st(a.gD + ro, off, fmaf(dt * (fmaf(L, lap, ex) + ey), inv_dx2, gd[k]));
    }
    // tau gradients: d j_ion / d tau
    const float lt = out ? lus * dt : 0.0f;
    const float t_d = (q ? -vv[k] * a1 * c.inv_td : 0.0f) * lt;
    const float t_r = (q ? c.inv_tr * c.inv_tr * c.inv_cm : 0.0f) * lt;
    const float t_si = (-ww[k] * S * c.inv_tsi * c.inv_tsi * c.inv_cm) * lt;
    const float t[3] = {t_d, t_r, t_si};
#pragma unroll
    for (int f = 0; f < 3; ++f) {
      if (R > 1 && k % 2 == 0) {
        even[f] = t[f];
      } else {
        const float p = pair_sum16(R > 1 ? even[f] : t[f], t[f]);
        ts[f] = k == 3 ? pair_sum32(ts[f], p) : p;
      }
    }
  }
#pragma unroll
  for (int f = 0; f < 3; ++f) ts[f] = row_sum(R == 4 ? ts[f] : pair_sum32(ts[f], ts[f]));
  if (has_tau) *gt = g0 + (double)(tau_f == 0 ? ts[0] : tau_f == 1 ? ts[1] : ts[2]);
}

// Up to this many bands of 2 rows a reverse step runs a wave per row: the waves
// all run at once and an edge wave's rows, 1.2 us each, set the time. Forward and
// backward over 200 steps, 2 rows per wave and one: 128^2 1.79 and 1.54 ms, 256^2
// (640 bands) 1.83 and 1.61, 400^2 (1600) 2.23 and 2.16, 460^2 (2070) 2.28 and 2.34,
// 600^2 (3600) 2.96 and 2.99.
constexpr int kRevRowTiles = 2048;

// Whether the band of R rows at rs, the strip at cs take the edge rules.
__host__ __device__ inline bool adj_edge_band(int rs, int R, int H) {
  return rs < kAdjT || rs + R + kAdjT > H;
}
__host__ __device__ inline bool adj_edge_strip(int cs, int W) {
  return cs < kAdjT || cs + kRevOut + kAdjT > W;
}

// adj_tile with its edge flags (bit 0 band, bit 1 strip).
template <int R, class SV>
__device__ __forceinline__ void adj_tile_any(const Coef& c, const AdjArgs& a, int H, int W,
                                             const SV& sv, float dt, float inv_dx2, int rs, int cs,
                                             int flags, AdjAxisTab* tab) {
  switch (flags) {
    case 0: adj_tile<R, false, false>(c, a, H, W, sv, dt, inv_dx2, rs, cs, tab); break;
    case 1: adj_tile<R, true, false>(c, a, H, W, sv, dt, inv_dx2, rs, cs, tab); break;
    case 2: adj_tile<R, false, true>(c, a, H, W, sv, dt, inv_dx2, rs, cs, tab); break;
    default: adj_tile<R, true, true>(c, a, H, W, sv, dt, inv_dx2, rs, cs, tab); break;
  }
}

// Blocks of the first pass of the tau reduction (k_adj_reduce).
constexpr int kRedBlocks = 512;

// Workspace layout: [tables (2 axes)][tau accumulators: 3 doubles per group]
// [cotangent ping-pong: 3 fields][tau block sums]
struct AdjLayout {
  size_t tab, part, lam, red, total;
};

inline AdjLayout adj_layout(int H, int W) {
  AdjLayout L;
  const size_t cells = (size_t)H * W;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  L.tab = take(2 * sizeof(AdjAxisTab));
  L.part = take(3 * adj_n_groups(H, W) * sizeof(double));
  L.lam = take(3 * cells * sizeof(float));
  L.red = take(3 * kRedBlocks * sizeof(double));
  L.total = o;
  return L;
}

}  // namespace fk
