// The device half of the reference's random scar D-map generator
// (deepx/utils_scars.py:246-426, called by deepx/generate.py:79-83): the
// rasterisation of the closed spline contours into a mask and the Gaussian
// blur that tapers its edges. The contours themselves (a few hundred points)
// are built on the host, as the reference builds them with scipy.
//
// Rasterisation (drawpolyintoemptycanvas, :79-97, via skimage.draw.polygon):
// a pixel (r, c) is inside a polygon when it lies in the polygon's bounding
// box [int(max(0, min r)), ceil(max r)] x [int(max(0, min c)), ceil(max c)]
// and the crossing-number test at its centre (integer coordinates) holds:
// an edge (i, j) counts when (r_i <= r < r_j or r_j <= r < r_i) and
// c < (c_j - c_i)(r - r_i) / (r_j - r_i) + c_i, in double precision. The
// blobs of one scar are OR'ed (MakeAndSumCompositeBlob, :377-381: summed and
// clipped to 1); pixels outside the image are dropped, as JAX's scatter drops
// them.
//
// Blur (blur_scar, :402-406): scipy.signal.convolve2d(scar, kernel, "same"):
// out[i, j] = sum_{p, q} k[p, q] in[i + (kh-1)/2 - p, j + (kw-1)/2 - q]
// (integer halves), zero outside the image; products and sums in double. A
// kernel that is an outer product (the generator's Gaussian, unless its tail
// was cut) and not small runs as a column pass and a row pass.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "cardiax_amd.h"
#include "fk_host.h"
#include "fk_stream.h"

namespace fk {

struct PolyBox {
  int r0, r1, c0, c1;  // inclusive bounding box of tested pixels
  int begin, end;      // vertex range
};

// Crossing-number test at (x, y) = (column, row) of the closed polygon with
// vertices (cp[k], rp[k]), k in [b, e).
__device__ __forceinline__ bool inside_polygon(const double* __restrict__ rp,
                                               const double* __restrict__ cp, int b, int e,
                                               double y, double x) {
#pragma clang fp contract(off)
  bool in = false;
  int j = e - 1;
  for (int i = b; i < e; ++i) {
    const double yi = rp[i], yj = rp[j], xi = cp[i], xj = cp[j];
    if (((yi <= y && y < yj) || (yj <= y && y < yi)) && (x < (xj - xi) * (y - yi) / (yj - yi) + xi))
      in = !in;
    j = i;
  }
  return in;
}

// One wave per row and kRasterCols columns of it. An edge's part of the test at
// row y is the column where the edge crosses y, the same for every pixel of the
// row: the wave collects a polygon's crossings once (a ballot per 64 edges), and a
// pixel is inside when an odd number of them lie to its right. A pixel then costs
// a comparison per crossing (two to six on the generator's contours) instead of
// one per vertex: 47 us before, 13 us now for 5 contours of 101 vertices at
// 1200 x 1200. Columns per wave: 64 take 27 us there, 128 18, 512 14, and a
// whole row 19 (and 4 x 100000 up to 800, where 256 take 10). A polygon with more
// crossings than the list has room for is tested pixel by pixel; polygons beyond
// kRasterPolys are a second pass over the row.
constexpr int kRasterCross = 256, kRasterPolys = 32;
constexpr int kRasterCols = 256;

__global__ void __launch_bounds__(256)
k_raster_polygons(float* __restrict__ mask, int H, int W, const double* __restrict__ rp,
                  const double* __restrict__ cp, const PolyBox* __restrict__ boxes, int n_polys) {
#pragma clang fp contract(off)
  __shared__ double s_cross[4][kRasterCross];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int r = blockIdx.x * 4 + wave;
  if (r >= H) return;  // whole wave; the kernel has no barrier
  double* cross = s_cross[wave];
  float* out = mask + (size_t)r * W;
  const double y = (double)r;
  for (int g = 0; g == 0 || g < n_polys; g += kRasterPolys) {
    const int np = min(n_polys - g, kRasterPolys);
    // lane p keeps polygon g + p: its columns and crossings (first, count; a
    // count of -1: test by pixel)
    int c0 = 0, c1 = -1, first = 0, count = 0, used = 0;
    for (int p = 0; p < np; ++p) {
      const PolyBox bx = boxes[g + p];
      if (r < bx.r0 || r > bx.r1) continue;
      int n = 0;
      for (int e = bx.begin; e < bx.end; e += 64) {
        const int i = min(e + lane, bx.end - 1), j = i == bx.begin ? bx.end - 1 : i - 1;
        const double yi = rp[i], yj = rp[j], xi = cp[i], xj = cp[j];
        const bool hit = e + lane < bx.end && ((yi <= y && y < yj) || (yj <= y && y < yi));
        const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
        const int at = used + n + __popcll(m & ((1ull << lane) - 1));
        if (hit && at < kRasterCross) cross[at] = (xj - xi) * (y - yi) / (yj - yi) + xi;
        n += __popcll(m);
      }
      const bool fits = used + n <= kRasterCross;
      if (lane == p) {
        c0 = bx.c0;
        c1 = bx.c1;
        first = used;
        count = fits ? n : -1;
      }
      if (fits) used += n;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // the wave's own LDS writes
    __builtin_amdgcn_wave_barrier();
    // this block's columns, run by run (one run unless W exceeds 65535 of them)
    for (int64_t x = (int64_t)blockIdx.y * kRasterCols; x < W;
         x = (x + 64) % kRasterCols ? x + 64 : x + 64 + (int64_t)(gridDim.y - 1) * kRasterCols) {
      const int cb = (int)x;
      const int c = cb + lane;
      bool on = false;
      for (int p = 0; p < np; ++p) {
        const int p0 = __builtin_amdgcn_readlane(c0, p), p1 = __builtin_amdgcn_readlane(c1, p);
        if (p1 < cb || p0 > cb + 63) continue;
        const int f = __builtin_amdgcn_readlane(first, p), n = __builtin_amdgcn_readlane(count, p);
        bool in = false;
        if (n >= 0) {
          for (int k = 0; k < n; ++k) in ^= (double)c < cross[f + k];
        } else {
          in = inside_polygon(rp, cp, boxes[g + p].begin, boxes[g + p].end, y, (double)c);
        }
        on |= in && c >= p0 && c <= p1;
      }
      if (c < W && (g == 0 || on)) out[c] = on ? 1.0f : 0.0f;
    }
    __builtin_amdgcn_wave_barrier();  // the list is read before the next group fills it
  }
}

// R outputs down a column per thread. With d = s - (i0 + oi) the offset of
// input row s from the thread's first output row, output r takes tap row
// p = r - d. The thread walks d over [-(kh-1), R-1] in chunks of R rows and,
// within a chunk, every tap column q: R input values (one load each, reused
// by up to R outputs; the chunk's rows stay in L1 across q) and the chunk's
// 2R - 1 taps of column q, contiguous and wave-uniform in the padded,
// transposed copy of the kernel (k_conv_prepare: zeros outside [0, kh), so no
// test per tap). The inputs come from a zero-padded copy of the image
// (pad_image) wide enough for every row and column a thread reaches, so
// the loads need no clamp and no select. Per output the sum runs over
// chunks, then q, then d, in double; rounded once.
constexpr int kConvRows = 8;
constexpr int kConvPadFront = 2 * kConvRows - 2;

__host__ __device__ constexpr int conv_padded_rows(int kh) { return kh + 3 * kConvRows - 3; }

// The zero-padded image: PT rows above and below, PL columns left and PR
// right of the H x W image.
struct ConvPad {
  int PT, PL, Hp, Wp;
};

__host__ __device__ inline ConvPad conv_pad(int H, int W, int kh, int kw) {
  ConvPad p;
  p.PT = kh + 2 * kConvRows;
  p.PL = kw;
  p.Hp = H + 2 * p.PT;
  p.Wp = W + 2 * kw + 64;
  return p;
}

// The factors of an outer product k[p][q] = c[p] r[q]: c is the column of the
// centre tap, r the row of it over the tap itself. Both are stored in the
// order the passes walk them, last tap first.
constexpr int kSepR = 8;  // outputs per thread of a pass

// Blocks of k_conv_prepare, and a flag of each; then one that is set when the image
// holds a value that is not finite.
constexpr int kConvFlags = 64;

struct ConvWork {  // offsets of the workspace, bytes
  size_t taps, col, row, flag, image, total;
};

inline ConvWork conv_work(int H, int W, int kh, int kw) {
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  const ConvPad pd = conv_pad(H, W, kh, kw);
  ConvWork w;
  w.taps = 0;
  w.col = up((size_t)kw * conv_padded_rows(kh) * sizeof(double));
  w.row = w.col + up((size_t)kh * sizeof(double));
  w.flag = w.row + up((size_t)kw * sizeof(double));
  w.image = w.flag + up((kConvFlags + 1) * sizeof(int));
  // the padded image, or the column pass's result in double
  w.total = w.image + std::max((size_t)pd.Hp * pd.Wp * sizeof(float),
                               (size_t)H * W * sizeof(double));
  return w;
}

// Whether an outer-product kernel takes the two passes: from kMinPasses units of the
// direct sum on, a unit being one tap column of one chunk of rows. Direct and passes,
// us a call: 10 x 10 taps (30 units) 22.7 and 22.0 at 1000 x 700, 18.7 and 14.2 at 64^2;
// 9 x 9 (18) 18.2 and 19.9, 16.1 and 12.5; 60 x 2 (18) 20.0 and 25.6; 3 x 3 13.7 and 19.5.
constexpr int kMinPasses = 24;

// The padded, transposed taps and, with `passes`, the factors and whether the kernel
// is the outer product of them: every tap c[p] r[q] within 2^-48 of itself (flags all
// 1). The passes' error is then below the direct sum's: at most 2^-50.8 of the result
// and 2^-49.0 with 10 to 19 taps a side, 2^-49.9 and 2^-46.4 with 40 to 69. The
// Gaussian's taps are exp(-(x^2 + y^2) / 2 s^2), whose argument (at most 16 before the
// tail is cut) carries a few roundings of 2^-53 of itself: over 1400 draws of the
// generator's width at sides from 4 to 130 no tap was off by more than 2^-48.7. A zero
// or non-finite centre tap fails (its row is not finite), and so does a tap cut to zero.
__global__ void __launch_bounds__(256)
k_conv_prepare(const double* __restrict__ k, int kh, int kw, bool passes,
               double* __restrict__ kt, double* __restrict__ col, double* __restrict__ row,
               int* __restrict__ flags) {
  const int kp = conv_padded_rows(kh);
  const int pc = (kh - 1) / 2, qc = (kw - 1) / 2;
  const int64_t t0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = 256 * kConvFlags;
  bool outer = passes;
  for (int64_t t = t0; t < (int64_t)kw * kp; t += step) {
    const int q = (int)(t / kp), p = (int)(t - (int64_t)q * kp) - kConvPadFront;
    const bool in = p >= 0 && p < kh;
    const double x = in ? k[(size_t)p * kw + q] : 0.0;
    kt[t] = x;
    if (!passes || !in) continue;
    const double c = k[(size_t)p * kw + qc], r = k[(size_t)pc * kw + q] / k[(size_t)pc * kw + qc];
    outer = outer && fabs(x - c * r) <= 0x1p-48 * fabs(x) && isfinite(x);
    if (q == qc) col[kh - 1 - p] = c;
    if (p == pc) row[kw - 1 - q] = r;
  }
  outer = __syncthreads_and(outer);
  if (threadIdx.x == 0) flags[blockIdx.x] = outer;
  if (t0 == 0) flags[kConvFlags] = 0;
}

__device__ __forceinline__ bool is_outer(const int* __restrict__ flags) {
  static_assert(kConvFlags == 64, "a flag per lane");
  return __builtin_amdgcn_ballot_w64(flags[threadIdx.x & 63] != 0) == ~0ull;
}

__device__ __forceinline__ void pad_image(const float* __restrict__ src, int H, int W, ConvPad pd,
                                          float* __restrict__ pad, int* __restrict__ nonfinite) {
  const size_t n = (size_t)pd.Hp * pd.Wp, step = (size_t)gridDim.x * 256;
  const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int dr = (int)(step / pd.Wp), dc = (int)(step - (size_t)dr * pd.Wp);
  int r = (int)(first / pd.Wp), c = (int)(first - (size_t)r * pd.Wp);
  bool bad = false;
  for (size_t idx = first; idx < n; idx += step) {
    const int i = r - pd.PT, j = c - pd.PL;
    const float x = (i >= 0 && i < H && j >= 0 && j < W) ? src[(size_t)i * W + j] : 0.0f;
    pad[idx] = x;
    bad = bad || !isfinite(x);
    r += dr;
    c += dc;
    if (c >= pd.Wp) {
      c -= pd.Wp;
      ++r;
    }
  }
  if (bad) *nonfinite = 1;
}

// Block b of the direct sum. FINITE: the zero taps around the kernel may be
// multiplied by any input; else they are left out, so that an infinite input
// reaches the outputs of its window only.
template <bool FINITE>
__device__ __forceinline__ void convolve_same(const float* __restrict__ pad, int H, int W,
                                              ConvPad pd, const double* __restrict__ kt, int kh,
                                              int kw, float* __restrict__ dst, int b) {
  constexpr int R = kConvRows;
  const int bx = (W + 63) / 64;
  const int j = b % bx * 64 + (threadIdx.x & 63);
  const int i0 = __builtin_amdgcn_readfirstlane((b / bx * 4 + (int)(threadIdx.x >> 6)) * R);
  if (i0 >= H) return;  // wave-uniform
  const int oi = (kh - 1) / 2, oj = (kw - 1) / 2;
  const int kp = conv_padded_rows(kh);
  const int n_chunks = (kh + 2 * R - 2) / R;
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  for (int ch = 0; ch < n_chunks; ++ch) {
    const int d0 = -(kh - 1) + ch * R;
    // padded row of input row i0 + oi + d0 + m (wave-uniform)
    const float* row0 = pad + (size_t)(i0 + oi + d0 + pd.PT) * pd.Wp;
    // taps p = -d0 - (R-1) + e of column q sit at kt[q kp + R - 1 - d0 + e]
    const double* tcol = kt + (R - 1 - d0);
    for (int q = 0; q < kw; ++q) {
      const uint32_t cb = (uint32_t)(j + oj - q + pd.PL) * 4u;  // padded column, bytes
      double x[R];
#pragma unroll
      for (int m = 0; m < R; ++m)
        x[m] = (double)ld(row0 + (size_t)m * pd.Wp, cb);
      const double* t = tcol + (size_t)q * kp;
#pragma unroll
      for (int m = 0; m < R; ++m)    // d = d0 + m
#pragma unroll
        for (int r = 0; r < R; ++r)  // p = r - d: tap index r - m + R - 1
        {
          const double a = fma(t[r - m + R - 1], x[m], acc[r]);
          const int p = r - d0 - m;
          acc[r] = FINITE || (p >= 0 && p < kh) ? a : acc[r];
        }
    }
  }
  if (j < W) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (i0 + r < H) dst[(size_t)(i0 + r) * W + j] = (float)acc[r];
  }
}

// kSepR inputs m0 + m into kSepR outputs r, each by tap m0 + m - r of the n
// reversed taps t[0 .. n-1]. The first and the last inputs reach outputs whose
// tap lies outside: those terms are left out rather than multiplied by a zero
// tap, so an infinite input reaches the outputs of its window only.
__device__ __forceinline__ void sep_fma(double acc[kSepR], const double x[kSepR],
                                        const double* __restrict__ t, int m0, int n) {
  constexpr int R = kSepR;
  if (m0 >= R - 1 && m0 + R <= n) {
#pragma unroll
    for (int m = 0; m < R; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = fma(t[m0 + m - r], x[m], acc[r]);
  } else {
#pragma unroll
    for (int m = 0; m < R; ++m)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int e = m0 + m - r;
        const double a = fma(t[min(max(e, 0), n - 1)], x[m], acc[r]);
        acc[r] = e >= 0 && e < n ? a : acc[r];
      }
  }
}

// Column pass of an outer-product kernel: tmp[i, j] = sum_p c[p] src[i + oi - p, j]
// in double, kSepR outputs down a column per thread. Walking input rows
// m = 0 .. kh + kSepR - 2 from i0 + oi - (kh - 1), output r takes tap m - r of
// the reversed column: one coalesced load per row feeds kSepR multiply-adds
// with wave-uniform taps. Block b of (W + 63) / 64 across.
__device__ __forceinline__ void conv_cols(const float* __restrict__ src, int H, int W,
                                          const double* __restrict__ col, int kh,
                                          double* __restrict__ tmp, int b) {
  constexpr int R = kSepR;
  const int bx = (W + 63) / 64;
  const int j = b % bx * 64 + (threadIdx.x & 63);
  const int i0 = __builtin_amdgcn_readfirstlane((b / bx * 4 + (int)(threadIdx.x >> 6)) * R);
  if (i0 >= H) return;  // wave-uniform
  const uint32_t cb = (uint32_t)min(j, W - 1) * 4u;
  const int top = i0 + (kh - 1) / 2 - (kh - 1);
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  for (int m0 = 0; m0 < kh + R - 1; m0 += R) {
    double x[R];
#pragma unroll
    for (int m = 0; m < R; ++m) {
      const int i = top + m0 + m;
      const float f = ld(src + (size_t)min(max(i, 0), H - 1) * W, cb);
      x[m] = i >= 0 && i < H ? (double)f : 0.0;
    }
    sep_fma(acc, x, col, m0, kh);
  }
  if (j < W) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (i0 + r < H) tmp[(size_t)(i0 + r) * W + j] = acc[r];
  }
}

// Row pass: dst[i, j] = sum_q r[q] tmp[i, j + oj - q], rounded once. One wave
// per row segment of 64 kSepR outputs, kSepR adjacent outputs per lane; the
// segment is staged in LDS in spans of kSepSpan inputs (one double of padding
// per kSepR, so lanes kSepR apart fall on different banks), each input read
// once for kSepR multiply-adds. Together the passes take kh + kw
// multiply-adds per pixel instead of kh kw: at 1200 x 1200 with 120 x 120
// taps 47 us (26 + 21) in place of 1213 us (bounded by latency: 2850 and 3600
// waves over 1024 SIMDs, where the arithmetic alone is 9 us).
constexpr int kSepSeg = 64 * kSepR;
constexpr int kSepSpan = 256;

__device__ __forceinline__ void conv_rows(const double* __restrict__ tmp, int H, int W,
                                          const double* __restrict__ row, int kw,
                                          float* __restrict__ dst, int b) {
  constexpr int R = kSepR, N = kSepSeg + kSepSpan;
  __shared__ double s[4][N + N / R];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int bx = (H + 3) / 4;
  const int i = b % bx * 4 + wave, j0 = b / bx * kSepSeg;
  const int left = j0 + (kw - 1) / 2 - (kw - 1);  // column of input m = 0 of output j0
  const double* src = tmp + (size_t)min(i, H - 1) * W;
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.0;
  for (int m0 = 0; m0 < kw + R - 1; m0 += kSepSpan) {
    __syncthreads();  // the last span has been read
    for (int x = lane; x < N; x += 64) {
      const int j = left + m0 + x;
      s[wave][x + x / R] = j >= 0 && j < W ? src[j] : 0.0;
    }
    __syncthreads();
    const int end = min(kSepSpan, kw + R - 1 - m0);
    for (int b = 0; b < end; b += R) {
      double x[R];
#pragma unroll
      for (int m = 0; m < R; ++m) x[m] = s[wave][(R * lane + b) / R * (R + 1) + m];
      sep_fma(acc, x, row, m0 + b, kw);
    }
  }
  if (i < H) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = j0 + R * lane + r;
      if (j < W) dst[(size_t)i * W + j] = (float)acc[r];
    }
  }
}

// Either route's first launch (the column pass; the padded image) and second one
// (the row pass; the direct sum), each in the blocks it needs. With a launch for
// each, those not wanted cost 4 to 10 us a call: 12 x 12 taps at 128 x 128 take 14
// us as an outer product, 18 then.
__global__ void __launch_bounds__(256)
k_conv_first(const float* __restrict__ src, int H, int W, ConvPad pd,
             const double* __restrict__ col, int kh, float* __restrict__ pad,
             double* __restrict__ tmp, bool passes, int n_cols, int* __restrict__ flags) {
  if (!passes || !is_outer(flags))
    pad_image(src, H, W, pd, pad, flags + kConvFlags);
  else if ((int)blockIdx.x < n_cols)
    conv_cols(src, H, W, col, kh, tmp, blockIdx.x);
}

__global__ void __launch_bounds__(256)
k_conv_last(const float* __restrict__ pad, const double* __restrict__ tmp, int H, int W,
            ConvPad pd, const double* __restrict__ kt, const double* __restrict__ row, int kh,
            int kw, float* __restrict__ dst, bool passes, int n_rows, int n_direct,
            const int* __restrict__ flags) {
  const int b = blockIdx.x;
  if (passes && is_outer(flags)) {  // uniform over the block, as is b: conv_rows has barriers
    if (b < n_rows) conv_rows(tmp, H, W, row, kw, dst, b);
  } else if (b < n_direct) {
    if (flags[kConvFlags] == 0)
      convolve_same<true>(pad, H, W, pd, kt, kh, kw, dst, b);
    else
      convolve_same<false>(pad, H, W, pd, kt, kh, kw, dst, b);
  }
}

// The scar-to-diffusivity map of random_diffusivity (deepx/generate.py:79-83,
// deepx/utils_scars.py:426, cardiax/convert.py:23-26): c = 1 - scar, then
// (c - min c) (hi - lo) / (max c - min c) + lo, in double (1 - x is exact
// there for a float x in [0, 1]), rounded once. min and max in two passes
// (per-block partials, then a fixed-order scan of them): deterministic.
constexpr int kMmBlocks = 256;

__global__ void __launch_bounds__(256)
k_minmax_partial(const float* __restrict__ x, int64_t n, double* __restrict__ part) {
  __shared__ double lo[256], hi[256];
  double a = INFINITY, b = -INFINITY;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double c = 1.0 - (double)x[i];
    a = fmin(a, c);
    b = fmax(b, c);
  }
  lo[threadIdx.x] = a;
  hi[threadIdx.x] = b;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      lo[threadIdx.x] = fmin(lo[threadIdx.x], lo[threadIdx.x + o]);
      hi[threadIdx.x] = fmax(hi[threadIdx.x], hi[threadIdx.x + o]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = lo[0];
    part[2 * blockIdx.x + 1] = hi[0];
  }
}

__global__ void __launch_bounds__(256)
k_scar_rescale(const float* __restrict__ x, int64_t n, const double* __restrict__ part,
               int n_part, double lo_d, double hi_d, float* __restrict__ D) {
#pragma clang fp contract(off)
  // every block reduces the partials (one per thread) in the same tree
  static_assert(kMmBlocks <= 256, "one partial per thread");
  __shared__ double s_lo[256], s_hi[256];
  s_lo[threadIdx.x] = (int)threadIdx.x < n_part ? part[2 * threadIdx.x] : INFINITY;
  s_hi[threadIdx.x] = (int)threadIdx.x < n_part ? part[2 * threadIdx.x + 1] : -INFINITY;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s_lo[threadIdx.x] = fmin(s_lo[threadIdx.x], s_lo[threadIdx.x + o]);
      s_hi[threadIdx.x] = fmax(s_hi[threadIdx.x], s_hi[threadIdx.x + o]);
    }
    __syncthreads();
  }
  // the reference's order of operations: (c - a) * (z - y) / (b - a) + y
  const double a = s_lo[0], span = s_hi[0] - a, range = hi_d - lo_d;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    D[i] = (float)((1.0 - (double)x[i] - a) * range / span + lo_d);
}

}  // namespace fk

using namespace fk;

extern "C" {

int32_t fk_rasterize_polygons(float* mask, int32_t H, int32_t W, const double* rows,
                              const double* cols, const int32_t* starts, int32_t n_polys,
                              void* work, size_t work_bytes, void* stream) {
  ErrorScope es;
  if (mask == nullptr || H < 1 || W < 1)
    return set_error(FK_ERR_ARG, "fk_rasterize_polygons: null mask or empty image");
  if (n_polys < 0 || (n_polys > 0 && (!rows || !cols || !starts)))
    return set_error(FK_ERR_ARG, "fk_rasterize_polygons: bad polygon list");
  const int32_t n_verts = n_polys > 0 ? starts[n_polys] : 0;
  for (int p = 0; p < n_polys; ++p)
    if (starts[p + 1] - starts[p] < 3 || starts[p] < 0)
      return set_error(FK_ERR_ARG, "polygon %d has fewer than 3 vertices", p);
  const size_t need = fk_rasterize_workspace_bytes(n_polys, n_verts);
  if (n_polys > 0 && (work == nullptr || work_bytes < need))
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu", need,
                     work_bytes);
  hipStream_t s = (hipStream_t)stream;
  // vertices and bounding boxes to the device (from host arrays; the call
  // waits for the stream before it returns, so they may be released then)
  char* wk = (char*)work;
  double* d_r = (double*)wk;
  double* d_c = d_r + n_verts;
  PolyBox* d_box = (PolyBox*)(wk + ((2 * (size_t)n_verts * sizeof(double) + 255) / 256) * 256);
  std::vector<PolyBox> boxes((size_t)n_polys);
  for (int p = 0; p < n_polys; ++p) {
    double rmin = rows[starts[p]], rmax = rmin, cmin = cols[starts[p]], cmax = cmin;
    for (int k = starts[p]; k < starts[p + 1]; ++k) {
      if (!std::isfinite(rows[k]) || !std::isfinite(cols[k]))
        return set_error(FK_ERR_ARG, "polygon %d has a non-finite vertex", p);
      rmin = std::fmin(rmin, rows[k]);
      rmax = std::fmax(rmax, rows[k]);
      cmin = std::fmin(cmin, cols[k]);
      cmax = std::fmax(cmax, cols[k]);
    }
    // skimage.draw.polygon's box, limited to the image (pixels beyond it are dropped)
    PolyBox b;
    b.r0 = (int)std::fmax(0.0, rmin);
    b.r1 = (int)std::fmin((double)(H - 1), std::ceil(rmax));
    b.c0 = (int)std::fmax(0.0, cmin);
    b.c1 = (int)std::fmin((double)(W - 1), std::ceil(cmax));
    b.begin = starts[p];
    b.end = starts[p + 1];
    boxes[p] = b;
  }
  if (n_polys > 0) {
    HIP_CHECK(hipMemcpyAsync(d_r, rows, n_verts * sizeof(double), hipMemcpyHostToDevice, s));
    HIP_CHECK(hipMemcpyAsync(d_c, cols, n_verts * sizeof(double), hipMemcpyHostToDevice, s));
    HIP_CHECK(hipMemcpyAsync(d_box, boxes.data(), n_polys * sizeof(PolyBox),
                             hipMemcpyHostToDevice, s));
  }
  const dim3 grid((H + 3) / 4, std::min((W - 1) / kRasterCols + 1, 65535));
  k_raster_polygons<<<grid, 256, 0, s>>>(mask, H, W, d_r, d_c, d_box, n_polys);
  HIP_CHECK(hipGetLastError());
  // the host-side staging of boxes must outlive the copy
  HIP_CHECK(hipStreamSynchronize(s));
  return FK_OK;
}

int32_t fk_scar_to_diffusivity(const float* scar, int64_t n_cells, double lo, double hi,
                               float* D, void* work, size_t work_bytes, void* stream) {
  ErrorScope es;
  if (!check_ptrs({scar, D, work}) || n_cells < 1)
    return set_error(FK_ERR_ARG, "fk_scar_to_diffusivity: null pointer or empty field");
  if (!std::isfinite(lo) || !std::isfinite(hi))
    return set_error(FK_ERR_ARG, "the diffusivity range must be finite");
  if (work_bytes < 2 * kMmBlocks * sizeof(double))
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu",
                     2 * kMmBlocks * sizeof(double), work_bytes);
  hipStream_t s = (hipStream_t)stream;
  const int blocks = (int)std::min<int64_t>((n_cells + 255) / 256, kMmBlocks);
  k_minmax_partial<<<blocks, 256, 0, s>>>(scar, n_cells, (double*)work);
  k_scar_rescale<<<blocks, 256, 0, s>>>(scar, n_cells, (const double*)work, blocks, lo, hi, D);
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

size_t fk_rasterize_workspace_bytes(int32_t n_polys, int32_t n_vertices) {
  if (n_polys <= 0 || n_vertices <= 0) return 0;
  return ((2 * (size_t)n_vertices * sizeof(double) + 255) / 256) * 256 +
         (size_t)n_polys * sizeof(PolyBox);
}

size_t fk_convolve_workspace_bytes(int32_t H, int32_t W, int32_t kh, int32_t kw) {
  if (H < 1 || W < 1 || kh < 1 || kw < 1) return 0;
  return conv_work(H, W, kh, kw).total;
}

int32_t fk_convolve_same(const float* src, int32_t H, int32_t W, const double* kernel,
                         int32_t kh, int32_t kw, float* dst, void* work, size_t work_bytes,
                         void* stream) {
  ErrorScope es;
  if (!check_ptrs({src, kernel, dst, work})) return last_code();
  if (H < 1 || W < 1 || kh < 1 || kw < 1)
    return set_error(FK_ERR_ARG, "fk_convolve_same: empty image or kernel");
  if (kh > (1 << 16) || kw > (1 << 16) || H > (1 << 20) || W > (1 << 20))
    return set_error(FK_ERR_ARG, "fk_convolve_same: image %d x %d or kernel %d x %d too large",
                     H, W, kh, kw);
  if (src == dst) return set_error(FK_ERR_ARG, "fk_convolve_same: dst must not be src");
  const size_t need = fk_convolve_workspace_bytes(H, W, kh, kw);
  if (work_bytes < need)
    return set_error(FK_ERR_ARG, "workspace too small: need %zu bytes, got %zu", need,
                     work_bytes);
  hipStream_t s = (hipStream_t)stream;
  const ConvWork wo = conv_work(H, W, kh, kw);
  const ConvPad pd = conv_pad(H, W, kh, kw);
  char* wk = (char*)work;
  double *kt = (double*)wk, *col = (double*)(wk + wo.col), *row = (double*)(wk + wo.row);
  int* flags = (int*)(wk + wo.flag);
  float* pad = (float*)(wk + wo.image);
  double* tmp = (double*)(wk + wo.image);
  const bool passes = (int64_t)kw * ((kh + 2 * kConvRows - 2) / kConvRows) >= kMinPasses;
  k_conv_prepare<<<kConvFlags, 256, 0, s>>>(kernel, kh, kw, passes, kt, col, row, flags);
  // The host does not know the kernel's values: a launch holds both routes, by the
  // flags.
  const int64_t nc = (int64_t)((W + 63) / 64) * ((H + 4 * kSepR - 1) / (4 * kSepR));
  const int64_t np = std::min<int64_t>(((int64_t)pd.Hp * pd.Wp + 1023) / 1024, 4096);
  k_conv_first<<<(unsigned)std::max(nc, np), 256, 0, s>>>(src, H, W, pd, col, kh, pad, tmp, passes,
                                                          (int)nc, flags);
  const int64_t nr = (int64_t)((H + 3) / 4) * ((W + kSepSeg - 1) / kSepSeg);
  const int64_t nd = (int64_t)((W + 63) / 64) * ((H + 4 * kConvRows - 1) / (4 * kConvRows));
  k_conv_last<<<(unsigned)std::max(nr, nd), 256, 0, s>>>(pad, tmp, H, W, pd, kt, row, kh, kw, dst,
                                                         passes, (int)nr, (int)nd, flags);
  HIP_CHECK(hipGetLastError());
  return FK_OK;
}

}  // extern "C"
