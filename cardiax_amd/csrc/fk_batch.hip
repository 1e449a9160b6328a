// Batched forward Euler: many independent simulations of uneven sizes and
// parameter sets advanced together.
//
// One launch over a work list that holds every tile of every simulation
// advances the whole batch by one Euler step (streaming tiles, stream_tile) or
// by two to four (block tiles, block_tile, which read and write the state once
// for all of them); each tile takes its simulation's constants, D-map and
// stimuli from a device-resident descriptor. Stimulus activity follows the law of cardiax/solve.py:262-267
// (floor modulo in double precision, as on the host path), evaluated on the
// device by one small kernel for up to kGraphSteps steps at a time. Steps are
// recorded once into a hipGraph (that kernel, the step launches and a
// one-thread kernel that advances the device-side step counter) and the graph
// is replayed: the host issues one graph launch per graph_steps steps for the
// whole batch.
//
// Reference: the batch has no counterpart in the reference, which runs one
// simulation per call (experiments/generate_fd_data_128.py:25-56 loops over
// seeds); each simulation follows cardiax/solve.py:92-100.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "cardiax_amd.h"
#include "fk_batch.h"
#include "fk_device.h"
#include "fk_host.h"
#include "fk_stream.h"
#include "fk_stream_t.h"

namespace fk {

// Work-list options, chosen by fk_batch_autotune: one step per launch on bands
// of 2, 4, 8 or 16 rows, or several steps per launch on block tiles: of 32 rows
// (option 8 | FK_BATCH_TWO_STEP) or of 48 rows (16 | FK_BATCH_TWO_STEP). Block
// tiles cover every grid, but these two options are offered and accepted only
// for simulations of at least 2 R + 16 rows (R the option's number) and 56..96
// or >= 104 columns, the sizes they were first defined for. An untuned batch
// runs the block tiling that LeastRounds finds.
constexpr int kNumRowOpts = FK_BATCH_N_OPTIONS;
constexpr int kBatchRows[kNumRowOpts] = {2, 4, 8, 16, 8, 16};
constexpr bool kBatchTwo[kNumRowOpts] = {false, false, false, false, true, true};
constexpr int kGraphSteps = 32;  // Euler steps of one mask window; at most as many in a graph

// Block tiling of a batch option.
enum BatchBlock { kNone, kBatch32x4, kBatch32x2, kBatch48x3 };
constexpr int batch_steps(int blk) {
  return blk == kBatch32x4 ? 4 : blk == kBatch48x3 ? 3 : blk == kBatch32x2 ? 2 : 1;
}

struct SimDesc {
  Coef c;
  const float* D;
  float* buf[2][3];  // ping-pong state: [parity][v, w, u]
  float* user[3];    // the caller's state buffers
  int H, W;
  int n_stim;
  float dt, inv_dx2;
  double t0;  // time of the first step
  BatchStim stim[FK_BATCH_MAX_STIMULI];
};

struct TileItem {
  int sim, cs, rs, flags;  // flags: bit0 band near a row edge, bit1 strip near a column edge
};

// Stimulus activity of every simulation at the n_rel steps from the device
// step counter on: bit k of mask[r * n + i] = stimulus k of simulation i is
// active at step r of them.
__global__ void k_batch_masks(const SimDesc* __restrict__ sims, int n,
                              const int64_t* __restrict__ step_base, int n_rel,
                              uint32_t* __restrict__ mask) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n * n_rel) return;
  const int i = idx % n, r = idx / n;
  const SimDesc& S = sims[i];
  const double t = S.t0 + (double)(*step_base + r);
  uint32_t m = 0;
  for (int k = 0; k < S.n_stim; ++k)
    if (active_dev(t, S.stim[k])) m |= 1u << k;
  mask[idx] = m;
}

// One Euler step of every tile (bands of R rows). Reads state[parity],
// writes state[parity ^ 1].
template <int R>
__global__ void __launch_bounds__(256)
k_batch_step(const SimDesc* __restrict__ sims, const TileItem* __restrict__ items, int n_items,
             const uint32_t* __restrict__ masks, int parity) {
  const int it = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x >> 6));
  if (it >= n_items) return;
  // wave-uniform work item (scalar registers)
  TileItem item = items[it];
  item.sim = __builtin_amdgcn_readfirstlane(item.sim);
  item.cs = __builtin_amdgcn_readfirstlane(item.cs);
  item.rs = __builtin_amdgcn_readfirstlane(item.rs);
  item.flags = __builtin_amdgcn_readfirstlane(item.flags);
  const SimDesc& S = sims[item.sim];
  const uint32_t mask = __builtin_amdgcn_readfirstlane(masks[item.sim]);
  const BatchStimView sv{S.stim, uni(S.n_stim), mask};
  Coef c = S.c;
  c.V_c = uni(c.V_c); c.V_v = uni(c.V_v); c.V_csi = uni(c.V_csi); c.kk = uni(c.kk);
  c.kk_off = uni(c.kk_off);
  c.inv_tvp = uni(c.inv_tvp); c.inv_tv1m = uni(c.inv_tv1m); c.inv_tv2m = uni(c.inv_tv2m);
  c.inv_twp = uni(c.inv_twp); c.inv_twm = uni(c.inv_twm); c.inv_td = uni(c.inv_td);
  c.inv_t0 = uni(c.inv_t0); c.inv_tr = uni(c.inv_tr); c.inv_tsi = uni(c.inv_tsi);
  c.inv_cm = uni(c.inv_cm);
  const float* Dp = uni(S.D);
  const float* i0 = uni(S.buf[parity][0]);
  const float* i1 = uni(S.buf[parity][1]);
  const float* i2 = uni(S.buf[parity][2]);
  float* o0 = uni(S.buf[parity ^ 1][0]);
  float* o1 = uni(S.buf[parity ^ 1][1]);
  float* o2 = uni(S.buf[parity ^ 1][2]);
  const int H = uni(S.H), W = uni(S.W);
  const float dt = uni(S.dt), inv_dx2 = uni(S.inv_dx2);
  const int sel = item.flags | (mask ? 4 : 0);
#define FK_BT(X, Y, ST)                                                                    \
  stream_tile<R, true, X, Y, ST, BatchStimView, false, true>(c, Dp, nullptr, i0, i1, i2, H, W,  \
                                                                sv, dt, inv_dx2, o0, o1, o2,      \
                                                                item.rs, item.cs)
  switch (sel) {
    case 0: FK_BT(false, false, false); break;
    case 1: FK_BT(true, false, false); break;
    case 2: FK_BT(false, true, false); break;
    case 3: FK_BT(true, true, false); break;
    case 4: FK_BT(false, false, true); break;
    case 5: FK_BT(true, false, true); break;
    case 6: FK_BT(false, true, true); break;
    default: FK_BT(true, true, true); break;
  }
#undef FK_BT
}

// n_lev Euler steps of every block tile. Reads state[parity], writes
// state[parity ^ 1]; masks holds the activity of the steps, n_sims words each.
template <class Cfg>
__global__ void __launch_bounds__(Cfg::waves * 64)
k_batch_block(const SimDesc* __restrict__ sims, const BlockItem* __restrict__ items, int n_sims,
              const uint32_t* __restrict__ masks, int n_lev, int parity) {
  __shared__ float lds[Cfg::lds_floats];
  // each XCD's run forward and backward in turn, as in BlockOrder
  const int x = blockIdx.x % kXcds, j = blockIdx.x / kXcds;
  const BlockItem& it = items[kXcds * (parity ? (int)gridDim.x / kXcds - 1 - j : j) + x];
  const int sim = uni(it.sim);
  if (sim < 0) return;  // padding of the XCD order: the whole block leaves
  const SimDesc& S = sims[sim];
  const BatchBlockStim sv{S.stim, pack_masks(masks + sim, n_sims, n_lev)};
  Coef c = S.c;
  c.V_c = uni(c.V_c); c.V_v = uni(c.V_v); c.V_csi = uni(c.V_csi); c.kk = uni(c.kk);
  c.kk_off = uni(c.kk_off);
  c.inv_tvp = uni(c.inv_tvp); c.inv_tv1m = uni(c.inv_tv1m); c.inv_tv2m = uni(c.inv_tv2m);
  c.inv_twp = uni(c.inv_twp); c.inv_twm = uni(c.inv_twm); c.inv_td = uni(c.inv_td);
  c.inv_t0 = uni(c.inv_t0); c.inv_tr = uni(c.inv_tr); c.inv_tsi = uni(c.inv_tsi);
  c.inv_cm = uni(c.inv_cm);
  const BlockIO io{uni(S.D), uni(S.buf[parity][0]), uni(S.buf[parity][1]),
                   uni(S.buf[parity][2]), uni(S.buf[parity ^ 1][0]), uni(S.buf[parity ^ 1][1]),
                   uni(S.buf[parity ^ 1][2]), 0, false};
  const BlockSpan r{uni(it.r.o), uni(it.r.a), uni(it.r.b)};
  const BlockSpan q{uni(it.c.o), uni(it.c.a), uni(it.c.b)};
  block_tile_any<Cfg, false>(c, io, uni(S.H), uni(S.W), sv, n_lev, uni(S.dt), uni(S.inv_dx2), r,
                             q, lds);
}

// n floats from src to dst, blocks [blk, blk + stride, ...) of 1024: 16-byte
// moves where both pointers allow them.
__device__ __forceinline__ void copy_cells(float* __restrict__ dst, const float* __restrict__ src,
                                           size_t n, size_t blk, size_t stride) {
  const bool wide = (((uintptr_t)dst | (uintptr_t)src) & 15) == 0;
  const size_t n4 = wide ? n / 4 : 0;
  for (size_t i = blk * 256 + threadIdx.x; i < n4; i += stride * 256)
    ((float4*)dst)[i] = ((const float4*)src)[i];
  for (size_t i = 4 * n4 + blk * 256 + threadIdx.x; i < n; i += stride * 256) dst[i] = src[i];
}

// The whole batch's state between the callers' buffers and a pool, one launch
// in place of one copy per field (768 copies of 2.4 us for 256 simulations,
// 1.85 ms; 26.1 M cells now take 0.15 ms). blockIdx.y strides over the
// fields: LOAD callers -> pool 0 and resets the step counter; else pool
// `parity` -> callers and moves every simulation's time on by n_steps.

template <bool LOAD>
__global__ void __launch_bounds__(256)
k_batch_copy(SimDesc* __restrict__ sims, int n, int parity, int64_t* __restrict__ step_base,
             int64_t n_steps) {
  for (int64_t y = blockIdx.y; y < 3 * (int64_t)n; y += gridDim.y) {
    SimDesc& S = sims[y / 3];
    const int f = (int)(y % 3);
    const size_t cells = (size_t)S.H * S.W;
    if (LOAD)
      copy_cells(S.buf[0][f], S.user[f], cells, blockIdx.x, gridDim.x);
    else
      copy_cells(S.user[f], S.buf[parity][f], cells, blockIdx.x, gridDim.x);
    if (!LOAD && f == 0 && blockIdx.x == 0 && threadIdx.x == 0) S.t0 += (double)n_steps;
  }
  if (LOAD && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *step_base = 0;
}

__global__ void k_batch_bump(int64_t* step_base, int64_t by) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *step_base += by;
}

__global__ void k_batch_set(int64_t* step_base, int64_t value) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *step_base = value;
}

}  // namespace fk

using namespace fk;

// Opaque batch handle.
struct fk_batch {
  int n_sims = 0;
  int opt = 0, untuned = 0;        // index into kBatchRows: in use, until tuned
  int block[kNumRowOpts] = {};     // BatchBlock of the option
  bool offered[kNumRowOpts] = {};  // accepted by fk_batch_set_rows
  int n_items_opt[kNumRowOpts] = {};
  std::vector<fk_sim> host_sims;   // caller's descriptors (state pointers)
  std::vector<size_t> offset;      // per-sim cell offset in the pools
  size_t total_cells = 0;
  int copy_blocks = 0;             // blocks per field of k_batch_copy
  char* dev = nullptr;             // one allocation: descriptors, items, counter, pools
  SimDesc* d_sims = nullptr;
  char* d_items[kNumRowOpts] = {};  // TileItem (one step) or BlockItem
  int64_t* d_step = nullptr;
  uint32_t* d_mask = nullptr;  // stimulus activity: kGraphSteps x n_sims
  float* pool[2] = {nullptr, nullptr};  // ping-pong pools of 3 * total_cells floats
  hipStream_t cap = nullptr;            // private stream used for graph capture
  hipGraphExec_t exec[2] = {nullptr, nullptr};  // per starting parity
};

static int32_t batch_check_sim(const fk_sim& s, int i) {
  if (!check_params(&s.params) || !check_grid(s.H, s.W) ||
      !check_ptrs({s.D, s.v, s.w, s.u}) || !check_time(s.t, s.t) ||
      !check_scalar("dt", s.dt) || !check_dx(s.dx))
    return set_error(last_code(), "simulation %d: %s", i, fk_last_error());
  if (s.n_stimuli < 0 || s.n_stimuli > FK_BATCH_MAX_STIMULI)
    return set_error(FK_ERR_UNSUPPORTED, "simulation %d: %d stimuli, the batch limit is %d", i,
                     s.n_stimuli, FK_BATCH_MAX_STIMULI);
  if (!check_stimuli(s.stimuli, s.n_stimuli))
    return set_error(last_code(), "simulation %d: %s", i, fk_last_error());
  return FK_OK;
}

static void batch_free(fk_batch* b) {
  if (!b) return;
  for (auto& e : b->exec)
    if (e) (void)hipGraphExecDestroy(e);
  if (b->cap) (void)hipStreamDestroy(b->cap);
  if (b->dev) (void)hipFree(b->dev);
  delete b;
}

extern "C" {

int32_t fk_batch_create(const fk_sim* sims, int32_t n, fk_batch** out) {
  ErrorScope es;
  if (out == nullptr) return set_error(FK_ERR_ARG, "out is null");
  *out = nullptr;
  if (n <= 0 || sims == nullptr) return set_error(FK_ERR_ARG, "empty batch");
  for (int i = 0; i < n; ++i) {
    const int32_t rc = batch_check_sim(sims[i], i);
    if (rc != FK_OK) return rc;
  }
  fk_batch* b = new fk_batch();
  b->n_sims = n;
  b->host_sims.assign(sims, sims + n);
  std::vector<TileItem> items[kNumRowOpts];
  std::vector<BlockItem> tiles[kNumRowOpts];
  b->offset.resize(n);
  int64_t n32x4 = 0, n32x2 = 0, n48x3 = 0;
  bool fit[2] = {true, true};
  for (int i = 0; i < n; ++i) {
    const fk_sim& s = sims[i];
    b->offset[i] = b->total_cells;
    b->total_cells += (size_t)s.H * s.W;
    n32x4 += block_tiles<Block32x4>(s.H, s.W);
    n32x2 += block_tiles<Block32x2>(s.H, s.W);
    n48x3 += block_tiles<Block48x3>(s.H, s.W);
    fit[0] = fit[0] && stream_t_fits<8>(s.H, s.W);
    fit[1] = fit[1] && stream_t_fits<16>(s.H, s.W);
    for (int o = 0; o < kNumRowOpts; ++o) {
      if (kBatchTwo[o]) continue;
      const int R = kBatchRows[o];
      const StreamGeom g = o == 0   ? make_stream_geom<kBatchRows[0]>(s.H, s.W)
                           : o == 1 ? make_stream_geom<kBatchRows[1]>(s.H, s.W)
                           : o == 2 ? make_stream_geom<kBatchRows[2]>(s.H, s.W)
                                    : make_stream_geom<kBatchRows[3]>(s.H, s.W);
      for (int strip = 0; strip < g.n_strips; ++strip)
        for (int band = 0; band < g.n_bands; ++band) {
          TileItem t;
          t.sim = i;
          t.cs = std::min(kStripOut * strip, g.cs_last);
          t.rs = std::min(R * band, g.rs_last);
          const bool xg = edge_band(t.rs, R, s.H, s.W);
          const bool yg = t.cs < 3 || t.cs + kStripOut + 3 > s.W;
          t.flags = (xg ? 1 : 0) | (yg ? 2 : 0);
          items[o].push_back(t);
        }
    }
  }
  // blocks of a field's copy: 4096 cells each in the largest simulation, 16 at least,
  // about 2^16 in all. With 16 whatever the sizes, one step of a batch of one 4096^2
  // simulation took 1130 us (290 so), of one 2048^2 180 (60).
  size_t largest = 0;
  for (int i = 0; i < n; ++i) largest = std::max(largest, (size_t)sims[i].H * sims[i].W);
  b->copy_blocks =
      (int)std::max<size_t>(16, std::min<size_t>(largest / 4096, 65536 / (3 * (size_t)n)));
  // 32 rows: 4 steps per launch for batches of few tiles, else 2
  LeastRounds by32((int64_t)b->total_cells), least((int64_t)b->total_cells);
  by32.offer(kBatch32x4, Block32x4{}, n32x4);
  by32.offer(kBatch32x2, Block32x2{}, n32x2);
  b->block[4] = by32.best;
  b->block[5] = kBatch48x3;
  least.offer(4, Block32x4{}, n32x4);
  least.offer(4, Block32x2{}, n32x2);
  least.offer(5, Block48x3{}, n48x3);
  b->untuned = b->opt = least.best;
  for (int o = 0; o < kNumRowOpts; ++o) {
    b->offered[o] = !kBatchTwo[o] || fit[o - 4];
    if (!kBatchTwo[o]) continue;
    for (int i = 0; i < n; ++i) {
      const int H = sims[i].H, W = sims[i].W;
      switch (b->block[o]) {
        case kBatch32x4: append_block_items<Block32x4>(i, H, W, tiles[o]); break;
        case kBatch32x2: append_block_items<Block32x2>(i, H, W, tiles[o]); break;
        default: append_block_items<Block48x3>(i, H, W, tiles[o]); break;
      }
    }
    tiles[o] = block_work_list(tiles[o]);
  }
  size_t sz_it[kNumRowOpts], sz_items = 0;
  for (int o = 0; o < kNumRowOpts; ++o) {
    b->n_items_opt[o] = (int)(kBatchTwo[o] ? tiles[o].size() : items[o].size());
    const size_t bytes =
        kBatchTwo[o] ? sizeof(BlockItem) * tiles[o].size() : sizeof(TileItem) * items[o].size();
    sz_it[o] = ((bytes + 255) / 256) * 256;
    sz_items += sz_it[o];
  }
  const size_t sz_sims = ((sizeof(SimDesc) * n + 255) / 256) * 256;
  const size_t sz_pool = 3 * b->total_cells * sizeof(float);
  const size_t sz_mask = ((sizeof(uint32_t) * n * kGraphSteps + 255) / 256) * 256;
  const size_t total = sz_sims + sz_items + 256 + sz_mask + 2 * sz_pool;
  hipError_t e = hipMalloc((void**)&b->dev, total);
  if (e != hipSuccess) {
    batch_free(b);
    return set_error(FK_ERR_HIP, "hipMalloc(%zu) failed: %s", total, hipGetErrorString(e));
  }
  b->d_sims = (SimDesc*)b->dev;
  {
    size_t at = sz_sims;
    for (int o = 0; o < kNumRowOpts; ++o) {
      b->d_items[o] = b->dev + at;
      at += sz_it[o];
    }
  }
  b->d_step = (int64_t*)(b->dev + sz_sims + sz_items);
  b->d_mask = (uint32_t*)(b->dev + sz_sims + sz_items + 256);
  b->pool[0] = (float*)(b->dev + sz_sims + sz_items + 256 + sz_mask);
  b->pool[1] = b->pool[0] + 3 * b->total_cells;
  std::vector<SimDesc> desc(n);
  for (int i = 0; i < n; ++i) {
    const fk_sim& s = sims[i];
    SimDesc& d = desc[i];
    std::memset(&d, 0, sizeof d);
    d.c = make_coef(s.params);
    d.D = s.D;
    const size_t cells = (size_t)s.H * s.W;
    for (int p = 0; p < 2; ++p)
      for (int f = 0; f < 3; ++f) d.buf[p][f] = b->pool[p] + 3 * b->offset[i] + f * cells;
    d.user[0] = s.v;
    d.user[1] = s.w;
    d.user[2] = s.u;
    d.H = s.H;
    d.W = s.W;
    d.n_stim = s.n_stimuli;
    d.dt = s.dt;
    d.inv_dx2 = (float)(1.0 / ((double)s.dx * (double)s.dx));
    d.t0 = s.t;
    for (int k = 0; k < s.n_stimuli; ++k)
      d.stim[k] = {s.stimuli[k].start, s.stimuli[k].duration, s.stimuli[k].period,
                   s.stimuli[k].field};
  }
  e = hipMemcpy(b->d_sims, desc.data(), sizeof(SimDesc) * n, hipMemcpyHostToDevice);
  for (int o = 0; o < kNumRowOpts && e == hipSuccess; ++o)
    e = kBatchTwo[o] ? hipMemcpy(b->d_items[o], tiles[o].data(),
                                 sizeof(BlockItem) * tiles[o].size(), hipMemcpyHostToDevice)
                     : hipMemcpy(b->d_items[o], items[o].data(),
                                 sizeof(TileItem) * items[o].size(), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking);
  if (e != hipSuccess) {
    batch_free(b);
    return set_error(FK_ERR_HIP, "batch setup failed: %s", hipGetErrorString(e));
  }
  *out = b;
  return FK_OK;
}

int32_t fk_batch_destroy(fk_batch* b) {
  ErrorScope es;
  if (b == nullptr) return FK_OK;
  HIP_CHECK(hipDeviceSynchronize());
  batch_free(b);
  return FK_OK;
}

int32_t fk_batch_n_items(const fk_batch* b) { return b ? b->n_items_opt[b->opt] : 0; }

int32_t fk_batch_option(const fk_batch* b, int32_t* steps_per_launch) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "batch is null");
  if (steps_per_launch) *steps_per_launch = batch_steps(b->block[b->opt]);
  return kBatchRows[b->opt] | (kBatchTwo[b->opt] ? FK_BATCH_TWO_STEP : 0);
}

// Stimulus masks of the next n_rel (<= kGraphSteps) steps from the counter.
static hipError_t batch_masks(fk_batch* b, int n_rel, hipStream_t s) {
  const int total = b->n_sims * n_rel;
  k_batch_masks<<<(total + 255) / 256, 256, 0, s>>>(b->d_sims, b->n_sims, b->d_step, n_rel,
                                                    b->d_mask);
  return hipGetLastError();
}

// One launch of option o, n_lev steps from step rel of the current mask window
// on (its masks computed). Reads pool[parity], writes pool[parity ^ 1].
static hipError_t batch_launch(fk_batch* b, int o, int n_lev, int rel, int parity,
                               hipStream_t s) {
  const int n_items = b->n_items_opt[o], n = b->n_sims;
  const int blocks = (n_items + 3) / 4;
  const TileItem* it = (const TileItem*)b->d_items[o];
  const BlockItem* bi = (const BlockItem*)b->d_items[o];
  const uint32_t* m = b->d_mask + (size_t)rel * n;
  auto block = [&](auto cfg) {
    typedef decltype(cfg) Cfg;
    k_batch_block<Cfg><<<n_items, Cfg::waves * 64, 0, s>>>(b->d_sims, bi, n, m, n_lev, parity);
  };
  switch (b->block[o]) {
    case kBatch32x4: block(Block32x4{}); return hipGetLastError();
    case kBatch32x2: block(Block32x2{}); return hipGetLastError();
    case kBatch48x3: block(Block48x3{}); return hipGetLastError();
    default: break;
  }
  switch (o) {
    case 0: k_batch_step<kBatchRows[0]><<<blocks, 256, 0, s>>>(b->d_sims, it, n_items, m, parity); break;
    case 1: k_batch_step<kBatchRows[1]><<<blocks, 256, 0, s>>>(b->d_sims, it, n_items, m, parity); break;
    case 2: k_batch_step<kBatchRows[2]><<<blocks, 256, 0, s>>>(b->d_sims, it, n_items, m, parity); break;
    default: k_batch_step<kBatchRows[3]><<<blocks, 256, 0, s>>>(b->d_sims, it, n_items, m, parity); break;
  }
  return hipGetLastError();
}

// n (<= kGraphSteps) steps of option o from the counter on: their masks, the
// step launches and the counter bump. Starts at pool[*parity] and leaves the
// pool of the result in *parity.
static hipError_t batch_chunk(fk_batch* b, int o, int n, int* parity, hipStream_t s) {
  hipError_t e = batch_masks(b, n, s);
  const int per = batch_steps(b->block[o]);
  for (int r = 0; r < n && e == hipSuccess; r += per) {
    e = batch_launch(b, o, std::min(per, n - r), r, *parity, s);
    *parity ^= 1;
  }
  if (e == hipSuccess) {
    k_batch_bump<<<1, 64, 0, s>>>(b->d_step, n);
    e = hipGetLastError();
  }
  return e;
}

// Steps of a recorded graph of option o: whole launches.
static int graph_steps(const fk_batch* b, int o) {
  const int per = batch_steps(b->block[o]);
  return kGraphSteps / per * per;
}

// Records a chunk of graph_steps steps starting at `parity`.
static hipError_t batch_build_graph(fk_batch* b, int parity) {
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamBeginCapture(b->cap, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) return e;
  int p = parity;
  e = batch_chunk(b, b->opt, graph_steps(b, b->opt), &p, b->cap);
  const hipError_t e2 = hipStreamEndCapture(b->cap, &g);
  if (e == hipSuccess) e = e2;
  if (e == hipSuccess) e = hipGraphInstantiate(&b->exec[parity], g, nullptr, nullptr, 0);
  if (g) (void)hipGraphDestroy(g);
  return e;
}

int32_t fk_batch_autotune(fk_batch* b, int32_t n_steps, void* stream, float* times_ms,
                          int32_t* best_rows) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "batch is null");
  if (n_steps < 1 || n_steps > 10000)
    return set_error(FK_ERR_ARG, "n_steps must be in [1, 10000], got %d", n_steps);
  hipStream_t s = (hipStream_t)stream;
  // Queued runs may still replay this batch's graphs or use its pools.
  HIP_CHECK(hipDeviceSynchronize());
  // The pools are scratch between runs (fk_batch_run copies the state in),
  // so timing may overwrite them; the step counter is reset by every run.
  hipEvent_t e0 = nullptr, e1 = nullptr;
  hipError_t e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  float ms[kNumRowOpts];
  for (int o = 0; o < kNumRowOpts; ++o) ms[o] = -1.0f;
  const int untuned = b->untuned;
  for (int o = 0; o < kNumRowOpts && e == hipSuccess; ++o) {
    if (!b->offered[o] && o != untuned) continue;
    int parity = 0;
    k_batch_set<<<1, 64, 0, s>>>(b->d_step, 0);
    e = batch_chunk(b, o, 4, &parity, s);  // warm-up
    if (e == hipSuccess) e = hipEventRecord(e0, s);
    const int chunk = graph_steps(b, o);
    for (int k = 0; k < n_steps && e == hipSuccess; k += chunk)
      e = batch_chunk(b, o, std::min(chunk, n_steps - k), &parity, s);
    if (e == hipSuccess) e = hipEventRecord(e1, s);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms[o], e0, e1);
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  int best = untuned, best_offered = 0;
  if (e == hipSuccess)
    for (int o = 0; o < kNumRowOpts; ++o) {
      if (ms[o] < 0.0f) continue;
      if (ms[o] < ms[best]) best = o;
      if (b->offered[o] && ms[o] < ms[best_offered]) best_offered = o;
    }
  b->opt = best;
  // graphs recorded for another work list are stale
  for (auto& x : b->exec)
    if (x) {
      (void)hipGraphExecDestroy(x);
      x = nullptr;
    }
  if (e != hipSuccess) return set_error(FK_ERR_HIP, "batch autotune failed: %s",
                                        hipGetErrorString(e));
  if (times_ms)
    for (int o = 0; o < kNumRowOpts; ++o) times_ms[o] = b->offered[o] ? ms[o] : -1.0f;
  if (best_rows)
    *best_rows = kBatchRows[best_offered] | (kBatchTwo[best_offered] ? FK_BATCH_TWO_STEP : 0);
  return FK_OK;
}

int32_t fk_batch_set_rows(fk_batch* b, int32_t rows) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "batch is null");
  int o = -1;
  const bool two = (rows & FK_BATCH_TWO_STEP) != 0;
  for (int k = 0; k < kNumRowOpts; ++k)
    if ((rows & ~FK_BATCH_TWO_STEP) == kBatchRows[k] && two == kBatchTwo[k]) o = k;
  if (o < 0)
    return set_error(FK_ERR_ARG,
                     "band height must be 2, 4, 8 or 16, or 8 or 16 with FK_BATCH_TWO_STEP, "
                     "got %d", rows);
  if (!b->offered[o])
    return set_error(FK_ERR_UNSUPPORTED,
                     "two steps per launch need every simulation of at least 2R + 16 rows "
                     "and 56..96 or >= 104 columns");
  if (o != b->opt) {
    HIP_CHECK(hipDeviceSynchronize());  // no queued launch may still use the old list
    for (auto& x : b->exec)
      if (x) {
        (void)hipGraphExecDestroy(x);
        x = nullptr;
      }
    b->opt = o;
  }
  return FK_OK;
}

int32_t fk_batch_run(fk_batch* b, int64_t n_steps, int32_t use_graph, void* stream) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "batch is null");
  if (n_steps < 0) return set_error(FK_ERR_ARG, "negative step count");
  for (int i = 0; i < b->n_sims; ++i)
    if (!check_time(b->host_sims[i].t, b->host_sims[i].t + (double)n_steps)) return last_code();
  hipStream_t s = (hipStream_t)stream;
  const dim3 cg(b->copy_blocks, (unsigned)std::min<int64_t>(3 * (int64_t)b->n_sims, 65535));
  k_batch_copy<true><<<cg, 256, 0, s>>>(b->d_sims, b->n_sims, 0, b->d_step, 0);
  HIP_CHECK(hipGetLastError());
  int64_t k = 0;
  int parity = 0;
  if (use_graph) {
    const int chunk = graph_steps(b, b->opt);
    const int flips = chunk / batch_steps(b->block[b->opt]) & 1;
    while (n_steps - k >= chunk) {
      if (!b->exec[parity]) HIP_CHECK(batch_build_graph(b, parity));
      HIP_CHECK(hipGraphLaunch(b->exec[parity], s));
      k += chunk;
      parity ^= flips;
    }
  }
  // the remainder (or everything without graphs): direct launches
  while (k < n_steps) {
    const int n = (int)std::min<int64_t>(kGraphSteps, n_steps - k);
    HIP_CHECK(batch_chunk(b, b->opt, n, &parity, s));
    k += n;
  }
  k_batch_copy<false><<<cg, 256, 0, s>>>(b->d_sims, b->n_sims, parity, b->d_step, n_steps);
  HIP_CHECK(hipGetLastError());
  // the simulations' times advance by n_steps for a later run
  for (auto& sm : b->host_sims) sm.t += (double)n_steps;
  return FK_OK;
}

}  // extern "C"
