// Batched rollout and its adjoint: the frame-producing forward solve of many
// independent problems and the checkpointed reverse pass of their frame loss,
// advanced together, one launch per Euler step (and per reverse step) for all
// of them.
//
// Each problem is the forward-Euler solve of cardiax/solve.py:92-100 from its
// own initial state, D-map, parameters and stimuli, with u sampled every
// `frame_every` steps; the reverse pass is the adjoint of fk_adjoint.hip.
// Per problem the schedule is the one the per-grid path runs (adjoint.py
// with fk_forward_trajectory and fk_adjoint_segment): checkpoints every S
// steps; for each segment, in reverse, the states are recomputed from its
// checkpoint and the steps are reversed one by one, frame cotangents entering
// lam_u at the frame steps. Every launch covers all problems through a work
// list (forward steps a block per block tile, two to four steps, or a wave per
// streaming tile for a single one; reverse steps a wave per tile), and the tiles
// run the same device code as the per-grid kernels: the results are bitwise those
// of the per-grid path.
//
// Reference: there is no counterpart in the reference, whose inverse problem
// is learnt by a network (deepx); the forward step follows
// cardiax/solve.py:26-100 and the loss is the frame MSE of the inverse
// problem built on it.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "cardiax_amd.h"
#include "fk_adjoint.h"
#include "fk_batch.h"
#include "fk_device.h"
#include "fk_host.h"
#include "fk_stream.h"

namespace fk {

__device__ __forceinline__ Coef uni(const Coef& a) {
  Coef c = a;
  c.V_c = uni(c.V_c); c.V_v = uni(c.V_v); c.V_csi = uni(c.V_csi); c.kk = uni(c.kk);
  c.kk_off = uni(c.kk_off);
  c.inv_tvp = uni(c.inv_tvp); c.inv_tv1m = uni(c.inv_tv1m); c.inv_tv2m = uni(c.inv_tv2m);
  c.inv_twp = uni(c.inv_twp); c.inv_twm = uni(c.inv_twm); c.inv_td = uni(c.inv_td);
  c.inv_t0 = uni(c.inv_t0); c.inv_tr = uni(c.inv_tr); c.inv_tsi = uni(c.inv_tsi);
  c.inv_cm = uni(c.inv_cm);
  return c;
}

// Block tiling of the forward steps.
enum RollBlock { kRoll32x4, kRoll48x3, kRoll32x2 };
constexpr int roll_steps(int blk) { return blk == kRoll32x4 ? 4 : blk == kRoll48x3 ? 3 : 2; }

struct RollDesc {
  Coef c;
  int H, W;
  float dt, inv_dx2;
  size_t cells;
  const float* D;
  const float* x0[3];  // initial state (the caller's)
  float* ckpt;         // x_S, x_2S, ...: 3 planes each
  float* traj;         // one segment's states after its start: 3 planes each
  float* frames;       // forward output, one plane per frame
  const float* g_frames;  // backward input, one plane per frame
  float* gD;           // backward output
  float* lam;          // cotangent (v, w, u planes) at segment boundaries
  float* lam_alt;      // its ping-pong partner
  const AdjAxisTab* tab;
  double* part;        // tau accumulators
  int n_stim;
  BatchStim stim[FK_BATCH_MAX_STIMULI];
};

struct RollTile {
  int sim, cs, rs, flags;  // flags: bit0 band near a row edge, bit1 strip near a column edge
};

// A pointer field of a descriptor, read as a global-memory pointer. Pointers
// read from memory are generic, and the tile bodies index them directly, so
// without this they compile to flat loads (which also wait on the LDS
// counter). The field's bits are loaded as an address-space-1 pointer and
// then converted, which lets the compiler keep every access global. Every
// field lives in device memory.
template <class T>
__device__ __forceinline__ T* gfield(T* const& f) {
  typedef T __attribute__((address_space(1)))* GT;
  GT g;
  __builtin_memcpy(&g, &f, sizeof g);
  return (T*)g;
}

// State x_{c + k} of segment `seg` (c = seg S): the checkpoint at k = 0, else
// slot k - 1 of the segment's trajectory. Plane f: 0 v, 1 w, 2 u.
__device__ __forceinline__ const float* roll_state(const RollDesc& S, int seg, int k, int f) {
  if (k == 0)
    return seg == 0 ? gfield(S.x0[f]) : gfield(S.ckpt) + ((size_t)(seg - 1) * 3 + f) * S.cells;
  return gfield(S.traj) + ((size_t)(k - 1) * 3 + f) * S.cells;
}

// n_lev Euler steps of every block tile: x_{c+k} -> trajectory slots k ..
// k + n_lev - 1. masks: the steps' stimulus activity, n words each.
template <class Cfg>
__global__ void __launch_bounds__(Cfg::waves * 64)
k_roll_block(const RollDesc* __restrict__ sims, const BlockItem* __restrict__ items, int n,
             const uint32_t* __restrict__ masks, int seg, int k, int n_lev) {
  __shared__ float lds[Cfg::lds_floats];
  const BlockItem& it = items[blockIdx.x];
  const int sim = uni(it.sim);
  if (sim < 0) return;  // padding of the XCD order: the whole block leaves
  const RollDesc& S = sims[sim];
  const BatchBlockStim sv{S.stim, pack_masks(masks + sim, n, n_lev)};
  const Coef c = uni(S.c);
  const size_t cells = S.cells;
  float* out = uni(S.traj + (size_t)k * 3 * cells);
  const BlockIO io{uni(S.D), uni(roll_state(S, seg, k, 0)), uni(roll_state(S, seg, k, 1)),
                   uni(roll_state(S, seg, k, 2)), out, out + cells, out + 2 * cells, 3 * cells,
                   true};
  const BlockSpan r{uni(it.r.o), uni(it.r.a), uni(it.r.b)};
  const BlockSpan q{uni(it.c.o), uni(it.c.a), uni(it.c.b)};
  block_tile_any<Cfg, false>(c, io, uni(S.H), uni(S.W), sv, n_lev, uni(S.dt), uni(S.inv_dx2), r,
                             q, lds);
}

// One Euler step: x_{c+k} -> trajectory slot k, on streaming tiles of kRollRows
// rows, a wave each: the step that whole launches of the block tiles leave over, and
// every step of segments of one. A block tile's halo is made for several steps.
// Forward, us per step with segments of one and of three, on block tiles only and
// so: 1.05 M cells 18.6 and 11.2, 17.2 and 10.3; 3.1 M cells 38.9 and 24.5, 35.0
// and 22.9.
constexpr int kRollRows = 4;

__global__ void __launch_bounds__(256)
k_roll_step(const RollDesc* __restrict__ sims, const RollTile* __restrict__ items, int n_items,
            const uint32_t* __restrict__ masks, int seg, int k) {
  constexpr int R = kRollRows;
  const int it = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x >> 6));
  if (it >= n_items) return;
  const RollTile item = items[it];
  const int sim = uni(item.sim), rs = uni(item.rs), cs = uni(item.cs);
  if (sim < 0) return;  // padding of the XCD order
  const RollDesc& S = sims[sim];
  const uint32_t mask = (uint32_t)uni((int)masks[sim]);
  const BatchStimView sv{S.stim, uni(S.n_stim), mask};
  const Coef c = uni(S.c);
  const size_t cells = S.cells;
  const float *D = uni(S.D), *v = uni(roll_state(S, seg, k, 0)), *w = uni(roll_state(S, seg, k, 1)),
              *u = uni(roll_state(S, seg, k, 2));
  float* out = uni(S.traj + (size_t)k * 3 * cells);
  const int H = uni(S.H), W = uni(S.W);
  const float dt = uni(S.dt), inv_dx2 = uni(S.inv_dx2);
#define FK_RS(X, Y, ST)                                                                     \
  stream_tile<R, true, X, Y, ST, BatchStimView, false, true>(c, D, nullptr, v, w, u, H, W, sv, \
                                                             dt, inv_dx2, out, out + cells,    \
                                                             out + 2 * cells, rs, cs)
  switch (uni(item.flags) | (mask ? 4 : 0)) {
    case 0: FK_RS(false, false, false); break;
    case 1: FK_RS(true, false, false); break;
    case 2: FK_RS(false, true, false); break;
    case 3: FK_RS(true, true, false); break;
    case 4: FK_RS(false, false, true); break;
    case 5: FK_RS(true, false, true); break;
    case 6: FK_RS(false, true, true); break;
    default: FK_RS(true, true, true); break;
  }
#undef FK_RS
}

// After forward segment `seg` (steps c .. c + len - 1): the frames it holds
// (states x_j, j in (c, c + len], j a multiple of fe) and, when `ckpt`, its
// last state as the next checkpoint. blockIdx.y: problem.
__global__ void __launch_bounds__(256)
k_roll_gather(const RollDesc* __restrict__ sims, int seg, int c, int len, int fe, int ckpt) {
  const RollDesc& S = sims[blockIdx.y];
  const size_t cells = S.cells;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < cells;
       i += (size_t)gridDim.x * 256) {
    for (int j = (c / fe + 1) * fe; j <= c + len; j += fe)
      S.frames[(size_t)(j / fe - 1) * cells + i] = S.traj[((size_t)(j - c - 1) * 3 + 2) * cells + i];
    if (ckpt)
      for (int f = 0; f < 3; ++f)
        S.ckpt[((size_t)seg * 3 + f) * cells + i] = S.traj[((size_t)(len - 1) * 3 + f) * cells + i];
  }
}

// dL/dD and the cotangent start at zero.
__global__ void __launch_bounds__(256) k_roll_zero(const RollDesc* __restrict__ sims) {
  const RollDesc& S = sims[blockIdx.y];
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < S.cells;
       i += (size_t)gridDim.x * 256) {
    S.gD[i] = 0.0f;
    for (int f = 0; f < 3; ++f) S.lam[(size_t)f * S.cells + i] = 0.0f;
  }
}

// The cotangent back from the ping-pong partner (a segment of odd length).
__global__ void __launch_bounds__(256) k_roll_lam_back(const RollDesc* __restrict__ sims) {
  const RollDesc& S = sims[blockIdx.y];
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < 3 * S.cells;
       i += (size_t)gridDim.x * 256)
    S.lam[i] = S.lam_alt[i];
}

// Frame cotangent injected into x_j (null when j is not a frame step).
__device__ __forceinline__ const float* roll_inject(const RollDesc& S, int j, int fe) {
  return (j > 0 && j % fe == 0) ? gfield(S.g_frames) + (size_t)(j / fe - 1) * S.cells : nullptr;
}

// Reverse of step c + k of segment `seg` (j = c + k + 1): cotangent set `cur`
// (0 lam, 1 lam_alt) -> the other; x_j's frame cotangent enters first. R = 1: two
// rows per block.
template <int R>
__global__ void __launch_bounds__(R == 1 ? 128 : 256)
k_roll_rev(const RollDesc* __restrict__ sims, const RollTile* __restrict__ items, int n_items,
           const uint32_t* __restrict__ masks, int seg, int k, int j, int fe, int cur) {
  constexpr int kWaves = R == 1 ? 2 : 4;
  __shared__ AdjAxisTab tab[kWaves][2];
  const int it = __builtin_amdgcn_readfirstlane(blockIdx.x * kWaves + (int)(threadIdx.x >> 6));
  if (it >= n_items) return;
  RollTile item = items[it];
  if (uni(item.sim) < 0) return;  // padding of the XCD order
  item.sim = uni(item.sim);
  const RollDesc& S = sims[item.sim];
  const size_t n = S.cells;
  const float* lin = uni(cur ? S.lam_alt : S.lam);
  float* lout = uni(cur ? S.lam : S.lam_alt);
  const AdjArgs a{uni(roll_state(S, seg, k, 0)), uni(roll_state(S, seg, k, 1)),
                  uni(roll_state(S, seg, k, 2)), uni(S.D), lin, lin + n, lin + 2 * n,
                  uni(roll_inject(S, j, fe)), lout, lout + n, lout + 2 * n, uni(S.gD),
                  uni(S.part), uni(S.tab)};
  const uint32_t mask = uni((int)masks[item.sim]);
  const BatchStimView sv{S.stim, mask ? uni(S.n_stim) : 0, mask};
  const Coef c = uni(S.c);
  adj_tile_any<R>(c, a, uni(S.H), uni(S.W), sv, uni(S.dt), uni(S.inv_dx2), uni(item.rs),
                  uni(item.cs), uni(item.flags), tab[threadIdx.x >> 6]);
}

}  // namespace fk

using namespace fk;

struct fk_rollout_batch {
  int n = 0, n_steps = 0, fe = 1, S = 1, n_seg = 0;
  std::vector<fk_rollout_spec> specs;
  std::vector<size_t> work_off;  // adjoint workspace of each problem (byte offset)
  std::vector<size_t> work_bytes;
  char* dev = nullptr;
  size_t dev_bytes = 0;
  RollDesc* d_sims = nullptr;
  BlockItem* d_tiles = nullptr;  // forward
  RollTile* d_step = nullptr;    // forward, single steps
  RollTile* d_rev = nullptr;     // reverse
  uint32_t* d_masks = nullptr;  // n_steps x n
  int n_tiles = 0, n_step = 0, n_rev = 0;
  int block = kRoll32x4;  // RollBlock of the forward steps
  int rev_rows = 4;       // band rows of the reverse tiles
  size_t max_cells = 0;
  int traj_seg = -1;  // segment whose states the trajectory buffer holds (-1: none)
};

static int32_t roll_check(const fk_rollout_spec& s, int i) {
  if (!check_params(&s.params) || !check_grid(s.H, s.W) ||
      !check_ptrs({s.D, s.v0, s.w0, s.u0, s.frames, s.g_frames, s.grad_D}) ||
      !check_time(s.t0, s.t0) || !check_scalar("dt", s.dt) || !check_dx(s.dx))
    return set_error(last_code(), "problem %d: %s", i, fk_last_error());
  if (s.n_stimuli < 0 || s.n_stimuli > FK_BATCH_MAX_STIMULI)
    return set_error(FK_ERR_UNSUPPORTED, "problem %d: %d stimuli, the limit is %d", i,
                     s.n_stimuli, FK_BATCH_MAX_STIMULI);
  if (!check_stimuli(s.stimuli, s.n_stimuli))
    return set_error(last_code(), "problem %d: %s", i, fk_last_error());
  return FK_OK;
}

static size_t align256(size_t x) { return (x + 255) / 256 * 256; }

static dim3 roll_cell_grid(const fk_rollout_batch* b) {
  const size_t blocks = std::min<size_t>((b->max_cells + 255) / 256, 1024);
  return dim3((unsigned)std::max<size_t>(blocks, 1), (unsigned)b->n);
}

static void roll_free(fk_rollout_batch* b) {
  if (!b) return;
  if (b->dev) (void)hipFree(b->dev);
  delete b;
}

extern "C" {

int32_t fk_rollout_batch_create(const fk_rollout_spec* specs, int32_t n, int32_t n_steps,
                                int32_t frame_every, int32_t checkpoint_every,
                                fk_rollout_batch** out) {
  ErrorScope es;
  if (out == nullptr) return set_error(FK_ERR_ARG, "out is null");
  *out = nullptr;
  if (n <= 0 || specs == nullptr) return set_error(FK_ERR_ARG, "empty batch");
  if (n_steps < 1 || frame_every < 1 || checkpoint_every < 1)
    return set_error(FK_ERR_ARG, "n_steps, frame_every and checkpoint_every must be >= 1 "
                     "(got %d, %d, %d)", n_steps, frame_every, checkpoint_every);
  for (int i = 0; i < n; ++i) {
    const int32_t rc = roll_check(specs[i], i);
    if (rc != FK_OK) return rc;
    if (!check_time(specs[i].t0, specs[i].t0 + (double)n_steps)) return last_code();
  }
  fk_rollout_batch* b = new fk_rollout_batch();
  b->n = n;
  b->n_steps = n_steps;
  b->fe = frame_every;
  b->S = std::min(checkpoint_every, n_steps);
  b->n_seg = (n_steps + b->S - 1) / b->S;
  b->specs.assign(specs, specs + n);
  int64_t n32x4 = 0, n48x3 = 0, n32x2 = 0, n_rev4 = 0, n_rev2 = 0;
  for (int i = 0; i < n; ++i) {
    const int H = specs[i].H, W = specs[i].W;
    n32x4 += block_tiles<Block32x4>(H, W);
    n48x3 += block_tiles<Block48x3>(H, W);
    n32x2 += block_tiles<Block32x2>(H, W);
    n_rev4 += (int64_t)adj_strips(W) * ((H + 3) / 4);
    n_rev2 += (int64_t)adj_strips(W) * ((H + 1) / 2);
  }
  LeastRounds least(0);  // every step writes its state, whatever the cache holds
  least.offer(kRoll32x4, Block32x4{}, n32x4);
  least.offer(kRoll48x3, Block48x3{}, n48x3);
  least.offer(kRoll32x2, Block32x2{}, n32x2);
  b->block = least.best;
  // A row per wave as in the per-grid step; bands of 2 rows while the waves are few
  // and a wave's rows, one after the other, set the time (2 problems 64 to 200 wide, 100 steps: 1.07 ms, 1.33 with
  // 4; 10 of 128 to 480: 3.33 and 3.40); 4 rows for more (12 of 128 to 512: 4.63 and
  // 4.69; one reverse step of 3.84 M cells 60 and 68 us, 67 with 8). The bits do not
  // depend on it.
  b->rev_rows = n_rev2 <= kRevRowTiles ? 1 : n_rev4 <= 5000 ? 2 : 4;
  const int rows = b->rev_rows;
  // work lists over the dies: neighbouring forward tiles, and runs of vertically
  // adjacent reverse tiles (which share halo rows), whole on one die each
  constexpr int kRunTiles = 16;
  std::vector<BlockItem> blocks;
  std::vector<std::vector<RollTile>> step_runs, rev_runs;
  // whether some segment, or its recomputation, leaves a single step over
  const int per = roll_steps(b->block), last = n_steps - (b->n_seg - 1) * b->S;
  bool single = false;
  for (int len : {b->S, b->S - 1, last, last - 1}) single = single || len % per == 1;
  for (int i = 0; i < n; ++i) {
    const fk_rollout_spec& s = specs[i];
    switch (b->block) {
      case kRoll32x4: append_block_items<Block32x4>(i, s.H, s.W, blocks); break;
      case kRoll48x3: append_block_items<Block48x3>(i, s.H, s.W, blocks); break;
      default: append_block_items<Block32x2>(i, s.H, s.W, blocks); break;
    }
    const StreamGeom g = make_stream_geom<kRollRows>(s.H, s.W);
    for (int strip = 0; single && strip < g.n_strips; ++strip)
      for (int band = 0; band < g.n_bands; ++band) {
        RollTile t;
        t.sim = i;
        t.cs = std::min(kStripOut * strip, g.cs_last);
        t.rs = std::min(kRollRows * band, g.rs_last);
        const bool yg = t.cs < 3 || t.cs + kStripOut + 3 > s.W;
        t.flags = (edge_band(t.rs, kRollRows, s.H, s.W) ? 1 : 0) | (yg ? 2 : 0);
        if (band % kRunTiles == 0) step_runs.emplace_back();
        step_runs.back().push_back(t);
      }
    for (int strip = 0; strip < adj_strips(s.W); ++strip)
      for (int band = 0; band < (s.H + rows - 1) / rows; ++band) {
        RollTile t;
        t.sim = i;
        t.cs = kRevOut * strip;
        t.rs = rows * band;
        t.flags = (adj_edge_band(t.rs, rows, s.H) ? 1 : 0) |
                  (adj_edge_strip(t.cs, s.W) ? 2 : 0);
        if (band % kRunTiles == 0) rev_runs.emplace_back();
        rev_runs.back().push_back(t);
      }
  }
  const std::vector<BlockItem> tiles = block_work_list(blocks);
  const std::vector<RollTile> steps = xcd_order(step_runs, 4, RollTile{-1, 0, 0, 0});
  const std::vector<RollTile> rev = xcd_order(rev_runs, rows == 1 ? 2 : 4, RollTile{-1, 0, 0, 0});
  b->n_tiles = (int)tiles.size();
  b->n_step = (int)steps.size();
  b->n_rev = (int)rev.size();
  // stimulus activity of every step, as the per-grid path evaluates it
  std::vector<uint32_t> masks((size_t)n_steps * n);
  for (int i = 0; i < n; ++i) {
    StimSchedule sched(specs[i].stimuli, specs[i].n_stimuli);
    for (int k = 0; k < n_steps; ++k)
      masks[(size_t)k * n + i] = sched.mask(specs[i].t0 + (double)k);
  }
  // one allocation: descriptors, work lists, masks, then per problem its
  // checkpoints, segment trajectory, cotangent and adjoint workspace
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += align256(bytes);
    return at;
  };
  const size_t o_sims = take(sizeof(RollDesc) * n);
  const size_t o_tiles = take(sizeof(BlockItem) * tiles.size());
  const size_t o_step = take(sizeof(RollTile) * steps.size());
  const size_t o_rev = take(sizeof(RollTile) * rev.size());
  const size_t o_masks = take(sizeof(uint32_t) * masks.size());
  std::vector<size_t> o_ckpt(n), o_traj(n), o_lam(n);
  b->work_off.resize(n);
  b->work_bytes.resize(n);
  for (int i = 0; i < n; ++i) {
    const size_t cells = (size_t)specs[i].H * specs[i].W;
    b->max_cells = std::max(b->max_cells, cells);
    o_ckpt[i] = take((size_t)(b->n_seg - 1) * 3 * cells * sizeof(float));
    o_traj[i] = take((size_t)b->S * 3 * cells * sizeof(float));
    o_lam[i] = take(3 * cells * sizeof(float));
    b->work_bytes[i] = adj_layout(specs[i].H, specs[i].W).total;
    b->work_off[i] = take(b->work_bytes[i]);
  }
  b->dev_bytes = o;
  hipError_t e = hipMalloc((void**)&b->dev, o);
  if (e != hipSuccess) {
    roll_free(b);
    return set_error(FK_ERR_HIP, "hipMalloc(%zu) failed: %s", o, hipGetErrorString(e));
  }
  b->d_sims = (RollDesc*)(b->dev + o_sims);
  b->d_tiles = (BlockItem*)(b->dev + o_tiles);
  b->d_step = (RollTile*)(b->dev + o_step);
  b->d_rev = (RollTile*)(b->dev + o_rev);
  b->d_masks = (uint32_t*)(b->dev + o_masks);
  std::vector<RollDesc> desc(n);
  for (int i = 0; i < n; ++i) {
    const fk_rollout_spec& s = specs[i];
    RollDesc& d = desc[i];
    std::memset(&d, 0, sizeof d);
    const size_t cells = (size_t)s.H * s.W;
    d.c = make_coef(s.params);
    d.H = s.H;
    d.W = s.W;
    d.dt = s.dt;
    d.inv_dx2 = (float)(1.0 / ((double)s.dx * (double)s.dx));
    d.cells = cells;
    d.D = s.D;
    d.x0[0] = s.v0;
    d.x0[1] = s.w0;
    d.x0[2] = s.u0;
    d.ckpt = (float*)(b->dev + o_ckpt[i]);
    d.traj = (float*)(b->dev + o_traj[i]);
    d.frames = s.frames;
    d.g_frames = s.g_frames;
    d.gD = s.grad_D;
    d.lam = (float*)(b->dev + o_lam[i]);
    char* wk = b->dev + b->work_off[i];
    const AdjLayout L = adj_layout(s.H, s.W);
    d.lam_alt = (float*)(wk + L.lam);
    d.tab = (const AdjAxisTab*)(wk + L.tab);
    d.part = (double*)(wk + L.part);
    d.n_stim = s.n_stimuli;
    for (int k = 0; k < s.n_stimuli; ++k)
      d.stim[k] = {s.stimuli[k].start, s.stimuli[k].duration, s.stimuli[k].period,
                   s.stimuli[k].field};
  }
  e = hipMemcpy(b->d_sims, desc.data(), sizeof(RollDesc) * n, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b->d_tiles, tiles.data(), sizeof(BlockItem) * tiles.size(),
                  hipMemcpyHostToDevice);
  if (e == hipSuccess && !steps.empty())
    e = hipMemcpy(b->d_step, steps.data(), sizeof(RollTile) * steps.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b->d_rev, rev.data(), sizeof(RollTile) * rev.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b->d_masks, masks.data(), sizeof(uint32_t) * masks.size(),
                  hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    roll_free(b);
    return set_error(FK_ERR_HIP, "rollout batch setup failed: %s", hipGetErrorString(e));
  }
  *out = b;
  return FK_OK;
}

size_t fk_rollout_batch_device_bytes(const fk_rollout_batch* b) { return b ? b->dev_bytes : 0; }

// Steps c .. c + n_steps - 1 of segment `seg` (c = seg S) into the trajectory.
static void roll_steps_of(fk_rollout_batch* b, int seg, int n_steps, hipStream_t s) {
  const int per = roll_steps(b->block);
  auto masks = [&](int k) { return b->d_masks + (size_t)(seg * b->S + k) * b->n; };
  auto go = [&](auto cfg, int k, int n_lev) {
    typedef decltype(cfg) Cfg;
    k_roll_block<Cfg><<<b->n_tiles, Cfg::waves * 64, 0, s>>>(b->d_sims, b->d_tiles, b->n, masks(k),
                                                            seg, k, n_lev);
  };
  for (int k = 0; k < n_steps; k += per) {
    const int n_lev = std::min(per, n_steps - k);
    if (n_lev == 1) {
      k_roll_step<<<b->n_step / 4, 256, 0, s>>>(b->d_sims, b->d_step, b->n_step, masks(k), seg, k);
      continue;
    }
    switch (b->block) {
      case kRoll32x4: go(Block32x4{}, k, n_lev); break;
      case kRoll48x3: go(Block48x3{}, k, n_lev); break;
      default: go(Block32x2{}, k, n_lev); break;
    }
  }
}

int32_t fk_rollout_batch_forward(fk_rollout_batch* b, void* stream) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "null rollout batch");
  hipStream_t s = (hipStream_t)stream;
  const dim3 cg = roll_cell_grid(b);
  for (int seg = 0; seg < b->n_seg; ++seg) {
    const int c = seg * b->S, len = std::min(b->S, b->n_steps - c);
    roll_steps_of(b, seg, len, s);
    k_roll_gather<<<cg, 256, 0, s>>>(b->d_sims, seg, c, len, b->fe,
                                     seg + 1 < b->n_seg ? 1 : 0);
  }
  HIP_CHECK(hipGetLastError());
  b->traj_seg = b->n_seg - 1;
  return FK_OK;
}

int32_t fk_rollout_batch_backward(fk_rollout_batch* b, float* g_tau, void* stream) {
  ErrorScope es;
  if (b == nullptr) return set_error(FK_ERR_ARG, "null rollout batch");
  hipStream_t s = (hipStream_t)stream;
  for (int i = 0; i < b->n; ++i) {  // boundary tables, tau accumulators
    const fk_rollout_spec& sp = b->specs[i];
    const int32_t rc = fk_adjoint_prepare(sp.D, sp.H, sp.W, b->dev + b->work_off[i],
                                          b->work_bytes[i], stream);
    if (rc != FK_OK) return rc;
  }
  const dim3 cg = roll_cell_grid(b);
  k_roll_zero<<<cg, 256, 0, s>>>(b->d_sims);
  const int rev_blocks = b->n_rev / (b->rev_rows == 1 ? 2 : 4);  // whole blocks, padded
  for (int seg = b->n_seg - 1; seg >= 0; --seg) {
    const int c = seg * b->S, len = std::min(b->S, b->n_steps - c);
    // recompute x_{c+1} .. x_{c+len-1}, unless the forward's last segment is
    // still in place (the same states: same kernels from the same checkpoint)
    if (seg != b->traj_seg) roll_steps_of(b, seg, len - 1, s);
    b->traj_seg = seg;
    int cur = 0;
    for (int k = len - 1; k >= 0; --k) {
      const uint32_t* m = b->d_masks + (size_t)(c + k) * b->n;
      if (b->rev_rows == 1)
        k_roll_rev<1><<<rev_blocks, 128, 0, s>>>(b->d_sims, b->d_rev, b->n_rev, m, seg, k,
                                                 c + k + 1, b->fe, cur);
      else if (b->rev_rows == 2)
        k_roll_rev<2><<<rev_blocks, 256, 0, s>>>(b->d_sims, b->d_rev, b->n_rev, m, seg, k,
                                                 c + k + 1, b->fe, cur);
      else
        k_roll_rev<4><<<rev_blocks, 256, 0, s>>>(b->d_sims, b->d_rev, b->n_rev, m, seg, k,
                                                 c + k + 1, b->fe, cur);
      cur ^= 1;
    }
    if (cur == 1) k_roll_lam_back<<<cg, 256, 0, s>>>(b->d_sims);
  }
  HIP_CHECK(hipGetLastError());
  if (g_tau)
    for (int i = 0; i < b->n; ++i) {
      const fk_rollout_spec& sp = b->specs[i];
      const int32_t rc =
          fk_adjoint_tau_grads(b->dev + b->work_off[i], sp.H, sp.W, g_tau + 3 * i, stream);
      if (rc != FK_OK) return rc;
    }
  return FK_OK;
}

int32_t fk_rollout_batch_destroy(fk_rollout_batch* b) {
  ErrorScope es;
  if (b == nullptr) return FK_OK;
  HIP_CHECK(hipDeviceSynchronize());
  roll_free(b);
  return FK_OK;
}

}  // extern "C"
