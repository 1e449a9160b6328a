// Helpers shared by the batched kernels (fk_batch.hip, and the batched
// rollout of fk_rollout_batch.hip): stimuli with a per-step activity mask,
// wave-uniform (scalar register) copies of descriptor values, and the XCD
// order of a work list.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "fk_block.h"
#include "fk_device.h"

namespace fk {

struct BatchStim {
  double start, duration, period;
  const float* field;
};

__device__ __forceinline__ bool active_dev(double t, const BatchStim& s) {
  if (!(t >= s.start)) return false;
  double r = fmod(s.start - t + 1.0, s.period);
  if (r != 0.0 && ((r < 0.0) != (s.period < 0.0))) r += s.period;
  return r < s.duration;
}

// Wave-uniform copies (scalar registers) of descriptor values.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ float uni(float x) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
template <class P>
__device__ __forceinline__ P* uni(P* p) {
  const uint64_t a = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return (P*)(((uint64_t)hi << 32) | lo);
}

// The simulation's stimuli with this step's activity mask.
struct BatchStimView {
  const BatchStim* s;
  int n;
  uint32_t mask;
  __device__ int count() const { return n; }
  __device__ bool on(int m) const { return (mask >> m) & 1u; }
  __device__ const float* field(int m) const { return s[m].field; }
};

// Work-list order for the chip's placement of workgroup w on XCD w % 8 (each
// XCD has its own L2): `runs` are groups of consecutive workgroups that share
// halo rows (a column of tiles); each run goes whole to the XCD with the least
// work so far, and the XCD lists are interleaved, short ones padded with
// `pad` items that exit at once. `per_wg` items make one workgroup.

template <class T>
inline std::vector<T> xcd_order(const std::vector<std::vector<T>>& runs, int per_wg, T pad) {
  std::vector<std::vector<T>> lists(kXcds);
  for (const auto& r : runs) {
    size_t best = 0;
    for (int x = 1; x < kXcds; ++x)
      if (lists[x].size() < lists[best].size()) best = x;
    lists[best].insert(lists[best].end(), r.begin(), r.end());
  }
  size_t m = 0;
  for (auto& l : lists) {
    while (l.size() % per_wg) l.push_back(pad);
    m = std::max(m, l.size() / per_wg);
  }
  std::vector<T> out;
  out.reserve(m * kXcds * per_wg);
  for (size_t j = 0; j < m; ++j)
    for (int x = 0; x < kXcds; ++x)
      for (int k = 0; k < per_wg; ++k)
        out.push_back(j * per_wg + k < lists[x].size() ? lists[x][j * per_wg + k] : pad);
  return out;
}

// One block tile (fk_block.h) of problem `sim`; sim < 0: padding.
struct BlockItem {
  int sim;
  BlockSpan r, c;
  int pad;
};

// The simulation's stimuli at the levels of a launch: bits 4 l .. 4 l + 3 of
// `packed` are the activity mask of level l.
static_assert(FK_BATCH_MAX_STIMULI <= 4 && kBlockMaxSteps <= 8, "masks of a launch in one word");
struct BatchBlockStim {
  const BatchStim* s;
  uint32_t packed;
  __device__ uint32_t active(int l) const { return (packed >> (4 * l)) & 15u; }
  __device__ const float* field(int m) const { return s[m].field; }
};

// masks: the activity words of one simulation, `stride` apart per step.
__device__ __forceinline__ uint32_t pack_masks(const uint32_t* masks, int stride, int n_lev) {
  uint32_t p = 0;
  for (int l = 0; l < n_lev; ++l) p |= (masks[(size_t)l * stride] & 15u) << (4 * l);
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
}

// The tiles of an H x W problem, in the patches of block_place.
template <class Cfg>
inline void append_block_items(int sim, int H, int W, std::vector<BlockItem>& out) {
  const BlockAxis ra = Cfg::row_axis(H), ca = Cfg::col_axis(W);
  for (int g = 0; g < ra.n; g += kBlockGroup)
    for (int strip = 0; strip < ca.n; ++strip)
      for (int band = g; band < std::min(g + kBlockGroup, ra.n); ++band)
        out.push_back({sim, block_span(ra, band), block_span(ca, strip), 0});
}

// The work list of block tiles over the XCDs: runs of neighbouring tiles, at
// least eight runs per XCD so that the lists come out even.
inline std::vector<BlockItem> block_work_list(const std::vector<BlockItem>& items) {
  const size_t run = std::max<size_t>(1, items.size() / (8 * kXcds));
  std::vector<std::vector<BlockItem>> runs;
  for (size_t k = 0; k < items.size(); k += run)
    runs.emplace_back(items.begin() + k, items.begin() + std::min(k + run, items.size()));
  BlockItem pad{};
  pad.sim = -1;
  return xcd_order(runs, 1, pad);
}

}  // namespace fk
