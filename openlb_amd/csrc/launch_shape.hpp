// Launch shapes of the step kernels (host code without HIP calls).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "lbmh.h"

namespace lbmh {

// The collision of a split lattice, all blocks in one launch: by what the blocks
// hold together, and without a cap on the resident workgroups if any block has
// local boundaries, as flat faces are then collided in the same pass.  FP32,
// uncapped against a 40 KB reservation, us per step: 128^3 in 8 blocks (159 MB)
// 85.0 and 86.3, 184^3 in 8 (473 MB) 258.8 and 254.9, 256^3 in 64 (1275 MB) 935
// and 918; FP64, against 48 KB: 128^3 in 8 (319 MB) 149.2 and 145.6, 184^3 in 32
// (947 MB) 687 and 674; FP16 128^3 (80 MB) 59.3 and 66.7; LocalVelocity cavity
// 161^3 in 8, FP32, 208 and 239.  The line is the Infinity Cache's size.  XCD
// groups as in an ensemble.
inline lbmh_launch_config split_launch(int storage, bool local, uint64_t bytes)
{
  lbmh_launch_config c{0, 32};
  if (storage == LBMH_F16 || local || bytes < 256000000u) return c;
  c.lds_bytes = storage == LBMH_F64 ? 49152 : 40960;
  return c;
}

// The XCD group a pass of `chunks` chunks runs with (chunk_of_block): a window
// of 8 x group chunks that the pass does not fill leaves every chunk in
// dispatch order, whatever the group.
inline uint32_t effective_group(int group, uint32_t chunks)
{
  const uint32_t g = group > 0 ? uint32_t(group) : 1u;
  return 8u * g <= chunks ? g : 0u;
}

inline bool same_shape(const lbmh_launch_config& a, const lbmh_launch_config& b, uint32_t chunks)
{
  return a.lds_bytes == b.lds_bytes && effective_group(a.xcd_group, chunks) == effective_group(b.xcd_group, chunks);
}

// The shapes an autotuner times: every (group, LDS reservation), and the shape
// in use and the default where these are not among them, each once.  The shape
// in use comes first.  (Without the last two, tuning replaced the default of a
// 48^3 FP32 D3Q27 block, group 54, by one of group 16: 7.5 -> 8.0 us per step.)
inline std::vector<lbmh_launch_config> tuning_shapes(const lbmh_launch_config& in_use, const lbmh_launch_config& standard,
                                                     const std::vector<int>& groups, const std::vector<int>& lds,
                                                     uint32_t chunks)
{
  std::vector<lbmh_launch_config> all;
  auto find = [&](const lbmh_launch_config& c) {
    return std::find_if(all.begin(), all.end(), [&](const lbmh_launch_config& o) { return same_shape(c, o, chunks); });
  };
  auto add = [&](const lbmh_launch_config& c) {
    if (find(c) == all.end()) all.push_back(c);
  };
  for (int g : groups)
    for (int l : lds) add(lbmh_launch_config{l, g});
  add(standard);
  add(in_use);
  std::iter_swap(all.begin(), find(in_use));
  return all;
}

// The fastest of `shapes`, by `time(shape, &ms)`; the first, which is in use,
// gives way only to one that is also faster when the two are timed again in
// turn (the least of some thirty readings is mostly the luckiest one).
template <typename Time>
int fastest_shape(const std::vector<lbmh_launch_config>& shapes, Time&& time, lbmh_launch_config& best)
{
  constexpr int kAgain = 3;
  size_t at = 0;
  float least = 0.f;
  for (size_t k = 0; k < shapes.size(); ++k) {
    float ms = 0.f;
    const int rc = time(shapes[k], &ms);
    if (rc != LBMH_OK) return rc;
    if (k == 0 || ms < least) {
      least = ms;
      at = k;
    }
  }
  if (at != 0) {
    float both[2] = {0.f, 0.f};
    for (int r = 0; r < kAgain; ++r) {
      for (int k = 0; k < 2; ++k) {
        float ms = 0.f;
        const int rc = time(shapes[k ? at : 0], &ms);
        if (rc != LBMH_OK) return rc;
        both[k] = r == 0 ? ms : std::min(both[k], ms);
      }
    }
    if (both[1] >= both[0]) at = 0;
  }
  best = shapes[at];
  return LBMH_OK;
}

}  // namespace lbmh
