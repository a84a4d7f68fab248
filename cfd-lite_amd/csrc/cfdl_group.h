// cfdl_group.h -- grouped launches (HIP translation units only): one launch
// runs the same step for several independent systems ("slots").  Block b of
// the launch belongs to the slot whose range [b0[i], b0[i+1]) holds it, and
// runs as one of that slot's blocks 0 .. b0[i+1]-b0[i]-1 (xcd_item).
#pragma once

#include <hip/hip_runtime.h>

#include "cfdl_internal.h"

namespace cfdl {

// Work item of block b of n (a bijection): blocks go to the 8 XCDs round robin,
// so items in block order would put neighbouring cells' blocks on different
// XCDs, each with an L2 of its own, and the values they share would be fetched
// once per XCD.  This gives the blocks of one XCD a contiguous range (96^3:
// colour sweeps 10.6 -> 9.7 us, k_coef_uvw6 272 -> 224 us; renumbered 96^3
// channel: k_mip 425 -> 332 us, k_coef_p6 150 -> 118 us).
constexpr int kXcds = 8;
__device__ inline int xcd_item(int b, int n) {
  const int x = b % kXcds, q = n / kXcds, r = n % kXcds;
  return x * q + min(x, r) + b / kXcds;
}
__device__ inline int xcd_block() {
  return xcd_item(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
}

// the slot of this block and its work item; spread: items in block order, for
// launches whose items differ in cost along the range
__device__ inline int group_slot(const GroupMap &g, int &lb, bool spread = false) {
  int i = 0;
  while (i + 1 < g.n && static_cast<int>(blockIdx.x) >= g.b0[i + 1]) i++;
  lb = static_cast<int>(blockIdx.x) - g.b0[i];
  if (!spread) lb = xcd_item(lb, g.b0[i + 1] - g.b0[i]);
  return g.slot[i];
}

// host: the map of slots taking part (slot ids and their block counts);
// returns the total block count
inline int group_map(GroupMap &g, const int *slot, const int *blocks, int n) {
  g.n = 0;
  g.b0[0] = 0;
  for (int i = 0; i < n; i++) {
    if (blocks[i] <= 0) continue;
    g.slot[g.n] = slot[i];
    g.b0[g.n + 1] = g.b0[g.n] + blocks[i];
    g.n++;
  }
  return g.b0[g.n];
}

}  // namespace cfdl
