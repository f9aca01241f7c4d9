// Places of the chunk walks' workgroups, grid (column slabs, heads, runs).  Workgroup i of a launch runs on XCD i % 8, whose L2 is its
// own, so the `unit` workgroups that read the same rows (the slabs of a head) take places of one XCD's turn: the delta rule's walk, 3
// runs of 510 tokens, 8 heads x 128 x 256, 57.7 -> 53 us, with decays per channel 70 -> 59.5; the channel gate's 195 -> 191.  (The heads
// of a group, which share q and k, gain nothing: the state-space walk, 8 runs of 1000, 187 -> 208.)
#pragma once
#include "common.h"

struct WalkPlace {
  int slab, head, run;
};

SYM_DEV WalkPlace walk_place(int unit) {
  if (unit <= 1) return {(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  const unsigned i = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), n = i >> 3;
  const unsigned at = (n / (unsigned)unit * 8 + (i & 7)) * unit + n % (unsigned)unit, r = at / gridDim.x;
  return {(int)(at % gridDim.x), (int)(r % gridDim.y), (int)(r / gridDim.y)};
}

// the largest unit, halved from `unit`, that the workgroups are whole rounds of; 1: in the order of the places
inline int walk_unit(long long total, int unit) {
  while (unit > 1 && (total % (8LL * unit) || total >= 1LL << 31)) unit = unit % 2 ? 1 : unit / 2;
  return unit;
}
