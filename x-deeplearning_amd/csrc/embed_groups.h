// embed_groups.h -- which samples a workgroup of the specialised pooling kernel has.
//
// A plan counts workgroups of one size, just as many a slot as have samples.  A launch whose workgroups are a part of those has that
// many times as many, the last of which may begin behind the slot's last sample: with nothing to add up, and no counts of
// their own that may be read, let alone all those in front of their first sample.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bz_common.h"

namespace bz {

// the grid of a launch that has `split` workgroups for each of the plan's, XCD by XCD a contiguous range of them
struct PoolGrid {
  int total_wg, wg_per_slot, wg_per_xcd, blocks;
  PoolGrid(int planned, int planned_per_slot, int split)
      : total_wg(split * planned), wg_per_slot(split * planned_per_slot), wg_per_xcd((total_wg + kNumXcd - 1) / kNumXcd), blocks(wg_per_xcd * kNumXcd) {}
};

// first sample of a slot's workgroup `wg`, each of which has `groups`; below zero: it has none
__host__ __device__ inline int64_t first_sample(int wg, int groups, int32_t batch) {
  const int64_t first = (int64_t)wg * groups;
  return first < batch ? first : -1;
}

}  // namespace bz
