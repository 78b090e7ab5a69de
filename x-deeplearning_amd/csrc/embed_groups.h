// embed_groups.h -- which samples a workgroup of the specialised pooling kernel has.
//
// A plan counts workgroups of one size, just as many a slot as have samples.  A launch whose workgroups are a part of those has that
// many times as many, the last of which may begin behind the slot's last sample: the counts in front of theirs are not all there to be read.
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

// How many of a slot's counts a workgroup whose first sample is `first` adds up for its offsets.  (It goes on where it has no sample, too: told to
// return, it asked for its record's `batch` alone and for the rest a trip to memory later, keyed 1000 x 24 lists of rows of 100 14.1 -> 14.4 us.)
__host__ __device__ inline int64_t counts_before(int64_t first, int32_t batch) { return first < batch ? first : 0; }

}  // namespace bz
