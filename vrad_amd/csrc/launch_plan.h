// Arithmetic of the launches whose grids grow with the largest inputs (host
// code, no HIP).
#pragma once
#include <algorithm>
#include <cstdint>

namespace vr {

// HIP takes fewer than 2^32 work-items a launch; longer grids go in parts of
// at most 2^31.  Workgroups of the part that starts at workgroup `at`:
inline int64_t grid_part(int64_t at, int64_t groups, int threads) {
  return std::min(groups - at, ((int64_t)1 << 31) / threads);
}

// Owner slots per wave of the blocked copy (k_block_fill): 16 where that still
// makes 16 K waves (with a PVS most of a large system's blocks are empty, and
// a wave costs more than its lookups), else 4.
inline int block_fill_slots(int64_t blocks) { return blocks * 64 >= 16384 ? 16 : 4; }
// and its workgroups of 4 waves; a block has 1024 slots
inline int64_t block_fill_groups(int64_t blocks) {
  return blocks * (1024 / block_fill_slots(blocks)) / 4;
}

// Workgroups per launch of MakeTransfers' trace, of `chunk` candidate pairs
// each: 16 M (a launch's tail costs more than it could give back), or as many
// as the caller's batch_pairs (> 0) allow, at least one.
inline int64_t pair_launch_groups(int64_t batch_pairs, int chunk) {
  constexpr int64_t kMost = (int64_t)1 << 24;
  if (batch_pairs <= 0) return kMost;
  return std::min(kMost, std::max<int64_t>(1, batch_pairs / chunk));
}

}  // namespace vr
