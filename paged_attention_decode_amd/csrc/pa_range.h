// pa_range.h - host interface of the range kernel (pa_range.hip), used by the
// launcher in pa_decode.hip.
#ifndef PA_RANGE_H_
#define PA_RANGE_H_

#include "pa_device.h"

namespace pad {

// Largest batch a range launch takes: its planner holds a sequence per lane in
// up to 4 registers (and reads a larger batch twice, in steps), its work list
// two sequences per record.
constexpr int kRangeMaxBatch = 512;

// Work list of a range launch: as many int32 per record, and in the header, as
// in the per-unit kernel's lists (pa_decode.hip checks both sizes at once).
constexpr int kRlHeaderInts = 32;
constexpr int kRlRecordInts = 32;

// A range launch: Phase1Args with hkv counting head groups, and
struct RangeArgs : Phase1Args {
  int groups;        // workgroups of the grid (G)
  int nh_shift;      // a head group is 2^nh_shift consecutive kv heads
  int rows;          // query heads of a head group
  int unit_extra;    // positions a unit counts beyond its pages
  uint32_t gqa_rcp;  // (row * gqa_rcp) >> 16 = row / gqa for row < rows
};

// Queues the decode, or the kernel that writes its work list.
hipError_t launch_range(const RangeArgs& a, int head_dim, int kvf, int nw, size_t lds, hipStream_t st);
hipError_t launch_range_plan(const RangeArgs& a, int32_t* wl, hipStream_t st);

}  // namespace pad

#endif  // PA_RANGE_H_
