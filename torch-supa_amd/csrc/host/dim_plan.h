// How a reduction over some dims reads a tensor where it lies.
#pragma once

#include <vector>

#include "common.h"

namespace supa {

// How a reduction over `red` dims reads x where it lies: x dense in some dim
// order, the kept dims in their own order within it, the reduced dims first
// (columns), last (segments of one run), between kept ones (columns) or around
// them (segments: a channel's planes).  kNone: any other pattern.
struct DimPlan {
  enum Kind { kNone, kCols, kSegments } kind = kNone;
  int64_t outer = 1, red = 1, inner = 1;                    // kCols; outer = rows of kSegments
  int64_t segs = 1, len = 1, row_stride = 0, seg_stride = 0;  // kSegments
};
DimPlan dim_plan(const at::Tensor& x, const std::vector<bool>& red);

}  // namespace supa
