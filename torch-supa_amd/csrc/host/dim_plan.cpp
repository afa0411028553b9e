#include "dim_plan.h"

namespace supa {

DimPlan dim_plan(const at::Tensor& x, const std::vector<bool>& red) {
  DimPlan p;
  int64_t order[64];  // dims of more than one element, slowest first
  int n = 0;
  const int64_t nd = x.dim();
  if (nd > 64) return p;
  for (int64_t i = 0; i < nd; ++i) {
    if (x.size(i) == 1) continue;
    int k = n++;
    for (; k > 0 && x.stride(order[k - 1]) < x.stride(i); --k) order[k] = order[k - 1];
    order[k] = i;
  }
  int64_t dense = 1, last_kept = nd;
  for (int k = n; k-- > 0;) {
    const int64_t d = order[k];
    if (x.stride(d) != dense) return p;
    dense *= x.size(d);
    if (!red[d]) {
      if (d > last_kept) return p;
      last_kept = d;
    }
  }
  c10::SmallVector<std::pair<bool, int64_t>, 8> g;  // runs of kept / reduced dims, slowest first
  for (int k = 0; k < n; ++k) {
    const int64_t d = order[k];
    if (!g.empty() && g.back().first == (bool)red[d]) g.back().second *= x.size(d);
    else g.emplace_back((bool)red[d], x.size(d));
  }
  if (g.empty() || g.size() > 3) return p;
  if (g.size() == 1 && g[0].first) g.insert(g.begin(), std::make_pair(false, int64_t(1)));  // one row
  else if (g.size() == 1) g.emplace_back(true, int64_t(1));
  const bool first = g[0].first;
  if (g.size() == 2 && !first) {  // [K, R]
    p.kind = DimPlan::kSegments;
    p.outer = g[0].second;
    p.len = p.row_stride = g[1].second;
  } else if (g.size() == 3 && first) {  // [R, K, R]
    p.kind = DimPlan::kSegments;
    p.segs = g[0].second;
    p.outer = g[1].second;
    p.len = p.row_stride = g[2].second;
    p.seg_stride = p.outer * p.len;
  } else {  // [R, K] or [K, R, K]
    p.kind = DimPlan::kCols;
    if (!first) p.outer = g[0].second;
    p.red = g[first ? 0 : 1].second;
    p.inner = g.back().second;
  }
  constexpr int64_t lim = int64_t(1) << 31;  // 32-bit rows, runs and positions
  if (p.outer >= lim || p.outer * p.inner >= lim || p.segs * p.len >= lim) p.kind = DimPlan::kNone;
  return p;
}

}  // namespace supa
