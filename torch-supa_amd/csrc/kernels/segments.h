// Rows made of runs: how the dim reductions (sums, moments) read a row of a
// tensor where it lies.  Row r is `segs` runs of `len` contiguous elements,
// run s at element r row_stride + s seg_stride (a matrix row is one run; a
// channel of [N, C, H, W] is N planes).  Its 16-byte vectors, ceil(len / VW) a
// run, are numbered across the runs.
#pragma once

#include "ew_launch.h"
#include "unaligned.h"

namespace sa {

template <typename T> constexpr bool dim_sum_vec() { return is_floating_st<T>::value; }
template <typename T> constexpr int dim_sum_vw() { return dim_sum_vec<T>() ? 16 / (int)sizeof(T) : 1; }

// VW elements of T as loaded, and element k as ACC.
template <typename T, int VW> struct SumRaw {
  using type = uint4;
};
template <typename T> struct SumRaw<T, 1> {
  using type = T;
};
template <typename T, int VW> using sum_raw_t = typename SumRaw<T, VW>::type;

template <typename T, int VW, bool STREAM = true> __device__ __forceinline__ sum_raw_t<T, VW> sum_load(const T* p) {
  if constexpr (VW == 1) return *p;
  else return STREAM ? ld_any_stream(p) : ld_any(p);
}
template <typename T, int VW, typename ACC>
__device__ __forceinline__ ACC sum_elem(const sum_raw_t<T, VW>& w, int k) {
  if constexpr (VW == 1) {
    return (ACC)to_arith(w);
  } else {
    T v[VW];
    __builtin_memcpy(v, &w, 16);
    return (ACC)to_arith(v[k]);
  }
}

struct SegGeom {
  int64_t rows, row_stride, seg_stride;
  int64_t runs, len;
  FastDiv vps;      // vectors per run (several runs: their vectors fit 32 bits)
  int64_t nvec;     // vectors per row
  uint32_t chunk;   // vectors per chunk of a row
};

// Vector i of a row (across its runs).  A run's last short vector comes back
// with zeros in place of the elements that are not its own; bit k of `valid`
// is set for element k that is.
template <typename T, int VW, bool STREAM = true>
__device__ __forceinline__ sum_raw_t<T, VW> seg_load(const T* row, const SegGeom& g, int64_t i, uint32_t& valid) {
  valid = (1u << VW) - 1u;
  const T* p = row + i * VW;
  int64_t left = g.len - i * VW;
  if (g.runs > 1) {  // uniform
    uint32_t s, v;
    g.vps.divmod((uint32_t)i, s, v);
    p = row + (int64_t)s * g.seg_stride + (int64_t)v * VW;
    left = g.len - (int64_t)v * VW;
  }
  if constexpr (VW == 1) {
    return *p;
  } else {
    if (left >= VW) return sum_load<T, VW, STREAM>(p);
    T w[VW];
    uint4 q;
    if (g.len >= VW) {  // the run's last vector, zeros for what the one before holds
      q = ld_any(p + left - VW);
      valid &= valid << (VW - left);
      __builtin_memcpy(w, &q, 16);
#pragma unroll
      for (int k = 0; k < VW; ++k)
        if (k < VW - left) w[k] = T{};
    } else {
      valid >>= VW - left;
#pragma unroll
      for (int k = 0; k < VW; ++k) w[k] = k < left ? p[k] : T{};
    }
    __builtin_memcpy(&q, w, 16);
    return q;
  }
}

}  // namespace sa
