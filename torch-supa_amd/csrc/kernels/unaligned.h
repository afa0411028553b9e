// 16-byte vector accesses at element alignment.  Global memory instructions
// take any byte address on gfx950 (the amdhsa default, unaligned-access-mode),
// so a row of odd length still moves in 16-byte vectors: a wavefront's 1 KiB
// run at an odd address touches one cache line more than an aligned one.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dtypes.h"

namespace sa {

typedef u32x4_t u32x4_any __attribute__((aligned(1)));

__device__ __forceinline__ uint4 ld_any(const void* p) {
  const u32x4_t v = *reinterpret_cast<const u32x4_any*>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 ld_any_stream(const void* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void st_any(void* p, const uint4& w) {
  *reinterpret_cast<u32x4_any*>(p) = u32x4_t{w.x, w.y, w.z, w.w};
}
__device__ __forceinline__ void st_any_stream(void* p, const uint4& w) {
  __builtin_nontemporal_store(u32x4_t{w.x, w.y, w.z, w.w}, reinterpret_cast<u32x4_any*>(p));
}

// Rows of c elements written in aligned VEC-wide vectors: how many elements
// before the row at p the vectors start, and the most a row takes.  Rows whose
// length is a multiple of VEC (all at one alignment) start at the 16-byte
// boundary; others at the 128-byte line boundary, so that a wavefront writes
// whole lines.
template <typename T, int VEC> __device__ __forceinline__ int grid_off(const T* p, int64_t c) {
  const int at = (int)(reinterpret_cast<uintptr_t>(p) / sizeof(T) % (128 / sizeof(T)));
  return c % VEC == 0 ? at % VEC : at;
}
template <typename T, int VEC> inline int64_t grid_vecs(const T* p, int64_t c) {
  if (c % VEC == 0) return c / VEC + (reinterpret_cast<uintptr_t>(p) % (VEC * sizeof(T)) ? 1 : 0);
  return (c + 128 / (int64_t)sizeof(T) - 1 + VEC - 1) / VEC;
}

// A vector of VEC elements at element alignment; 16-byte ones stream
// (nontemporal) when STREAM.
template <bool STREAM, typename T, int VEC> __device__ __forceinline__ Vec<T, VEC> ld_vec_any(const T* p) {
  Vec<T, VEC> w;
  if constexpr (sizeof(w) % 16 == 0) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(w) / 16); ++i) {
      const char* q = reinterpret_cast<const char*>(p) + 16 * i;
      const uint4 v = STREAM ? ld_any_stream(q) : ld_any(q);
      __builtin_memcpy(reinterpret_cast<char*>(&w) + 16 * i, &v, 16);
    }
  } else {
    __builtin_memcpy(&w, p, sizeof(w));
  }
  return w;
}
template <typename T, int VEC> __device__ __forceinline__ void st_vec_any(T* p, const Vec<T, VEC>& w) {
  if constexpr (sizeof(w) % 16 == 0) {
#pragma unroll
    for (int i = 0; i < (int)(sizeof(w) / 16); ++i) {
      uint4 v;
      __builtin_memcpy(&v, reinterpret_cast<const char*>(&w) + 16 * i, 16);
      st_any_stream(reinterpret_cast<char*>(p) + 16 * i, v);
    }
  } else {
    __builtin_memcpy(p, &w, sizeof(w));
  }
}

}  // namespace sa
