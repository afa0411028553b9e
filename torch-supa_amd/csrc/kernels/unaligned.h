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

}  // namespace sa
