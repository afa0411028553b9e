// Pieces the softmax kernels share: raw-word rows, the hardware base-2
// exponential, (max, sum of exp) arithmetic and row stores.
#pragma once

#include "devmath.h"
#include "ew_launch.h"
#include "unaligned.h"

namespace sa {

constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ float fast_exp(float x) {
  // e^x = 2^(x * log2 e); v_exp_f32 for the power of two
  return __builtin_amdgcn_exp2f(x * kLog2e);
}

template <typename T> struct VecOf {
  static constexpr int V = 16 / sizeof(T);
  using type = Vec<T, V>;
};

// The register-resident kernels keep each 16-byte vector as four raw 32-bit
// words and widen an element to float only where it is used; an empty asm
// statement between phases tells the compiler the words may have changed, so
// it never keeps a second, unpacked copy of the row alive (which would spill).
__device__ __forceinline__ uint32_t word_of(const uint4& w, int i) {
  return i == 0 ? w.x : (i == 1 ? w.y : (i == 2 ? w.z : w.w));
}

template <typename T>
__device__ __forceinline__ float elem_f(const uint4& w, int k) {
  if constexpr (std::is_same<T, float>::value) {
    return __uint_as_float(word_of(w, k));
  } else {
    const uint32_t word = word_of(w, k >> 1);
    const uint32_t h = (k & 1) ? (word >> 16) : (word & 0xffffu);
    if constexpr (std::is_same<T, bf16>::value) {
      return __uint_as_float(h << 16);
    } else {
      return (float)__builtin_bit_cast(f16, (uint16_t)h);
    }
  }
}

template <int VPT>
__device__ __forceinline__ void opaque(uint4 (&x)[VPT]) {
#pragma unroll
  for (int j = 0; j < VPT; ++j) asm volatile("" : "+v"(x[j].x), "+v"(x[j].y), "+v"(x[j].z), "+v"(x[j].w));
}

// Row results: 16-byte vectors of TO built from V floats.  bf16 pairs go
// through the gfx950 packed convert (round to nearest even; a NaN keeps its
// NaN-ness, its payload may differ from c10's canonical 0x7FC0).
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

template <typename TO, int V>
__device__ __forceinline__ void store_row_vec(Vec<TO, V>* dst, int v, const float (&f)[V]) {
  if constexpr (std::is_same<TO, bf16>::value) {
    uint32_t w[V / 2];
#pragma unroll
    for (int k = 0; k < V / 2; ++k) {
      const float2_t p = {f[2 * k], f[2 * k + 1]};
      w[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2_t));
    }
    st_stream(reinterpret_cast<Vec<uint32_t, V / 2>*>(dst + v), *reinterpret_cast<const Vec<uint32_t, V / 2>*>(w));
  } else {
    Vec<TO, V> o;
#pragma unroll
    for (int k = 0; k < V; ++k) o.v[k] = from_arith<TO>(f[k]);
    st_stream(dst + v, o);
  }
}

// The same at any element alignment.
template <typename TO, int V>
__device__ __forceinline__ void store_any(TO* p, const float (&f)[V]) {
  if constexpr (std::is_same<TO, bf16>::value) {
    uint4 q;
    uint32_t w[V / 2];
#pragma unroll
    for (int k = 0; k < V / 2; ++k) {
      const float2_t v = {f[2 * k], f[2 * k + 1]};
      w[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    }
    __builtin_memcpy(&q, w, 16);
    st_any_stream(p, q);
  } else {
    Vec<TO, V> o;
#pragma unroll
    for (int k = 0; k < V; ++k) o.v[k] = from_arith<TO>(f[k]);
#pragma unroll
    for (int w = 0; w < (int)(sizeof(o) / 16); ++w) {
      uint4 q;
      __builtin_memcpy(&q, reinterpret_cast<const char*>(&o) + 16 * w, 16);
      st_any_stream(reinterpret_cast<char*>(p) + 16 * w, q);
    }
  }
}

// s = sum of exp(x - m) rescaled to a maximum M >= m: s e^(m - M) (an all
// -inf M leaves s, which is then 0; a NaN s stays NaN).
__device__ __forceinline__ float lse_rescale(float s, float m, float M) {
  return M != -__builtin_inff() ? s * __builtin_amdgcn_exp2f((m - M) * kLog2e) : s;
}

// (max, sum of exp) pairs of `width` lanes (a power of two; lanes w apart in
// the XOR pattern hold the other pairs) combined: a max butterfly, one
// rescale per lane to that max, and a sum butterfly -- one exponential per
// lane where pairwise (m, s) combining takes two per step.  Every butterfly
// step is symmetric in its operands, so every lane ends with the same value.
template <int WIDTH>
__device__ __forceinline__ void lanes_lse(float& m, float& s) {
  float M = m;
#pragma unroll
  for (int off = WIDTH / 2; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
  s = lse_rescale(s, m, M);
#pragma unroll
  for (int off = WIDTH / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  m = M;
}

template <typename F>
int with_float_storage(int dtype, F&& f) {
  switch (dtype) {
    case SUPA_AMD_F32: return f((float*)nullptr);
    case SUPA_AMD_BF16: return f((bf16*)nullptr);
    case SUPA_AMD_F16: return f((f16*)nullptr);
    default: return SUPA_AMD_EDTYPE;
  }
}

}  // namespace sa
