// max / min (with their index) along the last dim of a contiguous [outer,
// inner] input, or along the middle dim of [outer, red, inner] where it lies:
// amax / amin, max.dim / min.dim, argmax / argmin and the full max() / min().
//
// Selection order (a total order on (value, index) pairs, so the result does
// not depend on the reduction tree): a NaN beats every number (upstream's
// max / min propagate NaN, and argmax / argmin point at a NaN); between two
// NaNs or two equal values the smaller index wins (upstream returns the first
// extremal index); otherwise the larger (max) or smaller (min) value wins.
//
// Rows: 16, 64 or 256 threads per (row, chunk of `chunk` elements) by its
// length, each keeping its best pair over 16-byte vectors at any alignment,
// four in flight; a thread meets its elements in order, so a running pair only
// gives way to a strictly better value and its index is 32 bits within the
// chunk.  The pairs meet through shuffles (and LDS for 256).  Long rows take
// two launches: the first writes one pair per chunk, the second (k_argext)
// reduces each row's chunk pairs, reading their indices from `in_idx`.
// Measured on MI355X, us, before (a workgroup and scalar loads for every row)
// -> now, bf16: [131072, 50] 196 -> 9.8, [16384, 1000] 40 -> 9.2,
// [4096, 50257] 227 -> 89; float32 [8192, 8192] 50.5 -> 41 (6.5 TB/s, HBM
// bound; bf16 65.6 -> 25, 5.4 TB/s, bound by the compares: six instructions an
// element).
//
// Middle dim: a thread owns a 16-byte vector of positions and walks the
// reduced dim, TY threads apart where positions alone would leave the chip
// idle; the planes are read once where a transposing copy and a workgroup per
// position came before: classes of float32
// [32, 19, 256, 256] 3415 us -> 30 (5.9 TB/s), of bf16 [4, 21, 513, 513]
// 1583 -> 17.
//
// Replaces amax.out NF:3926, amin.out NF:4115, max.dim_max NF:3894,
// min.dim_min NF:4091, argmax.out NF:839, argmin.out NF:852, max.unary_out
// NF:10274, min.unary_out NF:10204 (upstream ReduceMinMaxKernel.cu /
// ReduceArgMaxKernel.cu / ReduceArgMinKernel.cu).
#include "ew_launch.h"
#include "unaligned.h"

namespace sa {

constexpr int kExtBlock = 256;

template <typename A> __device__ __forceinline__ bool is_nan_v(A a) {
  if constexpr (std::is_floating_point<A>::value) return a != a;
  else return false;
}

// true when (a, ai) comes before (b, bi)
template <bool MIN, typename A, typename I>
__device__ __forceinline__ bool ext_better(A a, I ai, A b, I bi) {
  const bool na = is_nan_v(a), nb = is_nan_v(b);
  if (na != nb) return na;
  if (na || a == b) return ai < bi;
  return MIN ? a < b : a > b;
}

template <bool MIN, typename A, typename I>
__device__ __forceinline__ void ext_take(A& v, I& i, A b, I bi) {
  if (ext_better<MIN>(b, bi, v, i)) {
    v = b;
    i = bi;
  }
}

// One pair per row (or chunk) of pairs whose indices are in_idx, and of rows
// too long for a 32-bit index.  A = the comparison type (float for the float
// family, double, int64 for integers and bool); T = storage.
template <bool MIN, typename T, typename A>
__global__ void __launch_bounds__(kExtBlock)
k_argext(const T* __restrict__ in, const int64_t* __restrict__ in_idx, int64_t inner, int64_t chunk,
         uint32_t nchunks, T* __restrict__ out_val, int64_t* __restrict__ out_idx) {
  __shared__ A lds_v[kExtBlock / 64];
  __shared__ int64_t lds_i[kExtBlock / 64];
  const uint32_t row = blockIdx.x / nchunks, c = blockIdx.x % nchunks;
  const int64_t lo = (int64_t)c * chunk;
  const int64_t hi = lo + chunk < inner ? lo + chunk : inner;
  const T* src = in + (int64_t)row * inner;
  const int64_t* isrc = in_idx ? in_idx + (int64_t)row * inner : nullptr;
  // start from the first element of the segment (always present)
  A bv = (A)to_arith(src[lo]);
  int64_t bi = isrc ? isrc[lo] : lo;
  constexpr int U = 8;
  for (int64_t j0 = lo + threadIdx.x; j0 < hi; j0 += (int64_t)U * kExtBlock) {
    A v[U];
    int64_t ix[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t j = j0 + (int64_t)u * kExtBlock;
      const bool in_r = j < hi;
      v[u] = in_r ? (A)to_arith(src[j]) : bv;
      ix[u] = in_r ? (isrc ? isrc[j] : j) : bi;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) ext_take<MIN>(bv, bi, v[u], ix[u]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const A ov = __shfl_xor(bv, off, 64);
    const int64_t oi = __shfl_xor(bi, off, 64);
    ext_take<MIN>(bv, bi, ov, oi);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    lds_v[wave] = bv;
    lds_i[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < kExtBlock / 64; ++w) ext_take<MIN>(bv, bi, lds_v[w], lds_i[w]);
    if (out_val) out_val[blockIdx.x] = from_arith<T>(bv);
    if (out_idx) out_idx[blockIdx.x] = bi;
  }
}

// Takes (b, bi) for an index above every one met so far.
template <bool MIN, typename A>
__device__ __forceinline__ void ext_next(A& v, uint32_t& i, A b, uint32_t bi) {
  // better, or b is a NaN, and v is none; no short circuit: as branches the
  // compares cost more than the loads (bf16 [65536, 1024]
  // 34.9 us, 23.3 now)
  bool take = MIN ? !(b >= v) : !(b <= v);
  if constexpr (std::is_floating_point<A>::value) take = take & (v == v);
  v = take ? b : v;
  i = take ? bi : i;
}

// The same type as ExtCmp, 32 bits where those hold the storage type.
template <typename T> struct ExtReg {
  using type = typename std::conditional<std::is_same<T, double>::value || std::is_same<T, int64_t>::value, T,
                                         typename std::conditional<std::is_integral<T>::value ||
                                                                       std::is_same<T, b8>::value,
                                                                   int32_t, float>::type>::type;
};

constexpr int kExtUnroll = 4;

template <bool MIN, typename T, int G>
__global__ void __launch_bounds__(kExtBlock)
k_argext_rows(const T* __restrict__ in, int64_t inner, int64_t chunk, FastDiv nchunks, uint32_t first, uint32_t nseg,
              T* __restrict__ out_val, int64_t* __restrict__ out_idx) {
  using A = typename ExtReg<T>::type;
  constexpr int V = 16 / sizeof(T);
  const int lane = threadIdx.x % G;
  uint32_t seg = first + blockIdx.x * (kExtBlock / G) + threadIdx.x / G;
  const bool valid = seg < nseg;
  if (!valid) seg = nseg - 1;  // the block's shuffles need every lane
  uint32_t row, c;
  nchunks.divmod(seg, row, c);
  const int64_t lo = (int64_t)c * chunk;
  const uint32_t len = (uint32_t)(lo + chunk < inner ? chunk : inner - lo);
  const T* src = in + (int64_t)row * inner + lo;
  A bv = (A)to_arith(src[0]);
  uint32_t bi = 0;
  const uint32_t nvec = len / V;
  for (uint32_t v0 = lane; v0 < nvec; v0 += kExtUnroll * G) {
    Vec<T, V> w[kExtUnroll];
#pragma unroll
    for (int u = 0; u < kExtUnroll; ++u)
      if (v0 + u * G < nvec) w[u] = ld_vec_any<true, T, V>(src + (int64_t)(v0 + u * G) * V);
#pragma unroll
    for (int u = 0; u < kExtUnroll; ++u) {
      if (v0 + u * G < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) ext_next<MIN>(bv, bi, (A)to_arith(w[u].v[k]), (v0 + u * G) * V + k);
      }
    }
  }
  const uint32_t t = nvec * V + lane;  // fewer than V <= G elements are left
  if (t < len) ext_next<MIN>(bv, bi, (A)to_arith(src[t]), t);
#pragma unroll
  for (int off = G < 64 ? G / 2 : 32; off > 0; off >>= 1) {
    const A ov = __shfl_xor(bv, off, 64);
    const uint32_t oi = __shfl_xor(bi, off, 64);
    ext_take<MIN>(bv, bi, ov, oi);
  }
  if constexpr (G > 64) {
    __shared__ A lds_v[kExtBlock / 64];
    __shared__ uint32_t lds_i[kExtBlock / 64];
    if ((threadIdx.x & 63) == 0) {
      lds_v[threadIdx.x >> 6] = bv;
      lds_i[threadIdx.x >> 6] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < kExtBlock / 64; ++w) ext_take<MIN>(bv, bi, lds_v[w], lds_i[w]);
    }
  }
  if (lane == 0 && valid) {
    if (out_val) out_val[seg] = from_arith<T>(bv);
    if (out_idx) out_idx[seg] = lo + bi;
  }
}

// [outer, red, inner], inner >= V: TX vectors of positions by TY threads.
template <bool MIN, typename T, int TY>
__global__ void __launch_bounds__(kExtBlock)
k_argext_dim(const T* __restrict__ in, uint32_t red, int64_t inner, FastDiv ivec, uint32_t npos,
             T* __restrict__ out_val, int64_t* __restrict__ out_idx) {
  using A = typename ExtReg<T>::type;
  constexpr int V = 16 / sizeof(T);
  constexpr int TX = kExtBlock / TY;
  const uint32_t tx = threadIdx.x % TX, ty = threadIdx.x / TX;
  uint32_t pos = blockIdx.x * TX + tx;
  const bool valid = pos < npos;
  if (!valid) pos = npos - 1;  // the block's barrier needs every thread
  uint32_t o, v;
  ivec.divmod(pos, o, v);
  int64_t at = (int64_t)v * V;
  int skip = 0;  // a plane's last vector ends at its end; its first elements are another's
  if (at + V > inner) {
    skip = (int)(at + V - inner);
    at = inner - V;
  }
  const T* src = in + (int64_t)o * red * inner + at;
  A bv[V];
  uint32_t bi[V];
  {
    const Vec<T, V> w = ld_vec_any<false, T, V>(src);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      bv[k] = (A)to_arith(w.v[k]);
      bi[k] = 0;
    }
  }
  for (uint32_t r0 = ty; r0 < red; r0 += kExtUnroll * TY) {
    Vec<T, V> w[kExtUnroll];
#pragma unroll
    for (int u = 0; u < kExtUnroll; ++u)
      if (r0 + u * TY < red) w[u] = ld_vec_any<true, T, V>(src + (int64_t)(r0 + u * TY) * inner);
#pragma unroll
    for (int u = 0; u < kExtUnroll; ++u) {
      if (r0 + u * TY < red) {
#pragma unroll
        for (int k = 0; k < V; ++k) ext_next<MIN>(bv[k], bi[k], (A)to_arith(w[u].v[k]), r0 + u * TY);
      }
    }
  }
  if constexpr (TY > 1) {
    __shared__ A lds_v[TY][V][TX];
    __shared__ uint32_t lds_i[TY][V][TX];
#pragma unroll
    for (int k = 0; k < V; ++k) {
      lds_v[ty][k][tx] = bv[k];
      lds_i[ty][k][tx] = bi[k];
    }
    __syncthreads();
    if (ty > 0) return;
    for (int y = 1; y < TY; ++y) {
#pragma unroll
      for (int k = 0; k < V; ++k) ext_take<MIN>(bv[k], bi[k], lds_v[y][k][tx], lds_i[y][k][tx]);
    }
  }
  if (!valid) return;
  const int64_t dst = (int64_t)o * inner + at;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (k < skip) continue;
    if (out_val) out_val[dst + k] = from_arith<T>(bv[k]);
    if (out_idx) out_idx[dst + k] = bi[k];
  }
}

template <typename T> struct ExtCmp {
  using type = typename std::conditional<std::is_same<T, double>::value, double,
                                         typename std::conditional<std::is_integral<T>::value ||
                                                                       std::is_same<T, b8>::value,
                                                                   int64_t, float>::type>::type;
};

template <typename F>
int with_ext_storage(int dtype, F&& f) {
  switch (dtype) {
    case SUPA_AMD_F32: return f((float*)nullptr);
    case SUPA_AMD_BF16: return f((bf16*)nullptr);
    case SUPA_AMD_F16: return f((f16*)nullptr);
    case SUPA_AMD_F64: return f((double*)nullptr);
    case SUPA_AMD_U8: return f((uint8_t*)nullptr);
    case SUPA_AMD_I8: return f((int8_t*)nullptr);
    case SUPA_AMD_I16: return f((int16_t*)nullptr);
    case SUPA_AMD_I32: return f((int32_t*)nullptr);
    case SUPA_AMD_I64: return f((int64_t*)nullptr);
    case SUPA_AMD_BOOL: return f((b8*)nullptr);
    default: return SUPA_AMD_EDTYPE;
  }
}

// Threads per row segment: 16 up to 64 vectors (four each), a wavefront up to
// 256, else a workgroup; with enough rows to fill the chip twice as many
// vectors a thread (bf16 [65536, 1024] 23.3 us with 16 threads, 29.8 with 64;
// [4096, 1024] 6.0 and 4.8; [16384, 4096] 24.3 with 64, 29.1 with 256;
// [512, 8192] 9.3 and 4.6).
template <bool MIN, typename T>
int launch_ext_rows(const T* in, int64_t outer, int64_t inner, int64_t chunk, int64_t nchunks, T* out_val,
                    int64_t* out_idx, hipStream_t st) {
  const uint32_t nseg = (uint32_t)(outer * nchunks);
  const int64_t vecs = std::min(chunk, inner) * (int64_t)sizeof(T) / 16;
  const FastDiv div((uint32_t)nchunks);
  auto go = [&](auto g) -> int {
    constexpr int64_t per = kExtBlock / g.value;
    constexpr int64_t slab = per * (((int64_t(1) << 32) - 1) / kExtBlock);  // HIP: fewer than 2^32 threads a launch
    for (int64_t s0 = 0; s0 < nseg; s0 += slab) {
      const int64_t n = std::min<int64_t>(slab, nseg - s0);
      k_argext_rows<MIN, T, g.value><<<(unsigned)((n + per - 1) / per), kExtBlock, 0, st>>>(
          in, inner, chunk, div, (uint32_t)s0, nseg, out_val, out_idx);
      const int rc = launch_status();
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  };
  if (vecs <= (nseg >= (1u << 15) ? 128 : 64)) return go(std::integral_constant<int, 16>{});
  if (vecs <= (nseg >= (1u << 13) ? 512 : 256)) return go(std::integral_constant<int, 64>{});
  return go(std::integral_constant<int, 256>{});
}

// TY: 4 or 16 threads along the reduced dim while the position vectors alone
// are fewer than the chip holds threads (256 CUs x 2048) and each of the TY
// keeps a batch of loads.
template <bool MIN, typename T>
int launch_ext_dim(const T* in, int64_t outer, int64_t red, int64_t inner, T* out_val, int64_t* out_idx,
                   hipStream_t st) {
  constexpr int64_t V = 16 / sizeof(T);
  const int64_t ivec = (inner + V - 1) / V, npos = outer * ivec;
  if (inner < V || npos >= (int64_t(1) << 31) || red >= (int64_t(1) << 31)) return SUPA_AMD_ELAYOUT;
  const FastDiv div((uint32_t)ivec);
  auto grid = [&](int ty) { return (unsigned)((npos * ty + kExtBlock - 1) / kExtBlock); };
  const uint32_t r = (uint32_t)red, np = (uint32_t)npos;
  if (npos >= (1 << 19) || red <= kExtUnroll)
    k_argext_dim<MIN, T, 1><<<grid(1), kExtBlock, 0, st>>>(in, r, inner, div, np, out_val, out_idx);
  else if (npos >= (1 << 17) || red <= 4 * kExtUnroll)
    k_argext_dim<MIN, T, 4><<<grid(4), kExtBlock, 0, st>>>(in, r, inner, div, np, out_val, out_idx);
  else k_argext_dim<MIN, T, 16><<<grid(16), kExtBlock, 0, st>>>(in, r, inner, div, np, out_val, out_idx);
  return launch_status();
}

}  // namespace sa

using namespace sa;

extern "C" {

int supa_amd_argext_rows(const void* in, int32_t dtype, const int64_t* in_idx, int64_t outer, int64_t inner,
                         int64_t chunk, int is_min, void* out_val, int64_t* out_idx, void* stream) {
  if (!in || outer < 0 || inner <= 0 || chunk <= 0 || (!out_val && !out_idx)) return SUPA_AMD_EINVAL;
  if (outer == 0) return SUPA_AMD_OK;
  const int64_t nchunks = (inner + chunk - 1) / chunk;
  if (outer * nchunks >= (int64_t(1) << 31)) return SUPA_AMD_ELAYOUT;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ext_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    using A = typename ExtCmp<T>::type;
    if (!in_idx && std::min(chunk, inner) < (int64_t(1) << 32)) {
      const T* src = static_cast<const T*>(in);
      T* val = static_cast<T*>(out_val);
      return is_min ? launch_ext_rows<true, T>(src, outer, inner, chunk, nchunks, val, out_idx, st)
                    : launch_ext_rows<false, T>(src, outer, inner, chunk, nchunks, val, out_idx, st);
    }
    const unsigned blocks = (unsigned)(outer * nchunks);
    if (is_min)
      k_argext<true, T, A><<<blocks, kExtBlock, 0, st>>>(static_cast<const T*>(in), in_idx, inner, chunk,
                                                         (uint32_t)nchunks, static_cast<T*>(out_val), out_idx);
    else
      k_argext<false, T, A><<<blocks, kExtBlock, 0, st>>>(static_cast<const T*>(in), in_idx, inner, chunk,
                                                          (uint32_t)nchunks, static_cast<T*>(out_val), out_idx);
    return launch_status();
  });
}

int supa_amd_argext_dim(const void* in, int32_t dtype, int64_t outer, int64_t red, int64_t inner, int is_min,
                        void* out_val, int64_t* out_idx, void* stream) {
  if (!in || outer < 0 || red <= 0 || inner < 0 || (!out_val && !out_idx)) return SUPA_AMD_EINVAL;
  if (outer == 0 || inner == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ext_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    const T* src = static_cast<const T*>(in);
    T* val = static_cast<T*>(out_val);
    return is_min ? launch_ext_dim<true, T>(src, outer, red, inner, val, out_idx, st)
                  : launch_ext_dim<false, T>(src, outer, red, inner, val, out_idx, st);
  });
}

}  // extern "C"
