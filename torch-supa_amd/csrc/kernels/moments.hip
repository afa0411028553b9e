// Variance / standard deviation (and the mean beside them) of rows made of
// runs of contiguous elements (segments.h): var / std / var_mean / std_mean
// with a correction, which LayerNorm and BatchNorm written by hand, and
// normalisation statistics, call next to the loss path.
//
// HBM-bound: one read of the input.  A chunk of up to 2048 16-byte vectors
// stays in the registers of the threads that share it (16 lanes or a
// wavefront, each with whole rows, or a workgroup of 256).  Two passes over
// the registers: a mean, summed as x (1 / n), then the deviations d from it,
// with the corrected two-pass formulas mean + sum d / n and M2 = sum d^2 -
// (sum d)^2 / n: no division per value, and the first mean's rounding drops
// out, however large the mean against the spread.  Longer rows are cut in such
// chunks; each chunk's (count, mean - K, M2), K the row's first element (so
// that the means keep their precision when they are merged), goes to the
// workspace and a second launch merges a row's triples by Chan et al.'s
// update.  The result is M2 / max(0, count - correction), its square root for
// std; a NaN propagates and a row with count <= correction divides by zero
// (inf or NaN), as upstream's device reduction (WelfordOps in
// SharedReduceOps.h) does.
//
// Measured on MI355X, us, before (Welford triples per thread, one element a
// load; planes copied to rows first) -> now: float32 [8192, 4096] 28.2 -> 21.5
// (6.2 TB/s, HBM bound), bf16 25.2 -> 14.7; [65536, 512] 40.8 -> 23.8, bf16
// 40.4 -> 21; [2048, 65536] 143 -> 85; dims (0, 2) of [32, 64, 12544]
// 74 -> 20; [64, 512, 49] 26 -> 5.8; all of 64 Mi elements 61 -> 47, bf16 55 ->
// 27.  float64 rows stream instead (k_moments_stream).
//
// Replaces var.correction_out NF:6629, std.correction_out NF:6088,
// var_mean.correction NF:6668, std_mean.correction NF:6063 (upstream
// ReduceMomentKernel.cu: std_var_kernel_cuda over WelfordOps).
#include "segments.h"

namespace sa {

constexpr int kMomBlock = 256;
constexpr int kMomVecs = 8;                                        // most vectors a thread holds
constexpr uint32_t kMomChunk = (uint32_t)kMomBlock * kMomVecs;     // most vectors a chunk holds
// float64 rows stream through (k_moments_stream) and are cut when few and long.
constexpr int64_t kMomStreamRow = 16384;   // vectors of the longest uncut row
constexpr int64_t kMomStreamRows = 2048;   // rows from which none is cut
constexpr int64_t kMomStreamChunk = 8192;  // vectors a chunk

template <typename A> struct Welford {
  A n, mean, m2;
};

template <typename A> __device__ __forceinline__ bool mom_finite(A x) { return x - x == A(0); }

// Means of +inf or -inf meet as they would in a sum (inf + finite is inf).
template <typename A> __device__ __forceinline__ Welford<A> wf_merge(Welford<A> a, Welford<A> b) {
  if (a.n == A(0)) return b;
  if (b.n == A(0)) return a;
  const A n = a.n + b.n;
  const A d = b.mean - a.mean;
  const A nb_n = b.n / n;
  return {n, mom_finite(d) ? a.mean + d * nb_n : a.mean + b.mean, a.m2 + b.m2 + d * d * a.n * nb_n};
}
// The value that chunk means are taken relative to: the row's first element.
template <typename A, typename T> __device__ __forceinline__ A mom_shift(T first) {
  const A k = (A)to_arith(first);
  return mom_finite(k) ? k : A(0);
}

template <typename A> __device__ __forceinline__ Welford<A> wf_shfl(Welford<A> w, int off) {
  return {__shfl_xor(w.n, off, 64), __shfl_xor(w.mean, off, 64), __shfl_xor(w.m2, off, 64)};
}

// Sums of two values over the G threads that share a chunk, in every one.
template <int G, typename A> __device__ __forceinline__ void mom_sum(A& u, A& v, A (*lds)[kMomBlock / 64]) {
#pragma unroll
  for (int off = (G < 64 ? G : 64) / 2; off > 0; off >>= 1) {
    u += __shfl_xor(u, off, 64);
    v += __shfl_xor(v, off, 64);
  }
  if constexpr (G > 64) {
    if ((threadIdx.x & 63) == 0) {
      lds[0][threadIdx.x >> 6] = u;
      lds[1][threadIdx.x >> 6] = v;
    }
    __syncthreads();
    u = lds[0][0];
    v = lds[1][0];
#pragma unroll
    for (int w = 1; w < G / 64; ++w) {
      u += lds[0][w];
      v += lds[1][w];
    }
    __syncthreads();  // the slots are free for the next sum
  }
}

template <typename A, typename OT>
__device__ __forceinline__ void mom_write(Welford<A> w, A correction, int take_sqrt, OT* var, OT* mean) {
  const A div = w.n > correction ? w.n - correction : A(0);
  const A v = w.m2 / div;
  *var = from_arith<OT>(take_sqrt ? sqrt(v) : v);
  if (mean) *mean = from_arith<OT>(w.mean);
}

// FINAL: the chunk is the whole row; else its triple goes to part[row nchunks
// + chunk].
template <typename T, typename A, int VW, int G, int NV, bool FINAL>
__global__ void __launch_bounds__(kMomBlock)
k_moments(const T* __restrict__ in, SegGeom g, FastDiv nch, A correction, int take_sqrt, T* __restrict__ out_var,
          T* __restrict__ out_mean, A* __restrict__ part) {
  __shared__ A lds[2][kMomBlock / 64];
  const int l = threadIdx.x & (G - 1);
  // G = 256: workgroup b takes chunk b % nch of row b / nch
  uint32_t wrow = blockIdx.x, c = 0;
  if constexpr (!FINAL) nch.divmod(blockIdx.x, wrow, c);
  const int64_t row = G < 256 ? (int64_t)blockIdx.x * (256 / G) + threadIdx.x / G : (int64_t)wrow;
  if (row >= g.rows) return;
  const T* src = in + row * g.row_stride;
  const int64_t lo = (int64_t)c * g.chunk;
  const int64_t hi = g.nvec - lo < g.chunk ? g.nvec : lo + g.chunk;
  sum_raw_t<T, VW> x[NV];
  uint32_t valid[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    valid[j] = 0;
    if (lo + l + j * G < hi) x[j] = seg_load<T, VW>(src, g, lo + l + j * G, valid[j]);
  }
  constexpr uint32_t kAll = (1u << VW) - 1u;
  auto in_row = [&](int j, int k) { return valid[j] == kAll || (valid[j] >> k & 1u); };
  A count;
  if constexpr (FINAL) {
    count = (A)(g.runs * g.len);
  } else {  // whole vectors but for the runs' ends
    int n = 0;
#pragma unroll
    for (int j = 0; j < NV; ++j) n += __popc(valid[j]);
    A dummy = A(0);
    count = (A)n;
    mom_sum<G, A>(count, dummy, lds);
  }
  const A inv = A(1) / count;
  A s = A(0), unused = A(0);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (valid[j] == 0) continue;
#pragma unroll
    for (int k = 0; k < VW; ++k) s = fma(sum_elem<T, VW, A>(x[j], k), inv, s);  // zeros outside the row
  }
  mom_sum<G, A>(s, unused, lds);
  const A mean = s;
  A sd = A(0), m2 = A(0);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (valid[j] == 0) continue;
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      const A d = in_row(j, k) ? sum_elem<T, VW, A>(x[j], k) - mean : A(0);
      sd += d;
      m2 = fma(d, d, m2);
    }
  }
  mom_sum<G, A>(sd, m2, lds);
  if (l == 0) {
    const A c1 = sd / count;
    const A q = m2 - sd * c1;
    const A corr = mom_finite(mean) ? c1 : A(0);  // an infinite mean stands: its deviations are NaN
    Welford<A> w{count, mean + corr, q < A(0) ? A(0) : q};
    if constexpr (FINAL) {
      mom_write<A, T>(w, correction, take_sqrt, out_var + row, out_mean ? out_mean + row : nullptr);
    } else {
      A* p = part + 3 * (int64_t)blockIdx.x;
      p[0] = w.n;
      p[1] = (mean - mom_shift<A>(src[0])) + corr;
      p[2] = w.m2;
    }
  }
}

// The same in one pass, as k_moments where a row's vectors are too many
// registers: each thread merges the triples of kMomStreamU vectors at a time
// into its own.  float64, whose vectors hold two elements and whose deviations
// take twice the registers: [8192, 4100] 45 us, 80 in register chunks;
// [2048, 10000] 30, 44; [512, 8192] 5.8, 13; 32 Mi elements in one row 50, 104.
constexpr int kMomStreamU = 4;
template <typename T, typename A, int VW, int G, bool FINAL>
__global__ void __launch_bounds__(kMomBlock)
k_moments_stream(const T* __restrict__ in, SegGeom g, FastDiv nch, A correction, int take_sqrt,
                 T* __restrict__ out_var, T* __restrict__ out_mean, A* __restrict__ part) {
  constexpr int U = kMomStreamU;
  const int l = threadIdx.x & (G - 1);
  uint32_t wrow = blockIdx.x, c = 0;
  if constexpr (!FINAL) nch.divmod(blockIdx.x, wrow, c);
  const int64_t row = G < 256 ? (int64_t)blockIdx.x * (256 / G) + threadIdx.x / G : (int64_t)wrow;
  if (row >= g.rows) return;
  const T* src = in + row * g.row_stride;
  const int64_t lo = (int64_t)c * g.chunk;
  const int64_t hi = g.nvec - lo < g.chunk ? g.nvec : lo + g.chunk;
  const A K = mom_shift<A>(src[0]);
  Welford<A> w{A(0), A(0), A(0)};
  // U vectors' triple from their elements less K (zeros where not the row's)
  auto merge = [&](const A (&x)[U * VW], const bool (&own)[U * VW], int n) {
    A s = A(0);
#pragma unroll
    for (int k = 0; k < U * VW; ++k) s += x[k];
    const A mean = s / (A)n;
    A m2 = A(0);
#pragma unroll
    for (int k = 0; k < U * VW; ++k) {
      const A d = own[k] ? x[k] - mean : A(0);
      m2 = fma(d, d, m2);
    }
    w = wf_merge(w, Welford<A>{(A)n, mean, m2});
  };
  const int64_t whole = g.runs > 1 ? 0 : min(hi, g.len / VW);
  int64_t i0 = lo + l;
  for (; i0 + (U - 1) * G < whole; i0 += U * G) {
    sum_raw_t<T, VW> q[U];
#pragma unroll
    for (int u = 0; u < U; ++u) q[u] = sum_load<T, VW, false>(src + (i0 + u * G) * VW);
    A x[U * VW];
    bool own[U * VW];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        x[u * VW + k] = sum_elem<T, VW, A>(q[u], k) - K;
        own[u * VW + k] = true;
      }
    merge(x, own, U * VW);
  }
  for (; i0 < hi; i0 += U * G) {
    A x[U * VW];
    bool own[U * VW];
    int n = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      sum_raw_t<T, VW> q;
      uint32_t valid = 0;
      if (i0 + u * G < hi) q = seg_load<T, VW, false>(src, g, i0 + u * G, valid);
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        own[u * VW + k] = valid >> k & 1u;
        x[u * VW + k] = own[u * VW + k] ? sum_elem<T, VW, A>(q, k) - K : A(0);
      }
      n += __popc(valid);
    }
    merge(x, own, n);
  }
#pragma unroll
  for (int off = 1; off < (G < 64 ? G : 64); off <<= 1) w = wf_merge(w, wf_shfl(w, off));
  if constexpr (G > 64) {
    __shared__ Welford<A> lds[G / 64];
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = w;
    __syncthreads();
    w = lds[0];
#pragma unroll
    for (int v = 1; v < G / 64; ++v) w = wf_merge(w, lds[v]);
  }
  if (l == 0) {
    if constexpr (FINAL) {
      w.mean += K;
      mom_write<A, T>(w, correction, take_sqrt, out_var + row, out_mean ? out_mean + row : nullptr);
    } else {
      A* p = part + 3 * (int64_t)blockIdx.x;
      p[0] = w.n;
      p[1] = w.mean;
      p[2] = w.m2;
    }
  }
}

// BS threads merge a row's chunk triples, each kMomMerge of them loaded ahead
// of its merges: a wavefront for up to 128, else 1024 threads (the variance of
// 64 Mi float32 elements, 8192 triples, 47 us, 84.5 with a wavefront of 128 merges
// a lane one after another).
constexpr int kMomMerge = 4;
template <typename T, typename A, int BS>
__global__ void __launch_bounds__(BS)
k_moments_final(const T* __restrict__ in, int64_t row_stride, const A* __restrict__ part, int64_t nch, A correction,
                int take_sqrt, T* __restrict__ out_var, T* __restrict__ out_mean) {
  const int64_t row = blockIdx.x;
  const A* src = part + 3 * row * nch;
  Welford<A> w{A(0), A(0), A(0)};
  for (int64_t i0 = threadIdx.x; i0 < nch; i0 += kMomMerge * BS) {
    Welford<A> t[kMomMerge];
#pragma unroll
    for (int u = 0; u < kMomMerge; ++u) {
      const int64_t i = i0 + u * BS;
      t[u] = i < nch ? Welford<A>{src[3 * i], src[3 * i + 1], src[3 * i + 2]} : Welford<A>{A(0), A(0), A(0)};
    }
#pragma unroll
    for (int u = 0; u < kMomMerge; ++u) w = wf_merge(w, t[u]);
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) w = wf_merge(w, wf_shfl(w, off));
  if constexpr (BS > 64) {
    __shared__ Welford<A> lds[BS / 64];
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = w;
    __syncthreads();
    w = lds[threadIdx.x & (BS / 64 - 1)];
#pragma unroll
    for (int off = 1; off < BS / 64; off <<= 1) w = wf_merge(w, wf_shfl(w, off));
  }
  w.mean += mom_shift<A>(in[row * row_stride]);
  if (threadIdx.x == 0)
    mom_write<A, T>(w, correction, take_sqrt, out_var + row,
                    out_mean ? out_mean + row : nullptr);
}

inline int64_t mom_vecs(int64_t segs, int64_t len, int vw) { return segs * ((len + vw - 1) / vw); }
inline int64_t mom_chunks(int64_t rows, int64_t nvec, int esize) {
  if (esize < 8) return (nvec + kMomChunk - 1) / kMomChunk;
  return nvec > kMomStreamRow && rows < kMomStreamRows ? (nvec + kMomStreamChunk - 1) / kMomStreamChunk : 1;
}

template <typename T>
int moments_launch(const T* in, T* out_var, T* out_mean, int64_t rows, int64_t segs, int64_t len, int64_t row_stride,
                   int64_t seg_stride, double correction, int take_sqrt, void* ws, hipStream_t st) {
  using A = opmath_t<T>;
  constexpr int VW = 16 / (int)sizeof(T);
  const int64_t nvec = mom_vecs(segs, len, VW), nch = mom_chunks(rows, nvec, (int)sizeof(T));
  const int64_t chunk = (nvec + nch - 1) / nch;
  const SegGeom g{rows, row_stride, seg_stride, segs, len, FastDiv(segs > 1 ? (uint32_t)((len + VW - 1) / VW) : 1u), nvec,
                  (uint32_t)chunk};
  if (nch > 1) {
    A* part = static_cast<A*>(ws);
    const unsigned blocks = (unsigned)(rows * nch);
    const FastDiv div((uint32_t)nch);
    if constexpr (sizeof(T) == 8)
      k_moments_stream<T, A, VW, 256, false>
          <<<blocks, kMomBlock, 0, st>>>(in, g, div, (A)correction, take_sqrt, nullptr, nullptr, part);
    else
      k_moments<T, A, VW, 256, kMomVecs, false>
          <<<blocks, kMomBlock, 0, st>>>(in, g, div, (A)correction, take_sqrt, nullptr, nullptr, part);
    const int rc = launch_status();
    if (rc) return rc;
    if (nch <= 128)
      k_moments_final<T, A, 64><<<(unsigned)rows, 64, 0, st>>>(in, row_stride, part, nch, (A)correction, take_sqrt,
                                                               out_var, out_mean);
    else
      k_moments_final<T, A, 1024><<<(unsigned)rows, 1024, 0, st>>>(in, row_stride, part, nch, (A)correction, take_sqrt,
                                                                   out_var, out_mean);
    return launch_status();
  }
  auto slabs = [&](int64_t per, auto&& launch) -> int {  // `per` rows a workgroup
    const int64_t slab = per * (((int64_t(1) << 32) - 1) / kMomBlock);  // HIP: fewer than 2^32 threads a launch
    for (int64_t r0 = 0; r0 < rows; r0 += slab) {
      SegGeom gs = g;
      gs.rows = std::min(slab, rows - r0);
      launch((unsigned)((gs.rows + per - 1) / per), in + r0 * row_stride, gs, out_var + r0,
             out_mean ? out_mean + r0 : nullptr);
      const int rc = launch_status();
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  };
  using std::integral_constant;
  using G16 = integral_constant<int, 16>;
  using G64 = integral_constant<int, 64>;
  using G256 = integral_constant<int, 256>;
  using N1 = integral_constant<int, 1>;
  using N2 = integral_constant<int, 2>;
  using N4 = integral_constant<int, 4>;
  using N8 = integral_constant<int, 8>;
  auto go = [&](auto G, auto NV) -> int {
    return slabs(256 / G.value, [&](unsigned blocks, const T* x, const SegGeom& gs, T* v, T* m) {
      k_moments<T, A, VW, G.value, NV.value, true>
          <<<blocks, kMomBlock, 0, st>>>(x, gs, FastDiv(), (A)correction, take_sqrt, v, m, nullptr);
    });
  };
  // the fewest threads a row, and of those the fewest vectors a thread
  if (nvec <= 16) return go(G16{}, N1{});
  if (nvec <= 64) return go(G64{}, N1{});
  if (nvec <= 128) return go(G64{}, N2{});
  if (nvec <= 256) return go(G64{}, N4{});
  if constexpr (sizeof(T) == 8) {
    auto stream = [&](auto G) -> int {
      return slabs(256 / G.value, [&](unsigned blocks, const T* x, const SegGeom& gs, T* v, T* m) {
        k_moments_stream<T, A, VW, G.value, true>
            <<<blocks, kMomBlock, 0, st>>>(x, gs, FastDiv(), (A)correction, take_sqrt, v, m, nullptr);
      });
    };
    return nvec <= 2048 && rows >= 1024 ? stream(G64{}) : stream(G256{});
  } else {
    if (nvec <= 512) return go(G256{}, N2{});
    if (nvec <= 1024) return go(G256{}, N4{});
    return go(G256{}, N8{});
  }
}

}  // namespace sa

using namespace sa;

extern "C" {

int64_t supa_amd_moments_segments_workspace_bytes(int64_t rows, int64_t segs, int64_t len, int32_t dtype) {
  if (rows < 0 || segs <= 0 || len <= 0) return SUPA_AMD_EINVAL;
  if (dtype != SUPA_AMD_F32 && dtype != SUPA_AMD_BF16 && dtype != SUPA_AMD_F16 && dtype != SUPA_AMD_F64)
    return SUPA_AMD_EDTYPE;
  const int64_t nch = mom_chunks(rows, mom_vecs(segs, len, 16 / dtype_size(dtype)), dtype_size(dtype));
  return nch == 1 ? 0 : rows * nch * 3 * (dtype == SUPA_AMD_F64 ? 8 : 4);
}

int64_t supa_amd_moments_rows_workspace_bytes(int64_t outer, int64_t inner, int32_t dtype) {
  return supa_amd_moments_segments_workspace_bytes(outer, 1, inner, dtype);
}

int supa_amd_moments_segments(const void* in, int32_t dtype, int64_t rows, int64_t segs, int64_t len,
                              int64_t row_stride, int64_t seg_stride, double correction, int take_sqrt, void* out_var,
                              void* out_mean, void* workspace, int64_t ws_bytes, void* stream) {
  if (!in || !out_var || rows < 0 || segs <= 0 || len <= 0 || correction != correction) return SUPA_AMD_EINVAL;
  if (rows == 0) return SUPA_AMD_OK;
  const int64_t need = supa_amd_moments_segments_workspace_bytes(rows, segs, len, dtype);
  if (need < 0) return (int)need;
  const int64_t nvec = mom_vecs(segs, len, 16 / dtype_size(dtype));
  if (rows * mom_chunks(rows, nvec, dtype_size(dtype)) >= (int64_t(1) << 31) || (segs > 1 && nvec >= (int64_t(1) << 31))) return SUPA_AMD_ELAYOUT;
  if (need > 0 && (!workspace || ws_bytes < need)) return SUPA_AMD_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto go = [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    return moments_launch<T>(static_cast<const T*>(in), static_cast<T*>(out_var), static_cast<T*>(out_mean), rows,
                             segs, len, row_stride, seg_stride, correction, take_sqrt ? 1 : 0, workspace, st);
  };
  switch (dtype) {
    case SUPA_AMD_F32: return go((float*)nullptr);
    case SUPA_AMD_BF16: return go((bf16*)nullptr);
    case SUPA_AMD_F16: return go((f16*)nullptr);
    case SUPA_AMD_F64: return go((double*)nullptr);
    default: return SUPA_AMD_EDTYPE;
  }
}

int supa_amd_moments_rows(const void* in, int32_t dtype, int64_t outer, int64_t inner, double correction,
                          int take_sqrt, void* out_var, void* out_mean, void* workspace, int64_t ws_bytes,
                          void* stream) {
  return supa_amd_moments_segments(in, dtype, outer, 1, inner, inner, 0, correction, take_sqrt, out_var, out_mean,
                                   workspace, ws_bytes, stream);
}

}  // extern "C"
