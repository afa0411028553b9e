// log_softmax and softmax, forward and backward, over the last dim of a
// contiguous [rows, cols] tensor.
//
// A row is read once and written once (the HBM minimum of these aten ops)
// wherever it fits the registers of the threads that share it, by its length
// in 16-byte vectors:
//   up to 512     a sub-wavefront of 16 lanes or a wavefront (k_row_fwd,
//                 k_row_bwd): statistics by shuffles alone;
//   up to 2560    (backward 2048) a workgroup of 256 to 1024 threads, the
//                 same kernels with one LDS exchange;
//   2 to 32 parts of that: split over K workgroups of 512 threads that
//                 exchange row partials through a small per-stream buffer, so
//                 four parts share a CU (the section below);
//   otherwise     (split rows switched off, under graph capture, or writing
//                 over the input) aligned rows of up to 16384 vectors in one
//                 1024-thread workgroup, the rest streaming twice.
// Rows of any length and alignment move in 16-byte vectors at element
// alignment (unaligned.h); the last cols mod V elements go one to a thread.
//
// exp() of the row statistics is the hardware base-2 exponential of
// (x - max) * log2 e: the row maximum's term is exactly 1, as upstream's
// exp(x - max) makes it (a pre-scaled x * log2 e - max * log2 e leaves max's
// term 1 +- 2^-18 at |max| near 60, and a row with one dominant logit then
// gets a log-probability of -1.7e-6 where upstream gives 0); the row results
// are rounded to bf16/f16 (or kept in f32) exactly once.
//
// Replaces _log_softmax.out (NF:3752), _log_softmax_backward_data.out
// (NF:3763), _softmax.out and _softmax_backward_data.out, upstream SoftMax.cu /
// PersistentSoftmax.cuh in the reference's operator library.  softmax's
// epilogue is exp(x - max) * (1 / sum) and its gradient y (g - sum(g y)).
#include <cstdlib>
#include <map>
#include <mutex>

#include "softmax_common.h"
#include "unaligned.h"

namespace sa {

constexpr int kRowBlock = 1024;
template <typename ACC>
__device__ __forceinline__ ACC wave_sum(ACC v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block-wide reductions returning the result to every thread.  `lds` holds
// one slot per wavefront; NW = blockDim / 64.
template <int NW>
__device__ __forceinline__ float block_sum_all(float v, float* lds) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  float r = lds[0];
#pragma unroll
  for (int w = 1; w < NW; ++w) r += lds[w];
  return r;
}

// ------------------------------------------------------------- forward
// Persistent: a fixed grid of kLsmGrid workgroups walks the rows, so the next
// row's loads issue right behind the current row's stores.  Row statistics
// in one pass ("online" softmax): each thread reduces its own elements to
// (m, s) = (max, sum of exp(x - m)), and the pairs are combined across the
// wavefront and the workgroup by (m, s) (+) (m', s') = (M, s e^(m-M) + s' e^(m'-M)),
// M = max(m, m'), which needs one workgroup exchange instead of two.  A NaN
// anywhere in a row turns the row's sum, hence every output of the row, into
// NaN, as in the upstream kernels.
constexpr int kLsmGrid = 512;  // 2 workgroups per CU on MI355X's 256 CUs

// ------------------------------------------------- rows in registers
// G threads share a row: 16 or 64 lanes of a wavefront (a 256-thread workgroup
// then holds 256 / G rows) or a workgroup of G = 256 or 512.  Thread l holds
// vectors l, l + G, ... (NV of them) and, where cols is no multiple of the
// vector, element nvec V + l of the rest as a float.  VW = 1: rows of up to
// G elements, one to a lane.
//
// A 1024-thread workgroup per row, as longer rows take, left most of its
// threads without a vector here; rows of odd length took a 256-thread
// workgroup of scalar loads and three passes.  Measured on MI355X, us before
// -> after, forward / backward: bf16 [1048576, 10] 830 -> 40 / 452 -> 40,
// [262144, 64] 1136 -> 20 / 685 -> 22, [65536, 1024] 292 -> 43 (6.2 TB/s) /
// 204 -> 65 (6.2 TB/s), [32768, 1659] 106 -> 41 / 140 -> 61, [16384, 4096]
// 89 -> 46 / 76 -> 70, [8192, 10000] 68 -> 57; float32 [65536, 1000] 290 ->
// 95 / 268 -> 145.
template <int G> constexpr int row_block() { return G <= 64 ? 256 : G; }

// This thread's row and place in it; false past the last row.
template <int G>
__device__ __forceinline__ bool row_place(int64_t rows, int64_t& row, int& l) {
  l = threadIdx.x & (G - 1);
  row = G <= 64 ? (int64_t)blockIdx.x * (256 / (G <= 64 ? G : 256)) + threadIdx.x / G : (int64_t)blockIdx.x;
  return row < rows;
}

template <typename T, int VW, int G, int NV>
__device__ __forceinline__ void row_load(uint4 (&x)[NV], const T* src, int l, int nvec) {
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
      if constexpr (VW == 1) x[j].x = __float_as_uint((float)to_arith(src[l + j * G]));
      else x[j] = ld_any_stream(src + (int64_t)(l + j * G) * VW);
    }
}
template <typename T, int VW>
__device__ __forceinline__ float row_elem(const uint4& w, int k) {
  if constexpr (VW == 1) return __uint_as_float(w.x);
  else return elem_f<T>(w, k);
}
template <typename TO, int VW>
__device__ __forceinline__ void row_store(TO* p, const float (&f)[VW]) {
  if constexpr (VW == 1) p[0] = from_arith<TO>(f[0]);
  else store_any<TO, VW>(p, f);
}

// Values of the G threads of a row combined; every thread ends with the total.
template <int G>
__device__ __forceinline__ void row_lse(float& m, float& s) {
  lanes_lse<(G < 64 ? G : 64)>(m, s);
  if constexpr (G > 64) {
    __shared__ float lds_m[G / 64], lds_s[G / 64];
    const int wave = threadIdx.x >> 6, i = threadIdx.x & 15;
    if ((threadIdx.x & 63) == 0) {
      lds_m[wave] = m;
      lds_s[wave] = s;
    }
    __syncthreads();
    m = i < G / 64 ? lds_m[i] : -__builtin_inff();
    s = i < G / 64 ? lds_s[i] : 0.0f;
    lanes_lse<16>(m, s);
  }
}
template <int G>
__device__ __forceinline__ float row_sum(float s) {
#pragma unroll
  for (int off = (G < 64 ? G : 64) / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if constexpr (G > 64) {
    __shared__ float lds[G / 64];
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
    __syncthreads();
    const int i = threadIdx.x & 15;
    s = i < G / 64 ? lds[i] : 0.0f;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  }
  return s;
}

template <typename TI, typename TO, int VW, int G, int NV, bool LOG>
__global__ void __launch_bounds__(row_block<G>())
k_row_fwd(const TI* __restrict__ in, TO* __restrict__ out, int64_t rows, int cols) {
  int64_t row;
  int l;
  if (!row_place<G>(rows, row, l)) return;
  const TI* src = in + row * cols;
  const int nvec = cols / VW, rest = cols - nvec * VW;
  uint4 x[NV];
  row_load<TI, VW, G, NV>(x, src, l, nvec);
  float xt = -__builtin_inff();  // the identity: adds exp(-inf) = 0
  if (VW > 1 && l < rest) xt = (float)to_arith(src[nvec * VW + l]);
  float m = xt;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
#pragma unroll
      for (int k = 0; k < VW; ++k) m = fmaxf(m, row_elem<TI, VW>(x[j], k));
    }
  const float mb = m == -__builtin_inff() ? 0.0f : m;  // all -inf: keep exp arguments finite
  if constexpr (VW > 1) opaque<NV>(x);
  // a vector's sum, then the sum of the thread's vectors: chains of NV and VW
  float s = VW > 1 ? __builtin_amdgcn_exp2f((xt - mb) * kLog2e) : 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
      float t = NV == 1 ? s : 0.0f;
#pragma unroll
      for (int k = 0; k < VW; ++k) t += __builtin_amdgcn_exp2f((row_elem<TI, VW>(x[j], k) - mb) * kLog2e);
      s = NV == 1 ? t : s + t;
    }
  row_lse<G>(m, s);
  // log: (x - M) - log S;  softmax: e^(x - M) / S (an all -inf row gives
  // 0 * inf = NaN, as upstream)
  const float a = LOG ? m : (m == -__builtin_inff() ? 0.0f : m);
  const float b = LOG ? sa_logf(s) : 1.0f / s;
  auto res = [&](float v) {
    if constexpr (LOG) return (v - a) - b;
    else return __builtin_amdgcn_exp2f((v - a) * kLog2e) * b;
  };
  if constexpr (VW > 1) opaque<NV>(x);
  TO* dst = out + row * cols;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
      float f[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) f[k] = res(row_elem<TI, VW>(x[j], k));
      row_store<TO, VW>(dst + (int64_t)(l + j * G) * VW, f);
    }
  if (VW > 1 && l < rest) dst[nvec * VW + l] = from_arith<TO>(res(xt));
}

// LOG: gi = g - exp(y) sum(g);  softmax: gi = y (g - sum(g y)).
template <typename TG, typename TO, int VW, int G, int NV, bool LOG>
__global__ void __launch_bounds__(row_block<G>())
k_row_bwd(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, int64_t rows, int cols) {
  int64_t row;
  int l;
  if (!row_place<G>(rows, row, l)) return;
  const TG* gsrc = grad + row * cols;
  const TG* ysrc = outp + row * cols;
  const int nvec = cols / VW, rest = cols - nvec * VW;
  uint4 g[NV], y[NV];
  // g, then y: the sum of g runs while y is in flight
  const bool more = VW > 1 && l < rest;
  row_load<TG, VW, G, NV>(g, gsrc, l, nvec);
  float gt = 0.0f, yt = 0.0f;
  if (more) gt = (float)to_arith(gsrc[nvec * VW + l]);
  row_load<TG, VW, G, NV>(y, ysrc, l, nvec);
  if (more) yt = (float)to_arith(ysrc[nvec * VW + l]);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
      float t = 0.0f;  // a vector's sum first, as in the forward
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        if constexpr (LOG) t += row_elem<TG, VW>(g[j], k);
        else t = fmaf(row_elem<TG, VW>(g[j], k), row_elem<TG, VW>(y[j], k), t);
      }
      s = NV == 1 ? t : s + t;
    }
  s = row_sum<G>(LOG ? s + gt : fmaf(gt, yt, s));
  auto res = [&](float gk, float yk) {
    if constexpr (LOG) return fmaf(-__builtin_amdgcn_exp2f(yk * kLog2e), s, gk);
    else return yk * (gk - s);
  };
  if constexpr (VW > 1) {
    opaque<NV>(g);
    opaque<NV>(y);
  }
  TO* dst = gin + row * cols;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (l + j * G < nvec) {
      float f[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) f[k] = res(row_elem<TG, VW>(g[j], k), row_elem<TG, VW>(y[j], k));
      row_store<TO, VW>(dst + (int64_t)(l + j * G) * VW, f);
    }
  if (VW > 1 && l < rest) dst[nvec * VW + l] = from_arith<TO>(res(gt, yt));
}

// Calls launch(VW, G, NV as integral constants, first row, rows, workgroups)
// for rows of `cols` elements in vectors of V and stores its status in rc;
// false when a row has more than MAXV vectors.  Up to 16 elements one lane per
// element; else the fewest lanes that hold the row in one vector each (16,
// 64), then 2, 4 and 8 vectors a lane of one wavefront, then workgroups:
// forward 256 threads by 4 and 512 by 4 or 5, backward 1024 by 1 or 2 (bf16
// [8192, 8192] forward 45 us against 56 with 1024 threads, backward 64 us
// against 66 with 256).
// Rows too few to fill the chip that way (256 CUs) take more threads each, so
// that a row waits for one or two loads a thread: bf16 [512, 4096] backward
// 11.3 us by wavefronts, 5.1 so, and forward 8.1, 4.6; [256, 8192] forward 5.5
// with 256 threads, 4.3 so.
// Launches stay below HIP's 2^32 threads: more rows go in several.
template <int V, int MAXV, bool BWD, typename F>
bool row_split(int64_t rows, int64_t cols, int& rc, F&& launch) {
  using std::integral_constant;
  const int64_t nv = (cols + V - 1) / V;
  if (nv > MAXV) return false;
  rc = SUPA_AMD_OK;
  auto go = [&](auto vw, auto g, auto n) {
    const int64_t per = g.value <= 64 ? 256 / g.value : 1;
    const int64_t slab = per * (((int64_t(1) << 32) - 1) / row_block<g.value>());
    for (int64_t r0 = 0; r0 < rows && rc == SUPA_AMD_OK; r0 += slab) {
      const int64_t nr = std::min(slab, rows - r0);
      rc = launch(vw, g, n, r0, nr, (unsigned)((nr + per - 1) / per));
    }
    return true;
  };
  using I1 = integral_constant<int, 1>;
  using I2 = integral_constant<int, 2>;
  using I4 = integral_constant<int, 4>;
  using IV = integral_constant<int, V>;
  using G16 = integral_constant<int, 16>;
  using G64 = integral_constant<int, 64>;
  using G256 = integral_constant<int, 256>;
  using G512 = integral_constant<int, 512>;
  using G1024 = integral_constant<int, 1024>;
  if (cols <= 16) return go(I1{}, G16{}, I1{});
  if (nv <= 16) return go(IV{}, G16{}, I1{});
  if (nv <= 64) return go(IV{}, G64{}, I1{});
  if (nv <= 128) return go(IV{}, G64{}, I2{});
  if (nv <= 256) return rows < 1536 ? go(IV{}, G256{}, I1{}) : go(IV{}, G64{}, I4{});
  if (nv <= 512) return rows < (BWD ? 3072 : 1024) ? go(IV{}, G256{}, I2{}) : go(IV{}, G64{}, integral_constant<int, 8>{});
  if constexpr (BWD) {
    return nv <= 1024 ? go(IV{}, G1024{}, I1{}) : go(IV{}, G1024{}, I2{});
  } else {
    const bool few = rows < 600;
    if (nv <= 1024) return few ? go(IV{}, G1024{}, I1{}) : go(IV{}, G256{}, I4{});
    if (nv <= 2048) return few ? go(IV{}, G1024{}, I2{}) : go(IV{}, G512{}, I4{});
    static_assert(MAXV <= 3 * 1024, "a forward row fits three vectors of 1024 threads");
    return few ? go(IV{}, G1024{}, integral_constant<int, 3>{}) : go(IV{}, G512{}, integral_constant<int, MAXV / 512>{});
  }
}

template <typename TI, typename TO, int VPT, bool LOG>
__global__ void __launch_bounds__(kRowBlock)
k_lsm_fwd_reg(const TI* __restrict__ in, TO* __restrict__ out, int64_t rows, int64_t cols) {
  constexpr int V = VecOf<TI>::V;
  constexpr int NW = kRowBlock / 64;
  __shared__ float lds_m[NW];
  __shared__ float lds_s[NW];
  const int nvec = (int)(cols / V);
  const int full = nvec / kRowBlock;  // vectors every thread has (uniform)
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const uint4* src = reinterpret_cast<const uint4*>(in + row * cols);
    uint4 x[VPT];
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (j < full) x[j] = ld_stream(src + tid + j * kRowBlock);
      else if (tid + j * kRowBlock < nvec) x[j] = ld_stream(src + tid + j * kRowBlock);
    }
    float m = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (j < full || tid + j * kRowBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) m = fmaxf(m, elem_f<TI>(x[j], k));
      }
    }
    const float mb = m == -__builtin_inff() ? 0.0f : m;  // all -inf: keep exp args finite
    opaque<VPT>(x);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (j < full || tid + j * kRowBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) s += __builtin_amdgcn_exp2f((elem_f<TI>(x[j], k) - mb) * kLog2e);
      }
    }
    lanes_lse<64>(m, s);
    __syncthreads();  // the previous row's readers are done with the slots
    if (lane == 0) {
      lds_m[wave] = m;
      lds_s[wave] = s;
    }
    __syncthreads();
    float M = lds_m[lane & 15], S = lds_s[lane & 15];
    lanes_lse<NW>(M, S);
    // log: (x - M) - log S;  softmax: 2^(x log2e - M log2e) / S with the
    // scaled max of the sum (an all -inf row gives 0 * inf = NaN, as upstream)
    const float logsum = LOG ? sa_logf(S) : 0.0f;
    const float inv = LOG ? 0.0f : 1.0f / S;
    const float Mb = M == -__builtin_inff() ? 0.0f : M;
    opaque<VPT>(x);
    Vec<TO, V>* dst = reinterpret_cast<Vec<TO, V>*>(out + row * cols);
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
      if (j < full || tid + j * kRowBlock < nvec) {
        float f[V];
#pragma unroll
        for (int k = 0; k < V; ++k) {
          if constexpr (LOG) f[k] = (elem_f<TI>(x[j], k) - M) - logsum;
          else f[k] = __builtin_amdgcn_exp2f((elem_f<TI>(x[j], k) - Mb) * kLog2e) * inv;
        }
        store_row_vec<TO, V>(dst, tid + j * kRowBlock, f);
      }
    }
  }
}

// Rows past every other kernel: an online (max, sum) pass, then the output
// from a second read, in 16-byte vectors with kStreamU in flight.
constexpr int kStreamU = 4;

template <typename TI, typename TO, bool LOG>
__global__ void __launch_bounds__(kRowBlock)
k_lsm_fwd_stream(const TI* __restrict__ in, TO* __restrict__ out, int64_t cols) {
  constexpr int V = VecOf<TI>::V, U = kStreamU, NW = kRowBlock / 64;
  __shared__ float lds_m[NW], lds_s[NW];
  const TI* src = in + (int64_t)blockIdx.x * cols;
  TO* dst = out + (int64_t)blockIdx.x * cols;
  const int64_t nvec = cols / V;
  const int tid = threadIdx.x, rest = (int)(cols - nvec * V);
  const float xt = tid < rest ? (float)to_arith(src[nvec * V + tid]) : -__builtin_inff();
  float m = xt, s = xt == -__builtin_inff() ? 0.0f : (xt != xt ? xt : fast_exp(xt - xt));  // e^0, NaN for NaN and inf
  for (int64_t v0 = tid; v0 < nvec; v0 += (int64_t)U * kRowBlock) {
    uint4 w[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kRowBlock < nvec) w[u] = ld_any(src + (v0 + (int64_t)u * kRowBlock) * V);
    float M = m;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kRowBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) M = fmaxf(M, elem_f<TI>(w[u], k));
      }
    const float mb = M == -__builtin_inff() ? 0.0f : M;
    s = lse_rescale(s, m, M);
    m = M;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kRowBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) s += __builtin_amdgcn_exp2f((elem_f<TI>(w[u], k) - mb) * kLog2e);
      }
  }
  lanes_lse<64>(m, s);
  if ((tid & 63) == 0) {
    lds_m[tid >> 6] = m;
    lds_s[tid >> 6] = s;
  }
  __syncthreads();
  m = lds_m[tid & 15];
  s = lds_s[tid & 15];
  lanes_lse<NW>(m, s);
  const float a = LOG ? m : (m == -__builtin_inff() ? 0.0f : m);
  const float b = LOG ? sa_logf(s) : 1.0f / s;
  auto res = [&](float v) {
    if constexpr (LOG) return (v - a) - b;
    else return __builtin_amdgcn_exp2f((v - a) * kLog2e) * b;
  };
  for (int64_t v = tid; v < nvec; v += kRowBlock) {
    const uint4 w = ld_any_stream(src + v * V);
    float f[V];
#pragma unroll
    for (int k = 0; k < V; ++k) f[k] = res(elem_f<TI>(w, k));
    store_any<TO, V>(dst + v * V, f);
  }
  if (tid < rest) dst[nvec * V + tid] = from_arith<TO>(res(xt));
}

// ------------------------------------------------------------ backward
// grad's row stays in registers (raw words) for the row sum; the output row
// streams through in chunks of CH = 4 vectors with the next chunk's loads
// issued before the current chunk's math (8 vectors in flight per thread; two
// measured 3 % slower).
template <typename TG, typename TO, int VPT>
__global__ void __launch_bounds__(kRowBlock)
k_lsm_bwd_reg(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, int64_t cols) {
  constexpr int V = VecOf<TG>::V;
  constexpr int CH = VPT < 4 ? VPT : 4;
  __shared__ float lds[kRowBlock / 64];
  const int64_t row = blockIdx.x;
  const uint4* g = reinterpret_cast<const uint4*>(grad + row * cols);
  const uint4* y = reinterpret_cast<const uint4*>(outp + row * cols);
  const int nvec = (int)(cols / V);
  const int full = nvec / kRowBlock;
  const int tid = threadIdx.x;
  uint4 gv[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j)
    if (j < full || tid + j * kRowBlock < nvec) gv[j] = ld_stream(g + tid + j * kRowBlock);
  uint4 yv[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j)
    if (j < full || tid + j * kRowBlock < nvec) yv[j] = ld_stream(y + tid + j * kRowBlock);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (j < full || tid + j * kRowBlock < nvec) {
#pragma unroll
      for (int k = 0; k < V; ++k) s += elem_f<TG>(gv[j], k);
    }
  }
  s = block_sum_all<kRowBlock / 64>(s, lds);
  opaque<VPT>(gv);
  Vec<TO, V>* dst = reinterpret_cast<Vec<TO, V>*>(gin + row * cols);
#pragma unroll
  for (int c = 0; c < VPT; c += CH) {
    uint4 yn[CH];
    if (c + CH < VPT) {
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int jj = c + CH + j;
        if (jj < full || tid + jj * kRowBlock < nvec) yn[j] = ld_stream(y + tid + jj * kRowBlock);
      }
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int jj = c + j;
      if (jj < full || tid + jj * kRowBlock < nvec) {
        float f[V];
#pragma unroll
        for (int k = 0; k < V; ++k)
          f[k] = fmaf(-__builtin_amdgcn_exp2f(elem_f<TG>(yv[j], k) * kLog2e), s, elem_f<TG>(gv[jj], k));
        store_row_vec<TO, V>(dst, tid + jj * kRowBlock, f);
      }
    }
    if (c + CH < VPT) {
#pragma unroll
      for (int j = 0; j < CH; ++j) yv[j] = yn[j];
    }
  }
}

// Rows past every other kernel: the sum, then the output from a second read.
template <typename TG, typename TO, bool LOG>
__global__ void __launch_bounds__(kRowBlock)
k_bwd_stream(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, int64_t cols) {
  constexpr int V = VecOf<TG>::V, U = kStreamU;
  __shared__ float lds[kRowBlock / 64];
  const int64_t base = (int64_t)blockIdx.x * cols, nvec = cols / V;
  const TG* gs = grad + base;
  const TG* ys = outp + base;
  TO* dst = gin + base;
  const int tid = threadIdx.x, rest = (int)(cols - nvec * V);
  const float gt = tid < rest ? (float)to_arith(gs[nvec * V + tid]) : 0.0f;
  const float yt = tid < rest ? (float)to_arith(ys[nvec * V + tid]) : 0.0f;
  float s = LOG ? gt : gt * yt;
  for (int64_t v0 = tid; v0 < nvec; v0 += (int64_t)U * kRowBlock) {
    uint4 g[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t v = v0 + (int64_t)u * kRowBlock;
      if (v < nvec) {
        g[u] = ld_any(gs + v * V);
        if constexpr (!LOG) y[u] = ld_any(ys + v * V);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kRowBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
          if constexpr (LOG) s += elem_f<TG>(g[u], k);
          else s = fmaf(elem_f<TG>(g[u], k), elem_f<TG>(y[u], k), s);
        }
      }
  }
  s = block_sum_all<kRowBlock / 64>(s, lds);
  auto res = [&](float gk, float yk) {
    if constexpr (LOG) return fmaf(-__builtin_amdgcn_exp2f(yk * kLog2e), s, gk);
    else return yk * (gk - s);
  };
  for (int64_t v = tid; v < nvec; v += kRowBlock) {
    const uint4 g = ld_any_stream(gs + v * V), y = ld_any_stream(ys + v * V);
    float f[V];
#pragma unroll
    for (int k = 0; k < V; ++k) f[k] = res(elem_f<TG>(g, k), elem_f<TG>(y, k));
    store_any<TO, V>(dst + v * V, f);
  }
  if (tid < rest) dst[nvec * V + tid] = from_arith<TO>(res(gt, yt));
}

// softmax backward: gi = y (g - sum(g y)).  Both rows stay in registers
// (up to 8 vectors each per thread); longer rows take the streaming kernel.
template <typename TG, typename TO, int VPT>
__global__ void __launch_bounds__(kRowBlock)
k_sm_bwd_reg(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, int64_t cols) {
  constexpr int V = VecOf<TG>::V;
  __shared__ float lds[kRowBlock / 64];
  const int64_t row = blockIdx.x;
  const uint4* g = reinterpret_cast<const uint4*>(grad + row * cols);
  const uint4* y = reinterpret_cast<const uint4*>(outp + row * cols);
  const int nvec = (int)(cols / V);
  const int full = nvec / kRowBlock;
  const int tid = threadIdx.x;
  uint4 gv[VPT], yv[VPT];
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (j < full || tid + j * kRowBlock < nvec) {
      gv[j] = ld_stream(g + tid + j * kRowBlock);
      yv[j] = ld_stream(y + tid + j * kRowBlock);
    }
  }
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (j < full || tid + j * kRowBlock < nvec) {
#pragma unroll
      for (int k = 0; k < V; ++k) s = fmaf(elem_f<TG>(gv[j], k), elem_f<TG>(yv[j], k), s);
    }
  }
  s = block_sum_all<kRowBlock / 64>(s, lds);
  opaque<VPT>(gv);
  opaque<VPT>(yv);
  Vec<TO, V>* dst = reinterpret_cast<Vec<TO, V>*>(gin + row * cols);
#pragma unroll
  for (int j = 0; j < VPT; ++j) {
    if (j < full || tid + j * kRowBlock < nvec) {
      float f[V];
#pragma unroll
      for (int k = 0; k < V; ++k) f[k] = elem_f<TG>(yv[j], k) * (elem_f<TG>(gv[j], k) - s);
      store_row_vec<TO, V>(dst, tid + j * kRowBlock, f);
    }
  }
}

// ------------------------------------------------------- split rows
// Rows of 2 to 32 parts (split_parts below says which) are split over K
// workgroups of 512 threads, one part each: the backward's parts are at most
// 2048 16-byte vectors (4 per thread, 32 KiB of grad and of output), the
// forward's 2560 (5 per thread, 40 KiB), and a row is spread evenly over its
// K parts (split_part_len below).  Four such workgroups share a CU, so one part's statistics and
// stores overlap other parts' loads; a whole row per 1024-thread workgroup
// leaves a CU with one row, whose stores never overlap the next row's loads.
// On c3's rows (bf16 [8192, 128256]) the backward ran 79.9-80.0 % of the HBM
// roofline against 75.5-76.3 % with 1024-thread parts of 4096 vectors and
// 73.2-73.6 % with a whole row per workgroup, the forward 75.3-75.6 %
// against 69.3-69.7 % and 71.0-71.3 % (parts of 2048 / 2304 / 2688 vectors,
// 256-768 threads: 59-76 %).  Workgroup b takes part b % K of row b / K.  Each
// part publishes its row partial -- (max, sum of exp) forward, sum of grad
// backward -- to slots[row * K + part] with a device-scope atomic store, then
// waits for the row's other parts by polling their slots (device-scope loads,
// a short s_sleep between polls), and every part folds the K partials in slot
// order, so the K parts of a row use one bit-identical total.
//
// A part that is still missing after spin_limit polls (a peer not yet
// resident) is computed by the waiting workgroup itself: it loads that part
// with the same thread layout and reduces it in the same order, so the value
// is bit-identical to the one the peer publishes, and no wait depends on
// another workgroup being scheduled.  The inputs must not overlap the output
// for this (the host checks it).
//
// Slots are 64-bit; 0 marks an empty slot (kSlotTag below).  done[row]
// counts the parts that have read the row's slots; the last one resets the
// row's slots and done[row] to 0, so a buffer is clean after every launch.
// A buffer belongs to one (device, stream) until the process ends; launches
// on one stream are ordered, so they never share it (a stream destroyed with
// split work still queued, whose handle a new stream then receives, would
// share it with that work).
constexpr int kSplitBlock = 512;
constexpr int kSplitNW = kSplitBlock / 64;
constexpr int kFwdNV = 5, kBwdNV = 4;  // vectors per thread of a forward / backward part
constexpr int kSplitMaxK = 32;
constexpr int64_t kSplitSlots = int64_t(1) << 16;  // row parts per launch (c3's 8192 rows x 8 parts: one)
// An empty slot holds 0; a partial v is published as v ^ kSlotTag, whose high
// word is never 0 (a forward partial's high word is its sum, a non-negative
// float or the canonical NaN, below 0x80000000; a backward partial's is 0).
constexpr uint64_t kSlotTag = 0xFFFFFFFF00000000ull;
constexpr uint32_t kSplitSpinDefault = 1u << 16;
// Slot buffers per device (in the library's own device memory, 6 MiB a
// device): streams past the 8th of a device that reach a split call take the
// one-row or streaming kernels instead.
constexpr int kSplitBuffers = 8;

__device__ __forceinline__ void slot_store(uint64_t* p, uint64_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void slot_publish(uint64_t* p, uint64_t v) { slot_store(p, v ^ kSlotTag); }
__device__ __forceinline__ uint64_t slot_load(const uint64_t* p) {
  return __hip_atomic_load(const_cast<uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Polls the row's K slots (wave 0; lane q < K reads slot q) for at most
// spin_limit rounds; stores every published partial to part_w[q] and returns
// the bit mask of parts still missing (same value in every thread).
__device__ __forceinline__ uint32_t split_wait(const uint64_t* rs, int K, uint32_t spin_limit, uint64_t* part_w,
                                               uint32_t* lds_missing) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave == 0) {
    uint64_t v = 0;
    if (lane < K) {
      v = slot_load(rs + lane);
      for (uint32_t n = 0; v == 0 && n < spin_limit; ++n) {
        __builtin_amdgcn_s_sleep(8);
        v = slot_load(rs + lane);
      }
      part_w[lane] = v ^ kSlotTag;
    }
    const uint64_t miss = __ballot(lane < K && v == 0);
    if (lane == 0) *lds_missing = (uint32_t)miss;  // K <= 32
  }
  __syncthreads();
  return *lds_missing;
}

// After every part of the row has read the slots, the last one clears them.
// A part's own publish is complete before its increment: thread 0 stores it
// and then waits on its own slot loads in split_wait, and on gfx9 the vector
// memory counter that wait drains covers stores too, so no slot is published
// after the last part's clear.
__device__ __forceinline__ void split_release(uint64_t* rs, uint32_t* done_row, int K) {
  if (threadIdx.x == 0) {
    const uint32_t d = __hip_atomic_fetch_add(done_row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d == (uint32_t)K - 1) {
      for (int q = 0; q < K; ++q) slot_store(rs + q, 0);
      __hip_atomic_store(done_row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// A whole part loads without per-vector guards (a uniform branch), so its
// loads are not split by divergent ones; a part that fills all but its
// threads' last vector guards only that one.  `end` is one past the part's
// last vector.
// Loads are written at element alignment also for aligned rows: the same
// instructions, and the float32 backward no longer spilled ([4096, 50304]
// 425 -> 391 us, [4096, 65536] 521 -> 496 us).
template <typename T, int NV>
__device__ __forceinline__ void split_load(uint4 (&x)[NV], const T* row, int base, int end) {
  constexpr int V = VecOf<T>::V;
  const int tid = threadIdx.x;
  auto at = [&](int v) { return ld_any_stream(row + (int64_t)v * V); };
  if (base + kSplitBlock * NV <= end) {
#pragma unroll
    for (int j = 0; j < NV; ++j) x[j] = at(base + tid + j * kSplitBlock);
  } else if (base + kSplitBlock * (NV - 1) <= end) {
#pragma unroll
    for (int j = 0; j < NV - 1; ++j) x[j] = at(base + tid + j * kSplitBlock);
    if (base + tid + (NV - 1) * kSplitBlock < end) x[NV - 1] = at(base + tid + (NV - 1) * kSplitBlock);
  } else {
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (base + tid + j * kSplitBlock < end) x[j] = at(base + tid + j * kSplitBlock);
  }
}

// RAGGED rows, whose cols is no multiple of the vector.  The forward moves
// floor(cols / V) vectors at element alignment; its last part also holds the
// rest of the row, element nvec V + t in thread t, as a float (-inf in every
// other thread).
template <bool RAGGED, typename T>
__device__ __forceinline__ float split_rest(const T* row, int64_t cols, int nvec, bool last) {
  if constexpr (!RAGGED) return -__builtin_inff();
  const int64_t i = (int64_t)nvec * VecOf<T>::V + threadIdx.x;
  return last && i < cols ? (float)to_arith(row[i]) : -__builtin_inff();
}

// The backward, with three streams, takes the vectors of the grid of 128-byte
// lines of grad instead, so that every access is aligned and a wavefront
// stores whole lines; a row starts o elements into its first line.  The
// elements of a row's first and last partial vectors that lie outside the row
// are never read or written: those vectors load and store element by element,
// with zeros in the places outside.  bf16 [4096, 50257]: 233 us, on the
// 16-byte grid 239, at element alignment 306 (the forward, 16-byte
// grid and element alignment, 160 and 151 us;
// aligned rows of 50304 200 and 135 us; streaming the rows twice by scalars,
// as rows of odd length did before, 501 and 551 us).
struct SplitRow {
  int o;         // elements between the line boundary and the row
  int vf0, vf1;  // vectors wholly inside the row
  int nvec;      // one past the last vector the row touches
};
template <typename T, bool RAGGED>
__device__ __forceinline__ SplitRow split_row(int o, int64_t cols) {
  constexpr int V = VecOf<T>::V;
  SplitRow r;
  r.o = RAGGED ? o : 0;
  r.vf0 = RAGGED ? (r.o + V - 1) / V : 0;
  r.vf1 = (int)((r.o + cols) / V);
  r.nvec = RAGGED ? (int)((r.o + cols + V - 1) / V) : r.vf1;
  return r;
}
// The row's elements in vector v are [lo, hi) of its V (none before the row).
template <typename T>
__device__ __forceinline__ void split_edge(const SplitRow& r, int64_t cols, int v, int& lo, int& hi) {
  constexpr int V = VecOf<T>::V;
  lo = max(r.o - v * V, 0);
  const int64_t left = r.o + cols - (int64_t)v * V;
  hi = left < V ? (int)left : V;
}

// `row` points at the first vector's first element (o before the row).
template <typename T, int NV, bool RAGGED>
__device__ __forceinline__ void split_load_grid(uint4 (&x)[NV], const T* row, const SplitRow& r, int64_t cols, int base,
                                                int end) {
  constexpr int V = VecOf<T>::V;
  if (RAGGED && (base < r.vf0 || end > r.vf1)) {
    using Bits = std::conditional_t<sizeof(T) == 2, uint16_t, uint32_t>;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int v = base + (int)threadIdx.x + j * kSplitBlock;
      const T* p = row + (int64_t)v * V;
      if (v >= r.vf0 && v < end && v < r.vf1) {
        x[j] = ld_any_stream(p);
      } else if (v < end) {
        int lo, hi;
        split_edge<T>(r, cols, v, lo, hi);
        Bits b[V];
#pragma unroll
        for (int k = 0; k < V; ++k) b[k] = k >= lo && k < hi ? reinterpret_cast<const Bits*>(p)[k] : Bits(0);
        __builtin_memcpy(&x[j], b, 16);
      }
    }
  } else {
    split_load<T, NV>(x, row, base, end);
  }
}

// Stores vector v of a row's results (dst as `row` above).
template <typename TI, typename TO, bool RAGGED>
__device__ __forceinline__ void split_store(TO* dst, const SplitRow& r, int64_t cols, int v,
                                            const float (&f)[VecOf<TI>::V]) {
  constexpr int V = VecOf<TI>::V;
  if (RAGGED && (v < r.vf0 || v >= r.vf1)) {
    int lo, hi;
    split_edge<TI>(r, cols, v, lo, hi);
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (k >= lo && k < hi) dst[(int64_t)v * V + k] = from_arith<TO>(f[k]);
  } else {
    store_any<TO, V>(dst + (int64_t)v * V, f);
  }
}

// The kSplitNW wavefront values of a workgroup, combined over 16 lanes (lane
// l reads wavefront l % 16, or the identity past kSplitNW).
__device__ __forceinline__ void block_lse(float& M, float& S, const float* lds_m, const float* lds_s) {
  const int i = threadIdx.x & 15;
  M = i < kSplitNW ? lds_m[i] : -__builtin_inff();
  S = i < kSplitNW ? lds_s[i] : 0.0f;
  lanes_lse<16>(M, S);
}
__device__ __forceinline__ float block_sum(const float* lds) {
  const int i = threadIdx.x & 15;
  float S = i < kSplitNW ? lds[i] : 0.0f;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) S += __shfl_xor(S, off, 64);
  return S;
}

// Per-thread (max, sum of exp(x - max)) over the thread's vectors of a part.
// The forward keeps its per-vector guards on whole parts too: a specialization
// without them took 62 VGPRs against 57 and ran at 71.1-71.9 % of the HBM
// roofline against 73.2-74.7 % on c3's rows.
template <typename TI, int NV, bool RAGGED>
__device__ __forceinline__ void thread_lse(uint4 (&x)[NV], float xt, int base, int nvec, float& m, float& s) {
  constexpr int V = VecOf<TI>::V;
  const int tid = threadIdx.x;
  m = RAGGED ? xt : -__builtin_inff();
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (base + tid + j * kSplitBlock < nvec) {
#pragma unroll
      for (int k = 0; k < V; ++k) m = fmaxf(m, elem_f<TI>(x[j], k));
    }
  const float mb = m == -__builtin_inff() ? 0.0f : m;
  opaque<NV>(x);
  s = RAGGED ? __builtin_amdgcn_exp2f((xt - mb) * kLog2e) : 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if (base + tid + j * kSplitBlock < nvec) {
#pragma unroll
      for (int k = 0; k < V; ++k) s += __builtin_amdgcn_exp2f((elem_f<TI>(x[j], k) - mb) * kLog2e);
    }
}

// (max, sum of exp(x - max)) of one part, the same in every thread; the
// sum's NaN is canonical.
template <typename TI, int NV, bool RAGGED>
__device__ __forceinline__ uint64_t part_lse(uint4 (&x)[NV], float xt, int base, int nvec, float* lds_m, float* lds_s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float m, s;
  thread_lse<TI, NV, RAGGED>(x, xt, base, nvec, m, s);
  lanes_lse<64>(m, s);
  __syncthreads();
  if (lane == 0) {
    lds_m[wave] = m;
    lds_s[wave] = s;
  }
  __syncthreads();
  float M, S;
  block_lse(M, S, lds_m, lds_s);
  const uint32_t sb = S != S ? 0x7fc00000u : __float_as_uint(S);
  return ((uint64_t)sb << 32) | __float_as_uint(M);
}

template <typename TI, typename TO, bool LOG>
__device__ __forceinline__ void fwd_split_out(const uint4 (&x)[kFwdNV], TO* dst, int base, int nvec, float M, float logsum, float Mb, float inv) {
  constexpr int V = VecOf<TI>::V;
#pragma unroll
  for (int j = 0; j < kFwdNV; ++j) {
    const int v = base + (int)threadIdx.x + j * kSplitBlock;
    if (v < nvec) {
      float f[V];
#pragma unroll
      for (int k = 0; k < V; ++k) {
        if constexpr (LOG) f[k] = (elem_f<TI>(x[j], k) - M) - logsum;
        else f[k] = __builtin_amdgcn_exp2f((elem_f<TI>(x[j], k) - Mb) * kLog2e) * inv;
      }
      store_any<TO, V>(dst + (int64_t)v * V, f);
    }
  }
}

template <typename TI, typename TO, bool LOG, bool RAGGED>
__global__ void __launch_bounds__(kSplitBlock, 8)
k_lsm_fwd_split(const TI* __restrict__ in, TO* __restrict__ out, int64_t cols, int K, int plen,
                uint64_t* __restrict__ slots, uint32_t* __restrict__ done, uint32_t spin_limit) {
  constexpr int V = VecOf<TI>::V;
  __shared__ float lds_m[kSplitNW];
  __shared__ float lds_s[kSplitNW];
  __shared__ uint64_t part_w[kSplitMaxK];
  __shared__ uint32_t lds_missing;
  const int row = (int)(blockIdx.x / (unsigned)K);
  const int part = (int)(blockIdx.x - (unsigned)row * (unsigned)K);
  const int nvec = (int)(cols / V);
  const int base = part * plen;
  const int end = min(base + plen, nvec);
  const TI* src = in + (int64_t)row * cols;
  uint4 x[kFwdNV];
  split_load<TI, kFwdNV>(x, src, base, end);
  const float xt = split_rest<RAGGED>(src, cols, nvec, part == K - 1);
  const uint64_t mine = part_lse<TI, kFwdNV, RAGGED>(x, xt, base, end, lds_m, lds_s);
  opaque<kFwdNV>(x);
  uint64_t* rs = slots + (int64_t)row * K;
  if (threadIdx.x == 0) slot_publish(rs + part, mine);
  uint32_t miss = split_wait(rs, K, spin_limit, part_w, &lds_missing);
  split_release(rs, done + row, K);
  if (miss) {  // uniform; the own part is loaded again afterwards, so the fallback reuses its registers
    do {
      const int q = __builtin_ctz(miss);
      miss &= miss - 1;
      const int qb = q * plen, qe = min(qb + plen, nvec);
      split_load<TI, kFwdNV>(x, src, qb, qe);
      const float qt = split_rest<RAGGED>(src, cols, nvec, q == K - 1);
      const uint64_t w = part_lse<TI, kFwdNV, RAGGED>(x, qt, qb, qe, lds_m, lds_s);
      if (threadIdx.x == 0) part_w[q] = w;
    } while (miss);
    split_load<TI, kFwdNV>(x, src, base, end);
  }
  __syncthreads();
  // the row's (max, sum) from the K part pairs, in part order: the max, then
  // each part's sum rescaled to it (K exponentials)
  float M = __uint_as_float((uint32_t)part_w[0]);
  for (int q = 1; q < K; ++q) M = fmaxf(M, __uint_as_float((uint32_t)part_w[q]));
  auto part_sum_at = [&](int q) {
    return lse_rescale(__uint_as_float((uint32_t)(part_w[q] >> 32)), __uint_as_float((uint32_t)part_w[q]), M);
  };
  float S = 0.0f;
  if (K <= 8) {
    for (int q = 0; q < K; ++q) S += part_sum_at(q);
  } else {  // four sums side by side: fewer roundings at the size of the whole
    float S1 = 0.0f, S2 = 0.0f, S3 = 0.0f;
    int q = 0;
    for (; q + 3 < K; q += 4) {
      S += part_sum_at(q);
      S1 += part_sum_at(q + 1);
      S2 += part_sum_at(q + 2);
      S3 += part_sum_at(q + 3);
    }
    for (; q < K; ++q) S += part_sum_at(q);
    S = (S + S1) + (S2 + S3);
  }
  const float logsum = LOG ? sa_logf(S) : 0.0f;
  const float inv = LOG ? 0.0f : 1.0f / S;
  const float Mb = M == -__builtin_inff() ? 0.0f : M;
  opaque<kFwdNV>(x);
  TO* dst = out + (int64_t)row * cols;
  fwd_split_out<TI, TO, LOG>(x, dst, base, end, M, logsum, Mb, inv);
  if constexpr (RAGGED) {
    const int64_t i = (int64_t)nvec * V + threadIdx.x;
    if (part == K - 1 && i < cols)
      dst[i] = from_arith<TO>(LOG ? (xt - M) - logsum : __builtin_amdgcn_exp2f((xt - Mb) * kLog2e) * inv);
  }
}

template <typename TG, bool WHOLE>
__device__ __forceinline__ float thread_sum(const uint4 (&g)[kBwdNV], int base, int nvec) {
  constexpr int V = VecOf<TG>::V;
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < kBwdNV; ++j)
    if (WHOLE || base + (int)threadIdx.x + j * kSplitBlock < nvec) {
#pragma unroll
      for (int k = 0; k < V; ++k) s += elem_f<TG>(g[j], k);
    }
  return s;
}

// Sum of one part of grad, the same in every thread.
template <typename TG>
__device__ __forceinline__ uint64_t part_sum(uint4 (&g)[kBwdNV], int base, int nvec, float* lds) {
  float s = base + kSplitBlock * kBwdNV <= nvec ? thread_sum<TG, true>(g, base, nvec)
                                                : thread_sum<TG, false>(g, base, nvec);
  s = wave_sum(s);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = s;
  __syncthreads();
  return (uint64_t)__float_as_uint(block_sum(lds));
}

template <typename TG, typename TO, bool WHOLE, bool RAGGED>
__device__ __forceinline__ void bwd_split_out(const uint4 (&gv)[kBwdNV], const uint4 (&yv)[kBwdNV],
                                              TO* dst, const SplitRow& r, int64_t cols, int base, int nvec,
                                              float S) {
  constexpr int V = VecOf<TG>::V;
#pragma unroll
  for (int j = 0; j < kBwdNV; ++j) {
    const int v = base + (int)threadIdx.x + j * kSplitBlock;
    if (WHOLE || v < nvec) {
      float f[V];
#pragma unroll
      for (int k = 0; k < V; ++k)
        f[k] = fmaf(-__builtin_amdgcn_exp2f(elem_f<TG>(yv[j], k) * kLog2e), S, elem_f<TG>(gv[j], k));
      split_store<TG, TO, RAGGED>(dst, r, cols, v, f);
    }
  }
}

template <typename TG, typename TO, bool RAGGED>
__global__ void __launch_bounds__(kSplitBlock, 8)
k_lsm_bwd_split(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, int64_t cols, int K,
                int plen, uint64_t* __restrict__ slots, uint32_t* __restrict__ done, uint32_t spin_limit) {
  constexpr int V = VecOf<TG>::V;
  __shared__ float lds[kSplitNW];
  __shared__ uint64_t part_w[kSplitMaxK];
  __shared__ uint32_t lds_missing;
  const int row = (int)(blockIdx.x / (unsigned)K);
  const int part = (int)(blockIdx.x - (unsigned)row * (unsigned)K);
  const SplitRow r = split_row<TG, RAGGED>(RAGGED ? grid_off<TG, VecOf<TG>::V>(grad + (int64_t)row * cols, cols) : 0, cols);
  const int nvec = r.nvec;
  const int base = part * plen;
  const int end = min(base + plen, nvec);
  const TG* g = grad + (int64_t)row * cols - r.o;
  const TG* y = outp + (int64_t)row * cols - r.o;
  uint4 gv[kBwdNV], yv[kBwdNV];
  split_load_grid<TG, kBwdNV, RAGGED>(gv, g, r, cols, base, end);
  split_load_grid<TG, kBwdNV, RAGGED>(yv, y, r, cols, base, end);
  // every load of the part in flight before the sum: float32 parts, whose
  // sum is short, otherwise had it scheduled between the loads (75.2 ->
  // 76.3 % on [8192, 64128], 72.8 -> 75.3 % on [16384, 28672]; bf16 rows
  // unchanged)
  opaque<kBwdNV>(gv);
  opaque<kBwdNV>(yv);
  const uint64_t mine = part_sum<TG>(gv, base, end, lds);
  opaque<kBwdNV>(gv);
  uint64_t* rs = slots + (int64_t)row * K;
  if (threadIdx.x == 0) slot_publish(rs + part, mine);
  uint32_t miss = split_wait(rs, K, spin_limit, part_w, &lds_missing);
  split_release(rs, done + row, K);
  if (miss) {  // uniform; the own part is loaded again afterwards, so the fallback reuses its registers
    do {
      const int q = __builtin_ctz(miss);
      miss &= miss - 1;
      const int qb = q * plen, qe = min(qb + plen, nvec);
      split_load_grid<TG, kBwdNV, RAGGED>(gv, g, r, cols, qb, qe);
      const uint64_t w = part_sum<TG>(gv, qb, qe, lds);
      if (threadIdx.x == 0) part_w[q] = w;
    } while (miss);
    split_load_grid<TG, kBwdNV, RAGGED>(gv, g, r, cols, base, end);
  }
  __syncthreads();
  float S = __uint_as_float((uint32_t)part_w[0]);
  for (int q = 1; q < K; ++q) S += __uint_as_float((uint32_t)part_w[q]);
  opaque<kBwdNV>(gv);
  opaque<kBwdNV>(yv);
  TO* dst = gin + (int64_t)row * cols - r.o;
  if (base + kSplitBlock * kBwdNV <= end) bwd_split_out<TG, TO, true, RAGGED>(gv, yv, dst, r, cols, base, end, S);
  else bwd_split_out<TG, TO, false, RAGGED>(gv, yv, dst, r, cols, base, end, S);
}

__global__ void __launch_bounds__(kBlock) k_split_init(uint64_t* slots, uint32_t* done, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) {
    slots[i] = 0;
    done[i] = 0u;
  }
}

// The slot buffers live in the library's own device memory (a copy on every
// device), so the entry points allocate nothing.  Host code reaches them only
// through the addresses hipGetSymbolAddress gives on each device.
static __device__ __align__(256) uint64_t g_split_slots[kSplitBuffers * kSplitSlots];
static __device__ __align__(256) uint32_t g_split_done[kSplitBuffers * kSplitSlots];

struct SplitScratch {
  uint64_t* slots = nullptr;
  uint32_t* done = nullptr;
};

// The split kernels' buffer for (current device, st): one of the device's
// kSplitBuffers, given to the stream on its first split call (and cleared on
// it then) and kept; false when the split path is switched off
// (SUPA_AMD_ROW_SPLIT=0), the stream is capturing a graph, or the device has
// given out every buffer -- the caller then takes the one-row kernels.
inline bool split_scratch(hipStream_t st, SplitScratch& out, uint32_t& spin_limit) {
  const char* e = std::getenv("SUPA_AMD_ROW_SPLIT");
  if (e && e[0] == '0') return false;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) return false;
  const char* sp = std::getenv("SUPA_AMD_ROW_SPLIT_SPIN");
  spin_limit = sp ? (uint32_t)std::strtoul(sp, nullptr, 10) : kSplitSpinDefault;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, SplitScratch> bufs;
  static std::map<int, std::pair<SplitScratch, int>> base;  // device -> (symbol addresses, buffers given out)
  std::lock_guard<std::mutex> lock(mu);
  const auto key = std::make_pair(dev, st);
  auto it = bufs.find(key);
  if (it != bufs.end()) {
    out = it->second;
    return true;
  }
  auto bt = base.find(dev);
  if (bt == base.end()) {
    SplitScratch a;
    void* ps = nullptr;
    void* pd = nullptr;
    if (hipGetSymbolAddress(&ps, HIP_SYMBOL(g_split_slots)) != hipSuccess ||
        hipGetSymbolAddress(&pd, HIP_SYMBOL(g_split_done)) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    a.slots = static_cast<uint64_t*>(ps);
    a.done = static_cast<uint32_t*>(pd);
    bt = base.emplace(dev, std::make_pair(a, 0)).first;
  }
  if (bt->second.second >= kSplitBuffers) return false;
  const int idx = bt->second.second;
  SplitScratch b;
  b.slots = bt->second.first.slots + (int64_t)idx * kSplitSlots;
  b.done = bt->second.first.done + (int64_t)idx * kSplitSlots;
  k_split_init<<<(unsigned)(kSplitSlots / kBlock), kBlock, 0, st>>>(b.slots, b.done, kSplitSlots);
  if (hipGetLastError() != hipSuccess) return false;
  ++bt->second.second;
  bufs.emplace(key, b);
  out = b;
  return true;
}

// Parts per row for the split kernels (at most `part` vectors each), 0 when
// the row takes another kernel: 2 to kSplitMaxK parts, inputs that do not
// overlap the output.
inline int split_parts(int64_t nvec, int part, const void* a, const void* b, int64_t a_bytes, const void* o,
                       int64_t o_bytes) {
  const int64_t K = (nvec + part - 1) / part;
  if (K < 2 || K > kSplitMaxK) return 0;
  auto overlap = [](const void* x, int64_t xb, const void* y, int64_t yb) {
    const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), y0 = reinterpret_cast<uintptr_t>(y);
    return x0 < y0 + (uintptr_t)yb && y0 < x0 + (uintptr_t)xb;
  };
  if (overlap(a, a_bytes, o, o_bytes) || (b && overlap(b, a_bytes, o, o_bytes))) return 0;
  return (int)K;
}

// Vectors per part when a row of nvec vectors is split in K parts of at most
// `part`: the row spread evenly, rounded up to whole wavefronts (a part's
// guards are then uniform in every wavefront but the last part's), or, from
// `whole_from` parts on, full parts and a short last one (the backward's
// whole parts run unguarded loops).  Measured on MI355X, % of the HBM
// roofline, even parts / full parts and a short last / one-row kernel:
// forward bf16 [8192, 128256] (7 parts) 77.6 / 76.7 / 71.8, [16384, 65536]
// (4) 79.0 / 73.5 / 73.1, [16384, 50304] (3) 78.8 / 77.9 / 70.2; backward
// bf16 [16384, 50304] (4) 79.8 / 74.9 / 75.3, [2048, 57344] (4) 78.3 /
// 76.3 / 73.6, float32 [5120, 50304] (7) 68.4 / 71.2 / 72.5 (bf16 rows of
// those 12576 vectors 74.6 / 76.0 / 74.0).
inline int split_part_len(int64_t nvec, int K, int part, int whole_from) {
  if (K >= whole_from) return part;
  return (int)(((nvec + K - 1) / K + 63) / 64 * 64);
}

// The most vectors a backward row of cols elements takes: those of the line
// grid when cols is no multiple of the vector.
inline int64_t split_vecs(int64_t cols, int v) { return cols % v == 0 ? cols / v : (cols + 8 * v - 1 + v - 1) / v; }

// Aligned backward rows of 513 to 2048 whole vectors stay on the unguarded
// 1024-thread kernels (bf16 [8192, 10000] 78 us against 88 on k_row_bwd,
// [4096, 16384] 62 against 65; float32 rows within 2 %).
// Not past 2^22 rows, 2^32 threads.
inline bool bwd_reg_rows(int64_t rows, int64_t cols, int v) {
  return cols % v == 0 && cols / v > 512 && cols / v <= 2 * kRowBlock && rows < (int64_t(1) << 22);
}

template <bool LOG>
int softmax_forward(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t rows, int64_t cols,
                    void* stream) {
  if (!in || !out || rows < 0 || cols < 0 || rows >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (rows == 0 || cols == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_float_storage(in_dtype, [&](auto* ti) -> int {
    return with_float_storage(out_dtype, [&](auto* to) -> int {
      using TI = std::remove_pointer_t<decltype(ti)>;
      using TO = std::remove_pointer_t<decltype(to)>;
      if constexpr (!std::is_same<TI, TO>::value && !std::is_same<TO, float>::value) return SUPA_AMD_EDTYPE;
      else {
      constexpr int V = VecOf<TI>::V;
      const TI* pi = static_cast<const TI*>(in);
      TO* po = static_cast<TO*>(out);
      // aligned float32 rows of 1025 to 2048 vectors: the persistent kernel
      // ([8192, 8192] 92 us, k_row_fwd 94)
      if constexpr (sizeof(TI) == 4) {
        if (cols % V == 0 && cols / V > kRowBlock && cols / V <= 2 * kRowBlock && aligned(in, 16) && aligned(out, 16)) {
          k_lsm_fwd_reg<TI, TO, 2, LOG>
              <<<(unsigned)std::min<int64_t>(rows, kLsmGrid), kRowBlock, 0, st>>>(pi, po, rows, cols);
          return launch_status();
        }
      }
      int rc;
      if (row_split<V, kSplitBlock * kFwdNV, false>(
              rows, cols, rc, [&](auto vw, auto g, auto nv, int64_t r0, int64_t nr, unsigned blocks) {
                k_row_fwd<TI, TO, vw.value, g.value, nv.value, LOG>
                    <<<blocks, row_block<g.value>(), 0, st>>>(pi + r0 * cols, po + r0 * cols, nr, (int)cols);
                return launch_status();
              }))
        return rc;
      const int64_t nvec = (cols + V - 1) / V;
      const int K = split_parts(nvec, kSplitBlock * kFwdNV, in, nullptr, rows * cols * (int64_t)sizeof(TI), out,
                                rows * cols * (int64_t)sizeof(TO));
      SplitScratch sb;
      uint32_t spin = 0;
      if (K > 0 && split_scratch(st, sb, spin)) {
        const int plen = split_part_len(nvec, K, kSplitBlock * kFwdNV, kSplitMaxK + 1);
        const int64_t chunk = kSplitSlots / K;
        for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
          const int64_t nr = std::min(chunk, rows - r0);
          if (cols % V)
            k_lsm_fwd_split<TI, TO, LOG, true><<<(unsigned)(nr * K), kSplitBlock, 0, st>>>(
                pi + r0 * cols, po + r0 * cols, cols, K, plen, sb.slots, sb.done, spin);
          else
            k_lsm_fwd_split<TI, TO, LOG, false><<<(unsigned)(nr * K), kSplitBlock, 0, st>>>(
                pi + r0 * cols, po + r0 * cols, cols, K, plen, sb.slots, sb.done, spin);
        }
        return launch_status();
      }
      if (cols % V == 0 && aligned(in, 16) && aligned(out, 16) && nvec <= 16 * kRowBlock) {
        const int vpt = (int)((nvec + kRowBlock - 1) / kRowBlock);
        const unsigned grid = (unsigned)std::min<int64_t>(rows, kLsmGrid);
        if (vpt <= 4) k_lsm_fwd_reg<TI, TO, 4, LOG><<<grid, kRowBlock, 0, st>>>(pi, po, rows, cols);
        else if (vpt <= 8) k_lsm_fwd_reg<TI, TO, 8, LOG><<<grid, kRowBlock, 0, st>>>(pi, po, rows, cols);
        else k_lsm_fwd_reg<TI, TO, 16, LOG><<<grid, kRowBlock, 0, st>>>(pi, po, rows, cols);
        return launch_status();
      }
      k_lsm_fwd_stream<TI, TO, LOG><<<(unsigned)rows, kRowBlock, 0, st>>>(pi, po, cols);
      return launch_status();
      }
    });
  });
}

}  // namespace sa

using namespace sa;

extern "C" {

int supa_amd_log_softmax_forward(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t rows,
                                 int64_t cols, void* stream) {
  return softmax_forward<true>(in, in_dtype, out, out_dtype, rows, cols, stream);
}

int supa_amd_softmax_forward(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t rows,
                             int64_t cols, void* stream) {
  return softmax_forward<false>(in, in_dtype, out, out_dtype, rows, cols, stream);
}

int supa_amd_log_softmax_backward(const void* grad, const void* output, int32_t gy_dtype, void* grad_in,
                                  int32_t gin_dtype, int64_t rows, int64_t cols, void* stream) {
  if (!grad || !output || !grad_in || rows < 0 || cols < 0 || rows >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (rows == 0 || cols == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_float_storage(gy_dtype, [&](auto* tg) -> int {
    return with_float_storage(gin_dtype, [&](auto* to) -> int {
      using TG = std::remove_pointer_t<decltype(tg)>;
      using TO = std::remove_pointer_t<decltype(to)>;
      if constexpr (!std::is_same<TG, TO>::value && !std::is_same<TO, float>::value) return SUPA_AMD_EDTYPE;
      else {
      constexpr int V = VecOf<TG>::V;
      const TG* pg = static_cast<const TG*>(grad);
      const TG* py = static_cast<const TG*>(output);
      TO* po = static_cast<TO*>(grad_in);
      const bool al = aligned(grad, 16) && aligned(output, 16) && aligned(grad_in, 16);
      const int64_t nvec = split_vecs(cols, V);
      if (al && bwd_reg_rows(rows, cols, V)) {
        if (nvec <= kRowBlock) k_lsm_bwd_reg<TG, TO, 1><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        else k_lsm_bwd_reg<TG, TO, 2><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        return launch_status();
      }
      int rc;
      if (row_split<V, kSplitBlock * kBwdNV, true>(
              rows, cols, rc, [&](auto vw, auto g, auto nv, int64_t r0, int64_t nr, unsigned blocks) {
                k_row_bwd<TG, TO, vw.value, g.value, nv.value, true><<<blocks, row_block<g.value>(), 0, st>>>(
                    pg + r0 * cols, py + r0 * cols, po + r0 * cols, nr, (int)cols);
                return launch_status();
              }))
        return rc;
      const int K = al ? split_parts(nvec, kSplitBlock * kBwdNV, grad, output, rows * cols * (int64_t)sizeof(TG),
                                     grad_in, rows * cols * (int64_t)sizeof(TO))
                       : 0;
      SplitScratch sb;
      uint32_t spin = 0;
      if (K > 0 && split_scratch(st, sb, spin)) {
        const int plen = split_part_len(nvec, K, kSplitBlock * kBwdNV, 6);
        const int64_t chunk = kSplitSlots / K;
        for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
          const int64_t nr = std::min(chunk, rows - r0);
          if (cols % V)
            k_lsm_bwd_split<TG, TO, true><<<(unsigned)(nr * K), kSplitBlock, 0, st>>>(
                pg + r0 * cols, py + r0 * cols, po + r0 * cols, cols, K, plen, sb.slots, sb.done, spin);
          else
            k_lsm_bwd_split<TG, TO, false><<<(unsigned)(nr * K), kSplitBlock, 0, st>>>(
                pg + r0 * cols, py + r0 * cols, po + r0 * cols, cols, K, plen, sb.slots, sb.done, spin);
        }
        return launch_status();
      }
      if (al && cols % V == 0 && nvec <= 16 * kRowBlock) {
        const int vpt = (int)((nvec + kRowBlock - 1) / kRowBlock);
        if (vpt <= 4) k_lsm_bwd_reg<TG, TO, 4><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        else if (vpt <= 8) k_lsm_bwd_reg<TG, TO, 8><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        else k_lsm_bwd_reg<TG, TO, 16><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        return launch_status();
      }
      k_bwd_stream<TG, TO, true><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
      return launch_status();
      }
    });
  });
}

int supa_amd_softmax_backward(const void* grad, const void* output, int32_t gy_dtype, void* grad_in,
                              int32_t gin_dtype, int64_t rows, int64_t cols, void* stream) {
  if (!grad || !output || !grad_in || rows < 0 || cols < 0 || rows >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (rows == 0 || cols == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_float_storage(gy_dtype, [&](auto* tg) -> int {
    return with_float_storage(gin_dtype, [&](auto* to) -> int {
      using TG = std::remove_pointer_t<decltype(tg)>;
      using TO = std::remove_pointer_t<decltype(to)>;
      if constexpr (!std::is_same<TG, TO>::value && !std::is_same<TO, float>::value) return SUPA_AMD_EDTYPE;
      else {
      constexpr int V = VecOf<TG>::V;
      const bool reg_ok = (cols % V) == 0 && aligned(grad, 16) && aligned(output, 16) && aligned(grad_in, V * sizeof(TO)) &&
                          (cols / V) <= 8 * kRowBlock;
      const TG* pg = static_cast<const TG*>(grad);
      const TG* py = static_cast<const TG*>(output);
      TO* po = static_cast<TO*>(grad_in);
      if (reg_ok && bwd_reg_rows(rows, cols, V)) {
        if (cols / V <= kRowBlock) k_sm_bwd_reg<TG, TO, 1><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        else k_sm_bwd_reg<TG, TO, 2><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        return launch_status();
      }
      int rc;
      if (row_split<V, kSplitBlock * kBwdNV, true>(
              rows, cols, rc, [&](auto vw, auto g, auto nv, int64_t r0, int64_t nr, unsigned blocks) {
                k_row_bwd<TG, TO, vw.value, g.value, nv.value, false><<<blocks, row_block<g.value>(), 0, st>>>(
                    pg + r0 * cols, py + r0 * cols, po + r0 * cols, nr, (int)cols);
                return launch_status();
              }))
        return rc;
      if (reg_ok) {
        const int64_t nvec = cols / V;
        const int vpt = (int)((nvec + kRowBlock - 1) / kRowBlock);
        if (vpt <= 4) k_sm_bwd_reg<TG, TO, 4><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        else k_sm_bwd_reg<TG, TO, 8><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
        return launch_status();
      }
      k_bwd_stream<TG, TO, false><<<(unsigned)rows, kRowBlock, 0, st>>>(pg, py, po, cols);
      return launch_status();
      }
    });
  });
}

}  // extern "C"
