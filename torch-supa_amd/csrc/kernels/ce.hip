// Fused cross-entropy over a contiguous [n, c] logit matrix with int64
// targets and ignore_index: the forward reads the logits once and keeps one
// float32 log-sum-exp per row; the backward reads the logits once more and
// writes grad = (softmax - onehot) * g in one pass.  12 N C bytes of the
// log_softmax + nll_loss decomposition (bf16) become 6 N C.
//
// Forward, per row (one 256-thread workgroup; rows in a grid of n):
//   each thread folds its 16-byte vectors into an online (max, sum exp) pair,
//   pairs combine across the wavefront and the workgroup, lse = m + log(s),
//   loss = lse - x[t] in float32.  Rows whose target is ignore_index get
//   loss 0 and are not counted.  Stage 2 (one workgroup): the sum over rows
//   in a fixed order, and for mean the division by the kept-row count (NaN
//   for none, as CrossEntropyLossKernel.cu:67 / :191-193 of the reference).
// Backward, per (row, 16-byte vector) thread: g_i * (exp(x - lse_i) - [j == t_i]).
//
// Out-of-range targets set *error_flag (when given); their rows count as
// ignored.
//
// Probability targets (a float [n, c] target of the logits' dtype, the
// reference's other fp32 fast-path case): the forward reads logits and
// target once each, folds per thread an online (max m, sum of exp(x - m) s,
// sum of t T, sum of t (x - m) B) state, combines it across the workgroup and
// writes loss = T log(s) - B = sum_j t_j (lse - x_j) with lse and T saved per
// row; the backward writes g_i (exp(x - lse_i) T_i - t) in one pass.
#include "softmax_common.h"

namespace sa {

constexpr int kCeBlock = 256;
// The backward is a pure stream (one vector in, one out per thread): one
// wavefront per workgroup, as the elementwise kernels.
constexpr int kCeBwdBlock = 64;
constexpr int kCeUnroll = 4;  // 16-byte vectors in flight per thread in the forward
constexpr float kCeLog2e = 1.44269504088896340736f;

template <typename T> struct CeVec {
  static constexpr int V = 16 / sizeof(T);
};

template <typename T>
__device__ __forceinline__ float ce_elem(const uint4& w, int k) {
  if constexpr (std::is_same<T, float>::value) {
    return __uint_as_float(k == 0 ? w.x : (k == 1 ? w.y : (k == 2 ? w.z : w.w)));
  } else {
    const int wi = k >> 1;
    const uint32_t u = wi == 0 ? w.x : (wi == 1 ? w.y : (wi == 2 ? w.z : w.w));
    const uint32_t h = (k & 1) ? (u >> 16) : (u & 0xffffu);
    if constexpr (std::is_same<T, bf16>::value) return __uint_as_float(h << 16);
    else return (float)__builtin_bit_cast(f16, (uint16_t)h);
  }
}

__device__ __forceinline__ bool ce_kept(int64_t t, int64_t c, int64_t ignore_index) {
  return t != ignore_index && t >= 0 && t < c;
}

// loss_rows[i] (float32): the row's loss, 0 for an ignored row.  lse[i]: the
// row's log-sum-exp (0 for an ignored row).  out_none (may be null): the loss
// in the logits dtype, for reduction 'none'.
// Rows stream as 16-byte vectors at any alignment, their last c mod V elements
// one to a thread (rows of odd length took two exponentials per element
// through the pairwise update: float32 [4096, 50257] 259 us, 130 now, HBM
// bound at 6.3 TB/s; with the gradient 900, 384).
// G threads share a row: a wavefront (four rows a workgroup) up to
// kCeWaveVecs vectors, else the workgroup (float32 [65536, 1000] 109 us with
// a workgroup per row, 46 with a wavefront; from 257 vectors on a wavefront
// would hold a second batch of loads while the next row's wait).
constexpr int kCeWaveVecs = 64 * kCeUnroll;
// Workgroups of a launch: HIP takes fewer than 2^32 threads.
constexpr int64_t kCeSlab = ((int64_t(1) << 32) - 1) / kCeBlock;

template <typename T, int G>
__global__ void __launch_bounds__(kCeBlock)
k_ce_fwd(const T* __restrict__ x, const int64_t* __restrict__ target, int64_t n, int64_t c, int64_t ignore_index,
         float* __restrict__ loss_rows, float* __restrict__ lse, T* __restrict__ out_none, int32_t* error_flag) {
  constexpr int V = CeVec<T>::V;
  constexpr int NW = G / 64;
  const int l = threadIdx.x & (G - 1);
  int64_t row = blockIdx.x;
  if constexpr (G < kCeBlock) row = (int64_t)blockIdx.x * (kCeBlock / G) + threadIdx.x / G;
  if (row >= n) return;
  const T* xr = x + row * c;
  const int64_t nvec = c / V;
  // a wavefront's rows issue their loads before the target arrives (an
  // ignored row then reads logits it does not need)
  uint4 first[kCeUnroll];
  if constexpr (G < kCeBlock) {
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u)
      if (l + u * G < nvec) first[u] = ld_any_stream(xr + (int64_t)(l + u * G) * V);
  }
  const int64_t t = target[row];
  if (!ce_kept(t, c, ignore_index)) {  // the whole row's threads
    if (l == 0) {
      if (t != ignore_index && error_flag) *error_flag = 1;
      loss_rows[row] = 0.0f;
      lse[row] = 0.0f;
      if (out_none) out_none[row] = from_arith<T>(0.0f);
    }
    return;
  }
  float xt = 0.0f;  // a wavefront's, early; a workgroup reads it at the end
  if constexpr (G < kCeBlock) xt = (float)to_arith(xr[t]);
  float m = -__builtin_inff(), s = 0.0f;
  for (int64_t v0 = l; v0 < nvec; v0 += (int64_t)G * kCeUnroll) {
    uint4 w[kCeUnroll];
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u) {
      const int64_t v = v0 + (int64_t)u * G;
      if constexpr (G < kCeBlock) {  // the row's only step
        w[u] = first[u];
      } else {
        if (v < nvec) w[u] = ld_any_stream(xr + v * V);
      }
    }
    float mb = -__builtin_inff();
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u) {
      if (v0 + (int64_t)u * G < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) mb = fmaxf(mb, ce_elem<T>(w[u], k));
      }
    }
    // fmaxf passes over a NaN, so M says nothing of them: the sum is always
    // taken, and a NaN (or +inf) logit makes it, and the row's loss, NaN
    const float M = fmaxf(m, mb), base = M == -__builtin_inff() ? 0.0f : M;
    float sb = 0.0f;
#pragma unroll
    for (int u = 0; u < kCeUnroll; ++u) {
      if (v0 + (int64_t)u * G < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) sb += __builtin_amdgcn_exp2f((ce_elem<T>(w[u], k) - base) * kCeLog2e);
      }
    }
    s = lse_rescale(s, m, M) + sb;
    m = M;
  }
  // the elements after the whole vectors
  for (int64_t j = nvec * V + l; j < c; j += G) {
    const float xv = (float)to_arith(xr[j]);
    const float M = fmaxf(m, xv), base = M == -__builtin_inff() ? 0.0f : M;
    s = lse_rescale(s, m, M) + __builtin_amdgcn_exp2f((xv - base) * kCeLog2e);
    m = M;
  }
  lanes_lse<64>(m, s);
  if constexpr (NW > 1) {
    __shared__ float lds_m[NW];
    __shared__ float lds_s[NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
      lds_m[wave] = m;
      lds_s[wave] = s;
    }
    __syncthreads();
    m = lds_m[lane & (NW - 1)];
    s = lds_s[lane & (NW - 1)];
    lanes_lse<NW>(m, s);
  }
  if (l == 0) {
    const float lg = m + sa_logf(s);
    if constexpr (G == kCeBlock) xt = (float)to_arith(xr[t]);
    const float loss = lg - xt;
    loss_rows[row] = loss;
    lse[row] = lg;
    if (out_none) out_none[row] = from_arith<T>(loss);
  }
}

// Stage 2: sum of the row losses and the kept-row count, fixed order
// (target null: every row counts, the probability-target form).  Up to
// kCeSumRows rows one workgroup, all loads in flight; of more, a first launch
// (PART) sums whole chunks of that many, each workgroup leaving (sum, count) in
// its chunk's first two loss slots, which nobody else reads, and the last
// launch adds those and the rows after the chunks.
constexpr int kCeSumBlock = 1024;
constexpr int64_t kCeSumRows = 8192;

template <typename T, bool PART>
__global__ void __launch_bounds__(kCeSumBlock)
k_ce_final(float* __restrict__ loss_rows, const int64_t* __restrict__ target, int64_t n, int64_t nparts, int64_t c,
           int64_t ignore_index, int mean, T* __restrict__ out, float* __restrict__ count) {
  constexpr int NW = kCeSumBlock / 64;
  constexpr int U = (int)(kCeSumRows / kCeSumBlock);
  __shared__ float lds_v[NW];
  __shared__ float lds_c[NW];
  float v = 0.0f, k = 0.0f;
  if constexpr (!PART) {
    for (int64_t p = threadIdx.x; p < nparts; p += kCeSumBlock) {
      v += loss_rows[p * kCeSumRows];
      k += loss_rows[p * kCeSumRows + 1];
    }
  }
  const int64_t i0 = (PART ? (int64_t)blockIdx.x : nparts) * kCeSumRows + threadIdx.x;
  float lv[U];
  int64_t tg[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t i = i0 + (int64_t)u * kCeSumBlock;
    lv[u] = i < n ? loss_rows[i] : 0.0f;
    tg[u] = i < n && target ? target[i] : ignore_index;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (i0 + (int64_t)u * kCeSumBlock < n) {
      v += lv[u];
      k += (!target || ce_kept(tg[u], c, ignore_index)) ? 1.0f : 0.0f;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v += __shfl_xor(v, off, 64);
    k += __shfl_xor(k, off, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    lds_v[wave] = v;
    lds_c[wave] = k;
  }
  __syncthreads();
  // the wavefronts' sums by a tree too: one after another their roundings, at
  // the size of the whole sum, were half of the mean's error
  float sv = lds_v[lane & (NW - 1)], sk = lds_c[lane & (NW - 1)];
#pragma unroll
  for (int off = NW / 2; off > 0; off >>= 1) {
    sv += __shfl_xor(sv, off, 64);
    sk += __shfl_xor(sk, off, 64);
  }
  if (threadIdx.x == 0) {
    if constexpr (PART) {  // every row of the chunk is read: the barrier
      loss_rows[(int64_t)blockIdx.x * kCeSumRows] = sv;
      loss_rows[(int64_t)blockIdx.x * kCeSumRows + 1] = sk;
    } else {
      out[0] = from_arith<T>(mean ? sv / sk : sv);  // 0/0 = NaN for a mean over no rows
      if (count) count[0] = sk;
    }
  }
}

template <typename T>
int ce_final(float* rows, const int64_t* target, int64_t n, int64_t c, int64_t ignore_index, int reduction, T* out,
             float* count, hipStream_t st) {
  const int mean = reduction == SUPA_AMD_REDUCTION_MEAN ? 1 : 0;
  const int64_t nparts = n > kCeSumRows ? n / kCeSumRows : 0;
  if (nparts > 0) {
    k_ce_final<T, true><<<(unsigned)nparts, kCeSumBlock, 0, st>>>(rows, target, n, 0, c, ignore_index, mean, nullptr,
                                                                 nullptr);
    const int rc = launch_status();
    if (rc) return rc;
  }
  k_ce_final<T, false><<<1, kCeSumBlock, 0, st>>>(rows, target, n, nparts, c, ignore_index, mean, out, count);
  return launch_status();
}

// A row's output vectors are those of unaligned.h's grid, which starts
// grid_off elements before the row: its stores, and with the logits at the
// same alignment its loads, are aligned; the first and the last partial vector
// go element by element.
//
// grad[i, :] over a 2-d grid: blockIdx.y = row in the slab, x = column blocks
// of kCeBwdBlock vectors.  WHOLE: rows of whole aligned vectors.  A vector's
// logits load then goes out unconditionally, before the row's target, and the
// scale and lse that depend on it, have arrived (an ignored row then reads
// logits it does not need); waiting for the target first, as the kernel does
// that has partial vectors to tell from whole ones, held it at 75 % of the HBM
// roofline on c3's bf16 rows, against 85 % with the load first (forward and
// backward 1002 us and 921; float32 1837 and 1804).
template <typename T, bool WHOLE>
__global__ void __launch_bounds__(kCeBwdBlock)
k_ce_bwd(const T* __restrict__ grad_out, const T* __restrict__ x, const int64_t* __restrict__ target,
         const float* __restrict__ lse, const float* __restrict__ count, int64_t c, int64_t ignore_index,
         int reduction, T* __restrict__ gx) {
  constexpr int V = CeVec<T>::V;
  const int64_t row = blockIdx.y;
  const T* xr = x + row * c;
  T* dst = gx + row * c;
  const int64_t col0 = ((int64_t)blockIdx.x * kCeBwdBlock + threadIdx.x) * V - (WHOLE ? 0 : grid_off<T, V>(dst, c));
  if (col0 >= c) return;
  Vec<T, V> w;
  const bool whole = WHOLE || (col0 >= 0 && col0 + V <= c);
  if (whole) w = ld_vec_any<true, T, V>(xr + col0);
  const int64_t t = target[row];
  const bool kept = ce_kept(t, c, ignore_index);
  float g = 0.0f;
  if (kept) {
    if (reduction == SUPA_AMD_REDUCTION_NONE) g = (float)to_arith(grad_out[row]);
    else if (reduction == SUPA_AMD_REDUCTION_MEAN) g = (float)to_arith(grad_out[0]) / count[0];
    else g = (float)to_arith(grad_out[0]);
  }
  const float l = kept ? lse[row] : 0.0f;
  if (whole) {
    // p g everywhere, (p - 1) g at the target: the one thread of the row that
    // holds the target patches its element in a branch, so the other threads
    // spend no compare or select per element (the same values as
    // (p - [j == t]) g; ignored rows, uniform in the workgroup, store zeros)
    Vec<T, V> o;
    if (kept) {
      float p[V];
#pragma unroll
      for (int k = 0; k < V; ++k) p[k] = __builtin_amdgcn_exp2f(((float)to_arith(w.v[k]) - l) * kCeLog2e);
      float r[V];
#pragma unroll
      for (int k = 0; k < V; ++k) r[k] = p[k] * g;
      if ((uint64_t)(t - col0) < (uint64_t)V) {
#pragma unroll
        for (int k = 0; k < V; ++k)
          if (col0 + k == t) r[k] = (p[k] - 1.0f) * g;
      }
#pragma unroll
      for (int k = 0; k < V; ++k) o.v[k] = from_arith<T>(r[k]);
    } else {
#pragma unroll
      for (int k = 0; k < V; ++k) o.v[k] = from_arith<T>(0.0f);
    }
    st_vec_any<T, V>(dst + col0, o);
  } else {
    for (int k = col0 < 0 ? (int)-col0 : 0; k < V && col0 + k < c; ++k) {
      float r = 0.0f;
      if (kept) {
        const float p = __builtin_amdgcn_exp2f(((float)to_arith(xr[col0 + k]) - l) * kCeLog2e);
        r = (p - (col0 + k == t ? 1.0f : 0.0f)) * g;
      }
      dst[col0 + k] = from_arith<T>(r);
    }
  }
}

// ------------------------------------------------- probability targets
// Online state of a row: max m, s = sum exp(x - m), T = sum t,
// B = sum t (x - m).  (+) of two states rebases both to M = max(m, m2):
// s -> s e^{m - M}, B -> B + T (m - M).  A state whose elements are all -inf
// keeps m = -inf, s = 0 and B = sum t x (-inf, or NaN where a t is 0), which
// no rebase changes: its elements add t (lse - x) = +inf (or NaN for t = 0)
// to the loss, as -t log_softmax(x) does in the decomposition.
struct CeProbState {
  float m, s, T, B;
};
__device__ __forceinline__ CeProbState ce_prob_elem(float x, float t) {
  if (x == -__builtin_inff()) return CeProbState{x, 0.0f, t, t * x};
  return CeProbState{x, 1.0f, t, 0.0f};
}
__device__ __forceinline__ void ce_prob_combine(CeProbState& a, const CeProbState& b) {
  const float M = fmaxf(a.m, b.m);
  const bool fa = a.m != -__builtin_inff(), fb = b.m != -__builtin_inff();
  const float ea = fa ? __builtin_amdgcn_exp2f((a.m - M) * kCeLog2e) : 0.0f;
  const float eb = fb ? __builtin_amdgcn_exp2f((b.m - M) * kCeLog2e) : 0.0f;
  const float Ba = fa ? fmaf(a.T, a.m - M, a.B) : a.B;
  const float Bb = fb ? fmaf(b.T, b.m - M, b.B) : b.B;
  a.s = a.s * ea + b.s * eb;
  a.B = Ba + Bb;
  a.T = a.T + b.T;
  a.m = M;
}

// loss_rows[i] = T log(s) - B (float32); lse[i] = m + log(s); tsum[i] = T;
// out_none (may be null): the loss in the logits dtype.
template <typename T>
__global__ void __launch_bounds__(kCeBlock)
k_ce_prob_fwd(const T* __restrict__ x, const T* __restrict__ tgt, int64_t c, float* __restrict__ loss_rows,
              float* __restrict__ lse, float* __restrict__ tsum, T* __restrict__ out_none) {
  constexpr int V = CeVec<T>::V;
  constexpr int NW = kCeBlock / 64;
  constexpr int U = 2;  // vectors of each stream in flight per thread
  __shared__ CeProbState lds[NW];
  const int64_t row = blockIdx.x;
  const T* xr = x + row * c;
  const T* tr = tgt + row * c;
  const int64_t nvec = c / V;
  CeProbState st{-__builtin_inff(), 0.0f, 0.0f, 0.0f};
  for (int64_t v0 = threadIdx.x; v0 < nvec; v0 += (int64_t)kCeBlock * U) {
    uint4 wx[U], wt[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t v = v0 + (int64_t)u * kCeBlock;
      if (v < nvec) {
        wx[u] = ld_any_stream(xr + v * V);
        wt[u] = ld_any_stream(tr + v * V);
      }
    }
    float mb = -__builtin_inff();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kCeBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) mb = fmaxf(mb, ce_elem<T>(wx[u], k));
      }
    // every value so far -inf, or NaN: s stays 0, or NaN; B = sum t x
    const float M = fmaxf(st.m, mb), base = M == -__builtin_inff() ? 0.0f : M;
    if (st.m != -__builtin_inff()) {
      st.s *= __builtin_amdgcn_exp2f((st.m - M) * kCeLog2e);
      st.B = fmaf(st.T, st.m - M, st.B);
    }
    st.m = M;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (v0 + (int64_t)u * kCeBlock < nvec) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
          const float xv = ce_elem<T>(wx[u], k), tv = ce_elem<T>(wt[u], k);
          st.s += __builtin_amdgcn_exp2f((xv - base) * kCeLog2e);
          st.T += tv;
          st.B = fmaf(tv, xv - base, st.B);
        }
      }
  }
  // the elements after the whole vectors
  for (int64_t j = nvec * V + threadIdx.x; j < c; j += kCeBlock)
    ce_prob_combine(st, ce_prob_elem((float)to_arith(xr[j]), (float)to_arith(tr[j])));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const CeProbState o{__shfl_xor(st.m, off, 64), __shfl_xor(st.s, off, 64), __shfl_xor(st.T, off, 64),
                        __shfl_xor(st.B, off, 64)};
    ce_prob_combine(st, o);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = st;
  __syncthreads();
  if (threadIdx.x == 0) {
    CeProbState a = lds[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) ce_prob_combine(a, lds[w]);
    const float L = sa_logf(a.s);
    const float loss = fmaf(a.T, L, -a.B);
    loss_rows[row] = loss;
    lse[row] = a.m + L;
    tsum[row] = a.T;
    if (out_none) out_none[row] = from_arith<T>(loss);
  }
}

// grad[i, j] = g_i (exp(x - lse_i) T_i - t_ij); g_i = grad_out[i] (none),
// grad_out[0] (sum) or grad_out[0] / n (mean).
template <typename T>
__global__ void __launch_bounds__(kCeBwdBlock)
k_ce_prob_bwd(const T* __restrict__ grad_out, const T* __restrict__ x, const T* __restrict__ tgt,
              const float* __restrict__ lse, const float* __restrict__ tsum, int64_t c, int reduction, float inv_n,
              T* __restrict__ gx) {
  constexpr int V = CeVec<T>::V;
  const int64_t row = blockIdx.y;
  float g;
  if (reduction == SUPA_AMD_REDUCTION_NONE) g = (float)to_arith(grad_out[row]);
  else if (reduction == SUPA_AMD_REDUCTION_MEAN) g = (float)to_arith(grad_out[0]) * inv_n;
  else g = (float)to_arith(grad_out[0]);
  const float l = lse[row];
  const float Tr = tsum[row];
  const T* xr = x + row * c;
  const T* tr = tgt + row * c;
  T* dst = gx + row * c;
  const int64_t col0 = ((int64_t)blockIdx.x * kCeBwdBlock + threadIdx.x) * V - grid_off<T, V>(dst, c);
  if (col0 >= c) return;
  if (col0 >= 0 && col0 + V <= c) {
    const Vec<T, V> w = ld_vec_any<true, T, V>(xr + col0);
    const Vec<T, V> wt = ld_vec_any<true, T, V>(tr + col0);
    Vec<T, V> o;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const float p = __builtin_amdgcn_exp2f(((float)to_arith(w.v[k]) - l) * kCeLog2e);
      o.v[k] = from_arith<T>(fmaf(p, Tr, -(float)to_arith(wt.v[k])) * g);
    }
    st_vec_any<T, V>(dst + col0, o);
  } else {
    for (int k = col0 < 0 ? (int)-col0 : 0; k < V && col0 + k < c; ++k) {
      const float p = __builtin_amdgcn_exp2f(((float)to_arith(xr[col0 + k]) - l) * kCeLog2e);
      dst[col0 + k] = from_arith<T>(fmaf(p, Tr, -(float)to_arith(tr[col0 + k])) * g);
    }
  }
}

template <typename F>
int with_ce_storage(int dtype, F&& f) {
  switch (dtype) {
    case SUPA_AMD_F32: return f((float*)nullptr);
    case SUPA_AMD_BF16: return f((bf16*)nullptr);
    case SUPA_AMD_F16: return f((f16*)nullptr);
    default: return SUPA_AMD_EDTYPE;
  }
}

}  // namespace sa

using namespace sa;

extern "C" {

int64_t supa_amd_cross_entropy_workspace_bytes(int64_t n) { return n > 0 ? 4 * n : 0; }

int supa_amd_cross_entropy_forward(const void* logits, int32_t dtype, const int64_t* target, int64_t n, int64_t c,
                                   int64_t ignore_index, int reduction, void* out, float* lse, float* count,
                                   void* workspace, int64_t workspace_bytes, int32_t* error_flag, void* stream) {
  if (n < 0 || c <= 0 || n >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (reduction != SUPA_AMD_REDUCTION_NONE && reduction != SUPA_AMD_REDUCTION_MEAN &&
      reduction != SUPA_AMD_REDUCTION_SUM)
    return SUPA_AMD_EINVAL;
  if (!out || (n > 0 && (!logits || !target || !lse))) return SUPA_AMD_EINVAL;
  if (n > 0 && (!workspace || workspace_bytes < supa_amd_cross_entropy_workspace_bytes(n))) return SUPA_AMD_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ce_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    float* rows = static_cast<float*>(workspace);
    T* o = static_cast<T*>(out);
    if (n > 0) {
      const T* x = static_cast<const T*>(logits);
      T* on = reduction == SUPA_AMD_REDUCTION_NONE ? o : nullptr;
      const bool wave = (c + CeVec<T>::V - 1) / CeVec<T>::V <= kCeWaveVecs;
      const int64_t per = wave ? kCeBlock / 64 : 1, slab = per * kCeSlab;
      for (int64_t r0 = 0; r0 < n; r0 += slab) {
        const int64_t nr = std::min(slab, n - r0);
        const unsigned blocks = (unsigned)((nr + per - 1) / per);
        T* const o0 = on ? on + r0 : nullptr;
        if (wave)
          k_ce_fwd<T, 64><<<blocks, kCeBlock, 0, st>>>(x + r0 * c, target + r0, nr, c, ignore_index, rows + r0, lse + r0,
                                                       o0, error_flag);
        else
          k_ce_fwd<T, kCeBlock><<<blocks, kCeBlock, 0, st>>>(x + r0 * c, target + r0, nr, c, ignore_index, rows + r0,
                                                             lse + r0, o0, error_flag);
        const int rc = launch_status();
        if (rc) return rc;
      }
    }
    if (reduction == SUPA_AMD_REDUCTION_NONE) return SUPA_AMD_OK;
    return ce_final<T>(rows, target, n, c, ignore_index, reduction, o, count, st);
  });
}

int supa_amd_cross_entropy_backward(const void* grad_out, const void* logits, int32_t dtype, const int64_t* target,
                                    const float* lse, const float* count, int64_t n, int64_t c, int64_t ignore_index,
                                    int reduction, void* grad_logits, int32_t* error_flag, void* stream) {
  (void)error_flag;  // out-of-range targets were flagged by the forward
  if (n < 0 || c <= 0 || n >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (n == 0) return SUPA_AMD_OK;
  if (!grad_out || !logits || !target || !lse || !grad_logits) return SUPA_AMD_EINVAL;
  if (reduction == SUPA_AMD_REDUCTION_MEAN && !count) return SUPA_AMD_EINVAL;
  if (reduction != SUPA_AMD_REDUCTION_NONE && reduction != SUPA_AMD_REDUCTION_MEAN &&
      reduction != SUPA_AMD_REDUCTION_SUM)
    return SUPA_AMD_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ce_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    constexpr int V = CeVec<T>::V;
    const T* g = static_cast<const T*>(grad_out);
    const T* x = static_cast<const T*>(logits);
    T* gx = static_cast<T*>(grad_logits);
    const bool whole = c % V == 0 && aligned(x, 16) && aligned(gx, 16);
    const unsigned gx_blocks = (unsigned)((grid_vecs<T, V>(gx, c) + kCeBwdBlock - 1) / kCeBwdBlock);
    for (int64_t r0 = 0; r0 < n; r0 += 65535) {
      const int64_t rows = std::min<int64_t>(65535, n - r0);
      const T* gs = reduction == SUPA_AMD_REDUCTION_NONE ? g + r0 : g;
      const dim3 grid(gx_blocks, (unsigned)rows);
      if (whole)
        k_ce_bwd<T, true><<<grid, kCeBwdBlock, 0, st>>>(gs, x + r0 * c, target + r0, lse + r0, count, c, ignore_index,
                                                        reduction, gx + r0 * c);
      else
        k_ce_bwd<T, false><<<grid, kCeBwdBlock, 0, st>>>(gs, x + r0 * c, target + r0, lse + r0, count, c, ignore_index,
                                                         reduction, gx + r0 * c);
      const int rc = launch_status();
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  });
}

int supa_amd_cross_entropy_prob_forward(const void* logits, const void* target, int32_t dtype, int64_t n, int64_t c,
                                        int reduction, void* out, float* lse, float* tsum, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  if (n < 0 || c <= 0 || n >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (reduction != SUPA_AMD_REDUCTION_NONE && reduction != SUPA_AMD_REDUCTION_MEAN &&
      reduction != SUPA_AMD_REDUCTION_SUM)
    return SUPA_AMD_EINVAL;
  if (!out || (n > 0 && (!logits || !target || !lse || !tsum))) return SUPA_AMD_EINVAL;
  if (n > 0 && (!workspace || workspace_bytes < supa_amd_cross_entropy_workspace_bytes(n))) return SUPA_AMD_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ce_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    float* rows = static_cast<float*>(workspace);
    T* o = static_cast<T*>(out);
    if (n > 0) {
      const T* x = static_cast<const T*>(logits);
      const T* t = static_cast<const T*>(target);
      T* on = reduction == SUPA_AMD_REDUCTION_NONE ? o : nullptr;
      for (int64_t r0 = 0; r0 < n; r0 += kCeSlab) {
        k_ce_prob_fwd<T><<<(unsigned)std::min(kCeSlab, n - r0), kCeBlock, 0, st>>>(
            x + r0 * c, t + r0 * c, c, rows + r0, lse + r0, tsum + r0, on ? on + r0 : nullptr);
        const int rc = launch_status();
        if (rc) return rc;
      }
    }
    if (reduction == SUPA_AMD_REDUCTION_NONE) return SUPA_AMD_OK;
    return ce_final<T>(rows, nullptr, n, c, 0, reduction, o, nullptr, st);
  });
}

int supa_amd_cross_entropy_prob_backward(const void* grad_out, const void* logits, const void* target, int32_t dtype,
                                         const float* lse, const float* tsum, int64_t n, int64_t c, int reduction,
                                         void* grad_logits, void* stream) {
  if (n < 0 || c <= 0 || n >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (n == 0) return SUPA_AMD_OK;
  if (!grad_out || !logits || !target || !lse || !tsum || !grad_logits) return SUPA_AMD_EINVAL;
  if (reduction != SUPA_AMD_REDUCTION_NONE && reduction != SUPA_AMD_REDUCTION_MEAN &&
      reduction != SUPA_AMD_REDUCTION_SUM)
    return SUPA_AMD_EINVAL;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_ce_storage(dtype, [&](auto* tag) -> int {
    using T = std::remove_pointer_t<decltype(tag)>;
    constexpr int V = CeVec<T>::V;
    const T* g = static_cast<const T*>(grad_out);
    const T* x = static_cast<const T*>(logits);
    const T* t = static_cast<const T*>(target);
    T* gx = static_cast<T*>(grad_logits);
    const float inv_n = 1.0f / (float)n;
    const unsigned gx_blocks = (unsigned)((grid_vecs<T, V>(gx, c) + kCeBwdBlock - 1) / kCeBwdBlock);
    for (int64_t r0 = 0; r0 < n; r0 += 65535) {
      const int64_t rows = std::min<int64_t>(65535, n - r0);
      const T* gs = reduction == SUPA_AMD_REDUCTION_NONE ? g + r0 : g;
      const dim3 grid(gx_blocks, (unsigned)rows);
      k_ce_prob_bwd<T><<<grid, kCeBwdBlock, 0, st>>>(gs, x + r0 * c, t + r0 * c, lse + r0, tsum + r0, c, reduction,
                                                     inv_n, gx + r0 * c);
      const int rc = launch_status();
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  });
}

}  // extern "C"
