// log_softmax and softmax, forward and backward, along a dim that is not the
// last one: a contiguous [outer, cols, inner] tensor reduced over cols (the
// class dim of [N, C, H, W] logits, where each plane of a class is contiguous).
//
// HBM-bound: the class planes are read once and written once where the
// classes of a position fit the registers of a workgroup.  A workgroup of 256
// threads covers TX vectors of positions (16 bytes of each plane) by TY = 256
// / TX groups of classes; thread (tx, ty) holds classes ty, ty + TY, ... of
// its position vector, NC of them, in registers.  (max, sum of exp) pairs, or
// the backward's sums, meet across the groups by shuffles inside a wavefront
// and through LDS across the four.  More groups for more classes keep NC, and
// so the registers, small: 1 group up to NC classes, 4 up to 4 NC, 16 up to
// 16 NC; more classes than that stream through the 16 groups twice.
//
// A plane whose length is no multiple of the vector: vectors load at element
// alignment (unaligned.h), and the last one of a plane is moved back to end
// at the plane's end and stores only the positions that no other vector
// covers, so every position is written once, by a thread that read it first
// (the output may be the input).
//
// Measured on MI355X, float32 [8, 19, 512, 512] (159 MB a tensor): forward 57
// us (5.6 TB/s), backward 80 us (6.0 TB/s), where copying the planes to rows,
// one 256-thread workgroup per 19-element row, and copying back took 2870 and
// 2440 us; bf16 37 and 42 us (1755 and 1190); planes of 262143 elements 65
// and 93 us; float32 [4, 150, 256, 256] 62 and 94 us (818 and 985).
//
// Replaces _log_softmax.out (NF:3752), _log_softmax_backward_data.out
// (NF:3763), _softmax.out and _softmax_backward_data.out over inner dims
// (upstream SoftMax.cu, spatial kernels).
#include "softmax_common.h"
#include "unaligned.h"

namespace sa {

constexpr int kDimBlock = 256;

// One vector of VW positions of one class as loaded.
template <typename T, int VW> struct DimRaw {
  using type = uint4;
};
template <typename T> struct DimRaw<T, 1> {
  using type = T;
};
template <typename T, int VW> using dim_raw_t = typename DimRaw<T, VW>::type;

template <typename T, int VW, bool STREAM>
__device__ __forceinline__ dim_raw_t<T, VW> dim_load(const T* p) {
  if constexpr (VW == 1) return *p;
  else if constexpr (STREAM) return ld_any_stream(p);
  else return ld_any(p);
}
// The vectors stay packed between phases (opaque in softmax_common.h).
template <typename T, int VW, int NC>
__device__ __forceinline__ void dim_opaque(dim_raw_t<T, VW> (&x)[NC]) {
  if constexpr (VW > 1) opaque<NC>(x);
}
template <typename T, int VW>
__device__ __forceinline__ float dim_elem(const dim_raw_t<T, VW>& w, int k) {
  if constexpr (VW == 1) return (float)to_arith(w);
  else return elem_f<T>(w, k);
}

// Stores elements [skip, VW) of f at p (p is the vector's first element).
template <typename TO, int VW>
__device__ __forceinline__ void dim_store(TO* p, const float (&f)[VW], int skip) {
  if constexpr (VW > 1) {
    if (skip == 0) {
      store_any<TO, VW>(p, f);
      return;
    }
  }
#pragma unroll
  for (int k = 0; k < VW; ++k)
    if (k >= skip) p[k] = from_arith<TO>(f[k]);
}

struct DimGeom {
  uint32_t npos;    // position vectors: outer * ceil(inner / VW)
  uint32_t first;   // the launch's first one
  FastDiv ivec;     // vectors per plane
  uint32_t cols;
  int64_t inner;
};

// This thread's place: the element offset of its vector in class 0, and how
// many of the vector's leading positions belong to the vector before it.
struct DimPlace {
  int64_t base;
  int skip;
  bool valid;
};
template <int VW, int TXL>
__device__ __forceinline__ DimPlace dim_place(const DimGeom& g) {
  const uint32_t tx = threadIdx.x & ((1u << TXL) - 1u);
  const uint32_t p = g.first + blockIdx.x * (1u << TXL) + tx;
  DimPlace r{0, 0, p < g.npos};
  uint32_t o, v;
  g.ivec.divmod(p, o, v);
  int64_t pos = (int64_t)v * VW;
  if (pos + VW > g.inner) {
    r.skip = (int)(pos + VW - g.inner);
    pos = g.inner - VW;
  }
  r.base = (int64_t)o * g.cols * g.inner + pos;
  return r;
}

// The maximum, or the sum, per position over the TY class groups; every thread
// of a position ends with the same values.
template <int VW, int TXL>
__device__ __forceinline__ void dim_max(float (&m)[VW], float* lds) {
  constexpr int TX = 1 << TXL, NW = kDimBlock / 64;
#pragma unroll
  for (int off = TX; off < 64; off <<= 1) {
#pragma unroll
    for (int k = 0; k < VW; ++k) m[k] = fmaxf(m[k], __shfl_xor(m[k], off, 64));
  }
  if constexpr (TX <= 64) {  // the wavefronts hold different classes of the same positions
    const int wave = threadIdx.x >> 6, tx = threadIdx.x & (TX - 1);
    if ((threadIdx.x & 63) < TX) {
#pragma unroll
      for (int k = 0; k < VW; ++k) lds[(wave * VW + k) * TX + tx] = m[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      float M = lds[k * TX + tx];
#pragma unroll
      for (int w = 1; w < NW; ++w) M = fmaxf(M, lds[(w * VW + k) * TX + tx]);
      m[k] = M;
    }
  }
}

// t[0] + ... + t[N - 1] by a tree.
template <int N>
__device__ __forceinline__ float dim_tree(float (&t)[N]) {
#pragma unroll
  for (int h = 1; h < N; h *= 2)
#pragma unroll
    for (int i = 0; i + h < N; i += 2 * h) t[i] += t[i + h];
  return t[0];
}

template <int VW, int TXL>
__device__ __forceinline__ void dim_sum(float (&s)[VW], float* lds) {
  constexpr int TX = 1 << TXL, NW = kDimBlock / 64;
#pragma unroll
  for (int off = TX; off < 64; off <<= 1) {
#pragma unroll
    for (int k = 0; k < VW; ++k) s[k] += __shfl_xor(s[k], off, 64);
  }
  if constexpr (TX <= 64) {
    const int wave = threadIdx.x >> 6, tx = threadIdx.x & (TX - 1);
    if ((threadIdx.x & 63) < TX) {
#pragma unroll
      for (int k = 0; k < VW; ++k) lds[(wave * VW + k) * TX + tx] = s[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      float w[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) w[i] = lds[(i * VW + k) * TX + tx];
      s[k] = dim_tree<NW>(w);
    }
  }
}

// HOLD: the thread's classes (at most NC) stay in registers between the
// statistics and the output; otherwise they stream through in groups of NC,
// twice (plain loads first, so that the second pass may find them cached).
// The maximum of all groups comes before the exponentials that are held, and
// before the one rescale of those that stream: each rescale costs the sum two
// roundings.
template <typename TI, typename TO, int VW, int TXL, int NC, bool HOLD, bool LOG>
__global__ void __launch_bounds__(kDimBlock)
k_dim_fwd(const TI* __restrict__ in, TO* __restrict__ out, DimGeom g) {
  constexpr int TX = 1 << TXL, TY = kDimBlock / TX;
  constexpr int GRP = VW <= 4 ? 4 : 2;  // classes added by a tree; of eight positions four cost registers
  constexpr int LDS_SUM = TX <= 64 ? (kDimBlock / 64) * TX * VW : 0;  // the sums' place, then the maxima's
  __shared__ float lds[TX <= 64 ? 2 * LDS_SUM : 1];
  const DimPlace at = dim_place<VW, TXL>(g);
  const uint32_t ty = threadIdx.x >> TXL;
  const TI* src = in + at.base;
  TO* dst = out + at.base;
  dim_raw_t<TI, VW> x[NC];
  float m[VW], s[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) {
    m[k] = -__builtin_inff();
    s[k] = 0.0f;
  }
  for (uint32_t c0 = ty; HOLD ? c0 == ty : c0 < g.cols; c0 += NC * TY) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const uint32_t c = c0 + j * TY;
      if (at.valid && c < g.cols) x[j] = dim_load<TI, VW, HOLD>(src + (int64_t)c * g.inner);
    }
    float M[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) M[k] = m[k];
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (at.valid && c0 + j * TY < g.cols) {
#pragma unroll
        for (int k = 0; k < VW; ++k) M[k] = fmaxf(M[k], dim_elem<TI, VW>(x[j], k));
      }
    if constexpr (HOLD) dim_max<VW, TXL>(M, lds + LDS_SUM);
    float mb[VW];  // all -inf: keep exp arguments finite
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      if constexpr (!HOLD) s[k] = lse_rescale(s[k], m[k], M[k]);
      m[k] = M[k];
      mb[k] = M[k] == -__builtin_inff() ? 0.0f : M[k];
    }
    dim_opaque<TI, VW, NC>(x);
    float t[VW];  // this step's NC classes by fours or twos, then the steps: no chain is as long as the class dim
#pragma unroll
    for (int k = 0; k < VW; ++k) t[k] = 0.0f;
#pragma unroll
    for (int j = 0; j < NC; j += GRP)
      if (at.valid && c0 + j * TY < g.cols) {
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          float e[GRP];
#pragma unroll
          for (int i = 0; i < GRP; ++i)
            e[i] = c0 + (j + i) * TY < g.cols
                       ? __builtin_amdgcn_exp2f((dim_elem<TI, VW>(x[j + i], k) - mb[k]) * kLog2e)
                       : 0.0f;
          t[k] += dim_tree<GRP>(e);
        }
      }
#pragma unroll
    for (int k = 0; k < VW; ++k) s[k] += t[k];
    if constexpr (HOLD) break;
  }
  if constexpr (!HOLD) {
    float M[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) M[k] = m[k];
    dim_max<VW, TXL>(M, lds + LDS_SUM);
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      s[k] = lse_rescale(s[k], m[k], M[k]);
      m[k] = M[k];
    }
  }
  dim_sum<VW, TXL>(s, lds);
  if constexpr (HOLD) dim_opaque<TI, VW, NC>(x);
  // log: (x - M) - log S;  softmax: e^(x - M) / S (an all -inf column gives
  // 0 * inf = NaN, a NaN anywhere a NaN sum)
  float a[VW], b[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) {
    a[k] = LOG ? m[k] : (m[k] == -__builtin_inff() ? 0.0f : m[k]);
    b[k] = LOG ? sa_logf(s[k]) : 1.0f / s[k];
  }
  for (uint32_t c0 = ty; HOLD ? c0 == ty : c0 < g.cols; c0 += NC * TY) {
    if constexpr (!HOLD) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const uint32_t c = c0 + j * TY;
        if (at.valid && c < g.cols) x[j] = dim_load<TI, VW, true>(src + (int64_t)c * g.inner);
      }
    }
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const uint32_t c = c0 + j * TY;
      if (at.valid && c < g.cols) {
        float f[VW];
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          const float v = dim_elem<TI, VW>(x[j], k);
          if constexpr (LOG) f[k] = (v - a[k]) - b[k];
          else f[k] = __builtin_amdgcn_exp2f((v - a[k]) * kLog2e) * b[k];
        }
        dim_store<TO, VW>(dst + (int64_t)c * g.inner, f, at.skip);
      }
    }
    if constexpr (HOLD) break;
  }
}

// LOG: gi = g - exp(y) sum(g);  softmax: gi = y (g - sum(g y)).
template <typename TG, typename TO, int VW, int TXL, int NC, bool HOLD, bool LOG>
__global__ void __launch_bounds__(kDimBlock)
k_dim_bwd(const TG* __restrict__ grad, const TG* __restrict__ outp, TO* __restrict__ gin, DimGeom g) {
  constexpr int TX = 1 << TXL, TY = kDimBlock / TX;
  constexpr int GRP = LOG && VW <= 4 ? 4 : 2;  // as in the forward; products by two, the second fused
  __shared__ float lds[TX <= 64 ? (kDimBlock / 64) * TX * VW : 1];
  const DimPlace at = dim_place<VW, TXL>(g);
  const uint32_t ty = threadIdx.x >> TXL;
  const TG* gs = grad + at.base;
  const TG* ys = outp + at.base;
  TO* dst = gin + at.base;
  dim_raw_t<TG, VW> gv[NC], yv[NC];
  float s[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) s[k] = 0.0f;
  for (uint32_t c0 = ty; HOLD ? c0 == ty : c0 < g.cols; c0 += NC * TY) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const uint32_t c = c0 + j * TY;
      if (at.valid && c < g.cols) {
        gv[j] = dim_load<TG, VW, HOLD>(gs + (int64_t)c * g.inner);
        if (HOLD || !LOG) yv[j] = dim_load<TG, VW, HOLD>(ys + (int64_t)c * g.inner);
      }
    }
    float t[VW];  // as in the forward
#pragma unroll
    for (int k = 0; k < VW; ++k) t[k] = 0.0f;
#pragma unroll
    for (int j = 0; j < NC; j += GRP)
      if (at.valid && c0 + j * TY < g.cols) {
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          float e[GRP];
#pragma unroll
          for (int i = 0; i < GRP; ++i) {
            e[i] = 0.0f;
            if (c0 + (j + i) * TY < g.cols) {
              const float gk = dim_elem<TG, VW>(gv[j + i], k);
              if constexpr (LOG) e[i] = gk;
              else e[i] = fmaf(gk, dim_elem<TG, VW>(yv[j + i], k), i > 0 ? e[i - 1] : 0.0f);
              if constexpr (!LOG) if (i > 0) e[i - 1] = 0.0f;
            }
          }
          t[k] += dim_tree<GRP>(e);
        }
      }
#pragma unroll
    for (int k = 0; k < VW; ++k) s[k] += t[k];
    if constexpr (HOLD) break;
  }
  dim_sum<VW, TXL>(s, lds);
  if constexpr (HOLD) {
    dim_opaque<TG, VW, NC>(gv);
    dim_opaque<TG, VW, NC>(yv);
  }
  for (uint32_t c0 = ty; HOLD ? c0 == ty : c0 < g.cols; c0 += NC * TY) {
    if constexpr (!HOLD) {
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const uint32_t c = c0 + j * TY;
        if (at.valid && c < g.cols) {
          gv[j] = dim_load<TG, VW, true>(gs + (int64_t)c * g.inner);
          yv[j] = dim_load<TG, VW, true>(ys + (int64_t)c * g.inner);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const uint32_t c = c0 + j * TY;
      if (at.valid && c < g.cols) {
        float f[VW];
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          const float gk = dim_elem<TG, VW>(gv[j], k), yk = dim_elem<TG, VW>(yv[j], k);
          if constexpr (LOG) f[k] = fmaf(-__builtin_amdgcn_exp2f(yk * kLog2e), s[k], gk);
          else f[k] = yk * (gk - s[k]);
        }
        dim_store<TO, VW>(dst + (int64_t)c * g.inner, f, at.skip);
      }
    }
    if constexpr (HOLD) break;
  }
}

// Fills the geometry for VW-wide vectors; false when the counts leave the
// kernels' 32-bit indices.
inline bool dim_geom(DimGeom& g, int64_t outer, int64_t cols, int64_t inner, int vw) {
  const int64_t ivec = (inner + vw - 1) / vw;
  if (cols >= (int64_t(1) << 31) || ivec >= (int64_t(1) << 31) || outer * ivec >= (int64_t(1) << 31)) return false;
  g.npos = (uint32_t)(outer * ivec);
  g.first = 0;
  g.ivec = FastDiv((uint32_t)ivec);
  g.cols = (uint32_t)cols;
  g.inner = inner;
  return true;
}

// Calls launch(TXL, NC, HOLD as integral constants, workgroups) with the split
// of the classes over class groups, once per slab of positions (g.first): HIP
// takes fewer than 2^32 threads a launch.
template <int NCMAX, typename F>
int dim_split(DimGeom& g, F&& launch) {
  using std::integral_constant;
  constexpr int H = NCMAX / 2;
  auto go = [&](auto txl, auto nc, auto hold) -> int {
    constexpr uint64_t slab = (((uint64_t(1) << 32) - 1) / kDimBlock) << txl.value;
    for (uint64_t p0 = 0; p0 < g.npos; p0 += slab) {
      g.first = (uint32_t)p0;
      const uint64_t n = std::min<uint64_t>(slab, g.npos - p0);
      const int rc = launch(txl, nc, hold, (unsigned)((n + (1u << txl.value) - 1) >> txl.value));
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  };
  using X8 = integral_constant<int, 8>;
  using X6 = integral_constant<int, 6>;
  using X4 = integral_constant<int, 4>;
  using NH = integral_constant<int, H>;
  if (g.cols <= H) return go(X8{}, NH{}, std::true_type{});
  if (g.cols <= 4 * H) return go(X6{}, NH{}, std::true_type{});
  if (g.cols <= 16 * H) return go(X4{}, NH{}, std::true_type{});
  if (g.cols <= 16 * NCMAX) return go(X4{}, integral_constant<int, NCMAX>{}, std::true_type{});
  return go(X4{}, NH{}, std::false_type{});
}

template <typename TI, typename TO, int VW, bool LOG>
int dim_forward(const TI* in, TO* out, int64_t outer, int64_t cols, int64_t inner, hipStream_t st) {
  DimGeom g;
  if (!dim_geom(g, outer, cols, inner, VW)) return SUPA_AMD_ELAYOUT;
  return dim_split<16>(g, [&](auto txl, auto nc, auto hold, unsigned blocks) {
    k_dim_fwd<TI, TO, VW, txl.value, nc.value, hold.value, LOG><<<blocks, kDimBlock, 0, st>>>(in, out, g);
    return launch_status();
  });
}

template <typename TG, typename TO, int VW, bool LOG>
int dim_backward(const TG* grad, const TG* y, TO* gin, int64_t outer, int64_t cols, int64_t inner, hipStream_t st) {
  DimGeom g;
  if (!dim_geom(g, outer, cols, inner, VW)) return SUPA_AMD_ELAYOUT;
  return dim_split<16>(g, [&](auto txl, auto nc, auto hold, unsigned blocks) {
    k_dim_bwd<TG, TO, VW, txl.value, nc.value, hold.value, LOG><<<blocks, kDimBlock, 0, st>>>(grad, y, gin, g);
    return launch_status();
  });
}

}  // namespace sa

using namespace sa;

extern "C" {

int supa_amd_softmax_dim_forward(int log, const void* in, int32_t in_dtype, void* out, int32_t out_dtype,
                                 int64_t outer, int64_t cols, int64_t inner, void* stream) {
  if (!in || !out || outer < 0 || cols < 0 || inner < 0) return SUPA_AMD_EINVAL;
  if (outer == 0 || cols == 0 || inner == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_float_storage(in_dtype, [&](auto* ti) -> int {
    return with_float_storage(out_dtype, [&](auto* to) -> int {
      using TI = std::remove_pointer_t<decltype(ti)>;
      using TO = std::remove_pointer_t<decltype(to)>;
      if constexpr (!std::is_same<TI, TO>::value && !std::is_same<TO, float>::value) {
        return SUPA_AMD_EDTYPE;
      } else {
        constexpr int V = VecOf<TI>::V;
        const TI* x = static_cast<const TI*>(in);
        TO* y = static_cast<TO*>(out);
        if (inner >= V)
          return log ? dim_forward<TI, TO, V, true>(x, y, outer, cols, inner, st)
                     : dim_forward<TI, TO, V, false>(x, y, outer, cols, inner, st);
        return log ? dim_forward<TI, TO, 1, true>(x, y, outer, cols, inner, st)
                   : dim_forward<TI, TO, 1, false>(x, y, outer, cols, inner, st);
      }
    });
  });
}

int supa_amd_softmax_dim_backward(int log, const void* grad, const void* output, int32_t gy_dtype, void* grad_in,
                                  int32_t gin_dtype, int64_t outer, int64_t cols, int64_t inner, void* stream) {
  if (!grad || !output || !grad_in || outer < 0 || cols < 0 || inner < 0) return SUPA_AMD_EINVAL;
  if (outer == 0 || cols == 0 || inner == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_float_storage(gy_dtype, [&](auto* tg) -> int {
    return with_float_storage(gin_dtype, [&](auto* to) -> int {
      using TG = std::remove_pointer_t<decltype(tg)>;
      using TO = std::remove_pointer_t<decltype(to)>;
      if constexpr (!std::is_same<TG, TO>::value && !std::is_same<TO, float>::value) {
        return SUPA_AMD_EDTYPE;
      } else {
        constexpr int V = VecOf<TG>::V;
        const TG* g = static_cast<const TG*>(grad);
        const TG* y = static_cast<const TG*>(output);
        TO* gi = static_cast<TO*>(grad_in);
        if (inner >= V)
          return log ? dim_backward<TG, TO, V, true>(g, y, gi, outer, cols, inner, st)
                     : dim_backward<TG, TO, V, false>(g, y, gi, outer, cols, inner, st);
        return log ? dim_backward<TG, TO, 1, true>(g, y, gi, outer, cols, inner, st)
                   : dim_backward<TG, TO, 1, false>(g, y, gi, outer, cols, inner, st);
      }
    });
  });
}

}  // extern "C"
