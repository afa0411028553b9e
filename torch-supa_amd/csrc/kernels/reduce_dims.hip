// Sums over some dims of a dense tensor, straight from its memory order:
//   columns   [outer, red, inner] summed over red (a bias gradient: the sum
//             over the leading dims);
//   segments  each row the sum of `segs` runs of `len` contiguous elements
//             (rows of a matrix; a channel's planes over a batch).
// Both read the input once in 16-byte vectors at any alignment; moving the
// reduced dims last first, as a row kernel alone needs, copies it once more.
//
// HBM-bound.  Two launches where one would leave the chip idle: the reduced
// range is cut in chunks, each chunk's partial goes to the workspace in the
// accumulation type (float32, float64 for float64, int64 for integers), and a
// second launch adds the partials.  The order of every addition depends only
// on the sizes, so reruns are bit-identical.
//
// Measured on MI355X, us, before (a copy where the reduced dims are not last,
// then a 256-thread workgroup of scalar loads per row) -> after: sum over dim 0
// of bf16 [8192, 4096] 58 -> 16, float32 76 -> 27, float32 [8192, 12288] 250 ->
// 67 (6.0 TB/s), bf16 [131072, 256] 208 -> 17; over dims 0 and 2 of float32
// [32, 64, 12544] 180 -> 20 (5.2 TB/s); over the rows of bf16 [8192, 4096] 23
// -> 12 (5.7 TB/s), [16, 1048576] 408 -> 6.7, [1048576, 10] 420 -> 44.
//
// Replaces sum_stub / mean_stub over dims
// (.../kernels/reduce/ReduceSumKernel.cu:102-113, ReduceMomentKernel.cu:37-55).
#include "segments.h"

namespace sa {

constexpr int kDimSumBlock = 256;
constexpr int64_t kDimSumBlocks = 1024;  // workgroups to aim at when cutting chunks: four per CU

// --------------------------------------------------------------- columns
// Thread (tx, ty) adds rows ty, ty + TY, ... of its chunk for VW columns; TX =
// 2^TXL position vectors by TY = 256 / TX row groups a workgroup.  The last
// vector of a plane is moved back to end at the plane's end and stores only
// the columns no other vector covers.
struct ColsGeom {
  uint32_t npos;    // position vectors: outer * ceil(inner / VW)
  uint32_t first;   // the launch's first one
  FastDiv ivec;     // vectors per row
  int64_t red, inner;
  int64_t chunk;    // rows per chunk (blockIdx.y)
  int64_t nout;     // outer * inner
};

template <typename T, typename OT, typename ACC, int VW, int TXL>
__global__ void __launch_bounds__(kDimSumBlock)
k_sum_cols(const T* __restrict__ in, OT* __restrict__ out, ColsGeom g, ACC scale) {
  constexpr int TX = 1 << TXL, TY = kDimSumBlock / TX, NW = kDimSumBlock / 64, U = 8;
  __shared__ ACC lds[TX <= 64 ? NW * TX * VW : 1];
  const uint32_t tx = threadIdx.x & (TX - 1), ty = threadIdx.x >> TXL;
  const uint32_t p = g.first + blockIdx.x * TX + tx;
  const bool valid = p < g.npos;
  uint32_t o, v;
  g.ivec.divmod(p, o, v);
  int64_t pos = (int64_t)v * VW;
  int skip = 0;
  if (pos + VW > g.inner) {
    skip = (int)(pos + VW - g.inner);
    pos = g.inner - VW;
  }
  const T* src = in + (int64_t)o * g.red * g.inner + pos;
  const int64_t lo = (int64_t)blockIdx.y * g.chunk;
  const int64_t hi = lo + g.chunk < g.red ? lo + g.chunk : g.red;
  ACC acc[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) acc[k] = ACC(0);
  if (valid) {
    int64_t r = lo + ty;
    for (; r + (U - 1) * TY < hi; r += U * TY) {
      sum_raw_t<T, VW> w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = sum_load<T, VW>(src + (r + u * TY) * g.inner);
      if constexpr (std::is_integral<ACC>::value) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int k = 0; k < VW; ++k) acc[k] += sum_elem<T, VW, ACC>(w[u], k);
      } else {  // U rows by a tree, then the steps (cols_chunk says how many)
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          ACC t[U];
#pragma unroll
          for (int u = 0; u < U; ++u) t[u] = sum_elem<T, VW, ACC>(w[u], k);
#pragma unroll
          for (int h = 1; h < U; h *= 2)
#pragma unroll
            for (int u = 0; u < U; u += 2 * h) t[u] += t[u + h];
          acc[k] += t[0];
        }
      }
    }
    for (; r < hi; r += TY) {
      const sum_raw_t<T, VW> w = sum_load<T, VW>(src + r * g.inner);
#pragma unroll
      for (int k = 0; k < VW; ++k) acc[k] += sum_elem<T, VW, ACC>(w, k);
    }
  }
#pragma unroll
  for (int off = TX; off < 64; off <<= 1)
#pragma unroll
    for (int k = 0; k < VW; ++k) acc[k] += __shfl_xor(acc[k], off, 64);
  if constexpr (TX <= 64) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) < TX) {
#pragma unroll
      for (int k = 0; k < VW; ++k) lds[(wave * VW + k) * TX + tx] = acc[k];
    }
    __syncthreads();
    if (ty == 0) {
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        acc[k] = lds[k * TX + tx];
#pragma unroll
        for (int w = 1; w < NW; ++w) acc[k] += lds[(w * VW + k) * TX + tx];
      }
    }
  }
  if (ty == 0 && valid) {
    OT* dst = out + (int64_t)blockIdx.y * g.nout + (int64_t)o * g.inner + pos;
#pragma unroll
    for (int k = 0; k < VW; ++k)
      if (k >= skip) dst[k] = from_arith<OT>(acc[k] * scale);
  }
}

inline int cols_txl(int64_t red, int64_t npos) { return red <= 16 ? 8 : (npos >= 32 ? 6 : 4); }

// Rows per chunk: enough chunks for kDimSumBlocks workgroups, each of at least
// 8 rows a thread, and no more than 64 rows a thread (or a 256th of the column,
// as a workgroup per column would give each of its threads): where the columns
// alone fill the chip a thread of a single chunk would add red / TY rows one
// after another, and its rounding errors with them (float32 against 64 bits,
// [8192, 128256]: 4.4e-7 in one chunk, 1.2e-7 so and with a workgroup per
// column).  The partials are a 64th of the rows at most.
inline int64_t cols_chunk(int64_t red, int64_t npos, int txl) {
  const int64_t blocks = (npos + (1 << txl) - 1) >> txl;
  const int64_t ty = kDimSumBlock >> txl, rows = 8 * ty;  // one unrolled step
  const int64_t fill = std::min<int64_t>((kDimSumBlocks + blocks - 1) / blocks, (red + rows - 1) / rows);
  const int64_t most = ty * std::max<int64_t>(64, red / kDimSumBlock);
  const int64_t want = std::max<int64_t>(fill, (red + most - 1) / most);
  if (want <= 1) return red;
  const int64_t per = (red + want - 1) / want;
  return (per + rows - 1) / rows * rows;
}

constexpr int64_t kDimSumSlab = ((int64_t(1) << 32) - 1) / kDimSumBlock;  // workgroups: HIP takes fewer than 2^32 threads

template <typename T, typename OT, typename ACC, int VW>
int cols_launch(const T* in, OT* out, ColsGeom g, int txl, ACC scale, hipStream_t st) {
  const unsigned chunks = (unsigned)((g.red + g.chunk - 1) / g.chunk);
  const int64_t slab = kDimSumSlab << txl;
  for (int64_t p0 = 0; p0 < g.npos; p0 += slab) {
    g.first = (uint32_t)p0;
    const int64_t n = std::min<int64_t>(slab, g.npos - p0);
    const dim3 grid((unsigned)((n + (1 << txl) - 1) >> txl), chunks);
    if (txl == 8) k_sum_cols<T, OT, ACC, VW, 8><<<grid, kDimSumBlock, 0, st>>>(in, out, g, scale);
    else if (txl == 6) k_sum_cols<T, OT, ACC, VW, 6><<<grid, kDimSumBlock, 0, st>>>(in, out, g, scale);
    else k_sum_cols<T, OT, ACC, VW, 4><<<grid, kDimSumBlock, 0, st>>>(in, out, g, scale);
    const int rc = launch_status();
    if (rc) return rc;
  }
  return SUPA_AMD_OK;
}

// Geometry of a [outer, red, inner] sum in VW-wide vectors; false when its
// indices leave 32 bits.
inline bool cols_geom(ColsGeom& g, int64_t outer, int64_t red, int64_t inner, int vw, int64_t chunk) {
  const int64_t ivec = (inner + vw - 1) / vw;
  if (ivec >= (int64_t(1) << 31) || outer * ivec >= (int64_t(1) << 31) || (red + chunk - 1) / chunk > 65535) return false;
  g = ColsGeom{(uint32_t)(outer * ivec), 0, FastDiv((uint32_t)ivec), red, inner, chunk, outer * inner};
  return true;
}

struct ColsPlan {
  int vw, txl;
  int64_t npos, chunk, nchunks;
};
inline ColsPlan cols_plan(int64_t outer, int64_t red, int64_t inner, int vmax) {
  ColsPlan p;
  p.vw = inner >= vmax ? vmax : 1;
  p.npos = outer * ((inner + p.vw - 1) / p.vw);
  p.txl = cols_txl(red, p.npos);
  p.chunk = cols_chunk(red, p.npos, p.txl);
  p.nchunks = (red + p.chunk - 1) / p.chunk;
  return p;
}

template <typename T, typename OT, typename ACC, int VW>
int cols_run(const T* in, OT* out, int64_t outer, int64_t red, int64_t inner, const ColsPlan& p, ACC scale, void* ws,
             hipStream_t st) {
  ColsGeom g;
  if (!cols_geom(g, outer, red, inner, VW, p.chunk)) return SUPA_AMD_ELAYOUT;
  if (p.nchunks == 1) return cols_launch<T, OT, ACC, VW>(in, out, g, p.txl, scale, st);
  ACC* part = static_cast<ACC*>(ws);
  const int rc = cols_launch<T, ACC, ACC, VW>(in, part, g, p.txl, ACC(1), st);
  if (rc) return rc;
  // the partials: [nchunks, outer * inner], 16 groups of rows a workgroup
  constexpr int PV = std::is_same<ACC, float>::value ? 4 : 1;
  const int64_t n = outer * inner;
  if (n >= PV) {
    if (!cols_geom(g, 1, p.nchunks, n, PV, p.nchunks)) return SUPA_AMD_ELAYOUT;
    return cols_launch<ACC, OT, ACC, PV>(part, out, g, 4, scale, st);
  }
  if (!cols_geom(g, 1, p.nchunks, n, 1, p.nchunks)) return SUPA_AMD_ELAYOUT;
  return cols_launch<ACC, OT, ACC, 1>(part, out, g, 4, scale, st);
}

// -------------------------------------------------------------- segments
// Row r is `segs` runs of `len` elements, run s at r row_stride + s
// seg_stride.  Its vectors (ceil(len / VW) a run, the last of a run short) are
// numbered across the runs; G threads share a row: 16 lanes or a wavefront
// for short rows, a workgroup of 256 for long ones, and chunks of `chunk`
// vectors in blockIdx.y for few long ones.
//
// STREAM: nontemporal loads, for inputs past 64 MiB; smaller ones were often
// written just before, are still in a cache and take plain loads (float32
// [2000, 4096] read over and over 3.8 us, 6.5 with the hint; [1400, 8000] 7.4,
// 8.5; [8000, 12000] 66 us, 58 with it; a normalisation of [8192, 4096], whose
// row sums read tensors that left the caches, 811 us, 803 with it).
template <typename T, typename OT, typename ACC, int VW, int G, bool STREAM>
__global__ void __launch_bounds__(kDimSumBlock)
k_sum_segs(const T* __restrict__ in, OT* __restrict__ out, SegGeom g, ACC scale) {
  constexpr int U = 4;
  const int l = threadIdx.x & (G - 1);
  const int64_t row = G < 256 ? (int64_t)blockIdx.x * (256 / G) + threadIdx.x / G : (int64_t)blockIdx.x;
  if (row >= g.rows) return;
  const T* src = in + row * g.row_stride;
  const uint32_t lo = blockIdx.y * g.chunk;
  const uint32_t nvec = (uint32_t)g.nvec;
  const uint32_t hi = nvec - lo < g.chunk ? nvec : lo + g.chunk;
  ACC acc = ACC(0);
  auto add = [&](const sum_raw_t<T, VW>& w) {
    ACC t = sum_elem<T, VW, ACC>(w, 0);
#pragma unroll
    for (int k = 1; k < VW; ++k) t += sum_elem<T, VW, ACC>(w, k);
    acc += t;
  };
  uint32_t i0 = lo + l;
  if constexpr (G > 16) {  // rows of one run: steps of whole vectors without a look at each
    const uint32_t whole = g.runs > 1 ? 0u : (uint32_t)min((int64_t)hi, g.len / VW);
    for (; i0 + (U - 1) * G < whole; i0 += U * G) {
      sum_raw_t<T, VW> w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) w[u] = sum_load<T, VW, STREAM>(src + (int64_t)(i0 + u * G) * VW);
#pragma unroll
      for (int u = 0; u < U; ++u) add(w[u]);
    }
  }
  for (; i0 < hi; i0 += U * G) {
    sum_raw_t<T, VW> w[U];
    uint32_t valid;  // elements past a run's end are zeros
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + u * G < hi) w[u] = seg_load<T, VW, STREAM>(src, g, i0 + u * G, valid);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i0 + u * G < hi) add(w[u]);
  }
#pragma unroll
  for (int off = (G < 64 ? G : 64) / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if constexpr (G > 64) {
    __shared__ ACC lds[G / 64];
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = acc;
    __syncthreads();
    acc = lds[0];
#pragma unroll
    for (int w = 1; w < G / 64; ++w) acc += lds[w];
  }
  if (l == 0) out[row * gridDim.y + blockIdx.y] = from_arith<OT>(acc * scale);
}

// Chunks per row: rows too few for kDimSumBlocks workgroups are cut in chunks
// of at least 8 vectors a thread, from 32 on (the second launch costs 2 us:
// float32 [700, 16384], 16 vectors a thread, 6.3 us in one launch, 10.8 in two;
// [1, 16384] 3.9, 6.7).
inline int64_t seg_chunks(int64_t rows, int64_t nvec) {
  const int64_t most = nvec >= 32 * kDimSumBlock ? nvec / (8 * kDimSumBlock) : 1;
  return std::max<int64_t>(1, std::min<int64_t>(most, kDimSumBlocks / rows));
}

constexpr int64_t kSegStreamBytes = int64_t(64) << 20;

template <typename T, typename OT, typename ACC, int VW>
int segs_launch(const T* in, OT* out, const SegGeom& g, unsigned nch, ACC scale, hipStream_t st) {
  const bool stream = VW > 1 && g.rows * g.nvec * 16 > kSegStreamBytes;
  auto go = [&](auto G) -> int {
    constexpr int64_t per = kDimSumBlock / G.value, slab = per * kDimSumSlab;
    for (int64_t r0 = 0; r0 < g.rows; r0 += slab) {
      SegGeom gs = g;
      gs.rows = std::min(slab, g.rows - r0);
      const T* x = in + r0 * g.row_stride;
      OT* y = out + r0 * nch;
      const dim3 grid((unsigned)((gs.rows + per - 1) / per), nch);
      if (stream) k_sum_segs<T, OT, ACC, VW, G.value, VW != 1><<<grid, kDimSumBlock, 0, st>>>(x, y, gs, scale);
      else k_sum_segs<T, OT, ACC, VW, G.value, false><<<grid, kDimSumBlock, 0, st>>>(x, y, gs, scale);
      const int rc = launch_status();
      if (rc) return rc;
    }
    return SUPA_AMD_OK;
  };
  using std::integral_constant;
  // a wavefront per row up to 512 vectors where the rows alone fill the chip
  // (bf16 [6007, 2047] 5.5 us, 11.5 with four)
  const bool wave = g.rows >= 4096 && g.nvec <= 512;
  if (nch == 1 && g.nvec <= 32) return go(integral_constant<int, 16>{});
  if (nch == 1 && wave) return go(integral_constant<int, 64>{});
  return go(integral_constant<int, 256>{});
}

inline int64_t segs_vecs(int64_t segs, int64_t len, int vw) { return segs * ((len + vw - 1) / vw); }

template <typename T, typename OT, typename ACC>
int segs_run(const T* in, OT* out, int64_t rows, int64_t segs, int64_t len, int64_t row_stride, int64_t seg_stride,
             ACC scale, void* ws, hipStream_t st) {
  constexpr int VW = dim_sum_vw<T>();
  const int64_t nvec = segs_vecs(segs, len, VW), vps = (len + VW - 1) / VW;
  if (nvec >= (int64_t(1) << 31) || rows >= (int64_t(1) << 31)) return SUPA_AMD_ELAYOUT;
  const int64_t want = ws ? seg_chunks(rows, nvec) : 1;
  const int64_t chunk = (nvec + want - 1) / want, nch = (nvec + chunk - 1) / chunk;
  SegGeom g{rows, row_stride, seg_stride, segs, len, FastDiv((uint32_t)vps), nvec, (uint32_t)chunk};
  if (nch == 1) return segs_launch<T, OT, ACC, VW>(in, out, g, 1, scale, st);
  ACC* part = static_cast<ACC*>(ws);
  const int rc = segs_launch<T, ACC, ACC, VW>(in, part, g, (unsigned)nch, ACC(1), st);
  if (rc) return rc;
  SegGeom h{rows, nch, 0, 1, nch, FastDiv((uint32_t)nch), nch, (uint32_t)nch};
  return segs_launch<ACC, OT, ACC, 1>(part, out, h, 1, scale, st);
}

// Rows of 2^31 vectors and more: one 256-thread workgroup each, 64-bit indices.
template <typename T, typename OT, typename ACC>
__global__ void __launch_bounds__(kDimSumBlock)
k_sum_rows(const T* __restrict__ in, OT* __restrict__ out, int64_t inner, ACC scale) {
  __shared__ ACC lds[kDimSumBlock / 64];
  const T* row = in + (int64_t)blockIdx.x * inner;
  ACC acc = fold_strided<8>(
      ACC(0), threadIdx.x, kDimSumBlock, inner, [&](int64_t i) { return (ACC)to_arith(row[i]); },
      [](ACC a, ACC b) { return a + b; });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = from_arith<OT>((((lds[0] + lds[1]) + lds[2]) + lds[3]) * scale);
}

// f(input tag, output tag) for the dtype pairs of a dim sum: floating input
// to a floating output, bool / integer input to int64.
template <typename F>
int with_dim_sum_types(int in_dtype, int out_dtype, F&& f) {
  auto outsel = [&](auto* ti) -> int {
    switch (out_dtype) {
      case SUPA_AMD_F32: return f(ti, (float*)nullptr);
      case SUPA_AMD_BF16: return f(ti, (bf16*)nullptr);
      case SUPA_AMD_F16: return f(ti, (f16*)nullptr);
      case SUPA_AMD_F64: return f(ti, (double*)nullptr);
      default: return SUPA_AMD_EDTYPE;
    }
  };
  auto intsel = [&](auto* ti) -> int {
    return out_dtype == SUPA_AMD_I64 ? f(ti, (int64_t*)nullptr) : SUPA_AMD_EDTYPE;
  };
  switch (in_dtype) {
    case SUPA_AMD_F32: return outsel((float*)nullptr);
    case SUPA_AMD_BF16: return outsel((bf16*)nullptr);
    case SUPA_AMD_F16: return outsel((f16*)nullptr);
    case SUPA_AMD_F64: return outsel((double*)nullptr);
    case SUPA_AMD_BOOL: return intsel((b8*)nullptr);
    case SUPA_AMD_U8: return intsel((uint8_t*)nullptr);
    case SUPA_AMD_I8: return intsel((int8_t*)nullptr);
    case SUPA_AMD_I16: return intsel((int16_t*)nullptr);
    case SUPA_AMD_I32: return intsel((int32_t*)nullptr);
    case SUPA_AMD_I64: return intsel((int64_t*)nullptr);
    default: return SUPA_AMD_EDTYPE;
  }
}

template <typename T, typename OT>
using dim_sum_acc = std::conditional_t<std::is_integral<OT>::value, int64_t,
                                       std::conditional_t<std::is_same<T, double>::value || std::is_same<OT, double>::value,
                                                          double, float>>;

// Elements a 16-byte vector of the dtype holds in these kernels (1 for the
// integer types), and the bytes of a partial.
inline int dim_sum_vmax(int dtype) { return dtype_is_floating(dtype) ? 16 / dtype_size(dtype) : 1; }
inline int64_t dim_sum_acc_bytes(int in_dtype, int out_dtype) {
  return in_dtype == SUPA_AMD_F64 || out_dtype == SUPA_AMD_F64 || !dtype_is_floating(in_dtype) ? 8 : 4;
}

}  // namespace sa

using namespace sa;

extern "C" {

int64_t supa_amd_sum_cols_workspace_bytes(int32_t in_dtype, int32_t out_dtype, int64_t outer, int64_t red,
                                          int64_t inner) {
  if (outer <= 0 || red <= 0 || inner <= 0) return 0;
  const ColsPlan p = cols_plan(outer, red, inner, dim_sum_vmax(in_dtype));
  return p.nchunks == 1 ? 0 : p.nchunks * outer * inner * dim_sum_acc_bytes(in_dtype, out_dtype);
}

int supa_amd_sum_cols(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t outer, int64_t red,
                      int64_t inner, double scale, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!in || !out || outer < 0 || red <= 0 || inner < 0) return SUPA_AMD_EINVAL;
  if (outer == 0 || inner == 0) return SUPA_AMD_OK;
  const int64_t need = supa_amd_sum_cols_workspace_bytes(in_dtype, out_dtype, outer, red, inner);
  if (need > 0 && (!workspace || workspace_bytes < need)) return SUPA_AMD_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_dim_sum_types(in_dtype, out_dtype, [&](auto* ti, auto* to) -> int {
    using T = std::remove_pointer_t<decltype(ti)>;
    using OT = std::remove_pointer_t<decltype(to)>;
    using ACC = dim_sum_acc<T, OT>;
    constexpr int VW = dim_sum_vw<T>();
    const ColsPlan p = cols_plan(outer, red, inner, VW);
    const T* x = static_cast<const T*>(in);
    OT* y = static_cast<OT*>(out);
    if (p.vw == VW) return cols_run<T, OT, ACC, VW>(x, y, outer, red, inner, p, (ACC)scale, workspace, st);
    return cols_run<T, OT, ACC, 1>(x, y, outer, red, inner, p, (ACC)scale, workspace, st);
  });
}

int64_t supa_amd_sum_segments_workspace_bytes(int32_t in_dtype, int32_t out_dtype, int64_t rows, int64_t segs,
                                              int64_t len) {
  if (rows <= 0 || segs <= 0 || len <= 0) return 0;
  const int64_t n = seg_chunks(rows, segs_vecs(segs, len, dim_sum_vmax(in_dtype)));
  return n == 1 ? 0 : n * rows * dim_sum_acc_bytes(in_dtype, out_dtype);
}

int supa_amd_sum_segments(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t rows, int64_t segs,
                          int64_t len, int64_t row_stride, int64_t seg_stride, double scale, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  if (!in || !out || rows < 0 || segs <= 0 || len <= 0) return SUPA_AMD_EINVAL;
  if (rows == 0) return SUPA_AMD_OK;
  const int64_t need = supa_amd_sum_segments_workspace_bytes(in_dtype, out_dtype, rows, segs, len);
  if (need > 0 && (!workspace || workspace_bytes < need)) return SUPA_AMD_EWORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_dim_sum_types(in_dtype, out_dtype, [&](auto* ti, auto* to) -> int {
    using T = std::remove_pointer_t<decltype(ti)>;
    using OT = std::remove_pointer_t<decltype(to)>;
    using ACC = dim_sum_acc<T, OT>;
    return segs_run<T, OT, ACC>(static_cast<const T*>(in), static_cast<OT*>(out), rows, segs, len, row_stride,
                                seg_stride, (ACC)scale, need > 0 ? workspace : nullptr, st);
  });
}

// One launch, no workspace: a long row is one workgroup's.
int supa_amd_sum_rows(const void* in, int32_t in_dtype, void* out, int32_t out_dtype, int64_t outer, int64_t inner,
                      double scale, void* stream) {
  if (!in || !out || outer < 0 || inner <= 0 || outer >= (int64_t(1) << 31)) return SUPA_AMD_EINVAL;
  if (outer == 0) return SUPA_AMD_OK;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return with_dim_sum_types(in_dtype, out_dtype, [&](auto* ti, auto* to) -> int {
    using T = std::remove_pointer_t<decltype(ti)>;
    using OT = std::remove_pointer_t<decltype(to)>;
    using ACC = dim_sum_acc<T, OT>;
    const T* x = static_cast<const T*>(in);
    OT* y = static_cast<OT*>(out);
    if (segs_vecs(1, inner, dim_sum_vw<T>()) >= (int64_t(1) << 31)) {
      k_sum_rows<T, OT, ACC><<<(unsigned)outer, kDimSumBlock, 0, st>>>(x, y, inner, (ACC)scale);
      return launch_status();
    }
    return segs_run<T, OT, ACC>(x, y, outer, 1, inner, inner, 0, (ACC)scale, nullptr, st);
  });
}

}  // extern "C"
