// kern_dequant.hip — bit-exact dequantization kernels and the embedding gather.
// Compiled with -ffp-contract=off (see inferox_amd/build.py).
#include <algorithm>

#include "kernels.h"

namespace ifx {

// Little-endian loads at any alignment (raw GGUF blocks of 18, 34 and 210
// bytes keep no more than 2): the compiler emits single unaligned loads.
template <class V>
__device__ __forceinline__ V ldu(const uint8_t* p) {
  V v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}

// Elements 4i .. 4i + 3 of a raw GGUF block stream, raw_elem's arithmetic (so
// its bits): a quad never straddles a scale group, so its scales are decoded
// once and its quants come from one or two loads.
template <uint32_t T>
__device__ __forceinline__ float4 raw_quad(const uint8_t* __restrict__ p, uint64_t i) {
  float y[4];
  if constexpr (T == T_F32) {
    return ldu<float4>(p + 16 * i);
  } else if constexpr (T == T_F16) {
    const uint2 w = ldu<uint2>(p + 8 * i);
    return make_float4(h2f(w.x), h2f(w.x >> 16), h2f(w.y), h2f(w.y >> 16));
  } else if constexpr (T == T_Q4_0) {
    const uint8_t* blk = p + (i >> 3) * 18;
    const int j = (int)(4 * i & 31);
    const float delta = h2f(ldu<uint16_t>(blk));
    const uint32_t w = ldu<uint32_t>(blk + 2 + (j & 15)) >> (j < 16 ? 0 : 4);
#pragma unroll
    for (int k = 0; k < 4; k++) y[k] = (float)((int)((w >> (8 * k)) & 15u) - 8) * delta;
  } else if constexpr (T == T_Q8_0) {
    const uint8_t* blk = p + (i >> 3) * 34;
    const float delta = h2f(ldu<uint16_t>(blk));
    const uint32_t w = ldu<uint32_t>(blk + 2 + (4 * i & 31));
#pragma unroll
    for (int k = 0; k < 4; k++) y[k] = (float)(int8_t)(w >> (8 * k)) * delta;
  } else if constexpr (T == T_Q4K) {
    const uint8_t* blk = p + (i >> 6) * 144;
    const uint32_t j = (uint32_t)(4 * i & 255), g = j >> 5;
    const uint4 h = ldu<uint4>(blk);  // d, dmin, 12 scale bytes
    const uint32_t w = ldu<uint16_t>(blk + 16 + (j >> 1));
    const uint32_t s8 = 8 * (g & 3), a = h.y >> s8, b = h.z >> s8, c = h.w >> s8;
    const uint32_t sc = g < 4 ? a & 63u : (c & 15u) | ((a >> 2) & 48u);
    const uint32_t mn = g < 4 ? b & 63u : ((c >> 4) & 15u) | ((b >> 2) & 48u);
    const float dall = h2f(h.x) * (float)sc, dm = h2f(h.x >> 16) * (float)mn;
#pragma unroll
    for (int k = 0; k < 4; k++) y[k] = dall * (float)((w >> (4 * k)) & 15u) - dm;
  } else if constexpr (T == T_Q6K) {
    const uint8_t* blk = p + (i >> 6) * 210;
    const uint32_t j = (uint32_t)(4 * i & 255);
    const uint32_t lo = ldu<uint16_t>(blk + 18 + (j >> 1)), hi = blk[146 + (j >> 2)];
    const float ds = h2f(ldu<uint16_t>(blk)) * (float)blk[2 + (j >> 4)];
#pragma unroll
    for (int k = 0; k < 4; k++)
      y[k] = ds * (float)((int)(((lo >> (4 * k)) & 15u) | (((hi >> (2 * k)) & 3u) << 4)) - 32);
  } else {  // Q8_K
    const uint8_t* blk = p + (i >> 6) * 292;
    const uint32_t j = (uint32_t)(4 * i & 255), dd = ldu<uint32_t>(blk), w = ldu<uint32_t>(blk + 36 + j);
    const float ds = h2f(dd) * (float)blk[4 + (j >> 3)], dmin = h2f(dd >> 16);
#pragma unroll
    for (int k = 0; k < 4; k++) y[k] = ds * (float)(int8_t)(w >> (8 * k)) - dmin;
  }
  return make_float4(y[0], y[1], y[2], y[3]);
}

// Raw GGUF stream -> f32 (gguf::dequantize_f32, src/gguf/dequant.rs:10-31).
// Bound by the f32 stores.  A thread takes kQuads quads 256 apart, so each
// wave's stores are whole kilobytes and kQuads loads are in flight per lane.
// A 14336 x 4096 Q4_K matrix: 56 us, 4.8 TB/s read and written (an element per
// thread with byte loads, the scales decoded for each: 154 us, 1.7 TB/s).
constexpr int kQuads = 4;
template <uint32_t T>
__global__ void __launch_bounds__(256) k_dequant_raw(const uint8_t* __restrict__ p, uint64_t n,
                                                     float* __restrict__ out) {
  const uint64_t nq = n / 4, base = (uint64_t)blockIdx.x * (256 * kQuads) + threadIdx.x;
  float4 v[kQuads];
#pragma unroll
  for (int k = 0; k < kQuads; k++) {
    const uint64_t q = base + 256 * k;
    if (q < nq) v[k] = raw_quad<T>(p, q);
  }
#pragma unroll
  for (int k = 0; k < kQuads; k++) {
    const uint64_t q = base + 256 * k;
    if (q < nq) __builtin_memcpy(out + 4 * q, &v[k], 16);
  }
  if ((T == T_F32 || T == T_F16) && blockIdx.x == 0 && threadIdx.x < n % 4)  // whole blocks elsewhere
    out[4 * nq + threadIdx.x] = raw_elem(T, p, 4 * nq + threadIdx.x);
}

// Elements 4i .. 4i + 3 of row `row` of a matrix in the device layout
// (ifx_common.h), dev_elem's arithmetic; i < cols / 4, cols % 4 == 0.
__device__ __forceinline__ float4 dev_quad(const DevW& w, uint64_t row, uint32_t i) {
  float y[4];
  const uint32_t col = 4 * i;
  switch (w.type) {
    case T_F32: return ((const float4*)w.body)[row * (w.cols / 4) + i];
    case T_F16: {
      const uint2 v = ((const uint2*)w.body)[row * (w.cols / 4) + i];
      return make_float4(h2f(v.x), h2f(v.x >> 16), h2f(v.y), h2f(v.y >> 16));
    }
    case T_Q4_0: {
      const uint64_t b = row * (w.cols / 32) + (col >> 5);
      const float delta = h2f(((const uint16_t*)w.scal)[b]);
      const uint32_t v = *(const uint32_t*)(w.body + b * 16 + (col & 15)) >> ((col & 16) ? 4 : 0);
#pragma unroll
      for (int k = 0; k < 4; k++) y[k] = (float)((int)((v >> (8 * k)) & 15u) - 8) * delta;
      break;
    }
    case T_Q8_0: {
      const uint64_t b = row * (w.cols / 32) + (col >> 5);
      const float delta = h2f(((const uint16_t*)w.scal)[b]);
      const uint32_t v = *(const uint32_t*)(w.body + b * 32 + (col & 31));
#pragma unroll
      for (int k = 0; k < 4; k++) y[k] = (float)(int8_t)(v >> (8 * k)) * delta;
      break;
    }
    case T_Q4K: {
      const uint8_t* u = w.body + (row >> 4) * w.tstride + (uint64_t)(col >> 8) * w.bstride;
      const uint32_t n = (uint32_t)(row & 15), j = col & 255, g = j >> 5;
      const uint4 h = *(const uint4*)(u + 16 * n);
      const uint32_t v = *(const uint16_t*)(u + 256 + (g >> 2) * 1024 + (n + 16 * (g & 3)) * 16 + ((j & 31) >> 1));
      const uint32_t s8 = 8 * (g & 3), a = h.y >> s8, b = h.z >> s8, c = h.w >> s8;
      const uint32_t sc = g < 4 ? a & 63u : (c & 15u) | ((a >> 2) & 48u);
      const uint32_t mn = g < 4 ? b & 63u : ((c >> 4) & 15u) | ((b >> 2) & 48u);
      const float dall = h2f(h.x) * (float)sc, dm = h2f(h.x >> 16) * (float)mn;
#pragma unroll
      for (int k = 0; k < 4; k++) y[k] = dall * (float)((v >> (4 * k)) & 15u) - dm;
      break;
    }
    case T_Q6K: {
      const uint8_t* u = w.body + (row >> 4) * w.tstride + (uint64_t)(col >> 8) * w.bstride;
      const uint32_t n = (uint32_t)(row & 15), j = col & 255, s = j >> 5, e = j & 15;
      const uint32_t lane = n + 16 * (s & 3), c = 2 * (s >> 2) + ((j >> 4) & 1);
      const uint32_t lo = *(const uint16_t*)(u + (s >> 2) * 1024 + lane * 16 + ((j >> 1) & 15));
      const uint32_t hw = *(const uint32_t*)(u + 2048 + lane * 16 + 4 * c);
      const uint32_t sb = u[3072 + 4 * lane + c];
      const float ds = h2f(*(const uint16_t*)(u + 3328 + 2 * n)) * (w.q6_signed ? (float)(int8_t)sb : (float)sb);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t f = e + k, hi = (hw >> (8 * ((f & 7) >> 1) + 2 * (f & 1) + 4 * (f >> 3))) & 3u;
        y[k] = ds * (float)((int)(((lo >> (4 * k)) & 15u) | (hi << 4)) - 32);
      }
      break;
    }
    default: {  // Q8_K
      const uint64_t b = row * (w.cols / 256) + (col >> 8);
      const uint32_t j = col & 255, dd = ((const uint32_t*)w.scal)[b];
      const uint8_t* blk = w.body + b * 288;
      const uint32_t v = *(const uint32_t*)(blk + 32 + j);
      const float ds = h2f(dd) * (float)blk[j >> 3], dmin = h2f(dd >> 16);
#pragma unroll
      for (int k = 0; k < 4; k++) y[k] = ds * (float)(int8_t)(v >> (8 * k)) - dmin;
      break;
    }
  }
  return make_float4(y[0], y[1], y[2], y[3]);
}

// o[0..cols) = row `row` of the matrix: workgroup bx of the nbx that share the
// row.  Rows of whole quads (every block type) go four elements at a time.
__device__ __forceinline__ void dev_row(const DevW& w, uint64_t row, float* o, uint32_t bx, uint32_t nbx) {
  if (w.cols % 4 == 0) {
    for (uint64_t i = (uint64_t)bx * blockDim.x + threadIdx.x; i < w.cols / 4; i += (uint64_t)nbx * blockDim.x) {
      const float4 v = dev_quad(w, row, (uint32_t)i);
      __builtin_memcpy(o + 4 * i, &v, 16);
    }
    return;
  }
  for (uint64_t c = (uint64_t)bx * blockDim.x + threadIdx.x; c < w.cols; c += (uint64_t)nbx * blockDim.x)
    o[c] = dev_elem(w, row * w.cols + c);
}

// Device-layout matrix -> f32, row by row.
__global__ void __launch_bounds__(256) k_dequant_dev(DevW w, uint64_t rows, float* __restrict__ out) {
  for (uint64_t r = blockIdx.y; r < rows; r += gridDim.y) dev_row(w, r, out + r * w.cols, blockIdx.x, gridDim.x);
}

// out[r][:] = row ids[r] of the table (embedding_lookup, src/ops.rs:246-258,
// over the dequantized table as src/model/forward.rs:505-507 builds it).
__global__ void __launch_bounds__(256) k_embed_rows(DevW w, const uint32_t* __restrict__ ids,
                                                    float* __restrict__ out) {
  dev_row(w, ids[blockIdx.y], out + (uint64_t)blockIdx.y * w.cols, blockIdx.x, gridDim.x);
}

// hidden = row cur_token (Model::decode_step, src/model/forward.rs:556-558).
// It also clears the rows of the step's first K-split q/k/v launch (clr).
__global__ void __launch_bounds__(256) k_embed_state(DevW w, const DevState* __restrict__ s,
                                                     float* __restrict__ hidden, QkvClear clr) {
  const uint64_t row = s->cur_token;
  const uint32_t len = s->len;
  qkv_clear(clr, len, blockIdx.x, gridDim.x, threadIdx.x, blockDim.x);
  dev_row(w, row, hidden, blockIdx.x, gridDim.x);
}

// workgroups of 256 threads that cover a row, a quad per thread
static unsigned row_groups(uint64_t cols) {
  const uint64_t per = cols % 4 ? 256 : 1024;
  return (unsigned)((cols + per - 1) / per);
}

hipError_t launch_dequant_raw(uint32_t type, const uint8_t* bytes, uint64_t n, float* out,
                              hipStream_t st) {
  const uint64_t wgs = (n + 1024 * kQuads - 1) / (1024 * kQuads);
  if (wgs == 0 || wgs > 0x7fffffffull) return wgs ? hipErrorInvalidValue : hipSuccess;
  auto go = [&](auto kern) { hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(256), 0, st, bytes, n, out); };
  switch (type) {
    case T_F32: go(k_dequant_raw<T_F32>); break;
    case T_F16: go(k_dequant_raw<T_F16>); break;
    case T_Q4_0: go(k_dequant_raw<T_Q4_0>); break;
    case T_Q8_0: go(k_dequant_raw<T_Q8_0>); break;
    case T_Q4K: go(k_dequant_raw<T_Q4K>); break;
    case T_Q6K: go(k_dequant_raw<T_Q6K>); break;
    case T_Q8K: go(k_dequant_raw<T_Q8K>); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_dequant_dev(const DevW& w, uint64_t n, float* out, hipStream_t st) {
  const uint64_t rows = w.cols ? n / w.cols : 0;
  if (rows == 0) return hipSuccess;
  hipLaunchKernelGGL(k_dequant_dev, dim3(row_groups(w.cols), (unsigned)std::min<uint64_t>(rows, 32768)), dim3(256), 0,
                     st, w, rows, out);
  return hipGetLastError();
}

hipError_t launch_embed_rows(const DevW& w, const uint32_t* ids, uint64_t n_ids, float* out,
                             hipStream_t st) {
  if (n_ids == 0) return hipSuccess;
  hipLaunchKernelGGL(k_embed_rows, dim3(row_groups(w.cols), (unsigned)n_ids), dim3(256), 0, st, w, ids, out);
  return hipGetLastError();
}

hipError_t launch_embed_state(const DevW& w, const DevState* state, float* hidden, hipStream_t st,
                              const QkvClear& clr) {
  const unsigned gx = (unsigned)std::max<uint64_t>(row_groups(w.cols), (clr.floats() + 1023) / 1024);
  hipLaunchKernelGGL(k_embed_state, dim3(gx), dim3(256), 0, st, w, state, hidden, clr);
  return hipGetLastError();
}

}  // namespace ifx
