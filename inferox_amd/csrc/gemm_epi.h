// gemm_epi.h — output epilogues of the prefill GEMMs (kern_gemm.hip,
// kern_gemm_skinny.hip).  Compiled with -ffp-contract=off.
#pragma once

#include "kernels.h"

namespace ifx {

// ---------------------------------------------------------------------------
// Epilogues: v(t, n) for token t < m and output column n.
// ---------------------------------------------------------------------------
struct EpStore {  // y[t * ld + n] = v
  float* y;
  uint32_t ld;
  __device__ void operator()(uint32_t t, uint32_t n, float v, float) const { y[(uint64_t)t * ld + n] = v; }
};

struct EpResid {  // x[t * ld + n] += v (src/ops.rs:212-217)
  float* x;
  uint32_t ld;
  __device__ void operator()(uint32_t t, uint32_t n, float v, float) const {
    float* p = x + (uint64_t)t * ld + n;
    *p = *p + v;
  }
};

// Output (t, n) of a q/k/v projection at y[(row0 + t) ld + (n / head_dim)
// hstride + n % head_dim]: a row-major [t][heads * head_dim] buffer, or the
// head-major KV cache.
__device__ __forceinline__ uint64_t head_addr(uint32_t t, uint32_t n, uint32_t row0, uint32_t ld, uint64_t hstride,
                                              uint32_t head_dim) {
  return (uint64_t)(row0 + t) * ld + (uint64_t)(n / head_dim) * hstride + n % head_dim;
}

// RoPE on adjacent pairs (src/ops.rs:273-284) at position pos0 + t; `partner`
// is column n ^ 1 of the same token.
// y_f16: y holds binary16 (the f16 KV cache), rounded to nearest even.
__device__ __forceinline__ void store_y(void* y, bool f16, uint64_t i, float v) {
  if (f16) ((_Float16*)y)[i] = (_Float16)v;
  else ((float*)y)[i] = v;
}

struct EpRope {
  void* y;
  uint64_t hstride;
  uint32_t ld, row0, pos0, head_dim, rope_dim, half;
  const float2* cs;  // [pos][rope_dim / 2]
  bool y_f16;
  __device__ void operator()(uint32_t t, uint32_t n, float v, float partner) const {
    const uint32_t c = n % head_dim;
    float out = v;
    if (c < rope_dim) {
      const float2 r = cs[(uint64_t)(pos0 + t) * half + (c >> 1)];
      out = (c & 1u) ? (partner * r.y) + (v * r.x) : (v * r.x) - (partner * r.y);
    }
    store_y(y, y_f16, head_addr(t, n, row0, ld, hstride, head_dim), out);
  }
};

struct EpRows {  // the V cache append
  void* y;
  uint64_t hstride;
  uint32_t ld, row0, head_dim;
  bool y_f16;
  __device__ void operator()(uint32_t t, uint32_t n, float v, float) const {
    store_y(y, y_f16, head_addr(t, n, row0, ld, hstride, head_dim), v);
  }
};

// swiglu (src/ops.rs:190-209): mid[t][n] = (g * (1 / (1 + expf(-clamp(g, -80, 80))))) * u
struct EpSwiglu {
  float* mid;
  uint32_t ld;
  __device__ void operator()(uint32_t t, uint32_t n, float g, float u) const {
    const float c = fminf(fmaxf(g, -80.f), 80.f);
    mid[(uint64_t)t * ld + n] = (g * (1.0f / (1.0f + expf(-c)))) * u;
  }
};

template <class Ep>
struct EpTraits {
  static constexpr bool kPaired = false, kNeighbor = false;
};
template <>
struct EpTraits<EpSwiglu> {
  static constexpr bool kPaired = true, kNeighbor = false;
};
template <>
struct EpTraits<EpRope> {
  static constexpr bool kPaired = false, kNeighbor = true;
};

}  // namespace ifx
