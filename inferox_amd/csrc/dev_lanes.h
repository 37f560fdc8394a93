// dev_lanes.h — lane exchanges and reductions within a wave (gfx950).
#pragma once

#include <hip/hip_runtime.h>

namespace ifx {

// ---- lane exchanges without LDS round trips (whole wave active) ----
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ float lane_xor1(float v) { return dpp_mov<0xb1>(v); }  // quad_perm [1,0,3,2]
__device__ __forceinline__ float lane_xor2(float v) { return dpp_mov<0x4e>(v); }  // quad_perm [2,3,0,1]
// One butterfly step: v op (v of lane ^ OFF) in every lane.  OFF 32 / 16: the
// gfx950 swaps of the two halves / of rows 0<->1, 2<->3 return {own, partner}
// in some order (the pair's op either way); 8: row_ror:8; 4: row_half_mirror
// then quad_perm [3,2,1,0]; 2, 1: quad_perm.  The operands are those of a
// __shfl_xor butterfly, so sums come out bit for bit the same.
template <int OFF, bool MAX>
__device__ __forceinline__ float bfly(float v) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8 || OFF == 16 || OFF == 32, "lane offset");
  float a = v, b;
  if constexpr (OFF == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else if constexpr (OFF == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
  } else if constexpr (OFF == 8) {
    b = dpp_mov<0x128>(v);
  } else if constexpr (OFF == 4) {
    b = dpp_mov<0x1b>(dpp_mov<0x141>(v));
  } else if constexpr (OFF == 2) {
    b = lane_xor2(v);
  } else {
    b = lane_xor1(v);
  }
  return MAX ? fmaxf(a, b) : a + b;
}
// sum / max over the 64 lanes, in every lane (the xor butterfly 32, 16, ..., 1)
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v) {
  v = bfly<32, MAX>(v);
  v = bfly<16, MAX>(v);
  v = bfly<8, MAX>(v);
  v = bfly<4, MAX>(v);
  v = bfly<2, MAX>(v);
  return bfly<1, MAX>(v);
}
__device__ __forceinline__ float wave_sum(float v) { return wave_reduce<false>(v); }

}  // namespace ifx
