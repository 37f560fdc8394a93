// kern_gemm_skinny.hip — one matrix against 2 to 64 tokens (gemm_skinny.h): the
// launches of matmul_qt and of a short prompt's residual projections.
#include "gemm_skinny.h"

namespace ifx {

namespace {

template <int T, int MT, int RP, class Ep>
__global__ void __launch_bounds__(kThreads, 1) k_gemm_skinny(SkinnyArgs a, Ep ep) {
  __shared__ __attribute__((aligned(16))) SkinnyLds lds;
  if constexpr (std::is_same_v<Ep, EpStore>) ep.y += (uint64_t)blockIdx.y * a.m * a.w[0].rows;  // a range's partial outputs
  skinny_tiles<T, MT, RP, false>(a, a.w[0], a.w[0], blockIdx.x, ep, lds);
}

// y = (ADD: y +) the sum of the K ranges' partial outputs, in range order.
template <bool ADD>
__global__ void __launch_bounds__(256) k_skinny_reduce(const float* __restrict__ part, uint64_t n, uint32_t ksplit,
                                                       float* __restrict__ y) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v = 0.f;
  for (uint32_t z = 0; z < ksplit; z++) v += part[z * n + i];
  y[i] = ADD ? y[i] + v : v;
}

// K is cut over workgroups only where the row tiles leave most of the chip
// idle: each range costs its partial outputs and the launch that adds them
// (~4 us), so a range keeps at least two sets of WK blocks.
Plan split_plan(uint32_t m, const GemmW& w) {
  Plan p = plan_of(m, w.cols);
  const uint32_t wk = 4 / p.mt, nblk = p.bps, nwg = workgroups(p, w.rows), sets = (nblk + wk - 1) / wk;
  const uint32_t split = std::max(1u, std::min(256u / nwg, sets / 2)), per = (sets + split - 1) / split;
  p.bps = per * wk;
  p.ksplit = (nblk + p.bps - 1) / p.bps;
  return p;
}

template <class Ep>
hipError_t launch(const SkinnyArgs& a, const Plan& p, const Ep& ep, hipStream_t st) {
  const dim3 grid(workgroups(p, a.w[0].rows), p.ksplit);
  auto go = [&](auto t) {
    constexpr int T = decltype(t)::value;
    with_tokens(a.m, [&](auto mt, auto rp) {
      hipLaunchKernelGGL((k_gemm_skinny<T, decltype(mt)::value, decltype(rp)::value, Ep>), grid, dim3(kThreads), 0, st, a, ep);
    });
    return hipGetLastError();
  };
  switch (a.w[0].type) {
    case T_Q4K: return go(std::integral_constant<int, T_Q4K>{});
    case T_Q6K: return go(std::integral_constant<int, T_Q6K>{});
    case T_Q8_0: return go(std::integral_constant<int, T_Q8_0>{});
    case T_Q4_0: return go(std::integral_constant<int, T_Q4_0>{});
    default: return hipErrorInvalidValue;
  }
}

// y (ADD: +)= x W^T
template <bool ADD>
hipError_t run(const float* x, uint32_t m, const GemmW& w, float* y, float* ws, hipStream_t st) {
  if (m == 0 || w.rows == 0) return hipSuccess;
  if (!skinny_shape(m, w)) return hipErrorInvalidValue;
  const Plan p = split_plan(m, w);
  if (p.ksplit > 1 && !ws) return hipErrorInvalidValue;
  SkinnyArgs a{};
  a.x = x;
  a.w[0] = w;
  a.m = m;
  a.k = (uint32_t)w.cols;
  a.nblk = (uint32_t)((w.cols + 255) / 256);
  a.bps = p.bps;
  if (p.ksplit == 1) return ADD ? launch(a, p, EpResid{y, w.rows}, st) : launch(a, p, EpStore{y, w.rows}, st);
  const hipError_t e = launch(a, p, EpStore{ws, w.rows}, st);
  if (e != hipSuccess) return e;
  const uint64_t n = (uint64_t)m * w.rows;
  hipLaunchKernelGGL(k_skinny_reduce<ADD>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, ws, n, p.ksplit, y);
  return hipGetLastError();
}

}  // namespace

uint64_t gemm_skinny_ws_bytes(uint32_t m, const GemmW& w) {
  if (m == 0 || w.rows == 0) return 0;
  const Plan p = split_plan(m, w);
  return p.ksplit > 1 ? (uint64_t)p.ksplit * m * w.rows * 4 : 0;
}

// ranges x workgroups <= 256 (split_plan), each p.rows x m outputs
uint64_t gemm_skinny_ws_most(uint32_t m) {
  m = std::min(m, kSkinnyRows);
  return m ? 256ull * plan_of(m, 256).rows * m * 4 : 0;
}

hipError_t gemm_skinny(const float* x, uint32_t m, const GemmW& w, float* y, float* ws, hipStream_t st) {
  return run<false>(x, m, w, y, ws, st);
}

hipError_t gemm_skinny_residual(const float* x, uint32_t m, const GemmW& w, float* h, float* ws, hipStream_t st) {
  return run<true>(x, m, w, h, ws, st);
}

}  // namespace ifx
