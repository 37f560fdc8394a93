// kern_gemm_skinny_layer.hip — a short prompt's normed projections
// (gemm_skinny.h): q/k/v with RoPE and the cache append, and gate/up with
// SwiGLU, RMSNorm included, one launch each (src/model/forward.rs:215-337).
#include "gemm_skinny.h"

namespace ifx {

namespace {

// Outputs of segment seg (0: q, 1: k, 2: v; uniform over the workgroup).
struct EpQkvRows {
  EpRope q, k;
  EpRows v;
  uint32_t seg;
  __device__ void operator()(uint32_t t, uint32_t n, float x, float partner) const {
    if (seg == 0) q(t, n, x, partner);
    else if (seg == 1) k(t, n, x, partner);
    else v(t, n, x, partner);
  }
};

}  // namespace
template <>
struct EpTraits<EpQkvRows> {
  static constexpr bool kPaired = false, kNeighbor = true;
};
namespace {

// one of three uniform values, kept in scalar registers (a segment indexed
// from the kernel's arguments would go through scratch memory)
template <class V>
__device__ __forceinline__ V pick(uint32_t seg, V a, V b, V c) {
  asm("" : "+s"(a), "+s"(b), "+s"(c));
  return seg == 0 ? a : seg == 1 ? b : c;
}

// TA: the type of q and k, TB: of v.
template <int TA, int TB, int MT, int RP>
__global__ void __launch_bounds__(kThreads, 1) k_skinny_qkv(SkinnyArgs a, EpQkvRows ep) {
  __shared__ __attribute__((aligned(16))) SkinnyLds lds;
  const uint32_t b = blockIdx.x, seg = b < a.wg[1] ? 0u : b < a.wg[2] ? 1u : 2u;
  ep.seg = seg;
  const uint32_t wgx = b - (seg == 0 ? 0u : seg == 1 ? a.wg[1] : a.wg[2]);
  GemmW w = a.w[0];
  w.body = pick(seg, a.w[0].body, a.w[1].body, a.w[2].body);
  w.scal = pick(seg, a.w[0].scal, a.w[1].scal, a.w[2].scal);
  w.rows = pick(seg, a.w[0].rows, a.w[1].rows, a.w[2].rows);
  w.q6_signed = pick(seg, a.w[0].q6_signed, a.w[1].q6_signed, a.w[2].q6_signed);
  w.tstride = pick(seg, a.w[0].tstride, a.w[1].tstride, a.w[2].tstride);
  w.bstride = pick(seg, a.w[0].bstride, a.w[1].bstride, a.w[2].bstride);
  if (TA == TB || seg < 2) skinny_tiles<TA, MT, RP, true>(a, w, w, wgx, ep, lds);
  else skinny_tiles<TB, MT, RP, true>(a, w, w, wgx, ep, lds);
}

template <int T, int MT, int RP>
__global__ void __launch_bounds__(kThreads, 1) k_skinny_swiglu(SkinnyArgs a, EpSwiglu ep) {
  __shared__ __attribute__((aligned(16))) SkinnyLds lds;
  skinny_tiles<T, MT, RP, true>(a, a.w[0], a.w[1], blockIdx.x, ep, lds);
}

SkinnyArgs args_of(const float* x, uint32_t m, const float* norm_w, float eps, uint64_t cols) {
  SkinnyArgs a{};
  a.x = x;
  a.norm_w = norm_w;
  a.eps = eps;
  a.m = m;
  a.k = (uint32_t)cols;
  a.nblk = a.bps = (uint32_t)((cols + 255) / 256);  // one range: the norm's sums need whole rows
  return a;
}

}  // namespace

bool skinny_qkv_types(uint32_t tq, uint32_t tk, uint32_t tv) {
  return tq == tk && gemm_type(tq) && (tv == tq || (tq == T_Q4K && tv == T_Q6K));
}

hipError_t skinny_qkv(const float* x, uint32_t m, const float* norm_w, float eps, const GemmW (&w)[3],
                      const SkinnyQkv& d, hipStream_t st) {
  if (!skinny_qkv_types(w[0].type, w[1].type, w[2].type) || d.head_dim == 0 || d.head_dim % 2 || d.rope_dim % 2 ||
      d.rope_dim > d.head_dim)
    return hipErrorInvalidValue;
  for (const GemmW& q : w)
    if (!skinny_shape(m, q) || q.cols != w[0].cols) return hipErrorInvalidValue;
  SkinnyArgs a = args_of(x, m, norm_w, eps, w[0].cols);
  const Plan p = plan_of(m, w[0].cols);
  uint32_t wgs = 0;
  for (int i = 0; i < 3; i++) {
    a.w[i] = w[i];
    a.wg[i] = wgs;
    wgs += workgroups(p, w[i].rows);
  }
  const uint32_t half = d.rope_dim / 2;
  const EpRope eq{d.q, d.head_dim, w[0].rows, 0, d.pos0, d.head_dim, d.rope_dim, half, d.cs, false};
  const EpRope ek{d.k, d.kv_stride, d.head_dim, d.row0, d.pos0, d.head_dim, d.rope_dim, half, d.cs, d.kv_f16};
  const EpRows ev{d.v, d.kv_stride, d.head_dim, d.row0, d.head_dim, d.kv_f16};
  const EpQkvRows ep{eq, ek, ev, 0};
  auto go = [&](auto ta, auto tb) {
    constexpr int TA = decltype(ta)::value, TB = decltype(tb)::value;
    with_tokens(m, [&](auto mt, auto rp) {
      hipLaunchKernelGGL((k_skinny_qkv<TA, TB, decltype(mt)::value, decltype(rp)::value>), dim3(wgs), dim3(kThreads), 0,
                         st, a, ep);
    });
    return hipGetLastError();
  };
  using Q4K = std::integral_constant<int, T_Q4K>;
  using Q6K = std::integral_constant<int, T_Q6K>;
  using Q80 = std::integral_constant<int, T_Q8_0>;
  using Q40 = std::integral_constant<int, T_Q4_0>;
  switch (w[0].type) {
    case T_Q4K: return w[2].type == T_Q6K ? go(Q4K{}, Q6K{}) : go(Q4K{}, Q4K{});
    case T_Q6K: return go(Q6K{}, Q6K{});
    case T_Q8_0: return go(Q80{}, Q80{});
    default: return go(Q40{}, Q40{});
  }
}

hipError_t skinny_swiglu(const float* x, uint32_t m, const float* norm_w, float eps, const GemmW& gate, const GemmW& up,
                         float* mid, hipStream_t st) {
  if (!skinny_shape(m, gate) || up.type != gate.type || up.rows != gate.rows || up.cols != gate.cols)
    return hipErrorInvalidValue;
  SkinnyArgs a = args_of(x, m, norm_w, eps, gate.cols);
  a.w[0] = gate;
  a.w[1] = up;
  const Plan p = plan_of(m, gate.cols);
  const uint32_t wgs = (gate.rows + p.rows / kNB - 1) / (p.rows / kNB);
  const EpSwiglu ep{mid, gate.rows};
  auto go = [&](auto t) {
    constexpr int T = decltype(t)::value;
    with_tokens(m, [&](auto mt, auto rp) {
      hipLaunchKernelGGL((k_skinny_swiglu<T, decltype(mt)::value, decltype(rp)::value>), dim3(wgs), dim3(kThreads), 0, st,
                         a, ep);
    });
    return hipGetLastError();
  };
  switch (gate.type) {
    case T_Q4K: return go(std::integral_constant<int, T_Q4K>{});
    case T_Q6K: return go(std::integral_constant<int, T_Q6K>{});
    case T_Q8_0: return go(std::integral_constant<int, T_Q8_0>{});
    case T_Q4_0: return go(std::integral_constant<int, T_Q4_0>{});
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ifx
