// gemm_skinny.h — C[t][n] = sum_k A[t][k] W[n][k] for a few tokens
// (m <= 64) against a quantized matrix: ops::matmul_t (src/ops.rs:33-44) of a
// short prompt, on the fp16 matrix cores, in one launch.
//
// Bound by the weight stream at 16 tokens and by the matrix cores at 64.  The
// tile GEMM (kern_gemm.hip) computes 128 token rows whatever m is, reads the
// operand a separate launch prepared, and cuts K over workgroups whose partial
// tiles a third launch adds: 8 tokens x 14336 x 4096 Q4_K took 38 us, this
// kernel takes 15.3 (2.2 TB/s of weights; splitting 16 instead of 8 rows, with
// its reductions through LDS, it took 20.7).
//
// Arithmetic: that of kern_gemm.hip.  Weights are the integers p of w = s p - c
// in fp16 (Q6_K: the weight as an fp16 pair), activations fp16 pairs a_hi +
// a_lo, products accumulated in f32, block scales applied in f32, the Q4_K
// minimum as one K = 32 MFMA per 256 columns against the activations' group
// sums.  The activation scale is 2^(14 - e) per row and 256-column block (there:
// per row), so the split needs no pass over the whole row first.  Products with
// a lo part go to a sum of their own (kLoSums), small beside the other: 8 steps
// of a block round at its size instead of 16 (Q4_K) or 24 (Q6_K), and the error
// against 64 bits is 0.82 (Q4_K) and 0.4 to 0.7 (Q6_K) of kern_gemm.hip's, for
// 0.4 to 0.7% of the time up to 32 tokens (8 tokens x 14336 x 4096: 15.2 -> 15.3).
// In one sum it was up to 1.06 of it over 512 columns whose largest activations
// come early.
//
// Layout: a wave owns NB = 2 tiles of 16 weight rows and every token tile; it
// loads its rows' blocks straight into registers in the layout they are
// stored in: lane n + 16g holds sub-blocks g and g + 4 of row n, and a K = 32
// step takes 8 elements of each of the four lanes' sub-blocks, so nothing is
// exchanged between lanes (Q8_0, Q4_0: 8 elements of one 32-block per lane, as
// its scale is applied per block).  The A fragments of a step are read with
// the same mapping from LDS, where the workgroup has split the f32 rows;
// 16-byte chunk c of row r lies at c ^ (r & 15), so the 16 rows of a fragment
// read fall on distinct banks.  WK of the 8 waves share a tile's K range,
// block by block (their sums meet in LDS): with few tokens the LDS holds WK
// blocks of A, and 64-row tiles fill the chip without cutting K over
// workgroups.  One barrier per WK blocks; the next blocks' weights and f32
// rows are in flight during the MFMAs.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dev_lanes.h"
#include "gemm_epi.h"
#include "kernels.h"

namespace ifx {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8, kThreads = 64 * kWaves, kNB = 2;
constexpr uint32_t kMagic = 0x64006400u;  // fp16 1024 in both halves: 0x6400 | u is 1024 + u (u < 1024)
constexpr int kSRow = 20;                 // halves per row of group sums: 8-byte reads of 16 rows on distinct banks

struct SkinnyArgs {
  const float* x;        // [m][k]
  const float* norm_w;   // NORM: x is rms_norm(x, norm_w, eps)
  float eps;
  GemmW w[3];            // one matrix; gate, up; q, k, v
  uint32_t wg[3];        // q, k, v: the first workgroup of each
  uint32_t m, k, nblk;   // nblk: 256-column blocks (the last may be short)
  uint32_t bps;          // blocks per K range (ranges over grid.y)
};

__device__ __forceinline__ h2 as_h2(uint32_t v) { return __builtin_bit_cast(h2, v); }
__device__ __forceinline__ uint32_t as_u32(h2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ h2 splat(float v) { return h2{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ h8 frag(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return __builtin_bit_cast(h8, make_uint4(a, b, c, d));
}
__device__ __forceinline__ f4 mfma(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// One wave's block (16 rows x 256 columns) of a weight matrix: load() issues
// the raw loads of tile `tile`, block b; step(s, lo) is the B operand of K
// step s in the element order 0 4 1 5 2 6 3 7 (lo: Q6_K's low part).
// Lane group g meets it with the 16-byte A chunk (8 columns) chunk0(g) ^ chunk_xor(s).
template <int T>
struct WB;

template <>
struct WB<T_Q4K> {
  static constexpr bool kMins = true, kPair = false, kPerStep = false;
  uint4 h, q[2];
  __device__ __forceinline__ void load(const GemmW& w, uint32_t tile, uint32_t b, int n, int g) {
    const uint8_t* u = w.body + (uint64_t)tile * w.tstride + (uint64_t)b * w.bstride;
    h = *(const uint4*)(u + 16 * n);
    q[0] = *(const uint4*)(u + 256 + 16 * (n + 16 * g));
    q[1] = *(const uint4*)(u + 1280 + 16 * (n + 16 * g));
  }
  static __device__ __forceinline__ int chunk0(int g) { return 4 * g; }
  static __device__ constexpr int chunk_xor(int s) { return 16 * (s >> 2) + (s & 3); }
  // 6-bit scale of sub-block g + 4 (s >> 2) (dequant.rs:141-149)
  __device__ __forceinline__ float scale(int half, int g) const {
    const uint32_t y = h.y >> (8 * g), w = h.w >> (8 * g);
    return (float)(half ? (w & 15u) | ((y >> 2) & 48u) : y & 63u);
  }
  // (1024 + q) sc - 1024 sc = q sc, one rounding of an exact integer <= 945
  __device__ __forceinline__ h8 step(int s, float sc) const {
    const uint4& Q = q[s >> 2];
    const uint32_t v = (s & 3) == 0 ? Q.x : (s & 3) == 1 ? Q.y : (s & 3) == 2 ? Q.z : Q.w;
    const h2 s2 = splat(sc), o2 = splat(-1024.f * sc);
    uint32_t r[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
      r[j] = as_u32(__builtin_elementwise_fma(as_h2(((v >> (4 * j)) & 0x000F000Fu) | kMagic), s2, o2));
    return frag(r[0], r[1], r[2], r[3]);
  }
  __device__ __forceinline__ float d() const { return h2f(h.x); }
  __device__ __forceinline__ float dstep(int) const { return 0.f; }
  // -32 dmin mn of groups 4 (g & 1) .. + 3, as fp16 hi and lo (checked to be in range at upload)
  __device__ __forceinline__ void mins(int g, h4& hi, h4& lo) const {
    const uint32_t m4 = (g & 1) ? (((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)) : h.z & 0x3F3F3F3Fu;
    const float dmin = h2f(h.x >> 16);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float c = -(dmin * (float)((m4 >> (8 * i)) & 0xffu)) * 32.f;
      hi[i] = (_Float16)c;
      lo[i] = (_Float16)(c - (float)hi[i]);
    }
  }
};

template <>
struct WB<T_Q6K> {
  static constexpr bool kMins = false, kPair = true, kPerStep = false;
  uint4 l[2], hq;
  uint32_t sc, dd;
  bool sgn;
  __device__ __forceinline__ void load(const GemmW& w, uint32_t tile, uint32_t b, int n, int g) {
    const uint8_t* u = w.body + (uint64_t)tile * w.tstride + (uint64_t)b * w.bstride;
    const int lane = n + 16 * g;
    l[0] = *(const uint4*)(u + 16 * lane);
    l[1] = *(const uint4*)(u + 1024 + 16 * lane);
    hq = *(const uint4*)(u + 2048 + 16 * lane);
    sc = *(const uint32_t*)(u + 3072 + 4 * lane);
    dd = *(const uint16_t*)(u + 3328 + 2 * n);
    sgn = w.q6_signed;
  }
  static __device__ __forceinline__ int chunk0(int g) { return 4 * g; }
  static __device__ constexpr int chunk_xor(int s) { return 16 * (s >> 2) + (s & 3); }
  __device__ __forceinline__ float dstep(int) const { return 0.f; }
  // The weight pair in packed fp16: d sc (19 bits) = dh + dl exactly; wh =
  // fl(dh t), r = dh t - wh exactly, wl = fl(dl t + r), t = q - 32
  // (kern_gemm.hip: within 3.3e-7 relative of the f32 weight).
  __device__ __forceinline__ void step(int s, h8& hi, h8& lo) const {
    const int c = 2 * (s >> 2) + ((s >> 1) & 1);  // the lane's 16-element part
    const uint4& Q = l[s >> 2];
    const uint32_t v = (s & 3) == 0 ? Q.x : (s & 3) == 1 ? Q.y : (s & 3) == 2 ? Q.z : Q.w;
    const uint32_t hw = c == 0 ? hq.x : c == 1 ? hq.y : c == 2 ? hq.z : hq.w;
    const uint32_t sb = (sc >> (8 * c)) & 0xffu;
    const float ds = h2f(dd) * (sgn ? (float)(int8_t)sb : (float)sb);  // exact: 11 x 8 bits
    const _Float16 dh = (_Float16)ds, dl = (_Float16)(ds - (float)dh);
    const h2 m2 = splat(-1056.f), dh2 = h2{dh, dh}, dl2 = h2{dl, dl};
    uint32_t vh[4], vl[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      // high parts of elements j, j + 4 of chunk s & 1: bits 8 (j / 2) + 2 (j & 1) + 4 (s & 1), 16 apart
      const int sh = 8 * (j >> 1) + 2 * (j & 1) + 4 * (s & 1);
      const uint32_t hb = (sh >= 4 ? hw >> (sh - 4) : hw << (4 - sh)) & 0x00300030u;
      const h2 t = as_h2(((v >> (4 * j)) & 0x000F000Fu) | hb | kMagic) + m2;
      const h2 wh = dh2 * t;
      const h2 r = __builtin_elementwise_fma(dh2, t, -wh);
      vh[j] = as_u32(wh);
      vl[j] = as_u32(__builtin_elementwise_fma(dl2, t, r));
    }
    hi = frag(vh[0], vh[1], vh[2], vh[3]);
    lo = frag(vl[0], vl[1], vl[2], vl[3]);
  }
};

// bytes j of x and y as the fp16-pair word (x_j, 0, y_j, 0)
__device__ __forceinline__ uint32_t byte_pair(uint32_t x, uint32_t y, int j) {
  return __builtin_amdgcn_perm(y, x, (uint32_t)j | (0x0cu << 8) | ((uint32_t)(4 + j) << 16) | (0x0cu << 24));
}

// Q8_0, Q4_0: rows of 32-blocks; a lane's 8 elements of each of the block's
// eight 32-blocks.  In a row's short last block the 32-blocks past its end
// are the next row's (past the last row, kTensorPad bytes of the allocation):
// the A chunks they meet are zero, and their scales are not applied.
template <bool Q8>
struct WB32 {
  static constexpr bool kMins = false, kPair = false, kPerStep = true;
  uint2 q[8];
  uint4 dd;
  __device__ __forceinline__ void load(const GemmW& w, uint32_t tile, uint32_t b, int n, int g) {
    const uint32_t row = min(tile * 16 + (uint32_t)n, w.rows - 1);
    const uint64_t i = (uint64_t)row * (uint32_t)(w.cols >> 5) + 8 * b;
    const uint8_t* p = w.body + (Q8 ? i * 32 + 8 * g : i * 16 + 8 * (g & 1));
#pragma unroll
    for (int s = 0; s < 8; s++) q[s] = *(const uint2*)(p + (Q8 ? 32 : 16) * s);
    __builtin_memcpy(&dd, w.scal + 2 * i, 16);  // 2-byte aligned where a row is no whole number of 256 columns
  }
  static __device__ __forceinline__ int chunk0(int g) { return g; }
  static __device__ constexpr int chunk_xor(int s) { return 4 * s; }
  __device__ __forceinline__ h8 step(int s, int g) const {
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (Q8)  // int8 -> 1024 + (q + 128) by flipping the sign bit under the fp16 1024 pattern
        v[j] = as_u32(as_h2(byte_pair(q[s].x, q[s].y, j) ^ 0x64806480u) + splat(-1152.f));
      else  // low nibbles: elements 0..15, high: 16..31; 1024 + q - 1032 = q - 8
        v[j] = as_u32(as_h2(((byte_pair(q[s].x, q[s].y, j) >> (4 * (g >> 1))) & 0x000F000Fu) | kMagic) + splat(-1032.f));
    }
    return frag(v[0], v[1], v[2], v[3]);
  }
  __device__ __forceinline__ float dstep(int s) const {
    const uint32_t v = s < 2 ? dd.x : s < 4 ? dd.y : s < 6 ? dd.z : dd.w;
    return h2f(v >> (16 * (s & 1)));
  }
};
template <>
struct WB<T_Q8_0> : WB32<true> {};
template <>
struct WB<T_Q4_0> : WB32<false> {};

// MT token tiles of 16; MT WK = 4 (the LDS holds two sets of 64 row-blocks).
// RP: the token rows staged, 16 MT, or 8 of 16 (the others' LDS rows hold
// anything: a fragment row reaches its own output row alone).
// PAIRED: w0 / w1 are gate and up, the wave's two tiles the same rows of both.
// NORM: x * norm_w is staged, each row's sum of squares gathered on the way,
// and the norm's scale (one scalar per row) applied to the row's outputs.
constexpr int kRb = 64;  // row-blocks per set
struct SkinnyLds {
  _Float16 pl[2][2][kRb * 256];  // [set][hi, lo][row-block][256]
  _Float16 gs[2][kRb][kSRow];    // group sums (Q4_K)
  float inv[2][kRb];             // 2^(e - 14) of each row-block
  float rss[kRb];                // NORM: sums of squares
};
template <int T, int MT, int RP, bool NORM, class Ep>
__device__ __forceinline__ void skinny_tiles(const SkinnyArgs& a, const GemmW& w0, const GemmW& w1, uint32_t wgx,
                                             const Ep& ep, SkinnyLds& lds) {
  using W = WB<T>;
  constexpr bool PAIRED = EpTraits<Ep>::kPaired;
  constexpr int WK = 4 / MT, WN = kWaves / WK, RB = 16 * MT * WK;
  static_assert(RB == kRb, "row-blocks per set");
  constexpr int NC = RP * WK * 32 / kThreads;                        // chunks per thread per set
  constexpr int NW = RP == 64 ? 1 : RP == 32 ? 2 : NC;               // different blocks among them
  auto& pl = lds.pl;
  auto& gs = lds.gs;
  auto& inv = lds.inv;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave / WK, wk = wave % WK, fi = lane & 15, fg = lane >> 4;
  const uint32_t rows = w0.rows, tiles = (rows + 15) / 16;
  // tile nb of the wave: tile0 + nb, or (PAIRED) tile0 of both matrices
  const uint32_t tile0 = (wgx * WN + (uint32_t)wn) * (PAIRED ? 1 : kNB);
  const uint32_t b0 = blockIdx.y * a.bps, b1 = min(a.nblk, b0 + a.bps), iters = (b1 - b0 + WK - 1) / WK;

  // staging role j: chunk ch of token row `row(j)`, block `blk(j)` of the set,
  // which is LDS row-block rb0 + kRbStep j
  const int g32 = tid >> 5, rb0 = RP == 8 ? (g32 >> 3) * 16 + (g32 & 7) : g32;
  constexpr int kRbStep = RP == 8 ? 32 : 16;
  float4 xr[NC][2], nr[NORM ? NW : 1][2];
  float ssq[NC];
#pragma unroll
  for (int j = 0; j < NC; j++) ssq[j] = 0.f;
  const int ch = tid & 31;
  static_assert(kThreads / 32 == 16, "row-blocks of one staging round");
  constexpr int kPlane = RB * 512, kSet = 2 * kPlane;  // bytes
  const uint32_t wr0 = (uint32_t)(rb0 * 512 + 16 * (ch ^ (rb0 & 15)));
  auto load_x = [&](uint32_t it) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; j++) {
      const int rb = rb0 + kRbStep * j, row = rb % (16 * MT), blk = rb / (16 * MT);
      const uint32_t b = b0 + it * WK + (uint32_t)blk, col = 256 * b + 8 * (uint32_t)ch;
      const bool ok = (uint32_t)row < a.m && b < b1 && col < a.k;
      const float4* p = (const float4*)(a.x + (uint64_t)(ok ? row : 0) * a.k + (ok ? col : 0));
      const float4 z = make_float4(0.f, 0.f, 0.f, 0.f), v0 = p[0], v1 = p[1];
      xr[j][0] = ok ? v0 : z;
      xr[j][1] = ok ? v1 : z;
      if constexpr (NORM) {
        if (j % (NC / NW) == 0) {  // the chunks of one block share its norm weights
          const float4* q = (const float4*)(a.norm_w + (col < a.k ? col : 0));
          nr[j / (NC / NW)][0] = q[0];
          nr[j / (NC / NW)][1] = q[1];
        }
      }
    }
  };
  auto stage = [&](int set) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; j++) {
      const int rb = rb0 + kRbStep * j;
      float v[8] = {xr[j][0].x, xr[j][0].y, xr[j][0].z, xr[j][0].w, xr[j][1].x, xr[j][1].y, xr[j][1].z, xr[j][1].w};
      if constexpr (NORM) {
        const float4 g0 = nr[j / (NC / NW)][0], g1 = nr[j / (NC / NW)][1];
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int k = 0; k < 8; k++) {
          ssq[j] = fmaf(v[k], v[k], ssq[j]);
          v[k] *= g[k];
        }
      }
      float mx = 0.f;
#pragma unroll
      for (int k = 0; k < 8; k++) mx = fmaxf(mx, fabsf(v[k]));
      mx = bfly<16, true>(mx);
      mx = bfly<8, true>(mx);
      mx = bfly<4, true>(mx);
      mx = bfly<2, true>(mx);
      mx = bfly<1, true>(mx);
      int e = (int)((__float_as_uint(mx) >> 23) & 255u) - 127;
      e = e < -100 ? -100 : e;
      const float sc = ldexpf(1.f, 14 - e);
      h8 vh, vl;
      float s8 = 0.f;
#pragma unroll
      for (int p = 0; p < 8; p++) {
        const float y = v[(p >> 1) + 4 * (p & 1)] * sc;
        vh[p] = (_Float16)y;
        vl[p] = (_Float16)(y - (float)vh[p]);
        s8 += y;
      }
      uint8_t* at = (uint8_t*)pl + (wr0 + (uint32_t)(kSet * set + kRbStep * 512 * j));  // rb & 15 == rb0 & 15
      *(h8*)at = vh;
      *(h8*)(at + kPlane) = vl;
      if (ch == 0) inv[set][rb] = ldexpf(1.f, e - 14);
      if constexpr (W::kMins) {
        s8 = bfly<1, false>(s8);
        s8 = bfly<2, false>(s8);
        if ((ch & 3) == 0) {
          const float sg = s8 * 0.03125f;
          const _Float16 sh = (_Float16)sg;
          gs[set][rb][ch >> 2] = sh;
          gs[set][rb][8 + (ch >> 2)] = (_Float16)(sg - (float)sh);
        }
      }
    }
  };
  // The products with a lo part summed apart; not in a layer's projections of
  // more than 32 tokens, whose registers are full (in one sum a short prompt's
  // logits are within 0.5 to 0.8 of the error that the same ids fed one at a
  // time have).
  constexpr bool kLoSums = !W::kPerStep && !(NORM && MT == 4);
  // two sets of weights (this iteration's, the next one's), or one, refilled
  // once it is used (64 tokens with Q8_0 and Q4_0, or with the second sums: the
  // registers are full; Q4_K 4096 x 14336 34.9 -> 34.1 us with the one set)
  constexpr int kWSets = MT == 4 && (W::kPerStep || kLoSums) ? 1 : 2;
  W wb[kWSets][kNB];
  auto load_w = [&](W (&w)[kNB], uint32_t it) __attribute__((always_inline)) {
    const uint32_t b = min(b0 + it * WK + (uint32_t)wk, a.nblk - 1);
#pragma unroll
    for (int nb = 0; nb < kNB; nb++)
      w[nb].load(PAIRED && nb ? w1 : w0, min(tile0 + (uint32_t)(PAIRED ? 0 : nb), tiles - 1), b, fi, fg);
  };

  f4 acc[kNB][MT];
#pragma unroll
  for (int nb = 0; nb < kNB; nb++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[nb][mt] = f4{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const W (&w)[kNB], uint32_t it) __attribute__((always_inline)) {
    const int set = (int)(it & 1);
    // 32-blocks of the wave's block that the row has
    const uint32_t have = min(8u, (a.k >> 5) - min(a.k >> 5, 8 * (b0 + it * WK + (uint32_t)wk)));
    const int r0 = wk * 16 * MT;  // the wave's block of the set
    // products of the hi parts, and (kLoSums) those with a lo part
    f4 cs[kNB][MT], cl[kNB][MT];
#pragma unroll
    for (int nb = 0; nb < kNB; nb++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) cs[nb][mt] = cl[nb][mt] = f4{0.f, 0.f, 0.f, 0.f};
    float sc[kNB];
    // the fragment address of step 0; step s differs by an exclusive or (kept
    // from being hoisted, as eight addresses per set, into spilled registers)
    uint32_t rd0 = (uint32_t)((r0 + fi) * 512 + 16 * (W::chunk0(fg) ^ fi) + kSet * set);
    asm volatile("" : "+v"(rd0));
#pragma unroll
    for (int s = 0; s < 8; s++) {
      const uint8_t* at = (const uint8_t*)pl + (rd0 ^ (uint32_t)(16 * W::chunk_xor(s)));
      h8 ah[MT], al[MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        ah[mt] = *(const h8*)(at + 16 * 512 * mt);
        al[mt] = *(const h8*)(at + 16 * 512 * mt + kPlane);
      }
      // every tile's product with a_hi, then with a_lo: independent chains
      h8 bh[kNB], bl[kNB];
      f4 t[kNB][MT], u[kNB][MT];
#pragma unroll
      for (int nb = 0; nb < kNB; nb++) {
        if constexpr (W::kPair) {
          w[nb].step(s, bh[nb], bl[nb]);
        } else if constexpr (W::kPerStep) {
          bh[nb] = w[nb].step(s, fg);
        } else {
          if ((s & 3) == 0) sc[nb] = w[nb].scale(s >> 2, fg);
          bh[nb] = w[nb].step(s, sc[nb]);
        }
      }
#pragma unroll
      for (int nb = 0; nb < kNB; nb++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
          t[nb][mt] = mfma(ah[mt], bh[nb], W::kPerStep ? f4{0.f, 0.f, 0.f, 0.f} : cs[nb][mt]);
#pragma unroll
      for (int nb = 0; nb < kNB; nb++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) u[nb][mt] = mfma(al[mt], bh[nb], kLoSums ? cl[nb][mt] : t[nb][mt]);
      if constexpr (W::kPair) {
#pragma unroll
        for (int nb = 0; nb < kNB; nb++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++) u[nb][mt] = mfma(ah[mt], bl[nb], u[nb][mt]);
      }
#pragma unroll
      for (int nb = 0; nb < kNB; nb++) {
        const float d = W::kPerStep && (uint32_t)s < have ? w[nb].dstep(s) : 0.f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          if constexpr (W::kPerStep) {
#pragma unroll
            for (int r = 0; r < 4; r++) cs[nb][mt][r] = fmaf(d, u[nb][mt][r], cs[nb][mt][r]);
            asm volatile("" : "+v"(cs[nb][mt]));  // summed here: not put off with the products held in registers
          } else {
            cs[nb][mt] = kLoSums ? t[nb][mt] : u[nb][mt];
            if (kLoSums) cl[nb][mt] = u[nb][mt];
          }
        }
      }
      // four steps' fragments live at once, or one (all eight hoisted spill)
      if (MT > 1 || W::kPerStep || (s & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (W::kMins) {
      // lanes of group g: S_hi (g < 2) or S_lo of groups 4 (g & 1) .. + 3
      // against the hi parts, and S_hi against the lo parts, as one K = 32 MFMA
      const h4 z = {0, 0, 0, 0};
      h8 as[MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const h4 s = *(const h4*)&gs[set][r0 + 16 * mt + fi][4 * fg];
        const h4 s2 = fg < 2 ? s : z;
        as[mt] = __builtin_shufflevector(s, s2, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int nb = 0; nb < kNB; nb++) {
        h4 hi, lo;
        w[nb].mins(fg, hi, lo);
        if (fg >= 2) lo = z;
        const h8 bm = __builtin_shufflevector(hi, lo, 0, 1, 2, 3, 4, 5, 6, 7);
        const float d = w[nb].d();
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          if (kLoSums) {  // d cs is rounded only with the minimum added
            const f4 mn = mfma(as[mt], bm, cl[nb][mt] * d);
#pragma unroll
            for (int r = 0; r < 4; r++) cs[nb][mt][r] = fmaf(d, cs[nb][mt][r], mn[r]);
          } else {
            cs[nb][mt] = mfma(as[mt], bm, cs[nb][mt] * d);
          }
        }
      }
    }
    if constexpr (kLoSums && !W::kMins) {
#pragma unroll
      for (int nb = 0; nb < kNB; nb++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) cs[nb][mt] += cl[nb][mt];
    }
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const float4 iv = *(const float4*)&inv[set][r0 + 16 * mt + 4 * fg];
#pragma unroll
      for (int nb = 0; nb < kNB; nb++) {
        acc[nb][mt][0] = fmaf(iv.x, cs[nb][mt][0], acc[nb][mt][0]);
        acc[nb][mt][1] = fmaf(iv.y, cs[nb][mt][1], acc[nb][mt][1]);
        acc[nb][mt][2] = fmaf(iv.z, cs[nb][mt][2], acc[nb][mt][2]);
        acc[nb][mt][3] = fmaf(iv.w, cs[nb][mt][3], acc[nb][mt][3]);
      }
    }
  };

  // set it & 1 is computed while set it + 1 is staged; its last readers left
  // before the barrier that ended iteration it - 1
  load_x(0);
  load_w(wb[0], 0);
  stage(0);
  __syncthreads();
  auto iter = [&](uint32_t it, W (&cur)[kNB], W (&next)[kNB]) __attribute__((always_inline)) {
    const bool more = it + 1 < iters;
    if (more) {
      load_x(it + 1);
      if (kWSets == 2) load_w(next, it + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    compute(cur, it);
    __builtin_amdgcn_sched_barrier(0);
    if (more) {
      if (kWSets == 1) load_w(next, it + 1);
      stage((int)((it + 1) & 1));
    }
    __syncthreads();
  };
  for (uint32_t it = 0; it < iters; it += 2) {
    iter(it, wb[0], wb[kWSets - 1]);
    if (it + 1 < iters) iter(it + 1, wb[kWSets - 1], wb[0]);
  }

  // the norm scale of a token: 1 / sqrt(mean(x^2) + eps) (src/ops.rs:162-167)
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < NC; j++) {
      float s = ssq[j];
      s = bfly<16, false>(s);
      s = bfly<8, false>(s);
      s = bfly<4, false>(s);
      s = bfly<2, false>(s);
      s = bfly<1, false>(s);
      if (ch == 0) lds.rss[rb0 + kRbStep * j] = s;
    }
    if (WK == 1) __syncthreads();
  }
  // the WK waves' sums through LDS (free after the last barrier)
  if constexpr (WK > 1) {
    f4* red = (f4*)pl;
#pragma unroll
    for (int nb = 0; nb < kNB; nb++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) red[((wave * kNB + nb) * MT + mt) * 64 + lane] = acc[nb][mt];
    __syncthreads();
#pragma unroll
    for (int nb = 0; nb < kNB; nb++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        f4 v = red[((wn * WK * kNB + nb) * MT + mt) * 64 + lane];
#pragma unroll
        for (int q = 1; q < WK; q++) v += red[(((wn * WK + q) * kNB + nb) * MT + mt) * 64 + lane];
        acc[nb][mt] = v;
      }
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    if constexpr (NORM) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float s = 0.f;
#pragma unroll
        for (int q = 0; q < WK; q++) s += lds.rss[16 * MT * q + 16 * mt + 4 * fg + r];
        const float sc = 1.0f / sqrtf(s / (float)a.k + a.eps);
#pragma unroll
        for (int nb = 0; nb < kNB; nb++) acc[nb][mt][r] *= sc;
      }
    }
#pragma unroll
    for (int nb = 0; nb < (PAIRED ? 1 : kNB); nb++) {
      if (WK > 1 && (nb * MT + mt) % WK != wk) continue;  // each wave stores its share
      const uint32_t n = 16 * (tile0 + (uint32_t)nb) + (uint32_t)fi;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const uint32_t t = 16 * mt + 4 * fg + r;
        const float v = acc[nb][mt][r];
        float partner = 0.f;
        if (PAIRED) partner = acc[kNB - 1][mt][r];
        else if (EpTraits<Ep>::kNeighbor) partner = lane_xor1(v);
        if (t >= a.m || n >= rows) continue;
        ep(t, n, v, partner);
      }
    }
  }
}

// The launch's token tiles, and how K is cut over workgroups.
struct Plan {
  uint32_t mt, rows, ksplit, bps;  // rows: weight rows per workgroup
};
inline Plan plan_of(uint32_t m, uint64_t cols) {
  Plan p;
  p.mt = m <= 16 ? 1 : m <= 32 ? 2 : 4;
  p.rows = kWaves / (4 / p.mt) * kNB * 16;
  p.ksplit = 1;
  p.bps = (uint32_t)((cols + 255) / 256);
  return p;
}
inline uint32_t workgroups(const Plan& p, uint32_t rows) { return (rows + p.rows - 1) / p.rows; }

// kern.template operator()<MT, RP>() for m tokens
template <class F>
void with_tokens(uint32_t m, F f) {
  if (m <= 8) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 8>{});
  else if (m <= 16) f(std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{});
  else if (m <= 32) f(std::integral_constant<int, 2>{}, std::integral_constant<int, 32>{});
  else f(std::integral_constant<int, 4>{}, std::integral_constant<int, 64>{});
}

inline bool skinny_shape(uint32_t m, const GemmW& w) {
  const bool k256 = w.type == T_Q4K || w.type == T_Q6K;
  return m >= 1 && m <= kSkinnyRows && w.rows && w.cols && w.cols % (k256 ? 256 : 32) == 0;
}

}  // namespace

}  // namespace ifx
