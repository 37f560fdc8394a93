// kern_gemv.hip — fused dequant-GEMV for batch-1 decode on gfx950.
//
// Replaces the decode use of ops::matmul_t (src/ops.rs:33-44,104-134) fed by
// the per-call f32 dequant of Weights::tensor_f32_by_index
// (src/gguf/weights.rs:66-74): y = W x with W read once from HBM in its
// quantized form and decoded in registers.  This file holds the f32-dot path
// (Q8_0, Q4_0, Q8_K, F32, F16) and the launcher of every GEMV; Q4_K and Q6_K
// matrices go to the int8-MFMA kernel of kern_gemv_mfma.hip.
//
// Work decomposition
//   * A row's 16-byte pieces lie one after another; lane l of the L lanes that
//     share a row takes pieces l, l + L, ... (K of them), so every weight load
//     of a wave covers contiguous memory.  The lane's x values (K pieces of
//     them) stay in registers for all the rows the wave runs: no barrier
//     between the kernel's start and its first dot product.  A launch
//     on a small matrix is that start (the x loads, a few hundred cycles of
//     arithmetic, the row reduction), not the stream: with x staged through
//     LDS, 9 of 64 lanes at work on rows of 288 and 9 workgroups for 288 rows,
//     a turn of the tiny model (24 steps) took 5534 us, now 4398.  A large
//     matrix streams: 14336 x 4096 Q8_0 takes 12.2 us (5.1 TB/s; 16.6 before,
//     with one unit of loads in flight).
//   * Rows of at most 64 pieces (K = 1): L = 16, 32 or 64 lanes per row, so a
//     wave runs 64 / L units at once.  Longer rows: a wave per unit up to
//     4096 columns; past that S waves of a workgroup share each row (their
//     sums meet in LDS, one barrier per unit).
//   * A unit is two rows (2u, 2u + 1: a RoPE pair), or row u of gate and up.
//     Each wave keeps the loads of two units in flight (one where a row takes
//     32 registers or more) and refills a row's registers as soon as it is
//     summed.
//   * RMSNorm (ops::rms_norm, src/ops.rs:155-168) costs no launch: x * w is
//     formed in registers, every group of lanes sums x . x over its own
//     pieces (the whole row), and the scale, one scalar per vector, is applied
//     to the row sums.
//   * The epilogue fuses RoPE + KV append (QKV), SwiGLU (gate/up), the
//     residual add (O, down) or the logits store + greedy argmax (head).
// Compiled with -ffp-contract=off: only the explicit fmaf below are fused.
#include <algorithm>

#include "dev_lanes.h"
#include "gemv_epi.h"

namespace ifx {

namespace {

constexpr int kWavesNarrow = 4;  // waves per workgroup, a wave per unit
constexpr int kWavesWide = 8;    // S = 2, 4 or 8 of them per row

struct KArgs {
  GemvSeg seg[3];
  uint32_t nunits[3];  // per logical segment (paired: one logical segment)
  uint32_t total;      // their sum
  uint32_t cols, pieces;
  uint32_t lg_lanes;   // log2 of the lanes per row (6 unless K = 1)
  uint32_t split;      // waves per row
  const float* x;
  const float* norm_w;
  float eps;
};

__device__ __forceinline__ float cvtb(uint32_t v, int b) { return (float)((v >> (8 * b)) & 0xffu); }
// Hides a masked word from the combiner so that cvtb(w, k) selects
// v_cvt_f32_ubyte<k> (one instruction) instead of a bit-field extract of the
// unmasked word followed by a convert.
__device__ __forceinline__ uint32_t opaque(uint32_t v) {
  asm("" : "+v"(v));
  return v;
}
// byte b of v as a signed int8, to f32 (v_bfe_i32 + v_cvt_f32_i32)
__device__ __forceinline__ float sbyte(int v, int b) { return (float)((v << (24 - 8 * b)) >> 24); }

typedef float f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ldw(const uint8_t* p) {
  return *(const uint4*)p;
}

// ---------------------------------------------------------------------------
// Per-type pieces: 16 bytes of a row's quants (and the scale they need) in
// registers, and their dot product with the piece's kE x values.  P: pieces
// per row.  sx: the sum of those x values.
// ---------------------------------------------------------------------------

// Q8_0 (device layout qs[32] | d): y = f32(i8 q) * delta (src/gguf/dequant.rs:101-109).
struct PieceQ80 {
  static constexpr int kE = 16;
  uint4 q;
  uint32_t d;
  __device__ __forceinline__ void load(const uint8_t* body, const uint8_t* scal, uint32_t row, uint32_t P, uint32_t p) {
    const uint64_t i = (uint64_t)row * P + p;
    q = ldw(body + i * 16);
    d = ((const uint16_t*)scal)[i >> 1];
  }
  // q x = (u - 128) x with u = q ^ 0x80 unsigned: one convert per byte, the
  // -128 sum(x) term from sx
  __device__ __forceinline__ float dot(const float* x, float sx) const {
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const uint32_t u = opaque(qw[w] ^ 0x80808080u);
      s0 = fmaf(cvtb(u, 0), x[4 * w], s0);
      s1 = fmaf(cvtb(u, 1), x[4 * w + 1], s1);
      s0 = fmaf(cvtb(u, 2), x[4 * w + 2], s0);
      s1 = fmaf(cvtb(u, 3), x[4 * w + 3], s1);
    }
    return h2f(d) * fmaf(-128.f, sx, s0 + s1);
  }
};

// Q4_0 (device layout qs[16] | d): low nibble -> element j, high -> j+16, value q-8.
struct PieceQ40 {
  static constexpr int kE = 32;
  uint4 q;
  uint32_t d;
  __device__ __forceinline__ void load(const uint8_t* body, const uint8_t* scal, uint32_t row, uint32_t P, uint32_t p) {
    const uint64_t i = (uint64_t)row * P + p;
    q = ldw(body + i * 16);
    d = ((const uint16_t*)scal)[i];
  }
  __device__ __forceinline__ float dot(const float* x, float sx) const {
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      const uint32_t lo = opaque(qw[w] & 0x0F0F0F0Fu), hi = opaque(qw[w] & 0xF0F0F0F0u);  // hi: 16 q
#pragma unroll
      for (int b = 0; b < 4; b++) {
        s0 = fmaf(cvtb(lo, b), x[4 * w + b], s0);
        s1 = fmaf(cvtb(hi, b), x[16 + 4 * w + b], s1);
      }
    }
    return h2f(d) * fmaf(-8.f, sx, fmaf(s1, 0.0625f, s0));
  }
};

// Q8_K (device layout sc[32] | qs[256]; {d, dmin}): y = ((d*sc)*q) - dmin.
struct PieceQ8K {
  static constexpr int kE = 16;
  uint4 q;
  uint32_t sc, dd;
  __device__ __forceinline__ void load(const uint8_t* body, const uint8_t* scal, uint32_t row, uint32_t P, uint32_t p) {
    const uint64_t b = (uint64_t)row * (P >> 4) + (p >> 4);
    const uint8_t* blk = body + b * 288;
    q = ldw(blk + 32 + 16 * (p & 15));
    sc = *(const uint16_t*)(blk + 2 * (p & 15));
    dd = ((const uint32_t*)scal)[b];
  }
  __device__ __forceinline__ float dot(const float* x, float sx) const {
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    const float d = h2f(dd), dmin = h2f(dd >> 16);
    float tot = 0.f;
#pragma unroll
    for (int k = 0; k < 2; k++) {  // sub-blocks of 8 elements share one scale byte
      float a8 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e++) a8 = fmaf(sbyte((int)qw[2 * k + e / 4], e % 4), x[8 * k + e], a8);
      tot = fmaf(d * cvtb(sc, k), a8, tot);
    }
    return fmaf(-dmin, sx, tot);
  }
};

struct PieceF32 {
  static constexpr int kE = 4;
  uint4 q;
  __device__ __forceinline__ void load(const uint8_t* body, const uint8_t*, uint32_t row, uint32_t P, uint32_t p) {
    q = ldw(body + ((uint64_t)row * P + p) * 16);
  }
  __device__ __forceinline__ float dot(const float* x, float) const {
    float s = __uint_as_float(q.x) * x[0];
    s = fmaf(__uint_as_float(q.y), x[1], s);
    s = fmaf(__uint_as_float(q.z), x[2], s);
    return fmaf(__uint_as_float(q.w), x[3], s);
  }
};

struct PieceF16 {
  static constexpr int kE = 8;
  uint4 q;
  __device__ __forceinline__ void load(const uint8_t* body, const uint8_t*, uint32_t row, uint32_t P, uint32_t p) {
    q = ldw(body + ((uint64_t)row * P + p) * 16);
  }
  __device__ __forceinline__ float dot(const float* x, float) const {
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      s0 = fmaf(h2f(qw[w]), x[2 * w], s0);
      s1 = fmaf(h2f(qw[w] >> 16), x[2 * w + 1], s1);
    }
    return s0 + s1;
  }
};

// Where the rows of the logical segments lie.  Held in registers behind an
// asm barrier: a segment chosen per unit from the kernel's arguments would be
// indexed through scratch memory.
template <class Epi>
struct Segs {
  static constexpr int kN = Epi::kPaired ? 2 : Epi::kNeighbor ? 3 : 1;  // gate/up; q/k/v; one matrix
  const uint8_t* body[kN];
  const uint8_t* scal[kN];
  uint32_t rows[kN];
  __device__ __forceinline__ explicit Segs(const KArgs& a) {
#pragma unroll
    for (int i = 0; i < kN; i++) {
      body[i] = a.seg[i].body;
      scal[i] = a.seg[i].scal;
      rows[i] = a.seg[i].rows;
      asm("" : "+s"(body[i]), "+s"(scal[i]), "+s"(rows[i]));
    }
  }
};

// (by value: a conditional over the members selects an address to load from;
// eight steps of two 288-wide Q8_0 layers 445 -> 362 us, 4096-wide 1310 -> 1137)
template <class V>
__device__ __forceinline__ V pick(int s, V a, V b, V c) {
  return s == 2 ? c : s == 1 ? b : a;
}

// Unit u of the launch: the rows of its two sums.  Units past the end read
// unit 0 (in bounds, unused); the row past an odd segment's end reads the last.
struct Unit {
  int s;
  uint32_t r0, r1;
  bool ok1;
};
template <class Epi>
__device__ __forceinline__ Unit unit_of(const KArgs& a, const Segs<Epi>& g, uint32_t u) {
  Unit n;
  u = u < a.total ? u : 0u;
  n.s = 0;
  if constexpr (Epi::kPaired) {
    n.r0 = n.r1 = u;
    n.ok1 = true;
  } else {
    uint32_t rows = g.rows[0];
    if constexpr (Segs<Epi>::kN == 3) {
      const uint32_t n1 = a.nunits[0], n2 = n1 + a.nunits[1];
      n.s = u >= n2 ? 2 : u >= n1 ? 1 : 0;
      rows = pick(n.s, rows, g.rows[1], g.rows[2]);
      u -= n.s == 2 ? n2 : n.s == 1 ? n1 : 0u;
    }
    n.r0 = 2 * u;
    n.ok1 = n.r0 + 1 < rows;
    n.r1 = n.ok1 ? n.r0 + 1 : n.r0;
  }
  return n;
}

template <class Epi, class Q, int K>
struct Buf {
  Q q[2][K];
  // row t of unit u
  template <int t>
  __device__ __forceinline__ void load(const KArgs& a, const Segs<Epi>& g, uint32_t u, const uint32_t (&pc)[K]) {
    const Unit n = unit_of<Epi>(a, g, u);
    const uint8_t *b = g.body[0], *sc = g.scal[0];
    if constexpr (Epi::kPaired) {
      b = g.body[t];
      sc = g.scal[t];
    } else if constexpr (Segs<Epi>::kN == 3) {
      b = pick(n.s, b, g.body[1], g.body[2]);
      sc = pick(n.s, sc, g.scal[1], g.scal[2]);
    }
#pragma unroll
    for (int i = 0; i < K; i++) q[t][i].load(b, sc, t ? n.r1 : n.r0, a.pieces, pc[i]);
    __builtin_amdgcn_sched_barrier(0);  // rows in order: the loop's waits assume it
  }
  __device__ __forceinline__ float dot(int t, const float (&x)[K][Q::kE], const float (&sx)[K], const bool (&valid)[K]) const {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < K; i++) {
      const float p = q[t][i].dot(x[i], sx[i]);
      v += valid[i] ? p : 0.f;
    }
    return v;
  }
};

// the sum of v over the lanes that share a row, in each of them
template <int K>
__device__ __forceinline__ float lanes_sum(float v, uint32_t lg) {
  v = bfly<1, false>(v);
  v = bfly<2, false>(v);
  v = bfly<4, false>(v);
  v = bfly<8, false>(v);
  if (K > 1 || lg > 4) v = bfly<16, false>(v);
  if (K > 1 || lg > 5) v = bfly<32, false>(v);
  return v;
}

constexpr int kMinWaves = 2;  // per SIMD

// Q4_0, several pieces per lane: the 64 pieces of 32 x values that a wave's
// lanes take come from memory whole lines at a time, through the wave's own
// part of LDS (no barrier).  Read where they lie, a lane's values are 128 bytes
// from the next lane's and every load touches 64 cache lines: 4096 x 4096 7.63
// -> 5.89 us, 14336 x 4096 10.14 -> 8.26, 512 x 8192 8.01 -> 5.99.  The row
// stride of 36 floats spreads 16 lanes' reads over all banks.
constexpr int kStageRow = 36, kStageFloats = 64 * kStageRow;
// floats first .. first + 2047 of v (past `n`: its last four, unused)
__device__ __forceinline__ void stage_load(f4 (&g)[8], const float* v, uint32_t first, uint32_t n, int lane) {
#pragma unroll
  for (int r = 0; r < 8; r++) g[r] = *(const f4*)(v + min(first + 4u * (uint32_t)(lane + 64 * r), n - 4));
}
// orders this wave's LDS accesses, which run in the order they are issued
__device__ __forceinline__ void stage_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void stage_put(const f4 (&g)[8], float* lds, int lane) {
  stage_order();
#pragma unroll
  for (int r = 0; r < 8; r++) *(f4*)(lds + (lane / 8 + 8 * r) * kStageRow + 4 * (lane % 8)) = g[r];
  stage_order();
}

// K pieces of a row per lane; WIDE: a.split waves of the workgroup per row.
template <class Epi, class Q, int K, bool WIDE>
__global__ void __launch_bounds__(64 * (WIDE ? kWavesWide : kWavesNarrow), kMinWaves) k_gemv(KArgs a, Epi epi) {
  constexpr int kW = WIDE ? kWavesWide : kWavesNarrow, kE = Q::kE;
  constexpr bool P2 = Epi::kPaired;
  // units in flight; 0: a row's loads go out when its turn comes (F32: 64
  // registers a row; the other waves of the CU cover them)
  constexpr int kDepth = sizeof(Q) * K > 128 ? 0 : sizeof(Q) * K > 100 ? 1 : 2;
  constexpr int kSlots = kDepth ? kDepth : 1;
  constexpr bool kStaged = kE == 32 && (K > 1 || WIDE);  // x by way of LDS
  __shared__ float part[2][kW][2];
  __shared__ float red[kW];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t lg = K > 1 ? 6u : a.lg_lanes, ll = (uint32_t)lane & ((1u << lg) - 1u), G = 64u >> lg;
  const uint32_t S = WIDE ? a.split : 1u, j = WIDE ? (uint32_t)wave % S : 0u;
  // groups of G units: this wave takes g0, g0 + TW, ...; `iters` covers the
  // workgroup's first wave, which has the most
  const uint32_t NG = (a.total + G - 1) >> (6 - lg);
  const uint32_t GPB = kW / S, TW = gridDim.x * GPB, gb = blockIdx.x * GPB, g0 = gb + (uint32_t)wave / S;
  const uint32_t iters = gb < NG ? (NG - 1 - gb) / TW + 1 : 0u;
  const uint32_t u0 = (g0 << (6 - lg)) + (K > 1 ? 0u : (uint32_t)lane >> lg), ustep = TW << (6 - lg);

  const Segs<Epi> sg(a);
  typename Epi::Wave ws;
  epi.begin(ws);
  uint32_t pc[K];
  bool valid[K];
#pragma unroll
  for (int i = 0; i < K; i++) {
    const uint32_t p = K > 1 || WIDE ? (uint32_t)lane + 64u * (j + S * i) : ll;
    valid[i] = p < a.pieces;
    pc[i] = min(p, a.pieces - 1);
  }
  // x w (norm) of the lane's pieces, and its part of x . x; the first units'
  // rows are in flight meanwhile
  float x[K][kE], sx[K];
  float nscale = 1.f, ss = 0.f;
  Buf<Epi, Q, K> buf[kSlots];
  // x[i][e ..] = t * w, as ss gathers t * t
  auto normed = [&](int i, int e, float4 v) __attribute__((always_inline)) {
    const float w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const float t = x[i][e + c];
      ss = valid[i] ? fmaf(t, t, ss) : ss;
      x[i][e + c] = t * w[c];
    }
  };
  f4 gx[kStaged ? K : 1][8], gn[kStaged ? K : 1][8];
  if constexpr (kStaged) {
#pragma unroll
    for (int i = 0; i < K; i++) {
      const uint32_t first = kE * 64u * (j + S * i);
      stage_load(gx[i], a.x, first, a.cols, lane);
      if (a.norm_w) stage_load(gn[i], a.norm_w, first, a.cols, lane);
    }
  } else {
#pragma unroll
    for (int i = 0; i < K; i++)
#pragma unroll
      for (int e = 0; e < kE; e += 4) {
        const float4 v = *(const float4*)(a.x + (uint64_t)pc[i] * kE + e);
        x[i][e] = v.x; x[i][e + 1] = v.y; x[i][e + 2] = v.z; x[i][e + 3] = v.w;
      }
    if (a.norm_w) {
#pragma unroll
      for (int i = 0; i < K; i++)
#pragma unroll
        for (int e = 0; e < kE; e += 4) normed(i, e, *(const float4*)(a.norm_w + (uint64_t)pc[i] * kE + e));
    }
  }
#pragma unroll
  for (int d = 0; d < kDepth; d++) {
    buf[d].template load<0>(a, sg, u0 + d * ustep, pc);
    buf[d].template load<1>(a, sg, u0 + d * ustep, pc);
  }
  if constexpr (kStaged) {
    __shared__ __attribute__((aligned(16))) float stage[kW][kStageFloats];
    float* mine = stage[wave];
#pragma unroll
    for (int i = 0; i < K; i++) {
      stage_put(gx[i], mine, lane);
#pragma unroll
      for (int e = 0; e < kE; e += 4) {
        const float4 v = *(const float4*)(mine + lane * kStageRow + e);
        x[i][e] = v.x; x[i][e + 1] = v.y; x[i][e + 2] = v.z; x[i][e + 3] = v.w;
      }
      if (a.norm_w) {
        stage_put(gn[i], mine, lane);
#pragma unroll
        for (int e = 0; e < kE; e += 4) normed(i, e, *(const float4*)(mine + lane * kStageRow + e));
      }
    }
  }
  if (a.norm_w) {  // rms_norm (src/ops.rs:162-167): scale = 1/sqrt(mean(x^2) + eps)
    ss = lanes_sum<K>(ss, lg);
    if (WIDE) {
      if (lane == 0) red[wave] = ss;
      __syncthreads();
      ss = 0.f;
      for (uint32_t q = 0; q < S; q++) ss += red[(wave - j) + q];
    }
    nscale = 1.0f / sqrtf(ss / (float)a.cols + a.eps);
  }
#pragma unroll
  for (int i = 0; i < K; i++) {
    sx[i] = 0.f;
#pragma unroll
    for (int e = 0; e < kE; e += 4) sx[i] += (x[i][e] + x[i][e + 1]) + (x[i][e + 2] + x[i][e + 3]);
  }

  for (uint32_t it0 = 0; it0 < iters; it0 += kSlots) {
#pragma unroll
    for (int d = 0; d < kSlots; d++) {
      const uint32_t it = it0 + d, u = u0 + it * ustep;
      // lane ll < 2 (paired: 0) of the first wave emits row ll of its unit
      const bool live = it < iters && u < a.total && (!WIDE || j == 0) && ll < (P2 ? 1u : 2u);
      const Unit n = unit_of<Epi>(a, sg, u);
      const bool mine = live && (ll == 0 || n.ok1);
      const uint32_t r = ll == 0 ? n.r0 : n.r1;
      typename Epi::Pre pre{};
      if (mine) pre = epi.pre(ws, Segs<Epi>::kN == 3 ? n.s : 0, r);
      if constexpr (kDepth == 0) buf[d].template load<0>(a, sg, u, pc);
      float v0 = buf[d].dot(0, x, sx, valid);
      if constexpr (kDepth > 0) buf[d].template load<0>(a, sg, u + kDepth * ustep, pc);
      else buf[d].template load<1>(a, sg, u, pc);
      float v1 = buf[d].dot(1, x, sx, valid);
      if constexpr (kDepth > 0) buf[d].template load<1>(a, sg, u + kDepth * ustep, pc);
      v0 = lanes_sum<K>(v0, lg);
      v1 = lanes_sum<K>(v1, lg);
      if (WIDE) {
        if (lane == 0) {
          part[it & 1][wave][0] = v0;
          part[it & 1][wave][1] = v1;
        }
        __syncthreads();
        v0 = v1 = 0.f;
        for (uint32_t q = 0; q < S; q++) {
          v0 += part[it & 1][(wave - j) + q][0];
          v1 += part[it & 1][(wave - j) + q][1];
        }
      }
      v0 *= nscale;
      v1 *= nscale;
      if (mine) epi.row(ws, Segs<Epi>::kN == 3 ? n.s : 0, r, ll == 0 ? v0 : v1, ll == 0 ? v1 : v0, pre);
    }
  }
  epi.finish(ws, lane);
}

// ---------------------------------------------------------------------------
// F32 / F16 rows that are not whole 32-element groups: x in LDS (optionally
// RMS-normalised), lanes stride over the elements of each row, a wave per tile
// of kR rows.
// ---------------------------------------------------------------------------
constexpr int kGWaves = 8, kGThreads = kGWaves * 64, kR = 4;
constexpr int kGroupStride = 36;
__device__ __forceinline__ uint32_t xpad(uint32_t i) { return (i >> 5) * kGroupStride + (i & 31); }

struct GArgs {
  GemvSeg seg[3];
  uint32_t ntiles[3];
  uint32_t rot[3];  // first-wave rotation per segment (balances small segments)
  int nseg;
  uint32_t cols;
  const float* x;
  const float* norm_w;
  float eps;
};

// Row r of tile `tile` of logical segment s.  Paired launches (gate/up) put
// rows 2t, 2t + 1 of segment 0 in r = 0, 1 and those of segment 1 in r = 2, 3.
struct RowRef {
  const uint8_t* body;
  uint64_t row;
  bool ok, f32;
};
template <bool PAIRED>
__device__ __forceinline__ RowRef row_of(const GArgs& a, int s, uint32_t tile, int r) {
  const GemvSeg& sg = a.seg[PAIRED ? (r < kR / 2 ? 0 : 1) : s];
  const uint32_t row = PAIRED ? tile * (kR / 2) + (r % (kR / 2)) : tile * kR + r;
  return RowRef{sg.body, row < sg.rows ? row : sg.rows - 1, row < sg.rows, sg.type == T_F32};
}

template <class Epi>
__global__ void __launch_bounds__(kGThreads) k_gemv_generic(GArgs a, Epi epi) {
  constexpr bool P = Epi::kPaired;
  extern __shared__ float xl[];
  __shared__ float red[kGWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  float ss = 0.f;
  for (uint32_t i = tid; i < a.cols; i += kGThreads) {
    const float v = a.x[i];
    xl[xpad(i)] = v;
    ss = fmaf(v, v, ss);
  }
  if (a.norm_w) {
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float tot = 0.f;
    for (int w = 0; w < kGWaves; w++) tot += red[w];
    const float scale = 1.0f / sqrtf(tot / (float)a.cols + a.eps);
    for (uint32_t i = tid; i < a.cols; i += kGThreads) xl[xpad(i)] = (xl[xpad(i)] * scale) * a.norm_w[i];
  }
  __syncthreads();
  const uint32_t W = gridDim.x * kGWaves, wid = blockIdx.x * kGWaves + wave;
  typename Epi::Wave ws;
  epi.begin(ws);
  for (int s = 0; s < a.nseg; s++) {
    for (uint32_t t = (wid + W - a.rot[s]) % W; t < a.ntiles[s]; t += W) {
      float acc[kR] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < kR; r++) {
        const RowRef rr = row_of<P>(a, s, t, r);
        const uint64_t base = rr.row * a.cols;
        float v = 0.f;
        for (uint32_t l = lane; l < a.cols; l += 64) {
          const float w = rr.f32 ? ((const float*)rr.body)[base + l] : h2f(((const uint16_t*)rr.body)[base + l]);
          v = fmaf(w, xl[xpad(l)], v);
        }
        acc[r] = wave_sum(v);
      }
      // lane r < kR owns row r (paired: lanes 0, 1 the gate rows)
      if (lane < (P ? kR / 2 : kR)) {
        const RowRef rr = row_of<P>(a, s, t, lane);
        const int o = P ? lane + kR / 2 : lane ^ 1;
        const float v = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
        const float partner = o == 0 ? acc[0] : o == 1 ? acc[1] : o == 2 ? acc[2] : acc[3];
        const int es = P ? 0 : s;
        if (rr.ok) epi.row(ws, es, (uint32_t)rr.row, v, P || Epi::kNeighbor ? partner : 0.f,
                           epi.pre(ws, es, (uint32_t)rr.row));
      }
    }
  }
  epi.finish(ws, lane);
}

int device_cu_count() {
  // initialised once, thread-safe (sessions may run on several threads)
  static const int n = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
      return v;
    return 256;
  }();
  return n;
}

// Rows of >14K columns need more than 64 KiB of LDS in the generic kernel:
// each instance opts in once, through a block-scope static of a function
// instantiated per kernel (initialised the first time a launch gets there,
// once even when sessions run on several threads).
template <class K>
hipError_t allow_lds(K kernel) {
  return hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024);
}

template <class Epi>
hipError_t launch_generic(const GemvLaunch& L, const Epi& epi, size_t lds, hipStream_t st) {
  GArgs a{};
  a.cols = L.cols;
  a.x = L.x;
  a.norm_w = L.norm_w;
  a.eps = L.eps;
  a.nseg = Epi::kPaired ? 1 : L.nseg;
  for (int s = 0; s < L.nseg; s++) a.seg[s] = L.seg[s];
  uint32_t total = 0;
  for (int s = 0; s < a.nseg; s++) {
    const uint32_t per = Epi::kPaired ? kR / 2 : kR;
    a.ntiles[s] = (L.seg[s].rows + per - 1) / per;
    total += a.ntiles[s];
  }
  if (total == 0) return hipSuccess;
  const uint32_t per_cu = (uint32_t)std::max<size_t>(1, std::min<size_t>(2, (160 * 1024) / lds));
  const uint32_t blocks = std::min<uint32_t>((total + kGWaves - 1) / kGWaves, per_cu * device_cu_count());
  uint32_t acc = 0;
  for (int s = 0; s < a.nseg; s++) {
    a.rot[s] = acc % (blocks * kGWaves);
    acc += a.ntiles[s];
  }
  if (lds > 64 * 1024) {
    static const hipError_t opted = allow_lds(k_gemv_generic<Epi>);
    if (opted != hipSuccess) return opted;
  }
  hipLaunchKernelGGL(k_gemv_generic<Epi>, dim3(blocks), dim3(kGThreads), lds, st, a, epi);
  return hipGetLastError();
}

template <class Epi, class Q, int K, bool WIDE>
hipError_t go(const KArgs& a, const Epi& epi, hipStream_t st) {
  constexpr uint32_t kW = WIDE ? kWavesWide : kWavesNarrow;
  const uint32_t G = 64u >> a.lg_lanes, groups = (a.total + G - 1) / G, per = kW / a.split;
  // persistent: as many workgroups as run at once (kMinWaves waves per SIMD)
  const uint32_t most = (uint32_t)device_cu_count() * (4 * kMinWaves / kW);
  const uint32_t blocks = std::min((groups + per - 1) / per, most);
  hipLaunchKernelGGL((k_gemv<Epi, Q, K, WIDE>), dim3(blocks), dim3(64 * kW), 0, st, a, epi);
  return hipGetLastError();
}

// K: the smallest of the type's piece counts that covers a row with one wave
// (x then takes at most 64 registers); longer rows: KM pieces and S waves.
template <class Epi, class Q, int K2, int K4, int KM>
hipError_t dispatch(KArgs a, const Epi& epi, hipStream_t st) {
  a.pieces = a.cols / Q::kE;
  a.lg_lanes = 6;
  a.split = 1;
  if (a.pieces <= 64) {
    a.lg_lanes = a.pieces <= 16 ? 4 : a.pieces <= 32 ? 5 : 6;
    return go<Epi, Q, 1, false>(a, epi, st);
  }
  if (K2 < K4 && a.pieces <= 64 * K2) return go<Epi, Q, K2, false>(a, epi, st);
  if (K4 < KM && a.pieces <= 64 * K4) return go<Epi, Q, K4, false>(a, epi, st);
  if (a.pieces <= 64 * KM) return go<Epi, Q, KM, false>(a, epi, st);
  a.split = a.pieces <= 128 * KM ? 2 : a.pieces <= 256 * KM ? 4 : 8;
  if (a.pieces > 64 * KM * a.split) return hipErrorInvalidValue;
  return go<Epi, Q, KM, true>(a, epi, st);
}

template <class Epi>
hipError_t launch(const GemvLaunch& L, const Epi& epi, hipStream_t st) {
  if (L.nseg < 1 || L.nseg > 3 || L.cols == 0) return hipErrorInvalidValue;
  // Q4_K / Q6_K (tiled layout): the int8-MFMA kernel; a launch does not mix the two families
  int n_mfma = 0;
  for (int s = 0; s < L.nseg; s++) n_mfma += mfma_type(L.seg[s].type) ? 1 : 0;
  if (n_mfma == L.nseg) return launch_mfma(L, epi, st);
  if (n_mfma != 0) return hipErrorInvalidValue;
  const bool generic = L.cols % 32 != 0;
  for (int s = 0; s < L.nseg; s++) {
    const uint32_t t = L.seg[s].type;
    if (t == T_Q8K && L.cols % 256) return hipErrorInvalidValue;
    if (generic && t != T_F32 && t != T_F16) return hipErrorInvalidValue;
  }
  if (Epi::kPaired &&
      (L.nseg != 2 || L.seg[0].rows != L.seg[1].rows || L.seg[0].type != L.seg[1].type))
    return hipErrorInvalidValue;
  // The longest rows taken: 32336 columns, 17552 of whole 32-groups with a norm
  // (what 150 KiB hold of x, its 16-element sums and the norm weights, as both
  // kernels once staged them; the generic one's LDS is less).
  const size_t lds = (size_t)((L.cols + 31) / 32) * kGroupStride * 4 + (size_t)((L.cols / 16 + 3) & ~3u) * 4 +
                     (L.norm_w && !generic ? (size_t)L.cols * 4 : 0);
  if (lds > 150 * 1024) return hipErrorInvalidValue;
  if (generic) return launch_generic(L, epi, lds, st);
  if (!Epi::kPaired && L.nseg > Segs<Epi>::kN) return hipErrorInvalidValue;
  KArgs a{};
  a.cols = L.cols;
  a.x = L.x;
  a.norm_w = L.norm_w;
  a.eps = L.eps;
  const int nseg = Epi::kPaired ? 1 : L.nseg;
  for (int s = 0; s < L.nseg; s++) a.seg[s] = L.seg[s];
  for (int s = 0; s < nseg; s++) {
    a.nunits[s] = Epi::kPaired ? L.seg[s].rows : (L.seg[s].rows + 1) / 2;
    a.total += a.nunits[s];
  }
  if (a.total == 0) return hipSuccess;
  // one type per launch on this path (the mixed Q4_K / Q6_K layers take the MFMA kernel)
  const uint32_t ta = L.seg[0].type;
  for (int s = 1; s < nseg; s++)
    if (L.seg[s].type != ta) return hipErrorInvalidValue;
  switch (ta) {
    case T_Q8_0: return dispatch<Epi, PieceQ80, 2, 4, 4>(a, epi, st);
    case T_Q4_0: return dispatch<Epi, PieceQ40, 2, 2, 2>(a, epi, st);
    case T_Q8K: return dispatch<Epi, PieceQ8K, 4, 4, 4>(a, epi, st);
    case T_F32: return dispatch<Epi, PieceF32, 4, 16, 16>(a, epi, st);
    case T_F16: return dispatch<Epi, PieceF16, 2, 4, 8>(a, epi, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int gemv_supported(uint32_t t) {
  return t == T_F32 || t == T_F16 || t == T_Q4_0 || t == T_Q8_0 || t == T_Q4K || t == T_Q6K ||
         t == T_Q8K;
}

hipError_t gemv_store(const GemvLaunch& L, float* y, hipStream_t st) {
  EpiStore e{};
  e.y = y;
  uint32_t off = 0;
  for (int s = 0; s < L.nseg; s++) { e.seg_out[s] = off; off += L.seg[s].rows; }
  return launch(L, e, st);
}

hipError_t gemv_residual(const GemvLaunch& L, float* hidden, hipStream_t st) {
  if (L.nseg != 1) return hipErrorInvalidValue;
  const hipError_t e = launch_mfma_residual_ks(L, hidden, st);
  if (e != hipErrorNotSupported) return e;
  return launch(L, EpiResidual{hidden}, st);
}

hipError_t gemv_residual_fixed(const GemvLaunch& L, float* hidden, hipStream_t st) {
  if (L.nseg != 1) return hipErrorInvalidValue;
  return launch(L, EpiResidual{hidden}, st);
}

hipError_t gemv_qkv(const GemvLaunch& L, const QkvEpi& e, hipStream_t st) {
  if (L.nseg != 3 || (e.head_dim & 1) || (e.rope_dim & 1)) return hipErrorInvalidValue;
  return launch(L, EpiQkv{e}, st);
}

hipError_t gemv_swiglu(const GemvLaunch& L, float* mid, hipStream_t st) {
  if (!L.paired) return hipErrorInvalidValue;
  return launch(L, EpiSwiglu{mid}, st);
}

hipError_t gemv_logits(const GemvLaunch& L, float* logits, DevState* state, hipStream_t st) {
  if (L.nseg != 1) return hipErrorInvalidValue;
  return launch(L, EpiLogits{logits, state}, st);
}

}  // namespace ifx
