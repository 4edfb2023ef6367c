// Whole steps of the operation in one kernel for small bf16 heads (feature sizes up to 128), whose products are so short that
// the separate kernels spend their time on the [tokens, hidden] arrays they hand to each other.
#pragma once
#include <type_traits>

#include "window_attention.h"
#include "gemm_dma_kernels.h"

namespace lact {

// ---- apply: out = (silu(q W0^T) * (q W2^T)) W1^T ----------------------------------------------------------------------------
// A wave owns 32 tokens as matrix columns, their query rows in registers, and walks the hidden units in stages of 64 whose weight
// rows (W0, W2: [64][d]; W1: [d][64]) travel through a ring of asynchronous copies shared by the block.  The gated hidden values
// feed the second product as they lie: slots 0..3 / 4..7 of lane half h stand for hidden units 4h + i / 8 + 4h + i of 16, on both
// operands (as in window_attention.h).  Nothing but q is read and nothing but out is written.
//
// SPLIT: two waves share 32 tokens and take a half of every stage each, their sums meet in LDS at the end: four groups of
// tokens a block instead of eight, as long as these blocks are all resident at once (256 of them).
// What bounds it: 8 us of start, first copies and stores around a serial chain of matrix instructions, roundings and two
// transcendental functions per hidden value on two waves a SIMD (1.6 us per 32 hidden units).  us, whole / SPLIT / the hidden stage
// and output product as kernels of their own: 12 x 4680 tokens, d = 128, dh = 256 23.4 / 30.2 / 35.4; 6 x 1024 tokens 18.1 / 14.3 / 10.7
// and a launch; 24 x 2500 tokens, d = dh = 96 12.1 / 16.6 / 23.0.
struct ApplyFusedParams {
  int T, dh;
  const uint16_t* X; int ldx; long long bsx;               // [T, d] queries
  const uint16_t* W0; const uint16_t* W1; const uint16_t* W2; long long bsw;
  uint16_t* out; int ldo; long long bso;
  StepBatch steps; long long gsx, gsw, gso;                // several steps of the program in one launch
  TileMap map;                                             // token blocks, 1, batch
};

// One stage in LDS: KC tiles [64 hidden][64 k] each of W0 and W2, one tile [d][64 hidden] of W1, rows of 128 bytes with the
// granules where gemm_dma.h puts them.
template <int D>
struct ApplyStage {
  static constexpr int KC = (D + 63) / 64;
  static constexpr int W2 = KC * 64 * 128, W1 = 2 * KC * 64 * 128, BYTES = W1 + D * 128;
  static constexpr int COPIES = BYTES / 1024, PER_WAVE = (COPIES + 7) / 8;
  static constexpr int STAGES = 3;
  static_assert(STAGES * BYTES <= 160 * 1024, "the ring does not fit the LDS");
};

// The copies of a wave: PER_WAVE of the stage's COPIES KiB (the last ones repeat the last copy, with the same bytes).
template <int D>
struct ApplyCopies {
  using ST = ApplyStage<D>;
  uint32_t voff[ST::PER_WAVE];      // within the operand's hidden units [0, 64)
  // hid: hidden units left from the stage's first on (rows and columns past them repeat the last ones)
  __device__ __forceinline__ uint32_t offset(int n, int dh, int hid) const {
    const int lane = threadIdx.x & 63;
    int row, kv = (lane & 7) ^ (((n * 8 + (lane >> 3)) >> 1) & 7);      // the key's row: tiles start at multiples of 16 rows
    if (n < 2 * ST::KC * 8) {
      const int t = n / 8 % ST::KC;                                     // W0 or W2: 64 k from 64 t
      row = min((n % 8) * 8 + (lane >> 3), hid - 1);
      kv = min(t * 8 + kv, D / 8 - 1);
      return (uint32_t)(row * D + kv * 8) * 2;
    }
    row = (n - 2 * ST::KC * 8) * 8 + (lane >> 3);
    return (uint32_t)(row * dh + min(kv, hid / 8 - 1) * 8) * 2;
  }
  __device__ __forceinline__ int number(int i, int wave) const { return min(wave + 8 * i, ST::COPIES - 1); }
  __device__ __forceinline__ void init(int wave, int dh) {
#pragma unroll
    for (int i = 0; i < ST::PER_WAVE; ++i) voff[i] = offset(number(i, wave), dh, 64);
  }
  __device__ __forceinline__ void issue(const uint16_t* w0, const uint16_t* w2, const uint16_t* w1, int j0, int dh, uint32_t lds, int wave) const {
    const bool whole = j0 + 64 <= dh;
#pragma unroll
    for (int i = 0; i < ST::PER_WAVE; ++i) {
      const int n = number(i, wave);
      const uint16_t* base = n < ST::KC * 8 ? w0 + (size_t)j0 * D : n < 2 * ST::KC * 8 ? w2 + (size_t)j0 * D : w1 + j0;
      uint32_t off = voff[i];
      if (!whole) off = offset(n, dh, dh - j0);
      dma16<false>(base, off, lds + n * 1024);
    }
  }
};

template <int D, bool SPLIT>
__global__ __launch_bounds__(512, 2) void k_apply_fused(const ApplyFusedParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using ST = ApplyStage<D>;
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, h = lane >> 5;
  constexpr int GROUPS = SPLIT ? 4 : 8;
  const int tg = wave % GROUPS, half = wave / GROUPS, row0 = (bx * GROUPS + tg) * 32;
  const uint16_t* X = p.X + p.steps.at(z, p.bsx, p.gsx);
  const long long w = p.steps.at(z, p.bsw, p.gsw);
  const uint16_t *W0 = p.W0 + w, *W1 = p.W1 + w, *W2 = p.W2 + w;
  const uint32_t lds0 = lds_addr(smem);
  ApplyCopies<D> cp;
  cp.init(wave, p.dh);
  const int n = (p.dh + 63) / 64;
  auto issue = [&](int t) { cp.issue(W0, W2, W1, t * 64, p.dh, lds0 + (t % 3) * ST::BYTES, wave); };
  bf16x8 qf[D / 16];
  attn_own_rows<D>(qf, X, p.ldx, row0 + (lane & 31), p.T);
  issue(0);
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  const uint32_t roff = (lane & 31) * 128, rkey = (uint32_t)((lane >> 1) & 7) << 4;   // (rows 32 apart have the same key)
  // One stage ahead: a block's copies take less time than its products, but issued at once they keep the waves from starting.  Three
  // slots because a half's gated values enter the second product behind the first products of the half after it, which may lie in
  // the next stage.
  auto open = [&](int t) {
    wait_vmcnt<0>();
    __syncthreads();
    if (t + 1 < n) issue(t + 1);
  };
  constexpr int KS = D / 16;
  auto rows = [&](const char* half_, int ks, bf16x8 (&f)[2]) {     // W0 and W2: the half's 32 hidden units over 16 of the d
    const char* row = half_ + (ks / 4) * 64 * 128 + roff + ((uint32_t)((ks % 4) * 32 + h * 16) ^ rkey);
    f[0] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(row));
    f[1] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(row + ST::W2));
  };
  auto cols = [&](const char* stage, int hf, int s, bf16x8 (&f)[D / 32]) {     // W1: all d over 16 of the half's hidden units
    const char* w1 = stage + ST::W1 + roff + h * 8;
    const uint32_t g0 = (uint32_t)(hf * 64 + s * 32);
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) {
      const uint2 a = *reinterpret_cast<const uint2*>(w1 + dt * 32 * 128 + (g0 ^ rkey)), b = *reinterpret_cast<const uint2*>(w1 + dt * 32 * 128 + ((g0 + 16) ^ rkey));
      f[dt] = __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
    }
  };
  // The first products of the half at `next` (FIRST), the gating of the half in g, u between their matrix instructions, and its second
  // product (GATE).  Left to itself the compiler lines everything up: reads, products and gating one after the other.
  auto step = [&](auto first, auto gate, const char* next, f32x16& gn, f32x16& un, const char* stage, int hf, const f32x16& g, const f32x16& u) {
    constexpr bool FIRST = decltype(first)::value, GATE = decltype(gate)::value;
    uint32_t hv[8];
    bf16x8 f[2][2], w[2][D / 32];
    if (FIRST) {
      rows(next, 0, f[0]);
#pragma unroll
      for (int j = 0; j < 16; ++j) gn[j] = un[j] = 0.f;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (FIRST && ks + 1 < KS) rows(next, ks + 1, f[(ks + 1) & 1]);
      if (GATE && ks + 1 == KS) cols(stage, hf, 0, w[0]);
      if (FIRST) {
        gn = mma32(f[ks & 1][0], qf[ks], gn);
        un = mma32(f[ks & 1][1], qf[ks], un);
      }
      if (GATE)
#pragma unroll
        for (int i = ks * 8 / KS; i < (ks + 1) * 8 / KS; ++i) {
          float va, vb;
          apply_pointwise2(g[2 * i], g[2 * i + 1], u[2 * i], u[2 * i + 1], va, vb);
          hv[i] = pack_bf16(va, vb);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (GATE)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if (s == 0) cols(stage, hf, 1, w[1]);
        const bf16x8 hid = __builtin_bit_cast(bf16x8, make_uint4(hv[4 * s], hv[4 * s + 1], hv[4 * s + 2], hv[4 * s + 3]));
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) o[dt] = mma32(w[s][dt], hid, o[dt]);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  auto at = [&](int t) { return smem + (t % 3) * ST::BYTES; };
  f32x16 ga, ua, gb, ub;
  open(0);
  if (!SPLIT) {
    step(yes, no, at(0), ga, ua, at(0), 0, gb, ub);
    for (int t = 0; t + 1 < n; ++t) {
      step(yes, yes, at(t) + 32 * 128, gb, ub, at(t), 0, ga, ua);
      open(t + 1);
      step(yes, yes, at(t + 1), ga, ua, at(t), 1, gb, ub);
    }
    const char* st = at(n - 1);
    if (p.dh % 64 == 0) {
      step(yes, yes, st + 32 * 128, gb, ub, st, 0, ga, ua);
      step(no, yes, st, ga, ua, st, 1, gb, ub);
    } else {
      step(no, yes, st, gb, ub, st, 0, ga, ua);
    }
  } else {
    const int mine = half && p.dh % 64 ? n - 1 : n;       // stages whose half exists
    const int ho = half * 32 * 128;
    if (mine > 0) step(yes, no, at(0) + ho, ga, ua, at(0), 0, gb, ub);
    for (int t = 1; t < n; ++t) {
      open(t);
      if (t < mine) {
        step(yes, yes, at(t) + ho, gb, ub, at(t - 1), half, ga, ua);
        ga = gb; ua = ub;
      }
    }
    if (mine > 0) step(no, yes, smem, gb, ub, at(mine - 1), half, ga, ua);
  }
  __syncthreads();
  if (SPLIT) {
    float* part = reinterpret_cast<float*>(smem) + (tg * 64 + lane) * 4;
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (half) *reinterpret_cast<float4*>(part + (i * 4 + q) * GROUPS * 64 * 4) = make_float4(o[i][4 * q], o[i][4 * q + 1], o[i][4 * q + 2], o[i][4 * q + 3]);
    __syncthreads();
    if (!half)
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4 a = *reinterpret_cast<const float4*>(part + (i * 4 + q) * GROUPS * 64 * 4);
          o[i][4 * q] += a.x; o[i][4 * q + 1] += a.y; o[i][4 * q + 2] += a.z; o[i][4 * q + 3] += a.w;
        }
    __syncthreads();
    if (half) return;
  }
  attn_store_rows<D>(smem + tg * 32 * (D + 8) * 2, o, 1.f, p.out + p.steps.at(z, p.bso, p.gso), (size_t)p.ldo, row0, p.T);
}
template <int D, bool SPLIT>
constexpr int apply_fused_lds() {
  using ST = ApplyStage<D>;
  return cmax(ST::STAGES * ST::BYTES, cmax(SPLIT ? 4 * 32 * D * 4 : 0, 8 * 32 * (D + 8) * 2));
}

}  // namespace lact
