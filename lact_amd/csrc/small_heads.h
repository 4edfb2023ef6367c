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
  prefetch_args<sizeof(p)>();
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
  attn_arrived(qf);
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

// ---- update: the three weight gradients of a step -----------------------------------------------------------------------------
//   g, u, e = k W0^T, k W2^T, v W1  ->  dW0 = dgate^T (k lr0), dW1 = v^T (hidden lr1), dW2 = dhidden^T (k lr2)
// A wave keeps 32 hidden units: their rows of W0, W2 and W1^T as fragments and their rows (columns for dW1) of the three gradients as
// accumulators, all in registers, and walks every fourth patch of 32 tokens of its block's split.  The products come out with a
// token per register and a hidden unit per lane, which is how the gradients' products read them: nothing is exchanged.  A wave's
// tokens travel through a ring of its own, five half patches (k and v of two patches and one under way), so that the waves of a block
// meet only at the end, where the sums of the four are added in LDS.
//
// What bounds it: issue of vector operations by the one wave on a SIMD -- 730 for a patch of d = 128, of which 30 % scale k and a third of
// the rest rounds, in 5300 clocks (the 48 matrix instructions take 1540 of them and hide behind the others; the copies always arrive
// in time) -- and 8 us a block to start, finish its last patch and add the sums.  us, this kernel against the hidden stage and the
// token reduction as kernels of their own (and a pass that scales k): 6 x 8192 tokens, d = 128, dh = 256 43 / 36 + 21 (+ 8); 12 x 4680
// tokens 55 / 65 + 27 (+ 10); 24 x 2500 tokens, d = dh = 96 23 / 28 + 14 (+ 7).  One matrix instruction after each pair of tokens'
// pointwise part: 52 (the pair's operations wait for each other); the rates by ds_bpermute, 48 a patch: 49.
struct UpdateFusedParams {
  int T, dh, split_len;
  const uint16_t* K; int ldk; long long bsk;               // [T, d]
  const uint16_t* V; int ldv; long long bsv;
  const uint16_t* W0; const uint16_t* W1; const uint16_t* W2; long long bsw;
  const float* lr0; const float* lr1; const float* lr2; long long bslr;
  float* partial; long long split_stride, mat_stride;      // sums of split s, matrix j, batch entry z: partial + s, j * strides + z * d * dh
  TileMap map;                                             // splits, 32 hidden units, batch
};

template <int D>
struct UpdatePatch {
  static constexpr int P = D == 64 ? 64 : 128;             // columns of a row in LDS (those past D repeat its last granule)
  using T = AttnTile<P>;
  static constexpr int THREADS = 256, BYTES = 32 * T::ROWB, COPIES = BYTES / 1024, UNITS = 5;
  static constexpr int RING = 4 * UNITS * BYTES, SUMS = 4 * D * 128;
  static constexpr int LDS = cmax(RING, 2 * SUMS);
  static_assert(LDS <= 160 * 1024, "the rings do not fit the LDS");
};
// Copies of one operand's patch: four offsets a lane, the fifth to eighth copy 16 rows further down.
template <int D>
struct UpdateCopies {
  using U = UpdatePatch<D>;
  uint32_t voff[4];
  __device__ __forceinline__ void init(int ld) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = i * 64 + (threadIdx.x & 63), row = n / U::T::G, slot = n % U::T::G;
      voff[i] = (uint32_t)(row * ld + min(slot ^ U::T::key(row), D / 8 - 1) * 8) * 2;
    }
  }
  __device__ __forceinline__ void issue_one(const uint16_t* base, int ld, uint32_t lds, int i) const {
    dma16<false>(base + (size_t)(i / 4) * 16 * ld, voff[i % 4], lds + i * 1024);
  }
  __device__ __forceinline__ void issue(const uint16_t* base, int ld, uint32_t lds) const {
#pragma unroll
    for (int i = 0; i < U::COPIES; ++i) issue_one(base, ld, lds, i);
  }
};

// The rate of the token in register I of an accumulator: lane i of every 16 holds that of the lane half's i-th token, and the
// multiplication that takes it reads it from there.
__device__ __forceinline__ int slot_token(int lane) { return 8 * ((lane & 15) / 4) + 4 * (lane >> 5) + lane % 4; }
template <int I>
__device__ __forceinline__ float of_slot(float v) {
  constexpr int ROW_NEWBCAST = 0x150;
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ROW_NEWBCAST + I, 0xf, 0xf, true));
}

// Eight tokens of k from slot I on, times their rates, as the reference rounds the product.
template <int I>
__device__ __forceinline__ bf16x8 scaled(const float (&k)[8], float r) {
  return __builtin_bit_cast(bf16x8, make_uint4(pack_bf16(k[0] * of_slot<I>(r), k[1] * of_slot<I + 1>(r)), pack_bf16(k[2] * of_slot<I + 2>(r), k[3] * of_slot<I + 3>(r)),
                                               pack_bf16(k[4] * of_slot<I + 4>(r), k[5] * of_slot<I + 5>(r)), pack_bf16(k[6] * of_slot<I + 6>(r), k[7] * of_slot<I + 7>(r))));
}

// update_pointwise2 on two pairs of tokens, and hidden * lr1, in six steps of some twenty operations each: a matrix instruction is
// issued after every step, and a wave that is alone on its SIMD needs independent operations to issue one every 4 clocks (one that
// waits for the last takes 8).
struct UpdateSteps {
  float g[4], h2[4], dh[4], sg[4], sb[4], t[4], hid[4];
  uint32_t z0[2], z1[2], z2[2];
  __device__ __forceinline__ void round4(float (&x)[4]) const {
    round_both(x[0], x[1]);
    round_both(x[2], x[3]);
  }
  template <int STEP, int I>
  __device__ __forceinline__ void step(const f32x16& ag, const f32x16& ah, const f32x16& ad, float lr1) {
    auto each = [](auto f) {
#pragma unroll
      for (int j = 0; j < 4; ++j) f(j);
    };
    if (STEP == 0) {
      each([&](int j) { g[j] = ag[4 * I + j]; h2[j] = ah[4 * I + j]; dh[j] = ad[4 * I + j]; });
      round4(g);
      round4(h2);
      round4(dh);
    } else if (STEP == 1) {
      each([&](int j) { const SiluParts s = silu_parts(g[j]); sg[j] = s.silu; sb[j] = s.sig; });
    } else if (STEP == 2) {
      round4(sg);
      round4(sb);
      each([&](int j) { hid[j] = sg[j] * h2[j]; });
    } else if (STEP == 3) {
      round4(hid);
      float x[4];
      each([&](int j) { x[j] = dh[j] * sg[j]; t[j] = dh[j] * h2[j]; });
      z2[0] = pack_bf16(x[0], x[1]); z2[1] = pack_bf16(x[2], x[3]);
      x[0] = hid[0] * of_slot<4 * I>(lr1); x[1] = hid[1] * of_slot<4 * I + 1>(lr1);
      x[2] = hid[2] * of_slot<4 * I + 2>(lr1); x[3] = hid[3] * of_slot<4 * I + 3>(lr1);
      z1[0] = pack_bf16(x[0], x[1]); z1[1] = pack_bf16(x[2], x[3]);
    } else if (STEP == 4) {
      round4(t);
      each([&](int j) { t[j] *= sb[j]; sb[j] = 1.f - sb[j]; });
      round4(t);
      round4(sb);
    } else {
      each([&](int j) { sb[j] *= g[j]; });
      round4(sb);
      each([&](int j) { sb[j] += 1.f; });
      round4(sb);
      each([&](int j) { t[j] *= sb[j]; });
      z0[0] = pack_bf16(t[0], t[1]); z0[1] = pack_bf16(t[2], t[3]);
    }
  }
};

template <int D>
__global__ __launch_bounds__(256, 1) void k_update_fused(const UpdateFusedParams p) {
  prefetch_args<sizeof(p)>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using U = UpdatePatch<D>;
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, h = lane >> 5;
  const int hid0 = by * 32, tok0 = bx * p.split_len, len = min(p.split_len, p.T - tok0);
  const uint16_t* K = p.K + z * p.bsk;
  const uint16_t* V = p.V + z * p.bsv;
  const float *lr0 = p.lr0 + z * p.bslr, *lr1 = p.lr1 + z * p.bslr, *lr2 = p.lr2 + z * p.bslr;
  // Patches of this wave; one that would run past the last token starts earlier, its `over` first rows are cleared after the copy.
  const int patches = (len + 31) / 32, mine = patches > wave ? (patches - wave + 3) / 4 : 0;
  auto token = [&](int i) { return min(tok0 + (wave + 4 * min(i, mine - 1)) * 32, p.T - 32); };
  const int over = mine > 0 ? tok0 + (wave + 4 * (mine - 1)) * 32 - token(mine - 1) : 0;

  // The weights' slices come once for the block, into units of the first wave's ring that its tokens need later: rows of W0 and W2 like
  // a patch of tokens, [d][32 hidden] of W1 in rows of 64 bytes, to be read transposed.  (Each wave's fragments straight from memory
  // are 96 KiB a block instead of 24, at 40 to 70 GB/s that reach a compute unit: 1.5 us.)
  constexpr int KS = D / 16;
  bf16x8 w0[KS], w1[KS], w2[KS];
  AttnFrag<U::P> frag;
  frag.init();
  char* const weights = smem + 2 * U::BYTES;
  {
    const uint32_t to = lds_addr(weights);
    const long long w = z * p.bsw;
    UpdateCopies<D> cw;
    cw.init(D);
#pragma unroll
    for (int i = 0; i < U::COPIES; ++i)
      if (i % 4 == wave) {
        cw.issue_one(p.W0 + w + (size_t)hid0 * D, D, to, i);
        cw.issue_one(p.W2 + w + (size_t)hid0 * D, D, to + U::BYTES, i);
      }
    for (int i = wave; i < D / 16; i += 4) {
      const int n = i * 64 + lane;
      dma16<false>(p.W1 + w + hid0, (uint32_t)((n >> 2) * p.dh + (n & 3) * 8) * 2, to + 2 * U::BYTES + i * 1024);
    }
  }
  char* ring = smem + wave * U::UNITS * U::BYTES;
  const uint32_t lds0 = lds_addr(ring);
  UpdateCopies<D> ck, cv;
  ck.init(p.ldk);
  cv.init(p.ldv);
  auto unit = [&](int n) { return ring + n * U::BYTES; };
  auto issue_k = [&](int i, int n) { ck.issue(K + (size_t)token(i) * p.ldk, p.ldk, lds0 + n * U::BYTES); };
  auto issue_v = [&](int i, int n) { cv.issue(V + (size_t)token(i) * p.ldv, p.ldv, lds0 + n * U::BYTES); };
  struct Rates { float r[3]; };
  auto rates = [&](int i) {
    const int t = token(i) + slot_token(lane);
    return Rates{{lr0[t], lr1[t], lr2[t]}};
  };
  Rates rc{};
  if (mine > 0) {
    rc = rates(0);
    issue_k(0, 0);
    issue_v(0, 1);
  }
  wait_vmcnt<0>();
  __syncthreads();
  {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const char* t = weights + 2 * U::BYTES + (8 * h + ((lane & 15) >> 2)) * 64 + ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      w0[s] = frag.rows(weights, 0, s);
      w2[s] = frag.rows(weights + U::BYTES, 0, s);
      const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + s * 1024)), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + s * 1024 + 256));
      const s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      w1[s] = __builtin_bit_cast(bf16x8, v);
    }
  }
  f32x16 d0[D / 32], d1[D / 32], d2[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) d0[i][j] = d1[i][j] = d2[i][j] = 0.f;
  __syncthreads();       // the first wave's units are its own again
  if (mine > 0) {
    auto settle = [&](Rates& r, int i) {
      const int cut = i == mine - 1 ? over : 0;
#pragma unroll
      for (int j = 0; j < 3; ++j) r.r[j] = slot_token(lane) < cut ? 0.f : r.r[j];
    };
    settle(rc, 0);
    issue_k(1, 2);
    issue_v(1, 3);
    Rates rn = rates(1);
    auto clear = [&](int i, int nk, int nv) {
      if (i != mine - 1 || over == 0) return;
      wait_vmcnt<0>();
      for (int e = lane; e < over * U::T::G; e += 64) {
        *reinterpret_cast<uint4*>(unit(nk) + e * 16) = make_uint4(0, 0, 0, 0);
        *reinterpret_cast<uint4*>(unit(nv) + e * 16) = make_uint4(0, 0, 0, 0);
      }
      wave_lds_fence();
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    uint32_t q0[8], q1[8], q2[8];      // dgate, hidden * lr1, dhidden of the patch in hand, two tokens a word
    // The products of the next patch (FIRST), between them the pointwise part of the patch in g, u, e (GATE).
    auto products = [&](auto first, auto gate, const char* kt, const char* vt, f32x16& gn, f32x16& un, f32x16& en, const f32x16& g, const f32x16& u,
                        const f32x16& e, float lr, auto between) {
      constexpr bool FIRST = decltype(first)::value, GATE = decltype(gate)::value;
      // fragments two ahead; the steps of the pointwise part spread over the matrix instructions
      constexpr int N = 2 * KS, STEPS = 24;
      bf16x8 f[3];
      auto read = [&](int ks) {
        if (ks == KS) between();
        if (ks < N) f[ks % 3] = ks < KS ? frag.rows(kt, 0, ks) : frag.rows(vt, 0, ks - KS);
      };
      if (FIRST) {
        read(0);
        read(1);
#pragma unroll
        for (int j = 0; j < 16; ++j) gn[j] = un[j] = en[j] = 0.f;
      }
      UpdateSteps st;
      int done = 0;
      auto round = [&](auto at, int n) {
        constexpr int I = decltype(at)::value;
        switch (n) {
          case 0: st.template step<0, I>(g, u, e, lr); break;
          case 1: st.template step<1, I>(g, u, e, lr); break;
          case 2: st.template step<2, I>(g, u, e, lr); break;
          case 3: st.template step<3, I>(g, u, e, lr); break;
          case 4: st.template step<4, I>(g, u, e, lr); break;
          default:
            st.template step<5, I>(g, u, e, lr);
#pragma unroll
            for (int w = 0; w < 2; ++w) { q0[2 * I + w] = st.z0[w]; q1[2 * I + w] = st.z1[w]; q2[2 * I + w] = st.z2[w]; }
        }
      };
      auto steps = [&](int upto) {
        if (!GATE) return;
#pragma unroll
        for (int n = 0; n < STEPS; ++n) {
          if (n < done || n >= upto) continue;
          switch (n / 6) {
            case 0: round(std::integral_constant<int, 0>{}, n % 6); break;
            case 1: round(std::integral_constant<int, 1>{}, n % 6); break;
            case 2: round(std::integral_constant<int, 2>{}, n % 6); break;
            default: round(std::integral_constant<int, 3>{}, n % 6);
          }
        }
        done = upto;
      };
#pragma unroll
      for (int ks = 0; ks < N; ++ks) {
        const int before = ks < KS ? 2 * ks : KS + ks;        // matrix instructions issued before this fragment's
        if (FIRST) {
          read(ks + 2);
          if (ks < KS) gn = mma32(f[ks % 3], w0[ks % KS], gn);
          else en = mma32(f[ks % 3], w1[ks % KS], en);
        }
        steps((before + 1) * STEPS / (3 * KS));
        __builtin_amdgcn_sched_barrier(0);
        if (ks < KS) {
          if (FIRST) un = mma32(f[ks % 3], w2[ks % KS], un);
          steps((before + 2) * STEPS / (3 * KS));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    auto slots = [&](const uint32_t* q, int st) { return __builtin_bit_cast(bf16x8, make_uint4(q[4 * st], q[4 * st + 1], q[4 * st + 2], q[4 * st + 3])); };
    // The gradients' products over the patch in hand.
    auto gradients = [&](const char* kt, const char* vt, const Rates& r, auto after_v) {
      constexpr int N = D / 32 * 2;
      bf16x8 fk[3], fv[3];
      auto read = [&](int n) {
        if (n >= N) return;
        fk[n % 3] = frag.cols(kt, n / 2, n % 2);
        fv[n % 3] = frag.cols(vt, n / 2, n % 2);
      };
      read(0);
      read(1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const int dt = n / 2, st = n % 2;
        read(n + 2);
        d1[dt] = mma32(fv[n % 3], slots(q1, st), d1[dt]);
        const uint4 x = __builtin_bit_cast(uint4, fk[n % 3]);
        const float k[8] = {bf16_lo(x.x), bf16_hi(x.x), bf16_lo(x.y), bf16_hi(x.y), bf16_lo(x.z), bf16_hi(x.z), bf16_lo(x.w), bf16_hi(x.w)};
        const bf16x8 k0 = st == 0 ? scaled<0>(k, r.r[0]) : scaled<8>(k, r.r[0]);
        __builtin_amdgcn_sched_barrier(0);
        d0[dt] = mma32(slots(q0, st), k0, d0[dt]);
        const bf16x8 k2 = st == 0 ? scaled<0>(k, r.r[2]) : scaled<8>(k, r.r[2]);
        __builtin_amdgcn_sched_barrier(0);
        d2[dt] = mma32(slots(q2, st), k2, d2[dt]);
      }
      __builtin_amdgcn_sched_barrier(0);
      after_v();
    };
    f32x16 g, u, e, gn, un, en;
    clear(0, 0, 1);
    products(yes, no, unit(0), unit(1), g, u, e, gn, un, en, 0.f, [] {});
    int kc = 0, vc = 1, k1 = 2, v1 = 3, idle = 4;      // units of the current and the next patch
    for (int i = 0; i + 1 < mine; ++i) {
      wait_vmcnt<U::COPIES>();          // the next patch's k: nothing but its v (and its rates) was asked for later
      clear(i + 1, k1, v1);
      products(yes, yes, unit(k1), unit(v1), gn, un, en, g, u, e, rc.r[1], [&] {
        wait_vmcnt<0>();
        settle(rn, i + 1);              // (before the copies to come, which would have to arrive first)
        __builtin_amdgcn_sched_barrier(0);
        issue_k(i + 2, idle);
      });
      gradients(unit(kc), unit(vc), rc, [&] { issue_v(i + 2, vc); });
      g = gn; u = un; e = en;
      rc = rn;
      rn = rates(i + 2);
      const int k2 = idle, v2 = vc;
      idle = kc; kc = k1; vc = v1; k1 = k2; v1 = v2;
    }
    products(no, yes, smem, smem, gn, un, en, g, u, e, rc.r[1], [] {});
    gradients(unit(kc), unit(vc), rc, [] {});
  }
  wait_vmcnt<0>();
  __syncthreads();

  // the waves' sums, a matrix at a time: [wave][32 columns or rows of d][four registers][lane]
  auto put = [&](const f32x16 (&d)[D / 32], int buf) {
    float4* o = reinterpret_cast<float4*>(smem + buf * U::SUMS) + wave * D * 8 + lane;
#pragma unroll
    for (int t = 0; t < D / 32; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) o[(t * 4 + q) * 64] = make_float4(d[t][4 * q], d[t][4 * q + 1], d[t][4 * q + 2], d[t][4 * q + 3]);
  };
  float* out = p.partial + bx * p.split_stride + (long long)z * D * p.dh;
  auto add = [&](int mat, int buf) {
    const float4* s = reinterpret_cast<const float4*>(smem + buf * U::SUMS) + wave * 64 + lane;
    float* o = out + mat * p.mat_stride;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) {
      float4 v = s[t * 256];
#pragma unroll
      for (int w = 1; w < 4; ++w) {
        const float4 a = s[t * 256 + w * D * 8];
        v.x += a.x; v.y += a.y; v.z += a.z; v.w += a.w;
      }
      const float x[4] = {v.x, v.y, v.z, v.w};
      const int row = 8 * wave + 4 * h, col = lane & 31;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (mat == 1) o[(size_t)(t * 32 + row + j) * p.dh + hid0 + col] = x[j];
        else o[(size_t)(hid0 + row + j) * D + t * 32 + col] = x[j];
    }
  };
  put(d0, 0);
  __syncthreads();
  put(d1, 1);
  add(0, 0);
  __syncthreads();
  put(d2, 0);
  add(1, 1);
  __syncthreads();
  add(2, 0);
}

// ---- backward of an update: the tokens' gradients -------------------------------------------------------------------------------
// From k, v, the weights and the gradients G of their gradients: the gradients of the pre-activations (stored, for the weights'
// reduction over the tokens), dk, dv and the learning rates'.  A wave owns 32 tokens as matrix columns and walks the hidden units 32
// at a time: six products, the pointwise part in registers, and the six terms of dk and dv, which take its results as they lie.  The
// weights' and gradients' 32 rows (or columns) travel through a ring shared by the block.
//
// What bounds it: issue of the one wave on a SIMD, 1130 vector operations a stage (64 a hidden value, of which 19 round) in 6300 clocks; the
// terms' matrix instructions hide behind them, the six products' do not (1800), and 512 registers hold no second set of their sums.
// Copies: 800.  us, this kernel and the reduction / hidden stage and the reduction with dk and dv beside it: 12 x 4680 tokens, d = 128,
// dh = 256 96 + 28 / 92 + 62; 24 x 2500 tokens, d = dh = 96 39 + 14 / 46 + 38.  Six arrays of [tokens, hidden] less written and nine
// less read than there: three are written here, for the reduction.
struct UpdateBwdFusedParams {
  int T, dh;
  const uint16_t* K; int ldk; long long bsk;               // [T, d]
  const uint16_t* V; int ldv; long long bsv;
  const uint16_t* W0; const uint16_t* W1; const uint16_t* W2;
  const uint16_t* G0; const uint16_t* G1; const uint16_t* G2; long long bsw;
  const float* lr0; const float* lr1; const float* lr2; long long bslr;
  uint16_t* O0; uint16_t* O1; uint16_t* O2; long long bso; // [T, dh]: gradients of k W0^T, v W1, k W2^T
  uint16_t* dk; uint16_t* dv; long long bsd;               // [T, d], rows one after the other
  float* lrpart; long long lr_stride;                      // [3][b][..]: sums for the learning rates
  int ldlr;
  TileMap map;                                             // 128 tokens, 1, batch
};

template <int D>
struct BwdStage {
  using U = UpdatePatch<D>;
  static constexpr int SIDE = U::BYTES, TALL = D * 64;     // 32 rows of W0, W2, G0, G2; [d][32] of W1, G1
  static constexpr int BYTES = 4 * SIDE + 2 * TALL, RING = 3 * BYTES, LDS = cmax(RING, 4 * 32 * (D + 8) * 2);
  static_assert(LDS <= 160 * 1024, "the ring does not fit the LDS");
};

// The barrier without the wait for the wave's stores to memory that __syncthreads adds.  The wave's reads of LDS are done, which a slot's
// next copy has to be sure of (they are used by then, so the wait costs nothing; but where their last uses stand is the compiler's
// choice), and its copies into LDS are waited for by name; no access of the program moves across.
__device__ __forceinline__ void block_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// A stage of W1 or G1 in LDS: [d][32 hidden], rows of 64 bytes, granule g of row r at slot g ^ (r >> 2) & 3.
struct TallFrag {
  uint32_t tr_off[2], row_off[2];
  // of a copy of 16 rows, within the operand
  __device__ static __forceinline__ uint32_t copy_offset(int dh) {
    const int lane = threadIdx.x & 63;
    return (uint32_t)((lane >> 2) * dh + ((lane & 3) ^ ((lane >> 4) & 3)) * 8) * 2;
  }
  __device__ __forceinline__ void init() {
    const int lane = threadIdx.x & 63, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      tr_off[i] = (8 * h + ((lane & 15) >> 2) + 4 * i) * 64 + (((2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ ((2 * h + i) & 3)) << 4) + (lane & 1) * 8;
      row_off[i] = (lane & 31) * 64 + ((i ^ ((lane >> 2) & 3)) << 4) + h * 8;
    }
  }
  // the 32 hidden units as matrix rows over 16 of d
  __device__ __forceinline__ bf16x8 columns(const char* m, int ks) const {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(m + tr_off[0] + ks * 1024)), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(m + tr_off[1] + ks * 1024));
    const s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(bf16x8, v);
  }
  // 32 of d as matrix rows over 16 hidden units in the order of the products' results (the upper 16: granules two on, a bit of the slot)
  __device__ __forceinline__ bf16x8 rows(const char* m, int dt, int st) const {
    const uint2 a = *reinterpret_cast<const uint2*>(m + dt * 2048 + (row_off[0] ^ (st << 5))), b = *reinterpret_cast<const uint2*>(m + dt * 2048 + (row_off[1] ^ (st << 5)));
    return __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
  }
};
// Sixteen hidden units (two rounds of four a lane half, two words each, r and r + 2) of a token, 16 bytes a lane: the lower half of
// the wave writes the eight units of the first round, the upper half those of the second.
__device__ __forceinline__ void store_units(uint16_t* out, const uint32_t* r) {
  const auto x = __builtin_amdgcn_permlane32_swap(r[0], r[2], false, false), y = __builtin_amdgcn_permlane32_swap(r[1], r[3], false, false);
  *reinterpret_cast<uint4*>(out) = make_uint4(x[0], y[0], x[1], y[1]);
}

// The pointwise part on four hidden units of a token, in eight steps.  Roundings as in update_pointwise2.  One operation on all four
// after the other: in the compiler's order, each result right behind its operands, a wave alone on its SIMD waits for most of them.
struct BwdSteps {
  float g[4], h2[4], dh[4], z0[4], z1[4], z2[4];           // the rounded products
  float sig[4], silu[4], om[4], d1[4], d2[4], sg[4], sb[4], hid[4], dh2[4], p[4], t[4], x[4];
  uint32_t w[6][2];                                        // gradients of k W0^T, k W2^T; lr-scaled dgate, dhidden; gradient of v W1; lr-scaled hidden
  template <class F>
  __device__ __forceinline__ void each(F f) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) f(j);
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void pack(uint32_t (&o)[2]) const {
    o[0] = pack_bf16(x[0], x[1]); o[1] = pack_bf16(x[2], x[3]);
  }
  template <int STEP, int I>
  __device__ __forceinline__ void step(const f32x16 (&a)[6], float l0, float l1, float l2, float& s0, float& s1, float& s2) {
    if (STEP == 0) {
      each([&](int j) { g[j] = round_bf16(a[0][4 * I + j]); h2[j] = round_bf16(a[1][4 * I + j]); dh[j] = round_bf16(a[4][4 * I + j]); });
      each([&](int j) { z0[j] = round_bf16(a[2][4 * I + j]); z2[j] = round_bf16(a[3][4 * I + j]); z1[j] = round_bf16(a[5][4 * I + j]); });
    } else if (STEP == 1) {
      each([&](int j) { sig[j] = sigmoidf_(g[j]); p[j] = dh[j] * h2[j]; });
      each([&](int j) { silu[j] = g[j] * sig[j]; om[j] = 1.f - sig[j]; });
      each([&](int j) { sg[j] = round_bf16(silu[j]); sb[j] = round_bf16(sig[j]); });
    } else if (STEP == 2) {
      each([&](int j) { hid[j] = sg[j] * h2[j]; dh2[j] = dh[j] * sg[j]; });
      each([&](int j) { hid[j] = round_bf16(hid[j]); dh2[j] = round_bf16(dh2[j]); t[j] = round_bf16(p[j]); });
      each([&](int j) { t[j] *= sb[j]; sb[j] = 1.f - sb[j]; d1[j] = __builtin_fmaf(g[j], om[j], 1.f); });
      each([&](int j) { t[j] = round_bf16(t[j]); sb[j] = round_bf16(sb[j]); d1[j] *= sig[j]; });
    } else if (STEP == 3) {
      each([&](int j) { sb[j] *= g[j]; d2[j] = __builtin_fmaf(-2.f, sig[j], 1.f); om[j] *= sig[j]; });
      each([&](int j) { sb[j] = round_bf16(sb[j]); d2[j] = __builtin_fmaf(g[j], d2[j], 2.f); });
      each([&](int j) { sb[j] += 1.f; d2[j] *= om[j]; });
      each([&](int j) { sb[j] = round_bf16(sb[j]); d2[j] *= p[j]; });
    } else if (STEP == 4) {
      each([&](int j) { t[j] *= sb[j]; s1 = __builtin_fmaf(z1[j], hid[j], s1); x[j] = hid[j] * l1; });
      pack(w[5]);
      each([&](int j) { t[j] = round_bf16(t[j]); s2 = __builtin_fmaf(z2[j], dh2[j], s2); x[j] = dh2[j] * l2; });      // t: dgate before the activation
      pack(w[3]);
    } else if (STEP == 5) {
      each([&](int j) { s0 = __builtin_fmaf(z0[j], t[j], s0); x[j] = t[j] * l0; });
      pack(w[2]);
      each([&](int j) { z0[j] *= l0; z1[j] *= l1; z2[j] *= l2; });
      each([&](int j) { h2[j] *= d1[j]; dh[j] *= d1[j]; });
    } else if (STEP == 6) {
      each([&](int j) { x[j] = z0[j] * h2[j]; t[j] = z0[j] * dh[j]; });
      each([&](int j) { x[j] = __builtin_fmaf(z2[j], silu[j], x[j]); t[j] = __builtin_fmaf(z1[j], silu[j], t[j]); });
      pack(w[4]);
      each([&](int j) { x[j] = t[j]; });
      pack(w[1]);
    } else {
      each([&](int j) { x[j] = z0[j] * d2[j]; });
      each([&](int j) { x[j] = __builtin_fmaf(z2[j], dh[j], x[j]); });
      each([&](int j) { x[j] = __builtin_fmaf(z1[j], h2[j], x[j]); });
      pack(w[0]);
    }
  }
};

template <int D>
__global__ __launch_bounds__(256, 1) void k_update_bwd_fused(const UpdateBwdFusedParams p) {
  prefetch_args<sizeof(p)>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using ST = BwdStage<D>;
  using U = UpdatePatch<D>;
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, h = lane >> 5;
  const int row0 = (bx * 4 + wave) * 32, row = row0 + (lane & 31), dh = p.dh, n = dh / 32;
  const uint32_t lds0 = lds_addr(smem);
  const long long w = z * p.bsw;
  // copies: a quarter of every operand's KiB each, the operands of a kind at the same offsets
  UpdateCopies<D> cp;
  cp.init(D);
  const uint32_t tall_off = TallFrag::copy_offset(dh);
  uint32_t side_off = cp.voff[0];
#pragma unroll
  for (int i = 1; i < 4; ++i) side_off = wave == i ? cp.voff[i] : side_off;
  auto issue = [&](int t, int slot) {
    const uint32_t to = lds0 + slot;
    const long long rows = w + (long long)t * 32 * D, cols = w + t * 32;
    const uint16_t* const side[4] = {p.W0 + rows, p.W2 + rows, p.G0 + rows, p.G2 + rows};
    const uint16_t* const tall[2] = {p.W1 + cols, p.G1 + cols};
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int j = 0; j < U::COPIES / 4; ++j) dma16<false>(side[m] + (size_t)j * 16 * D, side_off, to + m * ST::SIDE + (wave + 4 * j) * 1024);
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int j = 0; j < (D / 16 + 3) / 4; ++j)
        if (wave + 4 * j < D / 16)
          dma16<false>(tall[m] + (size_t)(wave + 4 * j) * 16 * dh, tall_off, to + 4 * ST::SIDE + m * ST::TALL + (wave + 4 * j) * 1024);
  };
  issue(0, 0);
  constexpr int KS = D / 16, DT = D / 32;
  bf16x8 kf[KS], vf[KS];
  attn_own_rows<D>(kf, p.K + z * p.bsk, p.ldk, row, p.T);
  attn_own_rows<D>(vf, p.V + z * p.bsv, p.ldv, row, p.T);
  const int token = min(row, p.T - 1);
  const float l0 = p.lr0[z * p.bslr + token], l1 = p.lr1[z * p.bslr + token], l2 = p.lr2[z * p.bslr + token];
  AttnFrag<U::P> frag;
  frag.init();
  TallFrag tall_frag;
  tall_frag.init();
  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) dk[i][j] = dv[i][j] = 0.f;
  uint32_t res[6][8];      // of the units in hand, two a word, in the order of the operands in LDS
#pragma unroll
  for (int m = 0; m < 6; ++m)
#pragma unroll
    for (int j = 0; j < 8; ++j) res[m][j] = 0;
  float s0 = 0.f, s1 = 0.f, s2 = 0.f;

  // terms [from, to) of dk and dv over 16 hidden units (half st of the stage), their weights read two ahead
  constexpr int TERMS = 6 * DT;
  bf16x8 tf[3];
  auto term_read = [&](const char* stage, int st, int i) {
    if (i >= TERMS) return;
    const int m = i / DT, dt = i % DT;
    tf[i % 3] = m < 4 ? frag.cols(stage + m * ST::SIDE, dt, st) : tall_frag.rows(stage + 4 * ST::SIDE + (m - 4) * ST::TALL, dt, st);
  };
  auto term = [&](const char* stage, int st, int i) {
    const int m = i / DT, dt = i % DT;
    term_read(stage, st, i + 2);
    const bf16x8 r = __builtin_bit_cast(bf16x8, make_uint4(res[m][4 * st], res[m][4 * st + 1], res[m][4 * st + 2], res[m][4 * st + 3]));
    if (m < 4) dk[dt] = mma32(tf[i % 3], r, dk[dt]);
    else dv[dt] = mma32(tf[i % 3], r, dv[dt]);
  };
  f32x16 a[6];
  // Two rounds of four hidden units, between their steps the terms of the 16 units before.
  auto rounds = [&](auto half, const char* stage, int st) {
    constexpr int H = decltype(half)::value;
    BwdSteps b;
    int done = 0;
    term_read(stage, st, 0);
    term_read(stage, st, 1);
    auto terms = [&](int upto) {
#pragma unroll
      for (int i = 0; i < TERMS; ++i)
        if (i >= done && i < upto) term(stage, st, i);
      done = upto;
      __builtin_amdgcn_sched_barrier(0);
    };
    auto round = [&](auto rd) {
      constexpr int I = decltype(rd)::value, AT = (I - 2 * H) * 8;
      b.step<0, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 1) * TERMS / 16);
      b.step<1, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 2) * TERMS / 16);
      b.step<2, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 3) * TERMS / 16);
      b.step<3, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 4) * TERMS / 16);
      b.step<4, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 5) * TERMS / 16);
      b.step<5, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 6) * TERMS / 16);
      b.step<6, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 7) * TERMS / 16);
      b.step<7, I>(a, l0, l1, l2, s0, s1, s2); terms((AT + 8) * TERMS / 16);
#pragma unroll
      for (int m = 0; m < 6; ++m)
#pragma unroll
        for (int i = 0; i < 2; ++i) res[m][2 * I + i] = b.w[m][i];
    };
    round(std::integral_constant<int, 2 * H>{});
    round(std::integral_constant<int, 2 * H + 1>{});
  };
  // (lanes past the last token hold its values and write them once more: no branch between the steps, across which the compiler would
  // move work that the matrix instructions are to hide behind)
  const long long mine = z * p.bso + (long long)token * dh + 8 * h;
  uint16_t* const out[3] = {p.O0 + mine, p.O2 + mine, p.O1 + mine};
  auto store = [&](int t, int H) {
#pragma unroll
    for (int o = 0; o < 3; ++o) store_units(out[o] + t * 32 + 16 * H, res[o == 2 ? 4 : o] + 4 * H);
  };
  wait_vmcnt<0>();
  int prev = 0, cur = 0, next = ST::BYTES;      // the ring's stages (the first one stands for the one before it)
  for (int t = 0; t < n; ++t) {
    wait_vmcnt<6>();      // behind this stage's copies come the six stores of the stage before only
    block_barrier();
    issue(min(t + 1, n - 1), next);
    const char* stage = smem + cur;
    {
      bf16x8 f[2][4];
      auto read = [&](int ks) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
          if (ks < KS) f[ks & 1][m] = frag.rows(stage + m * ST::SIDE, 0, ks);
        if (ks >= KS && ks < 2 * KS)
#pragma unroll
          for (int m = 0; m < 2; ++m) f[ks & 1][m] = tall_frag.columns(stage + 4 * ST::SIDE + m * ST::TALL, ks - KS);
      };
      read(0);
#pragma unroll
      for (int m = 0; m < 6; ++m)
#pragma unroll
        for (int j = 0; j < 16; ++j) a[m][j] = 0.f;
#pragma unroll
      for (int ks = 0; ks < 2 * KS; ++ks) {
        read(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
        if (ks < KS) {
#pragma unroll
          for (int m = 0; m < 4; ++m) a[m] = mma32(f[ks & 1][m], kf[ks % KS], a[m]);
        } else {
#pragma unroll
          for (int m = 0; m < 2; ++m) a[4 + m] = mma32(f[ks & 1][m], vf[ks % KS], a[4 + m]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rounds(std::integral_constant<int, 0>{}, smem + prev, 1);      // (the first time of zeros)
    store(t, 0);
    rounds(std::integral_constant<int, 1>{}, stage, 0);
    store(t, 1);
    prev = cur; cur = next; next = next == 2 * ST::BYTES ? 0 : next + ST::BYTES;
  }
  term_read(smem + prev, 1, 0);
  term_read(smem + prev, 1, 1);
#pragma unroll
  for (int i = 0; i < TERMS; ++i) term(smem + prev, 1, i);
  s0 += __shfl_xor(s0, 32, 64); s1 += __shfl_xor(s1, 32, 64); s2 += __shfl_xor(s2, 32, 64);
  if (lane < 32 && row < p.T) {
    float* o = p.lrpart + (size_t)z * p.ldlr + row;
    o[0] = s0; o[p.lr_stride] = s1; o[2 * p.lr_stride] = s2;
  }
  wait_vmcnt<0>();
  __syncthreads();
  char* t = smem + wave * 32 * (D + 8) * 2;
  if (row0 < p.T) {
    attn_store_rows<D>(t, dk, 1.f, p.dk + z * p.bsd, D, row0, p.T);
    attn_store_rows<D>(t, dv, 1.f, p.dv + z * p.bsd, D, row0, p.T);
  }
}

// ---- backward of an apply: the hidden stage and dq ------------------------------------------------------------------------------
//   g, u, e = q W0^T, q W2^T, dout W1  ->  hidden, dg, du [T, dh] (stored, for the weights' gradients);  dq = dg W0 + du W2
// As above with three products and two terms: two waves fit a SIMD and cover each other's latencies, 256 tokens a block.
//
// What bounds it: memory, 130 MB read and written at 12 x 4680 tokens, d = 128, dh = 256 in 35 us (27 at a large copy's rate); as kernels
// of their own the hidden stage takes 43 us and dq 17, and dq reads two of the arrays again.  24 x 2500 tokens, d = dh = 96: 20 / 23 + 9.
struct ApplyBwdFusedParams {
  int T, dh;
  const uint16_t* X; int ldx; long long bsx;               // [T, d] queries
  const uint16_t* Y; int ldy; long long bsy;               // [T, d] gradients of the output
  const uint16_t* W0; const uint16_t* W1; const uint16_t* W2; long long bsw;
  uint16_t* O0; uint16_t* O1; uint16_t* O2; long long bso; // [T, dh]: hidden, gradients of q W0^T and of q W2^T
  uint16_t* dq; long long bsd;
  StepBatch steps; long long gsx, gsy, gsw, gsd;           // several steps of the program in one launch
  TileMap map;                                             // 256 tokens, 1, batch
};
template <int D>
struct ApplyBwdStage {
  using U = UpdatePatch<D>;
  static constexpr int SIDE = U::BYTES, BYTES = 2 * SIDE + D * 64, LDS = cmax(2 * BYTES, 8 * 32 * (D + 8) * 2);
};

template <int D>
__global__ __launch_bounds__(512, 2) void k_apply_bwd_fused(const ApplyBwdFusedParams p) {
  prefetch_args<sizeof(p)>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using ST = ApplyBwdStage<D>;
  using U = UpdatePatch<D>;
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, h = lane >> 5;
  const int row0 = (bx * 8 + wave) * 32, row = row0 + (lane & 31), dh = p.dh, n = dh / 32;
  const long long w = p.steps.at(z, p.bsw, p.gsw);
  const uint32_t lds0 = lds_addr(smem), tall_off = TallFrag::copy_offset(dh);
  uint32_t side_off;
  {
    UpdateCopies<D> cp;
    cp.init(D);
    side_off = cp.voff[0];
#pragma unroll
    for (int i = 1; i < 4; ++i) side_off = wave % 4 == i ? cp.voff[i] : side_off;
  }
  auto issue = [&](int t) {
    const uint32_t to = lds0 + (t & 1) * ST::BYTES + wave * 1024;
    const long long rows = w + ((long long)t * 32 + wave / 4 * 16) * D;
    if (wave < U::COPIES) {
      dma16<false>(p.W0 + rows, side_off, to);
      dma16<false>(p.W2 + rows, side_off, to + ST::SIDE);
    }
    if (wave < D / 16) dma16<false>(p.W1 + w + (size_t)wave * 16 * dh + t * 32, tall_off, to + 2 * ST::SIDE);
  };
  issue(0);
  constexpr int KS = D / 16, DT = D / 32;
  bf16x8 qf[KS], gf[KS];
  attn_own_rows<D>(qf, p.X + p.steps.at(z, p.bsx, p.gsx), p.ldx, row, p.T);
  attn_own_rows<D>(gf, p.Y + p.steps.at(z, p.bsy, p.gsy), p.ldy, row, p.T);
  AttnFrag<U::P> frag;
  frag.init();
  TallFrag tall;
  tall.init();
  // (lanes past the last token hold its values and write them once more)
  const long long mine = z * p.bso + (long long)min(row, p.T - 1) * dh + 8 * h;
  uint16_t* const out[3] = {p.O0 + mine, p.O1 + mine, p.O2 + mine};
  f32x16 dq[DT];
#pragma unroll
  for (int i = 0; i < DT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) dq[i][j] = 0.f;
  wait_vmcnt<0>();
  for (int t = 0; t < n; ++t) {
    wait_vmcnt<6>();      // behind this stage's copies come the six stores of the stage before only
    block_barrier();
    issue(min(t + 1, n - 1));
    const char* stage = smem + (t & 1) * ST::BYTES;
    f32x16 g, u, e;
#pragma unroll
    for (int j = 0; j < 16; ++j) g[j] = u[j] = e[j] = 0.f;
    bf16x8 f[2][2];
    auto read = [&](int ks) {
      if (ks < KS) {
        f[ks & 1][0] = frag.rows(stage, 0, ks);
        f[ks & 1][1] = frag.rows(stage + ST::SIDE, 0, ks);
      } else if (ks < 2 * KS) {
        f[ks & 1][0] = tall.columns(stage + 2 * ST::SIDE, ks - KS);
      }
    };
    read(0);
#pragma unroll
    for (int ks = 0; ks < 2 * KS; ++ks) {
      read(ks + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (ks < KS) {
        g = mma32(f[ks & 1][0], qf[ks % KS], g);
        u = mma32(f[ks & 1][1], qf[ks % KS], u);
      } else {
        e = mma32(f[ks & 1][0], gf[ks % KS], e);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      uint32_t r[3][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float o[3][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float y0 = round_bf16(g[8 * st + 2 * i + j]), y2 = round_bf16(u[8 * st + 2 * i + j]), gh = round_bf16(e[8 * st + 2 * i + j]);
          const SiluParts s = silu_parts(y0);
          const float sg = round_bf16(s.silu), dy = round_bf16(gh * y2);
          o[0][j] = sg * y2; o[1][j] = dy * s.d1; o[2][j] = gh * sg;
        }
#pragma unroll
        for (int m = 0; m < 3; ++m) r[m][i] = pack_bf16(o[m][0], o[m][1]);
      }
#pragma unroll
      for (int m = 0; m < 3; ++m) store_units(out[m] + t * 32 + 16 * st, r[m]);
      const bf16x8 dg = __builtin_bit_cast(bf16x8, make_uint4(r[1][0], r[1][1], r[1][2], r[1][3])), du = __builtin_bit_cast(bf16x8, make_uint4(r[2][0], r[2][1], r[2][2], r[2][3]));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        dq[dt] = mma32(frag.cols(stage, dt, st), dg, dq[dt]);
        dq[dt] = mma32(frag.cols(stage + ST::SIDE, dt, st), du, dq[dt]);
      }
    }
  }
  wait_vmcnt<0>();
  __syncthreads();
  if (row0 < p.T) attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, dq, 1.f, p.dq + p.steps.at(z, p.bsd, p.gsd), D, row0, p.T);
}

}  // namespace lact
