// Hidden stages of an update and of an apply's backward on 256 x 128 tiles: eight waves that all copy and all compute.
//
// The 128 x 128 kernels of gemm_dma_kernels.h run at the rate a compute unit gets its operands (2 x 4680 tokens, d = 768, dh = 1536: 0.9 us
// per K-step of 40 KiB on average against 0.32 us of matrix work): a tile of twice the rows copies 0.7 of the bytes per product.  Its
// accumulators need all eight waves of the block, so the copies are theirs as well: four to eight instructions per wave and K-step, issued
// behind the barrier that frees the slots they fill, where the other wave of the SIMD has matrix work in flight.  us, 128 x 128 /
// these: at that shape update 140 / 118, apply backward 113 / 95; 12 x 4680 tokens, d = 384, dh = 768 276 / 261 and 210 / 197; 16 x 2048 tokens,
// d = dh = 384 (whole rounds of the small tiles, one and a half of these) 79 / 82 and even.  Of 24 K-steps' 37 us the copies alone take
// 28, matrix instructions and fragments 20.  The apply's two products run as fast on persistent 128 x 128 tiles.
//
// Ring: three slots of the token tile (32 KiB) and two of the weight tiles (2 x 16 KiB), all 160 KiB of LDS.  The token rows come
// from HBM and are asked for three K-steps ahead, the weights from the L2 two ahead.  One barrier per K-step.  All 256 registers of a wave
// are in use; eight more (36 bytes a lane) are stored and read back once a block, outside the loops.
#pragma once
#include <type_traits>

#include "gemm_dma_kernels.h"

namespace lact {

using TS_WIDE = TileShape<256, 128, 4, 2>;   // 64 x 64 per wave and accumulator
constexpr int WIDE_A = TS_WIDE::BM * 128, WIDE_B = TS_WIDE::BN * 128;
constexpr int WIDE_LDS = 3 * WIDE_A + 2 * 2 * WIDE_B;
static_assert(WIDE_LDS <= 160 * 1024, "the ring does not fit the LDS");

// One wave's share (one eighth) of the copies of a tile of ROWS rows and one K-step; layouts as in gemm_dma.h.
template <int ROWS>
struct WideLane {
  static constexpr int N = ROWS / 64;   // copies of 1 KiB
  uint32_t voff[N];
  __device__ __forceinline__ void init_kc(int ld, int rows, int wave) {
    const int lane = threadIdx.x & 63, row0 = wave * 8 + (lane >> 3), last = rows - 1;
    const uint32_t kv = ((lane & 7) ^ ((row0 >> 1) & 7)) * 16, ld2 = (uint32_t)ld * 2;   // the copies' rows differ by 64
#pragma unroll
    for (int i = 0; i < N; ++i) voff[i] = __umul24(min(row0 + i * 64, last), ld2) + kv;
  }
  __device__ __forceinline__ void init_ks(int ld, int rows, int wave) {   // [64 k][ROWS], the granules of k-row k rotated by 4 * (k % 4)
    constexpr int G = ROWS / 8;
    const int L = wave * 64 + (threadIdx.x & 63), last = rows / 8 - 1;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int k = (L + i * 512) / G, g = (L + i * 512 + G - (4 * (k & 3)) % G) % G;
      voff[i] = __umul24(k, (uint32_t)ld * 2) + min(g, last) * 16;
    }
  }
  template <int FROM = 0, int TO = N>
  __device__ __forceinline__ void issue(const uint16_t* base, uint32_t lds_tile, int wave) const {
#pragma unroll
    for (int i = FROM; i < TO; ++i) dma16<false>(base, voff[i], lds_tile + (wave + i * 8) * 1024);
  }
};

// One phase of a tile: acc[j] += A B_j^T over nk K-steps of 64, j < NB.  Both B operands have one layout (B_KS: K-strided).
template <int NB, bool B_KS>
struct WidePhase {
  static constexpr int COPIES_A = TS_WIDE::BM / 64;
  const uint16_t* a; const uint16_t* b[NB];   // first row of the tile, k = 0
  size_t bstep;                               // elements of B between K-steps
  int nk;
  WideLane<TS_WIDE::BM> la;
  WideLane<TS_WIDE::BN> lb;
  __device__ __forceinline__ void init(int lda, int rows_a, int ldb, int rows_b, int K, int wave) {
    la.init_kc(lda, rows_a, wave);
    if (B_KS) lb.init_ks(ldb, rows_b, wave);
    else lb.init_kc(ldb, rows_b, wave);
    bstep = B_KS ? (size_t)DMA_BK * ldb : (size_t)DMA_BK;
    nk = K / DMA_BK;
  }
};
struct WideNone {
  static constexpr int nk = 0;
};

// The ring: LDS offsets of the slots in use and of those to fill next.
struct WideRing {
  uint32_t lds, a_use, a_fill, b_use, b_fill;
  int wave;
  __device__ __forceinline__ void init(char* smem) {
    lds = lds_addr(smem);
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    a_use = a_fill = 0; b_use = b_fill = 3 * WIDE_A;
  }
  __device__ static __forceinline__ void next_a(uint32_t& o) { o = o == 2 * WIDE_A ? 0 : o + WIDE_A; }
  __device__ static __forceinline__ void next_b(uint32_t& o) { o = o == 3 * WIDE_A ? 3 * WIDE_A + 2 * WIDE_B : 3 * WIDE_A; }
  // K-step k's tiles in parts of two copies: part 0, 1 of the token tile; part j is operand j of the weights
  template <int PART, int NB, bool KS>
  __device__ __forceinline__ void issue_a(const WidePhase<NB, KS>& ph, int k) {
    ph.la.template issue<2 * PART, 2 * PART + 2>(ph.a + (size_t)k * DMA_BK, lds + a_fill, wave);
    if (PART == 1) next_a(a_fill);
  }
  template <int PART, int NB, bool KS>
  __device__ __forceinline__ void issue_b(const WidePhase<NB, KS>& ph, int k) {
    if constexpr (PART < NB) ph.lb.issue(ph.b[PART] + k * ph.bstep, lds + b_fill + PART * WIDE_B, wave);
    if (PART + 1 == NB) next_b(b_fill);
  }
  template <int PART> __device__ __forceinline__ void issue_a(const WideNone&, int) {}
  template <int PART> __device__ __forceinline__ void issue_b(const WideNone&, int) {}
  template <class PH>
  __device__ __forceinline__ void start(const PH& ph) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      issue_a<0>(ph, k); issue_a<1>(ph, k);
      if (k < 2) { issue_b<0>(ph, k); issue_b<1>(ph, k); }
    }
  }
};

// Runs one phase; `next` is the one behind it (WideNone: the last).  Every phase has three K-steps or more.  Opening K-step s
// asks for the weight tiles of s + 1 and the token tile of s + 2 (into the slots of s - 1, which every wave has left behind the
// barrier), so that of what was asked for behind the tiles of s only a token tile may be on its way when s opens.  The copies are
// issued two at a time in the middle of a sub-step's products: eight waves that issue eight each at once wait for the address
// queue instead of computing.  The last K-steps stand apart: no branch lies between the matrix instructions of a loop, around which the register allocator would move accumulators.
template <bool FIRST, int NB, bool B_KS, class NEXT>
__device__ __forceinline__ void wide_phase(char* smem, WideRing& ring, const WidePhase<NB, B_KS>& ph, const NEXT& next, f32x16 (&acc)[NB][TS_WIDE::TM][TS_WIDE::TN]) {
  using TS = TS_WIDE;
  constexpr bool LAST = std::is_same<NEXT, WideNone>::value;
  constexpr int CA = WidePhase<NB, B_KS>::COPIES_A;
  const int wave = threadIdx.x >> 6;
  FragSrc<TS::BM, false> sa[TS::TM];
  FragSrc<TS::BN, B_KS> sb[TS::TN];
#pragma unroll
  for (int i = 0; i < TS::TM; ++i) sa[i].init((wave / TS::WAVES_N) * TS::WM + i * 32);
#pragma unroll
  for (int n = 0; n < TS::TN; ++n) sb[n].init((wave % TS::WAVES_N) * TS::WN + n * 32);
  bf16x8 fa[2][TS::TM], fb[2][NB][TS::TN];
  const char *ta = nullptr, *tb = nullptr;
  auto fetch = [&](int buf, int ks) {
#pragma unroll
    for (int i = 0; i < TS::TM; ++i) fa[buf][i] = sa[i].fetch(ta, ks);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int n = 0; n < TS::TN; ++n) fb[buf][j][n] = sb[n].fetch(tb + j * WIDE_B, ks);
  };
  constexpr int READS = TS::TM + (B_KS ? 2 : 1) * NB * TS::TN, HALF = NB * TS::TM * TS::TN / 2;
  auto products = [&](int buf, int half) {
#pragma unroll
    for (int e = half * HALF; e < (half + 1) * HALF; ++e) {
      const int j = e / (TS::TM * TS::TN), i = e / TS::TN % TS::TM, n = e % TS::TN;
      acc[j][i][n] = mma32(fb[buf][j][n], fa[buf][i], acc[j][i][n]);
    }
  };
  // one sub-step's products, the fragments of the next behind the first of them, copies in the middle
  auto sub = [&](int buf, int ks, auto copies) {
    fetch(buf ^ 1, ks);
    products(buf, 0);
    sched_interleave<READS, HALF>();
    copies();
    products(buf, 1);
  };
  auto none = [] {};
  // K-step s opens behind the wait for this wave's copies; PB, PA: the phases whose tiles kb, ka are asked for
  auto open = [&]() {
    __syncthreads();
    ta = smem + ring.a_use; tb = smem + ring.b_use;
    WideRing::next_a(ring.a_use); WideRing::next_b(ring.b_use);
  };
  auto step = [&](const auto& pb, int kb, const auto& pa, int ka) {
    open();
    sub(1, 0, [&] { ring.template issue_b<0>(pb, kb); });      // the previous K-step's last products
    sub(0, 1, [&] { ring.template issue_b<1>(pb, kb); });
    sub(1, 2, [&] { ring.template issue_a<0>(pa, ka); });
    sub(0, 3, [&] { ring.template issue_a<1>(pa, ka); });
  };
  if (FIRST) wait_vmcnt<2 * CA>();      // two token tiles and more were asked for behind the first tiles
  else wait_vmcnt<CA>();
  open();
  fetch(0, 0);
  if (FIRST) {
    sub(0, 1, none); sub(1, 2, none); sub(0, 3, none);
  } else {
    ring.template issue_b<0>(ph, 1); ring.template issue_b<1>(ph, 1);
    sub(0, 1, none);
    sub(1, 2, [&] { ring.template issue_a<0>(ph, 2); });
    sub(0, 3, [&] { ring.template issue_a<1>(ph, 2); });
  }
  const int nk = ph.nk;
  for (int s = 1; s < nk - 2; ++s) {
    wait_vmcnt<CA>();
    step(ph, s + 1, ph, s + 2);
  }
  wait_vmcnt<CA>();
  step(ph, nk - 1, next, 0);
  wait_vmcnt<LAST ? 0 : CA>();
  step(next, 0, next, 1);
  products(1, 0);
  products(1, 1);
}

// ---- epilogue: every wave for itself ----------------------------------------------------------------------------------
// The wave's 64 x 64 patches of NP rounded products, 32 rows at a time, through LDS of its own and back row-wise: f(row, column,
// granules) gets row and column inside the tile and eight values of each product.
constexpr int WIDE_STAGE_LD = 64 + 8;                       // bf16 elements
constexpr int WIDE_STAGE = 32 * WIDE_STAGE_LD * 2;          // bytes of one product's 32 rows
template <int NP, class P, class F>
__device__ __forceinline__ void wide_epilogue(char* smem, P product, F f) {
  using TS = TS_WIDE;
  static_assert(8 * NP * WIDE_STAGE <= WIDE_LDS, "the waves' staging areas lie in the ring");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* area = smem + wave * NP * WIDE_STAGE;
  char* put = area + ((lane & 31) * WIDE_STAGE_LD + 4 * (lane >> 5)) * 2;
  const char* get = area + ((lane >> 3) * WIDE_STAGE_LD + (lane & 7) * 8) * 2;
  const int r0 = (wave / TS::WAVES_N) * TS::WM + (lane >> 3), c0 = (wave % TS::WAVES_N) * TS::WN + (lane & 7) * 8;
#pragma unroll
  for (int tm = 0; tm < TS::TM; ++tm) {
#pragma unroll
    for (int i = 0; i < NP; ++i)
#pragma unroll
      for (int tn = 0; tn < TS::TN; ++tn)
#pragma unroll
        for (int g = 0; g < 4; ++g) *reinterpret_cast<uint2*>(put + i * WIDE_STAGE + (tn * 32 + g * 8) * 2) = product(i, tm, tn, g);
    wave_lds_fence();
    uint4 u[4][NP];
#pragma unroll
    for (int ps = 0; ps < 4; ++ps)
#pragma unroll
      for (int i = 0; i < NP; ++i) u[ps][i] = *reinterpret_cast<const uint4*>(get + i * WIDE_STAGE + ps * 8 * WIDE_STAGE_LD * 2);
    wave_lds_fence();
#pragma unroll
    for (int ps = 0; ps < 4; ++ps) f(r0 + tm * 32 + ps * 8, c0, u[ps]);
  }
}
__device__ __forceinline__ uint2 pack4(const f32x16& v, int g) {
  return make_uint2(pack_bf16(v[4 * g], v[4 * g + 1]), pack_bf16(v[4 * g + 2], v[4 * g + 3]));
}

// The phases X (W0, W2)^T and Y W1 (W1 read K-strided).
__device__ __forceinline__ void wide_x_phase(const HiddenParams& p, int m0, int n0, int z, int wave, WidePhase<2, false>& ph) {
  const long long w = p.steps.at(z, p.bsw, p.gsw) + (long long)n0 * p.d;
  ph.a = reinterpret_cast<const uint16_t*>(p.X) + p.steps.at(z, p.bsx, p.gsx) + (size_t)m0 * p.ldx;
  ph.b[0] = reinterpret_cast<const uint16_t*>(p.W0) + w;
  ph.b[1] = reinterpret_cast<const uint16_t*>(p.W2) + w;
  ph.init(p.ldx, p.T - m0, p.d, p.dh - n0, p.d, wave);
}
__device__ __forceinline__ void wide_y_phase(const HiddenParams& p, int m0, int n0, int z, int wave, WidePhase<1, true>& ph) {
  ph.a = reinterpret_cast<const uint16_t*>(p.Y) + p.steps.at(z, p.bsy, p.gsy) + (size_t)m0 * p.ldy;
  ph.b[0] = reinterpret_cast<const uint16_t*>(p.W1) + p.steps.at(z, p.bsw, p.gsw) + n0;
  ph.init(p.ldy, p.T - m0, p.dh, p.dh - n0, p.d, wave);
}

// Main loop of the three-product kernels: the product with Y first, rounded and packed before the other two need its registers.
__device__ __forceinline__ void wide_three_products(const HiddenParams& p, char* smem, int m0, int n0, int z, uint2 (&y)[TS_WIDE::TM][TS_WIDE::TN][4],
                                                    f32x16 (&x)[2][TS_WIDE::TM][TS_WIDE::TN]) {
  using TS = TS_WIDE;
  WideRing ring;
  ring.init(smem);
  WidePhase<1, true> py;
  wide_y_phase(p, m0, n0, z, ring.wave, py);
  ring.start(py);
  WidePhase<2, false> px;
  wide_x_phase(p, m0, n0, z, ring.wave, px);
  {
    f32x16 ay[1][TS::TM][TS::TN];
    zero_acc<TS>(ay[0]);
    wide_phase<true>(smem, ring, py, px, ay);
#pragma unroll
    for (int tm = 0; tm < TS::TM; ++tm)
#pragma unroll
      for (int tn = 0; tn < TS::TN; ++tn)
#pragma unroll
        for (int g = 0; g < 4; ++g) y[tm][tn][g] = pack4(ay[0][tm][tn], g);
  }
  zero_acc<TS>(x[0]);
  zero_acc<TS>(x[1]);
  wide_phase<false>(smem, ring, px, WideNone(), x);
  __syncthreads();     // the ring becomes the epilogue's staging area
}

__global__ __launch_bounds__(512, 2) void k_update_hidden_wide(const HiddenDmaParams pp) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  prefetch_args<sizeof(pp)>();
  using TS = TS_WIDE;
  const HiddenParams& p = pp.h;
  int bx, by, z;
  if (!pp.map.locate(blockIdx.x, bx, by, z)) return;
  const int m0 = bx * TS::BM, n0 = by * TS::BN;
  uint2 y[TS::TM][TS::TN][4];
  f32x16 x[2][TS::TM][TS::TN];
  wide_three_products(p, smem, m0, n0, z, y, x);
  const bool keep = p.O3 != nullptr;
  wide_epilogue<3>(smem, [&](int i, int tm, int tn, int g) { return i == 2 ? y[tm][tn][g] : pack4(x[i][tm][tn], g); },
    [&](int r, int c, const uint4 (&u)[3]) {
      const int m = m0 + r;
      if (m >= p.T || n0 + c >= p.dh) return;
      const float l0 = p.lr0[z * p.bslr + m], l1 = p.lr1[z * p.bslr + m], l2 = p.lr2[z * p.bslr + m];
      update_pointwise8(p, z * p.bso + (size_t)m * p.dh + n0 + c, keep, u[0], u[1], u[2], l0, l1, l2);
    });
}

__global__ __launch_bounds__(512, 2) void k_apply_bwd_hidden_wide(const HiddenDmaParams pp) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  prefetch_args<sizeof(pp)>();
  using TS = TS_WIDE;
  const HiddenParams& p = pp.h;
  int bx, by, z;
  if (!pp.map.locate(blockIdx.x, bx, by, z)) return;
  const int m0 = bx * TS::BM, n0 = by * TS::BN;
  uint2 y[TS::TM][TS::TN][4];
  f32x16 x[2][TS::TM][TS::TN];
  wide_three_products(p, smem, m0, n0, z, y, x);
  wide_epilogue<3>(smem, [&](int i, int tm, int tn, int g) { return i == 2 ? y[tm][tn][g] : pack4(x[i][tm][tn], g); },
    [&](int r, int c, const uint4 (&u)[3]) {
      if (m0 + r >= p.T || n0 + c >= p.dh) return;
      apply_bwd_pointwise8(p, z * p.bso + (size_t)(m0 + r) * p.dh + n0 + c, u[0], u[1], u[2]);
    });
}

}  // namespace lact
