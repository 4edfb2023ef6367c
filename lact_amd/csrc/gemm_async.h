// GEMM pipeline for fp32, and for bf16 shapes whose K is not a whole number of the dedicated-loader engine's K-steps
// (gemm_dma.h): asynchronous global -> LDS copies through a ring, every wave of the block issuing a share of them.
//
// A kernel lists its contractions as phases (acc += A * B^T over K each); the copies of all phases run through one flat
// sequence, so the ring never drains between two accumulators.  One barrier per K-step of 128 bytes.
//
// A stage holds the A tile and the B tile.  K-contiguous operand: [row][128 bytes], the 16-byte granule j of row r at slot
// j ^ ((r >> 1) & 7).  K-strided operand: [k][rows].  bf16: one 32x32x16 instruction per 16 k; K-strided tiles, their granules
// rotated so that the rows of a transposing read fall into different banks, are read with ds_read_b64_tr_b16.  fp32: four 32x32x2
// instructions per eight k; instruction i takes k = i from the lanes of the lower half and k = 4 + i from those of the upper
// half, on both operands, so that a K-contiguous operand costs one ds_read_b128 per four instructions.
//
// What bounds it at the sizes that come here (fp32 heads of 64 to 256 and chunks of some hundred tokens; bf16 heads that are
// no multiple of 16, as 40 or 72): the number of blocks and the latency of a block's first copies, less the matrix rate.  Hence
// small tiles and everything of the first K-steps in flight at once.
#pragma once
#include "gemm_dma.h"

namespace lact {

// 64 x 64 tiles: measured at eight fp32 heads of 128, 512 tokens, against the register-staged loop on 128 x 128 tiles: apply
// hidden stage 35 -> 11 us, update 48 -> 17, update backward 53 -> 32, four-term row GEMM 72 -> 19, token reduction 55 + 5 (its
// partial sums) -> 17.  With one A tile for the B operands that share it and one small piece of code for the copies of all contractions,
// instead of a fully unrolled one for each, whose instructions a launch waited for: update backward 31 -> 24.5, apply hidden 14 -> 9.
// HALF, for launches whose 64 x 64 tiles leave compute units without a block: 64 x 32 tiles, two waves to each 32 x 32 of
// them, which take half of the k of every K-step each and add their halves of the sums at the end: twice the blocks, half the
// serial chain of matrix instructions in each (update backward 24.5 -> 18.9 us, apply hidden 9.0 -> 7.4).
template <typename T, bool HALF = false> struct AsyncTile {
  static_assert(!HALF || sizeof(T) == 4, "half tiles: fp32");
  using TS = TileShape<64, HALF ? 32 : 64, 2, HALF ? 1 : 2>;
  static constexpr int KG = HALF ? 2 : 1, NQ = 4 / KG;     // waves to a 32 x 32 tile; quads of its columns that one of them ends up with
  static constexpr int THREADS = TS::THREADS * KG;
  static constexpr int STAGES = sizeof(T) == 4 ? 4 : 3;
  static constexpr int GROUP = sizeof(T) == 4 ? 8 : 16;    // k of one group of matrix instructions
  static_assert(TS::TM == 1 && TS::TN == 1 && THREADS == 256, "a wave owns one 32 x 32 tile, or half the k of one");
  __device__ static __forceinline__ int place() { return (threadIdx.x >> 6) % (TS::WAVES_M * TS::WAVES_N); }   // of the wave's 32 x 32 tile
  __device__ static __forceinline__ int kgroup() { return KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) / (TS::WAVES_M * TS::WAVES_N); }
  // rows and columns of the accumulators inside the block's tile, as quad_m and quad_n; quad g < NQ is in entries 4g .. 4g + 3
  __device__ static __forceinline__ int m() { return place() / TS::WAVES_N * 32 + (threadIdx.x & 31); }
  __device__ static __forceinline__ int n(int g) { return place() % TS::WAVES_N * 32 + 8 * (g + NQ * kgroup()) + 4 * ((threadIdx.x & 63) >> 5); }
};

template <typename T>
struct AsyncOperand {
  const T* base;       // first row (k = 0) of this block's tile
  int ld, rows, ks;    // rows: valid rows from base on (may exceed the tile); ks: element (r, k) at base[k * ld + r]
};

// The lane's share of one MFMA k group of a 32-row tile: fp32: four k, one per instruction; bf16: the eight of one instruction.
template <typename T> struct AsyncFrag;
template <> struct AsyncFrag<float> {
  float v[4];
  template <int ROWS, bool KS>
  __device__ __forceinline__ void fetch(const char* tile, int row0, int g) {
    const int lane = threadIdx.x & 63, h = lane >> 5, row = row0 + (lane & 31);
    if (KS) {
      const float* t = reinterpret_cast<const float*>(tile) + (8 * g + 4 * h) * ROWS + row;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = t[i * ROWS];
    } else {
      const float4 u = *reinterpret_cast<const float4*>(tile + row * 128 + (((2 * g + h) ^ ((row >> 1) & 7)) << 4));
      v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
    }
  }
  // clears what lies at k >= left of the group
  __device__ __forceinline__ void mask(int left) {
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (4 * h + i >= left) v[i] = 0.f;
  }
};
template <> struct AsyncFrag<uint16_t> {
  bf16x8 v;
  template <int ROWS, bool KS>
  __device__ __forceinline__ void fetch(const char* tile, int row0, int g) {
    const int l = threadIdx.x & 63, h = l >> 5;
    if (KS) {
      constexpr int G = ROWS / 8, RB = ROWS * 2;
      typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      const int r = row0 + 16 * ((l >> 4) & 1) + 4 * (l & 3), k = g * 16 + 8 * h + ((l & 15) >> 2);
      const char* p = tile + k * RB + ((r / 8 + rotation<G>(k)) % G) * 16 + (l & 1) * 8;
      const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
      const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * RB));
      const s16x8 u = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
      v = __builtin_bit_cast(bf16x8, u);
    } else {
      v = dma_fetch(tile, row0 + (l & 31), 2 * g + h);
    }
  }
  __device__ __forceinline__ void mask(int left) {
    const int h = (threadIdx.x & 63) >> 5;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (8 * h + i >= left) v[i] = (__bf16)0.f;
  }
  // granules by which k-row k of a K-strided tile with G granules per row is rotated (the same for k and k + 4)
  template <int G>
  __device__ static __forceinline__ int rotation(int k) { return G >= 16 ? 4 * (k & 3) : 4 * ((k >> 1) & 1); }
};

// NB: B operands that share the A tile of a stage, up to.  PHASES: contractions one after the other; set(i) (the constructor's argument) calls
// phase() with the operands of contraction i when its copies begin, so that only these are held.
template <typename T, int NB, bool HALF = false>
struct AsyncRing {
  using AT = AsyncTile<T, HALF>;
  using TS = typename AT::TS;
  static constexpr int EPG = 16 / sizeof(T), BK = 8 * EPG, WAVES = AT::THREADS / 64;
  static constexpr int A_BYTES = TS::BM * 128, B_BYTES = TS::BN * 128, STAGE = A_BYTES + NB * B_BYTES;
  // Where several B operands share a stage two of them, for three blocks to a compute unit (two with four B operands: a third stage of those
  // would leave one).  us with a third stage of 24 KiB and two blocks, with two and three, at 768 blocks of fp32: update hidden stage at d = dh =
  // 64 33.2 / 27.6, 128 39.9 / 35.4, 384 82.7 / 74.0, apply 35.7 / 31.3, 50.5 / 44.7, 105 / 97, apply backward 56.1 / 55.9, 81 / 74, 166 / 150; at
  // 1024 blocks, whose last round is a third full, 189 / 194, 116 / 110, 183 / 180; bf16 (16 x 1024 tokens, d = 200, dh = 392) update 141 / 125,
  // apply 109 / 97, apply backward 184 / 168.  Half tiles, launched where there are fewer blocks than compute units, have three.
  static constexpr int STAGES = NB == 1 ? AT::STAGES : HALF ? 3 : 2, BYTES = STAGE * STAGES;
  static constexpr int NA = TS::BM / 8 / WAVES, NBC = TS::BN / 8 / WAVES, COPIES = NA + NBC;   // per wave and stage, with one B operand
  static_assert(TS::BM / 8 % WAVES == 0 && TS::BN / 8 % WAVES == 0, "copies must split evenly over the waves");
  static_assert(BYTES <= 160 * 1024, "ring does not fit the 160 KiB LDS");
};
template <typename T, int NB, int PHASES, bool HALF, class SET>
struct AsyncPipe : AsyncRing<T, NB, HALF> {
  using R = AsyncRing<T, NB, HALF>;
  using AT = typename R::AT;
  using TS = typename R::TS;
  using R::EPG; using R::BK; using R::WAVES; using R::A_BYTES; using R::B_BYTES; using R::STAGE; using R::STAGES; using R::NA; using R::NBC; using R::COPIES;
  static constexpr int GROUP = AT::GROUP, KG = AT::KG;

  char* smem;
  SET set;
  int total, issued = 0, used = 0;
  // the contraction that is being copied: operands at the next K-step, elements from one to the next, k left
  int cp = 0, cnb = 0, cleft = 0;
  AsyncOperand<T> a, b;
  const T* bs[NB];
  size_t astep = 0, bstep = 0;
  uint32_t va[NA], vb[NBC];   // this lane's offsets inside a K-step (the B operands' are alike)

  // steps: K-steps of all contractions
  __device__ __forceinline__ AsyncPipe(char* s, int steps, SET f) : smem(s), set(f), total(steps) {
    set(*this, 0);
    for (int i = 0; i < STAGES - 1 && issued < total; ++i) issue();
  }
  __host__ __device__ static constexpr int steps(int k) { return (k + BK - 1) / BK; }
  __device__ __forceinline__ void phase(int k, const T* A, int lda, int a_rows, bool a_ks, int ldb, int b_rows, bool b_ks, int nb) {
    a = AsyncOperand<T>{A, lda, a_rows, a_ks};
    b = AsyncOperand<T>{nullptr, ldb, b_rows, b_ks};
    astep = a_ks ? (size_t)BK * lda : (size_t)BK;
    bstep = b_ks ? (size_t)BK * ldb : (size_t)BK;
    cnb = nb; cleft = k;
    offsets<TS::BM, NA>(a, va);
    offsets<TS::BN, NBC>(b, vb);
  }
  // Rows and k past the operand repeat its last ones: they reach only output rows that are never stored, or are left
  // out of the sum by accumulate().
  template <int ROWS, int N>
  __device__ __forceinline__ void offsets(const AsyncOperand<T>& op, uint32_t (&off)[N]) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int n = (wave + i * WAVES) * 64 + lane;      // granule of the tile
      if (op.ks) {
        constexpr int G = ROWS / EPG;
        const int k = n / G, rot = sizeof(T) == 2 ? AsyncFrag<uint16_t>::rotation<G>(k) : 0, g = (n % G + G - rot) % G;
        off[i] = (uint32_t)(min(k, cleft - 1) * op.ld + min(g * EPG, op.rows - EPG)) * (uint32_t)sizeof(T);
      } else {
        const int row = n / 8, j = (n % 8) ^ ((row >> 1) & 7);
        off[i] = (uint32_t)(min(row, op.rows - 1) * op.ld + min(j * EPG, cleft - EPG)) * (uint32_t)sizeof(T);
      }
    }
  }
  __device__ __forceinline__ void issue() {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds = lds_addr(smem + (issued % STAGES) * STAGE) + wave * 1024;
#pragma unroll
    for (int i = 0; i < NA; ++i) dma16<false>(uniform(a.base), va[i], lds + i * WAVES * 1024);
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (j < cnb) {
#pragma unroll
        for (int i = 0; i < NBC; ++i) dma16<false>(uniform(bs[j]), vb[i], lds + A_BYTES + j * B_BYTES + i * WAVES * 1024);
        bs[j] += bstep;
      }
    a.base += astep;
    ++issued;
    cleft -= BK;
    if (cleft <= 0) {
      if (++cp < PHASES) set(*this, PHASES == 2 ? 1 : cp);   // a constant where it can be: a choice between operands keeps them all in memory
    } else if (cleft < BK) {      // a last K-step that K does not fill
      offsets<TS::BM, NA>(a, va);
      offsets<TS::BN, NBC>(b, vb);
    }
  }
  __device__ static __forceinline__ void mma(f32x16& acc, const AsyncFrag<float>& fb, const AsyncFrag<float>& fa) {
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = mma32(fb.v[k], fa.v[k], acc);
  }
  __device__ static __forceinline__ void mma(f32x16& acc, const AsyncFrag<uint16_t>& fb, const AsyncFrag<uint16_t>& fa) {
    acc = mma32(fb.v, fa.v, acc);
  }
  // The next contraction, over k, its B operands into one accumulator each.
  template <bool A_KS, bool B_KS, class... ACC>
  __device__ __forceinline__ void accumulate(int k, ACC&... acc) {
    static_assert(sizeof...(ACC) <= NB, "as many B operands as the stages hold");
    constexpr int GROUPS = BK / GROUP / KG;       // of a K-step that are this wave's, from first on
    const int place = AT::place(), wm0 = (place / TS::WAVES_N) * TS::WM, wn0 = (place % TS::WAVES_N) * TS::WN, first = AT::kgroup() * GROUPS;
    auto group = [&](const char* st, int g, int left) LACT_INLINE_LAMBDA {
      AsyncFrag<T> fa, fb[sizeof...(ACC)];
      fa.template fetch<TS::BM, A_KS>(st, wm0, g);
#pragma unroll
      for (int j = 0; j < (int)sizeof...(ACC); ++j) fb[j].template fetch<TS::BN, B_KS>(st + A_BYTES + j * B_BYTES, wn0, g);
      if (left < GROUP) {   // both operands: an infinity that one of them repeats there would make the other's zeros NaN
        fa.mask(left);
        // feature sizes come in eights: groups of eight end ragged in contractions over tokens only (masking everywhere costs the
        // fp32 training step of eight heads of 128, 2048 tokens, 2.5 of 478 us)
        if constexpr ((A_KS && B_KS) || GROUP > 8)
#pragma unroll
          for (int j = 0; j < (int)sizeof...(ACC); ++j) fb[j].mask(left);
      }
      int j = 0;
      (mma(acc, fb[j++], fa), ...);
    };
    for (int left = k; left > 0; left -= BK) {
      if (used + STAGES - 2 < total) wait_vmcnt<(STAGES - 2) * COPIES>();
      else wait_vmcnt<0>();
      __syncthreads();
      if (issued < total) issue();
      const char* st = smem + (used % STAGES) * STAGE;
      ++used;
      if (left >= BK) {
#pragma unroll
        for (int g = 0; g < GROUPS; ++g) group(st, first + g, GROUP);
      } else {
        for (int g = first; g < first + GROUPS && g * GROUP < left; ++g) group(st, g, left - g * GROUP);
      }
    }
  }
  // Behind the last contraction: the sums of the waves that share a tile.  Each hands the other two quads of its columns and adds the two it
  // gets to those it keeps, which end in entries 0 .. 7.
  template <class... ACC>
  __device__ __forceinline__ void combine(ACC&... acc) {
    if constexpr (KG == 2) {
      static_assert(sizeof...(ACC) * 2 * AT::THREADS * 16 <= R::BYTES, "the sums are exchanged inside the ring");
      const int kg = AT::kgroup();
      float4* const area = reinterpret_cast<float4*>(smem);
      __syncthreads();                     // the ring is free
      int slot = 0;
      ([&]() LACT_INLINE_LAMBDA {
#pragma unroll
        for (int q = 0; q < 2; ++q, ++slot)
          area[slot * AT::THREADS + threadIdx.x] = kg ? make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3])
                                                      : make_float4(acc[4 * q + 8], acc[4 * q + 9], acc[4 * q + 10], acc[4 * q + 11]);
      }(), ...);
      __syncthreads();
      slot = 0;
      ([&]() LACT_INLINE_LAMBDA {
#pragma unroll
        for (int q = 0; q < 2; ++q, ++slot) {
          const float4 o = area[slot * AT::THREADS + (threadIdx.x ^ TS::THREADS)];
          const float in[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[4 * q + j] = (kg ? acc[4 * q + j + 8] : acc[4 * q + j]) + in[j];
        }
      }(), ...);
    }
  }
};
template <typename T, int NB, int PHASES, bool HALF, class SET>
__device__ __forceinline__ AsyncPipe<T, NB, PHASES, HALF, SET> async_pipe(char* smem, int steps, SET set) {
  return AsyncPipe<T, NB, PHASES, HALF, SET>(smem, steps, set);
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 v;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = 0.f;
  return v;
}

}  // namespace lact
