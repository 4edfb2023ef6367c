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
// partial sums) -> 17.
template <typename T> struct AsyncTile {
  using TS = TileShape<64, 64, 2, 2>;
  static constexpr int STAGES = sizeof(T) == 4 ? 4 : 3;
  static constexpr int GROUP = sizeof(T) == 4 ? 8 : 16;    // k of one group of matrix instructions
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

template <typename T, int NPH>
struct AsyncPipe {
  using TS = typename AsyncTile<T>::TS;
  static constexpr int STAGES = AsyncTile<T>::STAGES, GROUP = AsyncTile<T>::GROUP;
  static constexpr int EPG = 16 / sizeof(T), BK = 8 * EPG, WAVES = TS::THREADS / 64;
  static constexpr int A_BYTES = TS::BM * 128, B_BYTES = TS::BN * 128, STAGE = A_BYTES + B_BYTES, BYTES = STAGE * STAGES;
  static constexpr int NA = TS::BM / 8 / WAVES, NB = TS::BN / 8 / WAVES, COPIES = NA + NB;   // per wave and stage
  static_assert(TS::BM / 8 % WAVES == 0 && TS::BN / 8 % WAVES == 0, "copies must split evenly over the waves");

  char* smem;
  AsyncOperand<T> a[NPH], b[NPH];
  int K[NPH];
  int total = 0, issued = 0, used = 0, cp = 0, ckt = 0;

  __device__ __forceinline__ AsyncPipe(char* s) : smem(s) {}
  __device__ __forceinline__ void phase(int i, const T* A, int lda, int a_rows, bool a_ks, const T* B, int ldb, int b_rows, bool b_ks, int k) {
    a[i] = AsyncOperand<T>{A, lda, a_rows, a_ks};
    b[i] = AsyncOperand<T>{B, ldb, b_rows, b_ks};
    K[i] = k;
    total += (k + BK - 1) / BK;
  }
  // Rows and k past the operand repeat its last ones: they reach only output rows that are never stored, or are left
  // out of the sum by accumulate().
  template <int ROWS, int N>
  __device__ __forceinline__ void copy(const AsyncOperand<T>& op, int k0, int k_end, uint32_t lds) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int n = (wave + i * WAVES) * 64 + lane;      // granule of the tile
      uint32_t off;
      if (op.ks) {
        constexpr int G = ROWS / EPG;
        const int k = n / G, rot = sizeof(T) == 2 ? AsyncFrag<uint16_t>::rotation<G>(k) : 0, g = (n % G + G - rot) % G;
        off = (uint32_t)(min(k, k_end - 1 - k0) * op.ld + min(g * EPG, op.rows - EPG)) * (uint32_t)sizeof(T);
      } else {
        const int row = n / 8, j = (n % 8) ^ ((row >> 1) & 7);
        off = (uint32_t)(min(row, op.rows - 1) * op.ld + min(j * EPG, k_end - EPG - k0)) * (uint32_t)sizeof(T);
      }
      dma16<false>(op.base + (op.ks ? (size_t)k0 * op.ld : (size_t)k0), off, lds + (wave + i * WAVES) * 1024);
    }
  }
  __device__ __forceinline__ void issue() {
    const uint32_t lds = lds_addr(smem + (issued % STAGES) * STAGE);
    int k = 0;
#pragma unroll
    for (int i = 0; i < NPH; ++i)
      if (i == cp) {
        copy<TS::BM, NA>(a[i], ckt * BK, K[i], lds);
        copy<TS::BN, NB>(b[i], ckt * BK, K[i], lds + A_BYTES);
        k = K[i];
      }
    if (++ckt * BK >= k) {
      ckt = 0;
      ++cp;
    }
    ++issued;
  }
  __device__ __forceinline__ void start() {
    for (int i = 0; i < STAGES - 1 && issued < total; ++i) issue();
  }
  __device__ static __forceinline__ void mma(f32x16& acc, const AsyncFrag<float>& fb, const AsyncFrag<float>& fa) {
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = mma32(fb.v[k], fa.v[k], acc);
  }
  __device__ static __forceinline__ void mma(f32x16& acc, const AsyncFrag<uint16_t>& fb, const AsyncFrag<uint16_t>& fa) {
    acc = mma32(fb.v, fa.v, acc);
  }
  // Phase i into acc; the phases run in their order, each once.
  template <bool A_KS, bool B_KS>
  __device__ __forceinline__ void accumulate(int i, f32x16 (&acc)[TS::TM][TS::TN]) {
    const int wave = threadIdx.x >> 6;
    const int wm0 = (wave / TS::WAVES_N) * TS::WM, wn0 = (wave % TS::WAVES_N) * TS::WN;
    auto group = [&](const char* st, int g, int left) {
      AsyncFrag<T> fa[TS::TM], fb[TS::TN];
#pragma unroll
      for (int m = 0; m < TS::TM; ++m) fa[m].template fetch<TS::BM, A_KS>(st, wm0 + m * 32, g);
#pragma unroll
      for (int n = 0; n < TS::TN; ++n) fb[n].template fetch<TS::BN, B_KS>(st + A_BYTES, wn0 + n * 32, g);
      if (left < GROUP) {   // both operands: an infinity that one of them repeats there would make the other's zeros NaN
#pragma unroll
        for (int m = 0; m < TS::TM; ++m) fa[m].mask(left);
        // feature sizes come in eights: groups of eight end ragged in contractions over tokens only (masking everywhere costs the
        // fp32 training step of eight heads of 128, 2048 tokens, 2.5 of 478 us)
        if constexpr ((A_KS && B_KS) || GROUP > 8)
#pragma unroll
          for (int n = 0; n < TS::TN; ++n) fb[n].mask(left);
      }
#pragma unroll
      for (int m = 0; m < TS::TM; ++m)
#pragma unroll
        for (int n = 0; n < TS::TN; ++n) mma(acc[m][n], fb[n], fa[m]);
    };
    for (int k0 = 0; k0 < K[i]; k0 += BK) {
      if (used + STAGES - 2 < total) wait_vmcnt<(STAGES - 2) * COPIES>();
      else wait_vmcnt<0>();
      __syncthreads();
      if (issued < total) issue();
      const char* st = smem + (used % STAGES) * STAGE;
      ++used;
      if (K[i] - k0 >= BK) {
#pragma unroll
        for (int g = 0; g < BK / GROUP; ++g) group(st, g, GROUP);
      } else {
        for (int g = 0; g * GROUP < K[i] - k0; ++g) group(st, g, K[i] - k0 - g * GROUP);
      }
    }
  }
};

}  // namespace lact
