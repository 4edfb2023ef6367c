// What the GEMM kernels share: the shape of a block's output tile, the 32x32 matrix instructions and the walk over a lane's
// accumulators.
//
// MFMA operands are swapped (the B tile is passed as the instruction's first operand), so each lane ends up owning 4
// consecutive n for one m: epilogues store 8- or 16-byte vectors along n.
#pragma once
#include "common.h"

namespace lact {

template <int BM_, int BN_, int WAVES_M_, int WAVES_N_>
struct TileShape {
  static constexpr int BM = BM_, BN = BN_;
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_;
  static constexpr int THREADS = 64 * WAVES_M * WAVES_N;
  static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
  static constexpr int TM = WM / 32, TN = WN / 32;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "wave tile must be a multiple of the 32x32 MFMA tile");
};

constexpr int cmax(int a, int b) { return a > b ? a : b; }

__device__ __forceinline__ f32x16 mma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mma32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <class TS>
__device__ __forceinline__ void zero_acc(f32x16 (&acc)[TS::TM][TS::TN]) {
#pragma unroll
  for (int i = 0; i < TS::TM; ++i)
#pragma unroll
    for (int j = 0; j < TS::TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}

// Epilogue iteration.  Inside the body:  tm, tn, g index the fragment; `m`, `n` are block-local
// coordinates of 4 consecutive n; the values are acc[tm][tn][4*g + j], j = 0..3.
#define LACT_FOR_QUADS(TS)                                                                     \
  _Pragma("unroll") for (int tm = 0; tm < TS::TM; ++tm)                                        \
  _Pragma("unroll") for (int tn = 0; tn < TS::TN; ++tn)                                        \
  _Pragma("unroll") for (int g = 0; g < 4; ++g)

template <class TS> __device__ __forceinline__ int quad_m(int tm) {
  return ((threadIdx.x >> 6) / TS::WAVES_N) * TS::WM + tm * 32 + (threadIdx.x & 31);
}
template <class TS> __device__ __forceinline__ int quad_n(int tn, int g) {
  return ((threadIdx.x >> 6) % TS::WAVES_N) * TS::WN + tn * 32 + 8 * g + 4 * ((threadIdx.x & 63) >> 5);
}

}  // namespace lact
