// Newton-Schulz of small matrices ([r, c], r = 32 .. 128, c <= 256 in steps of 32): one block per matrix, everything in LDS and
// registers.  Per iteration  A = X X^T;  B = b A + (c A) A;  X' = a X + B X  (ttt_operation.py:58-62), preceded by the
// Frobenius normalisation.
//
// X lives in LDS as bf16 (64 KiB at 128 x 256; read row-wise for the Gram matrix and transposed for B X), its fp32 iterate in
// the registers of the waves that own its tiles, A in LDS, c A and then B in one more square.  Eight waves, all of them on
// matrix instructions; five barriers per iteration and no traffic to memory but the input, the result and what a backward pass
// keeps.  Every value is rounded where the separate launches round it and every product runs over k in the same order: the
// same bits.
//
// What bounds it: the chain of the five dependent iterations on one compute unit -- 2.1 us of matrix instructions each at
// 128 x 256, as much again of LDS reads, and the roundings of 64 iterate elements per lane.  Measured at 18 matrices of
// 128 x 256: 40 us against 66-68 us as k_ns_fused (four compute units per matrix, every stage handed over through the L2); at 6
// of 64 x 64: 16 us against 74 us as three launches per iteration.
#pragma once
#include "ns_fused.h"

namespace lact {

struct NsLocalParams {
  int c, S, nb, mask;
  float coeffs[3 * NS_FUSED_MAX_STEPS];
  const uint16_t* g16;                      // [n][r, c] input, bf16
  const float* ss_part; int nparts, part0, part1;   // partial sums of squares (part1 < 0: none), as in k_ns_fused
  float* norms;
  // kept for the backward, each null when there is none: X_k, A_k, B_k per iteration
  uint16_t* xb; long long xb_it_stride;
  uint16_t* ab; uint16_t* bb; long long sq_it_stride;
  float* u_out;                             // [n] result, fp32, original orientation
};

// LDS matrices are [row][GR granules of 16 bytes], granule g of row i at slot g ^ ns_key(i) (low four bits): 16 consecutive rows
// of one granule, and 4 consecutive rows of 4 neighbouring granules, fall into different banks.
__device__ __forceinline__ int ns_key(int i) { return ((i & 3) << 2) | ((i >> 2) & 3); }
template <int GR>
__device__ __forceinline__ char* ns_at(char* m, int row, int g) { return m + (row * GR + (g ^ ns_key(row))) * 16; }
// Fragment addresses.  Tiles start at multiples of 32 rows and columns and a product runs over k in steps of 16, so the keys
// involved depend on the lane only: one xor or nothing per fragment.
template <int GR>
struct NsFrag {
  uint32_t row_off, row_key;     // rows: 32 from row0 over 16 k (granules 2 ks, 2 ks + 1)
  __device__ __forceinline__ NsFrag() {
    const int l = threadIdx.x & 63;
    row_off = (l & 31) * GR * 16;
    row_key = (uint32_t)(ns_key(l & 31) ^ (l >> 5)) << 4;
  }
  __device__ __forceinline__ bf16x8 rows(const char* m, int row0, int ks) const {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(m + row0 * GR * 16 + row_off + ((uint32_t)(ks * 32) ^ row_key)));
  }
};
// 32 columns from col0 over 16 rows (k) from 16 ks
template <int GR>
struct NsColFrag {
  uint32_t off[2];
  __device__ __forceinline__ void init(int col0) {
    const int l = threadIdx.x & 63, k = 8 * (l >> 5) + ((l & 15) >> 2), g = col0 / 8 + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) off[i] = ((k + 4 * i) * GR + (g ^ ns_key(k + 4 * i))) * 16 + (l & 1) * 8;
  }
  __device__ __forceinline__ bf16x8 cols(const char* m, int ks) const {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(m + off[0] + ks * 16 * GR * 16));
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(m + off[1] + ks * 16 * GR * 16));
    const s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(bf16x8, v);
  }
};
// this lane's four consecutive columns 8 q + 4 (lane / 32) of row (lane % 32) of the 32 x 32 tile at (row0, col0)
template <int GR>
__device__ __forceinline__ uint16_t* ns_quad(char* m, int row0, int col0, int q) {
  const int l = threadIdx.x & 63;
  return reinterpret_cast<uint16_t*>(ns_at<GR>(m, row0 + (l & 31), col0 / 8 + q) + (l >> 5) * 8);
}
template <int GR>
__device__ __forceinline__ void ns_copy_out(char* m, int rows, int cols, uint16_t* dst) {
  const int gpr = cols / 8;
#pragma unroll 1
  for (int id = threadIdx.x; id < rows * gpr; id += 512) {
    const int row = id / gpr, g = id % gpr;
    *reinterpret_cast<uint4*>(dst + (size_t)id * 8) = *reinterpret_cast<const uint4*>(ns_at<GR>(m, row, g));
  }
}

template <int RT, int XG>
constexpr int ns_local_lds() { return RT * 32 * (XG + 2 * 16) * 16; }

// RT = r / 32; XG: granules per row of X in LDS (16: c <= 128, 32: c <= 256).  Grid: one block of 512 threads per matrix.
// PLAIN: the reference without autocast, every value a bf16 tensor.
template <int RT, int XG, bool PLAIN>
__global__ __launch_bounds__(512, 2) void k_ns_local(const NsLocalParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int WPR = RT == 3 ? 2 : 8 / RT;                       // waves that share a row of tiles
  constexpr int CX = (XG / 4 + WPR - 1) / WPR, CS = (RT + WPR - 1) / WPR;   // tiles per wave of an [r, c] and of an [r, r] matrix
  char* X = smem;
  char* A = smem + RT * 32 * XG * 16;
  char* P = A + RT * 32 * 16 * 16;                                // c A, then B
  const int z = blockIdx.x, r = RT * 32, c = p.c, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave / WPR, wc = wave % WPR;
  const bool on = wr < RT;                                        // RT = 3 leaves two waves without tiles
  const size_t xo = (size_t)z * r * c, so = (size_t)z * r * r;
  auto x_tile = [&](int i) { return (wc * CX + i) * 32; };        // first column of the wave's i-th tile
  auto s_tile = [&](int i) { return (wc * CS + i) * 32; };
  // a wave's tiles past the matrix repeat its last one in the products (no branch between matrix instructions) and are not stored
  auto x_in = [&](int i) { return min(x_tile(i), c - 32); };
  auto s_in = [&](int i) { return min(s_tile(i), RT * 32 - 32); };
  const NsFrag<XG> fx;
  const NsFrag<16> fs;
  NsColFrag<XG> fc[CX];
#pragma unroll
  for (int i = 0; i < CX; ++i) fc[i].init(x_in(i));

  float ss = 0.f;
  for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part0 + z) * p.nparts + i];
  if (p.part1 >= 0)
    for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part1 + z) * p.nparts + i];
  float n = sqrtf(ss);
  if (PLAIN) n = round_bf16(n);
  if (threadIdx.x == 0) p.norms[z] = n;
  float den = n + 1e-7f;
  if (PLAIN) den = round_bf16(den);
  f32x16 xf[CX];
  if (on) {
#pragma unroll
    for (int i = 0; i < CX; ++i)
      if (x_tile(i) < c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[4];
          Elem<uint16_t>::load4(p.g16 + xo + (size_t)(wr * 32 + (lane & 31)) * c + x_tile(i) + 8 * q + 4 * (lane >> 5), v);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = __fdiv_rn(v[j], den);      // the quotient itself (ttt_operation.py:49), not a product with 1 / den
            if (PLAIN) v[j] = round_bf16(v[j]);
            xf[i][4 * q + j] = v[j];
          }
          Elem<uint16_t>::store4(ns_quad<XG>(X, wr * 32, x_tile(i), q), v[0], v[1], v[2], v[3]);
        }
      }
  }
  __syncthreads();
  if (p.xb) ns_copy_out<XG>(X, r, c, p.xb + xo);

  for (int it = 0; it < p.S; ++it) {
    const float ca = p.coeffs[3 * it], cb = p.coeffs[3 * it + 1], cc = p.coeffs[3 * it + 2];
    const bool last = it + 1 == p.S;
    f32x16 acc[CX > CS ? CX : CS];
    auto clear = [&](int tiles) {
#pragma unroll
      for (int i = 0; i < (CX > CS ? CX : CS); ++i)
        if (i < tiles)
#pragma unroll
          for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    };
    // A = X X^T and c A
    if (on) {
      clear(CS);
#pragma unroll 2
      for (int kq = 0; kq < c / 32; ++kq)
#pragma unroll
        for (int ks = 2 * kq; ks < 2 * kq + 2; ++ks) {
          const bf16x8 fa = fx.rows(X, wr * 32, ks);
#pragma unroll
          for (int i = 0; i < CS; ++i) acc[i] = mma32(fx.rows(X, s_in(i), ks), fa, acc[i]);
        }
#pragma unroll
      for (int i = 0; i < CS; ++i)
        if (s_tile(i) < r)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = round_bf16(acc[i][4 * q + j]);
            Elem<uint16_t>::store4(ns_quad<16>(A, wr * 32, s_tile(i), q), v[0], v[1], v[2], v[3]);
            Elem<uint16_t>::store4(ns_quad<16>(P, wr * 32, s_tile(i), q), cc * v[0], cc * v[1], cc * v[2], cc * v[3]);
          }
    }
    __syncthreads();
    if (p.ab) ns_copy_out<16>(A, r, r, p.ab + it * p.sq_it_stride + so);
    // B = b A + (c A) A
    if (on) {
      clear(CS);
#pragma unroll
      for (int ks = 0; ks < 2 * RT; ++ks) {
        const bf16x8 fa = fs.rows(P, wr * 32, ks);
#pragma unroll
        for (int i = 0; i < CS; ++i) acc[i] = mma32(fs.rows(A, s_in(i), ks), fa, acc[i]);
      }
    }
    __syncthreads();
    if (on)
#pragma unroll
      for (int i = 0; i < CS; ++i)
        if (s_tile(i) < r)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float a[4], v[4];
            Elem<uint16_t>::load4(ns_quad<16>(A, wr * 32, s_tile(i), q), a);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = round_bf16(acc[i][4 * q + j]) + round_bf16(cb * a[j]);
            Elem<uint16_t>::store4(ns_quad<16>(P, wr * 32, s_tile(i), q), v[0], v[1], v[2], v[3]);
          }
    __syncthreads();
    if (p.bb) ns_copy_out<16>(P, r, r, p.bb + it * p.sq_it_stride + so);
    // X' = a X + B X
    if (on) {
      clear(CX);
#pragma unroll
      for (int ks = 0; ks < 2 * RT; ++ks) {
        const bf16x8 fa = fs.rows(P, wr * 32, ks);
#pragma unroll
        for (int i = 0; i < CX; ++i) acc[i] = mma32(fc[i].cols(X, ks), fa, acc[i]);
      }
#pragma unroll
      for (int i = 0; i < CX; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) xf[i][j] = dual_blend(round_bf16(acc[i][j]), __fmul_rn(ca, xf[i][j]), PLAIN);
    }
    if (!last) {
      __syncthreads();
      if (on)
#pragma unroll
        for (int i = 0; i < CX; ++i)
          if (x_tile(i) < c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              Elem<uint16_t>::store4(ns_quad<XG>(X, wr * 32, x_tile(i), q), xf[i][4 * q], xf[i][4 * q + 1], xf[i][4 * q + 2], xf[i][4 * q + 3]);
      __syncthreads();
      if (p.xb) ns_copy_out<XG>(X, r, c, p.xb + (it + 1) * p.xb_it_stride + xo);
    }
  }
  if (!on) return;
  const bool transposed = (p.mask >> (z / p.nb)) & 1;
  const int m = wr * 32 + (lane & 31);
#pragma unroll
  for (int i = 0; i < CX; ++i)
    if (x_tile(i) < c)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int col = x_tile(i) + 8 * q + 4 * (lane >> 5);
        if (transposed) {
#pragma unroll
          for (int j = 0; j < 4; ++j) p.u_out[xo + (size_t)(col + j) * r + m] = xf[i][4 * q + j];
        } else {
          Elem<float>::store4(p.u_out + xo + (size_t)m * c + col, xf[i][4 * q], xf[i][4 * q + 1], xf[i][4 * q + 2], xf[i][4 * q + 3]);
        }
      }
}

}  // namespace lact
