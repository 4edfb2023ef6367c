// Newton-Schulz of small matrices ([r, c], r = 32 .. 128, c <= 256 in steps of 32): one block per matrix, everything in LDS and
// registers.  Per iteration  A = X X^T;  B = b A + (c A) A;  X' = a X + B X  (ttt_operation.py:58-62), preceded by the
// Frobenius normalisation.
//
// X lives in LDS as bf16 (64 KiB at 128 x 256; read row-wise for the Gram matrix and transposed for B X), its fp32 iterate in
// the registers of the waves that own its tiles, A, c A and B in LDS.  Of the symmetric A a wave forms a tile on the diagonal and
// the one beside it from the same rows, and writes what lies above the diagonal twice.  Eight waves, all of them on matrix
// instructions; four barriers per iteration and no traffic to memory but the input, the result and what a backward pass keeps.  Every
// value is rounded where the separate launches round it and every product runs over k in the same order: the same bits.
//
// What bounds it: the chain of the five dependent iterations on one compute unit.  At 128 x 256 an iteration takes 4.8 us: 1.5 of
// matrix instructions, the reads of their operands from LDS (1.5 us of the unit's rate), and the roundings and stores between the
// barriers, 1.7 us of vector issue of the two waves on a SIMD.  Measured at 18 matrices of 128 x 256: 33 us; all 16 tiles of A, c A
// from LDS for B only, divisions for the normalisation and the products in the compiler's order 40; 66-68 us as k_ns_fused (four
// compute units per matrix, every stage handed over through the L2).  24 of 96 x 96: 20 us against 25; 6 of 64 x 64 14 against 15, and
// 74 as three launches per iteration.  At 96 and 128 rows of more than 128 columns all 256 registers are in use and one or three
// addresses (up to 12 bytes a lane) are stored once and read back once an iteration, outside the products' loops.
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
  UDiv by_granules;                         // c / 8
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
__device__ __forceinline__ uint16_t* ns_quad(char* m, int row0, int col0, int q, int l) {
  return reinterpret_cast<uint16_t*>(ns_at<GR>(m, row0 + (l & 31), col0 / 8 + q) + (l >> 5) * 8);
}
template <int GR, class DIV>
__device__ __forceinline__ void ns_copy_out(char* m, int rows, int cols, DIV by_granules, uint16_t* dst) {
  const int gpr = cols / 8;
#pragma unroll 2
  for (int id = threadIdx.x; id < rows * gpr; id += 512) {
    const int row = by_granules(id), g = id - row * gpr;
    *reinterpret_cast<uint4*>(dst + (size_t)id * 8) = *reinterpret_cast<const uint4*>(ns_at<GR>(m, row, g));
  }
}

template <int GR>
__device__ __forceinline__ uint16_t* ns_element(char* m, int row, int col) { return reinterpret_cast<uint16_t*>(ns_at<GR>(m, row, col / 8)) + col % 8; }
// of two neighbouring lanes' words the lower halves (even lane) or the upper ones (odd lane), the even lane's first
__device__ __forceinline__ uint32_t ns_pair(uint32_t own, int lane) {
  const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)own, 0xb1, 0xf, 0xf, true);      // quad_perm 1 0 3 2
  return __builtin_amdgcn_perm(other, own, lane & 1 ? 0x03020706u : 0x05040100u);
}
template <int RT, int XG>
constexpr int ns_local_lds() { return RT * 32 * (XG + 3 * 16) * 16; }

// RT = r / 32; XG: granules per row of X in LDS (16: c <= 128, 32: c <= 256).  Grid: one block of 512 threads per matrix.
// PLAIN: the reference without autocast, every value a bf16 tensor.
template <int RT, int XG, bool PLAIN>
__global__ __launch_bounds__(512, 2) void k_ns_local(const NsLocalParams p) {
  prefetch_args<sizeof(p)>();
  extern __shared__ __attribute__((aligned(16))) char smem[];
  constexpr int WPR = RT == 3 ? 2 : 8 / RT;                       // waves that share a row of tiles
  constexpr int CX = (XG / 4 + WPR - 1) / WPR, CS = (RT + WPR - 1) / WPR;   // tiles per wave of an [r, c] and of an [r, r] matrix
  char* X = smem;
  char* A = smem + RT * 32 * XG * 16;
  char* P = A + RT * 32 * 16 * 16;                                // c A
  char* B = P + RT * 32 * 16 * 16;
  const int z = blockIdx.x, r = RT * 32, c = p.c, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave / WPR, wc = wave % WPR;
  const bool on = wr < RT;                                        // RT = 3 leaves two waves without tiles
  const size_t xo = (size_t)z * r * c, so = (size_t)z * r * r;
  auto x_tile = [&](int i) { return (wc * CX + i) * 32; };        // first column of the wave's i-th tile
  auto s_tile = [&](int i) { return (wc * CS + i) * 32; };
  // a wave's tiles past the matrix repeat its last one in the products (no branch between matrix instructions) and are not stored
  auto x_in = [&](int i) { return min(x_tile(i), c - 32); };
  auto s_in = [&](int i) { return min(s_tile(i), RT * 32 - 32); };
  // tiles (gi, gi) and (gi, gj) of the Gram matrix, of a fourth row of tiles' waves 4 and 5 the second one only
  const bool diag = wave < RT;
  const int gi = diag ? wave : RT == 4 && wave < 6 ? wave - 4 : -1, gj = diag ? (wave + 1) % RT : gi + 2;
  auto x_row = [&](int id) { return p.by_granules.div(id); };
  auto s_row = [&](int id) { return id / (RT * 4); };
  const NsFrag<XG> fx;
  const NsFrag<16> fs;
  NsColFrag<XG> fc[CX];
#pragma unroll
  for (int i = 0; i < CX; ++i) fc[i].init(x_in(i));

#pragma unroll
  for (int i = 0; i < RT * XG / 16; ++i) {     // (granules of a row past its last one repeat that)
    const int n = wave + 8 * i, id = n * 64 + lane, row = id / XG, slot = id % XG;
    dma16<false>(p.g16 + xo, (uint32_t)(row * c + min(slot ^ ns_key(row), c / 8 - 1) * 8) * 2, lds_addr(X) + n * 1024);
  }
  float ss = 0.f;
  for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part0 + z) * p.nparts + i];
  if (p.part1 >= 0)
    for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part1 + z) * p.nparts + i];
  float n = sqrtf(ss);
  if (PLAIN) n = round_bf16(n);
  if (threadIdx.x == 0) p.norms[z] = n;
  float den = n + 1e-7f;
  if (PLAIN) den = round_bf16(den);
  wait_vmcnt<0>();
  __syncthreads();
  f32x16 xf[CX];
  if (on) {
    uint2 in[CX][4];
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 least = {0x7f80, 0x7f80};
#pragma unroll
    for (int i = 0; i < CX; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        in[i][q] = *reinterpret_cast<const uint2*>(ns_quad<XG>(X, wr * 32, x_in(i), q, lane));
        least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, in[i][q].x & 0x7f807f80u));
        least = __builtin_elementwise_min(least, __builtin_bit_cast(u16x2, in[i][q].y & 0x7f807f80u));
      }
    // The quotient itself (ttt_operation.py:49), not a product with 1 / den: with y the rounded 1 / den and q = v y, q + (v - q den) y
    // rounds to v / den, the two fused multiply-adds exact inside, for all 2^23 significands of den and 128 of v (tried one by one),
    // as long as nothing leaves the normal range.  10 clocks a value; the division is 44.
    const bool normal = den >= 0x1p-100f && den <= 0x1p25f && least[0] >= 0x0d80 && least[1] >= 0x0d80;      // |v| >= 2^-100
    const float y = __fdiv_rn(1.f, den);
    auto divide = [&](auto quotient) {
#pragma unroll
      for (int i = 0; i < CX; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint2 u = in[i][q];
          float v[4] = {bf16_lo(u.x), bf16_hi(u.x), bf16_lo(u.y), bf16_hi(u.y)};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = quotient(v[j]);
            if (PLAIN) v[j] = round_bf16(v[j]);
            xf[i][4 * q + j] = v[j];
          }
          if (x_tile(i) < c) Elem<uint16_t>::store4(ns_quad<XG>(X, wr * 32, x_tile(i), q, lane), v[0], v[1], v[2], v[3]);
        }
    };
    if (__all(normal)) {
      divide([&](float v) {
        const float q = v * y, rest = __builtin_fmaf(-q, den, v);
        return __builtin_fmaf(rest, y, q);
      });
    } else {
      divide([&](float v) { return __fdiv_rn(v, den); });
    }
  }
  __syncthreads();
  if (p.xb) ns_copy_out<XG>(X, r, c, x_row, p.xb + xo);

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
    // A = X X^T: tiles on and above the diagonal, the others are their mirror images.  A wave's two tiles, on the diagonal and beside
    // it, read the same rows.
    if (gi >= 0) {
      f32x16 on_diag, beside;
#pragma unroll
      for (int j = 0; j < 16; ++j) on_diag[j] = beside[j] = 0.f;
      bf16x8 fi[2][2], fj[2][2];
      const int nq = c / 32;
      auto read = [&](int g, int b) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          fi[b][h] = fx.rows(X, gi * 32, 2 * min(g, nq - 1) + h);
          if (RT > 1) fj[b][h] = fx.rows(X, gj * 32, 2 * min(g, nq - 1) + h);
        }
      };
      auto multiply = [&](int b) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (RT < 4 || diag) on_diag = mma32(fi[b][h], fi[b][h], on_diag);
          if (RT > 1) beside = mma32(fj[b][h], fi[b][h], beside);
        }
      };
      // (in this order: left to itself the compiler moves the reads back to their products)
      auto turn = [&](int g, int b) {
        read(g + 1, 1 - b);
        __builtin_amdgcn_sched_barrier(0);
        multiply(b);
        __builtin_amdgcn_sched_barrier(0);
      };
      read(0, 0);
      int g = 0;
      for (; g + 2 <= nq; g += 2) {
        turn(g, 0);
        turn(g + 1, 1);
      }
      if (g < nq) multiply(0);
      auto put = [&](char* m, const f32x16& s, int ti, int tj, bool mirror) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint2 u = make_uint2(pack_bf16(s[4 * q], s[4 * q + 1]), pack_bf16(s[4 * q + 2], s[4 * q + 3]));
          *reinterpret_cast<uint2*>(ns_quad<16>(m, ti * 32, tj * 32, q, lane)) = u;
          if (mirror) {      // lane pairs swap: the even one writes columns 0 and 2 of both rows, the odd one 1 and 3
            const uint32_t e[2] = {ns_pair(u.x, lane), ns_pair(u.y, lane)};
#pragma unroll
            for (int w = 0; w < 2; ++w)
              *reinterpret_cast<uint32_t*>(ns_element<16>(m, tj * 32 + 8 * q + 4 * (lane >> 5) + 2 * w + (lane & 1), ti * 32 + (lane & 30))) = e[w];
          }
        }
      };
      auto both = [&](f32x16& s, int ti, int tj, bool mirror) {
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = round_bf16(s[j]);
        put(A, s, ti, tj, mirror);
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] *= cc;
        put(P, s, ti, tj, mirror);
      };
      if (diag) both(on_diag, gi, gi, false);
      if (RT > 1 && !(RT == 2 && gi == 1)) both(beside, gi, gj, true);
    }
    __syncthreads();
    if (p.ab) ns_copy_out<16>(A, r, r, s_row, p.ab + it * p.sq_it_stride + so);
    // B = b A + (c A) A
    if (on) {
      clear(CS);
      uint2 own[CS][4];
#pragma unroll
      for (int i = 0; i < CS; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) own[i][q] = *reinterpret_cast<const uint2*>(ns_quad<16>(A, wr * 32, s_in(i), q, lane));
      float ba[CS][16];
      bf16x8 fp[2], fa[2][CS];
      auto read = [&](int ks) {
        fp[ks & 1] = fs.rows(P, wr * 32, ks);
#pragma unroll
        for (int i = 0; i < CS; ++i) fa[ks & 1][i] = fs.rows(A, s_in(i), ks);
      };
      read(0);
#pragma unroll
      for (int ks = 0; ks < 2 * RT; ++ks) {
        if (ks + 1 < 2 * RT) read(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CS; ++i) acc[i] = mma32(fa[ks & 1][i], fp[ks & 1], acc[i]);
#pragma unroll
        for (int n = ks * CS * 4 / (2 * RT); n < (ks + 1) * CS * 4 / (2 * RT); ++n) {      // b A of the wave's tiles meanwhile
          const uint2 u = own[n / 4][n % 4];
          const float a[4] = {bf16_lo(u.x), bf16_hi(u.x), bf16_lo(u.y), bf16_hi(u.y)};
#pragma unroll
          for (int j = 0; j < 4; ++j) ba[n / 4][n % 4 * 4 + j] = round_bf16(cb * a[j]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < CS; ++i)
        if (s_tile(i) < r)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = round_bf16(acc[i][4 * q + j]) + ba[i][4 * q + j];
            Elem<uint16_t>::store4(ns_quad<16>(B, wr * 32, s_tile(i), q, lane), v[0], v[1], v[2], v[3]);
          }
    }
    __syncthreads();
    if (p.bb) ns_copy_out<16>(B, r, r, s_row, p.bb + it * p.sq_it_stride + so);
    // X' = a X + B X
    if (on) {
      clear(CX);
      bf16x8 fb[2], fq[2][CX];
      auto read = [&](int ks) {
        fb[ks & 1] = fs.rows(B, wr * 32, ks);
#pragma unroll
        for (int i = 0; i < CX; ++i) fq[ks & 1][i] = fc[i].cols(X, ks);
      };
      read(0);
#pragma unroll
      for (int ks = 0; ks < 2 * RT; ++ks) {
        if (ks + 1 < 2 * RT) read(ks + 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < CX; ++i) acc[i] = mma32(fq[ks & 1][i], fb[ks & 1], acc[i]);
#pragma unroll
        for (int n = ks * CX * 4 / (2 * RT); n < (ks + 1) * CX * 4 / (2 * RT); ++n)      // a X of the wave's tiles meanwhile
#pragma unroll
          for (int j = 0; j < 4; ++j) xf[n / 4][n % 4 * 4 + j] = __fmul_rn(ca, xf[n / 4][n % 4 * 4 + j]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < CX; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) xf[i][j] = dual_blend(round_bf16(acc[i][j]), xf[i][j], PLAIN);
    }
    if (!last) {
      __syncthreads();
      int l = lane;
      asm volatile("" : "+v"(l));
      if (on)
#pragma unroll
        for (int i = 0; i < CX; ++i)
          if (x_tile(i) < c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              Elem<uint16_t>::store4(ns_quad<XG>(X, wr * 32, x_tile(i), q, l), xf[i][4 * q], xf[i][4 * q + 1], xf[i][4 * q + 2], xf[i][4 * q + 3]);
      __syncthreads();
      if (p.xb) ns_copy_out<XG>(X, r, c, x_row, p.xb + (it + 1) * p.xb_it_stride + xo);
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
