// Causal attention inside a sliding window (query i sees keys i - window + 1 .. i), bf16, head sizes 64 and 128,
// forward and backward: what the causal layer asks of flash_attn_func(causal=True, window_size=(window-1, 0))
// (causal_lact_with_sliding_window_attn.py:371-375).
//
// q, k, v: [B, L, H, D] with strides; a head's D elements are contiguous and heads follow each other.  out: [B, L, H, D]
// contiguous.  lse: [B, H, L] fp32, log2 of the row's sum of exp2(c * q.k), c = log2(e) / sqrt(D).
//
// One wave owns 32 rows (queries in the forward and in dq, keys in dk/dv) and walks the 64-row tiles of the other side
// that its window touches; the tiles travel through a three-stage ring of asynchronous global -> LDS copies shared by
// the block, one barrier per tile.  Scores are formed with the wave's own rows as matrix columns, so that a lane holds
// one of them and the softmax needs a single exchange with lane ^ 32.  The exponentials then feed the next product as
// they lie: a matrix instruction's k slots 0..3 / 4..7 of lane half h stand for rows 4h + i / 8 + 4h + i of its 16,
// on both operands, which costs nothing because the other operand comes from transposing LDS reads of four rows each.
//
// What bounds it: vector-ALU issue (one exp2, one fma, one add and half a conversion per score against 32 clocks of
// matrix work per 16 scores and lane), which two waves per SIMD overlap with each other's matrix work.  Measured at
// B = 4, L = 4096, window 2048: 12 heads of 128 forward 219 us (707 TFLOP/s), backward 687 us (788 TFLOP/s over its seven
// products); 24 heads of 64 227 and 702 us.  torch's masked attention over window-sized blocks: 0.93 and 3.4 ms at 12 heads
// of 128, plus building its masks and copying around it (the causal layer's training step 9.46 -> 5.41 ms).  A single
// backward pass over the keys with atomic adds into dq would save two of the seven products and is not deterministic.
#pragma once
#include "gemm_dma.h"

namespace lact {

struct WindowAttnParams {
  int B, L, H, window;               // window >= L: plain causal attention
  const uint16_t* q; const uint16_t* k; const uint16_t* v;
  int ldq, ldk, ldv;                 // elements between tokens
  long long bsq, bsk, bsv;           // elements between batch entries
  uint16_t* out;                     // [B, L, H, D]
  float* lse;                        // [B, H, L]
  // backward
  const uint16_t* dout; int lddo; long long bsdo;
  const uint16_t* o;                 // forward output, contiguous
  float* delta;                      // [B, H, L]: sum_d dout * out, written by the dq kernel, read by the dk/dv kernel
  uint16_t* dq; uint16_t* dk; uint16_t* dv;   // [B, L, H, D] contiguous
  float scale;
  TileMap map;                       // row tiles, 1, B * H
};

// 64 x D bf16 tile in LDS, rows unpadded; the 16-byte granule g of row r lies at slot g ^ key(r).  The key lets 16
// consecutive rows of one granule (row fragments) and 4 consecutive rows of 4 neighbouring granules (transposing reads)
// fall into different banks.
template <int D>
struct AttnTile {
  static constexpr int G = D / 8, ROWB = D * 2, BYTES = 64 * ROWB;
  __device__ static __forceinline__ int key(int r) {
    return D == 128 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
  }
};

// The copies of one 64-row tile that wave `wave` of NW issues.
template <int D, int NW>
struct AttnCopy {
  using T = AttnTile<D>;
  static constexpr int NC = T::G / NW;
  static_assert(T::G % NW == 0, "copies must split evenly over the waves");
  uint32_t voff[NC];
  __device__ __forceinline__ uint32_t offset(int i, int wave, int ld, int last_row) const {
    const int n = (wave + i * NW) * 64 + (threadIdx.x & 63), row = n / T::G, slot = n % T::G;
    return (uint32_t)(min(row, last_row) * ld + (slot ^ T::key(row)) * 8) * 2;
  }
  __device__ __forceinline__ void init(int wave, int ld) {
#pragma unroll
    for (int i = 0; i < NC; ++i) voff[i] = offset(i, wave, ld, 63);
  }
  // base: first element of the head's row 0; rows past the end of the sequence repeat its last row
  __device__ __forceinline__ void issue(const uint16_t* base, int ld, int t0, int L, uint32_t lds, int wave) const {
    const uint16_t* b = base + (size_t)t0 * ld;
    if (t0 + 64 <= L) {
#pragma unroll
      for (int i = 0; i < NC; ++i) dma16<false>(b, voff[i], lds + (wave + i * NW) * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < NC; ++i) dma16<false>(b, offset(i, wave, ld, L - 1 - t0), lds + (wave + i * NW) * 1024);
    }
  }
};

// 4 bytes per lane to LDS: lane i lands at lds_base + 4 * i
__device__ __forceinline__ void dma4(const void* sbase, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\t" ::"s"(lds_base), "v"(voff), "s"(sbase) : "memory", "m0");
}

// Fragments of a tile: rows [32 * rt, +32) as matrix rows over 16 of the D columns; or 32 of the D columns as matrix
// rows over 16 tile rows (transposed, k slots permuted as described above).
template <int D>
struct AttnFrag {
  using T = AttnTile<D>;
  uint32_t row_base, row_key;      // row fragments
  uint32_t tr_off[D / 32][2];      // transposing reads
  __device__ __forceinline__ void init() {
    const int l = threadIdx.x & 63, h = l >> 5;
    row_base = (l & 31) * T::ROWB;
    row_key = (uint32_t)(T::key(l & 31) ^ h) << 4;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 4 * h + 8 * i + ((l & 15) >> 2), g = dt * 4 + 2 * ((l >> 4) & 1) + ((l & 3) >> 1);
        tr_off[dt][i] = row * T::ROWB + ((g ^ T::key(row)) << 4) + (l & 1) * 8;
      }
  }
  __device__ __forceinline__ bf16x8 rows(const char* tile, int rt, int ks) const {
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(tile + rt * 32 * T::ROWB + row_base + ((uint32_t)(ks * 32) ^ row_key)));
  }
  // tile rows [16 * st, +16)
  __device__ __forceinline__ bf16x8 cols(const char* tile, int dt, int st) const {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + tr_off[dt][0] + st * 16 * T::ROWB));
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + tr_off[dt][1] + st * 16 * T::ROWB));
    const s16x8 v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(bf16x8, v);
  }
};

// The wave's own 32 rows as matrix columns: lane l holds row l & 31, 8 columns from 8 * (l >> 5) of every 16.
template <int D>
__device__ __forceinline__ void attn_own_rows(bf16x8 (&f)[D / 16], const uint16_t* base, int ld, int row, int L) {
  const uint16_t* p = base + (size_t)min(row, L - 1) * ld + 8 * ((threadIdx.x & 63) >> 5);
#pragma unroll
  for (int s = 0; s < D / 16; ++s) f[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p + s * 16));
}

__device__ __forceinline__ bf16x8 attn_pack(const f32x16& s, int st) {
  uint32_t r[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = pack_bf16(s[8 * st + 2 * i], s[8 * st + 2 * i + 1]);
  return __builtin_bit_cast(bf16x8, make_uint4(r[0], r[1], r[2], r[3]));
}

// A wave's [D][32] accumulator (rows = D, columns = its own rows), times `f`, to 32 rows of a contiguous [B, L, H, D]
// tensor, through 32 x (D + 8) halves of LDS of its own.
template <int D>
__device__ __forceinline__ void attn_store_rows(char* lds, const f32x16 (&acc)[D / 32], float f, uint16_t* out, size_t ld, int row0, int L) {
  constexpr int LD = D + 8;
  const int l = threadIdx.x & 63;
  uint16_t* t = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      Elem<uint16_t>::store4(t + (l & 31) * LD + dt * 32 + 8 * g + 4 * (l >> 5), acc[dt][4 * g] * f, acc[dt][4 * g + 1] * f, acc[dt][4 * g + 2] * f,
                             acc[dt][4 * g + 3] * f);
  wave_lds_fence();
  constexpr int LPR = D / 8;
#pragma unroll
  for (int i = 0; i < 32 * LPR / 64; ++i) {
    const int id = i * 64 + l, r = id / LPR, c = (id % LPR) * 8;
    const uint4 u = *reinterpret_cast<const uint4*>(t + r * LD + c);
    if (row0 + r < L) *reinterpret_cast<uint4*>(out + (size_t)(row0 + r) * ld + c) = u;
  }
  wave_lds_fence();
}

constexpr float ATTN_LOG2E = 1.4426950408889634f;
template <int D, int NW>
constexpr int attn_lds_bytes(bool stats) {
  constexpr int ring = 3 * (2 * AttnTile<D>::BYTES), stage = NW * 32 * (D + 8) * 2;
  return cmax(ring + (stats ? 3 * 512 : 0), stage);
}

// Walks the tiles [0, n) of 64 rows: `issue(t, slot)` starts the copies of tile t into ring slot `slot` (COPIES vector
// memory instructions per wave), `body(t, slot)` uses it.  Every wave of the block takes part in every tile's barrier.
template <int COPIES, typename Issue, typename Body>
__device__ __forceinline__ void attn_walk(int n, Issue issue, Body body) {
  if (n > 0) issue(0, 0);
  if (n > 1) issue(1, 1);
  int slot = 0, fill = 2;
  for (int t = 0; t < n; ++t) {
    if (t + 1 < n) wait_vmcnt<COPIES>();
    else wait_vmcnt<0>();
    __syncthreads();
    if (t + 2 < n) issue(t + 2, fill);
    body(t, slot);
    slot = slot == 2 ? 0 : slot + 1;
    fill = fill == 2 ? 0 : fill + 1;
  }
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 2 : 1) void k_window_attn_fwd(const WindowAttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using T = AttnTile<D>;
  using Copy = AttnCopy<D, NW>;
  constexpr int STAGE = 2 * T::BYTES;
  prefetch_args<sizeof(p)>();
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  bx = p.map.gx - 1 - bx;      // the longest windows first
  const int b = z / p.H, h = z % p.H, L = p.L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int blk0 = bx * 32 * NW, row0 = blk0 + wave * 32, row = row0 + (lane & 31);
  const uint16_t* K = p.k + b * p.bsk + h * D;
  const uint16_t* V = p.v + b * p.bsv + h * D;
  bf16x8 qf[D / 16];
  attn_own_rows<D>(qf, p.q + b * p.bsq + h * D, p.ldq, row, L);
  Copy ck, cv;
  ck.init(wave, p.ldk);
  cv.init(wave, p.ldv);
  AttnFrag<D> fr;
  fr.init();
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  const float c = p.scale * ATTN_LOG2E;
  float mc = -1e30f, sum = 0.f;        // running row maximum (times c) and this lane's share of the row sum
  const int first = max(0, blk0 - p.window + 1) / 64 * 64, last = min(L, blk0 + 32 * NW);
  const uint32_t lds0 = lds_addr(smem);
  attn_walk<2 * Copy::NC>((last - first + 63) / 64,
    [&](int t, int slot) {
      ck.issue(K, p.ldk, first + t * 64, L, lds0 + slot * STAGE, wave);
      cv.issue(V, p.ldv, first + t * 64, L, lds0 + slot * STAGE + T::BYTES, wave);
    },
    [&](int t, int slot) {
      const int k0 = first + t * 64;
      if (k0 > row0 + 31 || k0 + 63 < row0 - p.window + 1) return;     // nothing of this tile in the wave's windows
      const char* kt = smem + slot * STAGE;
      const char* vt = kt + T::BYTES;
      f32x16 s[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) s[i][j] = 0.f;
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i) s[i] = mma32(fr.rows(kt, i, ks), qf[ks], s[i]);
      if (k0 + 63 > row0 || k0 < row0 + 31 - p.window + 1) {
        const int lo = row - p.window - k0 - 4 * (lane >> 5), hi = row - k0 - 4 * (lane >> 5);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int key = i * 32 + 8 * (j / 4) + j % 4;
            s[i][j] = (key <= hi && key > lo) ? s[i][j] : -__builtin_inff();
          }
      }
      float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
      for (int j = 1; j < 16; ++j) mx = fmaxf(mx, fmaxf(s[0][j], s[1][j]));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * c;
      // The maximum only has to keep exp2 in range: it follows the row when it is exceeded by more than 2^8.
      if (__any(mx > mc + 8.f)) {
        const float nm = fmaxf(mc, mx), f = __builtin_amdgcn_exp2f(mc - nm);
        mc = nm;
        sum *= f;
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) o[i][j] *= f;
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          s[i][j] = __builtin_amdgcn_exp2f(fmaf(s[i][j], c, -mc));
          sum += s[i][j];
        }
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const bf16x8 pf = attn_pack(s[st >> 1], st & 1);
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) o[dt] = mma32(fr.cols(vt, dt, st), pf, o[dt]);
      }
    });
  sum += __shfl_xor(sum, 32, 64);
  if (lane < 32 && row < L) p.lse[(size_t)z * L + row] = mc + __builtin_amdgcn_logf(sum);   // v_log_f32 is base 2
  __syncthreads();
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, o, 1.f / sum, p.out + ((size_t)b * L * p.H + h) * D, (size_t)p.H * D, row0, L);
}

// dq = scale * sum_keys p (dp - delta) k, and delta itself.
template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 2 : 1) void k_window_attn_dq(const WindowAttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using T = AttnTile<D>;
  using Copy = AttnCopy<D, NW>;
  constexpr int STAGE = 2 * T::BYTES;
  prefetch_args<sizeof(p)>();
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  bx = p.map.gx - 1 - bx;
  const int b = z / p.H, h = z % p.H, L = p.L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int blk0 = bx * 32 * NW, row0 = blk0 + wave * 32, row = row0 + (lane & 31);
  const uint16_t* K = p.k + b * p.bsk + h * D;
  const uint16_t* V = p.v + b * p.bsv + h * D;
  bf16x8 qf[D / 16], gf[D / 16];
  attn_own_rows<D>(gf, p.dout + b * p.bsdo + h * D, p.lddo, row, L);
  float delta = 0.f;
  {
    bf16x8 of[D / 16];
    attn_own_rows<D>(of, p.o + ((size_t)b * L * p.H + h) * D, p.H * D, row, L);
#pragma unroll
    for (int s = 0; s < D / 16; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) delta += (float)gf[s][i] * (float)of[s][i];
    delta += __shfl_xor(delta, 32, 64);
  }
  if (lane < 32 && row < L) p.delta[(size_t)z * L + row] = delta;
  attn_own_rows<D>(qf, p.q + b * p.bsq + h * D, p.ldq, row, L);
  const float lse = p.lse[(size_t)z * L + min(row, L - 1)];
  Copy ck, cv;
  ck.init(wave, p.ldk);
  cv.init(wave, p.ldv);
  AttnFrag<D> fr;
  fr.init();
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  const float c = p.scale * ATTN_LOG2E;
  const int first = max(0, blk0 - p.window + 1) / 64 * 64, last = min(L, blk0 + 32 * NW);
  const uint32_t lds0 = lds_addr(smem);
  attn_walk<2 * Copy::NC>((last - first + 63) / 64,
    [&](int t, int slot) {
      ck.issue(K, p.ldk, first + t * 64, L, lds0 + slot * STAGE, wave);
      cv.issue(V, p.ldv, first + t * 64, L, lds0 + slot * STAGE + T::BYTES, wave);
    },
    [&](int t, int slot) {
      const char* kt = smem + slot * STAGE;
      const char* vt = kt + T::BYTES;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int k0 = first + t * 64 + i * 32;
        if (k0 > row0 + 31 || k0 + 31 < row0 - p.window + 1) continue;
        f32x16 s, dp;
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = dp[j] = 0.f;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
          s = mma32(fr.rows(kt, i, ks), qf[ks], s);
          dp = mma32(fr.rows(vt, i, ks), gf[ks], dp);
        }
        if (k0 + 31 > row0 || k0 < row0 + 31 - p.window + 1) {
          const int lo = row - p.window - k0 - 4 * (lane >> 5), hi = row - k0 - 4 * (lane >> 5);
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int key = 8 * (j / 4) + j % 4;
            s[j] = (key <= hi && key > lo) ? s[j] : -__builtin_inff();
          }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = __builtin_amdgcn_exp2f(fmaf(s[j], c, -lse)) * (dp[j] - delta);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 pf = attn_pack(s, st);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) o[dt] = mma32(fr.cols(kt, dt, 2 * i + st), pf, o[dt]);
        }
      }
    });
  __syncthreads();
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, o, p.scale, p.dq + ((size_t)b * L * p.H + h) * D, (size_t)p.H * D, row0, L);
}

// dv = sum_queries p dout, dk = scale * sum_queries p (dp - delta) q: a wave owns 32 keys and walks the queries that see them.
template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 2 : 1) void k_window_attn_dkv(const WindowAttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using T = AttnTile<D>;
  using Copy = AttnCopy<D, NW>;
  constexpr int STAGE = 2 * T::BYTES;
  prefetch_args<sizeof(p)>();
  int bx, by, z;
  if (!p.map.locate(blockIdx.x, bx, by, z)) return;
  const int b = z / p.H, h = z % p.H, L = p.L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int blk0 = bx * 32 * NW, row0 = blk0 + wave * 32, row = row0 + (lane & 31);
  const uint16_t* Q = p.q + b * p.bsq + h * D;
  const uint16_t* G = p.dout + b * p.bsdo + h * D;
  bf16x8 kf[D / 16], vf[D / 16];
  attn_own_rows<D>(kf, p.k + b * p.bsk + h * D, p.ldk, row, L);
  attn_own_rows<D>(vf, p.v + b * p.bsv + h * D, p.ldv, row, L);
  Copy cq, cg;
  cq.init(wave, p.ldq);
  cg.init(wave, p.lddo);
  AttnFrag<D> fr;
  fr.init();
  f32x16 ok[D / 32], ov[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) ok[i][j] = ov[i][j] = 0.f;
  const float c = p.scale * ATTN_LOG2E;
  const int first = blk0 / 64 * 64;
  const int last = p.window >= L ? L : min(L, blk0 + 32 * NW - 1 + p.window);     // one past the last query that sees a key here
  const uint32_t lds0 = lds_addr(smem);
  const char* stats = smem + 3 * STAGE;         // per ring slot: 64 lse, 64 delta
  // the even waves bring the slot's lse, the odd ones its delta: the same bytes from each, one copy per wave
  const float* st_src = (wave & 1 ? p.delta : p.lse) + (size_t)z * L;
  attn_walk<2 * Copy::NC + 1>((last - first + 63) / 64,
    [&](int t, int slot) {
      const int q0 = first + t * 64;
      cq.issue(Q, p.ldq, q0, L, lds0 + slot * STAGE, wave);
      cg.issue(G, p.lddo, q0, L, lds0 + slot * STAGE + T::BYTES, wave);
      dma4(st_src + q0, (uint32_t)min(lane, L - 1 - q0) * 4, lds0 + 3 * STAGE + slot * 512 + (wave & 1) * 256);
    },
    [&](int t, int slot) {
      const char* qt = smem + slot * STAGE;
      const char* gt = qt + T::BYTES;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int q0 = first + t * 64 + i * 32;
        if (q0 + 31 < row0 || q0 - p.window + 1 > row0 + 31 || q0 >= L) continue;
        f32x16 s, dp;
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = dp[j] = 0.f;
#pragma unroll
        for (int ks = 0; ks < D / 16; ++ks) {
          s = mma32(fr.rows(qt, i, ks), kf[ks], s);
          dp = mma32(fr.rows(gt, i, ks), vf[ks], dp);
        }
        const float* ls = reinterpret_cast<const float*>(stats + slot * 512) + i * 32 + 4 * (lane >> 5);
        if (q0 < row0 + 31 || q0 + 31 - p.window + 1 > row0 || q0 + 32 > L) {
          // query q0 + qi sees key `row` when row <= q0 + qi < row + window
          const int lo = row - q0 - 4 * (lane >> 5), hi = min(row + (p.window >= L ? L : p.window), L) - q0 - 4 * (lane >> 5);
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const int qi = 8 * (j / 4) + j % 4;
            s[j] = (qi >= lo && qi < hi) ? s[j] : -__builtin_inff();
          }
        }
        f32x16 ds;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 l4 = *reinterpret_cast<const float4*>(ls + 8 * g), d4 = *reinterpret_cast<const float4*>(ls + 64 + 8 * g);
          const float lv[4] = {l4.x, l4.y, l4.z, l4.w}, dv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            s[4 * g + j] = __builtin_amdgcn_exp2f(fmaf(s[4 * g + j], c, -lv[j]));
            ds[4 * g + j] = s[4 * g + j] * (dp[4 * g + j] - dv[j]);
          }
        }
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const bf16x8 pf = attn_pack(s, st), df = attn_pack(ds, st);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) {
            ov[dt] = mma32(fr.cols(gt, dt, 2 * i + st), pf, ov[dt]);
            ok[dt] = mma32(fr.cols(qt, dt, 2 * i + st), df, ok[dt]);
          }
        }
      }
    });
  __syncthreads();
  const size_t o = ((size_t)b * L * p.H + h) * D;
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, ok, p.scale, p.dk + o, (size_t)p.H * D, row0, L);
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, ov, 1.f, p.dv + o, (size_t)p.H * D, row0, L);
}

}  // namespace lact
