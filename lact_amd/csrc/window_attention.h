// Causal attention inside a sliding window (query i sees keys i - window + 1 .. i), bf16, head sizes 64 and 128,
// forward and backward: what the causal layer asks of flash_attn_func(causal=True, window_size=(window-1, 0))
// (causal_lact_with_sliding_window_attn.py:371-375).
//
// q, k, v: [B, L, H, D] with strides; a head's D elements are contiguous and heads follow each other.  out: [B, L, H, D]
// contiguous.  lse: [B, H, L] fp32, log2 of the row's sum of exp2(c * q.k), c = log2(e) / sqrt(D).
//
// One wave owns 32 rows (queries in the forward and in dq, keys in dk/dv) and walks the 64-row tiles of the other side
// that its window touches; the tiles travel through a ring of four slots of asynchronous global -> LDS copies shared by
// the block.  Scores are formed with the wave's own rows as matrix columns, so that a lane holds
// one of them and the softmax needs no exchange but where the row's maximum is moved.  The exponentials then feed the next product as
// they lie: a matrix instruction's k slots 0..3 / 4..7 of lane half h stand for rows 4h + i / 8 + 4h + i of its 16,
// on both operands, which costs nothing because the other operand comes from transposing LDS reads of four rows each.
//
// What bounds it: the issue of vector operations.  Beside a matrix instruction (32 clocks) a SIMD issues six of them for nothing;
// the forward needs seven for every instruction that forms scores (a fused multiply-add, an exponential of two issue slots and an
// add per score, half a conversion): 48 clocks measured in a loop of nothing else, with an LDS read.  Left to itself the compiler put
// the products of a tile in front and the vector work behind them, on both waves of a SIMD at once, and the two added up (111 us
// without the softmax, 128 with nothing but it, 226 together).  Hence the forward and dq form the scores of a tile while they
// work on those of the one before, instruction by instruction in a written order (sched_barrier).  dk/dv has no registers for
// that: its two accumulators and its own rows fill 192 of 256, and with half the waves and 512 registers each the vector
// work on accumulators in the second register file and the bare barriers cost more than the order gained (434 us against 394).
//
// Heads of 64 have as much vector work for half the products, and without a second tile's scores (119 and 128 registers instead of 186
// and 180) two blocks of eight waves fit a compute unit, which overlap better than one that forms them ahead: 4 x 24 heads, 4096 tokens, window
// 2048 / 512, forward 197 / 89 us against 214 / 108, dq 241 / 106 against 280 / 139.
//
// Measured at B = 4, L = 4096, window 2048, 12 heads of 128, before / now: forward 205 / 170 us (50 % of the matrix pipes' time), dq 260 / 238
// (54 %), dk and dv 402 / 350.  Of that a tenth is the order of the blocks (locate); the copies of dk/dv are two tiles ahead (three, or
// past the last tile without a branch, cost up to 3 % where a block has few).  Tried: the waves of a SIMD taking turns at the
// matrix pipe behind barriers (forward 208, dq 333); wave priorities that alternate from tile to tile (nothing); torch's masked
// attention over window-sized blocks: 930 and 3400 us, plus building its masks and copying around it.  A single
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
  UDiv by_heads;                     // B * H
  // Blocks of one row tile of every head follow each other, the tiles with the longest windows first.  (Heads one after the other
  // left the last ones' long blocks for the end: at 48 heads of 16 row tiles a CU worked 96 tiles where 81 are its share.)  A
  // head's blocks share a die where there is a multiple of eight heads.
  __device__ __forceinline__ void locate(int& x, int& z) const {
    x = by_heads.div(blockIdx.x);
    z = blockIdx.x - x * (int)by_heads.d;
  }
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

// The copies of the 64-row tiles [0, n) of one operand that wave `wave` of NW issues, NC a tile.
template <int D, int NW>
struct AttnCopy {
  using T = AttnTile<D>;
  static constexpr int NC = T::G / NW;
  static_assert(T::G % NW == 0, "copies must split evenly over the waves");
  uint32_t voff[NC], vlast[NC];   // of the last tile, whose rows past the end of the sequence repeat its last one
  const uint16_t* base;           // the head's first row that the tiles cover
  int step, last;
  __device__ __forceinline__ void init(int wave, const uint16_t* head, int ld, int first, int n, int L) {
    base = uniform(head + (size_t)first * ld);
    step = 64 * ld; last = n - 1;
    const int rows = L - 1 - (first + last * 64);
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = (wave + i * NW) * 64 + (threadIdx.x & 63), row = c / T::G, slot = c % T::G;
      voff[i] = (uint32_t)(row * ld + (slot ^ T::key(row)) * 8) * 2;
      vlast[i] = (uint32_t)(min(row, rows) * ld + (slot ^ T::key(row)) * 8) * 2;
    }
  }
  // Copy i of tile t; past the last tile that one again, so that no branch lies between the matrix instructions around this
  __device__ __forceinline__ void issue(int t, int i, uint32_t lds, int wave) const {
    dma16<false>(base + (long long)min(t, last) * step, t >= last ? vlast[i] : voff[i], lds + (wave + i * NW) * 1024);
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

// What was loaded is there behind this.  The compiler waits where a loaded value is first used; in a loop it waits again in every pass, by the
// counter of all vector-memory operations, and so for the copies just issued that it does not see: a tile then takes as long as they do.
template <int N>
__device__ __forceinline__ void attn_arrived(bf16x8 (&f)[N]) {
#pragma unroll
  for (int s = 0; s < N; ++s) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 u = __builtin_bit_cast(u32x4, f[s]);
    asm volatile("" : "+v"(u));
    f[s] = __builtin_bit_cast(bf16x8, u);
  }
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

// Heads of 128 form scores a tile ahead (forward and dq); of 64, where two blocks of eight waves share a compute unit, tile after tile.
template <int D> constexpr bool attn_ahead() { return D == 128; }
template <int D> constexpr int attn_waves() { return attn_ahead<D>() ? 2 : 4; }     // a SIMD's, forward and dq
constexpr float ATTN_LOG2E = 1.4426950408889634f;
constexpr int ATTN_RING = 4;   // slots of two tiles
template <int D, int NW>
constexpr int attn_lds_bytes(bool stats) {
  constexpr int ring = ATTN_RING * (2 * AttnTile<D>::BYTES), stage = NW * 32 * (D + 8) * 2;
  return cmax(ring + (stats ? ATTN_RING * 512 : 0), stage);
}

// Walks the tiles [0, n) of 64 rows: odd(t) and even(t) are called in turn for t = -1 .. n - 1 (and perhaps n) and issue COPIES of
// a wave's copies each, issue(t, i), spread over their matrix instructions: eight waves that issue all at once behind the barrier wait
// for the address queue, 600 clocks a tile.  The barriers lie in front of every step (EVERY) or of the odd ones; behind one lies there what was
// issued in front of the one before (EVERY) or of itself.
template <int COPIES, bool EVERY, typename Odd, typename Even>
__device__ __forceinline__ void attn_walk(int n, Odd odd, Even even) {
  auto open = [&]() LACT_INLINE_LAMBDA {
    wait_vmcnt<EVERY ? COPIES : 0>();
    __syncthreads();
  };
  for (int t = -1; t < n; t += 2) {
    open();
    odd(t);
    if (EVERY) open();
    even(t + 1);
  }
  wait_vmcnt<0>();
}

// Walks the tiles [0, n) one after the other: issue(t) starts the copies of tile t, COPIES of a wave, two tiles ahead; body(t) uses it.
template <int COPIES, typename Issue, typename Body>
__device__ __forceinline__ void attn_walk_in_order(int n, Issue issue, Body body) {
  issue(0);
  if (n > 1) issue(1);
  for (int t = 0; t < n; ++t) {
    if (t + 1 < n) wait_vmcnt<COPIES>();
    else wait_vmcnt<0>();
    __syncthreads();      // tile t is there for every wave, and all are through with t - 1
    if (t + 2 < n) issue(t + 2);
    body(t);
  }
}

template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? attn_waves<D>() : 1) void k_window_attn_fwd(const WindowAttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using T = AttnTile<D>;
  using Copy = AttnCopy<D, NW>;
  constexpr int STAGE = 2 * T::BYTES;
  prefetch_args<sizeof(p)>();
  int bx, z;
  p.locate(bx, z);
  bx = (p.L - 1) / (32 * NW) - bx;
  const int b = z / p.H, h = z % p.H, L = p.L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int blk0 = bx * 32 * NW, row0 = blk0 + wave * 32, row = row0 + (lane & 31);
  const uint16_t* K = p.k + b * p.bsk + h * D;
  const uint16_t* V = p.v + b * p.bsv + h * D;
  bf16x8 qf[D / 16];
  attn_own_rows<D>(qf, p.q + b * p.bsq + h * D, p.ldq, row, L);
  AttnFrag<D> fr;
  fr.init();
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  const float c = p.scale * ATTN_LOG2E;
  float mc = -1e30f, sum = 0.f;        // running row maximum (times c) and this lane's share of the row sum
  const int first = max(0, blk0 - p.window + 1) / 64 * 64, last = min(L, blk0 + 32 * NW), tiles = (last - first + 63) / 64;
  Copy ck, cv;
  ck.init(wave, K, p.ldk, first, tiles, L);
  cv.init(wave, V, p.ldv, first, tiles, L);
  const uint32_t lds0 = lds_addr(smem);
  const int ta = max(0, row0 - p.window + 1 - first) / 64, tb = (min(row0 + 31, last - 1) - first) / 64 + 1;   // the tiles in the wave's windows
  auto in_reach = [&](int t) { return t >= ta && t < tb; };
  constexpr int COPIES = 2 * Copy::NC;
  // The maximum only has to keep exp2 in range: it follows the row when it is exceeded by more than 2^8.
  auto follow = [&](float mx) LACT_INLINE_LAMBDA {     // of this lane's half of the row
    if (__any(mx > mc + 8.f)) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float nm = fmaxf(mc, mx), f = __builtin_amdgcn_exp2f(mc - nm);
      mc = nm;
      sum *= f;
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) o[i][j] *= f;
    }
  };
  auto mask = [&](int k0, f32x16 (&s)[2]) LACT_INLINE_LAMBDA {
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
  };
  auto larger = [](float a, float b) { return __builtin_amdgcn_fmed3f(a, b, __builtin_inff()); };   // one instruction; fmaxf quiets its operands first
  attn_arrived(qf);
  if constexpr (!attn_ahead<D>()) {
    attn_walk_in_order<COPIES>(tiles,
      [&](int t) LACT_INLINE_LAMBDA {
        const uint32_t slot = lds0 + t % ATTN_RING * STAGE;
#pragma unroll
        for (int i = 0; i < Copy::NC; ++i) {
          ck.issue(t, i, slot, wave);
          cv.issue(t, i, slot + T::BYTES, wave);
        }
      },
      [&](int t) LACT_INLINE_LAMBDA {
        if (!in_reach(t)) return;
        const char* kt = smem + t % ATTN_RING * STAGE;
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
        mask(first + t * 64, s);
        float mx = larger(s[0][0], s[1][0]);
#pragma unroll
        for (int j = 1; j < 16; ++j) mx = larger(mx, larger(s[0][j], s[1][j]));
        follow(mx * c);
        float part[2] = {0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            s[i][j] = __builtin_amdgcn_exp2f(fmaf(s[i][j], c, -mc));
            part[i] += s[i][j];
          }
        sum += part[0] + part[1];
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const bf16x8 pf = attn_pack(s[st >> 1], st & 1);
#pragma unroll
          for (int dt = 0; dt < D / 32; ++dt) o[dt] = mma32(fr.cols(vt, dt, st), pf, o[dt]);
        }
      });
  } else {
    // Step t brings the keys of tile t + 3 and the values of t + 2, which the next two steps do not use yet: one barrier for every two
    auto issue = [&](int t, int i) LACT_INLINE_LAMBDA {
      if (i < Copy::NC) ck.issue(t + 3, i, lds0 + (t + 3) % ATTN_RING * STAGE, wave);
      else cv.issue(t + 2, i - Copy::NC, lds0 + (t + 2) % ATTN_RING * STAGE + T::BYTES, wave);
    };
    // Step t: the exponentials of tile t between the matrix instructions that form the scores of t + 1, then the product with them,
    // the maximum of the new scores between its instructions.
    auto step = [&](int t, f32x16 (&cur)[2], f32x16 (&nxt)[2]) LACT_INLINE_LAMBDA {
      const bool here = in_reach(t), ahead = in_reach(t + 1);
      if (!here) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) issue(t, i);
        if (!ahead) return;
      }
      const char* kt = smem + (t + 1) % ATTN_RING * STAGE;
      const char* vt = smem + t % ATTN_RING * STAGE + T::BYTES;
      bf16x8 vb[4];
      uint32_t pw[16];
      bf16x8 kb[3][2];
      auto keys = [&](int ks) LACT_INLINE_LAMBDA {
#pragma unroll
        for (int i = 0; i < 2; ++i) kb[ks % 3][i] = fr.rows(kt, i, ks);
      };
      constexpr int KS = D / 16;
      keys(0);
      keys(1);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) nxt[i][j] = 0.f;
      if (here) {
#pragma unroll
        for (int i = 0; i < 3; ++i) vb[i] = fr.cols(vt, i % (D / 32), i / (D / 32));
        float part[4] = {0.f, 0.f, 0.f, 0.f};
        // two scores a step and instruction: product and offset, exponential, sum and conversion one step behind each other
        constexpr int PER = 16 / (2 * KS);      // pairs per matrix instruction
        auto soft = [&](int e) LACT_INLINE_LAMBDA {
#pragma unroll
          for (int x = 2 * e; x < 2 * e + 2; ++x)
            if (x < 32) cur[x / 16][x % 16] = fmaf(cur[x / 16][x % 16], c, -mc);
#pragma unroll
          for (int x = 2 * e - 2; x < 2 * e; ++x)
            if (x >= 0 && x < 32) cur[x / 16][x % 16] = __builtin_amdgcn_exp2f(cur[x / 16][x % 16]);
          const int x = 2 * e - 4;
          if (x >= 0) {
            part[(e & 1) * 2] += cur[x / 16][x % 16];
            part[(e & 1) * 2 + 1] += cur[x / 16][x % 16 + 1];
            pw[x / 2] = pack_bf16(cur[x / 16][x % 16], cur[x / 16][x % 16 + 1]);
          }
        };
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + 2 < KS) keys(ks + 2);
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            nxt[i] = mma32(kb[ks % 3][i], qf[ks], nxt[i]);
            if ((ks * 2 + i) % (2 * KS / COPIES) == 1 % (2 * KS / COPIES)) issue(t, (ks * 2 + i) / (2 * KS / COPIES));
#pragma unroll
            for (int e = 0; e < PER; ++e) soft((ks * 2 + i) * PER + e);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        soft(16);
        soft(17);
        sum += (part[0] + part[1]) + (part[2] + part[3]);
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + 2 < KS) keys(ks + 2);
#pragma unroll
          for (int i = 0; i < 2; ++i) nxt[i] = mma32(kb[ks % 3][i], qf[ks], nxt[i]);
        }
      }
      if (ahead) mask(first + (t + 1) * 64, nxt);
      float m4[4] = {nxt[0][0], nxt[1][0], nxt[0][1], nxt[1][1]};
      if (here) {
        constexpr int DT = D / 32, MM = 4 * DT;
#pragma unroll
        for (int e = 0; e < MM; ++e) {
          if (e + 3 < MM) vb[(e + 3) % 4] = fr.cols(vt, (e + 3) % DT, (e + 3) / DT);
          const bf16x8 pf = __builtin_bit_cast(bf16x8, make_uint4(pw[4 * (e / DT)], pw[4 * (e / DT) + 1], pw[4 * (e / DT) + 2], pw[4 * (e / DT) + 3]));
          o[e % DT] = mma32(vb[e % 4], pf, o[e % DT]);
#pragma unroll
          for (int j = e * 16 / MM; j < (e + 1) * 16 / MM; ++j)
            if (j >= 2) { m4[2 * (j & 1)] = larger(m4[2 * (j & 1)], nxt[0][j]); m4[2 * (j & 1) + 1] = larger(m4[2 * (j & 1) + 1], nxt[1][j]); }
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int j = 2; j < 16; ++j) { m4[2 * (j & 1)] = larger(m4[2 * (j & 1)], nxt[0][j]); m4[2 * (j & 1) + 1] = larger(m4[2 * (j & 1) + 1], nxt[1][j]); }
      }
      if (!ahead) return;
      follow(larger(larger(m4[0], m4[1]), larger(m4[2], m4[3])) * c);
    };
    f32x16 s[2][2];
#pragma unroll
    for (int t = -3; t < -1; ++t)
#pragma unroll
      for (int i = 0; i < COPIES; ++i)
        if (t == -2 || i < Copy::NC) issue(t, i);
    attn_walk<COPIES, false>(tiles,
      [&](int t) LACT_INLINE_LAMBDA { step(t, s[1], s[0]); }, [&](int t) LACT_INLINE_LAMBDA { step(t, s[0], s[1]); });
  }
  sum += __shfl_xor(sum, 32, 64);
  if (lane < 32 && row < L) p.lse[(size_t)z * L + row] = mc + __builtin_amdgcn_logf(sum);   // v_log_f32 is base 2
  __syncthreads();
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, o, 1.f / sum, p.out + ((size_t)b * L * p.H + h) * D, (size_t)p.H * D, row0, L);
}

// dq = scale * sum_keys p (dp - delta) k, and delta itself.
template <int D, int NW>
__global__ __launch_bounds__(64 * NW, NW == 8 ? attn_waves<D>() : 1) void k_window_attn_dq(const WindowAttnParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  using T = AttnTile<D>;
  using Copy = AttnCopy<D, NW>;
  constexpr int STAGE = 2 * T::BYTES;
  prefetch_args<sizeof(p)>();
  int bx, z;
  p.locate(bx, z);
  bx = (p.L - 1) / (32 * NW) - bx;
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
  float lse = p.lse[(size_t)z * L + min(row, L - 1)];
  AttnFrag<D> fr;
  fr.init();
  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  const float c = p.scale * ATTN_LOG2E;
  const int first = max(0, blk0 - p.window + 1) / 64 * 64, last = min(L, blk0 + 32 * NW), tiles = (last - first + 63) / 64;
  Copy ck, cv;
  ck.init(wave, K, p.ldk, first, tiles, L);
  cv.init(wave, V, p.ldv, first, tiles, L);
  const uint32_t lds0 = lds_addr(smem);
  const int ua = max(0, row0 - p.window + 1 - first) / 32, ub = (min(row0 + 31, last - 1) - first) / 32 + 1;   // the half tiles in the wave's windows
  auto in_reach = [&](int u) { return u >= ua && u < ub; };
  struct Scores { f32x16 s, dp; };
  constexpr int COPIES = 2 * Copy::NC, HALF = COPIES / 2;
  auto issue = [&](int t, int i) LACT_INLINE_LAMBDA {
    const uint32_t slot = lds0 + t % ATTN_RING * STAGE;
    if (i < Copy::NC) ck.issue(t, i, slot, wave);
    else cv.issue(t, i - Copy::NC, slot + T::BYTES, wave);
  };
  auto mask = [&](int k0, f32x16& s) LACT_INLINE_LAMBDA {
    if (k0 + 31 > row0 || k0 < row0 + 31 - p.window + 1) {
      const int lo = row - p.window - k0 - 4 * (lane >> 5), hi = row - k0 - 4 * (lane >> 5);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int key = 8 * (j / 4) + j % 4;
        s[j] = (key <= hi && key > lo) ? s[j] : -__builtin_inff();
      }
    }
  };
  attn_arrived(qf);
  attn_arrived(gf);
  asm volatile("" : "+v"(lse), "+v"(delta));
  if constexpr (!attn_ahead<D>()) {
    attn_walk_in_order<COPIES>(tiles,
      [&](int t) LACT_INLINE_LAMBDA {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) issue(t, i);
      },
      [&](int t) LACT_INLINE_LAMBDA {
        const char* kt = smem + t % ATTN_RING * STAGE;
        const char* vt = kt + T::BYTES;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (!in_reach(2 * t + i)) continue;
          f32x16 s, dp;
#pragma unroll
          for (int j = 0; j < 16; ++j) s[j] = dp[j] = 0.f;
#pragma unroll
          for (int ks = 0; ks < D / 16; ++ks) {
            s = mma32(fr.rows(kt, i, ks), qf[ks], s);
            dp = mma32(fr.rows(vt, i, ks), gf[ks], dp);
          }
          mask(first + t * 64 + i * 32, s);
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
  } else {
    // Half tile u: its probabilities and their gradients between the matrix instructions that form the two products of u + 1, then the product with them.
    auto step = [&](int u, Scores& cur, Scores& nxt) LACT_INLINE_LAMBDA {
      const bool here = in_reach(u), ahead = in_reach(u + 1);
      const int t = (u + 2) / 2 - 1, part0 = (u & 1) * HALF;    // the half tile's share of its tile's copies
      if (!here) {
#pragma unroll
        for (int i = 0; i < HALF; ++i) issue(t + 3, part0 + i);
        if (!ahead) return;
      }
      const char* kn = smem + (u + 1) / 2 % ATTN_RING * STAGE;
      const int in = (u + 1) & 1, iu = u & 1;
      constexpr int KS = D / 16, DT = D / 32;
      bf16x8 kb[2], vb[2], cb[3];
      kb[0] = fr.rows(kn, in, 0);
      vb[0] = fr.rows(kn + T::BYTES, in, 0);
#pragma unroll
      for (int j = 0; j < 16; ++j) nxt.s[j] = nxt.dp[j] = 0.f;
      uint32_t pw[8];
      constexpr int PER = 16 / (2 * KS);
      auto soft = [&](int j) LACT_INLINE_LAMBDA {     // one score a step: product and offset, exponential, gradient one step behind each other
        if (j < 16) cur.s[j] = fmaf(cur.s[j], c, -lse);
        if (j >= 1 && j < 17) { cur.s[j - 1] = __builtin_amdgcn_exp2f(cur.s[j - 1]); cur.dp[j - 1] -= delta; }
        if (j >= 2 && j < 18) cur.s[j - 2] *= cur.dp[j - 2];
        if (j >= 3 && (j & 1)) pw[(j - 3) / 2] = pack_bf16(cur.s[j - 3], cur.s[j - 2]);
      };
      if (here) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + 1 < KS) { kb[(ks + 1) % 2] = fr.rows(kn, in, ks + 1); vb[(ks + 1) % 2] = fr.rows(kn + T::BYTES, in, ks + 1); }
          nxt.s = mma32(kb[ks % 2], qf[ks], nxt.s);
          if (ks % (KS / HALF) == 0) issue(t + 3, part0 + ks / (KS / HALF));
#pragma unroll
          for (int e = 0; e < PER; ++e) soft(2 * ks * PER + e);
          __builtin_amdgcn_sched_barrier(0);
          nxt.dp = mma32(vb[ks % 2], gf[ks], nxt.dp);
#pragma unroll
          for (int e = 0; e < PER; ++e) soft((2 * ks + 1) * PER + e);
          __builtin_amdgcn_sched_barrier(0);
        }
        const char* kt = smem + u / 2 % ATTN_RING * STAGE;
#pragma unroll
        for (int i = 0; i < 2; ++i) cb[i] = fr.cols(kt, i % DT, 2 * iu + i / DT);
        soft(16);
        soft(17);
#pragma unroll
        for (int e = 0; e < 2 * DT; ++e) {
          if (e + 2 < 2 * DT) cb[(e + 2) % 3] = fr.cols(kt, (e + 2) % DT, 2 * iu + (e + 2) / DT);
          const int st = e / DT;
          const bf16x8 pf = __builtin_bit_cast(bf16x8, make_uint4(pw[4 * st], pw[4 * st + 1], pw[4 * st + 2], pw[4 * st + 3]));
          o[e % DT] = mma32(cb[e % 3], pf, o[e % DT]);
        }
      } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          if (ks + 1 < KS) { kb[(ks + 1) % 2] = fr.rows(kn, in, ks + 1); vb[(ks + 1) % 2] = fr.rows(kn + T::BYTES, in, ks + 1); }
          nxt.s = mma32(kb[ks % 2], qf[ks], nxt.s);
          nxt.dp = mma32(vb[ks % 2], gf[ks], nxt.dp);
        }
      }
      if (ahead) mask(first + (u + 1) * 32, nxt.s);
    };
    Scores sc[2];
    auto tile = [&](int t) LACT_INLINE_LAMBDA {
      step(2 * t, sc[0], sc[1]);
      step(2 * t + 1, sc[1], sc[0]);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < COPIES; ++i) issue(t, i);
    attn_walk<COPIES, true>(tiles, tile, tile);
  }
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
  int bx, z;
  p.locate(bx, z);
  const int b = z / p.H, h = z % p.H, L = p.L;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int blk0 = bx * 32 * NW, row0 = blk0 + wave * 32, row = row0 + (lane & 31);
  const uint16_t* Q = p.q + b * p.bsq + h * D;
  const uint16_t* G = p.dout + b * p.bsdo + h * D;
  bf16x8 kf[D / 16], vf[D / 16];
  attn_own_rows<D>(kf, p.k + b * p.bsk + h * D, p.ldk, row, L);
  attn_own_rows<D>(vf, p.v + b * p.bsv + h * D, p.ldv, row, L);
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
  const char* stats = smem + ATTN_RING * STAGE;         // per ring slot: 64 lse, 64 delta
  // the even waves bring the slot's lse, the odd ones its delta: the same bytes from each, one copy per wave
  const float* st_src = (wave & 1 ? p.delta : p.lse) + (size_t)z * L;
  const int tiles = (last - first + 63) / 64;
  Copy cq, cg;
  cq.init(wave, Q, p.ldq, first, tiles, L);
  cg.init(wave, G, p.lddo, first, tiles, L);
  constexpr int COPIES = 2 * Copy::NC + 1;
  auto issue_all = [&](int t) LACT_INLINE_LAMBDA {
    const uint32_t slot = t % ATTN_RING;
#pragma unroll
    for (int i = 0; i < Copy::NC; ++i) {
      cq.issue(t, i, lds0 + slot * STAGE, wave);
      cg.issue(t, i, lds0 + slot * STAGE + T::BYTES, wave);
    }
    const int q0 = first + t * 64;
    dma4(st_src + q0, (uint32_t)min(lane, L - 1 - q0) * 4, lds0 + ATTN_RING * STAGE + slot * 512 + (wave & 1) * 256);
  };
  auto tile = [&](int t) LACT_INLINE_LAMBDA {
    const int slot = t % ATTN_RING;
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
  };
  attn_arrived(kf);
  attn_arrived(vf);
  attn_walk_in_order<COPIES>(tiles, issue_all, tile);
  __syncthreads();
  const size_t o = ((size_t)b * L * p.H + h) * D;
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, ok, p.scale, p.dk + o, (size_t)p.H * D, row0, L);
  attn_store_rows<D>(smem + wave * 32 * (D + 8) * 2, ov, 1.f, p.dv + o, (size_t)p.H * D, row0, L);
}

}  // namespace lact
