// Pre- and post-processing of the layer classes around the TTT operation, one pass over the data each:
//
//   pre :  qkv [B, L, 3, H, hd]  ->  q, k, v [(B H), L, hd]     silu, per-head L2 norm of q and k, head layout
//          (bidirectional_lact_layer.py:231-244, causal_lact_with_sliding_window_attn.py:313-322)
//          and, for the causal layer, the attention's q and k (rescaled per channel) and v in token layout
//   lr  :  raw [B, L, H, 3] -> lr0, lr1, lr2 [(B H), L]          softplus(raw + inverse-softplus(base lr))
//          momentum raw [B, L, H] -> [(B H), L]                  sigmoid
//          (bidirectional_lact_layer.py:248-256, causal_...:326-345)
//   post:  o [(B H), L, hd] -> y [B, L, H*hd]                    per-head RMSNorm (affine), optional silu gate per
//          token and head, head layout, optionally plus the attention branch  (bidirectional_lact_layer.py:268-270, causal_...:351-357)
//
// and their backward passes.  A group of lanes of a wave per (token, head) row of hd elements.
// Element type T = uint16_t (bf16) or float; all statistics in fp32.
#pragma once
#include "common.h"

namespace lact {

struct LayerGeom {
  int B, L, H, hd;
  __device__ __forceinline__ long long rows() const { return (long long)B * L * H; }
};

__device__ __forceinline__ float silu_f(float x) { return x * sigmoidf_(x); }
__device__ __forceinline__ float silu_grad_f(float x) {
  const float s = sigmoidf_(x);
  return s * (1.f + x * (1.f - s));
}

constexpr int LAYER_HD_MAX = 1024;   // 64 lanes, 4 chunks of 4 elements each

// How a wave's lanes share rows of hd elements: G lanes per row (64 / G rows a wave), NV chunks of 4 * G elements each, so that
// hd fills them: 96 = 8 lanes x 3 chunks, 384 = 32 x 3.  With all 64 lanes on one row 24 of them worked at hd = 96, three
// quarters of the chunks at 384.
template <int G, int NV>
struct RowLanes {
  static constexpr int ROWS = 64 / G;
  __device__ static __forceinline__ int group() { return (threadIdx.x & 63) / G; }
  __device__ static __forceinline__ int col(int i) { return (threadIdx.x & (G - 1)) * 4 + i * 4 * G; }
  // Sum over the row of f(i, j), in the order of one lane per four elements of every 256: per such lane over its chunks, then
  // over the lanes by halves.  The same bits for every split, which Newton-Schulz behind the L2 norms would amplify.
  template <class F>
  __device__ static __forceinline__ float sum(F f) {
    float part[ROWS];
#pragma unroll
    for (int m = 0; m < ROWS; ++m) part[m] = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) part[i % ROWS] = f(i, j, part[i % ROWS]);
#pragma unroll
    for (int d = ROWS / 2; d > 0; d /= 2)
#pragma unroll
      for (int m = 0; m < d; ++m) part[m] += part[m + d];
    float v = part[0];
#pragma unroll
    for (int o = G / 2; o > 0; o /= 2) v += __shfl_xor(v, o, 64);
    return v;
  }
};

// ---- pre ------------------------------------------------------------------------------------------
struct LayerPreParams {
  LayerGeom g;
  int l2norm;                 // L2-normalise q and k
  const void* qkv;            // [B, L, 3, H, hd]
  void* out[3];               // q, k, v  [(B H), L, hd]
  // ATT: what the causal layer's attention reads of the same projection, [B, L, H * hd] each: q and k rescaled per channel
  // (x * qk_scale + qk_offset), v as it is
  void* att[3];
  const float* qk_scale;      // [H * hd][2] (q, k), as is qk_offset
  const float* qk_offset;
  int round_product;          // the rescaling parameters have type T: so has the product in front of the sum
  // backward
  const void* dout[3];
  const void* datt[3];
  void* dqkv;
  float* part;                // ATT: [gridDim.x / H][4][H * hd] partial sums of the gradients of scale q, offset q, scale k, offset k
  int tokens_per_pass;        // tokens between two of a wave
};

// Grid: H * m blocks of 256 threads; a wave handles q, k and v of one head and 64 / G tokens at a time.
// HBM and vector-ALU issue bound it alike: one read of qkv and of the gradients, one write of every output; all loads of a token
// are issued before the first of them is used (the norms otherwise put three round trips in line).  The attention's inputs ride
// along because the projection's output is in registers here: as tensor operations of their own (slices, rescaling, and in the
// backward three zero-padded slice gradients to add up) they took 0.9 ms of a training step at 16384 tokens of 1536 channels.
// Waves in flight decide (layer_pre_waves): operands stay packed until they are used, and the backward keeps the rescaling in LDS and asks
// for v's when q is done.  bf16, us forward / backward, and unpacked, with three and two waves a SIMD instead of four and three: 16384
// tokens, 4 heads of 384 (ATT) 77 / 121 (134 / 172: 450 and 600 MB); 7500 tokens, 8 heads of 96 15.5 / 24.7 (17 / 31: 69 and 104 MB).
template <typename T, bool BWD, bool ATT, int NV> constexpr int layer_pre_waves() { return NV > 3 || std::is_same<T, float>::value ? 1 : BWD && ATT ? 3 : 4; }
template <typename T, bool BWD, bool ATT, int G, int NV>
__global__ __launch_bounds__(256, (layer_pre_waves<T, BWD, ATT, NV>())) void k_layer_pre(const LayerPreParams p) {
  prefetch_args<sizeof(p)>();
  using RL = RowLanes<G, NV>;
  const int wave = threadIdx.x >> 6, grp = RL::group();
  const int hd = p.g.hd, h = blockIdx.x % p.g.H;
  const size_t dim = (size_t)p.g.H * hd;
  float sc[2][NV][4], off[2][NV][4];           // ATT: this lane's channels of the rescaling; backward: in LDS, [q, k][channels of a row]
  __shared__ __attribute__((aligned(16))) float scl[BWD && ATT ? 2 * NV * 4 * G : 1];
  float acc[4][NV][4];                         // ATT && BWD: this lane's share of the parameter gradients
  if (ATT) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = min(RL::col(i), hd - 4);
      if (BWD) {
        if (threadIdx.x < G)
          for (int j = 0; j < 4; ++j)
            for (int a = 0; a < 2; ++a) scl[a * NV * 4 * G + RL::col(i) + j] = p.qk_scale[((size_t)h * hd + c + j) * 2 + a];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[a][i][j] = 0.f;
        continue;
      }
      const float* ps = p.qk_scale + ((size_t)h * hd + c) * 2;
      const float4 s0 = *reinterpret_cast<const float4*>(ps), s1 = *reinterpret_cast<const float4*>(ps + 4);
      sc[0][i][0] = s0.x; sc[1][i][0] = s0.y; sc[0][i][1] = s0.z; sc[1][i][1] = s0.w;
      sc[0][i][2] = s1.x; sc[1][i][2] = s1.y; sc[0][i][3] = s1.z; sc[1][i][3] = s1.w;
      const float* po = p.qk_offset + ((size_t)h * hd + c) * 2;
      const float4 o0 = *reinterpret_cast<const float4*>(po), o1 = *reinterpret_cast<const float4*>(po + 4);
      off[0][i][0] = o0.x; off[1][i][0] = o0.y; off[0][i][1] = o0.z; off[1][i][1] = o0.w;
      off[0][i][2] = o1.x; off[1][i][2] = o1.y; off[0][i][3] = o1.z; off[1][i][3] = o1.w;
    }
    if (BWD) __syncthreads();
  }
  for (long long bl = ((long long)(blockIdx.x / p.g.H) * 4 + wave) * RL::ROWS + grp; bl < (long long)p.g.B * p.g.L; bl += p.tokens_per_pass) {
    const int l = (int)(bl % p.g.L);
    const long long b = bl / p.g.L;
    const size_t oi = ((size_t)(b * p.g.H + h) * p.g.L + l) * hd, ai = (size_t)bl * dim + (size_t)h * hd;
    using Raw = typename Elem<T>::Raw4;
    Raw xs[3][NV], gs[3][NV], as[3][NV];       // unpacked where they are used: half the registers
    auto load = [&](int which) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = RL::col(i);
        xs[which][i] = gs[which][i] = as[which][i] = Raw{};
        if (c < hd) {
          xs[which][i] = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(p.qkv) + ((size_t)(bl * 3 + which) * p.g.H + h) * hd + c);
          if (BWD) gs[which][i] = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(p.dout[which]) + oi + c);
          if (BWD && ATT) as[which][i] = *reinterpret_cast<const Raw*>(reinterpret_cast<const T*>(p.datt[which]) + ai + c);
        }
      }
    };
    constexpr int FIRST = BWD && ATT ? 2 : 3;  // (the third's registers are those of the first)
#pragma unroll
    for (int which = 0; which < FIRST; ++which) load(which);
#pragma unroll
    for (int which = 0; which < 3; ++which) {
      const bool norm = p.l2norm && which < 2;
      float x[NV][4], g[NV][4], y[NV][4];
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        Elem<T>::unpack4(xs[which][i], x[i]);
        if (BWD) Elem<T>::unpack4(gs[which][i], g[i]);
      }
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) y[i][j] = Elem<T>::rnd(silu_f(x[i][j]));       // silu output is a tensor of type T in the reference
      float n = 0.f;
      if (norm) n = sqrtf(RL::sum([&](int i, int j, float s) { return s + y[i][j] * y[i][j]; }));
      const float inv = norm ? 1.f / (n + 1e-5f) : 1.f;
      float c1 = 0.f;
      if (BWD && norm) {
        // z = y / (n + eps):  dy = dz / (n + eps) - y <dz, y> / (n (n + eps)^2);  dx = dy silu'(x)
        const float dot = RL::sum([&](int i, int j, float s) { return s + g[i][j] * y[i][j]; });
        c1 = n > 0.f ? dot / (n * (n + 1e-5f) * (n + 1e-5f)) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = RL::col(i);
        if (c >= hd) continue;
        if (!BWD) {
          Elem<T>::store4(reinterpret_cast<T*>(p.out[which]) + oi + c, y[i][0] * inv, y[i][1] * inv, y[i][2] * inv, y[i][3] * inv);
          if (ATT) {
            float a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              a[j] = x[i][j];
              if (which < 2) {
                a[j] = __fmul_rn(a[j], sc[which & 1][i][j]);
                if (p.round_product) a[j] = Elem<T>::rnd(a[j]);
                a[j] = __fadd_rn(a[j], off[which & 1][i][j]);
              }
            }
            Elem<T>::store4(reinterpret_cast<T*>(p.att[which]) + ai + c, a[0], a[1], a[2], a[3]);
          }
        } else {
          float o[4], at[4], s[4];
          if (ATT) {
            Elem<T>::unpack4(as[which][i], at);
            if (which < 2) {
              const float4 t = *reinterpret_cast<const float4*>(&scl[which * NV * 4 * G + c]);
              s[0] = t.x; s[1] = t.y; s[2] = t.z; s[3] = t.w;
            }
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            o[j] = (g[i][j] * inv - y[i][j] * c1) * silu_grad_f(x[i][j]);
            if (ATT) {
              const float a = at[j];
              if (which < 2) {
                acc[2 * (which & 1)][i][j] += a * x[i][j];
                acc[2 * (which & 1) + 1][i][j] += a;
                o[j] += a * s[j];
              } else {
                o[j] += a;
              }
            }
          }
          Elem<T>::store4(reinterpret_cast<T*>(p.dqkv) + ((size_t)(bl * 3 + which) * p.g.H + h) * hd + c, o[0], o[1], o[2], o[3]);
        }
      }
      if (FIRST < 3 && which == 0) load(2);
    }
  }
  if (ATT && BWD) {      // the shares of the wave's rows, then the four waves', in a fixed order
    __shared__ float red[4][NV * 4 * G];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int o = G; o < 64; o *= 2) acc[a][i][j] += __shfl_xor(acc[a][i][j], o, 64);
    for (int w = 0; w < 4; ++w) {
      if (wave == w && grp == 0) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              float* r = &red[a][RL::col(i) + j];
              *r = w == 0 ? acc[a][i][j] : *r + acc[a][i][j];
            }
      }
      __syncthreads();
    }
    for (int a = 0; a < 4; ++a)
      for (int c = threadIdx.x; c < hd; c += 256) p.part[((size_t)(blockIdx.x / p.g.H) * 4 + a) * dim + (size_t)h * hd + c] = red[a][c];
  }
}

// Sums the partial rows of k_layer_pre's parameter gradients into dscale, doffset [dim][2].  Grid ceil(dim / 64) x 4 blocks
// of 256 threads: 64 columns, four groups of rows.
__global__ __launch_bounds__(256) void k_layer_qk_reduce(const float* part, int rows, int dim, float* dscale, float* doffset) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), a = blockIdx.y, grp = threadIdx.x >> 6;
  float s = 0.f;
  if (c < dim)
#pragma unroll 8
    for (int r = grp; r < rows; r += 4) s += part[((size_t)r * 4 + a) * dim + c];
  red[grp][threadIdx.x & 63] = s;
  __syncthreads();
  if (grp == 0 && c < dim) {
    const int i = threadIdx.x & 63;
    (a & 1 ? doffset : dscale)[(size_t)c * 2 + a / 2] = red[0][i] + red[1][i] + red[2][i] + red[3][i];
  }
}

// ---- learning rates and momentum ------------------------------------------------------------------
struct LayerLrParams {
  LayerGeom g;
  float base_lr_inv;
  const float* lr_raw;        // [B, L, H, 3], or [B, L, 3, H] when rates_major
  int rates_major;
  float* lr[3];               // [(B H), L]
  const float* mom_raw;       // [B, L, H] or null
  float* mom;                 // [(B H), L]
  // backward
  const float* dlr[3]; const float* dmom;
  float* dlr_raw; float* dmom_raw;
};
template <bool BWD>
__global__ void k_layer_lr(const LayerLrParams p) {
  prefetch_args<sizeof(p)>();
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;   // over (b, l, h)
  if (i >= p.g.rows()) return;
  const int h = (int)(i % p.g.H);
  const long long bl = i / p.g.H;
  const int l = (int)(bl % p.g.L);
  const long long b = bl / p.g.L;
  const size_t o = (size_t)(b * p.g.H + h) * p.g.L + l;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const long long ri = p.rates_major ? (bl * 3 + s) * p.g.H + h : i * 3 + s;
    const float x = p.lr_raw[ri] + p.base_lr_inv;
    if (!BWD) p.lr[s][o] = x > 20.f ? x : log1pf(__expf(x));          // softplus (threshold as in torch)
    else p.dlr_raw[ri] = p.dlr[s] ? p.dlr[s][o] * (x > 20.f ? 1.f : sigmoidf_(x)) : 0.f;
  }
  if (p.mom_raw) {
    const float s = sigmoidf_(p.mom_raw[i]);
    if (!BWD) p.mom[o] = s;
    else p.dmom_raw[i] = p.dmom ? p.dmom[o] * s * (1.f - s) : 0.f;
  }
}

// ---- post -----------------------------------------------------------------------------------------
struct LayerPostParams {
  LayerGeom g;
  float eps;
  int use_norm;
  const void* o;              // [(B H), L, hd]
  const float* w;             // [hd] RMSNorm weight (null = ones)
  const void* gate_raw;       // [B, L, H] type T, or null: y *= silu(gate_raw)
  const void* add;            // [B, L, H*hd] type T, or null: y += add (the layer's attention branch)
  void* y;                    // [B, L, H*hd]
  // backward
  const void* dy; void* d_o; void* dgate_raw;
  float* dw_part;             // [gridDim.x][hd] partial sums of the weight gradient, or null
};
// Backward: each wave walks rows row0, row0 + stride, ... so that its partial weight gradient stays in registers.
// HBM bound.  bf16, us forward / backward, with all 64 lanes and four chunks on a row before: 16384 tokens, 4 heads of 384 31 / 45
// (53 / 71: 150 MB each; the forward with one row a wave and its gate asked for behind the sum 43); 7500 tokens, 8 heads of 96 8.7 / 13 (22 / 36).
template <typename T, bool BWD, int G, int NV>
__global__ __launch_bounds__(256, (NV > 3 || std::is_same<T, float>::value ? 1 : 4)) void k_layer_post(const LayerPostParams p) {
  prefetch_args<sizeof(p)>();
  using RL = RowLanes<G, NV>;
  const int wave = threadIdx.x >> 6, grp = RL::group();
  const long long step = (long long)gridDim.x * 4 * RL::ROWS;
  const int hd = p.g.hd;
  float wv[NV][4], dwacc[NV][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = RL::col(i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wv[i][j] = (p.w && c < hd) ? p.w[c + j] : 1.f;
      dwacc[i][j] = 0.f;
    }
  }
  using Raw = typename Elem<T>::Raw4;
  struct Row {
    size_t oi, yi;                // in o and in y
    long long gi;                 // its gate
    Raw x[NV], z[NV];             // z: what is added, or the gradient
    float gate;
  };
  auto load = [&](long long row, Row& r) {
    const int h = (int)(row % p.g.H);
    const long long bl = row / p.g.H;
    const int l = (int)(bl % p.g.L);
    const long long b = bl / p.g.L;
    r.oi = ((size_t)(b * p.g.H + h) * p.g.L + l) * hd;
    r.yi = ((size_t)bl * p.g.H + h) * hd;
    r.gi = bl * p.g.H + h;
    const T* src = reinterpret_cast<const T*>(p.o) + r.oi;
    const T* other = BWD ? reinterpret_cast<const T*>(p.dy) + r.yi : p.add ? reinterpret_cast<const T*>(p.add) + r.yi : nullptr;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = RL::col(i);
      r.x[i] = r.z[i] = Raw{};
      if (c < hd) {
        r.x[i] = *reinterpret_cast<const Raw*>(src + c);
        if (other) r.z[i] = *reinterpret_cast<const Raw*>(other + c);
      }
    }
    r.gate = p.gate_raw ? Elem<T>::load(reinterpret_cast<const T*>(p.gate_raw) + r.gi) : 0.f;
  };
  // Forward: a row ahead, so that the loads of the next one are on their way while this one is summed.  (The backward has too few
  // registers left for it: 45 -> 47 us.)
  Row cur, next;
  long long row = ((long long)blockIdx.x * 4 + wave) * RL::ROWS + grp;
  if (!BWD && row < p.g.rows()) load(row, cur);
  for (; row < p.g.rows(); row += step) {
    if (BWD) load(row, cur);
    else if (row + step < p.g.rows()) load(row + step, next);
    const size_t oi = cur.oi, yi = cur.yi;
    const float graw = cur.gate;
    float x[NV][4], z[NV][4];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      Elem<T>::unpack4(cur.x[i], x[i]);
      Elem<T>::unpack4(cur.z[i], z[i]);
    }
    float rstd = 1.f;
    if (p.use_norm) rstd = rsqrtf(RL::sum([&](int i, int j, float s) { return s + x[i][j] * x[i][j]; }) / (float)hd + p.eps);
    const float gate = p.gate_raw ? Elem<T>::rnd(silu_f(graw)) : 1.f;
    if (!BWD) {
      T* dst = reinterpret_cast<T*>(p.y) + yi;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = RL::col(i);
        if (c < hd) {
          float o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float t = x[i][j] * rstd;
            if (p.use_norm) t = Elem<T>::rnd(t * wv[i][j]);     // the normalised tensor has type T in the reference
            o[j] = t * gate;
            if (p.add) o[j] = z[i][j] + Elem<T>::rnd(o[j]);
          }
          Elem<T>::store4(dst + c, o[0], o[1], o[2], o[3]);
        }
      }
    } else {
      // n = x rstd; t = n w; y = t g.   dt = dy g; dg = <dy, t>; dn = dt w; dw += dt n; dx = rstd (dn - n mean(dn n))
      float dn[NV][4];
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float dt = z[i][j] * gate;
          if (p.use_norm) dwacc[i][j] += dt * (x[i][j] * rstd);
          dn[i][j] = p.use_norm ? dt * wv[i][j] : dt;
        }
      float dnn = 0.f;
      if (p.use_norm) dnn = RL::sum([&](int i, int j, float s) { return s + dn[i][j] * (x[i][j] * rstd); }) / (float)hd;
      if (p.gate_raw) {
        const float dg = RL::sum([&](int i, int j, float s) {
          const float n = x[i][j] * rstd;
          return s + z[i][j] * (p.use_norm ? n * wv[i][j] : n);
        });
        if ((threadIdx.x & (G - 1)) == 0) Elem<T>::store(reinterpret_cast<T*>(p.dgate_raw) + cur.gi, dg * silu_grad_f(graw));
      }
      T* dx = reinterpret_cast<T*>(p.d_o) + oi;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int c = RL::col(i);
        if (c < hd) {
          float o[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] = p.use_norm ? rstd * (dn[i][j] - x[i][j] * rstd * dnn) : dn[i][j];
          Elem<T>::store4(dx + c, o[0], o[1], o[2], o[3]);
        }
      }
    }
    if (!BWD) cur = next;
  }
  if (BWD && p.dw_part) {      // the shares of the wave's rows, then the four waves', in a fixed order
    __shared__ float red[NV * 4 * G];
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int o = G; o < 64; o *= 2) dwacc[i][j] += __shfl_xor(dwacc[i][j], o, 64);
    for (int w = 0; w < 4; ++w) {
      if (wave == w && grp == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float* r = &red[RL::col(i) + j];
            *r = w == 0 ? dwacc[i][j] : *r + dwacc[i][j];
          }
      }
      __syncthreads();
    }
    for (int c = threadIdx.x; c < hd; c += 256) p.dw_part[(size_t)blockIdx.x * hd + c] = red[c];
  }
}

// out[c] = sum over the rows of part [rows][dim], in a fixed order: 64 columns and 16 groups of rows a block.  Grid ceil(dim / 64),
// 1024 threads.
__global__ __launch_bounds__(1024) void k_layer_sum_rows(const float* part, int rows, int dim, float* out) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (c < dim)
#pragma unroll 16
    for (int r = grp; r < rows; r += 16) s += part[(size_t)r * dim + c];
  red[grp][lane] = s;
  __syncthreads();
  if (grp == 0 && c < dim) {
    for (int i = 1; i < 16; ++i) s += red[i][lane];
    out[c] = s;
  }
}

// ---- small projections of the layer input -------------------------------------------------------------
// lr_proj (fp32, outside autocast) and, in the causal layer, momentum_proj[0] and ttt_scale_proj (bf16 under autocast) read the
// layer's input like to_qkv does, but have a handful of outputs.  One pass over the fp32 input makes the bf16 copy that the
// to_qkv GEMM reads and the latter two, one all their parameter gradients, one the gradient of the input.
//
// Output n of the launch: n < NL * 4: rate row n (valid below n1), from the fp32 input and weights; behind them the rows of the
// two bf16 maps, from input and weights rounded to bf16, the sum in fp32, the result rounded: what the GEMMs of autocast do.
// Bound by HBM and vector-ALU issue alike.  16384 tokens of 1536 channels, 12 + 8 outputs, us: forward 28 (the two products and four
// casts 85), gradient of the input 37 (51 with a token's row asked for behind the one before it), of the parameters 37 + 8 (six
// products with a dozen rows or columns each, two bias sums and seven additions and casts: 520).  7500 tokens of 768 channels, 24 outputs: 15.5 and 18 + 5 (85).
struct LayerInMap {
  const float* w;      // [n][dim] fp32
  const float* bias;   // [n] or null (forward)
  int n;
};
struct LayerInParams {
  long long rows;      // tokens
  int dim;
  const float* x;      // [rows, dim]
  uint16_t* xb;        // forward: bf16 copy of x
  LayerInMap lr, mom, gate;
  float* mom_raw;      // [rows, mom.n], bf16 values
  uint16_t* gate_raw;  // [rows, gate.n]
  // backward
  const float* dlr; const float* dmom; const uint16_t* dgate;   // each nullable: no gradient
  const uint16_t* dxq; // gradient of the input through to_qkv, [rows, dim]
  float* dx;           // [rows, dim]
  float* part;         // [parts][(NL + NB) * 4][dim] partial sums of the weight gradients
  float* bpart;        // [parts * 4][(NL + NB) * 4] and of the bias gradients
  int parts, dw_tok;   // dw_tok: tokens of a wave in the weight gradients, at most LAYER_IN_DWTOK
  float* dw[3]; float* db[3];   // by map; each nullable
};
constexpr int LAYER_IN_TOK = 4;     // tokens of a wave in the forward
constexpr int LAYER_IN_DXTOK = 32;  // tokens of a block in the input gradient
constexpr int LAYER_IN_DWTOK = 32;  // most tokens of a wave in the weight gradients

// row `n` of the launch as (map, row inside it); map -1: padding
template <int NL, int NB>
__device__ __forceinline__ int layer_in_row(const LayerInParams& p, int n, int& r) {
  if (n < 4 * NL) { r = n; return n < p.lr.n ? 0 : -1; }
  r = n - 4 * NL;
  if (r < p.mom.n) return 1;
  r -= p.mom.n;
  return r < p.gate.n ? 2 : -1;
}
template <int NL, int NB>
__device__ __forceinline__ float4 layer_in_weight(const LayerInParams& p, int n, int c) {
  int r;
  const int m = layer_in_row<NL, NB>(p, n, r);
  if (m < 0 || c >= p.dim) return make_float4(0.f, 0.f, 0.f, 0.f);
  const float* w = m == 0 ? p.lr.w : m == 1 ? p.mom.w : p.gate.w;
  float4 v = *reinterpret_cast<const float4*>(w + (size_t)r * p.dim + c);
  if (m > 0) v = make_float4(round_bf16(v.x), round_bf16(v.y), round_bf16(v.z), round_bf16(v.w));
  return v;
}
// The gradients that arrive at the outputs of `toks` tokens from t0 on, to g[token][output] in LDS by `threads` threads.  Each map's lie
// one after the other in memory: four loads of a thread at a time (one by one, each behind the last
// one's latency, k_layer_in_dw took 44 us instead of 37).
template <int NL, int NB>
__device__ __forceinline__ void layer_in_grads(const LayerInParams& p, float* g, long long t0, int toks, int tid, int threads) {
  constexpr int NO = 4 * (NL + NB);
  for (int i = tid; i < toks * NO; i += threads) g[i] = 0.f;
  __syncthreads();
  auto map = [&](int n, int first, auto load) {
    const int total = toks * n;
    const long long from = t0 * n;
    for (int i0 = tid; i0 < total; i0 += 4 * threads) {
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = load(from + min(i0 + j * threads, total - 1));
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + j * threads, k = i / n;
        if (i < total) g[k * NO + first + i - k * n] = v[j];
      }
    }
  };
  if (NL > 0 && p.dlr) map(p.lr.n, 0, [&](long long e) { return p.dlr[e]; });
  if (NB > 0 && p.dmom) map(p.mom.n, 4 * NL, [&](long long e) { return round_bf16(p.dmom[e]); });
  if (NB > 0 && p.dgate) map(p.gate.n, 4 * NL + p.mom.n, [&](long long e) { return bf16_to_f32(p.dgate[e]); });
}

// Forward: the bf16 copy and the bf16 maps.  (The rates stay a library product: they decide the roundings of everything that
// Newton-Schulz amplifies.)  A wave owns four tokens, its lanes the columns in chunks of 256; the chunk's weights are staged in
// LDS for the block's 16 tokens.  The sums over the lanes of all outputs together: every step of the exchange halves the values a
// lane holds (one shuffle a value instead of six).
template <int NB>
__global__ __launch_bounds__(256) void k_layer_in(const LayerInParams p) {
  prefetch_args<sizeof(p)>();
  constexpr int NO = 4 * NB, TOK = LAYER_IN_TOK;
  __shared__ float4 ws[NO][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long t0 = ((long long)blockIdx.x * 4 + wave) * TOK;
  float v[NO * TOK];
#pragma unroll
  for (int i = 0; i < NO * TOK; ++i) v[i] = 0.f;
  const int chunks = (p.dim + 255) / 256;
  float4 xn[TOK], wn[NB];
  auto fetch = [&](int ch) {   // the next chunk's input and weights, while this one's are used
    const int c = ch * 256 + lane * 4;
#pragma unroll
    for (int k = 0; k < TOK; ++k)
      xn[k] = (c < p.dim && t0 + k < p.rows) ? *reinterpret_cast<const float4*>(p.x + (t0 + k) * p.dim + c) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NB; ++i) wn[i] = layer_in_weight<0, NB>(p, i * 4 + wave, c);
  };
  fetch(0);
  for (int ch = 0; ch < chunks; ++ch) {
    const int c = ch * 256 + lane * 4;
    float4 x[TOK];
#pragma unroll
    for (int k = 0; k < TOK; ++k) x[k] = xn[k];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NB; ++i) ws[i * 4 + wave][lane] = wn[i];
    __syncthreads();
    if (ch + 1 < chunks) fetch(ch + 1);
#pragma unroll
    for (int k = 0; k < TOK; ++k) {
      const uint32_t lo = pack_bf16(x[k].x, x[k].y), hi = pack_bf16(x[k].z, x[k].w);
      if (c < p.dim && t0 + k < p.rows) *reinterpret_cast<uint2*>(p.xb + (t0 + k) * p.dim + c) = make_uint2(lo, hi);
      x[k] = make_float4(bf16_lo(lo), bf16_hi(lo), bf16_lo(hi), bf16_hi(hi));
    }
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      const float4 w = ws[n][lane];
#pragma unroll
      for (int k = 0; k < TOK; ++k) v[n * TOK + k] = fmaf(x[k].x, w.x, fmaf(x[k].y, w.y, fmaf(x[k].z, w.z, fmaf(x[k].w, w.w, v[n * TOK + k]))));
    }
  }
  // value 16 i + 8 b(2) + 4 b(3) + 2 b(4) + b(5) ends up in v[i] of the lanes with these bits b
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int d = 32 >> s;
    const bool up = (lane & d) != 0;
#pragma unroll
    for (int i = 0; i < (NO * TOK) >> (s + 1); ++i) {
      const float keep = up ? v[2 * i + 1] : v[2 * i], send = up ? v[2 * i] : v[2 * i + 1];
      v[i] = keep + __shfl_xor(send, d, 64);
    }
  }
  const int tok = 2 * ((lane >> 4) & 1) + (lane >> 5), sub = 2 * ((lane >> 2) & 1) + ((lane >> 3) & 1);
  const long long t = t0 + tok;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    float s = v[i];
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 1, 64);
    if ((lane & 3) == 0 && t < p.rows) {
      int r;
      const int m = layer_in_row<0, NB>(p, i * 4 + sub, r);
      if (m == 1) p.mom_raw[t * p.mom.n + r] = round_bf16(p.mom.bias ? s + round_bf16(p.mom.bias[r]) : s);
      else if (m == 2) p.gate_raw[t * p.gate.n + r] = f32_to_bf16(p.gate.bias ? s + round_bf16(p.gate.bias[r]) : s);
    }
  }
}

// Gradient of the input: dx = dxq + sum over the outputs of gradient times weight row.  A lane owns four columns and keeps their
// weights, the block's tokens have their output gradients in LDS.  Grid (token blocks, column blocks of blockDim.x * 4).  All 40 outputs take
// 216 registers, two waves a SIMD; more outputs would need a second pass.
template <int NL, int NB>
__global__ __launch_bounds__(256) void k_layer_in_dx(const LayerInParams p) {
  prefetch_args<sizeof(p)>();
  constexpr int NO = 4 * (NL + NB), TOK = LAYER_IN_DXTOK;
  __shared__ float gs[TOK][NO];
  const long long t0 = (long long)blockIdx.x * TOK;
  const int toks = (int)min((long long)TOK, p.rows - t0);
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  constexpr int AHEAD = 8;                   // tokens whose rows are asked for together
  uint2 in[AHEAD];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) in[k] = *reinterpret_cast<const uint2*>(p.dxq + (t0 + min(k0 + k, toks - 1)) * p.dim + min(c, p.dim - 4));
  };
  fetch(0);
  float4 w[NO];
#pragma unroll
  for (int n = 0; n < NO; ++n) w[n] = layer_in_weight<NL, NB>(p, n, c);
  layer_in_grads<NL, NB>(p, &gs[0][0], t0, toks, threadIdx.x, blockDim.x);
  __syncthreads();
  if (c >= p.dim) return;
  for (int k0 = 0; k0 < toks; k0 += AHEAD) {
    uint2 now[AHEAD];
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) now[k] = in[k];
    if (k0 + AHEAD < toks) fetch(k0 + AHEAD);
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      if (k0 + k >= toks) break;
      float o[4];
      Elem<uint16_t>::unpack4(now[k], o);
#pragma unroll
      for (int n = 0; n < NO; ++n) {
        const float g = gs[k0 + k][n];
        o[0] = fmaf(g, w[n].x, o[0]); o[1] = fmaf(g, w[n].y, o[1]); o[2] = fmaf(g, w[n].z, o[2]); o[3] = fmaf(g, w[n].w, o[3]);
      }
      *reinterpret_cast<float4*>(p.dx + (t0 + k0 + k) * p.dim + c) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

// Gradients of the small maps' parameters: a lane owns four columns of every row and sums its wave's tokens, the block its four
// waves', in a fixed order; k_layer_in_reduce sums the blocks.  Grid (token blocks, chunks of 256 columns).
template <int NL, int NB>
__global__ __launch_bounds__(256) void k_layer_in_dw(const LayerInParams p) {
  prefetch_args<sizeof(p)>();
  constexpr int NO = 4 * (NL + NB), TOK = LAYER_IN_DWTOK;
  __shared__ float lds[(4 * TOK > 256 ? 4 * TOK : 256) * NO];   // output gradients of the block's tokens, then the sums of its waves
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tok = p.dw_tok;
  const long long t0 = ((long long)blockIdx.x * 4 + wave) * tok;
  float* gs = lds + wave * TOK * NO;
  const int toks = (int)max(0LL, min((long long)tok, p.rows - t0));
  layer_in_grads<NL, NB>(p, gs, t0, toks, lane, 64);
  __syncthreads();
  const int c = blockIdx.y * 256 + lane * 4;
  if (blockIdx.y == 0 && lane < NO) {
    float s = 0.f;
    for (int k = 0; k < toks; ++k) s += gs[k * NO + lane];
    p.bpart[((size_t)blockIdx.x * 4 + wave) * NO + lane] = s;
  }
  float4 acc[NO];
#pragma unroll
  for (int n = 0; n < NO; ++n) acc[n] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c < p.dim) {
#pragma unroll 8
    for (int k = 0; k < toks; ++k) {
      float4 x = *reinterpret_cast<const float4*>(p.x + (t0 + k) * p.dim + c);
#pragma unroll
      for (int n = 0; n < NO; ++n) {
        if (n == 4 * NL) x = make_float4(round_bf16(x.x), round_bf16(x.y), round_bf16(x.z), round_bf16(x.w));
        const float g = gs[k * NO + n];
        acc[n].x = fmaf(g, x.x, acc[n].x); acc[n].y = fmaf(g, x.y, acc[n].y); acc[n].z = fmaf(g, x.z, acc[n].z); acc[n].w = fmaf(g, x.w, acc[n].w);
      }
    }
  }
  __syncthreads();
  float4* sums = reinterpret_cast<float4*>(lds);
  for (int w = 0; w < 4; ++w) {
    if (wave == w) {
#pragma unroll
      for (int n = 0; n < NO; ++n) {
        float4 v = acc[n];
        if (w > 0) {
          const float4 o = sums[n * 64 + lane];
          v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
        }
        sums[n * 64 + lane] = v;
      }
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < NO * 64; i += 256) {
    const int n = i / 64, cc = blockIdx.y * 256 + (i % 64) * 4;
    if (cc < p.dim) *reinterpret_cast<float4*>(p.part + ((size_t)blockIdx.x * NO + n) * p.dim + cc) = sums[i];
  }
}
// Grid (ceil(dim / 64), NO): 64 columns of one row, four groups of partial sums.
template <int NL, int NB>
__global__ __launch_bounds__(256) void k_layer_in_reduce(const LayerInParams p) {
  constexpr int NO = 4 * (NL + NB);
  __shared__ float red[4][64];
  const int n = blockIdx.y, lane = threadIdx.x & 63, grp = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
  int r;
  const int m = layer_in_row<NL, NB>(p, n, r);
  if (m < 0) return;
  float s = 0.f;
  if (c < p.dim)
#pragma unroll 8
    for (int i = grp; i < p.parts; i += 4) s += p.part[((size_t)i * NO + n) * p.dim + c];
  red[grp][lane] = s;
  __syncthreads();
  float* dw = m == 0 ? p.dw[0] : m == 1 ? p.dw[1] : p.dw[2];
  float* db = m == 0 ? p.db[0] : m == 1 ? p.db[1] : p.db[2];
  if (grp == 0 && c < p.dim && dw) dw[(size_t)r * p.dim + c] = red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane];
  if (grp == 1 && blockIdx.x == 0 && db) {
    float b = 0.f;
    for (int i = lane; i < p.parts * 4; i += 64) b += p.bpart[(size_t)i * NO + n];
    b = wave_sum(b);
    if (lane == 0) db[r] = b;
  }
}

}  // namespace lact
