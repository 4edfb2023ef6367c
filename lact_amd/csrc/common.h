// Shared device helpers for the LaCT HIP kernels (gfx950 / CDNA4 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// a lambda of many lines or calls stays a function of its own otherwise, its captures in memory
#define LACT_INLINE_LAMBDA __attribute__((always_inline))

namespace lact {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// bf16 is handled as raw uint16_t in memory; conversions go through __bf16 so that the
// compiler emits the hardware round-to-nearest-even convert.
struct bf16 {
  uint16_t bits;
};

__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float(((uint32_t)h) << 16); }
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  __bf16 h = (__bf16)f;
  return __builtin_bit_cast(uint16_t, h);
}
// Two values at once: one v_cvt_pk_bf16_f32 (lo in the lower half) where separate conversions take three instructions to pack.
// The GEMM epilogues are bound by vector-ALU issue.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
// Round a float to the nearest bf16-representable float.  Converted into the upper half beside a zero, the value is a float again
// where it stands: one instruction of 4 clocks.  (Clocks a wave-wide operation takes of a SIMD with several waves: 2 for fp32 multiply
// and add, and / or / right shift; 4 for conversions, fma and left shift; 8 for exp and rcp.  One wave alone: 4 at least.)
__device__ __forceinline__ float round_bf16(float f) { return __uint_as_float(pack_bf16(0.f, f)); }
__device__ __forceinline__ float bf16_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// Element-type policies: T = uint16_t (bf16 storage) or float.
template <typename T> struct Elem;
template <> struct Elem<uint16_t> {
  static constexpr bool kIsBf16 = true;
  __device__ static __forceinline__ float load(const uint16_t* p) { return bf16_to_f32(*p); }
  __device__ static __forceinline__ void store(uint16_t* p, float v) { *p = f32_to_bf16(v); }
  __device__ static __forceinline__ float rnd(float v) { return round_bf16(v); }
  __device__ static __forceinline__ void store4(uint16_t* p, float a, float b, float c, float d) {
    uint2 u;
    u.x = pack_bf16(a, b);
    u.y = pack_bf16(c, d);
    *reinterpret_cast<uint2*>(p) = u;
  }
  using Raw4 = uint2;       // four elements as they lie in memory
  __device__ static __forceinline__ void load4(const uint16_t* p, float* o) { unpack4(*reinterpret_cast<const uint2*>(p), o); }
  __device__ static __forceinline__ void unpack4(const uint2& u, float* o) {
    o[0] = __uint_as_float(u.x << 16);
    o[1] = __uint_as_float(u.x & 0xffff0000u);
    o[2] = __uint_as_float(u.y << 16);
    o[3] = __uint_as_float(u.y & 0xffff0000u);
  }
};
template <> struct Elem<float> {
  static constexpr bool kIsBf16 = false;
  __device__ static __forceinline__ float load(const float* p) { return *p; }
  __device__ static __forceinline__ void store(float* p, float v) { *p = v; }
  __device__ static __forceinline__ float rnd(float v) { return v; }
  __device__ static __forceinline__ void store4(float* p, float a, float b, float c, float d) {
    *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d);
  }
  using Raw4 = float4;
  __device__ static __forceinline__ void load4(const float* p, float* o) { unpack4(*reinterpret_cast<const float4*>(p), o); }
  __device__ static __forceinline__ void unpack4(const float4& u, float* o) {
    o[0] = u.x; o[1] = u.y; o[2] = u.z; o[3] = u.w;
  }
};

// one v_exp_f32 and one v_rcp_f32 (1 ulp) instead of the ten-instruction IEEE division: the epilogues that call
// this per element are bound by vector-ALU issue
__device__ __forceinline__ float sigmoidf_(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Sum over the threads of a block (blockDim.x multiple of 64, <= 1024). `red` holds >= 16 floats.
// Every thread receives the total.  Deterministic for a fixed block size.
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

// The arguments of a launch lie in memory, and the scalar cache is cold when a kernel begins: read one by one where the code
// first needs them, they cost one memory latency per 64-byte line, in a row.  One load from every line of the first BYTES up
// front makes that a single one: the token reduction's copy waves start 0.7 us after the block instead of 2.1 us (with the
// divisions gone and the offsets of the copies computed without 64-bit products), the hidden stage's 0.6 instead of 1.1 us.
#define LACT_TOUCH(o) "s_load_dword %0, %1, " #o "*64\n\t"
#define LACT_TOUCH3 LACT_TOUCH(0) LACT_TOUCH(1) LACT_TOUCH(2)
#define LACT_TOUCH4 LACT_TOUCH3 LACT_TOUCH(3)
#define LACT_TOUCH8 LACT_TOUCH4 LACT_TOUCH(4) LACT_TOUCH(5) LACT_TOUCH(6) LACT_TOUCH(7)
#define LACT_TOUCH12 LACT_TOUCH8 LACT_TOUCH(8) LACT_TOUCH(9) LACT_TOUCH(10) LACT_TOUCH(11)
#define LACT_TOUCH16 LACT_TOUCH12 LACT_TOUCH(12) LACT_TOUCH(13) LACT_TOUCH(14) LACT_TOUCH(15)
// one block with its wait: nothing else may hold the register while a load is on its way to it
#define LACT_TOUCH_ARGS(lines) asm volatile(lines "s_waitcnt lgkmcnt(0)" : "=&s"(unused) : "s"(args) : "memory")
template <int BYTES>
__device__ __forceinline__ void prefetch_args() {
  const uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  constexpr int N = (BYTES + 63) / 64;
  [[maybe_unused]] int unused;
  if constexpr (N < 3) return;   // what one load brings anyway, or two
  else if constexpr (N == 3) LACT_TOUCH_ARGS(LACT_TOUCH3);
  else if constexpr (N == 4) LACT_TOUCH_ARGS(LACT_TOUCH4);
  else if constexpr (N == 5) LACT_TOUCH_ARGS(LACT_TOUCH4 LACT_TOUCH(4));
  else if constexpr (N == 6) LACT_TOUCH_ARGS(LACT_TOUCH4 LACT_TOUCH(4) LACT_TOUCH(5));
  else if constexpr (N == 7) LACT_TOUCH_ARGS(LACT_TOUCH4 LACT_TOUCH(4) LACT_TOUCH(5) LACT_TOUCH(6));
  else if constexpr (N < 12) LACT_TOUCH_ARGS(LACT_TOUCH8);
  else if constexpr (N < 16) LACT_TOUCH_ARGS(LACT_TOUCH12);
  else LACT_TOUCH_ARGS(LACT_TOUCH16);
}

// A pointer that is the same for the whole wave, in scalar registers wherever it was computed.
template <class P>
__device__ __forceinline__ P* uniform(P* p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  return reinterpret_cast<P*>((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a) | (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32)) << 32);
}

// Side job of a kernel that runs right before a fused Newton-Schulz launch: its first block clears the barrier
// lines and the error word (a few KiB), which saves a launch of its own in the dependent chain.
struct ClearWords {
  unsigned* ptr; int n;
};
__device__ __forceinline__ void clear_words(const ClearWords& c, bool first_block) {
  if (c.n > 0 && first_block)
    for (int i = threadIdx.x; i < c.n; i += blockDim.x) c.ptr[i] = 0u;
}

// Division of 0 <= n < 2^31 by a number that the host knows, without a division's forty dependent instructions: with
// 2^(s-1) < d <= 2^s and m = ceil(2^(31+s) / d), the error n * (m d - 2^(31+s)) of the product stays below 2^(31+s).
struct UDiv {
  unsigned d, m, s;
  __host__ __device__ __forceinline__ int div(int n) const { return (int)((unsigned)(((uint64_t)(2u * (unsigned)n) * m) >> 32) >> s); }
};
inline UDiv make_udiv(int d) {
  UDiv u;
  u.d = d > 0 ? d : 1; u.s = 0;
  while ((1u << u.s) < u.d) ++u.s;
  u.m = (unsigned)((((uint64_t)1 << (31 + u.s)) + u.d - 1) / u.d);
  return u;
}

// Batch entry z = g * d + ib of a launch over several steps of a program: offset of an operand whose batch entries lie bs apart and
// whose steps gs apart.  All zero: one step, z = ib.
struct StepBatch {
  UDiv by_nb;
  __host__ __device__ __forceinline__ long long at(int z, long long bs, long long gs) const {
    const int g = by_nb.div(z);
    return (z - g * (int)by_nb.d) * bs + g * gs;
  }
};

}  // namespace lact
