// Newton-Schulz iterations (forward, and their backward) as ONE launch per batch of matrices.
//
// The unfused path runs three dependent GEMM kernels per iteration over 48 small matrices: 6 K-steps of
// matrix work per block between a launch gap and a cache write-back, 30 launches per update step.  Here the
// blocks that own the tiles of one matrix stay resident, run the stages back to back and meet at a barrier
// of their own between stages:
//
//   * the block -> tile map gives all tiles of a matrix linear ids that are congruent mod 8, i.e. the same
//     XCD (workgroups are dealt to the 8 XCDs round-robin), so everything the group exchanges lives in one L2;
//   * a stage's stores are complete in that L2 once the block has waited for them (vmcnt) -- no L2
//     write-back is needed inside an XCD -- and the operands written by the partner blocks are read with
//     device-scope loads that miss the (non-coherent) vector L1;
//   * the barrier is a counter in that L2: arrive = atomic add, wait = poll (measured ~0.6 us per barrier
//     against ~4.5 us of launch gap plus the write-back of everything the kernel stored).  Only the waves that copy
//     the operands wait, and only in front of the first operand that a partner block has just written.
//
// What bounds it: a stage is a main loop of six K-steps (twelve backwards), the staging of its tile and the exchange.  48 matrices
// of 384 x 384 on 192 compute units, forward / backward: a stage 11 / 16.5 us, of which the matrix instructions take 3.6 / 7.2; 6.5 /
// 13 main loop (8 matrices, whose operands stay in the L2s, 5.1 / 8.5: the rest is misses), 2.7 epilogue, 1.5 stores, barrier and set-up.
// Launch: 221 -> 190 and 271 -> 262 us in a training step (alone, by a probe's events, 214 -> 166 and 260 -> 249) against epilogues that
// chose their case element by element, read the auxiliary tile behind the staging and had every wave wait at the barrier; six matrices of 768 x 1536, three iterations: 195 -> 173.
// Matrices with c >= 2 r take half tiles in the r x r stages (NsHalfTile), where whole ones leave half of the blocks waiting: forward /
// backward us, six of 768 x 1536, three iterations 190 / 267 -> 175 / 248; 24 of 384 x 768, five 197 / 257 -> 178 / 224; 30 of 256 x 512
// 96 / 115 -> 81 / 97; 18 of 384 x 1152, where a third of the blocks still waits, 200 / 273 -> 180 / 235.
// Tried: the next stage's saved operand asked for into the L2 in the epilogue (-3 % there, +2 % at 12 matrices of 384 x 768);
// non-temporal loads where an operand is read for the last time (+5 %: the partner block reads it too).
//
// Should the hardware place a group's blocks on different XCDs (each block publishes its XCC id at the
// start and the group checks), the group falls back to device-scope release/acquire fences around every
// barrier -- correct anywhere, only slower.  Every poll loop is bounded: on a timeout the block raises
// the error word and moves on, so that all waves always exit.
//
// Deadlock freedom needs each group to become resident as a whole.  The host launches at most 256 blocks
// (one per compute unit at this LDS size) per kernel and orders fused launches of one process after each
// other with an event, so two such kernels never hold compute units while waiting for each other.
#pragma once
#include "gemm_dma_kernels.h"
#include "state_kernels.h"

namespace lact {

constexpr int NS_FUSED_MAX_STEPS = 8;
constexpr long long NS_FUSED_SPIN_LIMIT = 4000000;   // default bound of a barrier wait, in polls of ~64 clocks: a fraction of a second

struct NsFusedParams {
  int n, z0;                 // matrices of this launch: global indices z0 .. z0+n-1 of the packed [3b] arrays
  int r, c, S;               // Newton-Schulz orientation [r, c], r <= c, both multiples of the tile edge; iterations
  int nb, mask, plain;       // u_out is written transposed for matrices whose (z / nb) bit of mask is set
  float coeffs[3 * NS_FUSED_MAX_STEPS];
  // forward:  X_0 in xf[0] (fp32) and xb (bf16);  saves X_k, A_k, B_k (bf16) per iteration
  float* xf[2];
  uint16_t* xb; long long xb_it_stride;            // X_k at xb + k * xb_it_stride, k < S
  uint16_t* ab; uint16_t* bb; long long sq_it_stride;
  uint16_t* cab;                                   // forward: c * A of the running iteration (one [r, r] buffer per matrix)
  float* u_out;                                    // X_S, fp32, original orientation
  // backward: incoming gradient in gxf[0] / gxb[0]; the result ends in gxf[S & 1]
  float* gxf[2]; uint16_t* gxb[2]; uint16_t* sg; uint16_t* gas;
  // forward, optional first stage: X_0 = G / (|G|_F + 1e-7) from the bf16 gradient g16 (laid out like xb) and the
  // partial sums of its squares; writes xb (iteration 0) and the norms.  Null g16: X_0 is there already.
  const uint16_t* g16; const float* ss_part; int nparts, part0, part1;   // partial rows part0 + z and (if >= 0) part1 + z
  float* norms;              // [n] of this batch
  // backward, optional last stages (the backward of that normalisation): every block writes <G_final, g16> over
  // its tile to dot_part[z][member]; with gc set, the blocks then meet once more and each writes its tile of
  //   gc = G_final / (n + 1e-7) - g16 * <G_final, g16> / (n (n + 1e-7)^2)
  // (the gradient w.r.t. the Newton-Schulz input in the compute type; norms as written by the forward)
  float* dot_part; uint16_t* gc;
  // with gc and a momentum state in the program: the gradient that arrives at the state after this update is added
  // (carry_valid), the one for the state before it is written back (carry_write: g * mbar), and the partial dots
  // <g, M_prev> over this block's tile go to mdot_part[z][member] (m_prev set).  All arrays packed like gc.
  float* gm_carry; int carry_valid, carry_write;
  const float* m_prev; const float* mbar; float* mdot_part;
  unsigned* sync;            // [n][32] words, zeroed before the launch: word 0 = arrivals, word 1 = XCC id mask
  unsigned* error;           // set to 1 by a block whose barrier timed out
  unsigned* sticky;          // per-device count of such time-outs (not cleared between calls), or null
  long long spin_limit;      // polls a block waits at a barrier before it gives up
};

struct GroupBarrier {
  unsigned* ctr;
  unsigned* sticky;          // per-device count of blocks' timed-out waits, never cleared by a kernel (lact_check_async_error reads it)
  unsigned* counted;         // in LDS: the last of this block's waits that was counted there, which several waves may have waited
  unsigned members, epoch;
  long long limit;
  bool split;                // group spread over several XCDs: fence at device scope
  __device__ __forceinline__ void init(unsigned* line, unsigned nmembers, unsigned* error, long long spin_limit, unsigned* sticky_count) {
    __shared__ unsigned last_counted;
    ctr = line; members = nmembers; epoch = 0; split = false; limit = spin_limit; sticky = sticky_count; counted = &last_counted;
    if (threadIdx.x == 0) last_counted = 0;
    unsigned xcc = 0;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    if (threadIdx.x == 0) __hip_atomic_fetch_or(line + 1, 1u << (xcc & 0xf), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sync(error, true);
    unsigned m = __hip_atomic_load(line + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    split = (m & (m - 1)) != 0;
  }
  // All threads of the block call it: the block's stores are there for its partners.
  __device__ __forceinline__ void arrive(bool heavy = false) {
    // Every wave waits for its own stores of the stage: a store that has been waited for is in this XCD's L2 (the
    // vector L1 writes through), which is where the partner blocks' device-scope loads look.  Without the wait the
    // arrival below could overtake a store that is still on its way to another L2 channel.
    wait_vmcnt<0>();
    __syncthreads();
    ++epoch;
    if (threadIdx.x == 0) {
      if (heavy || split) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  // One lane of every wave that is going to read what the partners stored polls until all of them have arrived.
  __device__ __forceinline__ void wait(unsigned* error, bool heavy = false) const {
    const unsigned target = members * epoch;
    long long spins = 0;
    while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins >= limit) {
        __hip_atomic_store(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (sticky && atomicMax(counted, epoch) < epoch) __hip_atomic_fetch_add(sticky, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    if (heavy || split) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  }
  // All threads of the block call it.  A block waits for every arrival of its own before the next one: the count tells no two apart.
  __device__ __forceinline__ void pass(unsigned* error, bool heavy = false) const {
    if (threadIdx.x == 0) wait(error, heavy);
    __syncthreads();
  }
  __device__ __forceinline__ void sync(unsigned* error, bool heavy = false) {
    arrive(heavy);
    pass(error, heavy);
  }
};

template <int NT>
__device__ __forceinline__ RowGemmDmaParams<NT> ns_row_params() {
  RowGemmDmaParams<NT> q;
  q.g.accumulate = 0; q.g.aux = nullptr; q.g.ldaux = 0; q.g.bsaux = 0; q.g.alpha = 1.f; q.g.beta = 0.f;
  q.g.out_c = nullptr; q.g.out_t = nullptr; q.g.transpose_mask = 0; q.g.nb = 1; q.g.round_out_bf16 = 0;
  q.g.out2 = nullptr; q.g.alpha2 = 0.f;
  q.g.steps = StepBatch{{0, 0, 0}}; q.g.gso = 0;
  q.out_ct = nullptr;
  return q;
}
__device__ __forceinline__ void ns_term(RowGemmTerm& t, const void* A, int lda, long long bsA, const void* B, int ldb, long long bsB, int K) {
  t.A = A; t.lda = lda; t.bsA = bsA; t.B = B; t.ldb = ldb; t.bsB = bsB; t.gsB = 0; t.K = K;
}

// <gx, g16> over one TS::BM x TS::BN tile whose first element is at offset zo of both arrays (row stride c): every thread
// takes the granules of 8 elements threadIdx.x, threadIdx.x + DMA_THREADS, ... and keeps what it read (ga, gb: the fp32
// values, gi: the bf16 ones).  Returns this thread's partial sum.  The fused kernel and k_ns_bwd_dot_tiles both sum a
// tile through this one function and block_sum, so the two paths produce the same bits.
template <class TS, int NG>
__device__ __forceinline__ float ns_tile_dot(const float* gx, const uint16_t* g16, size_t zo, int c, float4 (&ga)[NG], float4 (&gb)[NG], uint4 (&gi)[NG]) {
  constexpr int GR = TS::BN / 8;
  static_assert(NG == (TS::BM * GR + DMA_THREADS - 1) / DMA_THREADS, "granules per thread");
  float dot = 0.f;
#pragma unroll
  for (int t = 0; t < NG; ++t) {
    const int id = threadIdx.x + t * DMA_THREADS;
    if (id < TS::BM * GR) {
      const size_t o = zo + (size_t)(id / GR) * c + (id % GR) * 8;
      ga[t] = *reinterpret_cast<const float4*>(gx + o);
      gb[t] = *reinterpret_cast<const float4*>(gx + o + 4);
      gi[t] = *reinterpret_cast<const uint4*>(g16 + o);
      const uint32_t w[4] = {gi[t].x, gi[t].y, gi[t].z, gi[t].w};
      dot += ga[t].x * __uint_as_float(w[0] << 16) + ga[t].y * __uint_as_float(w[0] & 0xffff0000u) +
             ga[t].z * __uint_as_float(w[1] << 16) + ga[t].w * __uint_as_float(w[1] & 0xffff0000u) +
             gb[t].x * __uint_as_float(w[2] << 16) + gb[t].y * __uint_as_float(w[2] & 0xffff0000u) +
             gb[t].z * __uint_as_float(w[3] << 16) + gb[t].w * __uint_as_float(w[3] & 0xffff0000u);
    }
  }
  return dot;
}

// The partial dots of the Frobenius normalisation's backward as the fused backward kernel forms them (one per tile of
// the fused kernel's tiling, summed in its order), for the unfused launches: the two paths then hand the same bits
// to everything downstream.  Grid (tiles per matrix, matrices); matrices are [r, c] one after the other.
struct NsTileDotParams {
  const float* gx; const uint16_t* g16; float* dot_part;
  int r, c;
};
template <class TS>
__global__ __launch_bounds__(DMA_THREADS) void k_ns_bwd_dot_tiles(const NsTileDotParams p) {
  __shared__ float red[16];
  constexpr int GR = TS::BN / 8, NG = (TS::BM * GR + DMA_THREADS - 1) / DMA_THREADS;
  const int tc = p.c / TS::BN, member = blockIdx.x, z = blockIdx.y;
  const int rx = member / tc, ry = member % tc;
  const size_t zo = (size_t)z * p.r * p.c + (size_t)rx * TS::BM * p.c + ry * TS::BN;
  float4 ga[NG], gb[NG];
  uint4 gi[NG];
  float dot = ns_tile_dot<TS>(p.gx, p.g16, zo, p.c, ga, gb, gi);
  dot = block_sum(dot, red);
  if (threadIdx.x == 0) p.dot_part[(size_t)z * gridDim.x + member] = dot;
}

// Granules of 8 elements of a TS tile, dealt to THREADS threads: LPR lanes cover CB neighbouring columns of a row and the threads RP
// rows; granule t of a thread lies at a distance from its first one that is a compile-time multiple of the row stride and columns.
template <class TS, int THREADS>
struct NsGranules {
  static constexpr int LPR = TS::BN % 64 == 0 ? 8 : 4, CB = LPR * 8, RP = THREADS / LPR, NR = (TS::BM + RP - 1) / RP, NC = TS::BN / CB, N = NR * NC;
  static_assert((TS::BM % RP == 0 || (THREADS == DMA_THREADS && TS::BM % RP == RP / 2)) && TS::BN % CB == 0, "granules split evenly over the threads");
  // rows end with a pass of the lower half of the threads (the matrix waves) only: row(t) is past the tile for the others
  static constexpr bool UPPER_SHORT = TS::BM % RP != 0;
  __device__ static constexpr bool none(bool upper, int t) { return UPPER_SHORT && upper && t % NR == NR - 1; }
  __device__ static __forceinline__ int row0() { return (threadIdx.x & (THREADS - 1)) / LPR; }
  __device__ static __forceinline__ int col0() { return (threadIdx.x % LPR) * 8; }
  __device__ static constexpr int row(int t) { return (t % NR) * RP; }
  __device__ static constexpr int col(int t) { return (t / NR) * CB; }
};

// The roles of a block's waves are split for the whole of the iterations, not stage by stage: the fp32 iterate (its gradient) of
// this block's tile then lives in the copy waves' registers, 18 granules of 8 elements per thread at 192 x 192, and only its bf16
// copy goes through memory.  In one code path for all waves it would have to live beside the matrix waves' accumulators.
// The tile of the r x r stages where c >= 2 r: their whole tiles would leave half of the matrix' blocks without work.
template <class TS> struct NsHalfTile { using type = void; };
template <> struct NsHalfTile<TS_NS> { using type = TS_H96; };
template <> struct NsHalfTile<TS_SQ> { using type = TS_BWD; };
template <class TS> constexpr int ns_stages() { return TS::BM == 192 && TS::BN == 96 ? 4 : row_stages<TS>(); }
template <class TS> constexpr int ns_waves() { return TS::WAVES_M * TS::WAVES_N; }   // that own a part of the tile
template <class TS> __device__ __forceinline__ bool ns_idle_wave() {
  return ns_waves<TS>() < 4 && __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= ns_waves<TS>();
}

template <class TS>
struct NsTileRegs {
  using G = NsGranules<TS, 256>;
  float v[G::N][8];
};

// One stage's product on this block's tile (bx, by): the copy waves' part ...  They wait at the group's barrier in front of the first
// copy of phase GATE, the matrix waves not at all (what they read comes through the ring): the phases before it run while the
// partner blocks finish the stage before this one.
template <class TS, int NT, bool B_KS, int GATE>
__device__ __forceinline__ void ns_stage_load(const RowGemmParams<NT>& p, int bx, int by, int z, char* smem, const GroupBarrier& bar, unsigned* error) {
  DmaPhase<1> ph[NT];
  row_gemm_phases<TS, NT, B_KS>(p, bx * TS::BM, by * TS::BN, z, ph);
  using Pipe = DmaPipe<TS, 1, NT, ns_stages<TS>(), true>;
  Pipe pipe(smem, ph);
  pipe.template load_all<Pipe::loads(1)>([&](int phase) {
    if (phase == GATE && (threadIdx.x & 63) == 0) bar.wait(error);
  });
}
// ... and the matrix waves'
template <class TS, int NT, bool B_KS>
__device__ __forceinline__ void ns_stage_mma(const RowGemmParams<NT>& p, int bx, int by, int z, char* smem, f32x16 (&acc)[1][TS::TM][TS::TN]) {
  DmaPhase<1> ph[NT];
  row_gemm_phases<TS, NT, B_KS>(p, bx * TS::BM, by * TS::BN, z, ph);
  DmaPipe<TS, 1, NT, ns_stages<TS>(), true> pipe(smem, ph);
  if (ns_idle_wave<TS>()) return pipe.idle();
  zero_acc<TS>(acc[0]);
  int step = 0;
#pragma unroll
  for (int t = 0; t < NT; ++t) pipe.template run_phase<1, false, B_KS>(p.t[t].K, step, acc);
}
template <class TS>
__device__ __forceinline__ void ns_put_tile(char* smem, const f32x16 (&acc)[1][TS::TM][TS::TN]) {   // rounded to bf16
  using ST = StageTile<TS, 2>;
  if (ns_idle_wave<TS>()) return;
  char* lb = smem + ST::lane_base();
  LACT_FOR_QUADS(TS) ST::put4(lb, tm, tn, g, acc[0][tm][tn][4 * g], acc[0][tm][tn][4 * g + 1], acc[0][tm][tn][4 * g + 2], acc[0][tm][tn][4 * g + 3]);
}
// EPI_STORE: out = round(product), and out2 = round(alpha2 * out) if there is one.  EPI_AXPBY: out = round(round(alpha product) + round(beta aux));
// the auxiliary tile is asked for in front of the staging.
template <class TS, int NT, int EPI, bool COPY>
__device__ __forceinline__ void ns_stage_b16(const RowGemmParams<NT>& p, int bx, int by, int z, char* smem, const GroupBarrier& bar, unsigned* error) {
  using G = NsGranules<TS, DMA_THREADS>;
  using ST = StageTile<TS, 2>;
  f32x16 acc[1][TS::TM][TS::TN];   // matrix waves only
  if constexpr (COPY) ns_stage_load<TS, NT, false, 0>(p, bx, by, z, smem, bar, error);
  else ns_stage_mma<TS, NT, false>(p, bx, by, z, smem, acc);
  __syncthreads();   // the matrix waves are through with the ring
  const int r0 = G::row0(), c0 = G::col0();
  const size_t o0 = z * p.bso + (size_t)(bx * TS::BM + r0) * p.ldo + by * TS::BN + c0;
  uint4 w[G::N];
  if constexpr (EPI == EPI_AXPBY) {
#pragma unroll
    for (int t = 0; t < G::N; ++t)
      if (!G::none(COPY, t)) w[t] = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.aux) + o0 + (size_t)G::row(t) * p.ldo + G::col(t));
  }
  if constexpr (!COPY) ns_put_tile<TS>(smem, acc);
  __syncthreads();
  const char* src = smem + (r0 * ST::LD + c0) * 2;
  constexpr int LG = COPY ? 3 : G::N;   // LDS reads in flight together: the copy waves are short of registers
  uint4 u[LG];
#pragma unroll
  for (int t = 0; t < G::N; ++t) {
    if (t % LG == 0) {
      if (COPY) asm volatile("" ::: "memory");
#pragma unroll
      for (int g = 0; g < LG; ++g)
        if (t + g < G::N && !G::none(COPY, t + g)) u[g] = *reinterpret_cast<const uint4*>(src + (G::row(t + g) * ST::LD + G::col(t + g)) * 2);
    }
    if (G::none(COPY, t)) continue;
    const size_t o = o0 + (size_t)G::row(t) * p.ldo + G::col(t);
    uint32_t uu[4] = {u[t % LG].x, u[t % LG].y, u[t % LG].z, u[t % LG].w};
    if constexpr (EPI == EPI_AXPBY) {
      const uint32_t ww[4] = {w[t].x, w[t].y, w[t].z, w[t].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float alo = NT == 1 ? bf16_lo(uu[j]) : p.alpha * bf16_lo(uu[j]), ahi = NT == 1 ? bf16_hi(uu[j]) : p.alpha * bf16_hi(uu[j]);   // one term: alpha is 1
        if (NT > 1) round_both(alo, ahi);
        float blo = p.beta * bf16_lo(ww[j]), bhi = p.beta * bf16_hi(ww[j]);
        round_both(blo, bhi);
        uu[j] = pack_bf16(alo + blo, ahi + bhi);
      }
    }
    *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.out) + o) = make_uint4(uu[0], uu[1], uu[2], uu[3]);
    if (EPI == EPI_STORE && NT == 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) uu[j] = pack_bf16(p.alpha2 * bf16_lo(uu[j]), p.alpha2 * bf16_hi(uu[j]));
      *reinterpret_cast<uint4*>(reinterpret_cast<uint16_t*>(p.out2) + o) = make_uint4(uu[0], uu[1], uu[2], uu[3]);
    }
  }
}

// The stage that makes the next iterate, X' = beta X + product (B K-strided): the staged product, a bf16 tensor in the reference
// (ttt_operation.py:62), blended with the fp32 tile in the copy waves' registers.  out_c: bf16 copy; of the last one instead out_t: fp32
// ([r, c]; transposed, [c, r], if `tr`).  PLAIN: X' is a bf16 tensor; decided inside the loop it costs as much as the blend (5.7 us a
// tile of 192 x 192).
template <class TS, int NT, bool COPY, int GATE, bool PLAIN>
__device__ __forceinline__ void ns_stage_iterate(const RowGemmParams<NT>& p, int bx, int by, int z, char* smem, NsTileRegs<TS>* x, bool tr, const GroupBarrier& bar, unsigned* error) {
  using G = NsGranules<TS, 256>;
  const int m0 = bx * TS::BM, n0 = by * TS::BN;
  if constexpr (COPY) {
    using ST = StageTile<TS, 2>;
    ns_stage_load<TS, NT, true, GATE>(p, bx, by, z, smem, bar, error);
    __syncthreads();   // the matrix waves are through with the ring
    __syncthreads();   // and have staged the tile
    const char* src = smem + (G::row0() * ST::LD + G::col0()) * 2;
    const size_t o = z * p.bso + (size_t)(m0 + G::row0()) * p.ldo + n0 + G::col0();
    uint16_t* oc = reinterpret_cast<uint16_t*>(p.out_c) + o;
#pragma unroll
    for (int t = 0; t < G::N; ++t) {
      if (t % 3 == 0) asm volatile("" ::: "memory");   // three granules' reads at a time: more of them do not fit beside the tile
      float in[8];
      unpack8(*reinterpret_cast<const uint4*>(src + (G::row(t) * ST::LD + G::col(t)) * 2), in);
      float (&v)[8] = x->v[t];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = dual_blend(in[i], __fmul_rn(p.beta, v[i]), PLAIN);
      if (p.out_c) *reinterpret_cast<uint4*>(oc + (size_t)G::row(t) * p.ldo + G::col(t)) = pack8(v);
    }
  } else {
    f32x16 acc[1][TS::TM][TS::TN];
    ns_stage_mma<TS, NT, true>(p, bx, by, z, smem, acc);
    __syncthreads();
    ns_put_tile<TS>(smem, acc);
    __syncthreads();
  }
  if (!p.out_t) return;
  const bool turn = NT == 1 && tr;
  if (turn) __syncthreads();   // the staged product has been read
  if constexpr (COPY) {
    using ST = StageTile<TS, 4>;
    float* dst = turn ? reinterpret_cast<float*>(smem) + G::row0() * ST::LD + G::col0()
                      : p.out_t + z * p.bso + (size_t)(m0 + G::row0()) * p.ldo + n0 + G::col0();
    const int ld = turn ? ST::LD : p.ldo;
#pragma unroll
    for (int t = 0; t < G::N; ++t) {
      const float (&v)[8] = x->v[t];
      float4* f = reinterpret_cast<float4*>(dst + (size_t)G::row(t) * ld + G::col(t));
      f[0] = make_float4(v[0], v[1], v[2], v[3]);
      f[1] = make_float4(v[4], v[5], v[6], v[7]);
    }
  }
  if (NT == 1 && turn) {
    __syncthreads();
    row_gemm_copy_out_transposed<TS, NT>(p, nullptr, true, m0, n0, z, smem);
  }
}

__device__ __forceinline__ void ns_load8(const float* src, float (&v)[8]) {
  const float4 lo = reinterpret_cast<const float4*>(src)[0], hi = reinterpret_cast<const float4*>(src)[1];
  v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
}

// This block's place in its matrix
struct NsPlace {
  int z;
  bool sq_tile;              // owns a tile of the r x r stages: (sx, sy)
  int sx, sy, rx, ry;        // (rx, ry): its tile of the r x c stages
};
// BWD = false: S iterations  A = X X^T;  B = b A + c A A;  X' = a X + B X
// BWD = true:  the same iterations backwards:  Sg = G X^T + X G^T;  H = b Sg + c (Sg A + A Sg);  G' = a G + B G + H X
// COPY: on the copy waves, else on the matrix waves.  PLAIN: the iterate is a bf16 tensor (reference without autocast).
// TSQ: tile of the r x r stages, TS or half of one.
template <class TS, class TSQ, bool BWD, bool COPY, bool PLAIN = false>
__device__ __forceinline__ void ns_iterations(const NsFusedParams& p, GroupBarrier& bar, const NsPlace& b, char* smem) {
  const int z = b.z;
  NsTileRegs<TS> x;
  if constexpr (COPY) {
    using G = NsGranules<TS, 256>;
    if (!BWD && p.g16) {          // staged in LDS by the normalisation
      using ST = StageTile<TS, 4>;
      const char* src = smem + (G::row0() * ST::LD + G::col0()) * 4;
#pragma unroll
      for (int t = 0; t < G::N; ++t) ns_load8(reinterpret_cast<const float*>(src) + G::row(t) * ST::LD + G::col(t), x.v[t]);
    } else {
      const float* src = (BWD ? p.gxf[0] : p.xf[0]) + (size_t)z * p.r * p.c + (size_t)(b.rx * TS::BM + G::row0()) * p.c + b.ry * TS::BN + G::col0();
#pragma unroll
      for (int t = 0; t < G::N; ++t) ns_load8(src + (size_t)G::row(t) * p.c + G::col(t), x.v[t]);
    }
  }
  if (!BWD) __syncthreads();      // the staging area becomes the ring
  const bool tr = (p.mask >> (z / p.nb)) & 1;
  for (int step = 0; step < p.S; ++step) {
    const int it = BWD ? p.S - 1 - step : step;
    const bool last = step + 1 == p.S;
    // r and c are made opaque once per iteration: otherwise the compiler hoists every stage's loop-invariant
    // per-lane address registers out of this loop, keeps them all live and spills
    int r = p.r, c = p.c;
    asm volatile("" : "+s"(r), "+s"(c));
    const long long xe = (long long)r * c, se = (long long)r * r;
    const float ca = p.coeffs[3 * it], cb = p.coeffs[3 * it + 1], cc = p.coeffs[3 * it + 2];
    const uint16_t* X = p.xb + it * p.xb_it_stride;
    uint16_t* A = p.ab + it * p.sq_it_stride;
    uint16_t* B = p.bb + it * p.sq_it_stride;
    if (!BWD) {
      if (b.sq_tile) {
        auto q = ns_row_params<1>();
        ns_term(q.g.t[0], X, c, xe, X, c, xe, c);
        q.g.M = r; q.g.N = r; q.g.out = A; q.g.ldo = r; q.g.bso = se;
        q.g.out2 = p.cab; q.g.alpha2 = cc;
        ns_stage_b16<TSQ, 1, EPI_STORE, COPY>(q.g, b.sx, b.sy, z, smem, bar, p.error);
      } else bar.pass(p.error);
      bar.arrive();
      if (b.sq_tile) {
        auto q = ns_row_params<1>();
        ns_term(q.g.t[0], p.cab, r, se, A, r, se, r);
        q.g.M = r; q.g.N = r; q.g.out = B; q.g.ldo = r; q.g.bso = se;
        q.g.aux = A; q.g.ldaux = r; q.g.bsaux = se; q.g.alpha = 1.f; q.g.beta = cb;
        ns_stage_b16<TSQ, 1, EPI_AXPBY, COPY>(q.g, b.sx, b.sy, z, smem, bar, p.error);
      } else bar.pass(p.error);
      bar.arrive();
      {
        auto q = ns_row_params<1>();
        ns_term(q.g.t[0], B, r, se, X, c, xe, r);
        q.g.M = r; q.g.N = c; q.g.ldo = c; q.g.bso = xe;
        q.g.alpha = 1.f; q.g.beta = ca;
        q.g.out_c = last ? nullptr : p.xb + (it + 1) * p.xb_it_stride;   // nothing multiplies by the last iterate
        q.g.out_t = last ? p.u_out : nullptr;
        ns_stage_iterate<TS, 1, COPY, 0, PLAIN>(q.g, b.rx, b.ry, z, smem, &x, tr, bar, p.error);
      }
      if (!last) bar.arrive();
    } else {
      const int cur = step & 1;
      const uint16_t* gb = p.gxb[cur];
      if (b.sq_tile) {   // Sg = G X^T + X G^T
        auto q = ns_row_params<2>();
        ns_term(q.g.t[0], gb, c, xe, X, c, xe, c);
        ns_term(q.g.t[1], X, c, xe, gb, c, xe, c);
        q.g.M = r; q.g.N = r; q.g.out = p.sg; q.g.ldo = r; q.g.bso = se;
        ns_stage_b16<TSQ, 2, EPI_STORE, COPY>(q.g, b.sx, b.sy, z, smem, bar, p.error);
      } else bar.pass(p.error);
      bar.arrive();
      if (b.sq_tile) {   // H = b Sg + c (Sg A + A Sg)
        auto q = ns_row_params<2>();
        ns_term(q.g.t[0], p.sg, r, se, A, r, se, r);
        ns_term(q.g.t[1], A, r, se, p.sg, r, se, r);
        q.g.M = r; q.g.N = r; q.g.out = p.gas; q.g.ldo = r; q.g.bso = se;
        q.g.aux = p.sg; q.g.ldaux = r; q.g.bsaux = se; q.g.alpha = cc; q.g.beta = cb;
        ns_stage_b16<TSQ, 2, EPI_AXPBY, COPY>(q.g, b.sx, b.sy, z, smem, bar, p.error);
      } else bar.pass(p.error);
      bar.arrive();
      {                  // G' = a G + B G + H X
        auto q = ns_row_params<2>();
        ns_term(q.g.t[0], B, r, se, gb, c, xe, r);
        ns_term(q.g.t[1], p.gas, r, se, X, c, xe, r);
        q.g.M = r; q.g.N = c; q.g.ldo = c; q.g.bso = xe;
        q.g.alpha = 1.f; q.g.beta = ca;
        q.g.out_t = last ? p.gxf[p.S & 1] : nullptr;
        q.g.out_c = last ? nullptr : p.gxb[cur ^ 1];   // nothing multiplies by the final gradient
        ns_stage_iterate<TS, 2, COPY, 1, false>(q.g, b.rx, b.ry, z, smem, &x, false, bar, p.error);   // B G needs nothing that this stage's barrier waits for
      }
      if (!last) bar.arrive();
    }
  }
}

// TS: 192 x 192 tiles, or 128 x 128 / 128 x 64 when there are too few matrices to fill the chip with the large tile.
template <class TS, bool BWD, class TSQ = TS>
__global__ __launch_bounds__(DMA_THREADS) void k_ns_fused(const NsFusedParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  prefetch_args<sizeof(p)>();
  const int tr = p.r / TS::BM, tc = p.c / TS::BN, ts = p.r / TSQ::BN;   // tile rows; tile columns of [r, c] and of [r, r]
  static_assert(TSQ::BM == TS::BM, "the tiles of both kinds of stages have the same rows");
  const int nbm = tr * tc;                           // blocks per matrix (c >= r: the r x c stages have the most tiles)
  const int L = blockIdx.x, j = L >> 3;
  const int group = (L & 7) + 8 * (j / nbm), member = j % nbm;
  if (group >= p.n) return;
  const int z = p.z0 + group;
  GroupBarrier bar;
  bar.init(p.sync + (size_t)group * 32, nbm, p.error, p.spin_limit, p.sticky);
  const bool sq_tile = member < tr * ts;             // this block owns a tile of the r x r stages
  const int sx = member / ts, sy = member % ts;      // its tile there
  const int rx = member / tc, ry = member % tc;      // its tile of the r x c stages

  if (!BWD && p.g16) {
    // Frobenius normalisation in front of the first iteration: every block of the group sums the same partials
    // in the same order, then scales its own tile of [r, c], for its copy waves in LDS and in bf16 for its partners
    float ss = 0.f;
#pragma unroll 4
    for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part0 + z) * p.nparts + i];
    if (p.part1 >= 0)
      for (int i = 0; i < p.nparts; ++i) ss += p.ss_part[(size_t)(p.part1 + z) * p.nparts + i];
    float n = sqrtf(ss);
    if (p.plain) n = round_bf16(n);
    if (member == 0 && threadIdx.x == 0) p.norms[z] = n;
    float den = n + 1e-7f;
    if (p.plain) den = round_bf16(den);
    using G = NsGranules<TS, DMA_THREADS>;
    using ST = StageTile<TS, 4>;
    const size_t o = (size_t)z * p.r * p.c + (size_t)(rx * TS::BM + G::row0()) * p.c + ry * TS::BN + G::col0();
    float* stage = reinterpret_cast<float*>(smem) + G::row0() * ST::LD + G::col0();
    uint4 u[G::N];
#pragma unroll
    for (int t = 0; t < G::N; ++t) u[t] = *reinterpret_cast<const uint4*>(p.g16 + o + (size_t)G::row(t) * p.c + G::col(t));
#pragma unroll
    for (int t = 0; t < G::N; ++t) {
      float v[8];
      unpack8(u[t], v);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = __fdiv_rn(v[i], den);   // the quotient itself (ttt_operation.py:49), not a product with 1 / den
      if (p.plain) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = round_bf16(v[i]);
      }
      float4* f = reinterpret_cast<float4*>(stage + G::row(t) * ST::LD + G::col(t));   // for the copy waves, which keep the fp32 tile
      f[0] = make_float4(v[0], v[1], v[2], v[3]);
      f[1] = make_float4(v[4], v[5], v[6], v[7]);
      *reinterpret_cast<uint4*>(p.xb + o + (size_t)G::row(t) * p.c + G::col(t)) = pack8(v);
    }
    bar.arrive();
  }
  const NsPlace place{z, sq_tile, sx, sy, rx, ry};
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= 4) {
    if (!BWD && p.plain) ns_iterations<TS, TSQ, BWD, true, !BWD>(p, bar, place, smem);
    else ns_iterations<TS, TSQ, BWD, true>(p, bar, place, smem);
  }
  else ns_iterations<TS, TSQ, BWD, false>(p, bar, place, smem);
  wait_vmcnt<0>();   // the last stage's stores, for the other waves of this block
  __syncthreads();
  if (BWD && p.dot_part) {
    // the tile this block wrote in the last stage, and the same tile of the bf16 input: 12 granules of 8 elements
    // per thread at 192 x 192, kept in registers for the second pass
    constexpr int GR = TS::BN / 8, NG = (TS::BM * GR + DMA_THREADS - 1) / DMA_THREADS;
    const float* gx = p.gxf[p.S & 1];
    const size_t zo = (size_t)z * p.r * p.c + (size_t)rx * TS::BM * p.c + ry * TS::BN;
    float4 ga[NG], gb[NG];
    uint4 gi[NG];
    // No fence: this tile of gx was written by this very block, in the last stage only (before, the iterate stays in the copy
    // waves' registers), and the waves of a compute unit share its vector L1, which their own stores keep current.  The same
    // holds for the auxiliary bf16 tile that a blending epilogue reads (the block's own tile of a buffer it wrote itself).
    float dot = ns_tile_dot<TS>(gx, p.g16, zo, p.c, ga, gb, gi);
    dot = block_sum(dot, reinterpret_cast<float*>(smem));
    if (threadIdx.x == 0) p.dot_part[(size_t)z * nbm + member] = dot;
    if (p.gc) {
      bar.sync(p.error);
      float total = 0.f;
      for (int i = 0; i < nbm; ++i) total += __hip_atomic_load(p.dot_part + (size_t)z * nbm + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const float n = p.norms[z];
      float c0 = 1.f / (n + 1e-7f);
      const float c1 = n > 0.f ? total / (n * (n + 1e-7f) * (n + 1e-7f)) : 0.f;
      if (__hip_atomic_load(p.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) c0 = __uint_as_float(0x7fc00000u);
      const float mb = p.mbar ? p.mbar[z % p.nb] : 0.f;
      float md = 0.f;
#pragma unroll
      for (int t = 0; t < NG; ++t) {
        const int id = threadIdx.x + t * DMA_THREADS;
        if (id < TS::BM * GR) {
          const size_t o = zo + (size_t)(id / GR) * p.c + (id % GR) * 8;
          const uint32_t w[4] = {gi[t].x, gi[t].y, gi[t].z, gi[t].w};
          // the gradient that leaves Newton-Schulz through its input cast (G.bfloat16()) has that type
          const float gi0 = __uint_as_float(w[0] << 16), gi1 = __uint_as_float(w[0] & 0xffff0000u), gi2 = __uint_as_float(w[1] << 16),
                      gi3 = __uint_as_float(w[1] & 0xffff0000u), gi4 = __uint_as_float(w[2] << 16), gi5 = __uint_as_float(w[2] & 0xffff0000u),
                      gi6 = __uint_as_float(w[3] << 16), gi7 = __uint_as_float(w[3] & 0xffff0000u);
          float4 v0 = make_float4(ns_input_grad<uint16_t>(ga[t].x, gi0, c0, c1), ns_input_grad<uint16_t>(ga[t].y, gi1, c0, c1),
                                  ns_input_grad<uint16_t>(ga[t].z, gi2, c0, c1), ns_input_grad<uint16_t>(ga[t].w, gi3, c0, c1));
          float4 v1 = make_float4(ns_input_grad<uint16_t>(gb[t].x, gi4, c0, c1), ns_input_grad<uint16_t>(gb[t].y, gi5, c0, c1),
                                  ns_input_grad<uint16_t>(gb[t].z, gi6, c0, c1), ns_input_grad<uint16_t>(gb[t].w, gi7, c0, c1));
          if (p.gm_carry) {
            if (p.carry_valid) {
              const float4 a = *reinterpret_cast<const float4*>(p.gm_carry + o), b = *reinterpret_cast<const float4*>(p.gm_carry + o + 4);
              v0.x += a.x; v0.y += a.y; v0.z += a.z; v0.w += a.w;
              v1.x += b.x; v1.y += b.y; v1.z += b.z; v1.w += b.w;
            }
            if (p.carry_write) {
              *reinterpret_cast<float4*>(p.gm_carry + o) = make_float4(v0.x * mb, v0.y * mb, v0.z * mb, v0.w * mb);
              *reinterpret_cast<float4*>(p.gm_carry + o + 4) = make_float4(v1.x * mb, v1.y * mb, v1.z * mb, v1.w * mb);
            }
            if (p.m_prev) {
              const float4 a = *reinterpret_cast<const float4*>(p.m_prev + o), b = *reinterpret_cast<const float4*>(p.m_prev + o + 4);
              md += v0.x * a.x + v0.y * a.y + v0.z * a.z + v0.w * a.w + v1.x * b.x + v1.y * b.y + v1.z * b.z + v1.w * b.w;
            }
          }
          Elem<uint16_t>::store4(p.gc + o, v0.x, v0.y, v0.z, v0.w);
          Elem<uint16_t>::store4(p.gc + o + 4, v1.x, v1.y, v1.z, v1.w);
        }
      }
      if (p.gm_carry && p.m_prev) {
        __syncthreads();   // the block sum above may still be read from the same LDS words
        md = block_sum(md, reinterpret_cast<float*>(smem));
        if (threadIdx.x == 0) p.mdot_part[(size_t)z * nbm + member] = md;
      }
    }
  }
}

}  // namespace lact
